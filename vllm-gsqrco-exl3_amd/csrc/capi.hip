// C ABI of libgguf_mi355x.so (declared in include/gguf_mi355x.h): guards, workspace sizing and
// dispatch to the gfx950 kernels. Host code only; nothing here touches the GPU until every
// guard has passed.
//
// The guards restate the reference's run() type checks (lcpp_shim.cu:767-791) and check_inputs
// (lcpp_shim.cu:690-732) in the same order with the same message fragments, so callers (and the
// CPU guard tests) see the same rejections. Types served: the reference's Route L set (Q2_K,
// Q4_K, Q6_K, IQ2_XXS, IQ2_XS, IQ2_S, IQ3_XXS, IQ3_S, IQ4_XS, IQ1_M; lcpp_shim.cu:676-684).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <mutex>
#include <string>

#include "../../include/gguf_mi355x.h"
#include "gguf_common.h"
#include "split_k.h"

namespace gguf {
hipError_t launch_quantize(const void* x, int dtype, int64_t n, int64_t k, int64_t s01, int type, bool mmq, void* y,
                           hipStream_t stream);
hipError_t launch_gemv_raw(int type, const uint8_t* W, int64_t row_bytes, int nrows, int k, const uint8_t* q8, int n,
                           void* y, int y_dtype, hipStream_t stream);
hipError_t launch_gemm(int type, const uint8_t* W, int64_t row_bytes, int nrows, int k, const uint8_t* q8, int n,
                       void* y, int y_dtype, hipStream_t stream);
hipError_t launch_gemv_packed(const uint8_t* W, int64_t row_bytes, int nrows, int k, const uint8_t* q8, int n,
                              void* y, int y_dtype, hipStream_t stream);
hipError_t launch_quantize_xq(const void* x, int dtype, int64_t n, int64_t k, int64_t s01, int type, bool vec,
                              void* y, hipStream_t stream, uint32_t* zero = nullptr, int zero_words = 0);
hipError_t launch_q8_1_to_xq(const void* q8, int64_t n, int64_t k, int type, void* y, hipStream_t stream,
                             uint32_t* zero = nullptr, int zero_words = 0);
hipError_t launch_gemm_xq(int type, const uint8_t* W, int64_t row_bytes, int nrows, int k, const uint8_t* xq, int n,
                          void* y, int y_dtype, bool mmq, void* split_ws, hipStream_t stream);
int raw_split(int type, int64_t nrows, int64_t k, int64_t n);
int tile_split(int64_t nrows, int64_t k, int64_t n);
hipError_t launch_gemv_packed_x(const uint8_t* W, int64_t row_bytes, int nrows, int k, const void* x, int x_dtype,
                                int64_t s01, int n, void* y, int y_dtype, hipStream_t stream);
bool gemv_rows_supported(int type, int64_t nrows, int64_t row_bytes, int64_t k, int64_t n);
bool gemv_packed_x_supported(int64_t nrows, int64_t k, int64_t n);
hipError_t launch_gemv_rows_x(int type, const uint8_t* W, int64_t row_bytes, int nrows, int k, const void* x,
                              int x_dtype, int64_t s01, int n, void* y, int y_dtype, hipStream_t stream);
bool gemv_rows_x_supported(int type, int64_t nrows, int64_t row_bytes, int64_t k, int64_t n);
bool gemv_mfma4_supported(int type, int64_t nrows, int64_t row_bytes, int64_t k, int64_t n);
bool gemv_generic_x_supported(int type, int64_t nrows, int64_t row_bytes, int64_t k, int64_t n);
bool gemv_iq3xxs_stream_supported(int64_t nrows, int64_t row_bytes, int64_t k, int64_t n, bool fused);
hipError_t launch_gemv_iq3xxs_stream(const uint8_t* W, int64_t row_bytes, int nrows, int k, const void* x,
                                     int x_dtype, int64_t s01, int n, void* y, int y_dtype, hipStream_t stream);
hipError_t launch_gemm_iq3xxs_packed(const uint8_t* W, int64_t row_bytes, int nrows, int k, const uint8_t* xq, int n,
                                     void* y, int y_dtype, hipStream_t stream);
hipError_t launch_gemv_generic_x(int type, const uint8_t* W, int64_t row_bytes, int nrows, int k, const void* x,
                                 int x_dtype, int64_t s01, int n, void* y, int y_dtype, hipStream_t stream);
hipError_t launch_gemm_packed_xq(const uint8_t* W, int64_t row_bytes, int nrows, int k, const uint8_t* xq, int n,
                                 void* y, int y_dtype, void* split_ws, hipStream_t stream);
hipError_t launch_quantize_xh(const void* x, int dtype, int64_t n, int64_t k, int64_t s01, int type, void* y,
                              hipStream_t stream, uint32_t* zero = nullptr, int64_t zero_words = 0);
bool prefill_supported(int type, bool packed);
int64_t prefill_counters(int64_t nrows, int64_t k, int64_t n);
size_t prefill_slot_bytes(int64_t nrows, int64_t k, int64_t n);
bool small_h_supported(int type, bool packed);
bool small_h_range(int type, int64_t nrows, int64_t n);
hipError_t launch_gemm_small_h(int type, bool packed, const uint8_t* W, int64_t row_bytes, int nrows, int k,
                               const uint8_t* xh, int n, void* y, int y_dtype, hipStream_t stream);
double prefill_split_us(int type, bool exact, int64_t nrows, int64_t k, int64_t n);
double prefill_whole_us(int type, bool exact, int64_t nrows, int64_t k, int64_t n);
hipError_t launch_gemm_prefill(int type, bool exact, bool split, const uint8_t* W, int64_t row_bytes, int nrows, int k,
                               const uint8_t* xh, int n, void* y, int y_dtype, float* part, uint32_t* cnt,
                               hipStream_t stream);
hipError_t launch_iq3_pack(int type, uint8_t* w, int64_t rows, int64_t row_bytes, bool unpack, uint8_t* scratch,
                           size_t scratch_bytes, hipStream_t stream);
size_t iq3_pack_scratch_bytes(int64_t rows, int64_t row_bytes);
hipError_t launch_dense(int dtype, const void* W, int64_t ws0, int rows, int k, const void* X, int64_t xs0, int n,
                        void* y, hipStream_t stream);
}  // namespace gguf

namespace {

// the no-allocation entry point's static workspace
constexpr size_t kScratchBytes = GGUF_SCRATCH_BYTES;

thread_local std::string g_err;

int fail(const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_err = buf;
  return GGUF_EINVAL;
}

int hip_fail(hipError_t e, const char* op, const char* what) {
  char buf[512];
  snprintf(buf, sizeof(buf), "%s: HIP error in %s: %s", op, what, hipGetErrorString(e));
  g_err = buf;
  return GGUF_EHIP;
}

const char* op_name(int op) {
  switch (op) {
    case GGUF_OP_MUL_MAT_VEC_Q: return "lcpp_mul_mat_vec_q";
    case GGUF_OP_MUL_MAT_Q: return "lcpp_mul_mat_q";
    case GGUF_OP_MUL_MAT_VEC_IQ3: return "lcpp_mul_mat_vec_iq3";
    case GGUF_OP_MUL_MAT_VEC_IQ3_MMA: return "lcpp_mul_mat_vec_iq3_mma";
    case GGUF_OP_MUL_MAT_VEC_OWN: return "lcpp_mul_mat_vec_own";
    case GGUF_OP_MUL_MAT_MMA_K: return "lcpp_mul_mat_mma_k";
    case GGUF_OP_MUL_MAT_VEC_IQ3_MMA_PACKED: return "lcpp_mul_mat_vec_iq3_mma_packed";
    case GGUF_OP_MUL_MAT_IQ3_PACKED: return "lcpp_mul_mat_iq3_packed";
    default: return "gguf_mul_mat";
  }
}

// lcpp_type_supported (lcpp_shim.cu:676-684)
bool type_served(int64_t t) {
  return t == gguf::kQ4_K || t == gguf::kQ6_K || t == gguf::kIQ3_S || t == gguf::kIQ4_XS || t == gguf::kQ2_K ||
         t == gguf::kIQ2_XXS || t == gguf::kIQ2_XS || t == gguf::kIQ2_S || t == gguf::kIQ3_XXS || t == gguf::kIQ1_M;
}

using gguf::kIQ1_M;
using gguf::kIQ2_S;
using gguf::kIQ3_XXS;

// Q2_K, the IQ2 types, IQ3_XXS and IQ1_M run on the generic kernels: the dot4 GEMV for the decode
// ops, the per-slice MFMA GEMM for the product ops; the packed ops on IQ3_XXS read its unit layout
// (the IQ3 stream GEMV, and the generic GEMM staging the layout's fields into GGUF blocks)
bool generic(int64_t t) { return gguf::generic_type((int)t); }

// the generic types whose product ops run on the xq-layout GEMM (D4 scales); Q2_K's D2S6 layout
// stays on the per-slice GEMM over block_q8_1_mmq
bool generic_xq(int64_t t) { return generic(t) && t != gguf::kQ2_K && t != kIQ1_M; }

bool is_float(int32_t dt) { return dt == GGUF_DT_F32 || dt == GGUF_DT_F16 || dt == GGUF_DT_BF16; }

int64_t elem_size(int32_t dt) { return dt == GGUF_DT_F32 ? 4 : dt == GGUF_DT_U8 ? 1 : 2; }

bool op_packed(int op) { return op == GGUF_OP_MUL_MAT_VEC_IQ3_MMA_PACKED || op == GGUF_OP_MUL_MAT_IQ3_PACKED; }
bool op_gemm(int op) {
  return op == GGUF_OP_MUL_MAT_Q || op == GGUF_OP_MUL_MAT_MMA_K || op == GGUF_OP_MUL_MAT_IQ3_PACKED;
}
bool op_iq3(int op) {
  return op == GGUF_OP_MUL_MAT_VEC_IQ3 || op == GGUF_OP_MUL_MAT_VEC_IQ3_MMA || op_packed(op);
}
// activation-row limits of the ops (lcpp_shim.cu:775-777; mma_k_max_cols = 64)
int64_t op_max_rows(int op) {
  if (op == GGUF_OP_MUL_MAT_Q || op == GGUF_OP_MUL_MAT_IQ3_PACKED) return 0;
  if (op == GGUF_OP_MUL_MAT_MMA_K) return 64;
  if (op == GGUF_OP_MUL_MAT_VEC_IQ3_MMA_PACKED) return 32;
  return 8;
}

// check_inputs (lcpp_shim.cu:690-732). Returns K, or -1 with g_err set.
int64_t check_inputs(const gguf_view* W, const gguf_view* X, int64_t type, int64_t row, int64_t max_rows,
                     const char* op) {
  if (!type_served(type)) return fail("%s: unsupported ggml type %lld", op, (long long)type), -1;
  if (W->ndim != 2 || X->ndim != 2) return fail("%s: W and X must be 2-D", op), -1;
  if (W->dtype != GGUF_DT_U8) return fail("%s: W must be uint8", op), -1;
  if (!is_float(X->dtype)) return fail("%s: X must be fp32, fp16 or bf16", op), -1;
  const int64_t ts = gguf::block_bytes((int)type);
  const int64_t row_bytes = W->size[1];
  if (!(row_bytes > 0 && row_bytes % ts == 0))
    return fail("%s: W row bytes %lld not a multiple of the block size %lld", op, (long long)row_bytes,
                (long long)ts), -1;
  const int64_t k = row_bytes / ts * gguf::kQK;
  if (k % 512 != 0)
    return fail("%s: K=%lld must be a multiple of 512 (no weight tail padding)", op, (long long)k), -1;
  if (!(k <= INT_MAX && W->size[0] <= INT_MAX)) return fail("%s: W too large", op), -1;
  if (!(row > 0 && row <= W->size[0]))
    return fail("%s: row=%lld out of range (W has %lld rows)", op, (long long)row, (long long)W->size[0]), -1;
  if (W->stride[1] != 1) return fail("%s: W inner stride must be 1", op), -1;
  if (!(W->size[0] == 1 || W->stride[0] == row_bytes))
    return fail("%s: W rows must be contiguous (row stride %lld, row bytes %lld)", op, (long long)W->stride[0],
                (long long)row_bytes), -1;
  if (reinterpret_cast<uintptr_t>(W->data) % 16 != 0) return fail("%s: W data must be 16-byte aligned", op), -1;
  if (X->size[1] != k)
    return fail("%s: X has %lld columns, W rows hold K=%lld", op, (long long)X->size[1], (long long)k), -1;
  if (!(X->stride[1] == 1 && (X->size[0] <= 1 || X->stride[0] >= k))) return fail("%s: X inner stride must be 1", op), -1;
  if (max_rows > 0 && X->size[0] > max_rows)
    return fail("%s: at most %lld rows, got %lld", op, (long long)max_rows, (long long)X->size[0]), -1;
  if (X->size[0] > INT_MAX) return fail("%s: X too large", op), -1;
  // device checks last, so host views exercise every guard above and are then rejected
  if (W->device < 0 || X->device < 0) return fail("%s: W and X must be CUDA tensors", op), -1;
  if (W->device != X->device) return fail("%s: W and X must be on the same device", op), -1;
  return k;
}

// run()'s checks (lcpp_shim.cu:767-791) then check_inputs; returns K or -1.
int64_t check_op(int op, const gguf_view* W, const gguf_view* X, int64_t type, int64_t row, const gguf_view* x_q8) {
  if (op < 0 || op >= GGUF_OP_COUNT) return fail("gguf_mul_mat: unknown op %d", op), -1;
  const char* name = op_name(op);
  if (!W || !X) return fail("%s: W and X must be given", name), -1;
  if (op_iq3(op) && !(type == gguf::kIQ3_S || type == kIQ3_XXS))
    return fail("%s: IQ3_S or IQ3_XXS only, got type %lld", name, (long long)type), -1;
  if (op == GGUF_OP_MUL_MAT_VEC_OWN && !(type == gguf::kQ4_K || type == kIQ2_S))
    return fail("%s: Q4_K or IQ2_S only, got type %lld", name, (long long)type), -1;
  if (op == GGUF_OP_MUL_MAT_MMA_K && !(type == gguf::kQ4_K || type == gguf::kIQ4_XS || type == kIQ2_S))
    return fail("%s: Q4_K, IQ4_XS or IQ2_S only, got type %lld", name, (long long)type), -1;
  if (op == GGUF_OP_MUL_MAT_Q && type == kIQ1_M) return fail("%s: no MMQ for IQ1_M", name), -1;
  if (op_packed(op) && row % 16 != 0)
    return fail("%s: row=%lld must be a multiple of 16 (packed 16-row tiles)", name, (long long)row), -1;
  const int64_t k = check_inputs(W, X, type, row, op_max_rows(op), name);
  if (k < 0) return -1;
  if (x_q8) {
    const int64_t q8_bytes = X->size[0] * k / gguf::kQ81 * 36;
    if (!(x_q8->dtype == GGUF_DT_U8 && x_q8->ndim == 1 && x_q8->stride[0] == 1 && x_q8->size[0] >= q8_bytes))
      return fail("%s: x_q8 must be contiguous uint8 with at least %lld bytes", name, (long long)q8_bytes), -1;
    if (reinterpret_cast<uintptr_t>(x_q8->data) % 16 != 0) return fail("%s: x_q8 must be 16-byte aligned", name), -1;
    if (!(x_q8->device >= 0 && x_q8->device == X->device)) return fail("%s: x_q8 must be on X's device", name), -1;
  }
  return k;
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Makes `device` current for the call when it is not already (the reference's DeviceGuard,
// lcpp_shim.cu:796), restoring the caller's device after; no device call when nothing changes,
// so a call inside stream capture makes no device switch.
struct DeviceScope {
  int prev = -1;
  hipError_t err = hipSuccess;
  explicit DeviceScope(int device) {
    int cur = -1;
    err = hipGetDevice(&cur);
    if (err == hipSuccess && cur != device) {
      err = hipSetDevice(device);
      if (err == hipSuccess) prev = cur;
    }
  }
  ~DeviceScope() {
    if (prev >= 0) (void)hipSetDevice(prev);
  }
};

}  // namespace

extern "C" {

const char* gguf_last_error(void) { return g_err.c_str(); }

const char* gguf_version(void) { return "gguf_mi355x 0.1 (gfx950)"; }

int gguf_check_op(int op, const gguf_view* W, const gguf_view* X, int64_t type, int64_t row, const gguf_view* x_q8) {
  g_err.clear();
  return check_op(op, W, X, type, row, x_q8) < 0 ? GGUF_EINVAL : GGUF_OK;
}

size_t gguf_q8_1_bytes(int64_t n, int64_t k, int mmq) {
  return mmq ? (size_t)(n * k / 128 * 144) : (size_t)(n * k / gguf::kQ81 * 36);
}

namespace {

// Decode ops (1..8 rows; the packed IQ3 op up to 32) go to the int8-MFMA GEMM from this many
// activation rows on, measured against the dot4 GEMV at the 27B-layer shapes: the GEMV's time
// grows with every row, the GEMM's is flat up to 16. IQ3_S on plain rows stays on the GEMV.
// The packed decode op quantises X inside the GEMV when the caller gives no x_q8: at one
// activation row on weights of up to 32M values (the attention projections) block by block, and
// at one or two rows on larger weights by quantising all of X into LDS first.
bool packed_fused(int op, int64_t row, int64_t k, int64_t n, bool has_x_q8) {
  return op_packed(op) && !has_x_q8 && gguf::gemv_packed_x_supported(row, k, n);
}

// A Q4_K / IQ4_XS / Q6_K decode op on the row-chunk GEMV with no x_q8 from the caller quantises X
// inside the GEMV at one or two rows where each wave's part of X is small (K <= 8192).
bool rows_fused(int op, int64_t type, int64_t row, int64_t k, int64_t n, bool has_x_q8);

bool xxs_packed(int op, int64_t type);

bool small_fp16_shape(int op, int64_t type, int64_t k, int64_t n);

// The product ops that may run the prefill GEMM (gemm_prefill.hip) by the size that
// gguf_op_workspace_bytes reports, which has room for its activation copy there: from 65 rows on weights
// of 16M values or more (64 for IQ3_XXS and where the fp16 small GEMM's activation layout, the same, served
// 64), from 129 from 8M values, else from 257; Q2_K always, up to the K of which one column tile's copy fits
// the static scratch.
bool prefill_rows(int op, int64_t type, int64_t row, int64_t k, int64_t n) {
  if (!op_gemm(op) || !gguf::prefill_supported((int)type, op_packed(op))) return false;
  if (type == gguf::kQ2_K) return gguf::xh_bytes(16, k, (int)type) <= kScratchBytes;  // K <= 199k
  const int64_t values = row * k;
  if (values < (16 << 20)) return n >= (values >= (8 << 20) ? 129 : 257);
  return n >= (type == kIQ3_XXS || small_fp16_shape(op, type, k, 64) ? 64 : 65);
}

bool q6k_rounded(int64_t type, int64_t row, int64_t n);
double small_us(int64_t type, int64_t row, int64_t k, int64_t n);

// Whether one of them is the faster on the prefill GEMM where the workspace has room for the split plan: a
// tile of 128 weight rows decoded once per step for up to 256 columns, work split evenly over the CUs,
// against the small GEMMs' 16-row tiles that decode the weights again for every 4 column tiles. Measured
// (us per op, graph replays, prefill / the plan it replaces):
//   34816 x 5120, M = 65 / 256 / 512: IQ3_S 85 / 135 / 254 against 143 / 234 / 351, IQ4_XS 95 / 167 /
//   313 against 248 / 388 / 601, Q6_K 118 / 134 / 244 against 311 / 250 / 371, IQ2_S 82 / 130 / 250
//   against 305 / 635 / 1257; 5120 x 6144, M = 65: IQ3_S 33 against 45, Q6_K 38 against 67.
// It costs about 14 us at K = 512 and 18 to 28 where it adds parts, however small the product, so:
//  * weights of fewer than 8M values by the estimates of both plans, 1 us apart (within 1 % of the better
//    one on average over 8 shapes): 512 x 512 M = 257 / 1024 IQ3_S 14 / 15 against 9 / 12, IQ2_S 14 / 15
//    against 11 / 18; 1024 x 1024 M = 257 / 1024 18 / 20 against 13 / 23, 19 / 20 against 17 / 33; 1024 x 2048 M =
//    257 / 1024 IQ3_S 22 / 25 against 16 / 32;
//  * K > 8192 on few rows, where the int8 GEMM of Q4_K, IQ4_XS and Q6_K splits K as well and the prefill
//    GEMM adds up to 17 parts a tile: IQ4_XS 1024 x 17408 M = 65 / 129 39 / 43 against 31 / 53, 2048 x 17408 M
//    = 100 / 129 52 / 61 against 45 / 75, 512 x 17408 M = 160 / 512 / 1024 37 / 59 / 75 against 34 / 50 / 91;
//  * 64 rows of the fp16 small GEMM's types from 24M values: 4096 x 4096 IQ3_S 23 against 18;
//  * Q2_K, whose other GEMM is the per-slice one, by that one's estimate: M = 16 / 32 / 48 on 1024 x 1024 22 /
//    23 / 23 against 11 / 14 / 18, 1024 x 2048 24 / 25 / 25 against 15 / 22 / 28, 12288 x 5120 44 / 45 / 45 against
//    51 / 71 / 98.
bool split_route(int op, int64_t type, int64_t row, int64_t k, int64_t n) {
  if (!prefill_rows(op, type, row, k, n)) return false;
  if (type == gguf::kQ2_K) return small_us(type, row, k, n) > (k <= 512 ? 16 : k <= 1024 ? 22.5 : 25);
  const int64_t values = row * k;
  if (values < (8 << 20))
    return gguf::prefill_split_us((int)type, !q6k_rounded(type, row, n), row, k, n) + 1 < small_us(type, row, k, n);
  if (k > 8192 && row <= 2048 && !op_packed(op) && !generic(type)) return n >= (row <= 512 ? 1024 : 129);
  return n >= 65 || type == kIQ3_XXS || values >= (24 << 20);
}

// Q6_K products with the sub-scale folded into the fp16 operand, rounded beyond 2048 (pf_decode.h): from
// 256 rows on grids of 64 tiles of 128 x 256 or more. Elsewhere its operands are exact, as the int8
// GEMM's are: two MFMAs per slice instead of one.
bool q6k_rounded(int64_t type, int64_t row, int64_t n) {
  return type == gguf::kQ6_K && n >= 256 && (row + 127) / 128 * ((n + 255) / 256) >= 64;
}

// Estimated time of the small GEMM that a product runs without the prefill GEMM, us: K blocks x workgroups
// (a 16-row tile and up to four column tiles) per CU x a block's time in one. Q2_K's per-slice GEMM: a
// workgroup alone on its CU takes about 1.6 times that. Fitted like pf_whole_shape's.
double small_us(int64_t type, int64_t row, int64_t k, int64_t n) {
  const int64_t nct = (n + 15) / 16, nb = k / 256;
  const double tiles = (double)((row + 15) / 16) / 256;
  if (type == gguf::kQ2_K) {
    const double t = (double)std::min<int64_t>(nct, 4);
    const double wgs = std::ceil(tiles * std::max(1.0, (double)nct / 4));
    return 7 + (double)nb * std::max(1.6 * (0.2 + 0.47 * t), wgs * (0.35 + 0.33 * t));
  }
  if (row * k < (8 << 20)) {  // few workgroups: whole rounds of them over the CUs
    double a = 5, b = 4.2, c = 0.78;
    if (type == gguf::kIQ3_S) a = 6, b = 2, c = 0.52;
    if (type == gguf::kQ4_K) a = 6, b = 2.4, c = 0.60;
    if (type == gguf::kIQ4_XS) b = 4, c = 0.62;
    if (type == gguf::kIQ2_XXS) c = 0.65;
    return a + std::ceil(tiles * (double)((nct + 3) / 4)) * (b + c * (double)nb);
  }
  const bool deep = k > 8192;  // IQ3_S and Q4_K run the int8 GEMM instead of the fp16 one
  double per = deep ? 0.78 : 0.76;  // IQ3_XXS, IQ2_S, IQ2_XS
  if (type == gguf::kIQ2_XXS) per = deep ? 0.66 : 0.76;
  if (type == gguf::kIQ3_S) per = deep ? 0.76 : 0.42;
  if (type == gguf::kQ4_K) per = deep ? 0.52 : 0.50;
  if (type == gguf::kQ6_K) per = deep ? 0.64 : 0.94;
  if (type == gguf::kIQ4_XS) per = deep ? 0.56 : 0.60;
  return 12 + (double)nb * per * tiles * (double)((nct + 3) / 4);
}

// Whether a product of prefill_rows runs the prefill GEMM without room for the split plan's parts, in
// whole tiles: a tile walks all of K, so on a grid of few tiles most CUs idle, and the small GEMMs, whose
// 16-row tiles spread the same work, are the faster ones. By the estimates of both. Measured, us, whole
// tiles (their best width) / small GEMM / split plan: 5120 x 17408 M = 100 IQ3_S 140 / 132 / 63, Q2_K 226 /
// 323 / 78, M = 512 IQ3_S 200 / 432 / 145; 5120 x 6144 M = 65 IQ3_S 56 / 38 / 33, Q6_K 80 / 68 / 38; 1024 x
// 5120 M = 512 IQ3_S 52 / 31 / 30; 34816 x 5120 M = 65 IQ3_S 121 / 117 / 85, IQ2_S 121 / 299 / 82. Over 12
// shapes and 14 row counts of each type the choice is within 1 % of the better one on average, at worst
// 18 % (IQ3_S 34816 x 5120 M = 160 194 against 164), and at worst 4 % slower than the GEMM that ran before
// the split plan took the product over.
bool whole_route(int op, int64_t type, int64_t row, int64_t k, int64_t n) {
  return prefill_rows(op, type, row, k, n) &&
         gguf::prefill_whole_us((int)type, !q6k_rounded(type, row, n), row, k, n) < small_us(type, row, k, n);
}

// Where the split plan is the faster one below those rows, but its activation copy is twice the
// int8 layouts': taken when the library sizes the workspace itself (gguf_mul_mat_alloc), so that the
// size that gguf_op_workspace_bytes reports stays the smaller one. From 33 rows on weights of 24M
// values or more (M = 48: Q6_K 5120 x 6144 25 against 33 us, 34816 x 5120 76 against 135; Q4_K 73
// against 111; IQ2_S 17408 x 5120 41 against 53), there packed IQ3_S from 80M values (34816 x 5120 64
// against 80, 5120 x 17408 45 against 49; 8192 x 5120 25 against 24), IQ3_XXS and IQ2_XXS from 48M (8192 x
// 5120 25 against 23, 25 against 22), IQ4_XS with K > 8192 from 64M (3072 x 17408 40 against 34), and
// everything from 49 rows (M = 56: IQ3_S 8192 x 5120 25 against 37; M = 49 IQ4_XS 3072 x 17408 41 against 51);
// not where the fp16 range plan applies (17408 x 5120 M = 48 IQ3_S 42 against 41, Q4_K 45 against 40), nor
// where split_route leaves more rows to the int8 GEMM.
bool split_preferred(int op, int64_t type, int64_t row, int64_t k, int64_t n) {
  if (prefill_rows(op, type, row, k, n) || !op_gemm(op) || !gguf::prefill_supported((int)type, op_packed(op)))
    return split_route(op, type, row, k, n);
  if (small_fp16_shape(op, type, k, n) && gguf::small_h_range((int)type, row, n)) return false;
  if (k > 8192 && row <= 2048 && !op_packed(op) && !generic(type)) return false;
  const int64_t from = type == gguf::kIQ3_S                              ? 80
                       : type == kIQ3_XXS || type == gguf::kIQ2_XXS      ? 48
                       : type == gguf::kIQ4_XS && k > 8192               ? 64
                                                                         : 24;
  return row * k >= (n >= 49 ? 24 << 20 : n >= 33 ? from << 20 : INT64_MAX);
}

int64_t vec_mma_from(int op, int64_t type) {
  if (op_packed(op)) return 5;
  if (type == gguf::kQ4_K || type == gguf::kQ6_K) return 3;
  if (type == gguf::kIQ4_XS) return 5;
  return INT64_MAX;
}

// Bytes per 256-value block of the GGUF-row types with a row-chunk GEMV (0 for the others).
int64_t rows_block_bytes(int64_t type) {
  return type == gguf::kQ4_K ? 144 : type == gguf::kQ6_K ? 210 : type == gguf::kIQ4_XS ? 136 : 0;
}

// The MFMA decode GEMV (Q4_K / IQ4_XS / Q6_K at 2..4 rows, Q4_K / IQ4_XS at one row on long K;
// gemv_mfma4.hip) on a decode op's shape.
bool decode_mfma4(int op, int64_t type, int64_t row, int64_t k, int64_t n) {
  const int64_t bb = rows_block_bytes(type);
  return !op_gemm(op) && !op_packed(op) && bb > 0 && gguf::gemv_mfma4_supported((int)type, row, k / 256 * bb, k, n);
}

// A decode op runs the int8-MFMA small GEMM from vec_mma_from rows on, except at up to four rows
// of Q4_K / IQ4_XS / Q6_K where a GEMV takes the shape (X's q8_1 in LDS): the MFMA decode GEMV
// where it applies, else the row-chunk GEMV.
bool decode_mma(int op, int64_t type, int64_t row, int64_t k, int64_t n) {
  if (n < vec_mma_from(op, type) || decode_mfma4(op, type, row, k, n)) return false;
  const int64_t bb = rows_block_bytes(type);
  return !(op_packed(op) == false && bb > 0 && gguf::gemv_rows_supported((int)type, row, k / 256 * bb, k, n));
}

// A packed op on IQ3_XXS: the weight is in the build's IQ3_XXS unit layout (gguf_iq3_pack).
bool xxs_packed(int op, int64_t type) { return op_packed(op) && type == kIQ3_XXS; }


// A generic type's decode op with X quantised inside the stream GEMV (1-2 rows, K <= 8192).
bool generic_fused(int op, int64_t type, int64_t row, int64_t k, int64_t n) {
  if (xxs_packed(op, type)) return gguf::gemv_iq3xxs_stream_supported(row, k / 256 * 98, k, n, true);
  return gguf::gemv_generic_x_supported((int)type, row, k / 256 * gguf::block_bytes((int)type), k, n);
}

bool rows_fused(int op, int64_t type, int64_t row, int64_t k, int64_t n, bool has_x_q8) {
  if (op_gemm(op) || op_packed(op) || has_x_q8 || decode_mma(op, type, row, k, n) ||
      decode_mfma4(op, type, row, k, n))
    return false;
  const int64_t bb = rows_block_bytes(type);
  return bb > 0 && gguf::gemv_rows_x_supported((int)type, row, k / 256 * bb, k, n);
}

// The MFMA products with K <= 8192 off the prefill GEMM run the fp16 small GEMM (X in the xh
// layout) for packed IQ3_S and Q4_K from 64 activation rows, and below 64 where its
// one-workgroup-per-CU range plan applies (4..5 row tiles per CU; 33..48 rows for IQ3_S, 17..48 for
// Q4_K); the rest the int8 small GEMM (xq layout).
bool small_fp16_shape(int op, int64_t type, int64_t k, int64_t n) {
  return op_gemm(op) && k <= 8192 && n >= 17 && gguf::small_h_supported((int)type, op_packed(op));
}
bool small_fp16(int op, int64_t type, int64_t row, int64_t k, int64_t n) {
  if (!small_fp16_shape(op, type, k, n)) return false;
  return n >= 64 || gguf::small_h_range((int)type, row, n);
}

// The int8 small GEMM on Q4_K / IQ4_XS / Q6_K rows (gemm_raw_kernel): product ops off the prefill
// and the fp16 GEMM's plans, and decode ops from vec_mma_from rows on.
bool raw_gemm(int op, int64_t type, int64_t row, int64_t k, int64_t n) {
  if (op_packed(op) || !(type == gguf::kQ4_K || type == gguf::kIQ4_XS || type == gguf::kQ6_K)) return false;
  if (op_gemm(op)) return !small_fp16(op, type, row, k, n);
  return decode_mma(op, type, row, k, n);
}

// The int8 tile GEMM on packed IQ3_S (gemm_iq3s_tile_kernel), on the same terms.
bool tile_gemm(int op, int64_t type, int64_t row, int64_t k, int64_t n) {
  if (!op_packed(op) || type != gguf::kIQ3_S) return false;
  if (op_gemm(op)) return !small_fp16(op, type, row, k, n);
  return decode_mma(op, type, row, k, n);
}

// Either GEMM's K split over workgroups (split_k.h): the workgroups per tile and the row tiles.
struct SplitPlan {
  int split = 1;
  int64_t tiles = 0;
};

SplitPlan split_plan(int op, int64_t type, int64_t row, int64_t k, int64_t n) {
  SplitPlan p;
  if (raw_gemm(op, type, row, k, n)) p = {gguf::raw_split((int)type, row, k, n), (row + 15) / 16};
  else if (tile_gemm(op, type, row, k, n)) p = {gguf::tile_split(row, k, n), row / 16};
  return p;
}

// Bytes after the xq copy of X that a split GEMM needs (slots, then its counters).
size_t split_ws(int op, int64_t type, int64_t row, int64_t k, int64_t n) {
  const SplitPlan p = split_plan(op, type, row, k, n);
  return gguf::split_ws_bytes(p.split, p.tiles, n);
}

// Bytes of the activation copy of a prefill product, and with its split plan: the copy, the partial sums and
// the tile counters.
size_t prefill_ws(int64_t type, int64_t k, int64_t n) { return align256(gguf::xh_bytes(n, k, (int)type)); }
size_t prefill_split_ws(int64_t type, int64_t row, int64_t k, int64_t n) {
  const size_t slots = gguf::prefill_slot_bytes(row, k, n);
  const size_t cnt = slots ? align256((size_t)gguf::prefill_counters(row, k, n) * 4) : 0;
  return prefill_ws(type, k, n) + slots + cnt;
}

// Workspace bytes of an op off the prefill GEMM.
size_t small_ws(int op, int64_t type, int64_t row, int64_t k, int64_t n, bool has_x_q8) {
  if (generic(type)) {
    if (op_gemm(op)) return align256(generic_xq(type) ? gguf::xq_bytes(n, k) : gguf_q8_1_bytes(n, k, 1));
    return has_x_q8 || generic_fused(op, type, row, k, n) ? 0 : align256(gguf_q8_1_bytes(n, k, 0));
  }
  if (op_gemm(op)) {
    const bool mmq_layout = !op_packed(op) && type == gguf::kIQ3_S;
    if (!mmq_layout && small_fp16(op, type, row, k, n)) return align256(gguf::xh_bytes(n, k, (int)type));
    return align256(mmq_layout ? gguf_q8_1_bytes(n, k, 1) : gguf::xq_bytes(n, k)) + split_ws(op, type, row, k, n);
  }
  if (decode_mma(op, type, row, k, n))  // x_q8 is converted into it
    return align256(gguf::xq_bytes(n, k)) + split_ws(op, type, row, k, n);
  if (packed_fused(op, row, k, n, has_x_q8) || rows_fused(op, type, row, k, n, has_x_q8)) return 0;
  return has_x_q8 ? 0 : align256(gguf_q8_1_bytes(n, k, 0));
}

// How an op runs: off the prefill GEMM, or on it in whole tiles or with K split over the CUs.
enum class Plan { kSmall, kWhole, kSplit };

// The plan of a workspace of `bytes` bytes: the fastest one that fits it (kSmall, which may not fit either,
// if none does).
Plan plan_for(int op, int64_t type, int64_t row, int64_t k, int64_t n, size_t bytes) {
  if (!prefill_rows(op, type, row, k, n) || bytes < prefill_ws(type, k, n)) return Plan::kSmall;
  if (split_route(op, type, row, k, n) && bytes >= prefill_split_ws(type, row, k, n)) return Plan::kSplit;
  return whole_route(op, type, row, k, n) ? Plan::kWhole : Plan::kSmall;
}

}  // namespace

// The larger of the prefill GEMM's activation copy and the small GEMM's workspace where either may run.
size_t gguf_op_workspace_bytes(int op, int64_t type, int64_t row, int64_t k, int64_t n, int has_x_q8) {
  if (n <= 0) return 0;
  const size_t small = small_ws(op, type, row, k, n, has_x_q8 != 0);
  return prefill_rows(op, type, row, k, n) ? std::max(small, prefill_ws(type, k, n)) : small;
}

}  // extern "C"

namespace {

// One product whose guards have passed (check_op returned k): the buffer checks, the plan and the
// launches. Every entry point runs the guards once and then this. fixed_plan: how it runs, or null: as the
// workspace allows (plan_for, asked on X's device).
int run_checked(int op, const gguf_view* W, const gguf_view* X, int64_t type, int64_t row, const gguf_view* x_q8,
                int64_t k, void* y, size_t y_bytes, void* workspace, size_t workspace_bytes, void* stream,
                const Plan* fixed_plan = nullptr) {
  const char* name = op_name(op);
  const int64_t n = X->size[0];
  if (n == 0) return GGUF_OK;
  if (y_bytes < (size_t)(n * row * elem_size(X->dtype))) return fail("%s: output buffer too small", name);
  const bool packed = op_packed(op);
  const bool gemm = op_gemm(op);
  hipStream_t s = (hipStream_t)stream;
  const DeviceScope scope(X->device);
  if (scope.err != hipSuccess) return hip_fail(scope.err, name, "device select");
  // sized on X's device, as the dispatch below decides (some plans depend on its CU count)
  const Plan plan = fixed_plan ? *fixed_plan : plan_for(op, type, row, k, n, workspace_bytes);
  const size_t need = plan == Plan::kSplit   ? prefill_split_ws(type, row, k, n)
                      : plan == Plan::kWhole ? prefill_ws(type, k, n)
                                             : small_ws(op, type, row, k, n, x_q8 != nullptr);
  if (workspace_bytes < need || (need > 0 && !workspace))
    return fail("%s: workspace of %zu bytes needed, got %zu", name, need, workspace_bytes);
  if (reinterpret_cast<uintptr_t>(workspace) % 16 != 0) return fail("%s: workspace must be 16-byte aligned", name);
  hipError_t e;
  const int64_t s01 = n == 1 ? k : X->stride[0];
  const uint8_t* w = (const uint8_t*)W->data;
  const int64_t row_bytes = W->size[1];
  const int ydt = X->dtype;

  if (plan != Plan::kSmall) {
    uint8_t* ws = (uint8_t*)workspace;
    float* part = nullptr;
    uint32_t* cnt = nullptr;
    const bool split = plan == Plan::kSplit;
    const size_t slots = split ? gguf::prefill_slot_bytes(row, k, n) : 0;
    if (slots) {
      part = (float*)(ws + prefill_ws(type, k, n));
      cnt = (uint32_t*)((uint8_t*)part + slots);
    }
    e = gguf::launch_quantize_xh(X->data, X->dtype, n, k, s01, (int)type, ws, s, cnt,
                                 cnt ? gguf::prefill_counters(row, k, n) : 0);
    if (e != hipSuccess) return hip_fail(e, name, "quantize");
    e = gguf::launch_gemm_prefill((int)type, !q6k_rounded(type, row, n), split, w, row_bytes, (int)row, (int)k, ws, (int)n,
                                  y, ydt, part, cnt, s);
    if (e != hipSuccess) return hip_fail(e, name, "gemm");
    return GGUF_OK;
  }

  if (generic(type)) {
    const bool xxs = xxs_packed(op, type);
    if (gemm && generic_xq(type)) {  // the product ops' MMQ arithmetic in the xq layout
      e = gguf::launch_quantize_xq(X->data, X->dtype, n, k, s01, (int)type, false, workspace, s);
      if (e != hipSuccess) return hip_fail(e, name, "quantize");
      e = xxs ? gguf::launch_gemm_iq3xxs_packed(w, row_bytes, (int)row, (int)k, (const uint8_t*)workspace, (int)n, y,
                                               ydt, s)
              : gguf::launch_gemm_xq((int)type, w, row_bytes, (int)row, (int)k, (const uint8_t*)workspace, (int)n, y,
                                     ydt, true, nullptr, s);
      if (e != hipSuccess) return hip_fail(e, name, "gemm");
      return GGUF_OK;
    }
    if (xxs) {  // IQ3_XXS unit layout: the IQ3 stream GEMV
      if (!gguf::gemv_iq3xxs_stream_supported(row, row_bytes, k, 1, false))
        return fail("%s: K=%lld is past the packed IQ3_XXS GEMV's X staging", name, (long long)k);
      if (!x_q8 && generic_fused(op, type, row, k, n)) {
        e = gguf::launch_gemv_iq3xxs_stream(w, row_bytes, (int)row, (int)k, X->data, X->dtype, s01, (int)n, y, ydt, s);
        if (e != hipSuccess) return hip_fail(e, name, "gemv");
        return GGUF_OK;
      }
      const uint8_t* q8 = x_q8 ? (const uint8_t*)x_q8->data : (const uint8_t*)workspace;
      if (!x_q8) {
        e = gguf::launch_quantize(X->data, X->dtype, n, k, s01, (int)type, false, workspace, s);
        if (e != hipSuccess) return hip_fail(e, name, "quantize");
      }
      e = gguf::launch_gemv_iq3xxs_stream(w, row_bytes, (int)row, (int)k, q8, -1, 0, (int)n, y, ydt, s);
      if (e != hipSuccess) return hip_fail(e, name, "gemv");
      return GGUF_OK;
    }
    if (gemm) {  // Q2_K: the product ops' MMQ arithmetic, block_q8_1_mmq and the per-slice MFMA GEMM
      e = gguf::launch_quantize(X->data, X->dtype, n, k, s01, (int)type, true, workspace, s);
      if (e != hipSuccess) return hip_fail(e, name, "quantize");
      e = gguf::launch_gemm((int)type, w, row_bytes, (int)row, (int)k, (const uint8_t*)workspace, (int)n, y, ydt, s);
      if (e != hipSuccess) return hip_fail(e, name, "gemm");
      return GGUF_OK;
    }
    if (!x_q8 && generic_fused(op, type, row, k, n)) {  // quantisation inside the stream GEMV
      e = gguf::launch_gemv_generic_x((int)type, w, row_bytes, (int)row, (int)k, X->data, X->dtype, s01, (int)n, y,
                                      ydt, s);
      if (e != hipSuccess) return hip_fail(e, name, "gemv");
      return GGUF_OK;
    }
    const uint8_t* q8 = x_q8 ? (const uint8_t*)x_q8->data : (const uint8_t*)workspace;
    if (!x_q8) {
      e = gguf::launch_quantize(X->data, X->dtype, n, k, s01, (int)type, false, workspace, s);
      if (e != hipSuccess) return hip_fail(e, name, "quantize");
    }
    // the GEMV takes up to 8 activation rows per launch (the packed decode op allows 32)
    for (int64_t c = 0; c < n; c += 8) {
      const int64_t nc = n - c < 8 ? n - c : 8;
      e = gguf::launch_gemv_raw((int)type, w, row_bytes, (int)row, (int)k, q8 + c * (k / gguf::kQ81) * 36, (int)nc,
                                (uint8_t*)y + c * row * elem_size(X->dtype), ydt, s);
      if (e != hipSuccess) return hip_fail(e, name, "gemv");
    }
    return GGUF_OK;
  }

  // int8-MFMA GEMMs on the xq layout: the product ops with the MMQ arithmetic, the decode ops
  // (from vec_mma_from rows on, see decode_mma) with the decode ops' q8_1 arithmetic or the
  // caller's x_q8
  if ((gemm && (packed || type != gguf::kIQ3_S)) || (!gemm && decode_mma(op, type, row, k, n))) {
    const bool fp16 = small_fp16(op, type, row, k, n);
    // a K-split GEMM's slots and counters follow the xq copy; the quantise launch clears the
    // counters
    uint8_t* sws = nullptr;
    uint32_t* counters = nullptr;
    int nctr = 0;
    const SplitPlan sp = split_plan(op, type, row, k, n);
    if (sp.split > 1) {
      sws = (uint8_t*)workspace + align256(gguf::xq_bytes(n, k));
      counters = (uint32_t*)(sws + gguf::split_part_bytes(sp.split, sp.tiles, n));
      nctr = gguf::split_counters(sp.split, sp.tiles, n);
    }
    if (!gemm && x_q8)
      e = gguf::launch_q8_1_to_xq(x_q8->data, n, k, (int)type, workspace, s, counters, nctr);
    else if (fp16)
      e = gguf::launch_quantize_xh(X->data, X->dtype, n, k, s01, (int)type, workspace, s);
    else
      e = gguf::launch_quantize_xq(X->data, X->dtype, n, k, s01, (int)type, !gemm, workspace, s, counters, nctr);
    if (e != hipSuccess) return hip_fail(e, name, "quantize");
    if (fp16)
      e = gguf::launch_gemm_small_h((int)type, packed, w, row_bytes, (int)row, (int)k, (const uint8_t*)workspace,
                                    (int)n, y, ydt, s);
    else if (packed)
      e = gguf::launch_gemm_packed_xq(w, row_bytes, (int)row, (int)k, (const uint8_t*)workspace, (int)n, y, ydt, sws,
                                      s);
    else
      e = gguf::launch_gemm_xq((int)type, w, row_bytes, (int)row, (int)k, (const uint8_t*)workspace, (int)n, y, ydt,
                               gemm, sws, s);
    if (e != hipSuccess) return hip_fail(e, name, "gemm");
    return GGUF_OK;
  }
  if (gemm) {  // IQ3_S on plain rows: the MMQ layout and the per-slice MFMA GEMM
    e = gguf::launch_quantize(X->data, X->dtype, n, k, s01, (int)type, true, workspace, s);
    if (e != hipSuccess) return hip_fail(e, name, "quantize");
    e = gguf::launch_gemm((int)type, w, row_bytes, (int)row, (int)k, (const uint8_t*)workspace, (int)n, y, ydt, s);
    if (e != hipSuccess) return hip_fail(e, name, "gemm");
    return GGUF_OK;
  }
  if (packed_fused(op, row, k, n, x_q8 != nullptr)) {  // quantisation inside the GEMV
    e = gguf::launch_gemv_packed_x(w, row_bytes, (int)row, (int)k, X->data, X->dtype, s01, (int)n, y, ydt, s);
    if (e != hipSuccess) return hip_fail(e, name, "gemv");
    return GGUF_OK;
  }
  if (rows_fused(op, type, row, k, n, x_q8 != nullptr)) {  // quantisation inside the row-chunk GEMV
    e = gguf::launch_gemv_rows_x((int)type, w, row_bytes, (int)row, (int)k, X->data, X->dtype, s01, (int)n, y, ydt, s);
    if (e != hipSuccess) return hip_fail(e, name, "gemv");
    return GGUF_OK;
  }
  const uint8_t* q8 = (const uint8_t*)workspace;
  if (x_q8) {
    q8 = (const uint8_t*)x_q8->data;
  } else {
    e = gguf::launch_quantize(X->data, X->dtype, n, k, s01, (int)type, false, workspace, s);
    if (e != hipSuccess) return hip_fail(e, name, "quantize");
  }
  e = packed ? gguf::launch_gemv_packed(w, row_bytes, (int)row, (int)k, q8, (int)n, y, ydt, s)
             : gguf::launch_gemv_raw((int)type, w, row_bytes, (int)row, (int)k, q8, (int)n, y, ydt, s);
  if (e != hipSuccess) return hip_fail(e, name, "gemv");
  return GGUF_OK;
}

}  // namespace

extern "C" {

int gguf_mul_mat(int op, const gguf_view* W, const gguf_view* X, int64_t type, int64_t row, const gguf_view* x_q8,
                 void* y, size_t y_bytes, void* workspace, size_t workspace_bytes, void* stream) {
  g_err.clear();
  const int64_t k = check_op(op, W, X, type, row, x_q8);
  if (k < 0) return GGUF_EINVAL;
  return run_checked(op, W, X, type, row, x_q8, k, y, y_bytes, workspace, workspace_bytes, stream);
}

int gguf_mul_mat_alloc(int op, const gguf_view* W, const gguf_view* X, int64_t type, int64_t row,
                       const gguf_view* x_q8, gguf_alloc_fn alloc, void* alloc_ctx, void* stream) {
  g_err.clear();
  const int64_t k = check_op(op, W, X, type, row, x_q8);
  if (k < 0) return GGUF_EINVAL;
  const char* name = op_name(op);
  if (!alloc) return fail("%s: no allocator given", name);
  const int64_t n = X->size[0];
  const size_t y_bytes = (size_t)(n * row * elem_size(X->dtype));
  void* y = alloc(alloc_ctx, GGUF_ALLOC_OUTPUT, y_bytes);
  if (!y && y_bytes) return fail("%s: the allocator returned no output buffer", name);
  if (n == 0) return GGUF_OK;
  const DeviceScope scope(X->device);
  if (scope.err != hipSuccess) return hip_fail(scope.err, name, "device select");
  const Plan plan = split_preferred(op, type, row, k, n) ? Plan::kSplit : Plan::kSmall;
  const size_t need = plan == Plan::kSplit ? prefill_split_ws(type, row, k, n)
                                           : small_ws(op, type, row, k, n, x_q8 != nullptr);
  void* ws = nullptr;
  if (need) {
    ws = alloc(alloc_ctx, GGUF_ALLOC_WORKSPACE, need);
    if (!ws) return fail("%s: the allocator returned no workspace", name);
  }
  return run_checked(op, W, X, type, row, x_q8, k, y, y_bytes, ws, need, stream, &plan);
}

}  // extern "C"

namespace {

// The no-allocation variant's workspace: one statically sized device array per GPU, held until
// the process ends. Host code never uses the array's name as an address (on the host it is only
// a stand-in for the symbol); each device's address comes from hipGetSymbolAddress with that
// device current, once, and is kept here.
__device__ __align__(256) uint8_t scratch[kScratchBytes];

// Whether the no-allocation entry point takes a product whose reported workspace exceeds the scratch: where
// the small GEMM's fits it. Products on large grids of the types whose prefill GEMM has always read the
// fp16 copy are refused with it, as they always were.
bool noalloc_beyond_scratch(int op, int64_t type, int64_t row, int64_t k, int64_t n) {
  const int64_t groups = (row + 127) / 128 * ((n + 255) / 256);
  const bool fp16 = xxs_packed(op, type) ? (n >= 256 && groups >= 32) || (n >= 64 && groups >= 128)
                    : type == gguf::kIQ3_S || type == gguf::kQ4_K || type == gguf::kQ6_K ? n >= 256 && groups >= 64
                                                                                         : false;
  return prefill_rows(op, type, row, k, n) && !fp16 && small_ws(op, type, row, k, n, false) <= kScratchBytes;
}

void* g_scratch_ptr[gguf::kMaxDevices] = {};
std::mutex g_scratch_mu;

// The current device's scratch address (the caller has made X's device current). The first call
// on a device may come inside a caller's stream capture: the symbol lookup runs with the capture
// mode relaxed (gguf::outside_capture).
hipError_t scratch_address(int device, void** out) {
  if (device < 0 || device >= gguf::kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    void* p = nullptr;
    hipError_t e = hipSuccess;
    gguf::outside_capture([&] { e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)); });
    if (e != hipSuccess) return e;
    g_scratch_ptr[device] = p;
  }
  *out = g_scratch_ptr[device];
  return hipSuccess;
}

}  // namespace

extern "C" {

size_t gguf_scratch_bytes(void) { return kScratchBytes; }

int gguf_mul_mat_noalloc(int op, const gguf_view* W, const gguf_view* X, int64_t type, int64_t row,
                         const gguf_view* x_q8, void* y, size_t y_bytes, void* stream) {
  g_err.clear();
  const int64_t k = check_op(op, W, X, type, row, x_q8);
  if (k < 0) return GGUF_EINVAL;
  const char* name = op_name(op);
  const int64_t n = X->size[0];
  if (n == 0) return GGUF_OK;
  const DeviceScope scope(X->device);
  if (scope.err != hipSuccess) return hip_fail(scope.err, name, "device select");
  const size_t need = gguf_op_workspace_bytes(op, type, row, k, n, x_q8 != nullptr);
  if (need > kScratchBytes && !noalloc_beyond_scratch(op, type, row, k, n))
    return fail("%s: needs a %zu-byte workspace, more than the %zu-byte static scratch of the no-allocation "
                "entry point (use gguf_mul_mat with a workspace)", name, need, kScratchBytes);
  if (y_bytes < (size_t)(n * row * elem_size(X->dtype))) return fail("%s: output buffer too small", name);
  void* ws = nullptr;
  const hipError_t e = scratch_address(X->device, &ws);
  if (e != hipSuccess) return hip_fail(e, name, "scratch address");
  // the reported size, not the scratch's: the same plan and so the same bits as with a workspace of that size
  if (need <= kScratchBytes) return run_checked(op, W, X, type, row, x_q8, k, y, y_bytes, ws, need, stream);
  // whole tiles over activation rows in parts whose copy fits the scratch, one after the other on the
  // stream, where that is estimated the faster one; else the small GEMM
  const int64_t es = elem_size(X->dtype);
  int64_t part = (int64_t)(kScratchBytes / gguf::xh_bytes(16, k, (int)type)) * 16;
  if (part >= 256) part -= part % 256;  // whole column groups
  Plan plan = Plan::kSmall;
  if (part > 0) {
    const bool exact = !q6k_rounded(type, row, n);
    const double us = (double)(n / part) * gguf::prefill_whole_us((int)type, exact, row, k, part) +
                      (n % part ? gguf::prefill_whole_us((int)type, exact, row, k, n % part) : 0);
    if (us < small_us(type, row, k, n)) plan = Plan::kWhole;
  }
  if (plan == Plan::kSmall) part = n;
  for (int64_t c = 0; c < n; c += part) {
    gguf_view xp = *X;
    xp.data = (const uint8_t*)X->data + c * X->stride[0] * es;
    xp.size[0] = n - c < part ? n - c : part;
    const int rc = run_checked(op, W, &xp, type, row, x_q8, k, (uint8_t*)y + c * row * es, y_bytes - c * row * es, ws,
                               kScratchBytes, stream, &plan);
    if (rc != GGUF_OK) return rc;
  }
  return GGUF_OK;
}

#define GGUF_OP_Q8(fn, OP)                                                                                    \
  int fn(const gguf_view* W, const gguf_view* X, int64_t type, int64_t row, const gguf_view* x_q8, void* y,   \
         size_t y_bytes, void* ws, size_t ws_bytes, void* stream) {                                           \
    return gguf_mul_mat(OP, W, X, type, row, x_q8, y, y_bytes, ws, ws_bytes, stream);                         \
  }
#define GGUF_OP_OWN(fn, OP)                                                                                  \
  int fn(const gguf_view* W, const gguf_view* X, int64_t type, int64_t row, void* y, size_t y_bytes, void* ws, \
         size_t ws_bytes, void* stream) {                                                                     \
    return gguf_mul_mat(OP, W, X, type, row, nullptr, y, y_bytes, ws, ws_bytes, stream);                      \
  }
GGUF_OP_Q8(gguf_lcpp_mul_mat_vec_q, GGUF_OP_MUL_MAT_VEC_Q)
GGUF_OP_OWN(gguf_lcpp_mul_mat_q, GGUF_OP_MUL_MAT_Q)
GGUF_OP_Q8(gguf_lcpp_mul_mat_vec_iq3, GGUF_OP_MUL_MAT_VEC_IQ3)
GGUF_OP_Q8(gguf_lcpp_mul_mat_vec_iq3_mma, GGUF_OP_MUL_MAT_VEC_IQ3_MMA)
GGUF_OP_Q8(gguf_lcpp_mul_mat_vec_own, GGUF_OP_MUL_MAT_VEC_OWN)
GGUF_OP_OWN(gguf_lcpp_mul_mat_mma_k, GGUF_OP_MUL_MAT_MMA_K)
GGUF_OP_Q8(gguf_lcpp_mul_mat_vec_iq3_mma_packed, GGUF_OP_MUL_MAT_VEC_IQ3_MMA_PACKED)
GGUF_OP_OWN(gguf_lcpp_mul_mat_iq3_packed, GGUF_OP_MUL_MAT_IQ3_PACKED)
#undef GGUF_OP_Q8
#undef GGUF_OP_OWN

int gguf_lcpp_quantize_q8_1(const gguf_view* X, int64_t type, int mmq, int vendored, void* out, size_t out_bytes,
                            void* stream) {
  g_err.clear();
  // lcpp_shim.cu:950-955: one combined guard
  if (!(X && type_served(type) && X->device >= 0 && X->ndim == 2 && X->stride[1] == 1 && X->size[1] % 512 == 0 &&
        !(mmq && type == kIQ1_M) && is_float(X->dtype)))
    return fail("lcpp_quantize_q8_1: bad arguments");
  if (vendored) return fail("lcpp_quantize_q8_1: no vendored quantizer in this build (vendored must be false)");
  const int64_t n = X->size[0], k = X->size[1];
  if (out_bytes < gguf_q8_1_bytes(n, k, mmq)) return fail("lcpp_quantize_q8_1: output buffer too small");
  if (n == 0) return GGUF_OK;
  const DeviceScope scope(X->device);
  if (scope.err != hipSuccess) return hip_fail(scope.err, "lcpp_quantize_q8_1", "device select");
  hipError_t e;
  const int64_t s01 = n == 1 ? k : X->stride[0];
  e = gguf::launch_quantize(X->data, X->dtype, n, k, s01, (int)type, mmq != 0, out, (hipStream_t)stream);
  if (e != hipSuccess) return hip_fail(e, "lcpp_quantize_q8_1", "quantize");
  return GGUF_OK;
}

size_t gguf_iq3_pack_scratch_bytes(int64_t rows, int64_t row_bytes) { return gguf::iq3_pack_scratch_bytes(rows, row_bytes); }

int gguf_dense_mul_mat(const gguf_view* W, const gguf_view* X, void* y, size_t y_bytes, void* stream) {
  g_err.clear();
  const char* name = "gguf_dense_mul_mat";
  if (!W || !X) return fail("%s: W and X must be given", name);
  if (W->ndim != 2 || X->ndim != 2) return fail("%s: W and X must be 2-D", name);
  if (!is_float(W->dtype) || X->dtype != W->dtype) return fail("%s: W and X must share one float dtype", name);
  const int64_t rows = W->size[0], k = W->size[1], n = X->size[0];
  if (X->size[1] != k) return fail("%s: X has %lld columns, W has %lld", name, (long long)X->size[1], (long long)k);
  if (!(k > 0 && k % 32 == 0 && k <= INT_MAX)) return fail("%s: K=%lld must be a positive multiple of 32", name, (long long)k);
  if (!(rows >= 1 && rows <= INT_MAX)) return fail("%s: W must have rows", name);
  if (n > 8) return fail("%s: at most 8 rows, got %lld", name, (long long)n);
  const int64_t es = elem_size(X->dtype);
  if (W->stride[1] != 1 || X->stride[1] != 1) return fail("%s: W and X inner stride must be 1", name);
  if ((rows > 1 && (W->stride[0] < k || (W->stride[0] * es) % 16)) || (n > 1 && (X->stride[0] < k || (X->stride[0] * es) % 16)))
    return fail("%s: row strides must be at least K and 16-byte multiples", name);
  if (reinterpret_cast<uintptr_t>(W->data) % 16 || reinterpret_cast<uintptr_t>(X->data) % 16)
    return fail("%s: W and X data must be 16-byte aligned", name);
  if (W->device < 0 || X->device < 0) return fail("%s: W and X must be CUDA tensors", name);
  if (W->device != X->device) return fail("%s: W and X must be on the same device", name);
  if (n == 0) return GGUF_OK;
  if (y_bytes < (size_t)(n * rows * es)) return fail("%s: output buffer too small", name);
  const DeviceScope scope(X->device);
  if (scope.err != hipSuccess) return hip_fail(scope.err, name, "device select");
  const hipError_t e = gguf::launch_dense(X->dtype, W->data, rows > 1 ? W->stride[0] : k, (int)rows, (int)k, X->data,
                                          n > 1 ? X->stride[0] : k, (int)n, y, (hipStream_t)stream);
  if (e != hipSuccess) return hip_fail(e, name, "gemv");
  return GGUF_OK;
}

int gguf_iq3_pack(void* w, int64_t type, int64_t rows, int64_t row_bytes, int unpack, void* scratch,
                  size_t scratch_bytes, void* stream) {
  g_err.clear();
  if (type != gguf::kIQ3_S && type != kIQ3_XXS)
    return fail("gguf_iq3_pack: IQ3_S or IQ3_XXS only, got type %lld", (long long)type);
  const int64_t bs = type == kIQ3_XXS ? 98 : 110;
  if (!w || rows <= 0 || rows % 16 != 0 || row_bytes <= 0 || row_bytes % bs != 0)
    return fail("gguf_iq3_pack: rows must be a positive multiple of 16 and row bytes whole %s blocks",
                type == kIQ3_XXS ? "IQ3_XXS" : "IQ3_S");
  if (reinterpret_cast<uintptr_t>(w) % 16 != 0) return fail("gguf_iq3_pack: W data must be 16-byte aligned");
  if (scratch_bytes < gguf::iq3_pack_scratch_bytes(rows, row_bytes) || !scratch)
    return fail("gguf_iq3_pack: scratch of %zu bytes needed", gguf::iq3_pack_scratch_bytes(rows, row_bytes));
  const hipError_t e = gguf::launch_iq3_pack((int)type, (uint8_t*)w, rows, row_bytes, unpack != 0, (uint8_t*)scratch,
                                             scratch_bytes, (hipStream_t)stream);
  if (e != hipSuccess) return hip_fail(e, "gguf_iq3_pack", "pack");
  return GGUF_OK;
}

}  // extern "C"

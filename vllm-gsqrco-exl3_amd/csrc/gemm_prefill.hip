// Prefill GEMM (many activation rows) on fp16 MFMA: Y[c, r] = sum_k X[c, k] * W[r, k].
//
// Replaces the reference's large-M products (the IQ3 tiled kernel's wide plans,
// lcpp_owned_iq3_mma.cu:1022-1055, and vendored MMQ, mmq.cuh / mmq-load-tiles.cuh) for every type
// with a product op but IQ1_M (and IQ3 on GGUF rows).
//
// Arithmetic. The operand of a weight is its value times its sub-scale, an exact fp16 integer
// (pf_decode.h), the operand of an activation its q8 value (the xh layout, xq.h). One
// v_mfma_f32_16x16x32_f16 with a zero accumulator returns sub-scale x integer slice dot, exactly
// (every partial sum is an integer below 2^24), and the per-slice epilogue is one FMA by the
// activation scale (IQ4_XS: a multiply by the sub-scale first). The row's block scale d is not
// applied per slice: each row's accumulator is held in units of the d of the block being summed (e,
// the last nonzero d; a block with d = 0 decodes to zeros), and is multiplied by e_prev / e_cur when
// a new block starts and by the last e at the end. The min term of Q4_K, sum over slices of (-dmin / e)
// m_g s_g, is an integer-weighted sum of the activation sums s_g: one bf16 MFMA per block over m_g
// (exact in bf16) and s_g in bf16 pieces that add up to it exactly, then one FMA per output by -dmin /
// e. Q2_K rounds d times its sub-scale to fp16 (f), so its operands are f (q - 1) in units of a power of
// two and the slices are no integers: the two slices of 64 values, which share an activation scale, and
// the sum f x (sum of q8) that makes up for the - 1 are one chain of three MFMAs (one for f of 4 groups),
// one FMA per output and chain; its mins, over 16-value groups with the fp16 of dmin m_g, are two bf16
// MFMAs per half block (two pieces of it) onto the accumulator. 12288 x 5120, M = 24 / 512 / 1024: 44 / 133
// / 248 us; with 3f rounded off into a second plane of operands, four MFMAs per 64 values, 48 / 191 /
// 358; with d left outside (f not rounded) 40 / 132 / 253.
//
// Workgroup: 8 waves over 128 weight rows x 256 / RS activation rows. Wave w owns 2 column tiles of
// 16 and 8 / RS of the 8 row tiles (RS row parts share a column pair). Its B operands come straight
// from global memory into registers one step (half a K block) ahead; the decoded weights are shared
// through LDS, double-buffered, with one LDS-only barrier per step.
//
// What bounds it: MFMA and VALU work of a SIMD hardly overlap (counters at 17408 x 5120 M = 8192, IQ3_S: the
// matrix cores busy 39 % of the cycles, 20 of them per MFMA, and 6.7e8 VALU instructions of 4 cycles each,
// 57 %: together 96 %), so a step's time is their sum plus what is waited for. The decode of the next step
// is therefore cut into four parts that run between the MFMA groups of the four slices (table reads
// of a part at the start of its slice, its operands stored at the end), so that its LDS latencies
// and the raw loads (a step ahead, two register sets) hide under the MFMAs, and IQ3's two table
// reads per 8 values are 4 bytes each (a signed table biased by 128; the fp16 grid and sign masks it
// replaced took four times the LDS bytes).
//
// Work split: persistent workgroups (one per CU) over equal contiguous runs of (tile, K block)
// units, so a grid of 272 tiles takes 272 / 256 rounds, not 2. A run that ends inside a tile leaves
// its sums in its own slot of the workspace and counts itself in; the workgroup whose count
// completes the tile adds all parts in K order and writes the output, so the result does not depend
// on which one that is, and nothing waits.
#include <algorithm>
#include <type_traits>

#include "decode.h"
#include "iq3_tile.h"
#include "pf_decode.h"
#include "xh_decode.h"
#include "xq.h"

namespace gguf {

namespace {

typedef __bf16 b8 __attribute__((ext_vector_type(8)));

constexpr int kPfRowTiles = 8;  // 128 weight rows per workgroup
constexpr int kPfWaves = 8;
constexpr int kPfThreads = 64 * kPfWaves;

// The split of a launch: `units` runs of `ub` K blocks over the grid's workgroups; workgroup w takes
// units [w per + min(w, rem), ...), per or per + 1 of them.
struct PfPlan {
  int64_t per, rem;
  int ub;         // K blocks per unit: 1, or nb where there is no room for partial sums
  int nrg;        // row groups; tile t = column group t / nrg, row group t % nrg
  bool few;       // fewer tiles than workgroups (the numbering of the slots)
};

__device__ __forceinline__ int64_t pf_begin(const PfPlan& p, int64_t w) { return w * p.per + min(w, p.rem); }
// the workgroup that unit x belongs to
__device__ __forceinline__ int64_t pf_owner(const PfPlan& p, int64_t x) {
  const int64_t big = p.rem * (p.per + 1);
  return x < big ? x / (p.per + 1) : p.rem + (x - big) / p.per;
}

// Barrier that orders LDS only: __syncthreads()'s fences also order global memory, for which the
// compiler may wait for loads still in flight. The scheduling barriers keep each step's code in it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  __builtin_amdgcn_sched_barrier(0);
}

// four consecutive rows of one column; vec: their bytes are aligned as a whole
__device__ __forceinline__ void store_y4(void* y, int64_t i, f4 v, int y_dtype, bool vec, int rows) {
  if (vec) {
    if (y_dtype == kF32) {
      *(f4*)((float*)y + i) = v;
    } else if (y_dtype == kF16) {
      uint32_t h[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = __half_as_ushort(__float2half_rn(v[e]));
      *(uint2*)((uint16_t*)y + i) = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
    } else {
      uint32_t h[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = f32_to_bf16_bits(v[e]);
      *(uint2*)((uint16_t*)y + i) = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < rows) store_y(y, i + e, v[e], y_dtype);
  }
}

template <int TYPE, int RS>
__global__ void __launch_bounds__(kPfThreads) gemm_prefill_h_kernel(const uint8_t* __restrict__ W, int64_t row_bytes,
                                                                    int nrows, int k, const uint8_t* __restrict__ xh,
                                                                    int nct, int n, void* __restrict__ y, int y_dtype,
                                                                    PfPlan plan, float* __restrict__ part,
                                                                    uint32_t* __restrict__ cnt) {
  using Dec = PfDec<TYPE>;
  using Raw = typename Dec::Raw;
  constexpr bool IQ3 = pf_iq3(TYPE);   // the unit layouts: a 16-row tile is 4 units
  constexpr bool MIN = pf_min(TYPE);   // the min term
  constexpr int AMH = TYPE == kQ2_K ? 5120 : 2048;  // min operands of a half
  constexpr bool SUB = TYPE == kIQ4_XS;  // sub-scales applied to the dots
  constexpr bool LO = TYPE == kQ6_KX;   // two planes of operands, added in the MFMA
  // slices 2i, 2i + 1 in one chain of MFMAs: they share an activation scale (D2S6); the chain ends with
  // the sum that the operands' offset needs (pf_decode.h)
  constexpr bool PAIR = TYPE == kQ2_K;
  constexpr int RT = kPfRowTiles / RS;  // row tiles per wave
  constexpr int CG = kPfWaves / RS;     // column pairs per workgroup
  // row tiles per MFMA group: 4 MFMAs and their 16 FMAs in a row beat 2 and 8 by 3 %; with sub-scales
  // or two planes two row tiles' operands spill
  constexpr int GR = SUB || LO || PAIR ? 1 : 2;
  constexpr int NG = RT / GR;           // groups per slice (PAIR: per two slices)
  constexpr int GS = PAIR ? 2 : 4;      // groups of NG per step
  constexpr int AD = GR == 1 && !PAIR ? 2 : 1;  // groups ahead that A operands are read
  constexpr int BD = RS == 1 ? 1 : 2;   // steps ahead that B operands are loaded
  constexpr int SU = xh_scale_unit(TYPE);
  constexpr int TB = pf_table_bytes(TYPE);
  constexpr int kPfA = (LO ? 2 : 1) * kPfPlane;  // operands of a step
  __shared__ __attribute__((aligned(16))) uint8_t A[2 * kPfA];
  __shared__ __attribute__((aligned(16))) float RTs[128 + kPfRowTiles];
  __shared__ __attribute__((aligned(16))) float EFs[128];
  __shared__ __attribute__((aligned(16))) float RMs[TYPE == kQ4_K ? 128 : 4];
  __shared__ __attribute__((aligned(16))) uint16_t AMs[MIN ? 2 * AMH : 8];
  __shared__ __attribute__((aligned(16))) float LSs[SUB ? 2 * 512 : 4];
  __shared__ __attribute__((aligned(16))) uint4 tbl[TB ? TB / 16 : 1];
  __shared__ uint32_t last_flag;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, q = lane >> 4;
  int dj, dq;  // decode lane: row of the tile, index
  pf_lane(IQ3, lane, dj, dq);
  const int ntiles = (nrows + 15) / 16;
  const int nb = k / kQK;
  const int cw = wave % CG, r0 = wave / CG * RT;  // column pair and first row tile of this wave
  // 4 rows of a column in one store
  const bool vec = nrows % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;

  if constexpr (TB > 0) {
    const uint4* src = pf_table<TYPE>();
    for (int i = threadIdx.x; i < TB / 16; i += kPfThreads) tbl[i] = src[i];
  }
  const PfLds L0 = {A, RTs, EFs, AMs, RMs, LSs, (const uint8_t*)tbl};
  const PfLds L1 = {A + kPfA, RTs, EFs, AMs + (MIN ? AMH : 0), RMs, LSs + (SUB ? 512 : 0),
                    (const uint8_t*)tbl};

  // consecutive workgroups go round the 8 XCDs: give each XCD a contiguous range of units, so that
  // its workgroups share a column group (X stays in its L2)
  const int64_t nwg = gridDim.x;
  const int64_t wg = (nwg & 7) == 0 ? (int64_t)(blockIdx.x & 7) * (nwg >> 3) + (blockIdx.x >> 3) : (int64_t)blockIdx.x;
  int64_t at = pf_begin(plan, wg) * plan.ub;
  const int64_t end = pf_begin(plan, wg + 1) * plan.ub;

  while (at < end) {
    const int64_t tile = at / nb;
    const int b0 = (int)(at - tile * nb);
    const int b1 = (int)min((int64_t)nb, (int64_t)b0 + (end - at));
    at += b1 - b0;
    const int cgp = (int)(tile / plan.nrg), rg = (int)(tile % plan.nrg);
    const int tile0 = rg * kPfRowTiles;

    // this wave's column tiles (past nct: the last one again, never stored)
    const uint8_t* xv[2];
    const uint8_t* xs[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int ct = min((cgp * CG + cw) * 2 + c, nct - 1);
      xv[c] = xh + (int64_t)ct * nb * kXhUnit + 16 * lane;
      xs[c] = xh + xh_scale_base(nct, nb) + (int64_t)ct * nb * SU;
    }
    u32x4 bqs[BD][2][4];
    float dx[2][4];
    f4 dxn[2];
    u32x4 mb[2];  // the min term's activation sums of the coming step
    auto load_bq = [&](u32x4 (&bq)[2][4], int c, int u, int b, int h) {
      bq[c][u] = *(const u32x4*)(xv[c] + (int64_t)b * kXhUnit + 4096 * h + 1024 * u);
    };
    auto load_scales = [&](int b, int h) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const uint8_t* s = xs[c] + (int64_t)b * SU;
        dxn[c] = *(const f4*)(s + 32 * j + 16 * h);
        if constexpr (TYPE == kQ4_K)
          if (h == 0) mb[c] = *(const u32x4*)(s + 512 + 32 * j + 16 * (q & 1));
        if constexpr (TYPE == kQ2_K) mb[c] = *(const u32x4*)(s + 512 + 1024 * h + 64 * j + 16 * q);
      }
    };
    auto take_scales = [&]() {
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int u = 0; u < 4; ++u) dx[c][u] = dxn[c][u];
    };
    // the row tile this wave decodes (tiles past the weight's end, rows past nrows: copies of the
    // last, never stored)
    const uint8_t* wp;
    if constexpr (IQ3) wp = W + (int64_t)min(tile0 + wave, ntiles - 1) * kTileRows * row_bytes;
    else wp = W + (int64_t)min((tile0 + wave) * 16 + dj, nrows - 1) * row_bytes;

    float e = 1.0f;
    Raw raw0, raw1;
    f4 acc[RT][2];
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r][0] = acc[r][1] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    const f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};

    // One step: the 4 slices of half H of the block in A[H], with the decode of the following half
    // (raw bytes `raw`) into the other buffer; bnx: the block whose half 1 - H is the next step; bld:
    // the next block; braw: the block whose half 1 - H is decoded two steps on
    auto step = [&](auto HC, int bnx, Raw& raw, int bld, int braw) {
      constexpr int H = decltype(HC)::value;
      constexpr int HN = 1 - H;
      const uint8_t* Ab = A + H * kPfA;
      const PfLds& LN = H == 0 ? L1 : L0;
      typename Dec::Ctx ctx;
      typename Dec::Tmp tmp[2];
      u32x4 mbc[2];
      if constexpr (MIN) {  // before load_scales overwrites them
        mbc[0] = mb[0];
        mbc[1] = mb[1];
      }
      // the LDS reads that the step starts with go out first: what follows covers their latency
      h8 a[AD + 1][GR];  // the A operands (and sub-scales) of groups g .. g + AD
      h8 al[AD + 1][GR];
      f4 ls[AD + 1][GR];
      f4 p[GR][2];
      auto read_a = [&](int g) {
        const int u = g / NG * (4 / GS), r = g % NG * GR;
        if constexpr (PAIR) al[g % (AD + 1)][0] = *(const h8*)(Ab + pf_off(r0 + r, u + 1, j, q));
#pragma unroll
        for (int i = 0; i < GR; ++i) {
          a[g % (AD + 1)][i] = *(const h8*)(Ab + pf_off(r0 + r + i, u, j, q));
          if constexpr (LO) al[g % (AD + 1)][i] = *(const h8*)(Ab + kPfPlane + pf_off(r0 + r + i, u, j, q));
          if constexpr (SUB)
            ls[g % (AD + 1)][i] = *(const f4*)((H == 0 ? L0.LS : L1.LS) + ((r0 + r + i) * 4 + u) * 16 + 4 * q);
        }
      };
#pragma unroll
      for (int g = 0; g < AD; ++g) read_a(g);
      load_scales(bnx, HN);
      u32x4 (&bq)[2][4] = bqs[BD == 1 ? 0 : H];
      __builtin_amdgcn_sched_barrier(0);
      Dec::begin(raw, ctx, HN, e, LN, wave, dj, dq);
      Dec::template issue<0>(ctx, tmp[0], LN);
      // a new block: rescale the rows to its e; the min term
      if constexpr (PAIR) {
        // the mins' first pieces on all three pieces of the sums (q = 0, 1, 2), their second ones on the
        // first two; an infinite min meets the first piece only, which is 0 where the sum is (0 x inf
        // elsewhere would make a NaN of an inf)
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          const uint16_t* am = (H == 0 ? L0.AM : L1.AM) + ((r0 + r) * 16 + j) * 8;
          const b8 hi = __builtin_bit_cast(b8, *(const u32x4*)(am + (q == 0 ? 0 : 2048))),
                   lo = __builtin_bit_cast(b8, *(const u32x4*)(am + 1024));
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            const u32x4 b3 = q < 3 ? mbc[c] : u32x4{0, 0, 0, 0}, b2 = q < 2 ? mbc[c] : u32x4{0, 0, 0, 0};
            acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, __builtin_bit_cast(b8, b3), acc[r][c], 0, 0, 0);
            acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, __builtin_bit_cast(b8, b2), acc[r][c], 0, 0, 0);
          }
        }
      } else if constexpr (H == 0) {
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          const f4 rt = *(const f4*)(RTs + (r0 + r) * 16 + 4 * q);
          if constexpr (MIN) {
            const f4 rm = *(const f4*)(RMs + (r0 + r) * 16 + 4 * q);
            const b8 am8 = __builtin_bit_cast(b8, *(const u32x4*)(AMs + ((r0 + r) * 16 + j) * 16 + 8 * (q & 1)));
#pragma unroll
            for (int c = 0; c < 2; ++c) {
              const u32x4 bz = q < 2 ? mbc[c] : u32x4{0, 0, 0, 0};
              const f4 pm = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am8, __builtin_bit_cast(b8, bz), zero, 0, 0, 0);
#pragma unroll
              for (int v = 0; v < 4; ++v) {
                acc[r][c][v] *= rt[v];
                acc[r][c][v] = fmaf(pm[v], rm[v], acc[r][c][v]);
              }
            }
          } else {
            acc[r][0] *= rt;
            acc[r][1] *= rt;
          }
        }
      }
      if constexpr (PAIR) {  // of mbc the chains use what lanes q == 3 hold
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i) mbc[c][i] = q == 3 ? mbc[c][i] : 0;
      }
      __builtin_amdgcn_sched_barrier(0);
      // group g = (slice, GR row tiles): the A operands AD groups on are read, 2 GR MFMAs issued, and
      // the previous group's results folded into acc
      auto fold = [&](int g, const f4 (&lg)[GR]) {
        const int u = g / NG * (4 / GS), r = g % NG * GR;
#pragma unroll
        for (int i = 0; i < GR; ++i)
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              const float x = SUB ? p[i][c][v] * lg[i][v] : p[i][c][v];
              acc[r + i][c][v] = fmaf(x, dx[c][u], acc[r + i][c][v]);
            }
      };
#define GGUF_PF_SLICE(U)                                                                                              \
  if constexpr (U < 3) Dec::template issue<(U < 3 ? U + 1 : 3)>(ctx, tmp[(U + 1) & 1], LN);                           \
  if constexpr (!PAIR || (U & 1) == 0) _Pragma("unroll") for (int gr = 0; gr < NG; ++gr) {                            \
    const int g = U * GS / 4 * NG + gr;                                                                               \
    f4 nx[GR][2], lg[GR];                                                                                             \
    if constexpr (SUB) _Pragma("unroll") for (int i = 0; i < GR; ++i) lg[i] = ls[(g + AD) % (AD + 1)][i];             \
    if ((GR > 1 || PAIR) && g + AD < GS * NG) read_a(g + AD);                                                         \
    h8 af;                                                                                                            \
    if constexpr (PAIR) af = *(const h8*)((H == 0 ? L0.AM : L1.AM) + 3072 + 512 * U + ((r0 + gr) * 16 + j) * 8);      \
    _Pragma("unroll") for (int i = 0; i < GR; ++i) _Pragma("unroll") for (int c = 0; c < 2; ++c) nx[i][c] =           \
        __builtin_amdgcn_mfma_f32_16x16x32_f16(a[g % (AD + 1)][i], __builtin_bit_cast(h8, bq[c][U]), zero, 0, 0, 0);  \
    if constexpr (LO || PAIR) _Pragma("unroll") for (int i = 0; i < GR; ++i) _Pragma("unroll") for (int c = 0; c < 2; \
                                                                                                    ++c)              \
        nx[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(                                                            \
            al[g % (AD + 1)][i], __builtin_bit_cast(h8, bq[c][PAIR ? U | 1 : U]), nx[i][c], 0, 0, 0);                 \
    if constexpr (PAIR) _Pragma("unroll") for (int c = 0; c < 2; ++c) nx[0][c] =                                      \
        __builtin_amdgcn_mfma_f32_16x16x32_f16(af, __builtin_bit_cast(h8, mbc[c]), nx[0][c], 0, 0, 0);                \
    if (g > 0) fold(g - 1, lg);                                                                                       \
    if (GR == 1 && !PAIR && g + AD < GS * NG) read_a(g + AD);                                                         \
    _Pragma("unroll") for (int i = 0; i < GR; ++i) _Pragma("unroll") for (int c = 0; c < 2; ++c) p[i][c] = nx[i][c];  \
    __builtin_amdgcn_sched_barrier(0);                                                                                \
  }                                                                                                                   \
  load_bq(bq, 0, U, BD == 1 ? bnx : bld, BD == 1 ? HN : H);                                                           \
  load_bq(bq, 1, U, BD == 1 ? bnx : bld, BD == 1 ? HN : H);                                                           \
  Dec::template finish<U>(ctx, tmp[U & 1], LN, wave, dj, dq);                                                         \
  __builtin_amdgcn_sched_barrier(0);
      GGUF_PF_SLICE(0)
      GGUF_PF_SLICE(1)
      GGUF_PF_SLICE(2)
      GGUF_PF_SLICE(3)
#undef GGUF_PF_SLICE
      // last, so that no wait for B operands or scales waits for it: loads return in order
      Dec::load(raw, wp, row_bytes, nb, braw, HN, dj, dq);
      fold(GS * NG - 1, ls[(GS * NG - 1) % (AD + 1)]);
      take_scales();
    };

    // prologue: the first half decoded, the second's raw bytes and the first's operands in flight
    Dec::load(raw0, wp, row_bytes, nb, b0, 0, dj, dq);
    Dec::load(raw1, wp, row_bytes, nb, b0, 1, dj, dq);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
      for (int h = 0; h < BD; ++h) {
        load_bq(bqs[h], 0, u, b0, h);
        load_bq(bqs[h], 1, u, b0, h);
      }
    }
    load_scales(b0, 0);
    __syncthreads();  // the table; the previous tile's readers of A, RT and EF are done
    {
      typename Dec::Ctx ctx;
      typename Dec::Tmp tmp;
      Dec::begin(raw0, ctx, 0, e, L0, wave, dj, dq);
      Dec::template issue<0>(ctx, tmp, L0);
      Dec::template finish<0>(ctx, tmp, L0, wave, dj, dq);
      Dec::template issue<1>(ctx, tmp, L0);
      Dec::template finish<1>(ctx, tmp, L0, wave, dj, dq);
      Dec::template issue<2>(ctx, tmp, L0);
      Dec::template finish<2>(ctx, tmp, L0, wave, dj, dq);
      Dec::template issue<3>(ctx, tmp, L0);
      Dec::template finish<3>(ctx, tmp, L0, wave, dj, dq);
    }
    take_scales();
    Dec::load(raw0, wp, row_bytes, nb, min(b0 + 1, b1 - 1), 0, dj, dq);
    lds_barrier();
    for (int b = b0; b < b1; ++b) {
      const int bn = min(b + 1, b1 - 1);  // past the end: the last block again (never used; its
                                          // decode leaves e and EF as they are)
      step(std::integral_constant<int, 0>{}, b, raw1, bn, bn);
      lds_barrier();
      step(std::integral_constant<int, 1>{}, bn, raw0, bn, min(b + 2, b1 - 1));
      lds_barrier();
      if constexpr (PAIR) {  // the rows' e has moved: hardly ever
        if (__any(RTs[128 + (lane & 7)] != 0.0f)) {
#pragma unroll
          for (int r = 0; r < RT; ++r) {
            const f4 rt = *(const f4*)(RTs + (r0 + r) * 16 + 4 * q);
            acc[r][0] *= rt;
            acc[r][1] *= rt;
          }
        }
      }
    }
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const f4 ef = *(const f4*)(EFs + (r0 + r) * 16 + 4 * q);
      acc[r][0] *= ef;
      acc[r][1] *= ef;
    }

    if (b1 - b0 < nb) {  // a part of the tile's K
      constexpr int kSlot = RT * 2 * kPfThreads * 4;  // floats
      const int64_t first = pf_owner(plan, tile * nb);
      const int parts = (int)(pf_owner(plan, tile * nb + nb - 1) - first) + 1;
      const int mine = (int)(wg - first);
      // slot of a workgroup's part: 2 w where the part continues a tile, 2 w + 1 where it starts one; or
      // w + tile, which grows with every part in turn
      auto slot_of = [&](int i) {
        return part + (plan.few ? first + i + tile : (first + i) * 2 + (i == 0 ? 1 : 0)) * kSlot;
      };
      uint64_t* out = (uint64_t*)slot_of(mine);
#pragma unroll
      for (int i = 0; i < RT * 2; ++i) {
        const f4 v = acc[i >> 1][i & 1];
        const uint64_t lo = (uint64_t)__float_as_uint(v[0]) | ((uint64_t)__float_as_uint(v[1]) << 32);
        const uint64_t hi = (uint64_t)__float_as_uint(v[2]) | ((uint64_t)__float_as_uint(v[3]) << 32);
        __hip_atomic_store(out + (2 * i) * kPfThreads + threadIdx.x, lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(out + (2 * i + 1) * kPfThreads + threadIdx.x, hi, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      }
      // every wave's stores are complete before the workgroup counts itself in
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (threadIdx.x == 0)
        last_flag = __hip_atomic_fetch_add(cnt + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      if (last_flag != (uint32_t)parts - 1) continue;
      asm volatile("" ::: "memory");
      // all parts in K order; this workgroup's own come from its registers
      f4 own[RT * 2];
#pragma unroll
      for (int i = 0; i < RT * 2; ++i) own[i] = acc[i >> 1][i & 1];
      for (int z = 0; z < parts; ++z) {
        uint64_t* in = (uint64_t*)slot_of(z);
#pragma unroll
        for (int i = 0; i < RT * 2; ++i) {
          f4 v = own[i];
          if (z != mine) {
            const uint64_t lo = __hip_atomic_load(in + (2 * i) * kPfThreads + threadIdx.x, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT);
            const uint64_t hi = __hip_atomic_load(in + (2 * i + 1) * kPfThreads + threadIdx.x, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT);
            v = f4{__uint_as_float((uint32_t)lo), __uint_as_float((uint32_t)(lo >> 32)), __uint_as_float((uint32_t)hi),
                   __uint_as_float((uint32_t)(hi >> 32))};
          }
          acc[i >> 1][i & 1] = z == 0 ? v : acc[i >> 1][i & 1] + v;
        }
      }
    }

    const int col0 = (cgp * CG + cw) * 2 * kXqCols + j;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const int t = tile0 + r0 + r;
      const int row = t * 16 + 4 * q;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int col = col0 + c * kXqCols;
        if (col < n && row < nrows) store_y4(y, (int64_t)col * nrows + row, acc[r][c], y_dtype, vec, nrows - row);
      }
    }
  }
}

// The split of one product: row parts (a workgroup's columns are 256 / rs), tiles of 128 rows x those
// columns, workgroups.
struct PfShape {
  int rs;
  int64_t tiles, wgs;
};

// At most one workgroup per CU, each of at least 4 K blocks (a part of a tile costs its workgroup
// about two blocks' time to publish and another to add up). rs: least estimated time, in us
// fixed(rs) + blocks per workgroup x block(rs), a block's time growing with the workgroups at work.
// IQ3_S, K = 5120, slopes and intercepts over rows and K splits: block 3.5 / 2.3 / 1.7 us with a few
// workgroups and 5.6 / 3.0 / 2.3 with 256 for rs = 1 / 2 / 4, fixed 20 / 16 / 14. Measured at rs =
// 1 / 2 / 4: 1024 rows M = 256 47 / 32 / 25 us, 8192 rows M = 128 51 / 36 / 36, 34816 rows M = 100
// 130 / 86 / 111, M = 512 254 / 304 / 415. For the other types it takes the fastest rs as well, within 1 %
// on average over 12 shapes and 14 row counts each, at worst 19 % (6144 x 2048 M = 300 IQ4_XS, 40 us at rs = 2
// against 33 at 4).
PfShape pf_shape(int64_t nrows, int64_t k, int64_t n, double* us = nullptr) {
  static const double fixed[3] = {20, 16, 14}, few[3] = {3.5, 2.3, 1.7}, full[3] = {5.6, 3.0, 2.3};
  const int64_t nct = xq_col_tiles(n), nb = k / kQK, nrg = (nrows + 127) / 128, cus = device_cus();
  PfShape best{1, 0, 0};
  double least = 0;
  for (int i = 0; i < 3; ++i) {
    const int rs = 1 << i;
    const int64_t per = 16 / rs, tiles = nrg * ((nct + per - 1) / per), units = tiles * nb;
    const int64_t wgs = std::max<int64_t>(1, std::min<int64_t>(cus, units / 4));
    const double t = fixed[i] + (double)((units + wgs - 1) / wgs) * (few[i] + (full[i] - few[i]) * (double)wgs / (double)cus);
    if (i == 0 || t < least) least = t, best = {rs, tiles, wgs};
  }
  if (us) *us = least;
  return best;
}

// Whole tiles, where there is no room for parts: the rounds of tiles over the CUs, each whole[rs] + K
// blocks x block[cost class][rs] us, least squares over 12 shapes (1024 x 5120 .. 34816 x 5120, K 2048 ..
// 17408) and 65 .. 2048 rows, errors within -24 .. +14 % where one round fills few CUs, 10 % elsewhere.
// Measured at rs = 1 / 2 / 4: IQ3_S 5120 x 6144 M = 128 112 / 77 / 58 us, M = 1024 125 / 162 / 167; 34816 x
// 5120 M = 512 299 / 314 / 408.
PfShape pf_whole_shape(int type, bool exact, int64_t nrows, int64_t k, int64_t n, double* us) {
  static const double whole[3] = {14, 11, 8.5}, block[3][3] = {{4.1, 2.75, 2.0}, {5.5, 3.3, 2.2}, {6.2, 4.2, 3.2}};
  const int cost = type == kIQ4_XS ? 1 : type == kQ2_K || (type == kQ6_K && exact) ? 2 : 0;
  const int64_t nct = xq_col_tiles(n), nb = k / kQK, nrg = (nrows + 127) / 128, cus = device_cus();
  PfShape best{1, 0, 0};
  for (int i = 0; i < 3; ++i) {
    const int64_t per = 16 >> i, tiles = nrg * ((nct + per - 1) / per);
    const double t = (double)((tiles + cus - 1) / cus) * (whole[i] + (double)nb * block[cost][i]);
    if (i == 0 || t < *us) *us = t, best = {1 << i, tiles, std::min(cus, tiles)};
  }
  return best;
}

template <int TYPE, int RS>
void launch_prefill_h(const PfShape& s, const uint8_t* W, int64_t row_bytes, int nrows, int k, const uint8_t* xh, int n,
                      void* y, int y_dtype, float* part, uint32_t* cnt, hipStream_t stream) {
  const int64_t nb = k / kQK, tiles = s.tiles;
  const bool split = part != nullptr;  // else runs of whole tiles
  PfPlan p;
  p.ub = split ? 1 : (int)nb;
  p.nrg = (nrows + 127) / 128;
  p.few = tiles < s.wgs;
  const int64_t units = split ? tiles * nb : tiles;
  const int64_t wgs = split ? s.wgs : std::min<int64_t>(device_cus(), tiles);
  p.per = units / wgs;
  p.rem = units % wgs;
  gemm_prefill_h_kernel<TYPE, RS><<<dim3((unsigned)wgs), kPfThreads, 0, stream>>>(
      W, row_bytes, nrows, k, xh, (int)xq_col_tiles(n), n, y, y_dtype, p, part, cnt);
}

template <int TYPE>
void launch_prefill_t(const PfShape& s, const uint8_t* W, int64_t row_bytes, int nrows, int k, const uint8_t* xh, int n,
                      void* y, int y_dtype, float* part, uint32_t* cnt, hipStream_t stream) {
  switch (s.rs) {
    case 1: launch_prefill_h<TYPE, 1>(s, W, row_bytes, nrows, k, xh, n, y, y_dtype, part, cnt, stream); break;
    case 2: launch_prefill_h<TYPE, 2>(s, W, row_bytes, nrows, k, xh, n, y, y_dtype, part, cnt, stream); break;
    default: launch_prefill_h<TYPE, 4>(s, W, row_bytes, nrows, k, xh, n, y, y_dtype, part, cnt, stream); break;
  }
}

}  // namespace

// Whether the prefill GEMM serves the type: packed IQ3, and GGUF rows of every other type with a
// product op but IQ3 and IQ1_M.
bool prefill_supported(int type, bool packed) {
  if (packed) return type == kIQ3_S || type == kIQ3_XXS;
  return type == kQ4_K || type == kQ6_K || type == kIQ4_XS || type == kQ2_K || type == kIQ2_XXS || type == kIQ2_XS ||
         type == kIQ2_S;
}

// Tile counters of the split plan, and the bytes of its partial sums (a slot per workgroup and
// split tile; 0: the runs are whole tiles and nothing is split).
int64_t prefill_counters(int64_t nrows, int64_t k, int64_t n) { return pf_shape(nrows, k, n).tiles; }
size_t prefill_slot_bytes(int64_t nrows, int64_t k, int64_t n) {
  const int64_t nb = k / kQK;
  const PfShape s = pf_shape(nrows, k, n);
  if (s.tiles * nb % s.wgs == 0 && s.tiles * nb / s.wgs % nb == 0) return 0;
  return (size_t)(s.wgs + std::min(s.wgs, s.tiles)) * (16 / s.rs) * 2 * 4096;
}

// Estimated time of a product with K split over the CUs, us: pf_shape's, less on the shortest K
// (fewer parts or none), more where Q6_K's operands take two planes.
double prefill_split_us(int type, bool exact, int64_t nrows, int64_t k, int64_t n) {
  double us = 0;
  (void)pf_shape(nrows, k, n, &us);
  return us - (k <= 512 ? 7 : k <= 1024 ? 2.5 : 0) + (type == kQ6_K && exact ? 2.5 : 0);
}
// Estimated time of a product in whole tiles, us (512 x 512 M = 257 14, 1024 x 1024 18.6).
double prefill_whole_us(int type, bool exact, int64_t nrows, int64_t k, int64_t n) {
  double us = 0;
  (void)pf_whole_shape(type, exact, nrows, k, n, &us);
  return us + (k <= 1024 ? 2 : 0);
}

// Large-M products; xh: X in the xh layout of the type. split: K over the CUs, with prefill_slot_bytes of
// workspace at part and prefill_counters counters that the quantise launch cleared at cnt (both null where
// the split needs no slots); else whole tiles. exact: Q6_K's operands without the rounding beyond 2048 (two
// MFMAs per slice).
hipError_t launch_gemm_prefill(int type, bool exact, bool split, const uint8_t* W, int64_t row_bytes, int nrows, int k,
                               const uint8_t* xh, int n, void* y, int y_dtype, float* part, uint32_t* cnt,
                               hipStream_t stream) {
  double us = 0;
  const PfShape s = split ? pf_shape(nrows, k, n) : pf_whole_shape(type, exact, nrows, k, n, &us);
#define GGUF_PF(T) \
  case T: launch_prefill_t<T>(s, W, row_bytes, nrows, k, xh, n, y, y_dtype, part, cnt, stream); break;
  switch (type == kQ6_K && exact ? kQ6_KX : type) {
    GGUF_PF(kQ6_KX)
    GGUF_PF(kIQ3_S)
    GGUF_PF(kIQ3_XXS)
    GGUF_PF(kQ4_K)
    GGUF_PF(kQ6_K)
    GGUF_PF(kIQ4_XS)
    GGUF_PF(kQ2_K)
    GGUF_PF(kIQ2_XXS)
    GGUF_PF(kIQ2_XS)
    GGUF_PF(kIQ2_S)
    default: return hipErrorInvalidValue;
  }
#undef GGUF_PF
  return hipGetLastError();
}

}  // namespace gguf

// The build's q8 activation layout for the int8-MFMA GEMMs ("xq"), an internal workspace format
// (the reference's block_q8_1_mmq, mmq.cuh:27-56, serves its CUDA mma fragments; the values and
// scales here are the same, only their placement differs).
//
// Activation rows are grouped in column tiles of 16 (the B-operand width of
// v_mfma_i32_16x16x32_i8); rows past n in the last tile are zero. For column tile t and 256-value
// K block b (nb = K / 256 blocks):
//   values  4096 B at ((t * nb + b) * 4096): lane l = 16q + j of a wave owns, for the block's
//           slices u = 0..7, the eight q8 values 32u + 8q .. 32u + 8q + 7 of activation row
//           16t + j, 8 bytes at 1024 (u >> 1) + 16l + 8 (u & 1). One wave reads a (t, b) unit with
//           four 16-byte loads per lane, each a contiguous KB, and those bytes are the MFMA B
//           operands of the 8 slices. (With a lane's 64 bytes contiguous, each load went out as 64
//           L1 accesses instead of 16.)
//   scales  512 B at nct * nb * 4096 + (t * nb + b) * 512: one dword per slice u = 0..7 of activation
//           row 16t + j at 256 (u >> 2) + 16j + 4 (u & 3): fp32 d, or for Q4_K weights fp16 d in the
//           low half and, above it, the activation side of Q4_K's min term: with the decode ops' q8_1
//           arithmetic the slice's int16 sum of q (times d: the MMVQ form, |sum| <= 4064, exact
//           in fp32), with the MMQ arithmetic the fp16 of the slice's sum of x (the half2 sum of
//           block_q8_1_mmq's DS4 layout, the MMQ form, vecdotq.cuh:549-552).
// Quantisation per 32-value slice is the reference's MMQ arithmetic (lcpp_shim.cu:298-355):
// d_inv = 127 / amax, q = roundf(x * d_inv), d = 1 / d_inv, and q = 0, d = 0 for an all-zero
// slice; for Q4_K d is stored as fp16 as in the reference's half2 (DS4) MMQ layout.
#pragma once

#include "gguf_common.h"

namespace gguf {

constexpr int kXqCols = 16;         // activation rows per column tile
constexpr int kXqUnit = 4096;       // value bytes per (column tile, K block)
constexpr int kXqScaleUnit = 512;   // scale bytes per (column tile, K block)

__host__ __device__ inline int64_t xq_col_tiles(int64_t n) { return (n + kXqCols - 1) / kXqCols; }

// byte offsets inside a unit: the value bytes of slice u of lane l, and (for the scales) row j's word
__host__ __device__ constexpr int xq_value_off(int l, int u) { return 1024 * (u >> 1) + 16 * l + 8 * (u & 1); }
__host__ __device__ constexpr int xq_scale_off(int j, int u) { return 256 * (u >> 2) + 16 * j + 4 * (u & 3); }

__host__ __device__ inline int64_t xq_scale_base(int64_t nct, int64_t nb) { return nct * nb * kXqUnit; }

__host__ __device__ inline size_t xq_bytes(int64_t n, int64_t k) {
  const int64_t nct = xq_col_tiles(n), nb = k / kQK;
  return (size_t)(nct * nb * (kXqUnit + kXqScaleUnit));
}

// The prefill GEMM's fp16 variant of the layout ("xh"): the same q8 values held as fp16 (exact),
// the same column tiles and K blocks. For column tile t and block b:
//   values  8192 B at ((t * nb + b) * 8192): slice u at 1024u, lane l = 16q + j of a wave owns 16
//           bytes at 1024u + 16l: the fp16 values 32u + 8q .. 32u + 8q + 7 of activation row
//           16t + j (the f16 MFMA B operand of the slice). Slices 4h..4h+3 are 4 KB contiguous.
//   scales  1024 B at nct * nb * 8192 + (t * nb + b) * 1024: fp32 d of (row j, slice u) at 32j + 4u
//           (a lane reads the 4 scales of its half block with one 16-byte load). The activation side
//           of the min terms follows, in bf16 pieces that add up to it exactly (the B operand of a
//           bf16 MFMA whose A operand holds the integer mins):
//           Q4_K: d is the fp16-rounded scale; at 512 + 32j + 4u the two bf16 pieces (the first in the
//           low half) of the fp16 sum of the slice's x (DS4's half2 sum).
//           Q2_K (2560 B): d is the fp16-rounded scale of 64 values; for half block h at 512 + 1024h +
//           64j, + 16 and + 32: eight bf16 (16-value groups 0..7 of the half) of the first, second
//           and third pieces of, for groups 0..5, the fp16 sum of the group's x, and for groups 6
//           and 7 d x the sum of q (D2S6), with a sum that is not finite in the third place beside
//           +-1, 0 (the mins' second pieces, often 0, meet the first two places only: 0 x inf would
//           make a NaN of an inf); at + 48 the eight sums of q, as fp16 (exact).
constexpr int kXhUnit = 8192;       // fp16 value bytes per (column tile, K block)

// scale bytes per (column tile, K block)
__host__ __device__ constexpr int xh_scale_unit(int type) { return type == kQ2_K ? 2560 : 1024; }

__host__ __device__ inline int64_t xh_scale_base(int64_t nct, int64_t nb) { return nct * nb * kXhUnit; }

__host__ __device__ inline size_t xh_bytes(int64_t n, int64_t k, int type) {
  const int64_t nct = xq_col_tiles(n), nb = k / kQK;
  return (size_t)(nct * nb * (kXhUnit + xh_scale_unit(type)));
}

// MFMA B operand of slice 2i + h from the 16 bytes b[t][i] of a lane's xq unit
__device__ __forceinline__ long xq_b_operand(const u32x4& v, int h) {
  return h == 0 ? (long)(((uint64_t)v[1] << 32) | v[0]) : (long)(((uint64_t)v[3] << 32) | v[2]);
}

}  // namespace gguf

// fp16 decode of weight blocks for the prefill GEMM (gemm_prefill.hip), cut into four parts that the
// kernel spreads over the four slices of a step, so that a part's LDS table reads return under the
// MFMAs of the step instead of being waited for.
//
// A step decodes half a K block (4 slices of 32 values) of 16-row tiles; a lane (row j, index q = 0..3)
// of the wave that owns a tile decodes 32 values of one row: slice 4h + q, part i = values 8i ..
// 8i + 7 of it (Q6_K: values 8q .. 8q + 7 of every slice, part i = slice 4h + i). Lanes are numbered
// so that neighbours read neighbouring bytes (pf_lane): the loads of a tile's rows by lane = 16 q + j
// went out as nearly one L1 access per lane, 2400 of the 3560 a step of a workgroup made.
// The operand is the weight value times its sub-scale, an integer that fp16 holds exactly (IQ3_S
// <= 465, IQ3_XXS <= 1922, IQ2 <= 1333, Q4_K <= 945; Q6_K's (q - 32) * sc is exact up to 2048 and rounds to
// an even neighbour beyond, 2^-12, unless kQ6_KX keeps the rest), except IQ4_XS: codebook value x sub-scale
// reaches 4064, so its operand is the codebook value and the sub-scale multiplies the slice's dot; and
// Q2_K, see there.
// The row's block scale (d; d / 8 for the IQ2 types, d / 4 for IQ3_XXS) stays outside, see next_scale.
#pragma once

#include "xh_decode.h"

namespace gguf {

namespace {

// Row scales and the min operands a step's decoders leave in LDS for the multipliers.
struct PfLds {
  uint8_t* A;      // decoded operands of the step's half
  float* RT;       // [128] e_prev / e_cur, at block starts
  float* EF;       // [128] e_cur
  uint16_t* AM;    // the mins, bf16: Q2_K the half's in planes of [tile][row][8], Q4_K the block's in
                   // [tile][row][16]
  float* RM;       // Q4_K: [128] -dmin / e of the block
  float* LS;       // IQ4_XS: the half's sub-scales, [tile][slice][16 rows]
  const uint8_t* tbl;
};

// A slot of (row tile t, slice u of the half block, row j, quarter q): 16 bytes at 16 (16q + (j ^ 4u)) of
// the slice's KB. The operand read of MFMA lane 16q + j is a permutation of the KB's slots within each
// 256 bytes, free of bank conflicts (rows of 64 bytes with swizzled quarters had 4 conflict cycles in
// each ds_read_b128); the 4u keeps the stores of neighbouring decode lanes, which hold the 4 slices of
// a row, on different banks.
constexpr int kPfRegion = 1024;
__device__ __forceinline__ int pf_off(int t, int u, int j, int q) {
  return (t * 4 + u) * kPfRegion + (q * 16 + (j ^ (4 * u))) * 16;
}

constexpr int kPfPlane = 8 * 4 * kPfRegion;  // operands of half a K block of 128 rows: 32 KB

// Q6_K with its products kept exact, in two planes of operands
constexpr int kQ6_KX = 1000 + kQ6_K;

constexpr bool pf_iq3(int type) { return type == kIQ3_S || type == kIQ3_XXS; }
constexpr bool pf_min(int type) { return type == kQ4_K || type == kQ2_K; }

// bf16 bits of a small integer (exact up to 256)
__device__ __forceinline__ uint32_t small_bf16(uint32_t v) { return __float_as_uint((float)v) >> 16; }

// 4 unsigned bytes -> two dwords of fp16 (byte * mul + off): 1024 + byte by a byte permute, then one
// packed FMA. off = -1024 mul (or -(1024 + bias) mul for biased bytes), exact in fp16.
__device__ __forceinline__ void bytes_to_h4(uint32_t x, h2 mul, h2 off, uint32_t& a, uint32_t& b) {
  a = h2_bits(__builtin_elementwise_fma(bits_h2(__builtin_amdgcn_perm(0x64646464u, x, 0x04010400u)), mul, off));
  b = h2_bits(__builtin_elementwise_fma(bits_h2(__builtin_amdgcn_perm(0x64646464u, x, 0x04030402u)), mul, off));
}

// fp16 sign bits of values 2p, 2p + 1 from sign byte s, with x = s | s << 15
__device__ __forceinline__ uint32_t sign_pair(uint32_t x, int p) { return (x << (15 - 2 * p)) & 0x80008000u; }

__device__ __forceinline__ h2 h2_of(float v) {
  const _Float16 f = (_Float16)v;
  return h2{f, f};
}

// The biased signed tables (every byte + 128): IQ3_S index qs | ex << 8 (iq3_tile.h), IQ3_XXS index
// grid index | sign nibble << 8
constexpr Iq3sSignedTable make_pf_iq3s_table() {
  Iq3sSignedTable t = make_iq3s_signed_table();
  for (int i = 0; i < 8192; ++i) t.v[i] ^= 0x80808080u;
  return t;
}
__device__ const Iq3sSignedTable kPfIq3s = make_pf_iq3s_table();

struct PfXxsTable {
  uint32_t v[4096];
};
constexpr PfXxsTable make_pf_xxs_table() {
  PfXxsTable t{};
  for (int i = 0; i < 4096; ++i) {
    const uint32_t g = kIq3xxsGrid.v[i & 255], sg = (uint32_t)i >> 8;
    uint32_t out = 0;
    for (int b = 0; b < 4; ++b) {
      const uint32_t byte = (g >> (8 * b)) & 0xFF;
      out |= (((sg >> b) & 1 ? 256u - byte : byte) & 0xFF) << (8 * b);
    }
    t.v[i] = out ^ 0x80808080u;
  }
  return t;
}
__device__ const PfXxsTable kPfXxs = make_pf_xxs_table();
__device__ const Lattice64<256> kPfIq2xxs = kIq2xxsGrid;
__device__ const Lattice64<512> kPfIq2xs = kIq2xsGrid;
__device__ const Lattice64<1024> kPfIq2s = kIq2sGrid;

// bytes of a type's decode table in LDS
constexpr int pf_table_bytes(int type) {
  return type == kIQ3_S ? 32768 : type == kIQ3_XXS ? 16384 : type == kIQ2_XXS ? 2048 : type == kIQ2_XS ? 4096
         : type == kIQ2_S ? 8192 : 0;
}
template <int TYPE>
__device__ __forceinline__ const uint4* pf_table() {
  if constexpr (TYPE == kIQ3_S) return (const uint4*)kPfIq3s.v;
  else if constexpr (TYPE == kIQ3_XXS) return (const uint4*)kPfXxs.v;
  else if constexpr (TYPE == kIQ2_XXS) return (const uint4*)kPfIq2xxs.v;
  else if constexpr (TYPE == kIQ2_XS) return (const uint4*)kPfIq2xs.v;
  else if constexpr (TYPE == kIQ2_S) return (const uint4*)kPfIq2s.v;
  else return nullptr;
}

// PfDec<TYPE>: Raw (a lane's bytes of one step, loaded a step ahead), load(), begin() (the step's
// scales; writes RT / EF / AM / RM / LS), issue<I>() (part I's table reads) and finish<I>() (its 8
// values into A). wp: the row's first byte (the IQ3 unit layouts: the 16-row tile's).
template <int TYPE>
struct PfDec;

template <>
struct PfDec<kIQ3_S> {
  using Raw = RawIq3;
  struct Ctx {
    h2 mul, off;
    uint32_t P[4];  // two 13-bit table indices each
  };
  struct Tmp {
    int g[2];
  };
  __device__ __forceinline__ static void load(Raw& r, const uint8_t* wp, int64_t row_bytes, int nb, int b, int h, int j,
                                              int q) {
    load_step(r, wp, row_bytes, nb, b, h, j, q);
  }
  __device__ __forceinline__ static void begin(const Raw& w, Ctx& c, int h, float& e, const PfLds& s, int t, int j,
                                               int q) {
    const float d = half_bits_to_float(w.d);
    if (h == 0) next_scale(d, e, s.RT, s.EF, t * 16 + j);
    const uint32_t nib = (w.sc >> (4 * (q & 1))) & 0xF;  // slice 4h + q
    c.mul = h2_of(d != 0.0f ? (float)(1 + 2 * nib) : 0.0f);
    c.off = c.mul * (_Float16)(-1152.0f);
    uint32_t lo, hi;
    iq3_tile_ex(w.e8, w.l2, j & 1, lo, hi);
    c.P[0] = __builtin_amdgcn_perm(lo, w.qs.x, 0x05010400u);
    c.P[1] = __builtin_amdgcn_perm(lo, w.qs.x, 0x07030602u);
    c.P[2] = __builtin_amdgcn_perm(hi, w.qs.y, 0x05010400u);
    c.P[3] = __builtin_amdgcn_perm(hi, w.qs.y, 0x07030602u);
  }
  template <int I>
  __device__ __forceinline__ static void issue(const Ctx& c, Tmp& x, const PfLds& s) {
    tile_lookup2(s.tbl, c.P[I], x.g[0], x.g[1]);
  }
  template <int I>
  __device__ __forceinline__ static void finish(const Ctx& c, const Tmp& x, const PfLds& s, int t, int j, int q) {
    uint32_t v[4];
    bytes_to_h4((uint32_t)x.g[0], c.mul, c.off, v[0], v[1]);
    bytes_to_h4((uint32_t)x.g[1], c.mul, c.off, v[2], v[3]);
    *(uint4*)(s.A + pf_off(t, q, j, I)) = make_uint4(v[0], v[1], v[2], v[3]);
  }
};

// IQ3_XXS: value = (d / 4) * ls * w (ls = 2 * scale + 1). The second word of each 8-value group takes
// bits 4..6 of the group's 7-bit sign index and their parity with bits 0..3 (ksigns_iq2xs), all four
// parities from two three-way xors (bit 7g of t ^ t >> 3 ^ a >> 6, t = a ^ a >> 1 ^ a >> 2, is the
// xor of bits 7g .. 7g + 6).
template <>
struct PfDec<kIQ3_XXS> {
  using Raw = RawXxsH;
  struct Ctx {
    h2 mul, off;
    uint32_t a, hi;
    uint2 qs;
  };
  struct Tmp {
    uint32_t g[2];
  };
  __device__ __forceinline__ static void load(Raw& r, const uint8_t* wp, int64_t row_bytes, int nb, int b, int h, int j,
                                              int q) {
    load_step(r, wp, row_bytes, nb, b, h, j, q);
  }
  __device__ __forceinline__ static void begin(const Raw& w, Ctx& c, int h, float& e, const PfLds& s, int t, int j,
                                               int q) {
    const float d = half_bits_to_float(w.d) * 0.25f;
    if (h == 0) next_scale(d, e, s.RT, s.EF, t * 16 + j);
    const uint32_t a = w.aux, t3 = a ^ (a >> 1) ^ (a >> 2), par = t3 ^ (t3 >> 3) ^ (a >> 6);
    c.a = a;
    c.hi = ((par << 3) & 0x01020408u) | ((a >> 4) & ~0x01020408u);
    c.qs = w.qs;
    c.mul = h2_of(d != 0.0f ? (float)(2 * (a >> 28) + 1) : 0.0f);
    c.off = c.mul * (_Float16)(-1152.0f);
  }
  template <int I>
  __device__ __forceinline__ static void issue(const Ctx& c, Tmp& x, const PfLds& s) {
    const uint32_t qw = (I < 2 ? c.qs.x : c.qs.y) >> (16 * (I & 1));
    const uint32_t* tbl = (const uint32_t*)s.tbl;
    x.g[0] = tbl[(qw & 0xFF) | (((c.a >> (7 * I)) & 0xF) << 8)];
    x.g[1] = tbl[((qw >> 8) & 0xFF) | (((c.hi >> (7 * I)) & 0xF) << 8)];
  }
  template <int I>
  __device__ __forceinline__ static void finish(const Ctx& c, const Tmp& x, const PfLds& s, int t, int j, int q) {
    uint32_t v[4];
    bytes_to_h4(x.g[0], c.mul, c.off, v[0], v[1]);
    bytes_to_h4(x.g[1], c.mul, c.off, v[2], v[3]);
    *(uint4*)(s.A + pf_off(t, q, j, I)) = make_uint4(v[0], v[1], v[2], v[3]);
  }
};

// The IQ2 types: 8-value groups of unsigned grid bytes (8, 25 or 43), 8 sign bits each
struct PfIq2Ctx {
  h2 mul[2], off[2];  // values 0..15 and 16..31 of the slice
  uint32_t idx[4];    // grid index of each group
  uint32_t sg[4];     // sign byte of each group (s | s << 15)
};
struct PfIq2Tmp {
  uint2 g;
};
__device__ __forceinline__ void pf_iq2_scales(PfIq2Ctx& c, bool nz, uint32_t n0, uint32_t n1) {
  c.mul[0] = h2_of(nz ? (float)(2 * n0 + 1) : 0.0f);
  c.mul[1] = h2_of(nz ? (float)(2 * n1 + 1) : 0.0f);
  c.off[0] = c.mul[0] * (_Float16)(-1024.0f);
  c.off[1] = c.mul[1] * (_Float16)(-1024.0f);
}
template <int I>
__device__ __forceinline__ void pf_iq2_finish(const PfIq2Ctx& c, const PfIq2Tmp& x, const PfLds& s, int t, int j, int q) {
  uint32_t v[4];
  bytes_to_h4(x.g.x, c.mul[I >> 1], c.off[I >> 1], v[0], v[1]);
  bytes_to_h4(x.g.y, c.mul[I >> 1], c.off[I >> 1], v[2], v[3]);
#pragma unroll
  for (int p = 0; p < 4; ++p) v[p] ^= sign_pair(c.sg[I], p);
  *(uint4*)(s.A + pf_off(t, q, j, I)) = make_uint4(v[0], v[1], v[2], v[3]);
}

template <>
struct PfDec<kIQ2_XXS> {
  struct Raw {
    uint32_t idx, aux;
    uint16_t d;
  };
  using Ctx = PfIq2Ctx;
  using Tmp = PfIq2Tmp;
  __device__ __forceinline__ static void load(Raw& r, const uint8_t* wp, int64_t, int, int b, int h, int j, int q) {
    const uint8_t* blk = wp + (int64_t)b * 66;
    const uint64_t v = ld64(blk + 2 + 8 * (4 * h + q));
    r.idx = (uint32_t)v;
    r.aux = (uint32_t)(v >> 32);
    r.d = (uint16_t)ld16(blk);
  }
  __device__ __forceinline__ static void begin(const Raw& w, Ctx& c, int h, float& e, const PfLds& s, int t, int j,
                                               int q) {
    const float d = half_bits_to_float(w.d) * 0.125f;
    if (h == 0) next_scale(d, e, s.RT, s.EF, t * 16 + j);
    pf_iq2_scales(c, d != 0.0f, w.aux >> 28, w.aux >> 28);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const uint32_t sg = ksigns8((w.aux >> (7 * g)) & 127);
      c.sg[g] = sg | (sg << 15);
      c.idx[g] = (w.idx >> (8 * g)) & 0xFF;
    }
  }
  template <int I>
  __device__ __forceinline__ static void issue(const Ctx& c, Tmp& x, const PfLds& s) {
    x.g = ((const uint2*)s.tbl)[c.idx[I]];
  }
  template <int I>
  __device__ __forceinline__ static void finish(const Ctx& c, const Tmp& x, const PfLds& s, int t, int j, int q) {
    pf_iq2_finish<I>(c, x, s, t, j, q);
  }
};

template <>
struct PfDec<kIQ2_XS> {
  struct Raw {
    uint32_t v0, v1;  // four 16-bit codes: 9-bit grid index, 7-bit sign index
    uint8_t sc;
    uint16_t d;
  };
  using Ctx = PfIq2Ctx;
  using Tmp = PfIq2Tmp;
  __device__ __forceinline__ static void load(Raw& r, const uint8_t* wp, int64_t, int, int b, int h, int j, int q) {
    const uint8_t* blk = wp + (int64_t)b * 74;
    const uint64_t v = ld64(blk + 2 + 8 * (4 * h + q));
    r.v0 = (uint32_t)v;
    r.v1 = (uint32_t)(v >> 32);
    r.sc = blk[66 + 4 * h + q];
    r.d = (uint16_t)ld16(blk);
  }
  __device__ __forceinline__ static void begin(const Raw& w, Ctx& c, int h, float& e, const PfLds& s, int t, int j,
                                               int q) {
    const float d = half_bits_to_float(w.d) * 0.125f;
    if (h == 0) next_scale(d, e, s.RT, s.EF, t * 16 + j);
    pf_iq2_scales(c, d != 0.0f, w.sc & 0xF, w.sc >> 4);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const uint32_t v = (g < 2 ? w.v0 : w.v1) >> (16 * (g & 1));
      const uint32_t sg = ksigns8((v >> 9) & 127);
      c.sg[g] = sg | (sg << 15);
      c.idx[g] = v & 511;
    }
  }
  template <int I>
  __device__ __forceinline__ static void issue(const Ctx& c, Tmp& x, const PfLds& s) {
    x.g = ((const uint2*)s.tbl)[c.idx[I]];
  }
  template <int I>
  __device__ __forceinline__ static void finish(const Ctx& c, const Tmp& x, const PfLds& s, int t, int j, int q) {
    pf_iq2_finish<I>(c, x, s, t, j, q);
  }
};

template <>
struct PfDec<kIQ2_S> {
  struct Raw {
    uint32_t idx, sg;
    uint8_t qh, sc;
    uint16_t d;
  };
  using Ctx = PfIq2Ctx;
  using Tmp = PfIq2Tmp;
  __device__ __forceinline__ static void load(Raw& r, const uint8_t* wp, int64_t, int, int b, int h, int j, int q) {
    const uint8_t* blk = wp + (int64_t)b * 82;
    const int s = 4 * h + q;
    r.idx = ld32(blk + 2 + 4 * s);
    r.sg = ld32(blk + 34 + 4 * s);
    r.qh = blk[66 + s];
    r.sc = blk[74 + s];
    r.d = (uint16_t)ld16(blk);
  }
  __device__ __forceinline__ static void begin(const Raw& w, Ctx& c, int h, float& e, const PfLds& s, int t, int j,
                                               int q) {
    const float d = half_bits_to_float(w.d) * 0.125f;
    if (h == 0) next_scale(d, e, s.RT, s.EF, t * 16 + j);
    pf_iq2_scales(c, d != 0.0f, w.sc & 0xF, w.sc >> 4);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const uint32_t sg = (w.sg >> (8 * g)) & 0xFF;
      c.sg[g] = sg | (sg << 15);
      c.idx[g] = ((w.idx >> (8 * g)) & 0xFF) | (((uint32_t)w.qh << (8 - 2 * g)) & 0x300);
    }
  }
  template <int I>
  __device__ __forceinline__ static void issue(const Ctx& c, Tmp& x, const PfLds& s) {
    x.g = ((const uint2*)s.tbl)[c.idx[I]];
  }
  template <int I>
  __device__ __forceinline__ static void finish(const Ctx& c, const Tmp& x, const PfLds& s, int t, int j, int q) {
    pf_iq2_finish<I>(c, x, s, t, j, q);
  }
};

// Q4_K: nibble x sc. The block's 8 mins go out with half 0 (AM: each twice, for the two pieces of its
// slice's sum), as does RM.
template <>
struct PfDec<kQ4_K> {
  struct Raw {
    u32x4 hdr, v0, v1;  // d, dmin, scales[12]; the slice's 32 quant bytes (shared by slices 2i, 2i + 1)
  };
  struct Ctx {
    h2 mul, off;
    u32x4 v0, v1;  // the slice's nibbles
  };
  struct Tmp {};
  __device__ __forceinline__ static void load(Raw& r, const uint8_t* wp, int64_t, int, int b, int h, int j, int q) {
    const uint8_t* blk = wp + (int64_t)b * 144;
    r.hdr = *(const u32x4*)blk;
    r.v0 = *(const u32x4*)(blk + 16 + 64 * h + 32 * (q >> 1));
    r.v1 = *(const u32x4*)(blk + 32 + 64 * h + 32 * (q >> 1));
  }
  __device__ __forceinline__ static void begin(const Raw& w, Ctx& c, int h, float& e, const PfLds& s, int t, int j,
                                               int q) {
    const float d = half_bits_to_float(w.hdr[0] & 0xFFFF);
    const int row = t * 16 + j;
    const bool nz = d != 0.0f;
    // scales of slices 4h .. 4h + 3 (bytes); mins of all 8 slices, 4 per dword
    const uint32_t s0 = w.hdr[1], m0 = w.hdr[2], x = w.hdr[3];
    uint32_t sc;
    if (h == 0) {
      next_scale(d, e, s.RT, s.EF, row);
      s.RM[row] = -half_bits_to_float(w.hdr[0] >> 16) / e;
      sc = s0 & 0x3F3F3F3Fu;
      const uint32_t mlo = m0 & 0x3F3F3F3Fu, mhi = ((x >> 4) & 0x0F0F0F0Fu) | ((m0 >> 2) & 0x30303030u);
      const uint32_t mm = (q < 2 ? mlo : mhi) >> (16 * (q & 1));  // this lane: slices 2q, 2q + 1
      *(uint2*)(s.AM + row * 16 + 4 * q) = make_uint2(small_bf16(mm & 0xFF) * 0x10001u, small_bf16((mm >> 8) & 0xFF) * 0x10001u);
    } else {
      sc = (x & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u);
    }
    c.mul = h2_of(nz ? (float)((sc >> (8 * q)) & 0xFF) : 0.0f);
    c.off = c.mul * (_Float16)(-1024.0f);
    const int sh = 4 * (q & 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      c.v0[i] = (w.v0[i] >> sh) & 0x0F0F0F0Fu;
      c.v1[i] = (w.v1[i] >> sh) & 0x0F0F0F0Fu;
    }
  }
  template <int I>
  __device__ __forceinline__ static void issue(const Ctx&, Tmp&, const PfLds&) {}
  template <int I>
  __device__ __forceinline__ static void finish(const Ctx& c, const Tmp&, const PfLds& s, int t, int j, int q) {
    const u32x4 vv = I < 2 ? c.v0 : c.v1;
    uint32_t v[4];
    bytes_to_h4(vv[2 * (I & 1)], c.mul, c.off, v[0], v[1]);
    bytes_to_h4(vv[2 * (I & 1) + 1], c.mul, c.off, v[2], v[3]);
    *(uint4*)(s.A + pf_off(t, q, j, I)) = make_uint4(v[0], v[1], v[2], v[3]);
  }
};

// 1 / v of a power of two
__device__ __forceinline__ float pow2_inv(float v) { return __uint_as_float(0x7F000000u - __float_as_uint(v)); }

// Q2_K: 2-bit quant x f, the fp16 of d * sc, per 16 values, as the reference's MMQ tile loader rounds it
// (mmq-load-tiles.cuh:582-591). 3f may need two bits more than fp16 has, so the operand is f (q - 1), -f
// .. 2f, and the sum f x (sum of the group's q8) that it leaves out is an MFMA of its own per 64 values
// (f: AM + 3072 and AM + 4096, fp16, for groups 0..3 and 4..7 of the half, 0 for the others). Operands are
// in units of e, a power of two within 2^8 of d, so that f is exact there, and so are the mins: each half's
// 8 go out with the half, minus the fp16 of dmin * m (rounded there as well) in two bf16 pieces (AM, AM +
// 1024; the first again at AM + 2048, 0 where it is not finite). e moves only when a block's d leaves that range; the rows' accumulators are rescaled only then
// (RT, with a flag per row tile at RT + 128).
template <>
struct PfDec<kQ2_K> {
  struct Raw {
    u32x4 v0, v1;  // the half's 32 quant bytes (bits 2u: slice u)
    uint2 sc;      // the half's 8 scale bytes
    uint32_t dm;
  };
  struct Ctx {
    h2 mul[2];
    u32x4 v0, v1;
  };
  struct Tmp {};
  __device__ __forceinline__ static void load(Raw& r, const uint8_t* wp, int64_t, int, int b, int h, int j, int q) {
    const uint8_t* blk = wp + (int64_t)b * 84;  // 4-byte aligned: rows are
    r.v0 = ld128a4(blk + 16 + 32 * h);
    r.v1 = ld128a4(blk + 32 + 32 * h);
    const uint32_t* ps = (const uint32_t*)(blk + 8 * h);
    r.sc = make_uint2(ps[0], ps[1]);
    r.dm = *(const uint32_t*)(blk + 80);
  }
  __device__ __forceinline__ static void begin(const Raw& w, Ctx& c, int h, float& e, const PfLds& s, int t, int j,
                                               int q) {
    const float d = half_bits_to_float(w.dm & 0xFFFF);
    const int row = t * 16 + j;
    if (h == 0) {
      // the power of two of d, for an infinite one that of the largest fp16 (no short circuit: a branch
      // here made the step spill 140 registers)
      const uint32_t p = min(__float_as_uint(d) & 0x7F800000u, 0x47000000u);
      const bool move = (d != 0.0f) & (p - __float_as_uint(e) + (8u << 23) > (16u << 23));
      const float en = move ? __uint_as_float(p) : e;
      s.RT[row] = e * pow2_inv(en);
      s.EF[row] = en;
      s.RT[128 + t] = __any(en != e) ? 1.0f : 0.0f;
      e = en;
    }
    const float re = pow2_inv(e);
    const uint32_t mine = (q < 2 ? w.sc.x : w.sc.y) >> (16 * (q & 1));  // groups 2q, 2q + 1: slice q's
    const float dmin = half_bits_to_float(w.dm >> 16);
    uint32_t hi[2], lo[2], fin[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      c.mul[i] = h2_of(__half2float(__float2half_rn(d * (float)((mine >> (8 * i)) & 0xF))) * re);
      const float f = __half2float(__float2half_rn(dmin * (float)((mine >> (8 * i + 4)) & 0xF))) * -re;
      hi[i] = __float_as_uint(f) >> 16;  // the upper 8 bits of 11
      const float r = f - __uint_as_float(hi[i] << 16);
      lo[i] = __float_as_uint(r == r ? r : 0.0f) >> 16;
      fin[i] = r == r ? hi[i] : 0;
    }
    *(uint32_t*)(s.AM + row * 8 + 2 * q) = hi[0] | (hi[1] << 16);
    *(uint32_t*)(s.AM + 1024 + row * 8 + 2 * q) = lo[0] | (lo[1] << 16);
    *(uint32_t*)(s.AM + 2048 + row * 8 + 2 * q) = fin[0] | (fin[1] << 16);
    *(uint32_t*)(s.AM + 3072 + 1024 * (q >> 1) + row * 8 + 2 * q) = h2_bits(h2{c.mul[0][0], c.mul[1][0]});
    *(uint32_t*)(s.AM + 4096 - 1024 * (q >> 1) + row * 8 + 2 * q) = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      c.v0[i] = (w.v0[i] >> (2 * q)) & 0x03030303u;
      c.v1[i] = (w.v1[i] >> (2 * q)) & 0x03030303u;
    }
  }
  template <int I>
  __device__ __forceinline__ static void issue(const Ctx&, Tmp&, const PfLds&) {}
  template <int I>
  __device__ __forceinline__ static void finish(const Ctx& c, const Tmp&, const PfLds& s, int t, int j, int q) {
    const u32x4 vv = I < 2 ? c.v0 : c.v1;
    const h2 bias = {(_Float16)-1025.0f, (_Float16)-1025.0f};
    uint32_t v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[i] = h2_bits((bits_h2(__builtin_amdgcn_perm(0x64646464u, vv[2 * (I & 1) + (i >> 1)],
                                                    (i & 1) ? 0x04030402u : 0x04010400u)) + bias) * c.mul[I >> 1]);
    *(uint4*)(s.A + pf_off(t, q, j, I)) = make_uint4(v[0], v[1], v[2], v[3]);
  }
};

// Q6_K: q - 32 by one packed subtract, then times the 16-value sub-scale. LO: the rounding of the product
// (up to 1 where it passes 2048) goes into a second plane of operands at s.A + kPfPlane.
template <bool LO>
struct PfDecQ6k {
  using Raw = RawQ6k;
  struct Ctx {
    h2 mul[4];
    uint64_t la, lb, qh;
  };
  struct Tmp {};
  __device__ __forceinline__ static void load(Raw& r, const uint8_t* wp, int64_t, int, int b, int h, int j, int q) {
    load_step(r, wp + (int64_t)b * 210, h, q);
  }
  __device__ __forceinline__ static void begin(const Raw& w, Ctx& c, int h, float& e, const PfLds& s, int t, int j,
                                               int q) {
    const float d = half_bits_to_float(w.d);
    if (h == 0) next_scale(d, e, s.RT, s.EF, t * 16 + j);
    else e = d != 0.0f ? d : e;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int sc = (int)(int8_t)((w.sc >> (8 * (2 * u + (q >> 1)))) & 0xFF);
      c.mul[u] = h2_of(d != 0.0f ? (float)sc : 0.0f);
    }
    c.la = w.la;
    c.lb = w.lb;
    c.qh = w.qh;
  }
  template <int I>
  __device__ __forceinline__ static void issue(const Ctx&, Tmp&, const PfLds&) {}
  template <int I>
  __device__ __forceinline__ static void finish(const Ctx& c, const Tmp&, const PfLds& s, int t, int j, int q) {
    const uint64_t l = (I & 1) ? c.lb : c.la;
    constexpr int lsh = 4 * (I >> 1), hsh = 2 * I;
    const uint32_t x0 = (((uint32_t)l >> lsh) & 0x0F0F0F0Fu) | ((((uint32_t)c.qh >> hsh) & 0x03030303u) << 4);
    const uint32_t x1 =
        (((uint32_t)(l >> 32) >> lsh) & 0x0F0F0F0Fu) | ((((uint32_t)(c.qh >> 32) >> hsh) & 0x03030303u) << 4);
    const h2 bias = {(_Float16)-1056.0f, (_Float16)-1056.0f};
    uint32_t v[4], lo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const h2 x = bits_h2(__builtin_amdgcn_perm(0x64646464u, i < 2 ? x0 : x1, (i & 1) ? 0x04030402u : 0x04010400u)) + bias;
      const h2 p = x * c.mul[I];
      v[i] = h2_bits(p);
      if constexpr (LO) lo[i] = h2_bits(__builtin_elementwise_fma(x, c.mul[I], -p));
    }
    *(uint4*)(s.A + pf_off(t, I, j, q)) = make_uint4(v[0], v[1], v[2], v[3]);
    if constexpr (LO) *(uint4*)(s.A + kPfPlane + pf_off(t, I, j, q)) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
  }
};
template <>
struct PfDec<kQ6_K> : PfDecQ6k<false> {};
template <>
struct PfDec<kQ6_KX> : PfDecQ6k<true> {};

// IQ4_XS: the codebook value, exact; the sub-scales (-32 .. 31; 0 for a block of d = 0) go to LS. The
// slice's values 0..15 are the low nibbles of its 16 bytes, 16..31 the high ones.
template <>
struct PfDec<kIQ4_XS> {
  struct Raw {
    u32x4 v;    // the slice's 16 quant bytes (8-byte aligned)
    uint2 hdr;  // d, scales_h, scales_l
  };
  struct Ctx {
    u32x4 v;
  };
  struct Tmp {};
  __device__ __forceinline__ static void load(Raw& r, const uint8_t* wp, int64_t, int, int b, int h, int j, int q) {
    const uint8_t* blk = wp + (int64_t)b * 136;
    r.v = ld128a4(blk + 8 + 64 * h + 16 * q);
    r.hdr = *(const uint2*)blk;
  }
  __device__ __forceinline__ static void begin(const Raw& w, Ctx& c, int h, float& e, const PfLds& s, int t, int j,
                                               int q) {
    const float d = half_bits_to_float(w.hdr.x & 0xFFFF);
    if (h == 0) next_scale(d, e, s.RT, s.EF, t * 16 + j);
    const int u = 4 * h + q;
    const uint32_t ls = ((w.hdr.y >> (4 * u)) & 0xF) | (((w.hdr.x >> (16 + 2 * u)) & 3) << 4);
    s.LS[(t * 4 + q) * 16 + j] = d != 0.0f ? (float)((int)ls - 32) : 0.0f;
    c.v = w.v;
  }
  template <int I>
  __device__ __forceinline__ static void issue(const Ctx&, Tmp&, const PfLds&) {}
  template <int I>
  __device__ __forceinline__ static void finish(const Ctx& c, const Tmp&, const PfLds& s, int t, int j, int q) {
    const uint32_t x0 = (uint32_t)iq4nl(c.v[2 * (I & 1)], 4 * (I >> 1)) ^ 0x80808080u;
    const uint32_t x1 = (uint32_t)iq4nl(c.v[2 * (I & 1) + 1], 4 * (I >> 1)) ^ 0x80808080u;
    const h2 bias = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    uint32_t v[4];
    v[0] = h2_bits(bits_h2(__builtin_amdgcn_perm(0x64646464u, x0, 0x04010400u)) + bias);
    v[1] = h2_bits(bits_h2(__builtin_amdgcn_perm(0x64646464u, x0, 0x04030402u)) + bias);
    v[2] = h2_bits(bits_h2(__builtin_amdgcn_perm(0x64646464u, x1, 0x04010400u)) + bias);
    v[3] = h2_bits(bits_h2(__builtin_amdgcn_perm(0x64646464u, x1, 0x04030402u)) + bias);
    *(uint4*)(s.A + pf_off(t, q, j, I)) = make_uint4(v[0], v[1], v[2], v[3]);
  }
};

}  // namespace

}  // namespace gguf

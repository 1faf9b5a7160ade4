// Device helpers shared by the split-K kernels (attn_decode.hip, attn_block.hip): tile shapes, exchanges between the four 16-lane rows of a wavefront, int8 rows.
#pragma once
#include "pa_internal.h"
#include "glue_math.h"

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __fp16 hh4 __attribute__((__vector_size__(4 * sizeof(__fp16))));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));

#define TILE 32

#define NEG_INF (-__builtin_inff())
#define DEC_RESCALE_TH 8.f   // tile loop: a row maximum may pass the reference maximum by this much before O is rescaled

static __device__ inline h4 lds_read_tr16(const unsigned char* p) {
  hh4 t = __builtin_amdgcn_ds_read_tr16_b64_v4f16((hh4 __attribute__((address_space(3)))*)p);
  h4 r; __builtin_memcpy(&r, &t, 8); return r;
}

typedef _Float16 h2 __attribute__((ext_vector_type(2)));

// Exchanges between the four 16-lane rows of a wavefront on the VALU (gfx950 lane-swap instructions) instead of the LDS
// crossbar (ds_bpermute: a dependent round trip of ~100 clocks each, four of them on the critical path of every tile's
// softmax).  xrow16(v): lane i's own value and the value of lane i ^ 16; xrow32(v): the same for i ^ 32.  Both partners see
// the same pair, so a commutative combine gives both the same bits.
static __device__ inline void xrow16(float v, float& a, float& b) {
  const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  a = __uint_as_float(sw[0]); b = __uint_as_float(sw[1]);
}
static __device__ inline void xrow32(float v, float& a, float& b) {
  const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  a = __uint_as_float(sw[0]); b = __uint_as_float(sw[1]);
}
// maximum / sum over the four lanes {i, i ^ 16, i ^ 32, i ^ 48} (the four position groups of a query row), the same bits in all four
static __device__ inline float rows_max(float v) {
  float a, b;
  xrow16(v, a, b); v = fmaxf(a, b);
  xrow32(v, a, b); return fmaxf(a, b);
}
static __device__ inline float rows_sum(float v) {
  float a, b;
  xrow16(v, a, b); v = a + b;
  xrow32(v, a, b); return a + b;
}
// acc + the sum of eight f16 probabilities, as the numbers the PV product really uses (v_dot2_f32_f16 with ones: products
// exact, sums in f32): the row total l is then the total of the weights that were applied, so a row's output is a convex
// combination of value rows whatever the rounding of P did -- one visible row gives that row's bits back, constant
// values give the constant
static __device__ inline float sum_f16(const h8 pf, float acc) {
  const h2 ones = { (_Float16)1.f, (_Float16)1.f };
#pragma unroll
  for (int j = 0; j < 8; j += 2) { const h2 pp = { pf[j], pf[j + 1] }; acc = __builtin_amdgcn_fdot2(pp, ones, acc, false); }
  return acc;
}
// 16 int8 values x scale -> 16 f16 (see the Q8 note at the kernel)
static __device__ inline void dq16(const u4 raw, const float sc, h8& lo, h8& hi) {
  const h2 s2 = { (_Float16)sc, (_Float16)sc };
  const h2 off = { (_Float16)1152.f, (_Float16)1152.f };
  h2 o[8];
#pragma unroll
  for (int d = 0; d < 4; d++) {
    const uint32_t w = raw[d] ^ 0x80808080u;
    const uint32_t a = __builtin_amdgcn_perm(0x64646464u, w, 0x04010400u), b = __builtin_amdgcn_perm(0x64646464u, w, 0x04030402u);
    h2 xa, xb;
    __builtin_memcpy(&xa, &a, 4); __builtin_memcpy(&xb, &b, 4);
    o[2 * d] = (xa - off) * s2;
    o[2 * d + 1] = (xb - off) * s2;
  }
  lo = (h8){ o[0][0], o[0][1], o[1][0], o[1][1], o[2][0], o[2][1], o[3][0], o[3][1] };
  hi = (h8){ o[4][0], o[4][1], o[5][0], o[5][1], o[6][0], o[6][1], o[7][0], o[7][1] };
}

template <int HD> struct DecShape {
  static constexpr int LPR = HD / 8;            // lanes per f16 row at 16 bytes a lane
  static constexpr int RPL = 64 / LPR;          // rows per wave-wide load
  static constexpr int NLD = TILE / RPL;        // loads per tile and tensor
  static constexpr int KROW = HD * 2 + 16;      // staged K row stride (bytes): 16 rows x 16 B hit distinct banks
  static constexpr int VROW = HD * 2 + 32;      // staged V row stride (bytes)
  static constexpr int STAGE = TILE * VROW;     // wave-private staging bytes (>= 16 x (HD + 4) floats for the merge)
  static constexpr int QROW = HD * 2 + 16;      // staged q row stride (bytes)
  static constexpr int OROW = (HD + 4) * 4;     // merge row stride (bytes)
  // int8 caches: 16 values a lane
  static constexpr int LPR8 = HD / 16;          // lanes per int8 row
  static constexpr int RPL8 = 64 / LPR8;        // rows per wave-wide load
  static constexpr int NLD8 = TILE / RPL8;      // loads per tile and tensor
  static constexpr int SPR = HD / 32;           // scales per row
  static constexpr int LPS = SPR / 4;           // lanes per row of scales at 16 bytes a lane
  static constexpr int KS = HD / 32;            // k-steps of the QK product
  static constexpr int DB = HD / 16;            // 16-dim blocks of the output
};

// One-token projections either side of the attention block on gfx950: y = W x for f32, Q8_0 and Q4_0 weights,
// optionally over rmsnorm(x) computed in the kernel, optionally accumulated into y.
//
// Replaces the reference's matvec / matvec_q8 / matvec_q4 and their cooperative forms (engine/wgsl/base.js:15-118,
// engine/wgsl/coop.js:236-345), the accumulate variants (_coop_acc, coop.js:347-349: y[row] += W x, the residual add
// folded in) and the normed variants (_coop_n, coop.js:371-420: rmsnorm of the raw residual inside the GEMV).
// Weight formats are the reference's split planes:
//   Q8_0: int8 [d_out][d_in] + one f16 scale per 32 values; y_r = sum_b sc_rb * sum_j q_rbj * x_bj
//   Q4_0: nibbles [d_out][d_in / 2], byte j of a 16-byte block = element j (low nibble) and j + 16 (high nibble),
//         value = nibble - 8; same scales.
//
// A one-token GEMV reads every weight once and the 8-32 KB activation many times: it is HBM- and latency-bound,
// not arithmetic.  Shape here: a 64-lane wavefront owns RW output rows; lane l owns the 32-value blocks l, l + 64,
// ... of the input (one Q4_0 block = one 16-byte load, so a wave-wide load is 1 KB of one row, fully coalesced),
// keeps its slices of x in registers for all its rows (x reaches them through LDS, loaded coalesced once per
// workgroup), issues every weight and scale load of its rows before the first use, and sums the 64 lanes with DPP
// permutations.  All arithmetic is f32 as in the reference; the order of
// the additions differs from the reference's workgroup tree (the parity tests use a tolerance, as the reference's do).
#include "pa_internal.h"
#include "glue_math.h"
#include <algorithm>

typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));

// 32 weights of one block times the lane's 32 activations, scale not applied
template <int KIND> struct BlockRegs;
template <> struct BlockRegs<PA_W_F32> { f4 w[8]; };
template <> struct BlockRegs<PA_W_Q8_0> { u4 w[2]; };
template <> struct BlockRegs<PA_W_Q4_0> { u4 w[1]; };

template <int KIND>
static __device__ inline void load_block(BlockRegs<KIND>& r, const unsigned char* base, size_t row, uint32_t nb, uint32_t b) {
  if constexpr (KIND == PA_W_F32) {
    const f4* s = (const f4*)(base + ((size_t)row * nb + b) * 128);
#pragma unroll
    for (int i = 0; i < 8; i++) r.w[i] = s[i];
  } else if constexpr (KIND == PA_W_Q8_0) {
    const u4* s = (const u4*)(base + ((size_t)row * nb + b) * 32);
    r.w[0] = s[0]; r.w[1] = s[1];
  } else {
    r.w[0] = *(const u4*)(base + ((size_t)row * nb + b) * 16);
  }
}

template <int KIND>
static __device__ inline float dot_block(const BlockRegs<KIND>& r, const float (&x)[32], float sx) {
  float a = 0.f;
  if constexpr (KIND == PA_W_F32) {
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) a = __builtin_fmaf(r.w[i][j], x[4 * i + j], a);
    return a;
  } else if constexpr (KIND == PA_W_Q8_0) {
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int word = (int)r.w[i][k];
#pragma unroll
        for (int j = 0; j < 4; j++) a = __builtin_fmaf((float)((word << (24 - 8 * j)) >> 24), x[16 * i + 4 * k + j], a);
      }
    return a;
  } else {
    // sum (n - 8) x = sum n x - 8 sum x.  A nibble n in the low bits of a 16-bit half IS the f16 subnormal n x 2^-24, and
    // the mixed-precision fma takes an f16 operand as it is: two nibbles of a word are isolated by one shift and one mask
    // (15 instructions for 8 weights instead of 23 with byte-to-float conversions), the products are the same bits scaled
    // by a power of two, and the sum is scaled back once.
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t word = r.w[0][k];
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const uint32_t pr = (word >> (4 * t)) & 0x000F000Fu;          // nibble t of the word (low half) and nibble t + 4 (high half)
        h2v v; __builtin_memcpy(&v, &pr, 4);
        const int e = 4 * k + (t >> 1) + 16 * (t & 1);                 // nibble 2 j of a word is element j of its four bytes, nibble 2 j + 1 element j + 16
        a = __builtin_fmaf((float)v[0], x[e], a);
        a = __builtin_fmaf((float)v[1], x[e + 2], a);
      }
    }
    a *= 16777216.0f;
    return a - 8.0f * sx;
  }
}

// BPL: blocks per lane and pass; PASSES: passes over the input (d_in <= 2048 * BPL * PASSES; two for f32 weights past
// 4096 inputs, whose 32 registers a block leave no room for four blocks a lane: the second pass's weight rows are
// requested when the first pass's are consumed); RW: rows per wave; AT_ONCE: all of them requested in front
template <int KIND, int BPL, int RW, bool NORM, int PASSES, bool AT_ONCE>
__global__ __launch_bounds__(256)
void pa_gemv_kernel(const float* a_x, const float* a_norm_w, const void* a_w, const uint16_t* a_scales, float* a_y, uint32_t a_d_out, uint32_t a_d_in, GemvParams p_in) {
  // The leading arguments repeat fields of p_in: the first twelve dwords of the arguments are preloaded into scalar
  // registers, so every load address of the kernel is there when the wave starts; the other arguments are fetched in one
  // batch of scalar loads (the compiler would fetch each where it is first used, a dependent round trip each).
  GemvParams p = p_in;
  p.x = a_x; p.norm_w = a_norm_w; p.w = a_w; p.scales = a_scales; p.y = a_y; p.d_out = a_d_out; p.d_in = a_d_in;
  // Up to 4096 inputs, for up to three rows, and with AT_ONCE (pa_rule_gemv_at_once) a wave's rows are all requested at once; past that it keeps two or three in flight and asks for the next when
  // one is consumed.  With everything requested in front, a wave sat in the issue of its loads while the memory pipeline was full (of 14336 x 5120 Q4_0, seven rows a wave:
  // until 4.3 us after the first wave's entry on average, 7.4 at the latest), staged x behind that and did all of its arithmetic, 3 us, behind the last
  // byte; so the arithmetic runs under the stream (12.5 -> 10.8 us; 16384 x 5120 14.1 -> 11.9, 14336 x 8192 18.5 -> 14.3; one row in flight 13.3, three 11.0;
  // without the norm three are ahead, 12288 x 6144 10.35 / 10.15).  The rows of a wave are then dealt one of every 4 x gridDim.x: at any time the chip reads one
  // range of the matrix (10.8 -> 10.5 us), and the waves' counts differ by one at most.
  constexpr int AHEAD = AT_ONCE || BPL < 3 || KIND == PA_W_F32 || RW <= 3 ? RW : KIND == PA_W_Q4_0 && BPL == 3 && !NORM && RW >= 5 ? 3 : 2;
  constexpr bool STREAM = RW > AHEAD;
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t nb = p.d_in / 32;
  // rows of a wave: consecutive ones, or, where it streams them, one of every 4 x gridDim.x
  const size_t row0 = STREAM ? (size_t)__builtin_amdgcn_readfirstlane(wave) * gridDim.x + blockIdx.x : ((size_t)blockIdx.x * 4 + wave) * RW;
  const size_t row_step = STREAM ? 4 * (size_t)gridDim.x : 1;
  const unsigned char* wbase = (const unsigned char*)p.w;
  // x (and the norm weights) are requested FIRST, the wave's weight rows right behind them: the loads of a wave complete
  // in order, x comes from L2 in a fraction of the time the weight stream takes from HBM, and everything that depends
  // on x alone -- the sum of squares, two barriers, the trip through LDS -- then runs under the latency of the weights
  // instead of after it.
  extern __shared__ __attribute__((aligned(16))) float xs[];
  __shared__ float red[4];
  constexpr int XPT = 2 * BPL * PASSES;                                // float4 of x per thread (d_in <= 2048 * BPL * PASSES)
  const uint32_t n4 = p.d_in / 4;
  f4 xv[XPT], wv[NORM ? XPT : 1];
  float ss = 0.f;
  // Loads past the end of x re-read its last float4 instead of being guarded (their values are never stored, and are
  // masked out of the sum of squares by a factor, not by a select on the loaded value): a guarded load is a branch,
  // and between guarded blocks the compiler placed a full wait.
#pragma unroll
  for (int k = 0; k < XPT; k++) xv[k] = ((const f4*)p.x)[min(threadIdx.x + 256 * k, n4 - 1)];
  if constexpr (NORM) {
#pragma unroll
    for (int k = 0; k < XPT; k++) wv[k] = ((const f4*)p.norm_w)[min(threadIdx.x + 256 * k, n4 - 1)];
  }
  __builtin_amdgcn_sched_barrier(0);
  BlockRegs<KIND> wr[RW][BPL];
  uint16_t sc[RW][BPL];
  auto request = [&](int r, int pass) __attribute__((always_inline)) {
    const size_t row = min(row0 + r * row_step, (size_t)p.d_out - 1);            // rows past the end repeat the last one (not stored)
#pragma unroll
    for (int i = 0; i < BPL; i++) {
      const uint32_t b = min(lane + 64 * (i + BPL * pass), nb - 1);    // blocks past the end likewise (weighted by x = 0)
      load_block<KIND>(wr[r][i], wbase, row, nb, b);
      if constexpr (KIND != PA_W_F32) sc[r][i] = p.scales[row * nb + b];
    }
  };
#pragma unroll
  for (int r = 0; r < (RW < AHEAD ? RW : AHEAD); r++) request(r, 0);
  // accumulating calls: the old values of the wave's rows are requested here, with everything else, instead of in a
  // round trip of their own behind the reduction
  asm volatile("" :: "s"(p.xn_out), "s"(p.eps), "s"(p.acc));
  float yold[RW];
#pragma unroll
  for (int r = 0; r < RW; r++) yold[r] = p.acc ? p.y[min(row0 + r * row_step, (size_t)p.d_out - 1)] : 0.f;
  __builtin_amdgcn_sched_barrier(0);
  // x -> LDS (a lane's own slice is 32 consecutive floats: loaded directly, a wave-wide load would touch 64 cache lines
  // for 1 KB), normed on the way when asked; block b sits at xs[b * 36]: the 4-float pad makes the 8 lanes of a 128-bit
  // LDS read phase hit distinct banks
  if constexpr (NORM) {
#pragma unroll
    for (int k = 0; k < XPT; k++) {
      const float m = threadIdx.x + 256 * k < n4 ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < 4; j++) ss = __builtin_fmaf(xv[k][j] * m, xv[k][j], ss);
    }
    ss = wave_sum_f32(ss);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    // xn = (x * inv) * w with inv = 1 / sqrt(mean(x^2) + eps), as the reference's rmsnorm writes it
    // (engine/wgsl/base.js:119-152, coop.js:407-411); every workgroup recomputes it, as the reference's do
    const float inv = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)p.d_in + p.eps);
#pragma unroll
    for (int k = 0; k < XPT; k++)
#pragma unroll
      for (int j = 0; j < 4; j++) xv[k][j] = (xv[k][j] * inv) * wv[k][j];
    if (p.xn_out && blockIdx.x == 0) {
#pragma unroll
      for (int k = 0; k < XPT; k++) { const uint32_t e = threadIdx.x + 256 * k; if (e < n4) ((f4*)p.xn_out)[e] = xv[k]; }
    }
  }
#pragma unroll
  for (int k = 0; k < XPT; k++) {
    const uint32_t e = threadIdx.x + 256 * k;
    if (e < n4) *(f4*)(xs + (e / 8) * 36 + (e % 8) * 4) = xv[k];
  }
  __syncthreads();
  float part[RW];
#pragma unroll
  for (int r = 0; r < RW; r++) part[r] = 0.f;
#pragma unroll
  for (int pass = 0; pass < PASSES; pass++) {
  if (pass > 0) {                                                      // the next pass's weight rows
#pragma unroll
    for (int r = 0; r < (RW < AHEAD ? RW : AHEAD); r++) request(r, pass);
  }
  float x[BPL][32], sx[BPL];
#pragma unroll
  for (int i = 0; i < BPL; i++) {
    const uint32_t b = lane + 64 * (i + BPL * pass);
    const bool on = b < nb;
    const f4* src = (const f4*)(xs + min(b, nb - 1) * 36);
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const f4 v = src[k];
#pragma unroll
      for (int j = 0; j < 4; j++) x[i][4 * k + j] = on ? v[j] : 0.f;
    }
  }
  if constexpr (KIND == PA_W_Q4_0) {
#pragma unroll
    for (int i = 0; i < BPL; i++) {
      float t = 0.f;
#pragma unroll
      for (int j = 0; j < 32; j++) t += x[i][j];
      sx[i] = t;
    }
  } else {
#pragma unroll
    for (int i = 0; i < BPL; i++) sx[i] = 0.f;
  }
#pragma unroll
  for (int r = 0; r < RW; r++) {
    float a = part[r];
#pragma unroll
    for (int i = 0; i < BPL; i++) {
      const float d = dot_block<KIND>(wr[r][i], x[i], sx[i]);
      if constexpr (KIND == PA_W_F32) a += d;
      else a = __builtin_fmaf((float)__ushort_as_half(sc[r][i]), d, a);
    }
    part[r] = a;
    if constexpr (RW > AHEAD) {
      __builtin_amdgcn_sched_barrier(0);
      if (r + AHEAD < RW) request(r + AHEAD, pass);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  }
#pragma unroll
  for (int r = 0; r < RW; r++) part[r] = wave_sum_f32(part[r]);
  if (lane == 0) {
#pragma unroll
    for (int r = 0; r < RW; r++) {
      const size_t row = row0 + r * row_step;
      if (row < p.d_out) p.y[row] = p.acc ? yold[r] + part[r] : part[r];
    }
  }
}

template <int KIND, int BPL, int RW, bool NORM, int PASSES = 1, bool AT_ONCE = false>
static hipError_t launch_k(const GemvParams& p, hipStream_t s, uint32_t wgs = 0) {
  if (wgs == 0) wgs = (p.d_out + 4 * RW - 1) / (4 * RW);
  const size_t lds = (size_t)(p.d_in / 32) * 36 * sizeof(float);
  hipLaunchKernelGGL((pa_gemv_kernel<KIND, BPL, RW, NORM, PASSES, AT_ONCE>), dim3(wgs), dim3(256), lds, s, p.x, p.norm_w, p.w, p.scales, p.y, p.d_out, p.d_in, p);
  return hipGetLastError();
}

// rw of 1 .. R rows per wave
template <int KIND, int BPL, bool NORM, int R>
static hipError_t launch_rows(uint32_t rw, const GemvParams& p, hipStream_t s, uint32_t wgs = 0) {
  if constexpr (R > 1) { if (rw < (uint32_t)R) return launch_rows<KIND, BPL, NORM, R - 1>(rw, p, s, wgs); }
  return launch_k<KIND, BPL, R, NORM>(p, s, wgs);
}

// Rows per wave past 4096 inputs (quantised weights) of the calls that pa_rule_gemv_resident leaves.  Every workgroup fetches, norms and stages all of x -- 20 KB and the norm's
// 20 KB at 5120 inputs, twice the Q4_0 weights of its eight rows at two rows a wave -- so few large workgroups are faster as long as
// every SIMD keeps two waves and they come out even.  Time follows the rows of the busiest SIMD plus about 1.6 rows' worth for every
// wave it is dealt; measured at 1 .. 7 rows a wave with the norm (us, cold weights, Q4_0): 14336 x 5120 18.5 13.5 13.3 13.1 12.9 13.6 12.3;
// 10240 x 5120 14.6 11.3 11.3 10.7 9.7 10.5 11.6; 8192 x 5120 12.5 9.1 9.7 8.6 9.4 10.6 11.7; 17000 x 4608 20.8 15.5 15.0 14.7 14.8
// 14.0 15.0.  With fewer than six rows a SIMD two rows a wave are as good as any (5120 x 6144: 7.3, 7.4 at three, 7.3 at five).
// Q8_0 rows are twice the bytes to the same x: two rows a wave are ahead everywhere without the norm (14336 x 5120 18.9 16.4 16.9 17.5 17.6,
// accumulating 18.3 15.9 17.3 17.8 17.6; 17000 x 4608 21.6 17.4 18.5 18.9 20.1) and with it past 12 rows a SIMD or four blocks a lane
// (17000 x 4608 22.0 19.2 20.0 20.6 20.5; 16000 x 7168 35.9 26.9 28.1); below, the rule's choice (7168 x 5120 12.4 11.1 11.6 10.7 12.1; 9000 x 6016
// 15.6 14.4 13.8 15.4 13.9).  At most what fits the registers of two waves a SIMD.
static constexpr uint32_t wide_rows_max(int kind, int bpl, bool norm) {
  return kind == PA_W_Q4_0 ? (bpl == 3 ? 7 : 4) : norm && bpl == 3 ? 5 : 2;
}
extern "C" uint32_t pa_rule_gemv_wide_rows(int kind, uint32_t d_out, uint32_t d_in, int norm, int n_cu) {
  const uint32_t simds = 4u * (uint32_t)n_cu;
  if (d_out < 6 * simds) return d_out >= 4 * simds ? 2 : 1;
  const uint32_t rmax = wide_rows_max(kind, d_in <= 6144 ? 3 : 4, norm != 0);
  if (rmax == 2 || (kind == PA_W_Q8_0 && d_out > 12 * simds)) return 2;
  uint32_t best = 1;
  float cost = 1e30f;
  for (uint32_t r = 1; r <= rmax; r++) {
    const uint32_t waves = (d_out + r - 1) / r, per_simd = (waves + simds - 1) / simds;
    const float c = per_simd * (r + 1.6f);
    if (per_simd >= 2 && c < cost) { best = r; cost = c; }
  }
  return best;
}

// One or two workgroups a CU that stay for the whole call (<< 16 | the rows a wave; 0: neither): past 4096 inputs, quantised weights.  Every workgroup stages all of x and every
// wave reads it from LDS into its registers (10 waves a CU of 5120 x 6144: 240 KB, 0.8 us), so as few of them as keep the stream going are ahead.  One a CU with the norm
// in front up to eight rows a wave (Q4_0 2048 x 6144 5.6 -> 4.4 us, 3072 x 5120 6.5 -> 4.6, 5120 x 5120 7.4 -> 6.7, 6144 x 6144 8.1 -> 7.5, 8192 x 8192 12.0 -> 10.4; Q8_0
// 5120 x 6144 10.1 -> 8.7, 7168 x 5120 10.6 -> 9.7), but up to five for Q4_0 rows of at most 5120 inputs, whose arithmetic four waves a CU do not hide under so few bytes (5600 x 4128 7.3,
// one a CU 7.6; 7600 x 4128 8.2 and 8.8, x 5120 8.4 and 8.9, x 5632 8.9 and 9.0, x 6144 9.3 and 9.1).  Without the norm up to three rows and at five, where the rule above
// comes to 2.0 - 2.5 workgroups of two rows a wave a CU (Q4_0 4200, 4700 and 5120 rows of 6144 7.2 -> 7.0, 7.3 -> 6.9, 7.4 -> 7.1, of 8192 8.7 -> 8.2, 8.9 -> 8.3, 9.1 -> 8.4; Q8_0 of 6144 8.9 -> 8.1,
// 9.0 -> 8.4, 9.0 -> 8.7; the few workgroups of 4097 - 4112 rows past two a CU are not worth it: 4104 x 6144 6.65, one a CU 6.87, 4120 x 6144 6.96 and 6.88), but not at
// four or six (4096 x 6144 5.9, one a CU 6.3; 6144 x 6144 7.2 and 7.7; Q8_0 three rows 6.0 and 6.3).  Two a CU from there to eight rows
// (Q4_0 14336 x 5120 12.5 -> 10.5, 9500 x 7168 14.5 -> 11.3; Q8_0 14336 x 5120 17.5 -> 15.2, 9216 x 5120 without the norm 11.6 -> 10.8; at four rows Q8_0 6144 x 6144
// 9.1 -> 9.7), from six for Q4_0 rows of less than 5120 inputs without the norm (9000 x 4128 8.6, two a CU 9.0, x 5120 9.2 and 9.2).  More rows a wave were not built.
// (Up to three rows a wave do not stream and stay consecutive, so the last CUs may have none: 1025 rows of 5120 on 129 workgroups 4.2 us, dealt over all of them one
// row of every 1024 4.7; 2049 x 8192 with the norm 6.5 and 7.3.)
extern "C" uint32_t pa_rule_gemv_resident(int kind, uint32_t d_out, uint32_t d_in, int norm, int n_cu) {
  const uint32_t one = (d_out + 4 * n_cu - 1) / (4 * n_cu), two = (d_out + 8 * n_cu - 1) / (8 * n_cu);
  const bool q4 = kind == PA_W_Q4_0;
  if (norm ? one <= (q4 && d_in <= 5120 ? 5 : 8) : one <= 2 || (one == 3 && q4) || (one == 5 && d_out > 16u * n_cu + n_cu / 16)) return 1u << 16 | one;
  if (two >= (q4 && !norm && d_in < 5120 ? 6 : 5) && two <= 8) return 2u << 16 | two;
  return 0;
}
// Q4_0 calls of four or five rows a wave that the rule above leaves, without the norm: all rows requested in front where that is ahead of two or three in flight, over short rows and on
// tall weights, whose five waves a SIMD keep the stream going by themselves (us, in front / streamed: 7200 x 4128 7.3 / 7.7, x 4608 7.5 / 7.7, x 5120 7.7 / 7.8, x 6144 8.2 / 8.1, x 8192 11.0 / 10.4; 9000 x 4128
// 8.6 / 9.0; 19000 x 6400 19.0 / 21.0, x 8192 21.6 / 22.5).
extern "C" int pa_rule_gemv_at_once(int kind, uint32_t d_out, uint32_t d_in, int norm, uint32_t rows, int n_cu) {
  return kind == PA_W_Q4_0 && !norm && ((rows == 4 && (d_in <= 5120 || d_out > 64u * n_cu)) || (rows == 5 && d_in <= 5120));
}

template <int KIND, int BPL, bool NORM>
static hipError_t launch_rw(const GemvParams& p, int n_cu, hipStream_t s) {
  if constexpr (BPL >= 3) {
    const uint32_t resident = pa_rule_gemv_resident(KIND, p.d_out, p.d_in, NORM, n_cu);
    if (resident) return launch_rows<KIND, BPL, NORM, 8>(resident & 0xffff, p, s, std::min((resident >> 16) * (uint32_t)n_cu, (p.d_out + 3) / 4));
    const uint32_t rows = pa_rule_gemv_wide_rows(KIND, p.d_out, p.d_in, NORM, n_cu);
    if constexpr (KIND == PA_W_Q4_0 && !NORM) {
      if (pa_rule_gemv_at_once(KIND, p.d_out, p.d_in, NORM, rows, n_cu)) {
        if constexpr (BPL == 3) { if (rows == 5) return launch_k<KIND, BPL, 5, NORM, 1, true>(p, s); }
        return launch_k<KIND, BPL, 4, NORM, 1, true>(p, s);
      }
    }
    return launch_rows<KIND, BPL, NORM, wide_rows_max(KIND, BPL, NORM)>(rows, p, s);
  } else {
    // rows per wave: as many as still leave about two 4-wave workgroups per CU, within the registers that RW x BPL
    // blocks of weights take (f32: 32 registers a block, Q8_0: 8, Q4_0: 4)
    constexpr int RWMAX = (KIND == PA_W_F32 ? 2 : 8) / BPL > 0 ? (KIND == PA_W_F32 ? 2 : 8) / BPL : 1;
    const uint32_t waves_wanted = 8u * (uint32_t)n_cu;
    uint32_t rw = p.d_out >= 8 * waves_wanted ? 8 : p.d_out >= 4 * waves_wanted ? 4 : p.d_out >= 2 * waves_wanted ? 2 : 1;
    if (rw > (uint32_t)RWMAX) rw = RWMAX;
    // Once the weights are there the kernel is VALU work, and the SIMD with the most rows sets the time: with four rows a
    // wave the MoE model's 9216 [q|k|v] rows are 2304 waves, 2.25 a SIMD -- some SIMDs work through three waves (12 rows),
    // most through two.  Three rows a wave are 3072 waves, three on every SIMD (9 rows).  Taken when it lowers the busiest
    // SIMD's rows.
    if constexpr (RWMAX >= 4) {
      const uint32_t simds = 4u * (uint32_t)n_cu;
      auto busiest = [&](uint32_t r) { const uint32_t waves = (p.d_out + r - 1) / r; return ((waves + simds - 1) / simds) * r; };
      if (rw == 4 && busiest(3) < busiest(4)) return launch_k<KIND, BPL, 3, NORM>(p, s);
    }
    if constexpr (RWMAX >= 8) { if (rw == 8) return launch_k<KIND, BPL, 8, NORM>(p, s); }
    if constexpr (RWMAX >= 4) { if (rw >= 4) return launch_k<KIND, BPL, 4, NORM>(p, s); }
    if constexpr (RWMAX >= 2) { if (rw >= 2) return launch_k<KIND, BPL, 2, NORM>(p, s); }
    return launch_k<KIND, BPL, 1, NORM>(p, s);
  }
}

template <int KIND, bool NORM>
static hipError_t launch_bpl(const GemvParams& p, int n_cu, hipStream_t s) {
  const uint32_t nb = p.d_in / 32;
  if (nb <= 64) return launch_rw<KIND, 1, NORM>(p, n_cu, s);
  if (nb <= 128) return launch_rw<KIND, 2, NORM>(p, n_cu, s);
  if constexpr (KIND != PA_W_F32) {
    if (nb <= 192) return launch_rw<KIND, 3, NORM>(p, n_cu, s);
    if (nb <= 256) return launch_rw<KIND, 4, NORM>(p, n_cu, s);
  } else {
    if (nb <= 256) return launch_k<KIND, 2, 1, NORM, 2>(p, s);        // f32 weights past 4096 inputs: two passes of two blocks a lane
  }
  return hipErrorNotSupported;
}

hipError_t pa_launch_gemv(const GemvParams& p, int n_cu, hipStream_t s) {
  if (p.d_out == 0 || p.d_in == 0 || (p.d_in & 31)) return hipErrorInvalidValue;
  const bool norm = p.norm_w != nullptr;
  switch (p.kind) {
    case PA_W_F32: return norm ? launch_bpl<PA_W_F32, true>(p, n_cu, s) : launch_bpl<PA_W_F32, false>(p, n_cu, s);
    case PA_W_Q8_0: return norm ? launch_bpl<PA_W_Q8_0, true>(p, n_cu, s) : launch_bpl<PA_W_Q8_0, false>(p, n_cu, s);
    case PA_W_Q4_0: return norm ? launch_bpl<PA_W_Q4_0, true>(p, n_cu, s) : launch_bpl<PA_W_Q4_0, false>(p, n_cu, s);
    default: return hipErrorInvalidValue;
  }
}

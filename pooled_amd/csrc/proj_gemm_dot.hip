// Column-batched projections for one to four columns over long rows on gfx950, where the matrix-core kernel of proj_gemm_skinny.hip
// comes out slower: Y[c][r] = sum_k W[r][k] X[c][k] straight from the packed Q8_0 / Q4_0 planes, on the VALU's dot products.  Same
// operand precision (weights and activations f16, products and sums f32); the reference's counterpart is the batched cooperative
// matvec (engine/wgsl/coop.js).
//
// A wave owns RW rows, a lane the 32-value blocks lane + 64 i of each; the weights are widened once into f16 pairs in registers, the
// columns staged in LDS (80-byte block stride: conflict-free 128-bit reads), one v_dot2_f32_f16 runs per two weights and column, and
// the lanes' partial sums go through LDS: lane t of a wave adds up the 64 partials of its (row, column).
// What bounds it: the weight stream, and per column the dot products of lanes that hold whole blocks whatever d_in is (past 4096 inputs
// four blocks a lane).  Few workgroups' worth of rows still fill the chip, as a workgroup is 4 RW rows, where the matrix-core kernel takes
// 16 with all of K in one CU's LDS: with 16 Q8_0 rows of 6144 inputs staged a CU holds one workgroup, and 320 of them are two rounds.
#include "pf_common.h"

#define DOT_BLOCK 80    // bytes from one staged block of 32 activations to the next
#define DOT_COLS 4

static __device__ inline h2 dot_as_h2(uint32_t u) { h2 r; __builtin_memcpy(&r, &u, 4); return r; }
// two bytes of a word (byte indices by the selector) -> two f16 = (byte - bias) * scale
static __device__ inline h2 dot_widen(uint32_t w, uint32_t sel, h2 bias, h2 sc) { return (dot_as_h2(__builtin_amdgcn_perm(0x64646464u, w, sel)) - bias) * sc; }

template <int KIND, int BPL, int RW>
__global__ __launch_bounds__(256)
void pa_gemm_dot_kernel(const uint16_t* a_x, const void* a_w, const uint16_t* a_scales, uint32_t a_x_stride, uint32_t a_d_out, uint32_t a_d_in, uint32_t a_n_cols,
                        GemmParams p_in) {
  // (the leading arguments repeat fields of p_in: they are preloaded into scalar registers, so the loads below need no
  // scalar-load round trip; the other arguments are fetched in one batch behind them)
  GemmParams p = p_in;
  p.x = a_x; p.w = a_w; p.scales = a_scales; p.x_stride = a_x_stride; p.d_out = a_d_out; p.d_in = a_d_in; p.n_cols = a_n_cols;
  extern __shared__ __attribute__((aligned(16))) unsigned char dot_lds[];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t nb = p.d_in / 32, ncol = p.n_cols;
  const uint32_t xcol = nb * DOT_BLOCK;                               // bytes of a staged column
  const size_t row0 = ((size_t)blockIdx.x * 4 + wave) * RW;
  // The first eight 16-byte pieces a thread stages of the columns are requested FIRST, the wave's weight rows right behind them: a
  // wave's loads complete in order, the columns come from L2 in a fraction of the time the weight stream takes from HBM, and their trip
  // into LDS then runs under the latency of the weights instead of after it.
  const uint32_t cpc = p.d_in / 8, pieces = ncol * cpc;               // 16-byte pieces of a column, of all
  u4 xv0[8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const uint32_t e = min(tid + 256 * j, pieces - 1), c = e / cpc, k8 = e % cpc;
    xv0[j] = *(const u4*)((const unsigned char*)(p.x + (size_t)c * p.x_stride) + k8 * 16);
  }
  __builtin_amdgcn_sched_barrier(0);
  constexpr int WQ = KIND == PA_W_Q4_0 ? 1 : 2;                       // 16-byte words of a packed block
  u4 wq[RW][BPL][WQ];
  uint16_t wsc[RW][BPL];
#pragma unroll
  for (int r = 0; r < RW; r++) {
    const size_t row = min(row0 + r, (size_t)p.d_out - 1);            // rows past the end repeat the last one (not stored)
#pragma unroll
    for (int i = 0; i < BPL; i++) {
      const uint32_t b = min(lane + 64 * i, nb - 1);                  // blocks past the end likewise (scale forced to 0)
      const u4* src = (const u4*)((const unsigned char*)p.w + (row * nb + b) * (16 * WQ));
#pragma unroll
      for (int w = 0; w < WQ; w++) wq[r][i][w] = src[w];
      wsc[r][i] = p.scales[row * nb + b];
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" :: "s"(p.y), "s"(p.y_stride), "s"(p.acc));
  auto stage = [&](uint32_t e, const u4& v) __attribute__((always_inline)) {
    const uint32_t c = e / cpc, k8 = e % cpc;
    if (e < pieces) *(u4*)(dot_lds + c * xcol + (k8 >> 2) * DOT_BLOCK + (k8 & 3) * 16) = v;
  };
#pragma unroll
  for (int j = 0; j < 8; j++) stage(tid + 256 * j, xv0[j]);
  // any further pieces, eight loads a thread ahead of the first store (unconditional: one past the end re-reads the last piece)
  for (uint32_t e0 = tid + 256 * 8; e0 < pieces; e0 += 256 * 8) {
    u4 v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const uint32_t e = min(e0 + 256 * j, pieces - 1), c = e / cpc, k8 = e % cpc;
      v[j] = *(const u4*)((const unsigned char*)(p.x + (size_t)c * p.x_stride) + k8 * 16);
    }
#pragma unroll
    for (int j = 0; j < 8; j++) stage(e0 + 256 * j, v[j]);
  }
  // widen: pair k of a block = elements 2k, 2k + 1
  h2 wv[RW][BPL][16];
#pragma unroll
  for (int r = 0; r < RW; r++)
#pragma unroll
    for (int i = 0; i < BPL; i++) {
      const _Float16 s1 = __ushort_as_half(lane + 64 * i < nb ? wsc[r][i] : (uint16_t)0);
      const h2 sc = { s1, s1 };
      if constexpr (KIND == PA_W_Q4_0) {
        const h2 bias = { (_Float16)1032.f, (_Float16)1032.f };        // 0x6400 | n = 1024 + n; n - 8
#pragma unroll
        for (int d = 0; d < 4; d++) {
          const uint32_t l = wq[r][i][0][d] & 0x0F0F0F0Fu, h = (wq[r][i][0][d] >> 4) & 0x0F0F0F0Fu;
          wv[r][i][2 * d] = dot_widen(l, 0x04010400u, bias, sc); wv[r][i][2 * d + 1] = dot_widen(l, 0x04030402u, bias, sc);
          wv[r][i][8 + 2 * d] = dot_widen(h, 0x04010400u, bias, sc); wv[r][i][8 + 2 * d + 1] = dot_widen(h, 0x04030402u, bias, sc);
        }
      } else {
        const h2 bias = { (_Float16)1152.f, (_Float16)1152.f };        // 0x6400 | (v + 128) = 1152 + v
#pragma unroll
        for (int w = 0; w < 2; w++)
#pragma unroll
          for (int d = 0; d < 4; d++) {
            const uint32_t x = wq[r][i][w][d] ^ 0x80808080u;
            wv[r][i][8 * w + 2 * d] = dot_widen(x, 0x04010400u, bias, sc); wv[r][i][8 * w + 2 * d + 1] = dot_widen(x, 0x04030402u, bias, sc);
          }
      }
    }
  __syncthreads();
  float part[DOT_COLS][RW];
#pragma unroll
  for (int c = 0; c < DOT_COLS; c++) {
#pragma unroll
    for (int r = 0; r < RW; r++) part[c][r] = 0.f;
    if ((uint32_t)c < ncol) {
#pragma unroll
      for (int i = 0; i < BPL; i++) {
        const unsigned char* xb = dot_lds + c * xcol + min(lane + 64 * i, nb - 1) * DOT_BLOCK;
        h2 xv[16];
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const h8 v = *(const h8*)(xb + 16 * q);
          xv[4 * q] = (h2){ v[0], v[1] }; xv[4 * q + 1] = (h2){ v[2], v[3] }; xv[4 * q + 2] = (h2){ v[4], v[5] }; xv[4 * q + 3] = (h2){ v[6], v[7] };
        }
#pragma unroll
        for (int r = 0; r < RW; r++)
#pragma unroll
          for (int k = 0; k < 16; k++) part[c][r] = __builtin_amdgcn_fdot2(wv[r][i][k], xv[k], part[c][r], false);
      }
    }
  }
  __syncthreads();                                                    // every wave is done with the staged columns
  // partials -> LDS [wave][lane][DOT_COLS RW + 1], then lane t sums column t of its wave's table
  constexpr int PS = DOT_COLS * RW + 1;
  float* ps = (float*)dot_lds + (size_t)wave * 64 * PS;
#pragma unroll
  for (int c = 0; c < DOT_COLS; c++)
    if ((uint32_t)c < ncol)
#pragma unroll
      for (int r = 0; r < RW; r++) ps[lane * PS + c * RW + r] = part[c][r];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  for (uint32_t t = lane; t < ncol * RW; t += 64) {
    const uint32_t c = t / RW, r = t % RW;
    float* y = p.y + (size_t)c * p.y_stride + min(row0 + r, (size_t)p.d_out - 1);
    const float yo = p.acc ? *y : 0.f;                                // on its way while the partials are added up
    float a = 0.f;
    for (int l = 0; l < 64; l++) a += ps[l * PS + t];
    if (row0 + r < p.d_out) *y = p.acc ? yo + a : a;
  }
}

template <int KIND, int BPL, int RW>
static hipError_t dot_launch(const GemmParams& p, hipStream_t s) {
  const size_t x = (size_t)p.n_cols * (p.d_in / 32) * DOT_BLOCK, ps = (size_t)4 * 64 * (DOT_COLS * RW + 1) * sizeof(float), lds = x > ps ? x : ps;
  if (lds > 65536) {
    static PaPerDevice lds_set;
    const hipError_t e = pa_lds_limit(lds_set, (const void*)pa_gemm_dot_kernel<KIND, BPL, RW>, (size_t)DOT_COLS * (64 * BPL) * DOT_BLOCK);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((pa_gemm_dot_kernel<KIND, BPL, RW>), dim3((p.d_out + 4 * RW - 1) / (4 * RW)), dim3(256), lds, s, p.x, p.w, p.scales, p.x_stride, p.d_out, p.d_in,
                     p.n_cols, p);
  return hipGetLastError();
}

hipError_t pa_launch_gemm_dot(const GemmParams& p, hipStream_t s) {
  if (p.d_out == 0 || p.d_in == 0 || (p.d_in & 31) || p.d_in > 8192 || p.n_cols == 0 || p.n_cols > DOT_COLS) return hipErrorInvalidValue;
  if (p.d_in <= 4096) return p.kind == PA_W_Q4_0 ? dot_launch<PA_W_Q4_0, 2, 2>(p, s) : dot_launch<PA_W_Q8_0, 2, 2>(p, s);
  return p.kind == PA_W_Q4_0 ? dot_launch<PA_W_Q4_0, 4, 1>(p, s) : dot_launch<PA_W_Q8_0, 4, 1>(p, s);
}

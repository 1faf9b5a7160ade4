// Column-batched projections for a few columns on gfx950 (verify blocks, the reference's 16-column prefill passes, short
// rests of a prompt): Y[c][r] = sum_k W[r][k] X[c][k] straight from the packed Q8_0 / Q4_0 planes on the matrix cores.
//
// The reference's counterpart is the batched cooperative matvec (engine/wgsl/coop.js).  Same operand precision as the
// GEMMs of proj_gemm.hip: every dequantised weight and every activation rounded to f16, products and sums f32.
//
// The work is one pass over the packed weights.  What bounds it: the latency of that one pass on small matrices, the
// activations every workgroup pulls from L2 on wide ones, the widening arithmetic (16 VALU instructions for 8 weights) on
// large ones.  Measured (cold weights; against dot products on the VALU, kept in proj_gemm_dot.hip for where they are ahead): Q4_0 9216 x 2048,
// 8 / 16 columns 8.9 / 14.8 -> 7.3 / 8.3 us; 2048 x 4096 7.2 / 14.8 -> 6.1 / 7.1; 14336 x 5120 101 / 170 -> 15.3 / 17.3; 5120 x 6144
// 38 / 79 -> 10.0 / 12.0; Q8_0 4096 x 2048 6.3 / 8.3 -> 4.9 / 5.5.
//   * a workgroup is 16 RG weight rows; K is cut into chunks of CH = 8 or 16 quantisation blocks, one per wave, so every
//     weight byte the workgroup needs is requested in its first instructions and nothing is loaded twice;
//   * a wave's packed weights (16 rows x 128 to 512 bytes) go to LDS by LDS-direct loads that cover whole cache lines; the
//     XOR swizzle that keeps the fragment reads off each other's banks is applied on the global side.  A lane then reads
//     8 bytes a k-step (one quantisation block): the fragment of v_mfma_f32_16x16x32_f16 takes elements 8 kg .. + 7 of the
//     block, which in a Q4_0 block are the low (kg < 2) or high nibbles of 8 consecutive bytes;
//   * the activations of a k-step are 16 contiguous bytes a lane, straight from L2 into the registers the MFMA reads;
//   * the waves' partial tiles meet in LDS and are added up in wave order: deterministic, no partial sums in memory.
#include "pf_common.h"
#include <algorithm>
typedef unsigned int u2 __attribute__((ext_vector_type(2)));

static __device__ inline h2 sk_as_h2(uint32_t u) { h2 r; __builtin_memcpy(&r, &u, 4); return r; }
static __device__ inline h2 sk_bytes(uint32_t w, uint32_t sel, h2 bias, h2 sc) { return (sk_as_h2(__builtin_amdgcn_perm(0x64646464u, w, sel)) - bias) * sc; }


// A fragment (8 weights) of a k-step from the lane's 8 packed bytes
template <int KIND>
static __device__ inline h8 sk_frag(const u2 q, uint32_t nib, h2 sc) {
  h2 o[4];
  if constexpr (KIND == PA_W_Q4_0) {
    const h2 bias = { (_Float16)1032.f, (_Float16)1032.f };            // 0x6400 | n = 1024 + n; n - 8
    const uint32_t a = (q[0] >> nib) & 0x0F0F0F0Fu, b = (q[1] >> nib) & 0x0F0F0F0Fu;
    o[0] = sk_bytes(a, 0x04010400u, bias, sc); o[1] = sk_bytes(a, 0x04030402u, bias, sc);
    o[2] = sk_bytes(b, 0x04010400u, bias, sc); o[3] = sk_bytes(b, 0x04030402u, bias, sc);
  } else {
    const h2 bias = { (_Float16)1152.f, (_Float16)1152.f };            // 0x6400 | (v + 128) = 1152 + v
    const uint32_t a = q[0] ^ 0x80808080u, b = q[1] ^ 0x80808080u;
    o[0] = sk_bytes(a, 0x04010400u, bias, sc); o[1] = sk_bytes(a, 0x04030402u, bias, sc);
    o[2] = sk_bytes(b, 0x04010400u, bias, sc); o[3] = sk_bytes(b, 0x04030402u, bias, sc);
  }
  return (h8){ o[0][0], o[0][1], o[1][0], o[1][1], o[2][0], o[2][1], o[3][0], o[3][1] };
}

#define SK_MAXW 16       // waves of a workgroup

// RG: 16-row groups of a workgroup; NB: 16-column blocks; CH: quantisation blocks (k-steps) of a wave's chunk; WHOLE: d_in is a
// multiple of 32 CH (every chunk whole and its scales on 16 bytes).  Otherwise the last wave's chunk ends with the row: it begins inside
// the chunk before it, and the blocks they share get scale 0 (fewer blocks than a chunk: its tail past the row's end does).
template <int KIND, int RG, int NB, int CH, bool WHOLE>
__global__ __launch_bounds__(SK_MAXW * 64)
void pa_gemm_skinny_kernel(const void* a_w, const uint16_t* a_scales, const uint16_t* a_x, uint32_t a_x_stride, uint32_t a_d_out, uint32_t a_d_in, uint32_t a_n_cols,
                           GemmParams p_in) {
  // (the leading arguments repeat fields of p_in: they are preloaded into scalar registers, so the loads below need no
  // scalar-load round trip; the other arguments are fetched in one batch behind them)
  GemmParams p = p_in;
  p.x = a_x; p.w = a_w; p.scales = a_scales; p.x_stride = a_x_stride; p.d_out = a_d_out; p.d_in = a_d_in; p.n_cols = a_n_cols;
  constexpr uint32_t BB = KIND == PA_W_Q4_0 ? 16 : 32;                 // bytes of a packed block
  constexpr uint32_t RB = CH * BB;                                  // bytes of a row's chunk
  constexpr uint32_t SPR = RB / 16, RPL = 64 / SPR;                    // 16-byte slots of a row's chunk, rows of a load
  // slot of 16-byte piece c of row r: c ^ swz(r) -- any 16 rows' pieces c then sit in 16 different 16-byte bank groups
  auto swz = [](uint32_t r) __attribute__((always_inline)) -> uint32_t { return SPR >= 16 ? r & 15 : (r >> 1) & (SPR - 1); };
  constexpr int NLD = 16 / RPL;                                        // loads of a 16-row group
  // k-steps of activations in flight (16 halve the waves a CU holds: 5120 x 6144, 2 columns 9.7 -> 11.3 us)
  constexpr int XD = NB == 1 && RG < 4 ? 8 : 4;
  extern __shared__ __attribute__((aligned(1024))) unsigned char sk_lds[];   // [wave][RG][16][RB]; at the end [wave][RG NB][4][64] floats
  const uint32_t tid = threadIdx.x, lane = tid & 63, ln = lane & 15, kg = lane >> 4, nw = blockDim.x >> 6;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t nb = p.d_in / 32, first = wave * CH;               // the first block that the wave counts
  const uint32_t b0 = WHOLE ? first : nb < CH ? 0u : min(first, nb - CH);   // ... and that it loads
  const uint32_t r0 = blockIdx.x * (16 * RG);
  unsigned char* stage = sk_lds + (size_t)wave * (RG * 16 * RB);
#pragma unroll
  for (int r = 0; r < RG; r++)
#pragma unroll
    for (int i = 0; i < NLD; i++) {
      const uint32_t rl = i * RPL + lane / SPR, piece = (lane % SPR) ^ swz(rl);
      const size_t row = min(r0 + 16 * r + rl, p.d_out - 1);           // rows past the end repeat the last one (not stored)
      const uint32_t off = WHOLE ? b0 * BB + piece * 16 : min(b0 * BB + piece * 16, nb * BB - 16);    // past the row's end (rows of less than a chunk): its last piece, weighted 0
      PF_GLL((const unsigned char*)p.w + row * nb * BB + off, stage + (r * NLD + i) * 1024);
    }
  u4 sc4[RG][CH / 8];                                                     // the 16 scales of the lane's row(s), f16
#pragma unroll
  for (int r = 0; r < RG; r++) {
    const uint16_t* src = p.scales + (size_t)min(r0 + 16 * r + ln, p.d_out - 1) * nb;
    if constexpr (WHOLE) {
#pragma unroll
      for (int k = 0; k < CH / 8; k++) sc4[r][k] = *(const u4*)(src + b0 + 8 * k);
    } else {
      // 8 scales a 16-byte load here too, from any even address (vector loads take unaligned dwords); a load each cost 2 - 5 us a round
      // of the chip (1 column: Q8_0 9488 x 7456 32.0 -> 26.8 us, 4906 x 4864 13.2 -> 9.9, Q4_0 8624 x 7232 30.8 -> 20.4)
      uint16_t t[CH];
      if (CH == 16 || nb >= CH) __builtin_memcpy(t, src + b0, 2 * CH);     // (chunks of 16: d_in is past 4096)
      else {
#pragma unroll
        for (int k = 0; k < CH; k++) t[k] = src[min((uint32_t)k, nb - 1)];
      }
#pragma unroll
      for (int k = 0; k < CH; k++) if ((uint32_t)k < first - b0 || (CH == 8 && (uint32_t)k >= nb - b0)) t[k] = 0;
      __builtin_memcpy(sc4[r], t, 2 * CH);
    }
  }
  const unsigned char* xsrc[NB];
#pragma unroll
  for (int c = 0; c < NB; c++) xsrc[c] = (const unsigned char*)(p.x + (size_t)min(16 * c + ln, p.n_cols - 1) * p.x_stride) + kg * 16;
  u4 xr[XD][NB];
  auto load_x = [&](int t) __attribute__((always_inline)) {
    const uint32_t b = WHOLE ? b0 + t : min(b0 + t, nb - 1);
#pragma unroll
    for (int c = 0; c < NB; c++) xr[t % XD][c] = *(const u4*)(xsrc[c] + (size_t)b * 64);
  };
#pragma unroll
  for (int t = 0; t < XD; t++) load_x(t);
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" :: "s"(p.y), "s"(p.y_stride), "s"(p.acc));
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                     // the LDS-direct loads are not the compiler's to wait for
  f4 acc[RG][NB];
#pragma unroll
  for (int r = 0; r < RG; r++)
#pragma unroll
    for (int c = 0; c < NB; c++) acc[r][c] = (f4){0.f, 0.f, 0.f, 0.f};
  const uint32_t nib = (kg >> 1) * 4;
#pragma unroll
  for (int t = 0; t < CH; t++) {
    h8 a[RG];
#pragma unroll
    for (int r = 0; r < RG; r++) {
      const uint32_t piece = KIND == PA_W_Q4_0 ? (uint32_t)t : 2u * t + (kg >> 1);
      const u2 q = *(const u2*)(stage + r * 16 * RB + ln * RB + (piece ^ swz(ln)) * 16 + (kg & 1) * 8);
      const uint32_t w = sc4[r][t / 8][(t / 2) % 4], s = t & 1 ? w >> 16 : w & 0xffffu;
      a[r] = sk_frag<KIND>(q, nib, sk_as_h2(s | s << 16));
    }
#pragma unroll
    for (int c = 0; c < NB; c++) {
      h8 b; __builtin_memcpy(&b, &xr[t % XD][c], 16);
#pragma unroll
      for (int r = 0; r < RG; r++) acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[r], b, acc[r][c], 0, 0, 0);
    }
    if (t + XD < CH) load_x(t + XD);
  }
  // accumulator i of a tile: row 4 kg + i, column ln
  __syncthreads();                                                     // the staged weights are dead
  float* red = (float*)sk_lds;
#pragma unroll
  for (int r = 0; r < RG; r++)
#pragma unroll
    for (int c = 0; c < NB; c++)
#pragma unroll
      for (int i = 0; i < 4; i++) red[((wave * (RG * NB) + r * NB + c) * 4 + i) * 64 + lane] = acc[r][c][i];
  __syncthreads();
  // 16 consecutive rows of a column on 16 consecutive threads
  for (uint32_t e = tid; e < RG * NB * 256; e += nw * 64) {
    const uint32_t tl = e >> 8, lr = e & 15, lc = (e >> 4) & 15;
    const uint32_t row = r0 + tl / NB * 16 + lr, col = tl % NB * 16 + lc;
    if (row >= p.d_out || col >= p.n_cols) continue;
    float* y = p.y + (size_t)col * p.y_stride + row;
    const float yo = p.acc ? *y : 0.f;
    // four waves' values a turn, read together (a turn past the last wave re-reads it and counts it 0 times)
    float s = 0.f;
    for (uint32_t w0 = 0; w0 < nw; w0 += 4) {
      float v[4];
#pragma unroll
      for (uint32_t k = 0; k < 4; k++) v[k] = red[((min(w0 + k, nw - 1) * (RG * NB) + tl) * 4 + (lr & 3)) * 64 + (lr >> 2) * 16 + lc];
#pragma unroll
      for (uint32_t k = 0; k < 4; k++) s += w0 + k < nw ? v[k] : 0.f;
    }
    *y = p.acc ? yo + s : s;
  }
}

template <int KIND, int RG, int NB, int CH, bool WHOLE>
static hipError_t sk_launch(const GemmParams& p, hipStream_t s) {
  const uint32_t nw = (p.d_in / 32 + CH - 1) / CH;
  const uint32_t stage = RG * 16 * CH * (KIND == PA_W_Q4_0 ? 16 : 32), red = RG * NB * 1024;
  const size_t lds = (size_t)nw * (stage > red ? stage : red);
  if (nw > SK_MAXW || lds > 160 * 1024) return hipErrorNotSupported;
  if (lds > 65536) {
    static PaPerDevice lds_set;
    const hipError_t e = pa_lds_limit(lds_set, (const void*)pa_gemm_skinny_kernel<KIND, RG, NB, CH, WHOLE>, 160 * 1024);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((pa_gemm_skinny_kernel<KIND, RG, NB, CH, WHOLE>), dim3((p.d_out + 16 * RG - 1) / (16 * RG)), dim3(nw * 64), lds, s, p.w, p.scales, p.x, p.x_stride,
                     p.d_out, p.d_in, p.n_cols, p);
  return hipGetLastError();
}
template <int KIND, int RG, int CH>
static hipError_t sk_cols(const GemmParams& p, hipStream_t s) {
  if (p.d_in % (32 * CH) == 0) return p.n_cols <= 16 ? sk_launch<KIND, RG, 1, CH, true>(p, s) : sk_launch<KIND, RG, 2, CH, true>(p, s);
  return p.n_cols <= 16 ? sk_launch<KIND, RG, 1, CH, false>(p, s) : sk_launch<KIND, RG, 2, CH, false>(p, s);
}
// 16-row groups a workgroup.  Every workgroup reads all activations through its CU's L1 (n_cols x d_in x 2 bytes: 64 KB for
// 16 columns of 2048), so once there are more row groups than CUs larger workgroups cut that traffic; below that, and for
// few columns, they only leave CUs idle.  Measured (us, 1 / 2 / 4 groups): 9216 x 2048 Q4_0 2 columns 6.3 / 6.8 / 7.4, 8
// columns 7.3 / 7.4 / 7.6, 16 columns 9.2 / 9.0 / 8.3, 32 columns 14.7 / 12.7 / 10.6; 2048 x 4096 16 columns 7.1 / 8.5 / 11.2;
// 14336 x 5120 8 columns 18.0 / 15.3 / 15.7, 16 columns 25.1 / 18.6 / 17.3; 5120 x 6144 16 columns 16.4 / 12.0 / -.
static int sk_row_groups(uint32_t d_out, uint32_t d_in, uint32_t n_cols, int n_cu) {
  const uint32_t groups = (d_out + 15) / 16, cus = n_cu > 0 ? (uint32_t)n_cu : 256u;
  if (groups <= cus) return 1;
  if (n_cols <= 8) return d_in > 4096 ? 2 : 1;
  return groups >= 2 * cus ? 4 : 2;
}
// chunks of 8 blocks (twice the waves) while 16 waves cover d_in
static int sk_chunk(uint32_t d_in) { return d_in <= 4096 ? 8 : 16; }
// ... as many of them as the staged weights of a workgroup leave room for in its LDS
extern "C" int pa_rule_gemm_few_groups(int kind, uint32_t d_out, uint32_t d_in, uint32_t n_cols, int n_cu) {
  const int ch = sk_chunk(d_in);
  int rg = sk_row_groups(d_out, d_in, n_cols, n_cu);
  const uint32_t bytes = (d_in / 32 + ch - 1) / ch * ch * 16 * (kind == PA_W_Q4_0 ? 16 : 32);
  while (rg > 1 && rg * bytes > 160 * 1024) rg /= 2;
  return rg;
}
// Whether one to four columns over long rows go to the dot-product kernel (proj_gemm_dot.hip) instead.  This kernel costs whole rounds of
// the workgroups that the CUs' LDS and waves hold, the other follows rows x columns; both estimates in us were fitted to 604 measured
// calls (50 sizes of each kind, 1 to 6 columns, cold weights) and are within 6 % of most.  Always this kernel there: up to 1.65 times the other's time
// (Q8_0 885 x 6240), Q8_0 5120 x 6144 1 / 2 columns 13.7 / 14.2 us against 10.3 / 11.4; by the rule 0.3 % behind the better one on average,
// 17 % at worst.  Up to 2048 inputs the other kernel was never ahead; past two columns of more than 2048 rows by 10 % at most, past four by 15 %.
extern "C" int pa_rule_gemm_few_dot(int kind, uint32_t d_out, uint32_t d_in, uint32_t n_cols, int n_cu) {
  if (d_in <= 2048 || n_cols > 4 || (n_cols > 2 && d_out > 2048)) return 0;
  const bool q4 = kind == PA_W_Q4_0, longer = d_in > 4096;
  const uint32_t cus = n_cu > 0 ? (uint32_t)n_cu : 256u, ch = sk_chunk(d_in), nw = (d_in / 32 + ch - 1) / ch, rg = pa_rule_gemm_few_groups(kind, d_out, d_in, n_cols, n_cu);
  const uint32_t lds = nw * rg * std::max(16 * ch * (q4 ? 16u : 32u), 1024u), wgs = (d_out + 16 * rg - 1) / (16 * rg);
  const uint32_t held = std::max(1u, std::min(160u * 1024 / lds, 32u / nw)), rounds = (wgs + cus * held - 1) / (cus * held);
  const float mb = 1e-6f * d_out * d_in * (q4 ? 0.5625f : 1.0625f), rows = 1e-3f * d_out, n = (float)n_cols;
  const float dot = longer ? 3.25f + 0.41f * n + (0.44f + 0.27f * n) * rows + 0.091f * mb : 3.5f + 0.23f * n + (0.34f + 0.05f * n) * rows + 0.086f * mb;
  // start, a round, a round of ragged rows on top, a MB of weights, 100 KB of LDS a workgroup
  static const float cost[2][2][5] = { { { 1.8f, 0.f, 0.42f, 0.19f, 3.6f }, { 0.f, 3.8f, 0.64f, 0.13f, 1.9f } },          // Q8_0: up to 4096 inputs, longer
                                       { { 1.4f, 0.73f, 0.68f, 0.234f, 4.9f }, { 0.f, 2.9f, 0.97f, 0.206f, 3.2f } } };    // Q4_0
  const float* c = cost[q4][longer];
  return dot < c[0] + (c[1] + (d_in % (32 * ch) ? c[2] : 0.f)) * rounds + c[3] * mb + c[4] * 1e-5f * lds;
}
template <int KIND>
static hipError_t sk_shape(const GemmParams& p, int n_cu, hipStream_t s) {
  const int rg = pa_rule_gemm_few_groups(KIND, p.d_out, p.d_in, p.n_cols, n_cu);
  if (sk_chunk(p.d_in) == 16) return rg == 1 ? sk_cols<KIND, 1, 16>(p, s) : rg == 2 ? sk_cols<KIND, 2, 16>(p, s) : sk_cols<KIND, 4, 16>(p, s);
  return rg == 1 ? sk_cols<KIND, 1, 8>(p, s) : rg == 2 ? sk_cols<KIND, 2, 8>(p, s) : sk_cols<KIND, 4, 8>(p, s);
}

// Up to 16 columns, and up to 32 where that beats the mid-size kernel of proj_gemm_wide.hip (us at 32 columns, here / there:
// 9216 x 2048 10.6 / 13.4, 2048 x 4096 10.6 / 16.9, 14336 x 5120 21.9 / 30.7, 5120 x 6144 17.9 / 25.4, 4096 x 2048 6.5 / 9.8; with
// Q8_0 weights past 4096 inputs a workgroup's LDS holds too few rows: 14336 x 5120 36.4 / 30.7).
bool pa_gemm_skinny_serves(const GemmParams& p) {
  if (p.kind == PA_W_F32 || p.d_in > 8192 || (p.x_stride & 7) != 0 || ((uintptr_t)p.x & 15) != 0) return false;
  return p.n_cols <= 16 || (p.n_cols <= 32 && (p.kind == PA_W_Q4_0 || p.d_in <= 4096));
}
hipError_t pa_launch_gemm_skinny(const GemmParams& p, int n_cu, hipStream_t s) {
  if (p.d_out == 0 || p.d_in == 0 || (p.d_in & 31) || p.n_cols == 0) return hipErrorInvalidValue;
  if (pa_rule_gemm_few_dot(p.kind, p.d_out, p.d_in, p.n_cols, n_cu)) return pa_launch_gemm_dot(p, s);
  return p.kind == PA_W_Q4_0 ? sk_shape<PA_W_Q4_0>(p, n_cu, s) : sk_shape<PA_W_Q8_0>(p, n_cu, s);
}

// Column-batched projections for wide chunks on gfx950: Y[c][r] = sum_k W[r][k] X[c][k] over two f16 operands, the weights
// widened once into matrix-core fragment order (proj_gemm_wide.hip, which also says when this kernel is taken).
//
// Work decomposition
//   * a workgroup is eight wavefronts, two a SIMD, on a tile of BM columns x BN weight rows; WM x WN waves share the tile, and
//     where that would leave a wave too little to do, KG groups of waves split every stage's k-steps between them and
//     their copies of the tile meet in LDS at the end, added up in group order (no partial sums in memory);
//   * both operands go to LDS by LDS-direct loads (no staging registers): K in stages of 32 KG, S buffers, so S - 1 stages
//     are in flight.  Activation rows are staged with the 16-byte chunk order XORed by the row (conflict-free
//     ds_read_b128 fragments: SQ_LDS_BANK_CONFLICT = 0), the weights as the 1 KB fragments they are kept in;
//   * one barrier a stage, in the MIDDLE of its products: a stage is two k-steps a wave; the fragments of the next k-step are
//     read, and the stage's loads issued, one at a time between the MFMAs, so that behind the barrier a wave's next MFMA
//     has its operands.  (All reads and loads in front of the MFMAs: 8 % slower; the order left to the compiler: every
//     k-step waits out its own LDS reads.)
//   * a tile shape is picked per call, by the rule at pa_pick_tile.
//
// What bounds it: on full rounds of the chip the MFMA rate the power limit allows and the rounds' own ends (4096 columns:
// 14336 x 5120 1090 - 1130 TFLOP/s, 9216 x 2048 1000); on one round or less the LDS-direct loads' latency (a tile's 96 - 120 KB
// in flight a CU).  Measured against the kernel it replaced (128 columns x 256 / 384 / 512 rows, four waves, weight fragments
// from memory straight to registers) and the 64 x 64 kernel, Q8_0, five weights in rotation: 777 columns of 5120 x 6144 100 -> 64 us, of
// 14336 x 5120 143 -> 133, of 9216 x 2048 59 -> 36; 2048 columns of 2048 x 4096 76 -> 40; 512 of 14336 x 5120 141 -> 92, of 4096 x 2048
// 16.8 -> 15.0; 4096 of 9216 x 2048 161 -> 154, of 14336 x 5120 609 -> 568.  Not kept: a ninth wave that prefetches the weight stream into L2 (slower on every shape), activation
// rows at a padded stride (no change).
#include "pf_common.h"

struct GemmTileParams {
  const uint16_t* x; const uint16_t* w16; float* y;
  uint32_t x_stride, y_stride, d_out, d_in, n_cols;
};

template <int WM, int WN, int KG, int TM, int TN, int S, bool ACC>
__global__ __launch_bounds__(512, 2) void pa_gemm_tile_kernel(GemmTileParams p) {
  static_assert(WM * WN * KG == 8, "eight waves");
  constexpr int KS = 2;                                  // k-steps of a stage per wave
  constexpr int BM = WM * TM * 32, BN = WN * TN * 32, BK = 16 * KG * KS;
  constexpr int CH = BK / 8;                             // 16-byte chunks of a staged activation row
  constexpr int RPL = 64 / CH;                           // rows of a 1 KB load
  constexpr int ALD = BM * BK / 512, BLD = BN * BK / 512, LPW = (ALD + BLD + 7) / 8;
  constexpr int ABYTES = BM * BK * 2, STAGE = (BM + BN) * BK * 2;
  extern __shared__ __attribute__((aligned(1024))) unsigned char gt_lds[];
  const uint32_t tid = threadIdx.x, lane = tid & 63, fl = lane & 31, fk = lane >> 5;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t kgrp = wave / (WM * WN), wm = wave % (WM * WN) % WM, wn = wave % (WM * WN) / WM;
  const uint32_t n_cb = (p.n_cols + BM - 1) / BM, n_rb = (p.d_out + BN - 1) / BN, total = n_cb * n_rb;
  const uint32_t per = (total + 7) / 8, tile = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (tile >= total || blockIdx.x / 8 >= per) return;
  uint32_t cb = tile % n_cb, rb_ = tile / n_cb;
  if (n_cb % 8 == 0) {
    const uint32_t panel = tile / (4 * n_cb), r = tile % (4 * n_cb), h = min(4u, n_rb - panel * 4);
    cb = r / (8 * h) * 8 + r % 8; rb_ = panel * 4 + r % (8 * h) / 8;
  }
  const uint32_t c0 = cb * BM, r0 = rb_ * BN;
  const uint32_t n_stages = p.d_in / BK, n_rb32 = (p.d_out + 31) / 32;
  auto swz = [](uint32_t r) __attribute__((always_inline)) -> uint32_t { return BK >= 128 ? r & 15 : BK == 64 ? (r >> 1) & 7 : (r >> 2) & 3; };

  const unsigned char* xb = (const unsigned char*)(p.x + (size_t)c0 * p.x_stride);
  // load q of a stage fills the q-th KB of its buffer: ALD pieces of activations, then BLD weight fragments.  Wave w takes
  // q = w, w + 8, ...; where they do not come out even, the last ones repeat a piece (the same bytes twice)
  const unsigned char* src[LPW];
  uint32_t step[LPW], off[LPW], dofs[LPW];
#pragma unroll
  for (int i = 0; i < LPW; i++) {
    uint32_t q = i * 8 + wave;
    if (q >= ALD + BLD) q -= 8;
    dofs[i] = q * 1024;
    if (q < ALD) {
      const uint32_t row = q * RPL + lane / CH;
      src[i] = xb; step[i] = BK * 2;
      off[i] = min(row, p.n_cols - 1 - c0) * (p.x_stride * 2) + ((lane % CH) ^ swz(row)) * 16;
    } else {
      const uint32_t f = q - ALD, rb = min(r0 / 32 + f / (BK / 16), n_rb32 - 1), kb = f % (BK / 16);
      src[i] = (const unsigned char*)p.w16 + ((size_t)kb * n_rb32 + rb) * 1024; step[i] = n_rb32 * (BK * 64);
      off[i] = lane * 16;
    }
  }
  auto issue = [&](uint32_t st, uint32_t buf) __attribute__((always_inline)) {
    const uint32_t s = min(st, n_stages - 1);
#pragma unroll
    for (int i = 0; i < LPW; i++) PF_GLL_S(src[i] + (size_t)s * step[i], off[i], gt_lds + buf * STAGE + dofs[i]);
  };
  auto col_of = [&](int a, int i) { return c0 + (wm * TM + a) * 32 + 8 * (i / 4) + 4 * fk + (i % 4); };
  auto row_of = [&](int b) { return r0 + (wn * TN + b) * 32 + fl; };

  f16v acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; a++)
#pragma unroll
    for (int b = 0; b < TN; b++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[a][b][i] = 0.f;

#pragma unroll
  for (int j = 0; j < S; j++) issue(j, j);
  // fragment addresses
  uint32_t a_rd[TM];
#pragma unroll
  for (int t = 0; t < TM; t++) { const uint32_t row = (wm * TM + t) * 32 + fl; a_rd[t] = row * (BK * 2) + (((2 * kgrp + fk) ^ swz(row)) * 16); }
  const uint32_t b_rd = ABYTES + (wn * TN * (BK / 16) + kgrp) * 1024 + lane * 16;
  struct Frag { h8 a[TM], b[TN]; };
  auto rd = [&](Frag& f, const unsigned char* sb, int ks) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < TM; t++) f.a[t] = *(const h8*)(sb + (a_rd[t] ^ (2 * KG * ks * 16)));
#pragma unroll
    for (int t = 0; t < TN; t++) f.b[t] = *(const h8*)(sb + b_rd + (t * (BK / 16) + KG * ks) * 1024);
  };
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(LPW * (S - 1)) : "memory");       // stage 0 (S stages were issued)
  asm volatile("s_barrier" ::: "memory");
  Frag f0, f1;
  rd(f0, gt_lds, 0);
  uint32_t buf = 0;
  auto mma1 = [&](const Frag& f, int m) __attribute__((always_inline)) {
    acc[m % TM][m / TM] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[m % TM], f.b[m / TM], acc[m % TM][m / TM], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr int NM = TM * TN;
  for (uint32_t st = 0; st < n_stages; st++) {
    const uint32_t nbuf = buf + 1 == S ? 0 : buf + 1;
    __builtin_amdgcn_sched_barrier(0);
    mma1(f0, 0);
    rd(f1, gt_lds + buf * STAGE, 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 1; m < NM; m++) mma1(f0, m);
    // stage st + 1 is in LDS behind this barrier, and every wave has read stage st: its buffer takes stage st + S
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(LPW * (S - 2)) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    mma1(f1, 0);
    rd(f0, gt_lds + nbuf * STAGE, 0);
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t s_n = min(st + S, n_stages - 1);
#pragma unroll
    for (int m = 1; m < NM; m++) {
      mma1(f1, m);
#pragma unroll
      for (int i = 0; i < LPW; i++)
        if (i % (NM - 1) == m - 1) PF_GLL_S(src[i] + (size_t)s_n * step[i], off[i], gt_lds + buf * STAGE + dofs[i]);
      __builtin_amdgcn_sched_barrier(0);
    }
    buf = nbuf;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                       // (the stages past the end, never read)
  // accumulator i of a tile: column 8 (i / 4) + 4 fk + i % 4, row fl.  Accumulating calls: loads and stores share one counter,
  // and a wait for a loaded value with stores pending waits for those as well, so the old values are fetched several
  // tiles at a time, unconditionally (clamped addresses: a guarded load is a branch, one load a basic block), then added.
  if constexpr (KG == 1) {
    constexpr int D = TN <= 5 ? TN : 4;                                  // tiles of a phase: what fits next to the accumulators
#pragma unroll
    for (int m0 = 0; m0 < NM; m0 += D) {
      float old[D][16];
      if constexpr (ACC) {
#pragma unroll
        for (int m = 0; m < D && m0 + m < NM; m++)
#pragma unroll
          for (int i = 0; i < 16; i++) old[m][i] = p.y[(size_t)min(col_of((m0 + m) / TN, i), p.n_cols - 1) * p.y_stride + min(row_of((m0 + m) % TN), p.d_out - 1)];
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int m = 0; m < D && m0 + m < NM; m++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const int a = (m0 + m) / TN, b = (m0 + m) % TN;
          if (row_of(b) < p.d_out && col_of(a, i) < p.n_cols) p.y[(size_t)col_of(a, i) * p.y_stride + row_of(b)] = ACC ? old[m][i] + acc[a][b][i] : acc[a][b][i];
        }
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
    constexpr int NT = TM * TN, SPW = NT * 16 / KG;
    const uint32_t wt = wave % (WM * WN);
    auto col_s = [&](int k) { const uint32_t sl = kgrp * SPW + k; return c0 + (wm * TM + sl / (16 * TN)) * 32 + 8 * (sl % 16 / 4) + 4 * fk + (sl % 4); };
    auto row_s = [&](int k) { const uint32_t sl = kgrp * SPW + k; return r0 + (wn * TN + sl / 16 % TN) * 32 + fl; };
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    float* red = (float*)gt_lds;
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++)
#pragma unroll
        for (int i = 0; i < 16; i++) red[((wave * NT + a * TN + b) * 16 + i) * 64 + lane] = acc[a][b][i];
    float old[SPW];
    if constexpr (ACC) {
#pragma unroll
      for (int k = 0; k < SPW; k++) old[k] = p.y[(size_t)min(col_s(k), p.n_cols - 1) * p.y_stride + min(row_s(k), p.d_out - 1)];
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int k = 0; k < SPW; k++) {
      float s = 0.f;
#pragma unroll
      for (int g = 0; g < KG; g++) s += red[((g * (WM * WN) + wt) * NT * 16 + kgrp * SPW + k) * 64 + lane];
      if (row_s(k) < p.d_out && col_s(k) < p.n_cols) p.y[(size_t)col_s(k) * p.y_stride + row_s(k)] = ACC ? old[k] + s : s;
    }
  }
}

template <int WM, int WN, int KG, int TM, int TN, int S>
static hipError_t gt_launch(const GemmTileParams& q, int acc, hipStream_t s) {
  constexpr int BM = WM * TM * 32, BN = WN * TN * 32, BK = 32 * KG;
  constexpr int lds_st = S * (BM + BN) * BK * 2, lds_red = KG > 1 ? KG * BM * BN * 4 : 0, lds = lds_st > lds_red ? lds_st : lds_red;
  static_assert(lds <= 160 * 1024, "LDS");
  const uint32_t total = ((q.n_cols + BM - 1) / BM) * ((q.d_out + BN - 1) / BN);
  static PaPerDevice lds_set[2];
  const auto kernel = acc ? pa_gemm_tile_kernel<WM, WN, KG, TM, TN, S, true> : pa_gemm_tile_kernel<WM, WN, KG, TM, TN, S, false>;
  const hipError_t e = pa_lds_limit(lds_set[acc ? 1 : 0], (const void*)kernel, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3((total + 7) / 8 * 8), dim3(512), lds, s, q);
  return hipGetLastError();
}

// The tile shapes, with what a round of the chip costs: ns per k of d_in (measured on rounds of 200 - 256 workgroups) on top
// of about 6 us for a round's first loads and last stores.
struct TileShape { uint16_t bm, bn; float ns_k; hipError_t (*launch)(const GemmTileParams&, int, hipStream_t); };
static const TileShape tile_shapes[] = {
  { 64, 128, 6.5f, gt_launch<1, 2, 4, 2, 2, 3> },
  { 128, 128, 10.3f, gt_launch<2, 2, 2, 2, 2, 4> },
  { 128, 160, 11.8f, gt_launch<4, 1, 2, 1, 5, 4> },
  { 128, 192, 14.0f, gt_launch<4, 2, 1, 1, 3, 6> },
  { 128, 256, 15.5f, gt_launch<2, 4, 1, 2, 2, 6> },
  { 128, 320, 19.0f, gt_launch<4, 2, 1, 1, 5, 5> },
  { 128, 384, 21.5f, gt_launch<2, 4, 1, 2, 3, 4> },
  { 128, 448, 25.0f, gt_launch<4, 2, 1, 1, 7, 4> },
  { 256, 256, 27.0f, gt_launch<2, 4, 1, 4, 2, 4> },
};

// One workgroup is resident per CU, so a call costs whole rounds of n_cu workgroups: the shape with the cheapest rounds, and
// its estimate in us.  Larger tiles pay less traffic per product but are coarser: which one wins changes with every
// multiple of a tile edge (777 columns of 5120 x 6144: 128 x 160, 224 workgroups, 63 us; 128 x 128, 280 workgroups, 87 us).  Of
// 104 sizes measured on every tile and on the 64 x 64 kernel (8 weight shapes x 13 column counts, cold weights) the choice between
// all of them is the fastest at 84 and within 6 % at 8; it is 9 - 33 % behind at 12, most where one round of few workgroups (which
// costs less than a full one) is set against the 64 x 64 kernel: 9216 x 2048, 200 columns 27.9 us, on 128 x 128 21.1.
static int pa_pick_tile(uint32_t d_out, uint32_t d_in, uint32_t n_cols, int n_cu, float* us) {
  int best = 0;
  *us = 1e30f;
  for (int i = 0; i < (int)(sizeof tile_shapes / sizeof tile_shapes[0]); i++) {
    const TileShape& t = tile_shapes[i];
    const uint64_t wgs = (uint64_t)((n_cols + t.bm - 1) / t.bm) * ((d_out + t.bn - 1) / t.bn), cus = n_cu > 0 ? n_cu : 256;
    const float c = (float)((wgs + cus - 1) / cus) * (6.f + t.ns_k * 1e-3f * d_in);
    if (c < *us) { *us = c; best = i; }
  }
  return best;
}

float pa_gemm_tile_us(uint32_t d_out, uint32_t d_in, uint32_t n_cols, int n_cu, uint32_t* shape) {
  float us;
  const TileShape& t = tile_shapes[pa_pick_tile(d_out, d_in, n_cols, n_cu, &us)];
  *shape = (uint32_t)t.bm << 16 | t.bn;
  return us;
}

hipError_t pa_launch_gemm_tile(const GemmParams& p, const uint16_t* w16, int n_cu, hipStream_t s) {
  if (p.d_out == 0 || p.d_in == 0 || p.d_in % 128 != 0 || p.n_cols == 0 || p.x_stride > (1u << 22)) return hipErrorInvalidValue;   // (32-bit row offsets inside a tile)
  GemmTileParams q;
  q.x = p.x; q.w16 = w16; q.y = p.y; q.x_stride = p.x_stride; q.y_stride = p.y_stride; q.d_out = p.d_out; q.d_in = p.d_in; q.n_cols = p.n_cols;
  float us;
  return tile_shapes[pa_pick_tile(p.d_out, p.d_in, p.n_cols, n_cu, &us)].launch(q, p.acc, s);
}

// Column-batched projections for wide chunks on gfx950: Y[c][r] = sum_k W[r][k] X[c][k] over two f16 operands, the weights
// widened once into matrix-core fragment order (proj_gemm_wide.hip, which also says when this kernel is taken).
//
// Work decomposition
//   * a workgroup is eight wavefronts, two a SIMD, on a tile of BM columns x BN weight rows; WM x WN waves share the tile, and
//     where that would leave a wave too little to do, KG groups of waves split every stage's k-steps between them and
//     their copies of the tile meet in LDS at the end, added up in group order (no partial sums in memory);
//   * both operands go to LDS by LDS-direct loads (no staging registers): K in stages of 32 KG, S buffers, so S - 1 stages
//     are in flight.  Activation rows are staged with the 16-byte chunk order XORed by the row, the weights as the 1 KB fragments they
//     are kept in: fragments without bank conflicts where KG groups split K (SQ_LDS_BANK_CONFLICT = 0); the 16-row fragments of gt_whole_k have a swizzle of their
//     own (gt_swz64; under the other one 14 - 44 % of the LDS's active cycles were conflicts);
//   * one barrier a stage, in the MIDDLE of its products: a stage is two k-steps of 16 a wave, or, where a wave holds whole sums (KG = 1,
//     the shapes of the power-limited sizes), one of 32 on 16 x 16 x 32 products (gt_whole_k); the next fragments are
//     read, and the stage's loads issued, one at a time between the MFMAs, so that behind the barrier a wave's next MFMA
//     has its operands.  (All reads and loads in front of the MFMAs: 8 % slower; the order left to the compiler: every
//     k-step waits out its own LDS reads.)
//   * a tile shape is picked per call, by the rule at pa_pick_tile.
//
// What bounds it: on full rounds of the chip the MFMA rate the power limit allows and the rounds' own ends (4096 columns, on 32 x 32 x 16
// products: 14336 x 5120 1090 - 1130 TFLOP/s, 9216 x 2048 1000; the 16 x 16 x 32 ones are some 8 % faster there); on one round or less the LDS-direct loads' latency (a tile's 96 - 120 KB
// in flight a CU).  Measured against the kernel it replaced (128 columns x 256 / 384 / 512 rows, four waves, weight fragments
// from memory straight to registers) and the 64 x 64 kernel, Q8_0, five weights in rotation: 777 columns of 5120 x 6144 100 -> 64 us, of
// 14336 x 5120 143 -> 133, of 9216 x 2048 59 -> 36; 2048 columns of 2048 x 4096 76 -> 40; 512 of 14336 x 5120 141 -> 92, of 4096 x 2048
// 16.8 -> 15.0; 4096 of 9216 x 2048 161 -> 154, of 14336 x 5120 609 -> 568.  Not kept: a ninth wave that prefetches the weight stream into L2 (slower on every shape), activation
// rows at a padded stride (no change).
#include "pf_common.h"
#include "glue_math.h"
#include <algorithm>

struct GemmTileParams {
  const uint16_t* x; const uint16_t* w16; float* y;
  uint32_t x_stride, y_stride, d_out, d_in, n_cols;
};

// ---- the pre-step as the end of the [q | k | v] projection: whole heads in a workgroup's rows ----
// What the tile holds leaves as the pre-step would leave it (glue_kv.hip; the same arithmetic on the same f32 values, a head's sum of squares
// in f64 in another order: the same f32 factor but where that rounds the other way), and the f32 projections themselves are never stored: a launch less, and for 4096 columns of the gated 16 / 2-head
// shape 150 MB less written and as much less read.  It is LDS, VALU and store work behind a tile's products, with nothing to hide under, so it is dealt
// by what it is: columns on lanes for the sums of squares, rotation pairs on lanes for the rotation (both elements of a pair in one lane),
// the other dims a column at a time, everything read before the first store.  Layer pass, apart / so (us a layer, both on 32 x 32 x 16 products): 4096 columns
// of that shape 499 / 459, 2048 282 / 243, 300 71 / 66; 777 of the 24 / 4-head shape 292 / 280; 512 and 1024 of the 16 / 8-head shape 53 / 48 and 82 / 73.
enum { GT_STORE = 0, GT_ACC = 1, GT_HEADS = 2 };

#define GT_OLD 16                // old blocks of an accumulating call that a wave requests under its last products

// what a block of head_dim weight rows is: [q | gate] or q heads, then k, then v heads
enum { HB_Q = 0, HB_GATE = 1, HB_K = 2, HB_V = 3 };
static __device__ inline uint32_t head_block(const GlueParams& g, uint32_t b, uint32_t& h) {
  const uint32_t gated = g.flags & PA_FLAG_GATE ? 1 : 0, nq = g.n_heads << gated;
  if (b < nq) { h = b >> gated; return gated && (b & 1) ? HB_GATE : HB_Q; }
  h = b - nq;
  if (h < g.n_kv_heads) return HB_K;
  h -= g.n_kv_heads;
  return HB_V;
}

// four consecutive values of a finished k or v row (dims d0 ..; 8 lanes = 32 dims) to an f16 or int8 cache; every lane of the wave calls
static __device__ inline void cache_store4(const GlueParams& g, bool v, uint32_t h, uint32_t pos, uint32_t d0, const float (&x)[4], bool on) {
  const size_t row = (size_t)h * g.head_rows + pos;
  uint16_t* cache = v ? g.v_cache : g.k_cache;
  if (g.ks_cache) {
    uint32_t w; float sc;
    quant4_q8(x, w, sc);
    if (on) {
      *(uint32_t*)((unsigned char*)cache + row * g.head_dim + d0) = w;
      if (d0 % 32 == 0) (v ? g.vs_cache : g.ks_cache)[row * (g.head_dim / 32) + d0 / 32] = sc;
    }
  } else if (on) {
    *(h4*)((_Float16*)cache + row * g.head_dim + d0) = (h4){ (_Float16)x[0], (_Float16)x[1], (_Float16)x[2], (_Float16)x[3] };
  }
}

// LDS of it: CP columns x BN rows ([CP][BN + 4] f32), the slices' sums of squares, the heads' factors, the norm weights, then the (cos, sin)
// rows of the tile's BM columns where they fit.  Nothing is loaded from memory between the stores: loads and stores share one counter, and a
// wait for a loaded value with stores pending waits for those as well.
#define GT_LDS (160 * 1024)
template <int CP, int BN> struct HeadsLds {
  static constexpr int LR = BN + 4;
  static constexpr int part = CP * LR * 4, inv = part + 512 * 8, nw = inv + (BN / 128) * CP * 4, cs = nw + 2 * 256 * 4;
};
static __device__ __host__ inline bool cs_in_lds(uint32_t fixed, uint32_t bm, uint32_t half) { return fixed + bm * half * 8 <= GT_LDS; }

static __device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// requests the norm weights and the (cos, sin) rows of columns c0 .. c0 + BM; they are there behind the caller's wait and barrier
template <int CP, int BN, int BM>
static __device__ inline void heads_request(const GlueParams& g, unsigned char* lds, uint32_t c0) {
  typedef HeadsLds<CP, BN> H;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = g.n_rot / 2;
  if (g.flags & PA_FLAG_QK_NORM) ((float*)(lds + H::nw))[tid] = (tid < 256 ? g.qw : g.kw)[min(tid & 255, g.head_dim - 1)];
  if (cs_in_lds(H::cs, BM, half)) {
    const unsigned char* src = (const unsigned char*)(g.rope_tab + (size_t)(g.base_pos + c0) * half);
    const uint32_t last = (g.n_cols - c0) * half * 8 - 16;
    for (uint32_t q = wave; q * 1024 < BM * half * 8; q += 8) PF_GLL_S(src, min(q * 1024 + lane * 16, last), lds + H::cs + q * 1024);
  }
}

// global column of local column c: col_of(c); rows r0 ..  All 512 threads call, behind a barrier.
template <int HD, int CP, int BN, int BM, class ColOf>
static __device__ inline void finish_heads(const GlueParams& g, unsigned char* lds, uint32_t c0, uint32_t r0, uint32_t d_out, ColOf col_of) {
#pragma clang fp contract(off)
  typedef HeadsLds<CP, BN> H;
  constexpr int LR = H::LR, NS = 512 / CP, RS = BN / NS;               // slices a column, rows a slice
  constexpr int NHB = BN / HD, CPW = CP / 8;                           // heads of the tile, columns of a wave (consecutive ones)
  static_assert(RS % 16 == 0 && RS <= 128, "a slice is inside a head");
  const float* hx = (const float*)lds;
  double* part = (double*)(lds + H::part);                             // [NS][CP]
  float* inv = (float*)(lds + H::inv);                                 // [NHB][CP], a wave's columns its own
  uint32_t tid = threadIdx.x;
  asm volatile("" : "+v"(tid));                                        // (no lane's addresses are kept from phase to phase beside the accumulators)
  const uint32_t lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = g.n_rot / 2, lw = wave * CPW;
  const bool norm = (g.flags & PA_FLAG_QK_NORM) != 0, cs_lds = cs_in_lds(H::cs, BM, half);
  if (norm) {
    const uint32_t c = tid % CP, sl = tid / CP;
    uint32_t h;
    const uint32_t kind = head_block(g, (r0 + sl * RS) / HD, h);
    if (kind == HB_Q || kind == HB_K) {
      double ss[4] = { 0.0, 0.0, 0.0, 0.0 };
#pragma unroll
      for (int k = 0; k < RS; k += 4) {
        const f4 v = *(const f4*)(hx + c * LR + sl * RS + k);
#pragma unroll
        for (int i = 0; i < 4; i++) ss[i] = __builtin_fma((double)v[i], (double)v[i], ss[i]);
      }
      part[sl * CP + c] = (ss[0] + ss[1]) + (ss[2] + ss[3]);
    }
    lds_barrier();
    if (lane < NHB * CPW) {
      const uint32_t cc = lw + lane % CPW, hb = lane / CPW;
      double t[NS / NHB];
#pragma unroll
      for (int k = 0; k < NS / NHB; k++) t[k] = part[(hb * (NS / NHB) + k) * CP + cc];
      double s = t[0];
#pragma unroll
      for (int k = 1; k < NS / NHB; k++) s += t[k];
      inv[hb * CP + cc] = rms_inv(s, HD, g.eps);
    }
    wave_lds_fence();
  }
  const uint32_t qd = g.n_heads * HD;
  constexpr uint32_t Q4 = HD / 4, CPI = 64 / Q4, NI = CPW / CPI;       // quads of a head, columns an instruction, instructions
  const uint32_t cl = lane / Q4, d = 4 * (lane % Q4);
  for (int hb = 0; hb < NHB; hb++) {
    uint32_t h;
    const uint32_t row = r0 + hb * HD;
    if (row < d_out) {
    const uint32_t kind = head_block(g, row / HD, h);
    const float* hx0 = hx + hb * HD;
    const bool plain = kind == HB_GATE || kind == HB_V;
    const float* wp = (const float*)(lds + H::nw) + (kind == HB_Q ? 0 : 256);
    auto store4 = [&](uint32_t col, uint32_t dd, const float (&x)[4], bool on) __attribute__((always_inline)) {
      if (kind == HB_Q || kind == HB_GATE) { if (on) *(f4*)((kind == HB_Q ? g.q_out : g.gate_out) + (size_t)col * qd + h * HD + dd) = (f4){ x[0], x[1], x[2], x[3] }; }
      else cache_store4(g, kind == HB_V, h, g.base_pos + col, dd, x, on);
    };
    if (!plain) {
      // rotated dims: a lane holds elements da .. da + 3 and their partners
      const uint32_t U = half / 4, lgU = 31 - __builtin_clz(U), u = lane & (U - 1), da = 4 * u, db = da + half;
      f4 wa = { 1.f, 1.f, 1.f, 1.f }, wb = wa;
      if (norm) { wa = *(const f4*)(wp + da); wb = *(const f4*)(wp + db); }
      for (uint32_t e = lane; e < (CPW << lgU); e += 64) {
        const uint32_t c = lw + (e >> lgU), col = col_of(c);
        const bool on = col < g.n_cols;
        f4 t0, t1;
        if (cs_lds) { const f4* t = (const f4*)(lds + H::cs + (min(col - c0, (uint32_t)BM - 1) * half + da) * 8); t0 = t[0]; t1 = t[1]; }
        else { const f4* t = (const f4*)(g.rope_tab + (size_t)(g.base_pos + (on ? col : c0)) * half + da); t0 = t[0]; t1 = t[1]; }
        const float cs[4] = { t0[0], t0[2], t1[0], t1[2] }, sn[4] = { t0[1], t0[3], t1[1], t1[3] };
        const f4 va = *(const f4*)(hx0 + c * LR + da), vb = *(const f4*)(hx0 + c * LR + db);
        const float iv = norm ? inv[hb * CP + c] : 1.f;
        float oa[4], ob[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float a = va[i], b = vb[i];
          if (norm) { const float sa = iv * wa[i], sb = iv * wb[i]; a = a * sa; b = b * sb; }
          const float ac = a * cs[i], bs = b * sn[i], bc = b * cs[i], as = a * sn[i];    // rounded one by one
          oa[i] = ac - bs; ob[i] = bc + as;
        }
        store4(col, da, oa, on);
        store4(col, db, ob, on);
      }
    }
    // the rest (gate and v heads: all), a column or two an instruction; everything read before the first store
    if (plain || 2 * half < HD) {
      const bool scale = norm && !plain;
      f4 w = { 1.f, 1.f, 1.f, 1.f }, v[NI];
      float iv[NI];
      if (scale) w = *(const f4*)(wp + d);
#pragma unroll
      for (uint32_t k = 0; k < NI; k++) { v[k] = *(const f4*)(hx0 + (lw + k * CPI + cl) * LR + d); iv[k] = scale ? inv[hb * CP + lw + k * CPI + cl] : 1.f; }
#pragma unroll
      for (uint32_t k = 0; k < NI; k++) {
        const uint32_t col = col_of(lw + k * CPI + cl);
        float x[4];
#pragma unroll
        for (int i = 0; i < 4; i++) { x[i] = v[k][i]; if (scale) { const float sw = iv[k] * w[i]; x[i] = x[i] * sw; } }
        store4(col, d, x, col < g.n_cols && (plain || d >= 2 * half));
      }
    }
    }
  }
}

// The swizzle of 64-byte activation rows (KG = 1): chunk c of row r sits at c ^ (0, 2, 3, 1)[r / 4 % 4].  A 128-bit LDS read takes 16 lanes a clock, of a 16-row fragment rows 0 - 3 and
// 12 - 15 of one k quarter with rows 4 - 11 of the next: the four of r / 4 have to differ over those too, which (0, 1, 2, 3) does not give (rows 0 - 3 of
// quarter 0 and 4 - 7 of quarter 1 on the same banks: every activation read twice as long).
static __device__ inline uint32_t gt_swz64(uint32_t r) { return ((r >> 3) & 1) | (((r >> 2 ^ r >> 3) & 1) << 1); }

// The main loop of the shapes whose waves each hold whole sums (KG = 1), on 16 x 16 x 32 products: at the power limit they run faster than 32 x 32 x 16
// ones (half the accumulator traffic a product), and give the same bits.  Layer pass, 32 x 32 x 16 / so (us a layer): 4096 columns of the gated 16 / 2-head
// shape 430 / 408, 2048 of it 231 / 226, 2048 of the 24 / 4-head shape 534 / 510; one round of few workgroups (777 of that shape) 297 / 297.  A stage is one k-step of 32: the products with the first half of a wave's column blocks, the barrier,
// those with the second half; a fragment is read as soon as the products with the one in its registers are out, so a stage holds no more
// fragments than the two k-steps of 16 did.  Weights are the first operand: a lane holds four consecutive rows of a column.
template <int WM, int WN, int NA, int NB, int S, int EPI, int LPW, class Issue>
static __device__ __attribute__((always_inline)) inline void gt_whole_k(const GemmTileParams& p, const GlueParams& gp, unsigned char* lds, uint32_t c0, uint32_t r0, uint32_t wm, uint32_t wn, uint32_t n_stages,
                                              const unsigned char* const (&src)[LPW], const uint32_t (&step)[LPW], const uint32_t (&off)[LPW], const uint32_t (&dofs)[LPW], Issue issue) {
  constexpr int BM = WM * NA * 16, BN = WN * NB * 16, ABYTES = BM * 64, STAGE = (BM + BN) * 64;
  constexpr int N0 = (NA + 1) / 2, N1 = NA / 2;          // 16-column blocks of a wave in either half of a stage
  const uint32_t lane = threadIdx.x & 63, l16 = lane & 15, kq = lane >> 4;
  f4 acc[NA][NB];
#pragma unroll
  for (int a = 0; a < NA; a++)
#pragma unroll
    for (int b = 0; b < NB; b++) acc[a][b] = (f4){ 0.f, 0.f, 0.f, 0.f };
#pragma unroll
  for (int j = 0; j < S; j++) issue(j, j);
  // k 8 kq .. of a row: an activation row's chunk kq; of the weights' fragments, the half kq % 2 of k-step kq / 2
  const uint32_t x_rd = (wm * NA * 16 + l16) * 64 + ((kq ^ gt_swz64(l16)) * 16);
  // ... of a wave's 16-row block b, block wn NB + b of the tile: the half of a 32-row fragment that its parity says
  const uint32_t w_l = ABYTES + (kq >> 1) * 1024 + ((kq & 1) * 32 + l16) * 16, wb0 = wn * NB, wb1 = wb0 + 1;
  const uint32_t w_rd[2] = { w_l + (wb0 >> 1) * 2048 + (wb0 & 1) * 256, w_l + (wb1 >> 1) * 2048 + (wb1 & 1) * 256 };
  h8 x0[N0], x1[N1 > 0 ? N1 : 1], w[NB];
  auto rd_x = [&](h8& f, const unsigned char* sb, int a) __attribute__((always_inline)) { f = *(const h8*)(sb + x_rd + a * 1024); };
  auto rd_w = [&](h8& f, const unsigned char* sb, int b) __attribute__((always_inline)) { f = *(const h8*)(sb + w_rd[b % 2] + (b / 2) * 2048); };
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(LPW * (S - 1)) : "memory");       // stage 0 (S stages were issued)
  asm volatile("s_barrier" ::: "memory");
#pragma unroll
  for (int a = 0; a < N0; a++) rd_x(x0[a], lds, a);
#pragma unroll
  for (int b = 0; b < NB; b++) rd_w(w[b], lds, b);
  constexpr int H0 = N0 * NB, H1 = N1 * NB;              // products of either half of a stage
  static_assert(H1 >= N0 && N1 > 0, "a read behind each product of the second half");
  // Accumulating calls: the first NOLD of the wave's old blocks are requested behind the last stage's loads, under the products of the last S stages (addresses clamped
  // instead of guarded: a guarded load is a branch, one load a basic block, and the compiler waits for each).  Behind the loop, where every CU asks at once, they and the
  // stores took 7.4 of 61 us (4096 columns of 2048 x 4096): 69.8 -> 67.8 us a call, 4096 of 2048 x 2048 45.4 -> 44.2, 1300 of 5120 x 6144 86.5 -> 84.9.  Not on the 256 x 256 tile, whose
  // accumulators leave no room for a useful part of them (3000 of 5120 x 6144 160.0, with 16 of its 32 blocks 164.0, with 8 161.9).
  constexpr int NM = NA * NB, PHASE = NM > 28 ? 8 : NM < GT_OLD ? NM : GT_OLD, NOLD = EPI == GT_ACC && NM <= 28 ? PHASE : 0;
  typedef f4 f4u __attribute__((aligned(4)));                             // (y is aligned to its elements)
  auto col_of = [&](int a) { return c0 + (wm * NA + a) * 16 + l16; };
  auto row_of = [&](int b) { return r0 + (wn * NB + b) * 16 + 4 * kq; };
  const size_t last = EPI == GT_ACC ? (size_t)(p.n_cols - 1) * p.y_stride + p.d_out - 4 : 0;
  f4 old[EPI == GT_ACC ? PHASE : 1];
  auto request_old = [&](f4& o, int m) __attribute__((always_inline)) {
    const size_t at = (size_t)col_of(m / NB) * p.y_stride + row_of(m % NB);
    o = *(const f4u*)(p.y + (at < last ? at : last));
  };
  auto first_half = [&](const unsigned char* sb) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < H0; m++) {
      acc[m % N0][m / N0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[m / N0], x0[m % N0], acc[m % N0][m / N0], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (m < N1) { rd_x(x1[m], sb, N0 + m); __builtin_amdgcn_sched_barrier(0); }
    }
  };
  auto second_half = [&](const unsigned char* sn, auto READ, auto load) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < H1; m++) {
      acc[N0 + m % N1][m / N1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[m / N1], x1[m % N1], acc[N0 + m % N1][m / N1], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (decltype(READ)::value) {
        if (m < N0) rd_x(x0[m], sn, m);
        if (m % N1 == N1 - 1) rd_w(w[m / N1], sn, m / N1);
      }
      load(m);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  uint32_t buf = 0;
  const uint32_t n_main = n_stages > S ? n_stages - S : 0;
  for (uint32_t st = 0; st < n_main; st++) {
    const uint32_t nbuf = buf + 1 == S ? 0 : buf + 1;
    first_half(lds + buf * STAGE);
    // stage st + 1 is in LDS behind this barrier, and every wave has read stage st: its buffer takes stage st + S
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(LPW * (S - 2)) : "memory");
    second_half(lds + nbuf * STAGE, std::true_type{}, [&](int m) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < LPW; i++)
        if (i * (H1 - 1) / LPW == m) PF_GLL_S(src[i] + (size_t)(st + S) * step[i], off[i], lds + buf * STAGE + dofs[i]);
    });
    buf = nbuf;
  }
  // the last S stages, whose loads are all on their way (fewer stages than S: the ones past the end were requested as copies of the last, never read)
  auto tail = [&](auto J) __attribute__((always_inline)) {
    constexpr int j = decltype(J)::value;
    if (n_main + j >= n_stages) return;
    const uint32_t nbuf = buf + 1 == S ? 0 : buf + 1;
    first_half(lds + buf * STAGE);
    if constexpr (j < S - 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(LPW * (S - 2 - j) + (j > 0 ? NOLD : 0)) : "memory");
    second_half(lds + nbuf * STAGE, std::integral_constant<bool, (j < S - 1)>{}, [&](int m) __attribute__((always_inline)) {
      if constexpr (j == 0) {
#pragma unroll
        for (int i = 0; i < NOLD; i++) if (i * H1 / (NOLD > 0 ? NOLD : 1) == m) request_old(old[i], i);
      }
    });
    buf = nbuf;
  };
  static_assert(S >= 2 && S <= 6, "buffers");
  tail(std::integral_constant<int, 0>{}); tail(std::integral_constant<int, 1>{});
  if constexpr (S > 2) tail(std::integral_constant<int, 2>{});
  if constexpr (S > 3) tail(std::integral_constant<int, 3>{});
  if constexpr (S > 4) tail(std::integral_constant<int, 4>{});
  if constexpr (S > 5) tail(std::integral_constant<int, 5>{});
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(NOLD) : "memory");              // (copies past the end)
  if constexpr (EPI == GT_HEADS) {
    float* hx = (float*)lds;
    constexpr int LR = BN + 4;
    lds_barrier();
    heads_request<WM * 32, BN, BM>(gp, lds, c0);
    auto dump = [&](auto A) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 2; j++)
        if constexpr (2 * decltype(A)::value < NA)
          if (2 * decltype(A)::value + j < NA)
#pragma unroll
            for (int b = 0; b < NB; b++) *(f4*)(hx + (wm * 32 + j * 16 + l16) * LR + (wn * NB + b) * 16 + 4 * kq) = acc[2 * decltype(A)::value + j < NA ? 2 * decltype(A)::value + j : 0][b];
      asm volatile("; block %0" :: "n"(decltype(A)::value) : "memory");   // (the blocks' stores are not merged into one on selected registers)
    };
#pragma nounroll
    for (int a = 0; a < N0; a++) {                                       // a phase: 32 of every wave's columns (the last one of an odd number of blocks: 16)
      static_assert(N0 <= 5, "blocks of a wave");
      if (a == 0) dump(std::integral_constant<int, 0>{});
      if constexpr (N0 > 1) if (a == 1) dump(std::integral_constant<int, 1>{});
      if constexpr (N0 > 2) if (a == 2) dump(std::integral_constant<int, 2>{});
      if constexpr (N0 > 3) if (a == 3) dump(std::integral_constant<int, 3>{});
      if constexpr (N0 > 4) if (a == 4) dump(std::integral_constant<int, 4>{});
      if (a == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // what heads_request asked for
      lds_barrier();
      const auto col = [&](uint32_t c) -> uint32_t {
        if (NA % 2 && a * 32 + c % 32 >= NA * 16) return 0xffffffffu;      // no column: its row of LDS is an earlier phase's
        return c0 + c / 32 * (NA * 16) + a * 32 + c % 32;
      };
      if (gp.head_dim == 256) finish_heads<256, WM * 32, BN, BM>(gp, lds, c0, r0, p.d_out, col);
      else finish_heads<128, WM * 32, BN, BM>(gp, lds, c0, r0, p.d_out, col);
      lds_barrier();
    }
  } else {
    // Accumulating calls: loads and stores share one counter, and a wait for a loaded value waits for the stores in front of it as well, so the old values past the first
    // PHASE are requested, PHASE at a time, between the sums with those that are there and their stores.
    auto store = [&](int m) __attribute__((always_inline)) {
      const int a = m / NB, b = m % NB;
      const uint32_t col = col_of(a), row = row_of(b);
      if (col < p.n_cols) {
        float* y = p.y + (size_t)col * p.y_stride + row;
        if (row + 4 <= p.d_out) *(f4u*)y = acc[a][b];
        else
#pragma unroll
          for (int i = 0; i < 3; i++) if (row + i < p.d_out) y[i] = EPI == GT_ACC ? y[i] + acc[a][b][i] : acc[a][b][i];
      }
    };
    if constexpr (EPI != GT_ACC) {
#pragma unroll
      for (int m = 0; m < NM; m++) store(m);
    } else {
#pragma unroll
      for (int m0 = 0; m0 < NM; m0 += PHASE) {
        if (NOLD == 0 && m0 == 0) {
#pragma unroll
          for (int m = 0; m < PHASE; m++) request_old(old[m], m);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int m = m0; m < m0 + PHASE && m < NM; m++) if (row_of(m % NB) + 4 <= p.d_out) acc[m / NB][m % NB] = old[m - m0] + acc[m / NB][m % NB];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = m0 + PHASE; m < m0 + 2 * PHASE && m < NM; m++) request_old(old[m - m0 - PHASE], m);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = m0; m < m0 + PHASE && m < NM; m++) store(m);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

template <int WM, int WN, int KG, int TM, int TN, int S, int EPI>
__global__ __launch_bounds__(512, 2) void pa_gemm_tile_kernel(GemmTileParams p, GlueParams gp) {
  constexpr bool ACC = EPI == GT_ACC;
  static_assert(WM * WN * KG == 8, "eight waves");
  constexpr int KS = 2;                                  // k-steps of a stage per wave
  constexpr int U = KG == 1 ? 16 : 32;                   // columns and rows of a wave's blocks
  constexpr int BM = WM * TM * U, BN = WN * TN * U, BK = 16 * KG * KS;
  static_assert(BN % 32 == 0, "whole fragments of weights");
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
  auto swz = [](uint32_t r) __attribute__((always_inline)) -> uint32_t { return BK >= 128 ? r & 15 : BK == 64 ? (r >> 1) & 7 : gt_swz64(r); };

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
  if constexpr (KG == 1) {
    gt_whole_k<WM, WN, TM, TN, S, EPI>(p, gp, gt_lds, c0, r0, wm, wn, n_stages, src, step, off, dofs, issue);
  } else {
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
    if constexpr (EPI == GT_HEADS) {
      float sum[SPW];
#pragma unroll
      for (int k = 0; k < SPW; k++) {
        sum[k] = 0.f;
#pragma unroll
        for (int g = 0; g < KG; g++) sum[k] += red[((g * (WM * WN) + wt) * NT * 16 + kgrp * SPW + k) * 64 + lane];
      }
      lds_barrier();
      heads_request<BM, BN, BM>(gp, gt_lds, c0);
      float* hx = (float*)gt_lds;
#pragma unroll
      for (int k = 0; k < SPW; k++) hx[(col_s(k) - c0) * (BN + 4) + row_s(k) - r0] = sum[k];
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      lds_barrier();
      const auto col = [&](uint32_t c) { return c0 + c; };
      if constexpr (BN % 256 == 0) { if (gp.head_dim == 256) finish_heads<256, BM, BN, BM>(gp, gt_lds, c0, r0, p.d_out, col); }
      if (gp.head_dim == 128) finish_heads<128, BM, BN, BM>(gp, gt_lds, c0, r0, p.d_out, col);
      return;
    }
#pragma unroll
    for (int k = 0; k < SPW; k++) {
      float s = 0.f;
#pragma unroll
      for (int g = 0; g < KG; g++) s += red[((g * (WM * WN) + wt) * NT * 16 + kgrp * SPW + k) * 64 + lane];
      if (row_s(k) < p.d_out && col_s(k) < p.n_cols) p.y[(size_t)col_s(k) * p.y_stride + row_s(k)] = ACC ? old[k] + s : s;
    }
  }
}

template <int WM, int WN, int KG, int TM, int TN, int S, bool HEADS>
static hipError_t gt_launch(const GemmTileParams& q, int acc, const GlueParams* heads, hipStream_t s) {
  constexpr int U = KG == 1 ? 16 : 32, BM = WM * TM * U, BN = WN * TN * U, BK = 32 * KG;
  constexpr int lds_st = S * (BM + BN) * BK * 2, lds_red = KG > 1 ? KG * BM * BN * 4 : 0, lds_fixed = lds_st > lds_red ? lds_st : lds_red;
  typedef HeadsLds<(KG > 1 ? BM : WM * 32), BN> H;
  static_assert(lds_fixed <= GT_LDS && (!HEADS || H::cs <= GT_LDS), "LDS");
  int lds = lds_fixed;
  if (HEADS) lds = std::max(lds, H::cs + (cs_in_lds(H::cs, BM, heads->n_rot / 2) ? BM * (int)heads->n_rot * 4 : 0));
  const uint32_t total = ((q.n_cols + BM - 1) / BM) * ((q.d_out + BN - 1) / BN);
  static PaPerDevice lds_set[2];
  GlueParams none{};
  const auto kernel = HEADS ? pa_gemm_tile_kernel<WM, WN, KG, TM, TN, S, HEADS ? GT_HEADS : GT_STORE>
                            : acc ? pa_gemm_tile_kernel<WM, WN, KG, TM, TN, S, HEADS ? GT_HEADS : GT_ACC> : pa_gemm_tile_kernel<WM, WN, KG, TM, TN, S, HEADS ? GT_HEADS : GT_STORE>;
  const hipError_t e = pa_lds_limit(lds_set[acc ? 1 : 0], (const void*)kernel, HEADS ? GT_LDS : lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3((total + 7) / 8 * 8), dim3(512), lds, s, q, heads ? *heads : none);
  return hipGetLastError();
}

// The tile shapes, with what a round of the chip costs: ns per k of d_in (measured on rounds of 200 - 256 workgroups on 32 x 32 x 16 products; those of the kg = 1
// shapes are from before gt_whole_k, which takes some 5 % off several full rounds of them) on top of about 6 us for a round's first loads and last stores.
struct TileShape { uint16_t bm, bn, kg; float us, ns_k; hipError_t (*launch)(const GemmTileParams&, int, const GlueParams*, hipStream_t); };
static const TileShape tile_shapes[] = {
  { 64, 128, 4, 6.f, 6.5f, gt_launch<1, 2, 4, 2, 2, 3, false> },
  { 128, 128, 2, 6.f, 10.3f, gt_launch<2, 2, 2, 2, 2, 4, false> },
  { 128, 160, 2, 6.f, 11.8f, gt_launch<4, 1, 2, 1, 5, 4, false> },
  { 128, 192, 1, 6.f, 14.0f, gt_launch<2, 4, 1, 4, 3, 6, false> },
  { 128, 256, 1, 6.f, 15.5f, gt_launch<2, 4, 1, 4, 4, 6, false> },
  { 128, 320, 1, 6.f, 19.0f, gt_launch<2, 4, 1, 4, 5, 5, false> },
  { 128, 384, 1, 6.f, 21.5f, gt_launch<2, 4, 1, 4, 6, 4, false> },
  { 128, 448, 1, 6.f, 25.0f, gt_launch<2, 4, 1, 4, 7, 4, false> },
  { 256, 256, 1, 6.f, 27.0f, gt_launch<2, 4, 1, 8, 4, 4, false> },
};
// ... and those that hold whole heads (128 rows: of head_dim 128) and can end with the pre-step, whose work is part of a round's start here.
// Fitted to 75 sizes (the three model shapes, 33 to 4096 columns) on 32 x 32 x 16 products.  As the kernels are now, on 16 sizes (257 to 1024 columns) timed on every
// shape with the call's kg, the one taken is the fastest or within 1 % of it, but for 640 columns of the 24 / 4-head shape (205 us a layer, 199 on 192 columns).
static const TileShape head_shapes[] = {
  { 64, 128, 4, 3.5f, 7.1f, gt_launch<1, 2, 4, 2, 2, 3, true> },
  { 128, 128, 2, 4.3f, 8.9f, gt_launch<2, 2, 2, 2, 2, 4, true> },
  { 64, 256, 2, 5.6f, 11.8f, gt_launch<1, 4, 2, 2, 2, 3, true> },
  { 96, 256, 1, 5.f, 12.8f, gt_launch<2, 4, 1, 3, 4, 6, true> },
  { 128, 256, 1, 3.7f, 14.5f, gt_launch<2, 4, 1, 4, 4, 6, true> },
  { 160, 256, 1, 9.2f, 15.9f, gt_launch<2, 4, 1, 5, 4, 5, true> },
  { 192, 256, 1, 10.3f, 16.1f, gt_launch<2, 4, 1, 6, 4, 5, true> },
  { 224, 256, 1, 17.2f, 17.4f, gt_launch<2, 4, 1, 7, 4, 4, true> },
  { 256, 256, 1, 16.5f, 17.8f, gt_launch<2, 4, 1, 8, 4, 4, true> },
  { 320, 256, 1, 24.2f, 20.7f, gt_launch<2, 4, 1, 10, 4, 4, true> },
};

// One workgroup is resident per CU, so a call costs whole rounds of n_cu workgroups: the shape with the cheapest rounds, and
// its estimate in us.  Larger tiles pay less traffic per product but are coarser: which one wins changes with every
// multiple of a tile edge (777 columns of 5120 x 6144: 128 x 160, 224 workgroups, 63 us; 128 x 128, 280 workgroups, 87 us).  Of
// 104 sizes measured on every tile as they are and on the 64 x 64 kernel (8 weight shapes x 13 column counts, cold weights) the choice between
// all of them is the fastest at 90 and within 6 % at 2; it is 7 - 27 % behind at 12, most where one round of few workgroups (which
// costs less than a full one) is set against the 64 x 64 kernel: 9216 x 2048, 200 columns 27 % over 128 x 128.
static float rounds_us(const TileShape& t, uint32_t d_out, uint32_t d_in, uint32_t n_cols, int n_cu) {
  const uint64_t wgs = (uint64_t)((n_cols + t.bm - 1) / t.bm) * ((d_out + t.bn - 1) / t.bn), cus = n_cu > 0 ? n_cu : 256;
  return (float)((wgs + cus - 1) / cus) * (t.us + t.ns_k * 1e-3f * d_in);
}
static int pa_pick_tile(uint32_t d_out, uint32_t d_in, uint32_t n_cols, int n_cu, float* us) {
  int best = 0;
  *us = 1e30f;
  for (int i = 0; i < (int)(sizeof tile_shapes / sizeof tile_shapes[0]); i++) {
    const float c = rounds_us(tile_shapes[i], d_out, d_in, n_cols, n_cu);
    if (c < *us) { *us = c; best = i; }
  }
  return best;
}

float pa_gemm_tile_us(uint32_t d_out, uint32_t d_in, uint32_t n_cols, int n_cu, uint32_t* shape, uint32_t* kg) {
  float us;
  const TileShape& t = tile_shapes[pa_pick_tile(d_out, d_in, n_cols, n_cu, &us)];
  *shape = (uint32_t)t.bm << 16 | t.bn; *kg = t.kg;
  return us;
}

hipError_t pa_launch_gemm_tile(const GemmParams& p, const uint16_t* w16, int n_cu, hipStream_t s) {
  if (p.d_out == 0 || p.d_in == 0 || p.d_in % 128 != 0 || p.n_cols < 4 || p.x_stride > (1u << 22)) return hipErrorInvalidValue;   // (32-bit row offsets inside a tile)
  GemmTileParams q;
  q.x = p.x; q.w16 = w16; q.y = p.y; q.x_stride = p.x_stride; q.y_stride = p.y_stride; q.d_out = p.d_out; q.d_in = p.d_in; q.n_cols = p.n_cols;
  float us;
  return tile_shapes[pa_pick_tile(p.d_out, p.d_in, p.n_cols, n_cu, &us)].launch(q, p.acc, nullptr, s);
}

// kg: the groups of waves that a stage's k-steps are split over, which fixes the order of an element's sum
static int pick_heads(uint32_t d_out, uint32_t d_in, uint32_t n_cols, uint32_t head_dim, uint32_t kg, int n_cu, float* us) {
  int best = -1;
  *us = 1e30f;
  for (int i = 0; i < (int)(sizeof head_shapes / sizeof head_shapes[0]); i++) {
    const TileShape& t = head_shapes[i];
    if (t.bn % head_dim || t.kg != kg) continue;
    // 96 columns where 128 take as many blocks (65 - 96, 129 - 192, 257 - 288 columns): the wider tile is the faster one all the same, its last
    // block is the emptier and brings the weights in for the others (us a layer of the 24 / 4-head shape, 96 / 128 columns a tile: 144 columns 116 / 107,
    // 192 129 / 123, 257 133 / 118, 272 140 / 125, 288 143 / 133; 16 / 2-head shape, 257 66.8 / 64.1).
    if (t.bm == 96 && (n_cols + 95) / 96 == (n_cols + 127) / 128) continue;
    const float c = rounds_us(t, d_out, d_in, n_cols, n_cu);
    if (c < *us) { *us = c; best = i; }
  }
  return best;
}

float pa_gemm_heads_us(uint32_t d_out, uint32_t d_in, uint32_t n_cols, uint32_t head_dim, uint32_t kg, int n_cu, uint32_t* shape) {
  float us;
  const int i = pick_heads(d_out, d_in, n_cols, head_dim, kg, n_cu, &us);
  *shape = i < 0 ? 0 : (uint32_t)head_shapes[i].bm << 16 | head_shapes[i].bn;
  return us;
}

hipError_t pa_launch_gemm_heads(const GemmParams& p, const uint16_t* w16, const GlueParams& heads, uint32_t kg, int n_cu, hipStream_t s) {
  const uint32_t half = heads.n_rot / 2;
  if (p.d_out == 0 || p.d_in == 0 || p.d_in % 128 != 0 || p.n_cols == 0 || p.x_stride > (1u << 22) || p.d_out % heads.head_dim || half < (heads.ks_cache ? 32u : 4u) || (half & (half - 1)) || !heads.rope_tab) return hipErrorInvalidValue;
  GemmTileParams q;
  q.x = p.x; q.w16 = w16; q.y = nullptr; q.x_stride = p.x_stride; q.y_stride = 0; q.d_out = p.d_out; q.d_in = p.d_in; q.n_cols = p.n_cols;
  float us;
  const int i = pick_heads(p.d_out, p.d_in, p.n_cols, heads.head_dim, kg, n_cu, &us);
  return i < 0 ? hipErrorNotSupported : head_shapes[i].launch(q, 0, &heads, s);
}

// Column-batched projections for large chunks on gfx950: Y[c][r] = sum_k W[r][k] X[c][k] with the weights widened
// to f16 once and a matrix-core GEMM over two f16 operands.
//
// Same contract and the same operand precision as pa_gemm_kernel (proj_gemm.hip) -- the reference's "f16" prefill
// math, engine/wgsl/gemm.js:31-36: every dequantised weight and every activation rounded to f16, products and sums
// f32 -- for the chunks its batched GEMMs serve (engine/wgsl/gemm.js, gemm_sgm.js, gemm_wide.js; dispatched at
// engine/qwen35.js:2142-2170, :2600-2620).  What differs is where the widening happens.  The tiled kernel of
// proj_gemm.hip widens packed weights on their way into LDS inside its main loop; at 64 x 64 wave tiles that loop is
// bound by LDS traffic and by the widening arithmetic in front of every barrier.  For a chunk of many columns
// the weights are re-read by every column block anyway, so here they are widened once into an f16 staging matrix
// (pa_widen_w_kernel: one pass over the packed planes, HBM-bound; the caller keeps the matrix with the weight or
// widens per call), and the GEMM proper has nothing but loads and MFMAs in its loop:
//   * the staging matrix is in MFMA fragment order: for every block of 16 k and 32 rows the 64 lanes' 16 bytes are contiguous
//     (1 KB), so a weight fragment is one coalesced wave-wide load, straight into the registers the MFMA reads or into LDS.
//     The k blocks are outermost: workgroups walk K in step, and what all of them read at a time is one contiguous range
//     (rows outermost, every row block's stream sat at the same offset of its own 128 - 384 KB stripe: 5120 x 6144, 512
//     columns, 128 x 256 tiles 102 -> 97 us);
//   * chunks with enough 64 x 64 tiles to be worth larger ones: proj_gemm_tile.hip;
//   * smaller ones: the kernel below, 64 x 64 (or 32) tiles whose four waves split K.
#include "pf_common.h"
#include <algorithm>

struct Gemm16Params {
  const uint16_t* x; const uint16_t* w16; float* y;
  uint32_t x_stride, y_stride, d_out, d_in, n_cols;
  int acc;
};

// ---- weights -> f16 in MFMA fragment order: for row block rb (32 rows, the last one padded with copies of the last
//      row) and k block kb (16 values) the 1 KB at ((kb n_rb + rb) 64 + lane) 16 (n_rb row blocks in all) holds, for lane = 32 fk + fl, the 8
//      values k = 16 kb + 8 fk .. + 7 of row 32 rb + fl.  The arithmetic is the tiled kernel's staging: (nibble - 8) *
//      scale and int8 * scale in f16 (exact integer, one rounding), f32 rounded to nearest even ----
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
static __device__ inline h2v gw_as_h2(uint32_t u) { h2v r; __builtin_memcpy(&r, &u, 4); return r; }
static __device__ inline h2v gw_bytes(uint32_t w, uint32_t sel, h2v bias, h2v sc) { return (gw_as_h2(__builtin_amdgcn_perm(0x64646464u, w, sel)) - bias) * sc; }

// one thread per (row, quantisation block of 32 weights), the 32 rows of a row block on consecutive threads
template <int KIND>
__global__ __launch_bounds__(256) void pa_widen_w_kernel(const void* w, const uint16_t* scales, uint16_t* out, uint32_t d_out, uint32_t nb, size_t n_threads) {
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= n_threads) return;
  const uint32_t fl = (uint32_t)(idx % 32), bq = (uint32_t)((idx / 32) % nb);
  const size_t rb = idx / ((size_t)32 * nb);
  const size_t b = (size_t)min((uint32_t)(rb * 32 + fl), d_out - 1) * nb + bq;          // the packed block this thread widens
  h8 o[4];
  if constexpr (KIND == PA_W_Q4_0) {
    const u4 q = *(const u4*)((const unsigned char*)w + b * 16);       // byte j: element j (low nibble), element 16 + j (high)
    const _Float16 s = __ushort_as_half(scales[b]);
    const h2v sc = { s, s }, bias = { (_Float16)1032.f, (_Float16)1032.f };
    h2v lo[8], hi[8];
#pragma unroll
    for (int d = 0; d < 4; d++) {
      const uint32_t l = q[d] & 0x0F0F0F0Fu, h = (q[d] >> 4) & 0x0F0F0F0Fu;
      lo[2 * d] = gw_bytes(l, 0x04010400u, bias, sc); lo[2 * d + 1] = gw_bytes(l, 0x04030402u, bias, sc);
      hi[2 * d] = gw_bytes(h, 0x04010400u, bias, sc); hi[2 * d + 1] = gw_bytes(h, 0x04030402u, bias, sc);
    }
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
      for (int j = 0; j < 4; j++) { o[v][2 * j] = lo[4 * v + j][0]; o[v][2 * j + 1] = lo[4 * v + j][1]; o[2 + v][2 * j] = hi[4 * v + j][0]; o[2 + v][2 * j + 1] = hi[4 * v + j][1]; }
  } else if constexpr (KIND == PA_W_Q8_0) {
    const u4* src = (const u4*)((const unsigned char*)w + b * 32);
    const _Float16 s = __ushort_as_half(scales[b]);
    const h2v sc = { s, s }, bias = { (_Float16)1152.f, (_Float16)1152.f };
#pragma unroll
    for (int v = 0; v < 2; v++) {
      const u4 q = src[v];
#pragma unroll
      for (int d = 0; d < 4; d++) {
        const uint32_t x = q[d] ^ 0x80808080u;
        const h2v e0 = gw_bytes(x, 0x04010400u, bias, sc), e1 = gw_bytes(x, 0x04030402u, bias, sc);
        o[2 * v + d / 2][4 * (d & 1)] = e0[0]; o[2 * v + d / 2][4 * (d & 1) + 1] = e0[1];
        o[2 * v + d / 2][4 * (d & 1) + 2] = e1[0]; o[2 * v + d / 2][4 * (d & 1) + 3] = e1[1];
      }
    }
  } else {
    const f4* src = (const f4*)((const float*)w + b * 32);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const f4 x0 = src[2 * v], x1 = src[2 * v + 1];
      o[v] = (h8){ (_Float16)x0[0], (_Float16)x0[1], (_Float16)x0[2], (_Float16)x0[3], (_Float16)x1[0], (_Float16)x1[1], (_Float16)x1[2], (_Float16)x1[3] };
    }
  }
  // o[v] = values 8 v .. 8 v + 7 of the block: k block 2 bq + v / 2, half fk = v & 1
  const size_t n_rb32 = (d_out + 31) / 32;
#pragma unroll
  for (int v = 0; v < 4; v++) *(h8*)(out + ((((size_t)(2 * bq + v / 2) * n_rb32 + rb) * 64 + (v & 1) * 32 + fl) * 8)) = o[v];
}

// ---- chunks too small to give every CU one of the tiles above (a few dozen to a few hundred columns, or few weight
//      rows): 64 columns x 64 weight rows a workgroup, and the workgroup's four waves split K between them instead of
//      the tile -- of every K stage of 128 wave w takes the k-steps w and w + 4 -- so that all four share the staged
//      activations (one coalesced fetch per workgroup) while each loads only the weight fragments of its own
//      k-steps.  Every wave holds the whole 64 x 64 tile (4 MFMA tiles, 64 accumulators: two workgroups a CU); at the
//      end the four copies meet in LDS and wave w adds up MFMA tile w in a fixed order (((w0 + w1) + w2) + w3) and
//      stores it.  A workgroup walks all of K, so there are no partial sums in memory and no second launch; what
//      bounds it is the L2 -> CU traffic of 64 x 64 tiles (K (64 + 64) 2 bytes a tile), about twice its MFMA time.
#define GM_T 64              // columns per workgroup
#define GM_KS 128            // K per stage
#define GM_ROWB 256          // bytes of a staged activation row

template <int TN, int RING, bool ACC>
__global__ __launch_bounds__(256, 2) void pa_gemm16_mid_kernel(Gemm16Params p) {
  constexpr int STAGE = GM_T * GM_ROWB;                  // 16 KB
  constexpr int ROWS = 32 * TN;                          // weight rows per workgroup
  constexpr int NT = 2 * TN;                             // MFMA tiles per wave: 2 column blocks x TN row blocks
  __shared__ __attribute__((aligned(1024))) unsigned char smem[(4 * NT * 16 * 64 * 4 > 2 * STAGE) ? 4 * NT * 16 * 64 * 4 : 2 * STAGE];   // two stages; at the end the four waves' tiles
  const uint32_t tid = threadIdx.x, lane = tid & 63, fl = lane & 31, fk = lane >> 5;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // XCD k owns a contiguous range of tiles, column blocks fastest: neighbours stream the same weight rows through one L2
  const uint32_t n_cb = (p.n_cols + GM_T - 1) / GM_T, n_rb = (p.d_out + ROWS - 1) / ROWS, total = n_cb * n_rb;
  const uint32_t per = (total + 7) / 8, tile = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (tile >= total) return;
  const uint32_t c0 = (tile % n_cb) * GM_T, r0 = (tile / n_cb) * ROWS;
  const uint32_t n_stages = p.d_in / GM_KS;

  // A: a load covers 4 rows x 256 bytes; chunk c of row r is staged at slot c ^ (r & 15)
  const uint32_t lrow = lane >> 4, lchunk = lane & 15;
  const unsigned char* a_src[4];
  uint32_t a_dst[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t row = (wave * 4 + i) * 4 + lrow;
    const size_t col = min((size_t)c0 + row, (size_t)p.n_cols - 1);     // columns past the end repeat the last one (never stored)
    a_src[i] = (const unsigned char*)(p.x + col * p.x_stride) + lchunk * 16;
    a_dst[i] = row * GM_ROWB + ((lchunk ^ (row & 15)) * 16);
  }
  // a stage's activations are fetched two stages ahead (two register sets), its weight fragments RING stages ahead:
  // one stage of MFMAs is far less than a round trip to L2, let alone to HBM, and a workgroup's time is its number of
  // stages x that latency / the stages it keeps in flight
  u4 areg[2][4];
  auto fetch_a = [&](int set, uint32_t st) __attribute__((always_inline)) {
    const size_t off = (size_t)min(st, n_stages - 1) * GM_ROWB;       // past the last stage: the last one again, never used
#pragma unroll
    for (int i = 0; i < 4; i++) areg[set][i] = *(const u4*)(a_src[i] + off);
  };
  auto store_a = [&](int set, uint32_t buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; i++) *(u4*)(smem + buf * STAGE + a_dst[i]) = areg[set][i];
  };
  // fragment of column block t at k-step j of the stage: row 32 t + fl, chunk 2 j + fk
  uint32_t a_rd[2][2];
#pragma unroll
  for (int t = 0; t < 2; t++)
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const uint32_t row = t * 32 + fl, chunk = 2 * (wave + 4 * u) + fk;
      a_rd[t][u] = row * GM_ROWB + ((chunk ^ (row & 15)) * 16);
    }
  // B: this wave's k blocks 8 st + wave and 8 st + wave + 4 of the TN 32-row blocks
  const uint32_t n_rb32 = (p.d_out + 31) / 32;
  const unsigned char* b_src[TN];
#pragma unroll
  for (int t = 0; t < TN; t++) b_src[t] = (const unsigned char*)p.w16 + ((size_t)min(r0 / 32 + t, n_rb32 - 1) * 64 + lane) * 16;
  u4 bq[RING][2][TN];                                    // [stage % RING][u][row block]
  auto load_b = [&](int slot, uint32_t st) __attribute__((always_inline)) {
    const size_t off = (size_t)(min(st, n_stages - 1) * 8 + wave) * n_rb32 * 1024;
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int t = 0; t < TN; t++) bq[slot][u][t] = *(const u4*)(b_src[t] + off + (size_t)u * 4 * n_rb32 * 1024);
  };
  f16v acc[2][TN];
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < TN; b++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[a][b][i] = 0.f;

#pragma unroll
  for (int j = 0; j < RING; j++) load_b(j, j);
  fetch_a(0, 0);
  fetch_a(1, 1);
  store_a(0, 0);
  fetch_a(0, 2);
  __syncthreads();
  // stage st reads LDS buffer st % 2 and ring slot st % RING; register set p holds the stages of parity p: at the
  // end of stage st the other set (stage st + 1, fetched two stages ago) goes to the other buffer and then receives
  // stage st + 3
  auto stage = [&](auto J, uint32_t st) __attribute__((always_inline)) {
    constexpr int j = decltype(J)::value, par = j & 1;
    const unsigned char* sb = smem + par * STAGE;
#pragma unroll
    for (int u = 0; u < 2; u++) {
      h8 af[2], bf[TN];
#pragma unroll
      for (int t = 0; t < 2; t++) af[t] = *(const h8*)(sb + a_rd[t][u]);
#pragma unroll
      for (int t = 0; t < TN; t++) __builtin_memcpy(&bf[t], &bq[j][u][t], 16);
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < TN; b++) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[a], bf[b], acc[a][b], 0, 0, 0);
    }
    load_b(j, st + RING);
    store_a(par ^ 1, par ^ 1);          // stage st + 1 into the other buffer: every wave left it before the last barrier
    fetch_a(par ^ 1, st + 3);
    __syncthreads();
  };
  static_assert(RING == 4 || RING == 8, "the loop below is unrolled by the ring");
  for (uint32_t st = 0; st < n_stages; st += RING) {
    stage(std::integral_constant<int, 0>{}, st);
    if (st + 1 < n_stages) stage(std::integral_constant<int, 1>{}, st + 1);
    if (st + 2 < n_stages) stage(std::integral_constant<int, 2>{}, st + 2);
    if (st + 3 < n_stages) stage(std::integral_constant<int, 3>{}, st + 3);
    if constexpr (RING == 8) {
      if (st + 4 < n_stages) stage(std::integral_constant<int, 4>{}, st + 4);
      if (st + 5 < n_stages) stage(std::integral_constant<int, 5>{}, st + 5);
      if (st + 6 < n_stages) stage(std::integral_constant<int, 6>{}, st + 6);
      if (st + 7 < n_stages) stage(std::integral_constant<int, 7>{}, st + 7);
    }
  }
  // the four partial tiles meet in LDS (the stages are dead behind the loop's last barrier): [wave][slot][lane], slot =
  // 16 (TN a + b) + i for accumulator i of the MFMA tile of column block a and row block b
  float* red = (float*)smem;
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < TN; b++)
#pragma unroll
      for (int i = 0; i < 16; i++) red[((wave * NT + a * TN + b) * 16 + i) * 64 + lane] = acc[a][b][i];
  __syncthreads();
  // wave w finishes slots [w SPW, (w + 1) SPW); accumulator i of a tile = column 8 (i / 4) + 4 fk + i % 4, row fl
  constexpr int SPW = NT * 16 / 4;
  float sum[SPW];
#pragma unroll
  for (int k = 0; k < SPW; k++) {
    const uint32_t o = (wave * SPW + k) * 64 + lane;
    sum[k] = ((red[o] + red[o + NT * 16 * 64]) + red[o + 2 * NT * 16 * 64]) + red[o + 3 * NT * 16 * 64];
  }
  auto col_of = [&](int k) { const uint32_t sl = wave * SPW + k, a = sl / (16 * TN), i = sl % 16; return c0 + a * 32 + 8 * (i / 4) + 4 * fk + (i % 4); };
  auto row_of = [&](int k) { const uint32_t sl = wave * SPW + k, b = sl / 16 % TN; return r0 + b * 32 + fl; };
  float old[SPW];
  if constexpr (ACC) {
#pragma unroll
    for (int k = 0; k < SPW; k++) old[k] = p.y[(size_t)min(col_of(k), p.n_cols - 1) * p.y_stride + min(row_of(k), p.d_out - 1)];   // unconditional (clamped): guarded loads would go out one round trip at a time
  }
#pragma unroll
  for (int k = 0; k < SPW; k++)
    if (row_of(k) < p.d_out && col_of(k) < p.n_cols) p.y[(size_t)col_of(k) * p.y_stride + row_of(k)] = ACC ? old[k] + sum[k] : sum[k];
}

template <int TN, int RING>
static hipError_t launch_gemm16_mid(const Gemm16Params& q, hipStream_t s) {
  const uint32_t total = ((q.n_cols + GM_T - 1) / GM_T) * ((q.d_out + 32 * TN - 1) / (32 * TN));
  if (q.acc) hipLaunchKernelGGL((pa_gemm16_mid_kernel<TN, RING, true>), dim3((total + 7) / 8 * 8), dim3(256), 0, s, q);
  else hipLaunchKernelGGL((pa_gemm16_mid_kernel<TN, RING, false>), dim3((total + 7) / 8 * 8), dim3(256), 0, s, q);
  return hipGetLastError();
}

// chunks wider than the kernel for a few columns (proj_gemm_skinny.hip) serves
bool pa_gemm_wide_serves(const GemmParams& p) {
  return p.n_cols > 16 && p.d_in % GM_KS == 0 && (p.x_stride & 7) == 0 && ((uintptr_t)p.x & 15) == 0;
}

// bytes of the staging matrix of a weight: whole 32-row blocks
size_t pa_gemm_wide_staging_bytes(uint32_t d_out, uint32_t d_in) { return (size_t)((d_out + 31) / 32) * 32 * d_in * sizeof(uint16_t); }

// The 64 x 64 kernel runs two workgroups a CU and its time follows their number: about 4 us and 4.6 ns per k and workgroup a
// CU (cold weights, 4096 x 2048: 256 / 512 / 777 columns 13.0 / 19.8 / 32.3 us; past one a CU it is some 10 % longer on 9216 rows).  The larger tiles where their rounds come out cheaper, and their
// kernel takes the stride.
// Fewer 64 x 64 tiles than half the CUs: 32-row tiles (twice the workgroups) with twice the stages in flight (2048 x 4096 on up to
// 64 columns, cold: 20 -> 16.7 us; with 144 tiles, 9216 x 2048, it is 2 us slower).
static float mid_tile_us(uint32_t d_in, uint64_t tiles64, uint32_t cus) { return 4.f + 4.6e-3f * d_in * std::max(1.f, (float)tiles64 / cus); }
// Columns << 16 | rows of the tile a call takes; 64-column tiles of up to 64 rows are this file's kernel.
extern "C" uint32_t pa_rule_gemm_wide_tile(uint32_t d_out, uint32_t d_in, uint32_t n_cols, uint32_t x_stride, int n_cu) {
  const uint32_t cus = n_cu > 0 ? (uint32_t)n_cu : 256u;
  const uint64_t tiles64 = (uint64_t)((n_cols + GM_T - 1) / GM_T) * ((d_out + 63) / 64);
  const float mid_us = mid_tile_us(d_in, tiles64, cus);
  uint32_t shape, kg;
  if (x_stride <= (1u << 22) && pa_gemm_tile_us(d_out, d_in, n_cols, n_cu, &shape, &kg) < mid_us) return shape;
  return (uint32_t)GM_T << 16 | (tiles64 * 2 < cus ? 32u : 64u);
}

// How a chunk's [q | k | v] projection that ends with the pre-step runs (proj_gemm_tile.hip): k groups << 28 | columns << 16 | rows of its tile, or 0
// where the two apart are the faster form -- the tiles that hold whole heads are few, and below some 200 - 300 columns (64-column tiles of too
// few workgroups) they cost more than the pre-step's launch, 3.5 us and the f32 projections through memory at 6 TB/s (16 columns 3.9 us, 512 of
// the 16 / 8-head shape 6.5, 777 of the 24 / 4-head shape 19.6, 4096 of the 16 / 2-head shape 53.5).  Only tiles that split K as the call apart does:
// a projection has its bits.  Taken where its estimate is 3 % ahead: closer than that the estimates do not tell which is faster (24 / 4-head shape, 214 - 256 columns,
// estimates within 1.2 %: 118 - 126 us a layer apart, up to 1 % more so from position 0, up to 1 % less behind 1000 rows).  On 238 sizes (the three model
// shapes, 33 to 4096 columns) the choice is 7 % ahead of always apart (best 22 %) and at no size behind it.
extern "C" uint32_t pa_rule_gemm_heads(uint32_t d_out, uint32_t d_in, uint32_t n_cols, uint32_t n_heads, uint32_t head_dim, int gated, int n_cu) {
  const uint32_t cus = n_cu > 0 ? (uint32_t)n_cu : 256u;
  uint32_t shape, kg, whole;
  const uint64_t tiles64 = (uint64_t)((n_cols + GM_T - 1) / GM_T) * ((d_out + 63) / 64);
  float apart = pa_gemm_tile_us(d_out, d_in, n_cols, n_cu, &shape, &kg);
  const float mid = mid_tile_us(d_in, tiles64, cus);
  if (mid <= apart) { apart = mid; kg = 4; }                            // (the 64-column kernel's four waves: k-steps w and w + 4 of eight)
  apart += 3.5f + 0.166e-6f * 4.f * n_cols * ((float)d_out + n_heads * head_dim * (gated ? 2.f : 1.f));
  return pa_gemm_heads_us(d_out, d_in, n_cols, head_dim, kg, n_cu, &whole) * 1.03f < apart ? kg << 28 | whole : 0;
}
// ... whose arithmetic takes rotation tables of a power of two of pairs, on int8 caches whole blocks of them
bool pa_gemm_heads_serves(const GemmParams& p, const GlueParams& g, int n_cu) {
  const uint32_t half = g.n_rot / 2;
  if (!pa_gemm_wide_serves(p) || pa_gemm_skinny_serves(p) || p.x_stride > (1u << 22) || !g.rope_tab) return false;
  if ((half & (half - 1)) || half < (g.ks_cache ? 32u : 4u)) return false;
  return pa_rule_gemm_heads(p.d_out, p.d_in, p.n_cols, g.n_heads, g.head_dim, (g.flags & PA_FLAG_GATE) != 0, n_cu) != 0;
}

// w16: staging of pa_gemm_wide_staging_bytes (the caller's, 16-byte aligned); widen = false: it already holds these weights
hipError_t pa_launch_gemm_wide(const GemmParams& p, uint16_t* w16, bool widen, const GlueParams* heads, int n_cu, hipStream_t s) {
  if (widen) {
    const uint32_t nb = p.d_in / 32;
    const size_t n_threads = (size_t)((p.d_out + 31) / 32) * 32 * nb;
    const dim3 wgrid((unsigned)((n_threads + 255) / 256));
    switch (p.kind) {
      case PA_W_Q4_0: hipLaunchKernelGGL(pa_widen_w_kernel<PA_W_Q4_0>, wgrid, dim3(256), 0, s, p.w, p.scales, w16, p.d_out, nb, n_threads); break;
      case PA_W_Q8_0: hipLaunchKernelGGL(pa_widen_w_kernel<PA_W_Q8_0>, wgrid, dim3(256), 0, s, p.w, p.scales, w16, p.d_out, nb, n_threads); break;
      case PA_W_F32: hipLaunchKernelGGL(pa_widen_w_kernel<PA_W_F32>, wgrid, dim3(256), 0, s, p.w, p.scales, w16, p.d_out, nb, n_threads); break;
      default: return hipErrorInvalidValue;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (heads) return pa_launch_gemm_heads(p, w16, *heads, pa_rule_gemm_heads(p.d_out, p.d_in, p.n_cols, heads->n_heads, heads->head_dim, (heads->flags & PA_FLAG_GATE) != 0, n_cu) >> 28, n_cu, s);
  const uint32_t tile = pa_rule_gemm_wide_tile(p.d_out, p.d_in, p.n_cols, p.x_stride, n_cu);
  if (tile >> 16 != GM_T || (tile & 0xffff) > 64) return pa_launch_gemm_tile(p, w16, n_cu, s);
  Gemm16Params q;
  q.x = p.x; q.w16 = w16; q.y = p.y; q.x_stride = p.x_stride; q.y_stride = p.y_stride;
  q.d_out = p.d_out; q.d_in = p.d_in; q.n_cols = p.n_cols; q.acc = p.acc;
  return (tile & 0xffff) == 32 ? launch_gemm16_mid<1, 8>(q, s) : launch_gemm16_mid<2, 4>(q, s);
}

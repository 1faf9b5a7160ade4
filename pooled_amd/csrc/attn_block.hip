// Split-K attention of a verify block (two to four 16-row blocks of stacked query rows a workgroup) on gfx950: the workgroup's waves share one
// online softmax and divide the product O^T = V^T P^T by OUTPUT DIMS.
//
// Work decomposition: as the tile loop of attn_decode.hip -- one workgroup of 4 wavefronts per (split, kv head, column group), a kv head's 32-row tiles dealt
// round robin to the waves of all its splits, 32 KB of loads in flight a wave -- but what a wave holds of O is HD / 4 dims of ALL rows of the workgroup's four
// tiles instead of all dims of its own tile's:
//   * a wave scores its own tile (q fragments in registers: the K tile is all that the product reads from LDS) and publishes its row maxima; behind a
//     barrier every wave knows the workgroup's, so all of them work relative to one lazily updated reference and P of the four tiles can be added up by the MFMA;
//   * with one reference for four tiles only one of their largest weights is 1, and exact in f16, where a wave of its own has one in every tile: P's rounding alone would
//     make an output's error 1 - 2 % larger over several tiles a wave and 6 % over one (relative, against 64 bits; tile loop and single-round kernel 2.5 - 2.9e-4).  The scores
//     therefore see the first quarter of q's dims at f32 precision (f16 + f16, q_lo_row of attn_decode.hip), which takes a quarter of q's rounding out: 0.92 - 0.98 of
//     the others' error for 0.2 - 0.4 us a call (16 / 2-head shape, 5 columns at 8191 rows 14.3 -> 14.7, 24 / 4-head, 8 at 65536 54.0 -> 54.3; half of the dims 0.87 - 0.89
//     for 0.4 - 0.9 us, all of them spill; P in two halves 0.73 - 0.82 for 0.5 - 3 us);
//   * P goes to LDS, V to the wave's V region; behind a second barrier each wave multiplies the four tiles' V^T by their P for its dims.
// Nothing is merged at the end: the waves of the tile loop meet in LDS there, 1.9 / 2.6 / 4.3 us with two / two / three row blocks (in-kernel stamps: 16 / 2-head shape, 5
// columns at 8191 rows and 16 at 12345; 24 / 4-head shape, 8 at 65536), which no stream hides.  The price is two barriers a turn, so that the workgroup's
// waves move in step: calls whose turns are short of bytes (several column groups on the same rows) stay with the loop.  The rule, with both sides measured: plan_block.
//
// What bounds it: over short contexts the chain of one tile (stamps, 16 / 2-head shape, 4 columns at 8000 rows, us after the first wave's entry: loads issued 2.6, K staged
// 3.8, scores 4.2, P 4.9, V staged 5.3, product 5.8, partials stored 6.6: the 64-byte pieces of 16 rows a store leave at 16 bytes a clock), over long ones the stream.
// Not kept: four row blocks at head_dim 256 (spills; 8 columns of that shape at 8191 rows 18.3 us against 14.8 in two groups), three row blocks in one group where two groups of two
// have no more than two tiles a wave (24 / 4-head shape, 8 at 8000 16.9 / 15.1).
#include "attn_tile.h"

static __device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int HD, int NB> struct BlockLds {
  typedef DecShape<HD> S;
  static constexpr int W = 4;
  static constexpr int v = W * TILE * S::KROW, p = v + W * S::STAGE, mx = p + W * NB * 1024, l = mx + W * 16 * NB * 4, bytes = l + W * 16 * NB * 4;
  // the low halves of q's first HD / 4 dims (k-steps 0 .. QL - 1), rows of LROW bytes behind the q rows
  static constexpr int QL = S::KS / 4, LROW = QL * 64 + 16;
  static_assert(16 * NB * (S::QROW + LROW) <= W * S::STAGE, "the q rows and their low halves pass through the V regions");
};

template <int HD, int NB, bool Q8>
__global__ __launch_bounds__(256, HD == 128 && NB == 2 ? 2 : 1)
void pa_block_kernel(const uint16_t* a_k_cache, uint32_t a_base_pos, uint32_t a_max_seq, uint32_t a_n_splits, uint32_t a_col_groups, uint32_t a_ncg_magic,
                     uint32_t a_ns_magic, uint32_t a_group, uint32_t a_n_kv_heads, uint32_t a_cols_per_group, uint32_t a_n_cols, AttnParams p_in) {
  // (the leading arguments repeat fields of p_in: they are preloaded into scalar registers, see attn_decode.hip)
  AttnParams p = p_in;
  p.k_cache = a_k_cache; p.base_pos = a_base_pos; p.max_seq = a_max_seq; p.n_splits = a_n_splits; p.col_groups = a_col_groups; p.ncg_magic = a_ncg_magic;
  p.ns_magic = a_ns_magic; p.group = a_group; p.n_kv_heads = a_n_kv_heads; p.cols_per_group = a_cols_per_group; p.n_cols = a_n_cols;
  typedef DecShape<HD> S;
  typedef BlockLds<HD, NB> L;
  constexpr int W = 4, DBW = S::DB / W;                              // 16-dim output blocks of a wave
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  // dispatch id i runs on XCD i % 8, which owns a contiguous range of (kv head, split, column group) items, column group fastest (attn_decode.hip)
  const uint32_t ncg = p.col_groups, total = p.n_splits * p.n_kv_heads * ncg, per = (total + 7) / 8;
  const uint32_t item = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (item >= total) return;
  const uint32_t q1 = p.ncg_magic ? __umulhi(item, p.ncg_magic) : (ncg == 1 ? item : item / ncg);
  const uint32_t q2 = p.ns_magic ? __umulhi(q1, p.ns_magic) : (p.n_splits == 1 ? q1 : q1 / p.n_splits);
  const uint32_t cg = item - q1 * ncg, sp = q1 - q2 * p.n_splits, g = q2;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t ln = lane & 15, kg = lane >> 4;
  const uint32_t G = p.group, nH = p.n_heads, g_magic = (65536u + G - 1u) / G;
  auto div_g = [&](uint32_t r) __attribute__((always_inline)) -> uint32_t { return (r * g_magic) >> 16; };      // row r is (column r / G, head r % G)
  const uint32_t c0 = cg * p.cols_per_group, ncl = min(p.cols_per_group, p.n_cols - c0), R = ncl * G;
  const uint32_t seq_max = p.base_pos + c0 + ncl;                    // rows visible to the group's last column
  const uint32_t t_begin = sp * (uint32_t)(W * TILE);                // a split's first round of tiles; one tile a wave is one round
  if (t_begin >= seq_max) return;
  const uint32_t lim = t_begin + (seq_max - t_begin + TILE - 1) / TILE * TILE, step = p.n_splits * (uint32_t)(W * TILE);
  const size_t head_rows = (size_t)p.max_seq + TILE;                 // rows of one kv head's plane, padding included
  const size_t row_bytes = (size_t)HD * 2;
  const uint32_t lrow = lane / S::LPR, voff = lrow * (uint32_t)row_bytes + (lane % S::LPR) * 16;
  const uint32_t lrow8 = lane / S::LPR8, voff8 = lrow8 * HD + (lane % S::LPR8) * 16;
  const uint32_t srow = min(lane / S::LPS, (uint32_t)TILE - 1), soff = srow * S::SPR * 4 + (lane % S::LPS) * 16;
  const unsigned char* kbase = (const unsigned char*)p.k_cache + (size_t)g * head_rows * HD * (Q8 ? 1 : 2);
  const unsigned char* vbase = (const unsigned char*)p.v_cache + (size_t)g * head_rows * HD * (Q8 ? 1 : 2);
  const unsigned char* ksbase = (const unsigned char*)(p.k_scale + (Q8 ? (size_t)g * head_rows * S::SPR : 0));
  const unsigned char* vsbase = (const unsigned char*)(p.v_scale + (Q8 ? (size_t)g * head_rows * S::SPR : 0));
  unsigned char* kst = smem + wave * TILE * S::KROW;
  unsigned char* vst = smem + L::v + wave * S::STAGE;
  float* mex = (float*)(smem + L::mx);                               // [W][16 NB]
  float* lex = (float*)(smem + L::l);
  constexpr int NL = Q8 ? S::NLD8 : S::NLD;
  u4 kr[NL], vr[NL], ksr = {0u, 0u, 0u, 0u}, vsr = {0u, 0u, 0u, 0u};
  auto load_tile = [&](u4 (&r)[NL], u4& sr, const unsigned char* base, const unsigned char* sbase, uint32_t tp) __attribute__((always_inline)) {
    if constexpr (Q8) {
#pragma unroll
      for (int i = 0; i < NL; i++) r[i] = *(const u4*)(base + ((size_t)tp + i * S::RPL8) * HD + voff8);
      sr = *(const u4*)(sbase + (size_t)tp * S::SPR * 4 + soff);
    } else {
#pragma unroll
      for (int i = 0; i < NL; i++) r[i] = *(const u4*)(base + ((size_t)tp + i * S::RPL) * row_bytes + voff);
    }
  };
  // a tile's registers -> LDS rows of `stride` bytes (int8 rows widened, their scales through the region first); rows from `live` on as zeros
  auto store_tile = [&](const u4 (&r)[NL], const u4& sr, unsigned char* st, int stride, int live) __attribute__((always_inline)) {
    if constexpr (Q8) {
      if (lane / S::LPS < TILE) *(u4*)(st + soff) = sr;
      wave_lds_fence();
      float sc[NL];
#pragma unroll
      for (int i = 0; i < NL; i++) sc[i] = *(const float*)(st + ((i * S::RPL8 + lrow8) * S::SPR + (lane % S::LPR8) / 2) * 4);
      wave_lds_fence();
#pragma unroll
      for (int i = 0; i < NL; i++) {
        h8 lo, hi;
        dq16(r[i], sc[i], lo, hi);
        if ((int)(i * S::RPL8 + lrow8) >= live) { lo = (h8){0, 0, 0, 0, 0, 0, 0, 0}; hi = lo; }       // also rows whose scale is not a number
        unsigned char* d = st + (i * S::RPL8 + lrow8) * stride + (lane % S::LPR8) * 32;
        *(h8*)d = lo; *(h8*)(d + 16) = hi;
      }
    } else {
#pragma unroll
      for (int i = 0; i < NL; i++) *(u4*)(st + (i * S::RPL + lrow) * stride + (lane % S::LPR) * 16) = r[i];
      if (live < TILE) {
        const u4 z = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int i = 0; i < NL; i++) if ((int)(i * S::RPL + lrow) >= live) *(u4*)(st + (i * S::RPL + lrow) * stride + (lane % S::LPR) * 16) = z;
      }
    }
  };
  asm volatile("" :: "s"(p.q), "s"(p.v_cache), "s"(p.q_stride), "s"(p.n_heads));
  if constexpr (Q8) asm volatile("" :: "s"(p.k_scale), "s"(p.v_scale));
  // q first (it returns first), then the first tile.  Loads are unconditional: the caches carry TILE rows of padding past max_seq; a wave without a tile
  // of its own reads the last one, whose scores are masked and whose rows are staged as zeros.
  constexpr int QPT = 16 * NB * (HD / 4) / 256;
  f4 qv[QPT];
#pragma unroll
  for (int j = 0; j < QPT; j++) {
    const uint32_t e = tid + j * 256, r = min(e / (HD / 4), R - 1), d4 = e % (HD / 4), qc = div_g(r);      // padding rows copy the last live one (masked below)
    qv[j] = *(const f4*)(p.q + (size_t)(c0 + qc) * p.q_stride + (size_t)(g * G + r - qc * G) * HD + 4 * d4);
  }
  // (a quarter of the rows' dims once more: in the threads that have them already, the low halves cost four times the instructions; 0.2 us a call)
  constexpr int QL = L::QL, QL4 = QL * 8, LPT = (16 * NB * QL4 + 255) / 256;
  f4 qlv[LPT];
#pragma unroll
  for (int j = 0; j < LPT; j++) {
    const uint32_t e = min(tid + j * 256, 16u * NB * QL4 - 1), r = min(e / QL4, R - 1), qc = div_g(r);
    qlv[j] = *(const f4*)(p.q + (size_t)(c0 + qc) * p.q_stride + (size_t)(g * G + r - qc * G) * HD + 4 * (e % QL4));
  }
  uint32_t tp = t_begin + wave * TILE;
  load_tile(kr, ksr, kbase, ksbase, min(tp, lim - TILE));
  load_tile(vr, vsr, vbase, vsbase, min(tp, lim - TILE));
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < QPT; j++) {
    const uint32_t e = tid + j * 256;
    *(h4*)(smem + L::v + e / (HD / 4) * S::QROW + e % (HD / 4) * 8) = (h4){ (_Float16)qv[j][0], (_Float16)qv[j][1], (_Float16)qv[j][2], (_Float16)qv[j][3] };
  }
  unsigned char* qlo = smem + L::v + 16 * NB * S::QROW;
#pragma unroll
  for (int j = 0; j < LPT; j++) {
    const uint32_t e = min(tid + j * 256, 16u * NB * QL4 - 1);
    float lo[4];
#pragma unroll
    for (int i = 0; i < 4; i++) lo[i] = qlv[j][i] - (float)(_Float16)qlv[j][i];
    *(h4*)(qlo + e / QL4 * L::LROW + e % QL4 * 8) = (h4){ (_Float16)lo[0], (_Float16)lo[1], (_Float16)lo[2], (_Float16)lo[3] };
  }
  uint32_t end_pos[NB];                                              // a row sees cache rows below this; 0 for padding rows
#pragma unroll
  for (int nb = 0; nb < NB; nb++) { const uint32_t r = nb * 16 + ln; end_pos[nb] = r < R ? p.base_pos + c0 + div_g(r) + 1 : 0u; }
  lds_barrier();
  h8 qf[S::KS][NB];
#pragma unroll
  for (int ks = 0; ks < S::KS; ks++)
#pragma unroll
    for (int nb = 0; nb < NB; nb++) qf[ks][nb] = *(const h8*)(smem + L::v + (nb * 16 + ln) * S::QROW + ks * 64 + kg * 16);     // (the V tiles go there, behind the loop's first barrier)

  h8 ql[QL][NB];
#pragma unroll
  for (int ks = 0; ks < QL; ks++)
#pragma unroll
    for (int nb = 0; nb < NB; nb++) ql[ks][nb] = *(const h8*)(qlo + (nb * 16 + ln) * L::LROW + ks * 64 + kg * 16);
  f4 acc[DBW][NB];
#pragma unroll
  for (int j = 0; j < DBW; j++)
#pragma unroll
    for (int nb = 0; nb < NB; nb++) acc[j][nb] = (f4){0.f, 0.f, 0.f, 0.f};
  float m_run[NB], l_run[NB];
#pragma unroll
  for (int nb = 0; nb < NB; nb++) { m_run[nb] = NEG_INF; l_run[nb] = 0.f; }

  for (uint32_t t0 = t_begin; t0 < lim; t0 += step, tp += step) {
    const bool more = t0 + step < lim;
    const uint32_t tpn = min(tp + step, lim - TILE);
    store_tile(kr, ksr, kst, S::KROW, TILE);
    if (more) load_tile(kr, ksr, kbase, ksbase, tpn);
    wave_lds_fence();
    // S^T = K Q^T, the K fragments four k-steps ahead of their MFMAs
    f4 s[2][NB];
#pragma unroll
    for (int nb = 0; nb < NB; nb++) { s[0][nb] = (f4){0.f, 0.f, 0.f, 0.f}; s[1][nb] = (f4){0.f, 0.f, 0.f, 0.f}; }
    {
      constexpr int FD = 4;
      h8 a0r[FD], a1r[FD];
      auto fetch = [&](int ks) __attribute__((always_inline)) {
        a0r[ks % FD] = *(const h8*)(kst + ln * S::KROW + ks * 64 + kg * 16);
        a1r[ks % FD] = *(const h8*)(kst + (16 + ln) * S::KROW + ks * 64 + kg * 16);
      };
#pragma unroll
      for (int ks = 0; ks < FD; ks++) fetch(ks);
#pragma unroll
      for (int ks = 0; ks < S::KS; ks++) {
        const h8 a0 = a0r[ks % FD], a1 = a1r[ks % FD];
        if (ks + FD < S::KS) fetch(ks + FD);
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
          s[0][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, qf[ks][nb], s[0][nb], 0, 0, 0);
          s[1][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, qf[ks][nb], s[1][nb], 0, 0, 0);
        }
        if (ks < QL) {
#pragma unroll
          for (int nb = 0; nb < NB; nb++) {
            s[0][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, ql[ks < QL ? ks : 0][nb], s[0][nb], 0, 0, 0);
            s[1][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, ql[ks < QL ? ks : 0][nb], s[1][nb], 0, 0, 0);
          }
        }
      }
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * FD, 0);
#pragma unroll
      for (int ks = 0; ks < S::KS; ks++) {
        if (ks + FD < S::KS) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        if (ks < QL) __builtin_amdgcn_sched_group_barrier(0x008, 4 * NB, 0);
        else __builtin_amdgcn_sched_group_barrier(0x008, 2 * NB, 0);
      }
    }
    // a lane holds row nb 16 + ln, positions tp + pb 16 + 4 kg + i (a wave past the last tile: none, end_pos is below tp)
    const uint32_t vis = tp < lim ? tp : 0xffffff00u;
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
      float mx = NEG_INF;
#pragma unroll
      for (int pb = 0; pb < 2; pb++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float x = vis + pb * 16 + 4 * kg + i < end_pos[nb] ? s[pb][nb][i] * p.scale : NEG_INF;
          s[pb][nb][i] = x;
          mx = fmaxf(mx, x);
        }
      mx = rows_max(mx);
      if (kg == 0) mex[wave * 16 * NB + nb * 16 + ln] = mx;
    }
    lds_barrier();                                                   // the waves' maxima are there, and every wave has read the last turn's V and P
    // the reference of the rows: raised (O and l rescaled) only when a maximum passes it by more than DEC_RESCALE_TH, so that P <= e^8 in f16; from the same
    // values in every wave, so all of them decide alike
    float mxs[NB];
    bool grow = false;
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
      mxs[nb] = NEG_INF;
#pragma unroll
      for (int w = 0; w < W; w++) mxs[nb] = fmaxf(mxs[nb], mex[w * 16 * NB + nb * 16 + ln]);
      grow |= mxs[nb] > m_run[nb] + DEC_RESCALE_TH;
    }
    if (__any(grow)) {
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        const float m_new = fmaxf(m_run[nb], mxs[nb]);
        const float alpha = m_new == NEG_INF ? 1.f : __expf(m_run[nb] - m_new);
        l_run[nb] *= alpha;
        m_run[nb] = m_new;
#pragma unroll
        for (int j = 0; j < DBW; j++) acc[j][nb] *= alpha;
      }
    }
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
      const float m_safe = m_run[nb] == NEG_INF ? 0.f : m_run[nb];
      h8 pf;
#pragma unroll
      for (int j = 0; j < 8; j++) pf[j] = (_Float16)__expf(s[j / 4][nb][j % 4] - m_safe);
      l_run[nb] = sum_f16(pf, l_run[nb]);
      *(h8*)(smem + L::p + ((wave * NB + nb) * 64 + lane) * 16) = pf;
    }
    store_tile(vr, vsr, vst, S::VROW, (int)seq_max - (int)min(tp, seq_max));
    if (more) load_tile(vr, vsr, vbase, vsbase, tpn);
    lds_barrier();
    // O^T += V^T P^T over the four tiles, dims [wave HD / 4, + HD / 4); V^T fragments (two transpose reads each) VD steps ahead
    {
      constexpr int NS = W * DBW, VD = 4;
      h4 lor[VD], hir[VD];
      h8 pf[W][NB];
      auto fetch = [&](int st) __attribute__((always_inline)) {
        const unsigned char* vp = smem + L::v + st / DBW * S::STAGE + (4 * kg + (ln >> 2)) * S::VROW + ((wave * DBW + st % DBW) * 16 + 4 * (ln & 3)) * 2;
        lor[st % VD] = lds_read_tr16(vp);
        hir[st % VD] = lds_read_tr16(vp + 16 * S::VROW);
      };
#pragma unroll
      for (int w = 0; w < W; w++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++) pf[w][nb] = *(const h8*)(smem + L::p + ((w * NB + nb) * 64 + lane) * 16);
#pragma unroll
      for (int st = 0; st < VD; st++) fetch(st);
#pragma unroll
      for (int st = 0; st < NS; st++) {
        const h4 lo = lor[st % VD], hi = hir[st % VD];
        if (st + VD < NS) fetch(st + VD);
        const h8 a = { lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3] };
#pragma unroll
        for (int nb = 0; nb < NB; nb++) acc[st % DBW][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, pf[st / DBW][nb], acc[st % DBW][nb], 0, 0, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, W * NB, 1);
#pragma unroll
      for (int st = 0; st < VD; st++) __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
#pragma unroll
      for (int st = 0; st < NS; st++) {
        if (st + VD < NS) __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
        __builtin_amdgcn_sched_group_barrier(0x008, NB, 1);
      }
    }
  }
  // the rows' totals: the waves' sums over their own tiles, in wave order
#pragma unroll
  for (int nb = 0; nb < NB; nb++) {
    l_run[nb] = rows_sum(l_run[nb]);
    if (kg == 0) lex[wave * 16 * NB + nb * 16 + ln] = l_run[nb];
  }
  uint32_t rc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; nb++) rc[nb] = div_g(nb * 16 + ln);
  lds_barrier();
#pragma unroll
  for (int nb = 0; nb < NB; nb++) {
    const uint32_t r = nb * 16 + ln;
    if (r >= R) continue;
    float lr = 0.f;
#pragma unroll
    for (int w = 0; w < W; w++) lr += lex[w * 16 * NB + r];
    const size_t slot = ((size_t)(c0 + rc[nb]) * nH + g * G + r - rc[nb] * G) * p.slots + sp;
#pragma unroll
    for (int j = 0; j < DBW; j++) *(f4*)(p.part_o + slot * HD + (wave * DBW + j) * 16 + 4 * kg) = acc[j][nb];
    if (wave == 0 && kg == 0) *(float2*)(p.part_ml + slot * 2) = make_float2(m_run[nb], lr);
  }
}

template <int HD, int NB, bool Q8>
static hipError_t launch_block_t(const AttnParams& p, uint32_t col_groups, hipStream_t s, const PaTiming* t) {
  static PaPerDevice lds_set;
  const size_t lds = BlockLds<HD, NB>::bytes;
  static_assert(BlockLds<HD, NB>::bytes <= 160 * 1024 && (HD == 256 || NB > 2 || 2 * BlockLds<HD, NB>::bytes <= 160 * 1024), "workgroups a CU");
  const hipError_t e = pa_lds_limit(lds_set, (const void*)pa_block_kernel<HD, NB, Q8>, lds);
  if (e != hipSuccess) return e;
  if (col_groups != (p.n_cols + p.cols_per_group - 1) / p.cols_per_group || p.cols_per_group * p.group > 16 * NB) return hipErrorInvalidValue;
  AttnParams pk = p;
  const uint64_t total = (uint64_t)p.n_splits * p.n_kv_heads * col_groups;
  auto magic = [&](uint32_t d) -> uint32_t { return d > 1 && total * d < (1ull << 32) ? (uint32_t)(((1ull << 32) + d - 1) / d) : 0u; };
  PA_LAUNCH((pa_block_kernel<HD, NB, Q8>), dim3((unsigned)((total + 7) / 8 * 8)), dim3(256), lds, s, t, p.k_cache, p.base_pos, p.max_seq, p.n_splits, col_groups,
            magic(col_groups), magic(p.n_splits), p.group, p.n_kv_heads, p.cols_per_group, p.n_cols, pk);
  return hipGetLastError();
}

template <int HD, bool Q8>
static hipError_t launch_block_nb(const AttnParams& p, uint32_t nb, uint32_t col_groups, hipStream_t s, const PaTiming* t) {
  switch (nb) {
    case 2: return launch_block_t<HD, 2, Q8>(p, col_groups, s, t);
    case 3: return launch_block_t<HD, 3, Q8>(p, col_groups, s, t);
    case 4: if constexpr (HD == 128) return launch_block_t<HD, 4, Q8>(p, col_groups, s, t); else return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}

hipError_t pa_launch_block(const AttnParams& p, uint32_t hd, uint32_t nb, uint32_t col_groups, hipStream_t s, const PaTiming* t) {
  if (p.self_row || p.sel || p.part_f16 || p.direct_out || p.exact_cols || (p.split_len != 128 && p.tile_ilv != 128)) return hipErrorInvalidValue;
  if (hd == 256) return p.k_scale ? launch_block_nb<256, true>(p, nb, col_groups, s, t) : launch_block_nb<256, false>(p, nb, col_groups, s, t);
  if (hd == 128) return p.k_scale ? launch_block_nb<128, true>(p, nb, col_groups, s, t) : launch_block_nb<128, false>(p, nb, col_groups, s, t);
  return hipErrorInvalidValue;
}

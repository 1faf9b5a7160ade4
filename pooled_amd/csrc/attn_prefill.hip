// Causal prefill attention on f16 MFMA for gfx950 (MI355X).
//
// Replaces the reference's attn_flash_tile + attn_combine_tile + sigmoid_mul_mc
// (engine/wgsl/attn_tile.js:108-193, engine/wgsl/qwen35.js:877-887): a chunk of n_cols query columns at absolute
// positions base_pos + c attends causally to the f16 KV cache rows [0, base_pos + c].  One launch covers what
// the reference runs as consecutive 16-column passes.
//
// Work decomposition
//   * A workgroup owns one kv head and a block of columns; its 256 query rows are (column, head-in-group) pairs,
//     so every K/V tile it stages serves all G heads of the group (the reference's "up to 64 rows share a tile",
//     scaled to the MFMA shape).  8 wavefronts x 32 rows, two per SIMD: while one wave of a SIMD does its softmax
//     on the VALU the other one's MFMAs keep the matrix pipe busy.
//   * K/V tiles of 32 positions go global -> LDS directly (global_load_lds_dwordx4: no staging registers),
//     double buffered, one barrier a step; the next tile's loads are in flight while the current one is consumed.
//     An LDS-direct load writes 64 lanes x 16 B contiguously, so rows cannot be padded; bank conflicts are
//     avoided by an XOR swizzle applied on the *global* side (lane i fetches the chunk that belongs at its LDS
//     slot): K chunk c of row r sits at slot c ^ (r & 15) (conflict-free ds_read_b128 fragments), V chunk c at
//     c ^ 4 (r & 3) ^ 2 (r / 4 & 1) (2-way = optimal ds_read_b64_tr_b16).  Rows at or past the end of the context are fetched
//     from the cache's zero padding row instead, so 0 x stale bits never reaches O.
//   * S^T = K Q^T and O^T = V^T P^T on v_mfma_f32_16x16x32_f16, a wave's 32 rows as two blocks of 16.  Q fragments stay in registers for the
//     whole kernel; K fragments are ds_read_b128, V^T fragments come from the gfx950 LDS transpose read (ds_read_b64_tr_b16), each feeding
//     both blocks.  The S^T accumulator layout (lane = query row, 4 + 4 positions) is the B-operand layout of the PV product, so P never leaves
//     registers.  On a full chip of head_dim 256 the kernel runs at the power limit, where this shape has the better rate (products alone
//     on random operands: 1.73 - 1.80 PFLOP/s against 1.65 on 32 x 32 x 16), as long as the softmax's two rows a lane cost no
//     more than one did:
//   * Online softmax in f32 in the exp2 domain with a lazily updated reference maximum: O and l are rescaled only when a P comes out above 2^8
//     (exact enough in f16), which takes the 128-register O rescale, and with it every row maximum, off the common path: what is
//     looked at is the packed P itself, seven maxima a tile, and a tile that fails is taken again with raised references.  Row maxima of
//     every tile: 4 % slower at head_dim 256, 7 - 10 % at 128.
//     Both steps together against 32 x 32 x 16 with row maxima (us, 16 / 2-head shape): 4096 columns at 64K 3708 -> 3325, at 8192 658 -> 598, 2500
//     at 16384 (158 workgroups: below the limit) 778 -> 761; 16 / 8-head shape, 4096 at 28000 972 -> 878, 2500 at 8192 276 -> 272; 777 of the 24 / 4-head
//     shape at 5003, split, 142 -> 133.  Fragments three ahead in both products: two of K are 1 - 2 % slower, four spill.
//   * Workgroup ids are remapped so that each XCD (ids are dealt round-robin to the 8 XCDs) works on one
//     contiguous range of (kv head, column block): the K/V stream of a kv head is fetched into one L2.
//   * PAIRED (unsplit passes of one round whose chunk is a material part of the context, the rule at pairs_pay): waves 0-3 take a
//     half block of columns from the front of the chunk, waves 4-7 the one as far from its back, so that every workgroup has the same
//     work and the causal triangle of a chunk at the start of a prompt does not leave most CUs idle behind the last columns'
//     workgroups (with one block of neighbouring columns a workgroup, 4096 columns from 0 of the 16 / 2-head shape 190 us, paired 155 us: 128
//     steps at the pace of one wave a SIMD, which is some 0.7 of two waves').  Where half blocks would need a workgroup more than whole
//     ones, the blocks stay whole.
//   * Unsplit passes of more workgroups than CUs keep whole blocks (halves that end apart run one wave a SIMD for a while: more work
//     in all), dealt over the XCDs of a kv head in turn, the longest first.  In order of position, one XCD of a head had the front of the
//     triangle and another the back, the longest blocks last: 4096 columns of the 24 / 4-head shape from 0 420 -> 315 us, 3000 at
//     3000 567 -> 454.
//   * Optional split over the context (short chunks on long contexts would otherwise leave CUs idle): partial
//     (m, l, O) go to the same buffers the decode kernel uses and the same merge kernel finishes them.
#include "pf_common.h"

template <int HD, int W> struct PfShape {
  static constexpr int ROWB = HD * 2;             // bytes of one kv head's row
  static constexpr int TILE = PF_TN * ROWB;       // bytes of one staged tile (K or V)
  static constexpr int KS = HD / 32;              // k-steps of QK^T
  static constexpr int DB = HD / 16;              // 16-dim blocks of the output
  static constexpr int CPR = HD / 8;              // 16-byte chunks per row
  static constexpr int RPB = 64 / CPR;            // rows per 1 KB LDS-direct load
  static constexpr int NLD = PF_TN / RPB / W;   // LDS-direct loads per wave, tensor and step
  static_assert(NLD >= 1 && NLD * W * RPB == PF_TN, "tile must divide evenly over the waves");
};

template <int HD, int W, bool PAIRED>
__global__ __launch_bounds__(W * 64, W / 4) void pa_prefill_kernel(AttnParams p, uint32_t n_col_blocks, uint32_t half_cols, uint32_t head_xcds) {
  typedef PfShape<HD, W> S;
  constexpr int NB = 2;                            // 16-row blocks of a wave
  // four separate LDS objects (two K, two V buffers): the compiler then orders an LDS read only after the
  // LDS-direct loads into the *same* buffer, and the prefetch into the other buffer stays in flight
  __shared__ __attribute__((aligned(1024))) unsigned char kbuf0[S::TILE];
  __shared__ __attribute__((aligned(1024))) unsigned char kbuf1[S::TILE];
  __shared__ __attribute__((aligned(1024))) unsigned char vbuf0[S::TILE];
  __shared__ __attribute__((aligned(1024))) unsigned char vbuf1[S::TILE];

  // ---- XCD-aware id -> (kv head, split, column block) ----
  // Work items are (kv head, split, column block), column block fastest: the workgroups of one (kv head, split) read
  // the same K/V rows.  The grid is one-dimensional; dispatch id i runs on XCD i % 8, and XCD k owns the contiguous
  // item range [k per_xcd, (k + 1) per_xcd): every XCD gets the same number of workgroups whatever the split count,
  // and the workgroups that share a K/V stream share an L2.
  // head_xcds (unsplit passes of whole blocks): the XCDs of a kv head take its column blocks in turn, the longest first.
  uint32_t cb, sp, g;
  if (head_xcds) {
    const uint32_t xcd = blockIdx.x % 8, i = blockIdx.x / 8 * head_xcds + xcd % head_xcds;
    if (i >= n_col_blocks) return;
    cb = n_col_blocks - 1 - i; sp = 0; g = xcd / head_xcds;
  } else {
    const uint32_t total = n_col_blocks * p.n_kv_heads * p.n_splits;
    const uint32_t per_xcd = (total + 7) / 8;
    const uint32_t lid = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (lid >= total) return;
    cb = lid % n_col_blocks; sp = (lid / n_col_blocks) % p.n_splits; g = lid / (n_col_blocks * p.n_splits);
  }

  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform (scalar) so per-wave branches are scalar branches
  const uint32_t ln = lane & 15, kg = lane >> 4;    // MFMA row / column index, k group
  const uint32_t G = p.group, nH = p.n_heads;
  // r / G as a multiply and a shift (exact for r < 1024 and G <= 64)
  const uint32_t g_magic = (65536u + G - 1u) / G;
  auto div_g = [&](uint32_t r) __attribute__((always_inline)) -> uint32_t { return (r * g_magic) >> 16; };
  // the lane, counted anew: what depends on it is not kept in registers across the code before
  auto fresh_lane = []() __attribute__((always_inline)) -> uint32_t {
    uint32_t l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
  };
  // columns of this WAVE [c0, c0 + R / G): the workgroup's block, or (PAIRED) its half's block: waves of the lower half
  // take block cb from the front, the others the one as far from the back, so that every workgroup has the same work
  uint32_t c0 = cb * p.cols_per_group, wrow0 = wave * 32;       // wrow0: the wave's first row in its block
  uint32_t ncl = min(p.cols_per_group, p.n_cols - c0), c_end = c0 + ncl;
  if constexpr (PAIRED) {
    const uint32_t n_half = (p.n_cols + half_cols - 1) / half_cols, far = n_half - 1 - cb;
    const bool lower = wave < W / 2;
    c0 = (lower ? cb : far) * half_cols;
    if (!lower) wrow0 -= W / 2 * 32;
    c_end = min((far + 1) * half_cols, p.n_cols);
    ncl = min(half_cols, p.n_cols - c0);
    if (far == cb && lower) ncl = 0;               // an odd number of blocks: the middle one is alone
  }
  const uint32_t R = ncl * G;                      // live rows (<= 32 W)
  const uint32_t seq_max = p.base_pos + c_end;     // rows visible to the workgroup's last column
  const uint32_t t_begin = sp * p.split_len;
  if (t_begin >= seq_max) return;
  const uint32_t t_end = min(t_begin + p.split_len, seq_max);
  const uint32_t n_steps = (t_end - t_begin + PF_TN - 1) / PF_TN;
  const size_t row_bytes = (size_t)HD * 2;                       // head-major caches: a kv head's rows are contiguous
  const size_t head_rows = (size_t)p.max_seq + PF_TN;            // rows of one kv head's plane, padding included
  const unsigned char* kg_base = (const unsigned char*)(p.k_cache + (size_t)g * head_rows * HD);
  const unsigned char* vg_base = (const unsigned char*)(p.v_cache + (size_t)g * head_rows * HD);

  // ---- LDS-direct tile loads: load i of wave w fills the 1 KB block i W + w of a buffer, i.e. rows (i W + w) RPB ..;
  //      lane l of a block lands at (row l / CPR, slot l % CPR) and therefore fetches chunk slot ^ swizzle(row) of
  //      that row.  W RPB is a multiple of 16, so the swizzle -- and with it the lane's byte offset from the block's
  //      first row -- is the same for every i and every tile: one 32-bit offset per tensor, the rest of the address
  //      is wave-uniform (scalar registers) ----
  static_assert((W * S::RPB) % 16 == 0, "the swizzle must not depend on the load index");
  const uint32_t ld_row0 = wave * S::RPB + lane / S::CPR, ld_slot = lane % S::CPR;
  auto k_slot = [&](uint32_t row, uint32_t slot) { return slot ^ (row & 15); };
  auto v_slot = [&](uint32_t row, uint32_t slot) { return slot ^ (4 * (row & 3)) ^ (2 * ((row >> 2) & 1)); };
  auto k_off_of = [&](uint32_t row0, uint32_t slot) { return row0 * (uint32_t)row_bytes + k_slot(row0, slot) * 16; };
  auto v_off_of = [&](uint32_t row0, uint32_t slot) { return row0 * (uint32_t)row_bytes + v_slot(row0, slot) * 16; };
  const uint32_t k_off = k_off_of(ld_row0, ld_slot), v_off = v_off_of(ld_row0, ld_slot);
  constexpr uint32_t LD_STRIDE = W * S::RPB * S::ROWB;           // bytes between the rows of consecutive loads
  // Rows at or past t_end (only in the last tile of the context) come from the zero padding row max_seq; their addresses are worked out
  // there and one load at a time, so that nothing of them takes registers in the loop.
  auto issue = [&](unsigned char* kdst, unsigned char* vdst, const uint32_t tpos, const uint32_t ko, const uint32_t vo) __attribute__((always_inline)) {
    if (tpos + PF_TN <= t_end) {
      const unsigned char* kt = kg_base + (size_t)tpos * row_bytes;
      const unsigned char* vt = vg_base + (size_t)tpos * row_bytes;
#pragma unroll
      for (int i = 0; i < S::NLD; i++) PF_GLL_S(kt + i * LD_STRIDE, ko, kdst + (i * W + wave) * 1024);
#pragma unroll
      for (int i = 0; i < S::NLD; i++) PF_GLL_S(vt + i * LD_STRIDE, vo, vdst + (i * W + wave) * 1024);
    } else {
      const uint32_t l = fresh_lane(), row0 = wave * S::RPB + l / S::CPR, slot = l % S::CPR;
#pragma unroll
      for (int i = 0; i < S::NLD; i++) {
        const uint32_t row = tpos + i * W * S::RPB + row0;
        const size_t at = (size_t)(row < t_end ? row : p.max_seq) * row_bytes;
        PF_GLL(kg_base + at + k_slot(row0, slot) * 16, kdst + (i * W + wave) * 1024);
        PF_GLL(vg_base + at + v_slot(row0, slot) * 16, vdst + (i * W + wave) * 1024);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  issue(kbuf0, vbuf0, t_begin, k_off, v_off);

  // ---- per-lane rows: row r = wrow0 + 16 nb + ln of the wave's block of columns = (column c0 + r / G, head r % G) ----
  uint32_t w_min_end = 0xffffffffu, w_max_end = 0;                // positions seen by the wave's first row, by its last one
  if (wrow0 < R) { w_min_end = p.base_pos + c0 + div_g(wrow0) + 1; w_max_end = p.base_pos + c0 + div_g(min(wrow0 + NB * 16 - 1, R - 1)) + 1; }

  // ---- Q fragments (B operand of S^T = K Q^T): row ln of block nb, dims 32 ks + 8 kg .. + 7, as f16, in registers for the whole kernel ----
  h8 qf[NB][S::KS];
#pragma unroll
  for (int nb = 0; nb < NB; nb++) {
    const uint32_t r = wrow0 + nb * 16 + ln, rc = !PAIRED || R ? min(r, R - 1) : 0;
    const uint32_t qc = div_g(rc);
    const float* qrow = p.q + (size_t)(c0 + qc) * p.q_stride + (size_t)(g * G + rc - qc * G) * HD + 8 * kg;
#pragma unroll
    for (int ks = 0; ks < S::KS; ks++) {
      const f4 a = *(const f4*)(qrow + 32 * ks), b = *(const f4*)(qrow + 32 * ks + 4);
      qf[nb][ks] = (h8){ (_Float16)a[0], (_Float16)a[1], (_Float16)a[2], (_Float16)a[3],
                         (_Float16)b[0], (_Float16)b[1], (_Float16)b[2], (_Float16)b[3] };
    }
  }

  f4 acc[S::DB][NB];
#pragma unroll
  for (int db = 0; db < S::DB; db++)
#pragma unroll
    for (int nb = 0; nb < NB; nb++) acc[db][nb] = (f4){0.f, 0.f, 0.f, 0.f};
  float m_ref[NB], l_run[NB];
#pragma unroll
  for (int nb = 0; nb < NB; nb++) { m_ref[nb] = wrow0 + nb * 16 + ln < R ? NEG_INF : 0.f; l_run[nb] = 0.f; }   // (rows past the last: never counted as unseen)
  bool unseen = true;
  const float c1 = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(p.scale * 1.4426950408889634f)));   // scores -> log2 domain (scalar)

  // per-lane LDS read offsets with the swizzles folded in (buffer bases are 1 KB aligned, so XOR == add on the
  // swizzled bits, 256 bytes of a row): K fragment of k-step ks is at k_rd ^ (ks * 64); V fragment of dim block db at v_rd ^ (db * 32)
  const uint32_t k_rd = ln * S::ROWB + (kg ^ ln) * 16;
  const uint32_t v_rd = (4 * kg + (ln >> 2)) * S::ROWB + (((ln & 3) >> 1) ^ (4 * (ln >> 2)) ^ (2 * (kg & 1))) * 16 + (ln & 1) * 8;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  // The three phases of a tile.  s (raw scores) lives from qk to sm, pf (f16 probabilities) from sm to pv.
  f4 s[2][NB];
  h8 pf[NB];
  // ---- S^T = K Q^T : rows = 2 x 16 positions, columns = 16 query rows per block ----
  auto qk = [&](const unsigned char* kb, const uint32_t tp) {
#pragma unroll
    for (int pb = 0; pb < 2; pb++)
#pragma unroll
      for (int nb = 0; nb < NB; nb++) s[pb][nb] = (f4){0.f, 0.f, 0.f, 0.f};
    // fragment f = positions 16 (f % 2) .., k-step f / 2; fetched KD fragments ahead of the MFMAs that consume them
    constexpr int KD = PF_KD, NF = 2 * S::KS;
    h8 ka[KD];
    auto at = [&](int f) { return kb + (k_rd ^ (f / 2 % 4 * 64)) + f / 8 * 256 + f % 2 * 16 * S::ROWB; };
#pragma unroll
    for (int f = 0; f < KD; f++) ka[f] = *(const h8*)at(f);
#pragma unroll
    for (int f = 0; f < NF; f++) {
      const h8 a = ka[f % KD];
      if (f + KD < NF) ka[f % KD] = *(const h8*)at(f + KD);
#pragma unroll
      for (int nb = 0; nb < NB; nb++) s[f % 2][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, qf[nb][f / 2], s[f % 2][nb], 0, 0, 0);
    }
    // pin the issue order the source states: the first KD fetches up front, then each fragment's successor behind its MFMAs
#pragma unroll
    for (int f = 0; f < KD; f++) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
#pragma unroll
    for (int f = 0; f < NF; f++) {
      __builtin_amdgcn_sched_group_barrier(0x008, NB, 0);
      if (f + KD < NF) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
  };
  // ---- online softmax; lane holds query row ln of each block, positions tp + 16 pb + 4 kg + i ----
  // Raw scores stay unscaled: the scale rides in the exp2 argument (one fma per element), the row sum is a
  // v_dot2 over the f16-rounded probabilities (the values PV really uses), and the mask is a separate pass
  // that only tiles straddling a row end execute.
  auto sm = [&](const uint32_t tp) {
    if (tp + PF_TN > w_min_end) {
      // (volatile: keeps this a branch -- most tiles skip the 3 ops per element -- and what it works out in it)
      const uint32_t l = fresh_lane();
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        const uint32_t r = wrow0 + nb * 16 + (l & 15), end_pos = r < R ? p.base_pos + c0 + div_g(r) + 1 : 0u;
#pragma unroll
        for (int pb = 0; pb < 2; pb++)
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const uint32_t pos = tp + 16 * pb + 4 * (l >> 4) + i;
            s[pb][nb][i] = pos < end_pos ? s[pb][nb][i] : NEG_INF;
          }
      }
    }
    // P against the reference maxima as they are; where one of the wave's comes out above 2^PF_RESCALE_TH (on the packed values, seven maxima
    // a tile instead of the rows' own), the references are raised and P is taken again, below 1 this time.  So no row maximum is worked out on
    // the common path -- but on a wave's first tile, and for as long as one of its rows has seen nothing (a split before the row's end).
    auto raise = [&]() __attribute__((always_inline)) {
      bool none = false;
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        float mx = fmaxf(s[0][nb][0], s[0][nb][1]);
        mx = fmaxf(fmaxf(mx, s[0][nb][2]), s[0][nb][3]);
        mx = fmaxf(fmaxf(mx, s[1][nb][0]), s[1][nb][1]);
        mx = fmaxf(fmaxf(mx, s[1][nb][2]), s[1][nb][3]);
        const auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = fmaxf(__uint_as_float(s16[0]), __uint_as_float(s16[1]));
        const auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        const float m_new = fmaxf(m_ref[nb], fmaxf(__uint_as_float(s32[0]), __uint_as_float(s32[1])) * c1);   // all four position groups of the row, log2 domain
        const float alpha = m_new == NEG_INF ? 1.f : __builtin_amdgcn_exp2f(m_ref[nb] - m_new);
        m_ref[nb] = m_new;
        l_run[nb] *= alpha;
        none |= m_new == NEG_INF;
#pragma unroll
        for (int db = 0; db < S::DB; db++) acc[db][nb] *= alpha;
      }
      unseen = __any(none);
    };
    auto probs = [&]() __attribute__((always_inline)) -> bool {
      h2 top = { (_Float16)0.f, (_Float16)0.f };
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        const float nmr = m_ref[nb] == NEG_INF ? 0.f : -m_ref[nb];
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
          const float e0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[j / 4][nb][j % 4], c1, nmr));
          const float e1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[j / 4][nb][j % 4 + 1], c1, nmr));
          const h2 pp = { (_Float16)e0, (_Float16)e1 };
          top = __builtin_elementwise_max(top, pp);
          pf[nb][j] = pp[0]; pf[nb][j + 1] = pp[1];
        }
      }
      const _Float16 lim = (_Float16)(float)(1 << PF_RESCALE_TH);
      return __any(top[0] > lim || top[1] > lim);
    };
    if (__builtin_expect(unseen, 0)) raise();
    if (__builtin_expect(probs(), 0)) { raise(); probs(); }
    const h2 ones = { (_Float16)1.f, (_Float16)1.f };
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
#pragma unroll
      for (int j = 0; j < 8; j += 2) { const h2 pp = { pf[nb][j], pf[nb][j + 1] }; l_run[nb] = __builtin_amdgcn_fdot2(pp, ones, l_run[nb], false); }
    }
  };
  // ---- O^T += V^T P^T : rows = 16 dims a block, contraction over the 32 positions (slot 8 kg + j: position 4 kg + j, or 16 + 4 kg + j - 4) ----
  auto pv = [&](const unsigned char* vb, const uint32_t tp) {
    // dim block db's fragment is fetched VD blocks ahead
    constexpr int VD = PF_VD;
    h4 vlo[VD], vhi[VD];
    auto at = [&](int f) { return vb + (v_rd ^ (f % 8 * 32)) + f / 8 * 256; };
#pragma unroll
    for (int f = 0; f < VD; f++) {
      const unsigned char* vp = at(f);
      vlo[f] = lds_read_tr16(vp);
      vhi[f] = lds_read_tr16(vp + 16 * S::ROWB);
    }
#pragma unroll
    for (int f = 0; f < S::DB; f++) {
      const h4 lo = vlo[f % VD], hi = vhi[f % VD];
      if (f + VD < S::DB) {
        const unsigned char* vp = at(f + VD);
        vlo[f % VD] = lds_read_tr16(vp);
        vhi[f % VD] = lds_read_tr16(vp + 16 * S::ROWB);
      }
      const h8 a = { lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3] };
#pragma unroll
      for (int nb = 0; nb < NB; nb++) acc[f][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, pf[nb], acc[f][nb], 0, 0, 0);
    }
#pragma unroll
    for (int f = 0; f < VD; f++) __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
#pragma unroll
    for (int f = 0; f < S::DB; f++) {
      __builtin_amdgcn_sched_group_barrier(0x008, NB, 1);
      if (f + VD < S::DB) __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
    }
  };

  // ---- main loop ----
  // From its step n_live on a wave has no row left: it only stages its share of the remaining tiles.  Every wave passes n_steps barriers,
  // whichever loop it is in.  PAIRED: that is the near half of a pair.  Whole blocks: the waves past the last block's rows, from the start
  // (split passes, those waves computing / not: 24 / 4-head shape at 50000, 130 columns 214 / 205 us, 88 columns 170 / 160); a wave whose
  // rows end a tile before the workgroup's computes it, as an end of its own costs 0.3 % of a long pass.
  // It is a loop of its own: with the compute under a branch instead, the loop's blocks end where the compiler overlaps the end of a tile
  // with the start of the next (us, branch / two loops, pairs: 4096 columns at 8192 666 / 665, at 16384 1113 / 1108, at 64K 3833 / 3811).
  // For pairs at head_dim 128 the branch is the cheaper form (4096 columns at 28K 946 against 951, 2500 at 8192 253 against 257).
  constexpr bool TWO_LOOPS = !PAIRED || HD == 256;
  const uint32_t n_live = !PAIRED ? (wrow0 < R ? n_steps : 0u) : !TWO_LOOPS ? n_steps : w_max_end > t_begin ? min((w_max_end - t_begin + PF_TN - 1) / PF_TN, n_steps) : 0u;
  const uint32_t n_even = n_live & ~1u;
  uint32_t lane_e = lane;
  {
    // all waves in phase: QK, softmax, PV of a tile between two barriers (tile i + 1 of both K and V in flight)
    auto step_s = [&](auto PAR, const uint32_t i) {
      constexpr int par = decltype(PAR)::value;
      const uint32_t tp = t_begin + i * PF_TN;
      if (i + 1 < n_steps) issue(par ? kbuf0 : kbuf1, par ? vbuf0 : vbuf1, tp + PF_TN, k_off, v_off);
      if (TWO_LOOPS || tp < w_max_end) {
        qk(par ? kbuf1 : kbuf0, tp);
        sm(tp);
        pv(par ? vbuf1 : vbuf0, tp);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    };
    for (uint32_t i = 0; i < n_even; i += 2) {
      step_s(std::integral_constant<int, 0>{}, i);
      step_s(std::integral_constant<int, 1>{}, i + 1);
    }
    if (n_live & 1) step_s(std::integral_constant<int, 0>{}, n_even);
    if constexpr (HD == 256) {
      lane_e = fresh_lane();
    }
    if constexpr (TWO_LOOPS) {
      const uint32_t d_row0 = wave * S::RPB + lane_e / S::CPR, d_slot = lane_e % S::CPR;
      for (uint32_t i = n_live; i < n_steps; i++) {
        const uint32_t tp = t_begin + i * PF_TN;
        if (i + 1 < n_steps) issue(i & 1 ? kbuf0 : kbuf1, i & 1 ? vbuf0 : vbuf1, tp + PF_TN, k_off_of(d_row0, d_slot), v_off_of(d_row0, d_slot));
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
      }
    }
  }

  // ---- epilogue ----
  const uint32_t ln_e = lane_e & 15, kg_e = lane_e >> 4;
#pragma unroll
  for (int nb = 0; nb < NB; nb++) {
    l_run[nb] += __shfl_xor(l_run[nb], 16, 64);
    l_run[nb] += __shfl_xor(l_run[nb], 32, 64);
    const uint32_t r = wrow0 + nb * 16 + ln_e;
    if (r >= R) continue;
    const uint32_t rc = div_g(r), col = c0 + rc, hq = g * G + r - rc * G;
    if (p.n_splits == 1) {
      // the whole context was seen: normalise, gate, convert, store
      const float inv_l = 1.f / l_run[nb];
      const float* gate = p.gate ? p.gate + (size_t)col * p.gate_stride + (size_t)hq * HD : nullptr;
#pragma unroll
      for (int db = 0; db < S::DB; db++) {
        const uint32_t d = 16 * db + 4 * kg_e;
        f4 o = acc[db][nb] * inv_l;
        if (gate) {
          const f4 gt = *(const f4*)(gate + d);
#pragma unroll
          for (int i = 0; i < 4; i++) o[i] *= 1.f / (1.f + __expf(-gt[i]));
        }
        if (p.out_f16) {
          const h4 hv = { (_Float16)o[0], (_Float16)o[1], (_Float16)o[2], (_Float16)o[3] };
          *(h4*)((_Float16*)p.out + (size_t)col * p.out_stride + (size_t)hq * HD + d) = hv;
        } else {
          *(f4*)((float*)p.out + (size_t)col * p.out_stride + (size_t)hq * HD + d) = o;
        }
      }
    } else {
      // split partial: un-normalised O, m in natural-log units of the scaled scores, l
      const size_t slot = ((size_t)col * nH + hq) * p.slots + sp;
#pragma unroll
      for (int db = 0; db < S::DB; db++) *(f4*)(p.part_o + slot * HD + 16 * db + 4 * kg_e) = acc[db][nb];
      if (kg_e == 0) {
        p.part_ml[slot * 2] = m_ref[nb] * 0.6931471805599453f;
        p.part_ml[slot * 2 + 1] = l_run[nb];
      }
    }
  }
}

template <int HD, int W, bool PAIRED>
static hipError_t launch_prefill_k(const AttnParams& p, uint32_t col_groups, uint32_t half, uint32_t head_xcds, hipStream_t s, const PaTiming* t) {
  const uint32_t total = col_groups * p.n_kv_heads * p.n_splits;
  const uint32_t gx = 8 * (head_xcds ? (col_groups + head_xcds - 1) / head_xcds : (total + 7) / 8);       // whole rounds of the 8 XCDs
  PA_LAUNCH((pa_prefill_kernel<HD, W, PAIRED>), dim3(gx), dim3(W * 64), 0, s, t, p, col_groups, half, head_xcds);
  return hipGetLastError();
}

// Whether an unsplit pass of one round is paired.  Pairing takes the wait for the longest block away (n_cols / 2 positions at
// most) and pays for it in energy: every pair stages tiles up to its far half's end, and halves that end apart run one wave a SIMD
// for a while.  At head_dim 256 a full chip runs at the power limit, so once the triangle is a small part of the context pairs are at
// most as fast.  Measured (us, whole blocks / pairs, with the pre-step): 256 workgroups, 4096 columns of the 16 / 2-head shape at 0 244 / 209, at 8192
// 614 / 587, at 16384 979 / 965, at 32768 1748 / 1733, at 124K 6286 / 6269; 2650 columns of the 24 / 4-head shape at 4096 370 / 356, at 8192 555 / 551, at
// 16384 927 / 929; 158 workgroups, 2500 columns of the first at 8192 456 / 440, at 16384 763 / 754, at 32768 1387 / 1386, at 64K 2618 / 2646.
// Head_dim 128 stays ahead (4096 columns at 28672 920 / 888).
static bool pairs_pay(uint32_t hd, uint32_t base_pos, uint32_t n_cols, uint32_t total, uint32_t n_cu) {
  return hd == 128 || (uint64_t)base_pos * total <= 6ull * n_cols * n_cu;
}
extern "C" int pa_rule_prefill_paired(uint32_t hd, uint32_t base_pos, uint32_t n_cols, uint32_t group, uint32_t n_kv_heads, uint32_t n_splits, uint32_t col_groups, uint32_t n_cu) {
  const uint32_t half = PF_ROWS / 2 / group, total = col_groups * n_kv_heads * n_splits;
  return n_splits == 1 && half > 0 && total <= n_cu && ((n_cols + half - 1) / half + 1) / 2 == col_groups && pairs_pay(hd, base_pos, n_cols, total, n_cu);
}

template <int HD, int W>
static hipError_t launch_prefill_t(const AttnParams& p, uint32_t col_groups, uint32_t n_cu, hipStream_t s, const PaTiming* t) {
  static_assert(W * 32 == PF_ROWS, "the rule's rows of a workgroup");
  if (pa_rule_prefill_paired(HD, p.base_pos, p.n_cols, p.group, p.n_kv_heads, p.n_splits, col_groups, n_cu))
    return launch_prefill_k<HD, W, true>(p, col_groups, PF_ROWS / 2 / p.group, 0, s, t);
  // more workgroups than the chip holds at once: the longest blocks first
  const uint32_t head_xcds = p.n_splits == 1 && col_groups * p.n_kv_heads > n_cu && 8 % p.n_kv_heads == 0 ? 8 / p.n_kv_heads : 0;
  return launch_prefill_k<HD, W, false>(p, col_groups, 0, head_xcds, s, t);
}

// row_blocks = 32-row query blocks per workgroup (8: one per wavefront)
hipError_t pa_launch_prefill(const AttnParams& p, uint32_t hd, uint32_t row_blocks, uint32_t col_groups, uint32_t n_cu, hipStream_t s, const PaTiming* t) {
  if (row_blocks != 8) return hipErrorNotSupported;
  if (hd == 256) return launch_prefill_t<256, 8>(p, col_groups, n_cu, s, t);
  if (hd == 128) return launch_prefill_t<128, 8>(p, col_groups, n_cu, s, t);
  return hipErrorNotSupported;
}

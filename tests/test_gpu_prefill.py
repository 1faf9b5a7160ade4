"""GPU parity of causal prefill attention (MFMA kernel) through the C ABI against the CPU oracle.
Tolerance: max-abs <= 2e-3 and max|d|/max|ref| <= 1e-2 of the f32/f64 reference."""
import numpy as np
import pytest
from oracle import attn_oracle as O
from oracle import c_oracle as C
from pooled_amd import capi
from pooled_amd.capi import PooledAttn, PA_OUT_F16
from helpers import SHAPES, assert_parity, random_cache, oracle_cache

pytestmark = pytest.mark.gpu
NAN16 = 0x7E00


def _prefill(cfg, base, n, seed, max_seq=None, gate=True, out_dtype=0, check_rows=None, k_scale=1.0, tile=1):
    """tile: pa_set_prefill_tile mode -- 1 (default here) forces the matrix-core kernel, which the table would not pick
    for the small chunks most of these cases are; 0 = the table's choice."""
    rng = np.random.default_rng(seed)
    max_seq = max_seq or base + n + 7
    k16, v16 = random_cache(cfg, max_seq, seed=seed + 1, k_scale=k_scale)
    q = rng.standard_normal((n, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32)
    gt = rng.standard_normal(q.shape, dtype=np.float32) if (gate and cfg["gate"]) else None
    rows = check_rows if check_rows is not None else list(range(n))
    ref = C.attention(q, k16, v16, base, gate=gt, rows=rows)
    pa = PooledAttn(cfg, max_seq, n_layers=1, max_cols=n)
    try:
        pa.layer_alloc(0)
        K, V = k16.copy(), v16.copy()
        K[base + n:] = NAN16; V[base + n:] = NAN16        # rows past the chunk's end must never be used
        pa.kv_write(0, 0, 0, K); pa.kv_write(0, 1, 0, V)
        pa.set_prefill_tile(tile)
        plan = pa.plan("prefill", base, n)
        got = pa.run_attn("prefill", 0, q, base, gate=gt, out_dtype=out_dtype)
    finally:
        pa.close()
    return got[rows].astype(np.float32), ref, plan


@pytest.mark.parametrize("shape,base,n", [
    ("qwen36_moe", 0, 16), ("qwen36_moe", 301, 16), ("qwen36_moe", 0, 77), ("qwen36_moe", 1000, 200),
    ("qwen38_27b", 173, 16), ("qwen38_27b", 90, 130), ("qwen3_1p7b", 77, 8 * 16), ("qwen3_1p7b", 0, 300),
    ("qwen3_1p7b", 219, 257), ("qwen36_moe", 4000, 33),
])
def test_prefill_small(shape, base, n):
    """Shapes of tests/unit/attn_tile_test.js:102-109 (first pass, partial tiles, padded row groups) and wider chunks."""
    got, ref, plan = _prefill(SHAPES[shape], base, n, seed=base + n)
    assert plan["kernel"] == 1
    assert_parity(got, ref, "%s base %d n %d" % (shape, base, n))


@pytest.mark.parametrize("shape", ["qwen36_moe", "qwen38_27b", "qwen3_1p7b"])
@pytest.mark.parametrize("base,n", [(0, 37), (0, 129), (33, 200), (3, 449)])
def test_prefill_paired_halves(shape, base, n):
    """An unsplit pass gives a workgroup a half block of columns from the front and one from the back: one half block alone,
    odd and even numbers of them, a ragged last one, halves whose row ends are hundreds of positions apart."""
    got, ref, plan = _prefill(SHAPES[shape], base, n, seed=base + n + 3)
    assert plan["kernel"] == 1 and plan["n_splits"] == 1
    assert_parity(got, ref, "paired %s base %d n %d" % (shape, base, n))


@pytest.mark.parametrize("base,n,paired", [(3000, 1000, 1), (3200, 1000, 1), (3300, 1010, 1), (6107, 1010, 1), (6144, 1000, 1), (6145, 1000, 0), (6108, 1010, 0), (9000, 1024, 0)])
def test_prefill_long_context_keeps_whole_blocks(base, n, paired):
    """At head_dim 256 an unsplit pass that fills the chip pairs half blocks only while base_pos x workgroups is within 6 x n_cols x
    CUs (on a 256-CU part); past that the blocks stay whole: either side of the line, full and ragged last blocks on both."""
    cfg = dict(SHAPES["qwen36_moe"], n_heads=64, n_kv_heads=2)                      # 32 heads a kv head: blocks of eight columns
    rows = sorted(set(range(0, n, 50)) | set(range(5)) | set(range(n - 5, n)))
    got, ref, plan = _prefill(cfg, base, n, seed=base + n, check_rows=rows)
    assert plan["kernel"] == 1 and plan["n_splits"] == 1 and plan["col_groups"] * 2 == 2 * -(-n // 8) <= 256
    assert capi.load().pa_rule_prefill_paired(256, base, n, 32, 2, 1, plan["col_groups"], 256) == paired
    assert_parity(got, ref, "%s at base %d n %d" % ("pairs" if paired else "whole blocks", base, n))


@pytest.mark.parametrize("shape,base,n", [("qwen36_moe", 0, 33), ("qwen36_moe", 31, 17), ("qwen36_moe", 64, 514), ("qwen38_27b", 10, 106),
                                          ("qwen38_27b", 1500, 43), ("qwen36_moe", 900, 33)])
def test_prefill_waves_done_early(shape, base, n):
    """Waves whose rows end before the workgroup's last tile only stage what is left: none, one and many such steps, an odd and an
    even number of computed ones, waves without any row, with the context whole and split."""
    got, ref, plan = _prefill(SHAPES[shape], base, n, seed=base + 3 * n)
    assert plan["kernel"] == 1
    assert_parity(got, ref, "waves done early %s base %d n %d" % (shape, base, n))


@pytest.mark.parametrize("n_kv,n", [(4, 260), (4, 257), (8, 133), (1, 1027), (3, 345)])
def test_prefill_more_workgroups_than_cus(n_kv, n):
    """An unsplit pass of more workgroups than the chip holds takes whole blocks of columns, the longest first, dealt over the
    XCDs of a kv head: one, two or eight of them, numbers of blocks that do not come out even, and (three kv heads) the
    general mapping."""
    cfg = dict(SHAPES["qwen3_1p7b"], n_heads=64 * n_kv, n_kv_heads=n_kv)           # 64 heads a kv head: blocks of four columns
    rows = sorted(set(range(0, n, max(1, n // 60))) | set(range(8)) | set(range(n - 8, n)))
    got, ref, plan = _prefill(cfg, 21, n, seed=n, check_rows=rows)
    assert plan["kernel"] == 1 and plan["n_splits"] == 1 and plan["col_groups"] * n_kv > 256
    assert_parity(got, ref, "whole blocks, %d kv heads n %d" % (n_kv, n))


def test_prefill_equals_decode_columns():
    """Every prefill column equals a single-token decode at the same position (tolerance)."""
    cfg = SHAPES["qwen36_moe"]
    rng = np.random.default_rng(21)
    base, n = 700, 40
    k16, v16 = random_cache(cfg, base + n, seed=22)
    q = rng.standard_normal((n, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32)
    gt = rng.standard_normal(q.shape, dtype=np.float32)
    with PooledAttn(cfg, base + n, n_layers=1, max_cols=n) as pa:
        pa.layer_alloc(0); pa.kv_write(0, 0, 0, k16); pa.kv_write(0, 1, 0, v16)
        pre = pa.run_attn("prefill", 0, q, base, gate=gt)
        for c in (0, 1, 17, 39):
            dec = pa.run_attn("decode", 0, q[c:c + 1], base + c, gate=gt[c:c + 1])
            assert np.abs(dec[0] - pre[c]).max() <= 1e-3


def test_prefill_split_path_and_f16_out():
    """A chunk of a few column blocks on a long context is split over the context (partials + merge kernel)."""
    cfg = SHAPES["qwen36_moe"]
    got, ref, plan = _prefill(cfg, 20000, 80, seed=5, out_dtype=PA_OUT_F16)
    assert plan["kernel"] == 1 and plan["n_splits"] > 1
    assert_parity(got, ref, "split prefill")


@pytest.mark.parametrize("shape,base,n", [("qwen36_moe", 20000, 16), ("qwen36_moe", 20000, 64), ("qwen38_27b", 9000, 40), ("qwen3_1p7b", 5000, 100)])
def test_prefill_narrow_chunk_on_a_long_context_takes_the_stream_kernel(shape, base, n):
    """Chunks of at most 512 stacked rows over 4096 or more cache rows (the reference's own passes are 16 columns wide)
    are bound by the K/V stream: the plan hands them to the split-K kernel in column groups."""
    got, ref, plan = _prefill(SHAPES[shape], base, n, seed=base + n, tile=0)
    assert plan["kernel"] == 0 and plan["col_groups"] > 1
    assert_parity(got, ref, "narrow chunk")


@pytest.mark.parametrize("shape,base,n,rows", [
    ("qwen3_1p7b", 0, 256, 16), ("qwen3_1p7b", 0, 512, 32), ("qwen3_1p7b", 1536, 512, 32), ("qwen36_moe", 0, 256, 16), ("qwen36_moe", 0, 512, 32),
    ("qwen38_27b", 0, 300, 12), ("qwen36_moe", 77, 129, 16), ("qwen3_1p7b", 5, 40, 16),
])
def test_prefill_small_chunk_takes_the_stream_kernel_in_one_launch(shape, base, n, rows):
    """Chunks of little causal work (the first chunks of a prompt, configuration 2's 512 columns over 2K rows): the table
    hands them to the split-K kernel as one split per workgroup -- 16- or 32-row workgroups over the whole context of
    their columns -- which writes the gated output itself: no partials, no merge launch.  Rows past the chunk are NaN;
    f16 and f32 output."""
    cfg = SHAPES[shape]
    G = cfg["n_heads"] // cfg["n_kv_heads"]
    for out_dtype in (0, PA_OUT_F16):
        got, ref, plan = _prefill(cfg, base, n, seed=base + n + 7, tile=0, out_dtype=out_dtype)
        assert plan["kernel"] == 0 and plan["n_splits"] == 1 and plan["slots"] == 1 and plan["cols_per_group"] * G == rows, plan
        assert_parity(got, ref, "small chunk %s base %d n %d" % (shape, base, n))


@pytest.mark.parametrize("shape,base,n,kernel,split,blocks", [
    ("qwen36_moe", 0, 33, 0, False, 1), ("qwen36_moe", 1000, 5, 0, True, 2), ("qwen36_moe", 450, 320, 0, False, 2), ("qwen36_moe", 2000, 100, 0, True, 2),
    ("qwen36_moe", 3500, 256, 1, True, 8), ("qwen38_27b", 300, 512, 0, False, 3), ("qwen38_27b", 1500, 40, 0, True, 2), ("qwen38_27b", 3500, 200, 1, True, 8),
    ("qwen3_1p7b", 2000, 128, 0, True, 4), ("qwen3_1p7b", 300, 1000, 0, False, 2), ("qwen3_1p7b", 500, 400, 0, False, 2), ("qwen3_1p7b", 3000, 33, 1, True, 8),
])
def test_prefill_chunk_takes_the_cheapest_of_three(shape, base, n, kernel, split, blocks):
    """Both sides of the lines between the matrix-core kernel, the split-K kernel with its merge and the one-launch split-K
    kernel of one, two and more row blocks; rows past the chunk are NaN."""
    rows = sorted({0, 1, n // 3, n // 2, n - 2, n - 1})
    got, ref, plan = _prefill(SHAPES[shape], base, n, seed=base + n + 9, tile=0, check_rows=rows)
    assert (plan["kernel"], plan["n_splits"] > 1, plan["row_blocks"]) == (kernel, split, blocks), plan
    assert_parity(got, ref, "chunk %s base %d n %d" % (shape, base, n))


@pytest.mark.parametrize("shape", ["qwen36_moe", "qwen38_27b", "qwen3_1p7b"])
@pytest.mark.parametrize("total", [3, 32, 33, 128, 129, 256, 257])
def test_a_few_columns_over_a_short_context(shape, total):
    """Blocks of one row block (prefill and decode calls) and chunks of several, either side of the context that one
    launch serves (256 rows; 128 for one row block at head_dim 256): no column has more rows than one before the last, the first block starts at position 0."""
    cfg = SHAPES[shape]
    G = cfg["n_heads"] // cfg["n_kv_heads"]
    most = lambda n: 128 if cfg["head_dim"] == 256 and n * G <= 16 else 256  # noqa: E731
    for n in sorted({min(total, 2), min(total, 16 // G), min(total, 32 // G + 1)}):
        got, ref, plan = _prefill(cfg, total - n, n, seed=total + n, tile=0)
        assert plan["kernel"] == 0 and ((plan["n_splits"] == 1) == (total <= most(n))) and (total > 256 or plan["row_blocks"] == 1), plan
        assert_parity(got, ref, "short %s %d columns of %d" % (shape, n, total))
    n = min(total, 16 // G)
    rng = np.random.default_rng(total)
    k16, v16 = random_cache(cfg, total, seed=total)
    q = rng.standard_normal((n, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32)
    with PooledAttn(cfg, total, n_layers=1, max_cols=n) as pa:
        pa.layer_alloc(0)
        pa.kv_write(0, 0, 0, k16.copy()); pa.kv_write(0, 1, 0, v16.copy())
        assert pa.plan("decode", total - n, n)["n_splits"] == (1 if total <= most(n) else -(-total // 128))
        assert_parity(pa.run_attn("decode", 0, q, total - n), C.attention(q, k16, v16, total - n), "short decode block %s of %d" % (shape, total))


def test_prefill_tile_override():
    """pa_set_prefill_tile (the reference's attnPrefillTile option, engine/qwen35.js:389-401): 1 forces the matrix-core
    kernel, 2 the split-K kernel, 0 is the table; all three give the same result within tolerance."""
    cfg = SHAPES["qwen36_moe"]
    outs = {}
    for mode, kernel in ((0, 0), (1, 1), (2, 0)):
        got, ref, plan = _prefill(cfg, 900, 200, seed=3, tile=mode)
        assert plan["kernel"] == kernel, (mode, plan)
        assert_parity(got, ref, "tile mode %d" % mode)
        outs[mode] = got
    assert np.abs(outs[1] - outs[2]).max() <= 1e-3


def test_prefill_peaked_softmax():
    """Large score spread (K scaled x3: scores span about +-12, far beyond the 2^8 lazy-rescale threshold): the
    lazily updated reference maximum must keep exp2 in range.  (Larger K scales amplify the f16 rounding of q
    beyond the 2e-3 gate: at x6 the error is 4e-3, all of it from the MFMA operand precision.)"""
    cfg = SHAPES["qwen38_27b"]
    got, ref, _ = _prefill(cfg, 500, 96, seed=9, k_scale=3.0)
    assert_parity(got, ref, "peaked")


def test_c2_prefill_full():
    """Config 2: 512-token chunk at positions 1536-2047 over a 1536-token prefix, Qwen3-1.7B shape, pre-step on
    the GPU (QK-RMSNorm + full RoPE theta 1e6 + KV write for the chunk), f16 output."""
    cfg = SHAPES["qwen3_1p7b"]
    base, n = 1536, 512
    d = O.make_inputs(cfg, base, n, seed=0x5EED0002)
    k16, v16 = oracle_cache(cfg, d["kraw"], d["vraw"], d["kw"])          # all 2048 rows, oracle pre-step
    g = O.glue_kv(d["qraw"], d["kraw"][base:], d["vraw"][base:], d["qw"], d["kw"], base, cfg)
    ref = C.attention(g["q"], k16, v16, base)
    with PooledAttn(cfg, base + n, n_layers=1, max_cols=n) as pa:
        pa.layer_alloc(0)
        pa.kv_write(0, 0, 0, k16[:base]); pa.kv_write(0, 1, 0, v16[:base])
        pa.run_glue_kv(0, d["qraw"], d["kraw"][base:], d["vraw"][base:], d["qw"], d["kw"], base)
        assert np.array_equal(pa.kv_read(0, 0, base, n), k16[base:]) and np.array_equal(pa.kv_read(0, 1, base, n), v16[base:])
        dout = pa.alloc(n * pa.q_dim * 2)
        pa.attn("prefill", 0, None, 0, None, 0, base, n, dout, pa.q_dim, PA_OUT_F16)
        pa.sync()
        got = dout.download(np.float16, n * pa.q_dim).reshape(ref.shape).astype(np.float32)
    assert_parity(got, ref, "C2 prefill chunk", tight=True)


def test_c5_prefill_128k_row_sample():
    """Config 5: 4096-token chunk at positions 126976-131071 over a 126976-token prefix, MoE shape, gate, f16 out.
    The whole chunk runs on the GPU; 24 evenly spread columns (all 16 heads) are checked against the f64 oracle,
    plus the first and last column."""
    cfg = SHAPES["qwen36_moe"]
    base, n = 126976, 4096
    rows = sorted(set([0, n - 1] + list(range(5, n, n // 22))))
    got, ref, plan = _prefill(cfg, base, n, seed=0x5EED0005, max_seq=base + n, out_dtype=PA_OUT_F16, check_rows=rows)
    assert plan["kernel"] == 1 and plan["n_splits"] == 1
    assert_parity(got, ref, "C5 prefill 128K, column sample", tight=True)


@pytest.mark.parametrize("shape,base,n", [("qwen36_moe", 300, 40), ("qwen3_1p7b", 200, 120), ("qwen38_27b", 5000, 64)])
@pytest.mark.parametrize("one_row", [False, True])
@pytest.mark.parametrize("jump", [5.3, 5.5, 5.6, 6.0, 10.9, 11.2, 12.0])
def test_prefill_jumps_around_the_raise(shape, base, n, one_row, jump):
    """References are raised where a probability is past 2^8 (a score 5.55 above the reference) on its f16 value, which is infinite from 2^16 on (11.09):
    a flat context whose scores jump once by a little less and a little more than either, for all rows of a wave and for one row among others that
    must not notice; every row against the oracle, whole and split contexts."""
    cfg = SHAPES[shape]
    nH, nKV, hd = cfg["n_heads"], cfg["n_kv_heads"], cfg["head_dim"]
    rng = np.random.default_rng(base + n)
    rows = base + n
    k = rng.standard_normal((rows, nKV, hd)).astype(np.float32) * 0.02
    k[:, :, 0] = jump * (np.arange(rows) >= rows // 2)[:, None]   # q's first value is sqrt(hd) or 0: it adds the jump to a row's scores or not
    k16 = k.astype(np.float16).view(np.uint16)
    v16 = rng.standard_normal((rows, nKV, hd)).astype(np.float16).view(np.uint16)
    q = rng.standard_normal((n, nH, hd)).astype(np.float16).astype(np.float32)
    q[:, :, 0] = 0 if one_row else hd ** 0.5
    q[n // 2, 0, 0] = hd ** 0.5
    q = q.astype(np.float16).astype(np.float32)                   # f16 queries: the scores carry no rounding of q
    ref = C.attention(q, k16, v16, base, gate=None, rows=list(range(n)))
    with PooledAttn(cfg, rows + 3, n_layers=1, max_cols=n) as pa:
        pa.layer_alloc(0); pa.kv_write(0, 0, 0, k16); pa.kv_write(0, 1, 0, v16)
        pa.set_prefill_tile(1)
        assert pa.plan("prefill", base, n)["kernel"] == 1
        got = pa.run_attn("prefill", 0, q, base)
    assert_parity(got.astype(np.float32), ref, "jump %g %s" % (jump, shape))


@pytest.mark.parametrize("shape,base,n,tile", [("qwen36_moe", 0, 40, 1), ("qwen36_moe", 900, 33, 1), ("qwen3_1p7b", 70, 300, 1), ("qwen38_27b", 5000, 64, 1)])
@pytest.mark.parametrize("trend", ["up", "down", "jump", "late"])
def test_prefill_reference_maxima(shape, base, n, tile, trend):
    """Scores whose maximum rises by a few units a tile, falls, jumps by 60 in the middle of the context (exp2 of it is past the f16
    range before the references are raised) or only behind the chunk's first columns (rows of a wave that end before the jump must not
    notice): every row against the oracle, whole and split contexts."""
    cfg = SHAPES[shape]
    nH, nKV, hd = cfg["n_heads"], cfg["n_kv_heads"], cfg["head_dim"]
    rng = np.random.default_rng(base + n)
    rows = base + n
    t = np.arange(rows)
    level = {"up": t / 32 * 0.7 % 40, "down": 30 - 30 * t / rows, "jump": 60.0 * (t >= rows // 2), "late": 60.0 * (t >= base + n // 2)}[trend]
    k = rng.standard_normal((rows, nKV, hd)).astype(np.float32) * 0.25
    k[:, :, 0] = level[:, None]                                   # q's first value is sqrt(hd): it adds the level to every score
    k16 = k.astype(np.float16).view(np.uint16)
    v16 = rng.standard_normal((rows, nKV, hd)).astype(np.float16).view(np.uint16)
    q = rng.standard_normal((n, nH, hd)).astype(np.float16).astype(np.float32)
    q[:, :, 0] = hd ** 0.5
    q16 = q.astype(np.float16).astype(np.float32)                 # f16 queries: the scores carry no rounding of q
    ref = C.attention(q16, k16, v16, base, gate=None, rows=list(range(n)))
    with PooledAttn(cfg, rows + 3, n_layers=1, max_cols=n) as pa:
        pa.layer_alloc(0); pa.kv_write(0, 0, 0, k16); pa.kv_write(0, 1, 0, v16)
        pa.set_prefill_tile(tile)
        assert pa.plan("prefill", base, n)["kernel"] == 1
        got = pa.run_attn("prefill", 0, q16, base)
    assert_parity(got.astype(np.float32), ref, "maxima %s %s base %d" % (trend, shape, base))

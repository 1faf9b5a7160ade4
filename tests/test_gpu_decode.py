"""GPU parity of decode / speculative-verify attention through the C ABI against the CPU oracle.
Tolerance (floating point): max-abs <= 2e-3 and max|d|/max|ref| <= 1e-2 of the f32/f64 reference."""
import numpy as np
import pytest
from oracle import attn_oracle as O
from oracle import c_oracle as C
from pooled_amd.capi import PooledAttn, PA_OUT_F16
from helpers import BLOCK, LOOP, SHAPES, SINGLE_ROUND, assert_parity, attn_rule, random_cache, oracle_cache

pytestmark = pytest.mark.gpu

NAN16 = 0x7E00


def _ctx_with_cache(cfg, k16, v16, max_seq, max_cols=16, poison_from=None):
    pa = PooledAttn(cfg, max_seq, n_layers=1, max_cols=max_cols)
    pa.layer_alloc(0)
    K, V = k16.copy(), v16.copy()
    if poison_from is not None:
        K[poison_from:] = NAN16; V[poison_from:] = NAN16
    pa.kv_write(0, 0, 0, K); pa.kv_write(0, 1, 0, V)
    return pa


SEQ_LENS = [1, 2, 5, 31, 32, 33, 63, 64, 65, 127, 128, 129, 300, 1000, 2049, 4097]


@pytest.mark.parametrize("shape", ["qwen36_moe", "qwen38_27b", "qwen3_1p7b"])
def test_decode_seq_lens(shape):
    """The context lengths of tests/test_attn_dec.js:106-107 (split-length steps), K in +-0.3-like spread."""
    cfg = SHAPES[shape]
    rng = np.random.default_rng(7)
    max_seq = max(SEQ_LENS) + 40
    k16, v16 = random_cache(cfg, max_seq, seed=8)
    q = rng.standard_normal((1, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32) * 2
    with _ctx_with_cache(cfg, k16, v16, max_seq) as pa:
        for L in SEQ_LENS:
            # rows at or past L are NaN: any causal leak poisons the output (tests/unit/attn_tile_test.js:43-50)
            pa.kv_write(0, 0, 0, np.where(np.arange(max_seq)[:, None, None] < L, k16, NAN16).astype(np.uint16))
            pa.kv_write(0, 1, 0, np.where(np.arange(max_seq)[:, None, None] < L, v16, NAN16).astype(np.uint16))
            got = pa.run_attn("decode", 0, q, L - 1)
            ref = C.attention(q, k16, v16, L - 1)
            assert_parity(got, ref, "%s seqLen %d" % (shape, L))


def test_decode_closed_forms():
    cfg = SHAPES["qwen36_moe"]
    nH, nKV, hd = cfg["n_heads"], cfg["n_kv_heads"], cfg["head_dim"]
    rng = np.random.default_rng(9)
    L = 1500
    k16, v16 = random_cache(cfg, L, seed=10)
    q = rng.standard_normal((1, nH, hd), dtype=np.float32)
    v = v16.view(np.float16)
    with _ctx_with_cache(cfg, k16, v16, L) as pa:
        o = pa.run_attn("decode", 0, q, 0)                                 # one row -> that V row
        for h in range(nH):
            assert np.allclose(o[0, h], v[0, h // (nH // nKV)].astype(np.float32), atol=1e-6)
        o = pa.run_attn("decode", 0, np.zeros_like(q), L - 1)               # q = 0 -> mean of V rows
        assert np.abs(o[0, 3] - v[:, 0].astype(np.float64).mean(0)).max() < 2e-4
        pa.kv_write(0, 1, 0, np.full((L, nKV, hd), 0x3A00, np.uint16))      # constant V = 0.75
        assert np.abs(pa.run_attn("decode", 0, q, L - 1) - 0.75).max() < 1e-3


@pytest.mark.parametrize("shape", ["qwen36_moe", "qwen38_27b", "qwen3_1p7b"])
def test_outputs_are_convex_combinations_of_value_rows(shape):
    """Every value row the same vector => the output is that vector, whatever the scores: the row total l is summed
    from the f16-rounded probabilities the PV product uses, so the weights that are applied add up to exactly the
    divisor and the rounding of P cancels (with l summed from the unrounded exponentials the outputs were off by up to
    3e-4 of the value on short contexts).  What is left is f32 accumulation: a few 1e-7.  One-column decodes and verify
    blocks on the single-round kernel and on the tile loop, chunks on the split-K kernel with direct output and on the
    matrix-core kernel, with and without a split over the context."""
    cfg = SHAPES[shape]
    nH, nKV, hd = cfg["n_heads"], cfg["n_kv_heads"], cfg["head_dim"]
    rng = np.random.default_rng(5)
    L = 40000
    k16, _ = random_cache(cfg, L, seed=3, k_scale=2.0)
    vrow = rng.standard_normal((nKV, hd)).astype(np.float16)
    v16 = np.broadcast_to(vrow.view(np.uint16), (L, nKV, hd)).copy()
    want = np.repeat(vrow.astype(np.float64), nH // nKV, axis=0)
    with _ctx_with_cache(cfg, k16, v16, L, max_cols=400) as pa:
        kernels = set()
        for kind, n, lens in (("decode", 1, (1, 2, 3, 17, 40, 129, 1500, 33000, 39999)), ("decode", 5, (6, 40, 1500, 33000)),
                              ("prefill", 12, (12, 300)), ("prefill", 300, (300, 5000))):
            for Lc in lens:
                q = rng.standard_normal((n, nH, hd), dtype=np.float32)
                pl = pa.plan(kind, Lc - n, n)
                kernels.add((pl["kernel"], pl["n_splits"] > 1, pl["split_len"] == 128))
                o = pa.run_attn(kind, 0, q, Lc - n).astype(np.float64)
                err = np.abs(o - want[None]).max() / np.abs(want).max()
                assert err < 2e-6, "%s %s %d columns over %d rows: %.2e of the value (%s)" % (shape, kind, n, Lc, err, pl)
        assert {k[0] for k in kernels} == {0, 1} and any(k[1] and k[2] for k in kernels) and any(k[1] and not k[2] for k in kernels), kernels


@pytest.mark.parametrize("shape", ["qwen36_moe", "qwen38_27b", "qwen3_1p7b"])
def test_short_context_decode_sees_q_at_f32_precision(shape):
    """A block of at most eight stacked rows carries the f16 rounding error of q in rows 8 .. 15 of its q tile, so its
    scores see q at f32 precision.  Inputs that make the rounding of q visible (q of twice, keys of twice the
    benchmark's spread: scores of a spread of 4, a few rows share the weight whatever the length) come out within 6e-4 of
    the f64 oracle (measured: up to 4.1e-4, what the f16 rounding of P leaves); with q rounded to f16 the same inputs are
    off by 1.6e-3 to 4.7e-3."""
    cfg = SHAPES[shape]
    nH, nKV, hd = cfg["n_heads"], cfg["n_kv_heads"], cfg["head_dim"]
    rng = np.random.default_rng(11)
    Lmax = 4100
    k16, v16 = random_cache(cfg, Lmax, seed=13, k_scale=2.0)
    with _ctx_with_cache(cfg, k16, v16, Lmax) as pa:
        for n in sorted({1, 8 // (nH // nKV)}):
            for L in (2, 3, 5, 17, 33, 129, 300, 1000, 2047, 2049, 4097):
                if L <= n:
                    continue
                for rep in range(3):
                    q = rng.standard_normal((n, nH, hd), dtype=np.float32) * 2
                    got = pa.run_attn("decode", 0, q, L - n)
                    ref = C.attention(q, k16[:L], v16[:L], L - n)
                    d = float(np.abs(got - ref).max())
                    assert d < 6e-4, "%s %d columns over %d rows: max-abs %.3e" % (shape, n, L, d)


def test_decode_split_invariance_and_plan():
    cfg = SHAPES["qwen36_moe"]
    rng = np.random.default_rng(11)
    L = 5000
    k16, v16 = random_cache(cfg, L, seed=12)
    q = rng.standard_normal((1, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32) * 1.5
    ref = C.attention(q, k16, v16, L - 1)
    with _ctx_with_cache(cfg, k16, v16, L) as pa:
        outs = []
        for s in (0, 1, 3, 16, 40):
            pa.set_decode_splits(s)
            pl = pa.plan("decode", L - 1, 1)
            # a one-column decode streams rows 0 .. L - 2; its own row L - 1 is one more partial (slots = splits + 1)
            assert pl["n_splits"] * pl["split_len"] >= L - 1 and pl["split_len"] % 32 == 0 and pl["slots"] == pl["n_splits"] + 1
            if s:
                assert pl["n_splits"] <= s
            outs.append(pa.run_attn("decode", 0, q, L - 1))
            assert_parity(outs[-1], ref, "splits %d" % s)
        assert max(np.abs(o - outs[0]).max() for o in outs) < 2e-4
        # deterministic run to run
        pa.set_decode_splits(0)
        assert np.array_equal(pa.run_attn("decode", 0, q, L - 1), pa.run_attn("decode", 0, q, L - 1))


@pytest.mark.parametrize("pos", [63 * 128, 64 * 128, 64 * 128 + 77, 12000])
def test_decode_either_side_of_the_f16_partials_threshold(pos):
    """A one-column decode writes f16 O partials from 64 single-round splits on (f32 below): both sides of the threshold,
    a remainder split, and a longer context against the f64 oracle, with the margin the five configurations are held to."""
    cfg = SHAPES["qwen36_moe"]
    rng = np.random.default_rng(pos)
    k16, v16 = random_cache(cfg, pos + 1, seed=pos + 1)
    q = rng.standard_normal((1, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32)
    gate = rng.standard_normal(q.shape, dtype=np.float32)
    ref = C.attention(q, k16, v16, pos, gate=gate)
    with _ctx_with_cache(cfg, k16, v16, pos + 1) as pa:
        pl = pa.plan("decode", pos, 1)
        assert pl["split_len"] == 128 and (pl["n_splits"] >= 64) == (pos >= 64 * 128)
        for out_dtype in (0, PA_OUT_F16):
            assert_parity(pa.run_attn("decode", 0, q, pos, gate=gate, out_dtype=out_dtype), ref, "decode at %d, %d splits" % (pos, pl["n_splits"]), tight=True)


@pytest.mark.parametrize("shape,n_cols,base", [("qwen36_moe", 4, 996), ("qwen36_moe", 16, 3000), ("qwen38_27b", 8, 2040),
                                               ("qwen3_1p7b", 4, 510), ("qwen38_27b", 16, 17), ("qwen36_moe", 7, 0),
                                               ("qwen36_moe", 16, 20000), ("qwen38_27b", 12, 30000), ("qwen3_1p7b", 16, 9000)])
def test_verify_equals_sequential_decodes(shape, n_cols, base):
    """A verify block must equal n sequential single-token decodes (engine/wgsl/attn_dec.js:12-16;
    tests/test_attn_dec.js:89-97) -- here within tolerance -- and the oracle."""
    cfg = SHAPES[shape]
    rng = np.random.default_rng(base + n_cols)
    L = base + n_cols
    k16, v16 = random_cache(cfg, L + 5, seed=13)
    q = rng.standard_normal((n_cols, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32)
    gate = rng.standard_normal((n_cols, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32) if cfg["gate"] else None
    ref = C.attention(q, k16, v16, base, gate=gate)
    with _ctx_with_cache(cfg, k16, v16, L + 5, poison_from=L) as pa:
        multi = pa.run_attn("decode", 0, q, base, gate=gate)
        assert_parity(multi, ref, "verify block")
        for c in range(n_cols):
            single = pa.run_attn("decode", 0, q[c:c + 1], base + c, gate=None if gate is None else gate[c:c + 1])
            assert_parity(single, ref[c:c + 1], "single decode col %d" % c)
            assert np.abs(single[0] - multi[c]).max() <= 1e-3


@pytest.mark.parametrize("shape,n_cols,base", [("qwen36_moe", 4, 8000), ("qwen38_27b", 5, 5000), ("qwen3_1p7b", 12, 1900), ("qwen36_moe", 3, 16200),
                                               ("qwen36_moe", 8, 3900)])
def test_verify_block_on_the_single_round_kernel_with_two_row_blocks(shape, n_cols, base):
    """A verify block of 17 .. 32 stacked rows a workgroup over a context that fits one round of one-tile-per-wave splits
    at one workgroup a CU (half of that at head_dim 128 and with several column groups): the single-round kernel with two row blocks (f16 caches).  Causal ends differ by column, the
    last split is partial, rows past the context are poisoned; f32 and f16 out, with a gate where the shape has one."""
    cfg = SHAPES[shape]
    rng = np.random.default_rng(base + n_cols)
    L = base + n_cols
    k16, v16 = random_cache(cfg, L + 40, seed=base)
    q = rng.standard_normal((n_cols, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32)
    gate = rng.standard_normal(q.shape, dtype=np.float32) if cfg["gate"] else None
    ref = C.attention(q, k16, v16, base, gate=gate)
    with _ctx_with_cache(cfg, k16, v16, L + 40, max_cols=n_cols, poison_from=L) as pa:
        pl = pa.plan("decode", base, n_cols)
        assert pl["row_blocks"] == 2 and pl["split_len"] == 128 and pl["n_splits"] == -(-L // 128) and pl["slots"] == pl["n_splits"], pl
        assert attn_rule(cfg, "decode", base, n_cols) == (SINGLE_ROUND, pl)
        for out_dtype in (0, PA_OUT_F16):
            assert_parity(pa.run_attn("decode", 0, q, base, gate=gate, out_dtype=out_dtype), ref, "two row blocks, single round, %d columns at %d" % (n_cols, base), tight=True)
        fewer = max(2, pl["n_splits"] // 3)
        pa.set_decode_splits(fewer)                                  # the same block at several tiles a wave: the tile loop, or with one column group one softmax a workgroup
        assert attn_rule(cfg, "decode", base, n_cols, fewer) == (LOOP if pl["col_groups"] > 1 else BLOCK, pa.plan("decode", base, n_cols))
        assert np.abs(pa.run_attn("decode", 0, q, base, gate=gate) - pa_first(pa, q, base, gate)).max() <= 2e-4


def pa_first(pa, q, base, gate):
    """The table's plan again (after a splits override)."""
    pa.set_decode_splits(0)
    return pa.run_attn("decode", 0, q, base, gate=gate)


@pytest.mark.parametrize("shape,n_cols,base", [("qwen36_moe", 4, 996), ("qwen38_27b", 8, 2040), ("qwen3_1p7b", 5, 510), ("qwen36_moe", 3, 32767),
                                               ("qwen36_moe", 8, 9000), ("qwen36_moe", 16, 20000), ("qwen38_27b", 6, 8190), ("qwen3_1p7b", 13, 119),
                                               ("qwen36_moe", 5, 40000), ("qwen38_27b", 4, 33000), ("qwen38_27b", 8, 65533)])
def test_verify_exact_flag_gives_the_sequential_decodes_bits(shape, n_cols, base):
    """PA_FLAG_VERIFY_EXACT: every column of a verify block has the bits of the one-column decode at its position
    (the reference's invariant, engine/wgsl/attn_dec.js:12-16; tests/test_attn_dec.js:89-97 checks it with Object.is);
    the plan a plan query reports is unchanged.  Blocks whose columns share a one-column plan run as one pass (the first
    three cases and the 9000- and 20000-row ones, with f16 partials on the last two; the 40000- and 33000-row ones on the
    tile loop's longer splits); blocks that straddle a change of plan (32767 .. 32769, 8190 .. 8195, 119 .. 131, and
    65536 .. 65543 of the 27B shape, where the tile loop goes from eight to nine tiles a wave) run as one pass per run of
    columns with the same plan, a lone column as the one-column decode itself."""
    cfg = dict(SHAPES[shape], verify_exact=True)
    rng = np.random.default_rng(base + n_cols)
    L = base + n_cols
    k16, v16 = random_cache(cfg, L + 5, seed=14)
    q = rng.standard_normal((n_cols, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32)
    gate = rng.standard_normal(q.shape, dtype=np.float32) if cfg["gate"] else None
    ref = C.attention(q, k16, v16, base, gate=gate)
    with _ctx_with_cache(cfg, k16, v16, L + 5, poison_from=L) as pa:
        multi = pa.run_attn("decode", 0, q, base, gate=gate)
        assert_parity(multi, ref, "column-exact verify block")
        for c in range(n_cols):
            single = pa.run_attn("decode", 0, q[c:c + 1], base + c, gate=None if gate is None else gate[c:c + 1])
            assert np.array_equal(single[0].view(np.uint32), multi[c].view(np.uint32)), "column %d differs from its decode" % c


@pytest.mark.parametrize("shape,n_cols,base,more", [("qwen36_moe", 8, 9209, {}), ("qwen36_moe", 9, 9209, dict(kv_q8=True)), ("qwen38_27b", 15, 12000, {}),
                                                    ("qwen38_27b", 7, 12154, dict(kv_q8=True)), ("qwen3_1p7b", 9, 6137, {}), ("qwen36_moe", 2, 30001, {}),
                                                    ("qwen36_moe", 16, 16380, {}), ("qwen3_1p7b", 5, 7005, dict(n_heads=80, n_kv_heads=8)),
                                                    ("qwen36_moe", 10, 250, {}), ("qwen3_1p7b", 7, 253, dict(kv_q8=True))])
def test_verify_exact_two_columns_a_workgroup(shape, n_cols, base, more):
    """Column-exact blocks of more workgroups than the chip holds twice share their whole splits between two columns: odd and even
    numbers of columns, a last column that ends with a whole split (9216, 12160, 6144, 16384 rows) alone or before a change of plan, f16 and f32
    partials, more than eight heads a kv head, int8 caches; and short blocks of one workgroup a column and kv head up to 256 rows, splits past
    them.  Every column finite, with its decode's bits, and unchanged when all rows behind it are infinite (int8 caches: 3e4): no column may see them."""
    cfg = dict(SHAPES[shape], verify_exact=True, **more)
    rng = np.random.default_rng(base + n_cols)
    L = base + n_cols
    far = 3e4 if cfg.get("kv_q8") else np.inf
    q = rng.standard_normal((n_cols, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32)
    with PooledAttn(cfg, L + 5, n_layers=1, max_cols=2048) as pa:
        pa.layer_alloc(0)
        kvd = pa.kv_dim

        def store(r, k, v):
            dk, dv = pa.to_device(k), pa.to_device(v)
            pa.kv_store(0, dk, kvd, dv, kvd, r, len(k))
            pa.sync()

        for r in range(0, base, 2048):
            store(r, *rng.standard_normal((2, min(2048, base - r), kvd), dtype=np.float32))
        k, v = rng.standard_normal((2, n_cols + 5, kvd), dtype=np.float32)
        behind = lambda c: np.where(np.arange(n_cols + 5)[:, None] > c, np.float32(far), v)   # noqa: E731
        store(base, k, behind(n_cols - 1))
        multi = pa.run_attn("decode", 0, q, base)
        assert np.isfinite(multi).all()
        for c in range(n_cols):
            single = pa.run_attn("decode", 0, q[c:c + 1], base + c)
            assert np.array_equal(single[0].view(np.uint32), multi[c].view(np.uint32)), "column %d differs from its decode" % c
        for c in range(n_cols - 1):
            store(base, k, behind(c))
            assert np.array_equal(pa.run_attn("decode", 0, q, base)[c].view(np.uint32), multi[c].view(np.uint32)), "column %d sees rows behind it" % c


@pytest.mark.parametrize("shape,n_cols,base", [("qwen36_moe", 1, 200), ("qwen3_1p7b", 1, 256), ("qwen3_1p7b", 5, 120), ("qwen36_moe", 4, 250)])
@pytest.mark.parametrize("into", ["q", "gate", "behind q"])
def test_decode_output_over_its_inputs(shape, n_cols, base, into):
    """Results written over the queries or the gate, f16 and f32, from their first byte or from a column's middle on, where one workgroup a kv head
    writes the output itself (at most 256 rows, in column-exact blocks too): the bits of a call with a buffer of its own."""
    cfg = dict(SHAPES[shape], verify_exact=True)
    rng = np.random.default_rng(base + n_cols)
    k16, v16 = random_cache(cfg, base + n_cols, seed=5)
    with _ctx_with_cache(cfg, k16, v16, base + n_cols) as pa:
        qd = pa.q_dim
        q, gate = rng.standard_normal((2, n_cols, qd), dtype=np.float32)
        for out_dtype, np_dtype, stride in ((0, np.float32, qd), (PA_OUT_F16, np.float16, qd), (PA_OUT_F16, np.float16, qd + 4)):
            assert pa.plan("decode", base + n_cols - 1, 1)["waves"] == 8
            room = np.zeros(n_cols * qd + 4 * stride, np.float32)
            dq, dg, own = (pa.to_device(np.concatenate([a.ravel(), room])) for a in (q, gate, room))
            pa.attn("decode", 0, dq, qd, dg, qd, base, n_cols, own, stride, out_dtype)
            at = (dg if into == "gate" else dq).ptr + (qd * 2 if into == "behind q" else 0)
            pa.sync()
            want = own.download(np_dtype, n_cols * stride)
            pa._chk(pa.L.pa_attn_decode(pa.ctx, 0, dq.ptr, qd, dg.ptr, qd, base, n_cols, at, stride, out_dtype))
            pa.sync()
            got = np.empty(n_cols * stride, np_dtype)
            pa._chk(pa.L.pa_download(pa.ctx, got.ctypes.data, at, got.nbytes))
            cols = lambda a: a.reshape(n_cols, stride)[:, :qd]
            assert np.isfinite(cols(want).astype(np.float32)).all() and np.array_equal(cols(want), cols(got)), (out_dtype, stride)


def test_decode_f16_output_and_strides():
    cfg = SHAPES["qwen36_moe"]
    rng = np.random.default_rng(14)
    L, n = 700, 3
    k16, v16 = random_cache(cfg, L + n, seed=15)
    q = rng.standard_normal((n, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32)
    gate = rng.standard_normal(q.shape, dtype=np.float32)
    ref = C.attention(q, k16, v16, L, gate=gate)
    with _ctx_with_cache(cfg, k16, v16, L + n) as pa:
        got = pa.run_attn("decode", 0, q, L, gate=gate, out_dtype=PA_OUT_F16)
        assert got.dtype == np.float16
        assert_parity(got.astype(np.float32), ref, "f16 out")
        # padded column strides (the engine aligns columns to 256 bytes, engine/qwen35.js:2054-2055)
        qd, pad = pa.q_dim, 64
        qp = np.full((n, qd + pad), np.nan, np.float32); qp[:, :qd] = q.reshape(n, -1)
        gp = np.full((n, qd + pad), np.nan, np.float32); gp[:, :qd] = gate.reshape(n, -1)
        dq, dg = pa.to_device(qp), pa.to_device(gp)
        dout = pa.to_device(np.full((n, qd + pad), -7.0, np.float32))
        pa.attn("decode", 0, dq, qd + pad, dg, qd + pad, L, n, dout, qd + pad)
        pa.sync()
        o = dout.download(np.float32, n * (qd + pad)).reshape(n, qd + pad)
        assert_parity(o[:, :qd].reshape(ref.shape), ref, "padded strides")
        assert np.all(o[:, qd:] == -7.0), "wrote into the padding between columns"


def test_c1_decode_full_pipeline():
    """Config 1: Qwen3-1.7B shape, ctx 2048, pre-step (QK-RMSNorm + full RoPE theta 1e6) on the GPU for the
    query column, cache rows built by the oracle's pre-step; f32 softmax; f16 output."""
    cfg = SHAPES["qwen3_1p7b"]
    ctx = 2048
    d = O.make_inputs(cfg, ctx, 1, seed=0x5EED0001)
    k16, v16 = oracle_cache(cfg, d["kraw"][:ctx], d["vraw"][:ctx], d["kw"])
    g = O.glue_kv(d["qraw"], d["kraw"][ctx:], d["vraw"][ctx:], d["qw"], d["kw"], ctx, cfg)
    kall = np.concatenate([k16, g["k16"]]); vall = np.concatenate([v16, g["v16"]])
    ref = C.attention(g["q"], kall, vall, ctx)
    with PooledAttn(cfg, ctx + 1, n_layers=1, max_cols=1) as pa:
        pa.layer_alloc(0)
        pa.kv_write(0, 0, 0, k16); pa.kv_write(0, 1, 0, v16)
        pa.run_glue_kv(0, d["qraw"], d["kraw"][ctx:], d["vraw"][ctx:], d["qw"], d["kw"], ctx)
        assert np.array_equal(pa.kv_read(0, 0, ctx, 1), g["k16"])
        dout = pa.alloc(pa.q_dim * 2)
        pa.attn("decode", 0, None, 0, None, 0, ctx, 1, dout, pa.q_dim, PA_OUT_F16)    # q from the context's buffer
        pa.sync()
        got = dout.download(np.float16, pa.q_dim).reshape(ref.shape).astype(np.float32)
    assert_parity(got, ref, "C1 decode, f16 out", tight=True)


def test_c3_gated_decode_32k():
    """Config 3: Qwen3.6-35B-MoE attention shape, ctx 32768, partial RoPE (64 dims, theta 1e7), sigmoid gate."""
    cfg = SHAPES["qwen36_moe"]
    ctx = 32768
    d = O.make_inputs(cfg, ctx, 1, seed=0x5EED0003)
    k16, v16 = oracle_cache(cfg, d["kraw"][:ctx], d["vraw"][:ctx], d["kw"])
    g = O.glue_kv(d["qraw"], d["kraw"][ctx:], d["vraw"][ctx:], d["qw"], d["kw"], ctx, cfg)
    kall = np.concatenate([k16, g["k16"]]); vall = np.concatenate([v16, g["v16"]])
    ref = C.attention(g["q"], kall, vall, ctx, gate=g["gate"])
    with PooledAttn(cfg, ctx + 1, n_layers=1, max_cols=1) as pa:
        pa.layer_alloc(0)
        pa.kv_write(0, 0, 0, k16); pa.kv_write(0, 1, 0, v16)
        pa.run_glue_kv(0, d["qraw"], d["kraw"][ctx:], d["vraw"][ctx:], d["qw"], d["kw"], ctx)
        dout = pa.alloc(pa.q_dim * 4)
        pa.attn("decode", 0, None, 0, pa.gate_buffer_ptr(), pa.q_dim, ctx, 1, dout, pa.q_dim)
        pa.sync()
        got = dout.download(np.float32, pa.q_dim).reshape(ref.shape)
        # 32768 streamed rows over 256 workgroup slots per kv head = whole 128-row splits; the token's own row is
        # the 257th partial
        pl = pa.plan("decode", ctx, 1)
        assert pl["n_splits"] * pl["split_len"] == ctx and pl["split_len"] % 32 == 0 and pl["slots"] == pl["n_splits"] + 1
    assert_parity(got, ref, "C3 gated decode 32K", tight=True)


@pytest.mark.parametrize("extra", [1, 2, 3, 32, 33, 34, 128, 2000, 5000])
def test_decode_past_the_single_round_capacity(extra):
    """Contexts a little past what the single-round kernel holds in one round (256 one-tile-per-wave splits a kv head
    at this shape): the tile loop with one workgroup a CU, its tiles dealt round robin to the waves of all splits, the
    last tile partial (poisoned rows past the context must stay unused)."""
    cfg = SHAPES["qwen36_moe"]
    L = 32768 + extra
    rng = np.random.default_rng(40 + extra)
    k16, v16 = random_cache(cfg, L + 40, seed=41)
    q = rng.standard_normal((1, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32)
    ref = C.attention(q, k16, v16, L - 1)
    with _ctx_with_cache(cfg, k16, v16, L + 40, poison_from=L) as pa:
        pl = pa.plan("decode", L - 1, 1)
        if extra == 1:
            assert pl["n_splits"] * pl["split_len"] == L - 1 and pl["split_len"] == 128      # whole splits + the token's own row
        else:
            assert pl["n_splits"] <= 128 and pl["split_len"] > 128 and pl["n_splits"] * pl["split_len"] >= L - 1, pl
        got = pa.run_attn("decode", 0, q, L - 1)
    assert_parity(got, ref, "open-ended last split, +%d rows" % extra)


def test_decode_one_column_at_128k():
    """A one-column decode over 131072 cached rows (MoE shape): the tile loop with one workgroup a CU, a kv head's 4096
    tiles dealt round robin to the 512 waves of its 128 splits, eight a wave; with a gate, f32 and f16 out."""
    cfg = SHAPES["qwen36_moe"]
    pos = 131072
    rng = np.random.default_rng(131)
    k16, v16 = random_cache(cfg, pos + 1, seed=132)
    q = rng.standard_normal((1, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32)
    gate = rng.standard_normal(q.shape, dtype=np.float32)
    ref = C.attention(q, k16, v16, pos, gate=gate)
    with _ctx_with_cache(cfg, k16, v16, pos + 1, max_cols=1) as pa:
        pl = pa.plan("decode", pos, 1)
        assert pl["n_splits"] == 128 and pl["split_len"] == 1024 and pl["slots"] == 129 and pl["row_blocks"] == 1, pl
        for out_dtype in (0, PA_OUT_F16):
            assert_parity(pa.run_attn("decode", 0, q, pos, gate=gate, out_dtype=out_dtype), ref, "decode at 128K", tight=True)


def test_c4_verify_64k():
    """Config 4: 8-token draft block over a 65536-token cache, Qwen3.8-27B attention shape, gate; equals 8
    sequential decodes (checked on columns 0 and 7) and the oracle."""
    cfg = SHAPES["qwen38_27b"]
    ctx, n = 65536, 8
    rng = np.random.default_rng(0x5EED0004)
    k16, v16 = random_cache(cfg, ctx + n, seed=0x5EED0004)
    q = O.rope_neox(O.head_rmsnorm(rng.standard_normal((n, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32),
                                   np.ones(cfg["head_dim"], np.float32), cfg["eps"]), ctx + np.arange(n), cfg["n_rot"], cfg["rope_theta"])
    gate = rng.standard_normal(q.shape, dtype=np.float32)
    ref = C.attention(q, k16, v16, ctx, gate=gate)
    with _ctx_with_cache(cfg, k16, v16, ctx + n, max_cols=n) as pa:
        multi = pa.run_attn("decode", 0, q, ctx, gate=gate)
        assert_parity(multi, ref, "C4 verify block 64K", tight=True)
        for c in (0, 7):
            single = pa.run_attn("decode", 0, q[c:c + 1], ctx + c, gate=gate[c:c + 1])
            assert_parity(single, ref[c:c + 1], "C4 decode col %d" % c)
            assert np.abs(single[0] - multi[c]).max() <= 1e-3


@pytest.mark.parametrize("kind,shape,n_cols,base,blocks,kernel", [
    ("decode", "qwen36_moe", 1, 40000, 1, LOOP), ("decode", "qwen36_moe", 8, 20000, 2, LOOP), ("decode", "qwen38_27b", 11, 30000, 3, LOOP), ("decode", "qwen36_moe", 4, 40000, 2, BLOCK),
    ("decode", "qwen38_27b", 8, 50000, 3, BLOCK), ("decode", "qwen3_1p7b", 32, 20000, 4, BLOCK), ("prefill", "qwen3_1p7b", 512, 1536, 2, LOOP),
    ("prefill", "qwen36_moe", 320, 450, 2, LOOP), ("prefill", "qwen38_27b", 512, 300, 3, LOOP), ("prefill", "qwen3_1p7b", 400, 500, 2, LOOP)])
def test_decode_growing_maximum(kind, shape, n_cols, base, blocks, kernel):
    """Scores that jump along the context: K rows alternate between a scale of 0.1 and a scale of 4 every eighth of the
    context, so every wave of the tile loop (its tiles are spread over the whole context, three or more a wave) and every workgroup of the kernel with one softmax
    meets low tiles first and then row maxima far beyond the threshold of its lazily updated reference maximum, and has to take the
    rescale path -- with one to four row blocks per workgroup, over several splits and, chunks, in one launch."""
    cfg = SHAPES[shape]
    rng = np.random.default_rng(base + n_cols)
    rows = base + n_cols
    shp = (rows, cfg["n_kv_heads"], cfg["head_dim"])
    scale = np.where((np.arange(rows) // (rows // 8)) % 2 == 0, 0.1, 4.0).astype(np.float32)[:, None, None]
    k16 = (rng.standard_normal(shp, dtype=np.float32) * scale).astype(np.float16).view(np.uint16)
    v16 = rng.standard_normal(shp, dtype=np.float32).astype(np.float16).view(np.uint16)
    q = rng.standard_normal((n_cols, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32)
    ref = C.attention(q, k16, v16, base)
    with _ctx_with_cache(cfg, k16, v16, rows, max_cols=n_cols) as pa:
        plan = pa.plan(kind, base, n_cols)
        assert plan["row_blocks"] == blocks and plan["split_len"] >= 3 * 32 * plan["waves"], plan     # three tiles a wave or more
        assert attn_rule(cfg, kind, base, n_cols) == (kernel, plan) and (kind == "decode") == (plan["n_splits"] > 1)
        got = pa.run_attn(kind, 0, q, base)
        # scores of standard deviation 4 over q rounded to f16 (2^-12.3 rms of each product) move by 8e-4 rms, by five times that at most over these outputs, and the weights
        # with them; P's rounding and the sums are a quarter of it.  (A reference that is not raised overflows f16.)
        assert np.abs(got - ref).max() <= 4e-3 * np.abs(ref).max()
        if n_cols <= 8 and shape != "qwen3_1p7b":                     # ... which at few outputs is within the gate of the other tests
            assert_parity(got, ref, "jumping maximum, %d row blocks" % blocks)


@pytest.mark.parametrize("shape,kv_q8,n_cols,base,blocks,groups,tiles", [
    ("qwen36_moe", False, 5, 8191, 2, 2, 2), ("qwen36_moe", False, 6, 8100, 2, 2, 1), ("qwen36_moe", False, 4, 16385, 2, 1, 2), ("qwen36_moe", False, 3, 36000, 2, 1, 3),
    ("qwen38_27b", False, 8, 50000, 3, 1, 7), ("qwen38_27b", False, 10, 4000, 2, 2, 1), ("qwen3_1p7b", False, 9, 4000, 2, 1, 1), ("qwen3_1p7b", False, 24, 4200, 3, 1, 2),
    ("qwen3_1p7b", False, 32, 12345, 4, 1, 4), ("qwen36_moe", True, 16, 8000, 2, 4, 2), ("qwen38_27b", True, 5, 20001, 2, 1, 3), ("qwen3_1p7b", True, 32, 9000, 4, 1, 3),
    ("qwen3_1p7b", False, 12, 3000, 2, 1, 1), ("qwen36_moe", False, 8, 4090, 2, 2, 1)])
def test_blocks_whose_waves_share_one_softmax(shape, kv_q8, n_cols, base, blocks, groups, tiles):
    """Blocks of two row blocks or more over several splits on the kernel that divides O by output dims (test_plan_rules.py has the lines of its rule): against the oracle, with low and high keys in turn (a raised reference), rows past the context poisoned, f32 and f16 out.  Budget of the
    decode tests.  Then value rows that are all alike: that vector comes back, whatever the rounding of P (f32 sums of the same weights above and below the
    fraction bar, a reciprocal of 1 ulp: a few 1e-7), also in a third of the splits."""
    cfg = dict(SHAPES[shape], kv_q8=kv_q8)
    rng = np.random.default_rng(base + n_cols)
    rows, tail = base + n_cols, 40
    nKV, hd = cfg["n_kv_heads"], cfg["head_dim"]
    scale = np.where((np.arange(rows) // max(rows // 9, 1)) % 2 == 0, 0.2, 2.0).astype(np.float32)[:, None, None]
    k = rng.standard_normal((rows, nKV, hd), dtype=np.float32) * scale
    v = rng.standard_normal((rows, nKV, hd), dtype=np.float32)
    q = rng.standard_normal((n_cols, cfg["n_heads"], hd), dtype=np.float32)
    gate = rng.standard_normal(q.shape, dtype=np.float32) if cfg["gate"] else None
    same = np.ascontiguousarray(np.broadcast_to(v[:1], v.shape))
    with PooledAttn(cfg, rows + tail, n_layers=1, max_cols=n_cols) as pa:
        pa.layer_alloc(0)
        pl = pa.plan("decode", base, n_cols)
        assert (pl["row_blocks"], pl["col_groups"], pl["split_len"]) == (blocks, groups, 128 * tiles) and pl["n_splits"] > 1, pl
        assert attn_rule(cfg, "decode", base, n_cols) == (BLOCK, pl)

        first_v = []                     # int8 rows: the first value row as the kernels widen it, f16 value x f16 scale

        def fill(k, v):
            pa.kv_write(0, 2 if kv_q8 else 0, rows, np.full((tail, nKV, hd // 32), np.nan, np.float32) if kv_q8 else np.full((tail, nKV, hd), 0x7e00, np.uint16))
            pa.kv_write(0, 3 if kv_q8 else 1, rows, np.full((tail, nKV, hd // 32), np.nan, np.float32) if kv_q8 else np.full((tail, nKV, hd), 0x7e00, np.uint16))
            if not kv_q8:
                k16, v16 = k.astype(np.float16).view(np.uint16), v.astype(np.float16).view(np.uint16)
                pa.kv_write(0, 0, 0, k16); pa.kv_write(0, 1, 0, v16)
                return k16, v16
            kq, ks = O.q8_quantize(k); vq, vs = O.q8_quantize(v)
            for which, a in enumerate((kq, vq, ks, vs)):
                pa.kv_write(0, which, 0, a)
            first_v[:] = [(vq[:1].reshape(1, nKV, hd // 32, 32).astype(np.float16) * vs[:1].reshape(1, nKV, hd // 32, 1).astype(np.float16)).reshape(1, nKV, hd)]
            return O.q8_dequantize(kq, ks), O.q8_dequantize(vq, vs)

        kk, vv = fill(k, v)
        ref = O.attention_values(q, kk, vv, base, gate=gate) if kv_q8 else C.attention(q, kk, vv, base, gate=gate)
        for out_dtype in (0, PA_OUT_F16):
            assert_parity(pa.run_attn("decode", 0, q, base, gate=gate, out_dtype=out_dtype).astype(np.float32), ref, "one softmax, %s %d columns at %d" % (shape, n_cols, base))
        first = pa.run_attn("decode", 0, q, base, gate=gate)
        assert np.array_equal(first, pa.run_attn("decode", 0, q, base, gate=gate))          # no atomics, fixed orders
        _, vv = fill(k, same)
        vec = (first_v[0] if kv_q8 else vv.view(np.float16))[0].astype(np.float32)
        want = np.repeat(vec, cfg["n_heads"] // nKV, axis=0)[None]
        for splits in (0, max(2, pl["n_splits"] // 3)):
            pa.set_decode_splits(splits)
            assert np.abs(pa.run_attn("decode", 0, q, base) - want).max() <= 2e-6


@pytest.mark.parametrize("shape,n_cols,base", [("qwen36_moe", 16, 700), ("qwen36_moe", 16, 760), ("qwen36_moe", 16, 1000), ("qwen36_moe", 16, 1010), ("qwen36_moe", 25, 4500), ("qwen36_moe", 26, 4500), ("qwen3_1p7b", 51, 4300),
                                               ("qwen3_1p7b", 52, 4300), ("qwen38_27b", 17, 5000)])
def test_merge_of_sixteen_columns_and_more(shape, n_cols, base):
    """Either merge kernel behind a pass of 16 columns or more: up to eight splits and past them, two fifths of the CUs' worth of workgroups and past that."""
    cfg = SHAPES[shape]
    rng = np.random.default_rng(base + n_cols)
    k16, v16 = random_cache(cfg, base + n_cols, seed=base)
    q = rng.standard_normal((n_cols, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32)
    gate = rng.standard_normal(q.shape, dtype=np.float32) if cfg["gate"] else None
    ref = C.attention(q, k16, v16, base, gate=gate)
    with _ctx_with_cache(cfg, k16, v16, base + n_cols, max_cols=n_cols) as pa:
        assert pa.plan("decode", base, n_cols)["n_splits"] > 1
        for out_dtype in (0, PA_OUT_F16):
            assert_parity(pa.run_attn("decode", 0, q, base, gate=gate, out_dtype=out_dtype).astype(np.float32), ref, "merge of %d columns at %d" % (n_cols, base), tight=True)


def _own_reference_error(q, k, v, base, waves, q_f32=False):
    """Relative error against 64 bits of attention whose waves keep a softmax reference of their own: q (unless q_f32) and P rounded to f16, all else exact; wave w
    of `waves` takes the 32-row tiles w, w + waves, ... and raises its reference when a row's maximum passes it by 8."""
    n, nH, hd = q.shape
    rows, G = k.shape[0], nH // k.shape[1]
    k, v = k.astype(np.float64), v.astype(np.float64)
    vis = np.arange(rows)[None, :] <= base + np.arange(n)[:, None]
    err = nrm = 0.0
    exact = np.empty(q.shape)
    for h in range(nH):
        kh, vh = k[:, h // G], v[:, h // G]
        s = np.where(vis, q[:, h].astype(np.float64) @ kh.T / hd ** 0.5, -np.inf)
        w = np.exp(s - s.max(1, keepdims=True))
        exact[:, h] = w @ vh / w.sum(1, keepdims=True)
        s = np.where(vis, q[:, h].astype(np.float32 if q_f32 else np.float16).astype(np.float64) @ kh.T / hd ** 0.5, -np.inf)
        M, L, O_ = np.full((waves, n), -np.inf), np.zeros((waves, n)), np.zeros((waves, n, hd))
        for t in range(-(-rows // 32)):
            i, sl = t % waves, slice(32 * t, 32 * t + 32)
            top = s[:, sl].max(1)
            m = np.where(top > M[i] + 8, top, M[i])
            a = np.exp(np.subtract(M[i], m, out=np.zeros(n), where=~np.isneginf(m)))
            p = np.exp(s[:, sl] - np.where(np.isneginf(m), 0.0, m)[:, None]).astype(np.float16).astype(np.float64)
            M[i], L[i], O_[i] = m, L[i] * a + p.sum(1), O_[i] * a[:, None] + p @ vh[sl]
        c = np.exp(M - M.max(0))
        got = np.einsum("wn,wnd->nd", c, O_) / (c * L).sum(0)[:, None]
        err += ((got - exact[:, h]) ** 2).sum(); nrm += (exact[:, h] ** 2).sum()
    return (err / nrm) ** 0.5, exact


@pytest.mark.parametrize("shape,n_cols,base,blocks,tiles", [
    ("qwen36_moe", 6, 8000, 2, 1), ("qwen38_27b", 10, 2862, 2, 1), ("qwen3_1p7b", 16, 2137, 2, 1), ("qwen36_moe", 5, 8191, 2, 2), ("qwen38_27b", 5, 12001, 2, 2),
    ("qwen3_1p7b", 24, 4200, 3, 2), ("qwen38_27b", 8, 50000, 3, 7)])
def test_one_softmax_for_four_waves_is_as_exact_as_four(shape, n_cols, base, blocks, tiles):
    """The workgroup's one reference rounds P a little worse than a reference a wave does; the low halves of q make up for it: the error against 64 bits is
    at most that of waves with references of their own, on unit-variance keys, values and queries.  (2.5 to 2.9e-4 there; 0.92 to 0.98 of it measured, without the
    low halves 1.01 to 1.06.  f32 sums and exponentials add 1e-6.)"""
    cfg = SHAPES[shape]
    rng = np.random.default_rng(base + n_cols)
    k16, v16 = random_cache(cfg, base + n_cols, seed=base)
    q = rng.standard_normal((n_cols, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32)
    with _ctx_with_cache(cfg, k16, v16, base + n_cols, max_cols=n_cols) as pa:
        pl = pa.plan("decode", base, n_cols)
        assert (pl["row_blocks"], pl["split_len"]) == (blocks, 128 * tiles) and pl["n_splits"] > 1, pl
        assert attn_rule(cfg, "decode", base, n_cols) == (BLOCK, pl)
        got = pa.run_attn("decode", 0, q, base)
    limit, exact = _own_reference_error(q, k16.view(np.float16).reshape(base + n_cols, cfg["n_kv_heads"], -1), v16.view(np.float16).reshape(base + n_cols, cfg["n_kv_heads"], -1),
                                        base, 4 * pl["n_splits"])
    err = (((got - exact) ** 2).sum() / (exact ** 2).sum()) ** 0.5
    print("error %.4e, own references %.4e, ratio %.4f" % (err, limit, err / limit))
    assert err <= limit


WIDE_GROUPS = [(256, 34, 2, False, (0, 100, 128, 129, 300, 16384, 16390)), (256, 64, 2, True, (127, 2000, 16390, 33000)), (256, 24, 1, False, (200, 33000)),
               (128, 33, 1, False, (0, 127, 200, 300, 400, 2000, 4097)), (128, 64, 1, True, (130, 260, 300, 2000)), (128, 64, 2, False, (100, 2000, 10000, 33000)), (128, 20, 1, False, (128, 700, 33000))]


@pytest.mark.parametrize("kv_q8", [False, True])
@pytest.mark.parametrize("head_dim,n_heads,n_kv,gate,bases", WIDE_GROUPS)
def test_one_column_of_more_than_sixteen_heads_a_kv_head(head_dim, n_heads, n_kv, gate, bases, kv_q8):
    """Two to four row blocks whose own row is a partial of its own, either side of the lengths where the plan changes its kernel or its tiles a wave, with rows past the
    column poisoned; the same through the prefill entry point, under a splits override, and as the columns of a column-exact block (bit for bit)."""
    cfg = dict(n_heads=n_heads, n_kv_heads=n_kv, head_dim=head_dim, n_rot=64, rope_theta=1e6, eps=1e-6, qk_norm=True, gate=gate, kv_q8=kv_q8)
    rng = np.random.default_rng(n_heads + head_dim)
    rows = max(bases) + 40
    k, v = rng.standard_normal((2, rows, n_kv, head_dim), dtype=np.float32)
    q = rng.standard_normal((3, n_heads, head_dim), dtype=np.float32)
    g = rng.standard_normal(q.shape, dtype=np.float32) if gate else None
    if kv_q8:
        kq, ks = O.q8_quantize(k); vq, vs = O.q8_quantize(v)
        parts, bad = [kq, vq, ks, vs], {2: np.nan, 3: np.nan}
        kf, vf = O.q8_dequantize(kq, ks), O.q8_dequantize(vq, vs)
    else:
        parts, bad = [x.astype(np.float16).view(np.uint16) for x in (k, v)], {0: NAN16, 1: NAN16}
    def ref(base, n):
        return O.attention_values(q[:n], kf[:base + n], vf[:base + n], base, gate=None if g is None else g[:n]) if kv_q8 else \
            C.attention(q[:n], parts[0][:base + n], parts[1][:base + n], base, gate=None if g is None else g[:n])
    def fill(pa, live):
        for w, x in enumerate(parts):
            x = x.copy()
            if w in bad:
                x[live:] = bad[w]
            pa.kv_write(0, w, 0, x)
    one = lambda pa, c, base, kind="decode": pa.run_attn(kind, 0, q[c:c + 1], base, gate=None if g is None else g[c:c + 1])  # noqa: E731
    with PooledAttn(cfg, rows, n_layers=1, max_cols=4) as pa:
        pa.layer_alloc(0)
        for base in bases:
            fill(pa, base + 1)
            want = ref(base, 1)
            what = "%d / %d heads of %d, %s, at %d" % (n_heads, n_kv, head_dim, "q8" if kv_q8 else "f16", base)
            got = one(pa, 0, base)
            assert_parity(got, want, what)
            assert np.array_equal(got, one(pa, 0, base, "prefill"))
            for splits in (2, 5):
                pa.set_decode_splits(splits)
                assert_parity(one(pa, 0, base), want, what + ", splits %d" % splits)
            pa.set_decode_splits(0)
    with PooledAttn(dict(cfg, verify_exact=True), rows, n_layers=1, max_cols=4) as pa:
        pa.layer_alloc(0)
        base = bases[-2]
        fill(pa, base + 3)
        got = pa.run_attn("decode", 0, q, base, gate=g)
        assert_parity(got, ref(base, 3), "column-exact block of %d / %d heads" % (n_heads, n_kv))
        for c in range(3):
            assert np.array_equal(got[c], one(pa, c, base + c)[0])


@pytest.mark.parametrize("kind,shape,n_cols,rows", [("decode", "qwen3_1p7b", 2, 256), ("decode", "qwen3_1p7b", 4, 200), ("decode", "qwen3_1p7b", 8, 240), ("decode", "qwen36_moe", 2, 256),
                                                    ("decode", "qwen38_27b", 2, 200), ("prefill", "qwen36_moe", 4, 250), ("prefill", "qwen38_27b", 4, 256), ("prefill", "qwen3_1p7b", 16, 256)])
def test_a_few_columns_over_a_short_context_are_as_exact_as_a_tile_a_wave(kind, shape, n_cols, rows):
    """Blocks of a few columns over 129 to 256 rows, in one launch or two: the error against 64 bits is that of tiles with softmax references of their own.  (Which rows
    are a tile differs between the two, which moves it by 1 % at most; with two tiles a wave it is 1.06 to 1.2 times as large.)"""
    cfg = SHAPES[shape]
    rng = np.random.default_rng(rows + n_cols)
    base = rows - n_cols
    err2 = lim2 = 0.0
    for seed in range(8):
        k16, v16 = random_cache(cfg, rows, seed=seed)
        q = rng.standard_normal((n_cols, cfg["n_heads"], cfg["head_dim"]), dtype=np.float32)
        with _ctx_with_cache(cfg, k16, v16, rows, max_cols=n_cols) as pa:
            got = pa.run_attn(kind, 0, q, base)
        k, v = [x.view(np.float16).reshape(rows, cfg["n_kv_heads"], -1) for x in (k16, v16)]
        lim, exact = _own_reference_error(q, k, v, base, 8, n_cols * cfg["n_heads"] // cfg["n_kv_heads"] <= 8)
        err2 += ((got - exact) ** 2).sum() / (exact ** 2).sum(); lim2 += lim ** 2
    print("error %.4e, a tile a wave %.4e, ratio %.4f" % ((err2 / 8) ** 0.5, (lim2 / 8) ** 0.5, (err2 / lim2) ** 0.5))
    assert err2 <= lim2 * 1.02 ** 2

"""GPU tests of the one-token projections either side of the attention block (pa_gemv, pa_gemv_norm,
pa_attn_layer_decode) through the C ABI, against the oracle's dequantise-and-multiply in f64.

The reference checks its GEMVs against a CPU product of the dequantised weights with a tolerance relative to the
output scale (engine/selftest.js:120-139: max-abs / scale < 2e-3; tests/test_gemm.js:13-14, :105: ~1e-6 for
summation order alone).  Here: 2e-5 of the largest output for a GEMV alone, the path's 2e-3 / 1e-2 gate for the layer.
"""
import numpy as np
import pytest
from oracle import attn_oracle as O
from pooled_amd.capi import PooledAttn, PaError, PA_W_F32, PA_W_Q8_0, PA_W_Q4_0, PA_ERR_INVALID, PA_ERR_UNSUPPORTED
from helpers import SHAPES, assert_parity, oracle_cache

pytestmark = pytest.mark.gpu


def _weights(kind, d_out, d_in, rng, scale=0.02):
    """Random weight planes of a kind: (w, scales-or-None)."""
    if kind == PA_W_F32:
        return (rng.standard_normal((d_out, d_in)) * scale).astype(np.float32), None
    sc = np.asarray(rng.uniform(0.5, 1.5, (d_out, d_in // 32)) * scale / (127 if kind == PA_W_Q8_0 else 8) * 3, np.float16).view(np.uint16)
    if kind == PA_W_Q8_0:
        return rng.integers(-127, 128, (d_out, d_in)).astype(np.int8), sc
    return rng.integers(0, 256, (d_out, d_in // 2)).astype(np.uint8), sc


def _rel(got, ref):
    return np.abs(np.asarray(got, np.float64) - ref).max() / max(np.abs(ref).max(), 1e-30)


@pytest.mark.parametrize("kind", [PA_W_F32, PA_W_Q8_0, PA_W_Q4_0])
@pytest.mark.parametrize("d_out,d_in", [(9216, 2048), (2048, 4096), (1, 32), (37, 96), (5000, 6144), (130, 8192)])
def test_gemv_matches_oracle(kind, d_out, d_in):
    rng = np.random.default_rng(d_out * 7 + d_in + kind)
    w, sc = _weights(kind, d_out, d_in, rng)
    x = rng.standard_normal(d_in).astype(np.float32)
    y0 = rng.standard_normal(d_out).astype(np.float32)
    ref = O.gemv(kind, w, sc, x)
    with PooledAttn(SHAPES["qwen36_moe"], 64, n_layers=1, max_cols=1) as pa:
        wh = pa.weight(kind, w, sc)
        dx = pa.to_device(x); dy = pa.to_device(y0)
        pa.gemv(wh, dx, dy); pa.sync()
        got = dy.download(np.float32, d_out)
        assert _rel(got, ref) < 2e-5, "plain"
        pa.gemv(wh, dx, dy, acc=True); pa.sync()                      # y = W x, then y += W x
        assert _rel(dy.download(np.float32, d_out), 2.0 * ref) < 2e-5, "accumulate"
        # deterministic run to run
        pa.gemv(wh, dx, dy); pa.sync()
        assert np.array_equal(dy.download(np.float32, d_out), got)


# sizes past 4096 inputs that take every number of rows a wave with and without the norm (test_proj_rules.py asks the rule)
GEMV_WIDE_SIZES = [(6143, 4128), (6145, 4128), (8191, 5120), (11265, 4160), (14337, 6144), (9001, 6176), (6150, 8192),
                   (14335, 5120), (4000, 4128), (6144, 4128), (4111, 8192), (1000, 7968), (9003, 6016),
                   (7001, 6144), (7001, 4128), (8603, 4128), (18753, 7168)]


@pytest.mark.parametrize("kind", [PA_W_Q8_0, PA_W_Q4_0])
@pytest.mark.parametrize("d_out,d_in", GEMV_WIDE_SIZES)
def test_gemv_many_rows_a_wave(kind, d_out, d_in):
    """Past 4096 inputs: one to seven rows a wave (d_out over the SIMDs picks), the last wave's rows past the end repeating the last
    one.  Every tenth row and the last ones are checked."""
    rng = np.random.default_rng(d_out + d_in + kind)
    w, sc = _weights(kind, d_out, d_in, rng)
    x = rng.standard_normal(d_in).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(d_in)).astype(np.float32)
    y0 = rng.standard_normal(d_out).astype(np.float32)
    rows = np.unique(np.r_[0:d_out:10, d_out - 9:d_out])
    cfg = SHAPES["qwen36_moe"]
    ref = O.gemv(kind, w[rows], sc[rows], x)
    ref_n = O.gemv(kind, w[rows], sc[rows], O.rmsnorm(x, nw, cfg["eps"]).astype(np.float32))
    with PooledAttn(cfg, 64, n_layers=1, max_cols=1) as pa:
        wh = pa.weight(kind, w, sc)
        dx = pa.to_device(x); dn = pa.to_device(nw); dy = pa.to_device(np.r_[y0, np.float32(7)])
        pa.gemv(wh, dx, dy, acc=True); pa.sync()
        got = dy.download(np.float32, d_out + 1)
        assert got[d_out] == 7 and _rel(got[rows], ref + y0[rows]) < 2e-5
        pa.gemv_norm(wh, dx, dn, dy); pa.sync()
        got = dy.download(np.float32, d_out + 1)
        assert got[d_out] == 7 and _rel(got[rows], ref_n) < 2e-5


# one or two workgroups a CU that stay for the whole call, one to eight rows a wave (test_proj_rules.py asks the rule): counts that come out
# even, one row more or less, and the first size that is left to the rows above
GEMV_RESIDENT_SIZES = [(1024, 4128), (1025, 8192), (2047, 4160), (2049, 5120), (3071, 7008), (3073, 6144), (4001, 7008), (4097, 6400), (5120, 6144), (5121, 8192), (6145, 6208), (7169, 8192),
                       (8192, 4160), (8193, 8160), (10241, 6144), (10241, 7008), (12289, 8192), (14337, 6208), (16384, 6144), (16385, 4128),
                       (4112, 5120), (4113, 6400), (5501, 5152), (6803, 5632), (7901, 5152), (9001, 5120)]


@pytest.mark.parametrize("kind", [PA_W_Q8_0, PA_W_Q4_0])
@pytest.mark.parametrize("d_out,d_in", GEMV_RESIDENT_SIZES)
def test_gemv_resident_workgroups(kind, d_out, d_in):
    """Every row against the f64 product of the dequantised weights, with the norm, without it and accumulating: rows dealt to waves whose counts
    differ by one.  2e-5 of the largest output, the bound of the tests above: f32 sums of up to 8192 products, 4 to 8e-7 measured there."""
    rng = np.random.default_rng(d_out + 3 * d_in + kind)
    w, sc = _weights(kind, d_out, d_in, rng)
    x = rng.standard_normal(d_in).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(d_in)).astype(np.float32)
    y0 = rng.standard_normal(d_out).astype(np.float32)
    cfg = SHAPES["qwen36_moe"]
    ref = O.gemv(kind, w, sc, x)
    ref_n = O.gemv(kind, w, sc, O.rmsnorm(x, nw, cfg["eps"]).astype(np.float32))
    with PooledAttn(cfg, 64, n_layers=1, max_cols=1) as pa:
        wh = pa.weight(kind, w, sc)
        dx = pa.to_device(x); dn = pa.to_device(nw); dy = pa.to_device(np.r_[y0, np.float32(7)])
        for call, want in ((lambda: pa.gemv(wh, dx, dy, acc=True), ref + y0), (lambda: pa.gemv(wh, dx, dy), ref), (lambda: pa.gemv_norm(wh, dx, dn, dy), ref_n)):
            call(); pa.sync()
            got = dy.download(np.float32, d_out + 1)
            assert got[d_out] == 7 and _rel(got[:d_out], want) < 2e-5


@pytest.mark.parametrize("kind", [PA_W_F32, PA_W_Q4_0])
def test_gemv_norm_matches_rmsnorm_then_gemv(kind):
    cfg = SHAPES["qwen36_moe"]
    d_out, d_in = 1024 + 3, 2048
    rng = np.random.default_rng(11 + kind)
    w, sc = _weights(kind, d_out, d_in, rng)
    x = (rng.standard_normal(d_in) * 3.0).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(d_in)).astype(np.float32)
    xn_ref = O.rmsnorm(x, nw, cfg["eps"])
    ref = O.gemv(kind, w, sc, xn_ref)
    with PooledAttn(cfg, 64, n_layers=1, max_cols=1) as pa:
        wh = pa.weight(kind, w, sc)
        dx = pa.to_device(x); dnw = pa.to_device(nw); dy = pa.alloc(d_out * 4); dxn = pa.alloc(d_in * 4)
        pa.gemv_norm(wh, dx, dnw, dy, dxn); pa.sync()
        assert _rel(dxn.download(np.float32, d_in), xn_ref.astype(np.float64)) < 1e-6
        assert _rel(dy.download(np.float32, d_out), ref) < 2e-5
        pa.gemv_norm(wh, dx, dnw, dy); pa.sync()                      # without the xn copy
        assert _rel(dy.download(np.float32, d_out), ref) < 2e-5


def test_weight_and_gemv_errors():
    with PooledAttn(SHAPES["qwen36_moe"], 64, n_layers=1, max_cols=1) as pa:
        with pytest.raises(PaError) as e:
            pa.weight(PA_W_Q8_0, np.zeros((4, 48), np.int8), np.zeros((4, 1), np.uint16))       # d_in not a multiple of 32
        assert e.value.code == PA_ERR_INVALID
        with pytest.raises(PaError) as e:
            pa.weight(PA_W_Q4_0, np.zeros((4, 8192), np.uint8), np.zeros((4, 512), np.uint16))  # d_in 16384
        assert e.value.code == PA_ERR_UNSUPPORTED
        with pytest.raises(PaError) as e:
            pa.weight(7, np.zeros((4, 32), np.float32))
        assert e.value.code == PA_ERR_INVALID


@pytest.mark.parametrize("shape,dim,kind,pos", [("qwen36_moe", 2048, PA_W_Q4_0, 777), ("qwen36_moe", 2048, PA_W_Q8_0, 0),
                                                 ("qwen3_1p7b", 2048, PA_W_Q4_0, 300), ("qwen38_27b", 5120, PA_W_Q8_0, 1029)])
def test_attn_layer_decode_matches_oracle(shape, dim, kind, pos):
    """rmsnorm -> [q | k | v] -> pre-step -> attention over the cache -> gate -> wo, accumulated into x: the residual
    and the new cache rows against the oracle's composition of the same stages."""
    cfg = SHAPES[shape]
    nH, nKV, hd = cfg["n_heads"], cfg["n_kv_heads"], cfg["head_dim"]
    qd, kvd = nH * hd, nKV * hd
    q_rows = qd * (2 if cfg["gate"] else 1)
    rng = np.random.default_rng(pos + dim)
    w_qkv, s_qkv = _weights(kind, q_rows + 2 * kvd, dim, rng, scale=0.03)
    w_o, s_o = _weights(kind, dim, qd, rng, scale=0.03)
    x = rng.standard_normal(dim).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(dim)).astype(np.float32)
    qw = (1 + 0.1 * rng.standard_normal(hd)).astype(np.float32); kw = (1 + 0.1 * rng.standard_normal(hd)).astype(np.float32)
    k16, v16 = oracle_cache(cfg, rng.standard_normal((pos, kvd)).astype(np.float32), rng.standard_normal((pos, kvd)).astype(np.float32), kw)
    x_ref, k_row, v_row = O.attn_layer_decode(x, kind, w_qkv, s_qkv, kind, w_o, s_o, nw, qw, kw, k16, v16, pos, cfg)
    with PooledAttn(cfg, pos + 8, n_layers=1, max_cols=1) as pa:
        pa.layer_alloc(0)
        if pos:
            pa.kv_write(0, 0, 0, k16); pa.kv_write(0, 1, 0, v16)
        wq = pa.weight(kind, w_qkv, s_qkv); wo = pa.weight(kind, w_o, s_o)
        dx = pa.to_device(x); dnw = pa.to_device(nw); dqw = pa.to_device(qw); dkw = pa.to_device(kw)
        pa.attn_layer_decode(0, wq, wo, dnw, dqw, dkw, dx, pos); pa.sync()
        got = dx.download(np.float32, dim)
        kc = pa.kv_read(0, 0, pos, 1).view(np.float16).astype(np.float64); vc = pa.kv_read(0, 1, pos, 1).view(np.float16).astype(np.float64)
    assert_parity(got, x_ref, "layer %s pos %d" % (shape, pos))
    # the new cache rows: f16 of GEMV outputs that differ from the oracle's f64 products in the last f32 bits, so a
    # value next to a rounding boundary may land one f16 step away
    for a, b in ((kc, k_row), (vc, v_row)):
        ref = np.asarray(b).reshape(a.shape).view(np.float16).astype(np.float64)
        assert np.abs(a - ref).max() <= np.abs(ref).max() * 2.0 ** -10


# ---- column-batched passes: rmsnorm -> f16, GEMM on the matrix cores, the whole attention half of a layer ----

@pytest.mark.parametrize("kind", [PA_W_F32, PA_W_Q8_0, PA_W_Q4_0])
@pytest.mark.parametrize("d_out,d_in,n", [(9216, 2048, 300), (2048, 4096, 129), (37, 96, 5), (130, 8192, 40), (256, 32, 128), (384, 96, 700),
                                          (100, 384, 65), (64, 128, 33), (4096, 2048, 512),
                                          (9216, 2048, 8), (2048, 4096, 16), (130, 8192, 3), (70, 64, 1), (2048, 4096, 31), (130, 8192, 17)])
def test_gemm_matches_oracle(kind, d_out, d_in, n):
    """One size or more of every kernel (on a 256-CU part): 128 x 128 tiles (9216 rows, 300 columns) and 64 x 128 ones (4096 rows, 512
    columns); 64 columns x 32 rows with many stages, three and one (129, 40, 65 and 33 columns); d_in not a multiple of 128 past the few
    columns, and f32 weights up to 16 columns, on the kernel that widens in its loop; quantised weights from (37, 96, 5) and
    (9216, 2048, 8) on from the packed planes, but 17 columns of 8192 Q8_0 inputs on 64 x 32 tiles."""
    rng = np.random.default_rng(d_out + 3 * d_in + n + kind)
    w, sc = _weights(kind, d_out, d_in, rng)
    x16 = rng.standard_normal((n, d_in)).astype(np.float16)
    ref = O.gemm_f16(kind, w, sc, x16.astype(np.float32))
    xs, ys = d_in + 8, d_out + 5                                      # padded strides
    xpad = np.zeros((n, xs), np.float16); xpad[:, :d_in] = x16
    y0 = rng.standard_normal((n, ys)).astype(np.float32)
    with PooledAttn(SHAPES["qwen36_moe"], 64, n_layers=1, max_cols=1) as pa:
        wh = pa.weight(kind, w, sc)
        dx = pa.to_device(xpad.view(np.uint16)); dy = pa.to_device(y0)
        pa.gemm(wh, dx, xs, n, dy, ys); pa.sync()
        got = dy.download(np.float32, n * ys).reshape(n, ys)
        assert _rel(got[:, :d_out], ref) < 2e-5, "plain"
        assert np.array_equal(got[:, d_out:], y0[:, d_out:]), "the stride padding of y must stay untouched"
        pa.gemm(wh, dx, xs, n, dy, ys, acc=True); pa.sync()
        assert _rel(dy.download(np.float32, n * ys).reshape(n, ys)[:, :d_out], 2.0 * ref) < 2e-5, "accumulate"


@pytest.mark.parametrize("kind", [PA_W_F32, PA_W_Q8_0, PA_W_Q4_0])
@pytest.mark.parametrize("d_out,d_in,n", [(9216 - 40, 2048, 4096 - 3), (2048, 4096, 4000), (4090, 256, 4096), (600, 128, 11000),
                                          (2048, 4096, 600), (130, 8192, 513), (1000, 64, 1100)])
def test_gemm_large_chunks(kind, d_out, d_in, n):
    """Chunks of 512 columns and more over d_in a multiple of 128: the weights are widened to f16 in fragment order (a
    copy kept with the weight handle) and the GEMM runs over two f16 operands.  On a 256-CU part the sizes take tiles of 128 columns x
    384 rows, 128 x 256, 256 x 256, three times the 64-column kernel (64 rows, 64 and 32); d_in 64 stays on the kernel that widens
    in its loop, 256 columns a workgroup.  Ragged edges on both axes, padded strides that must stay untouched, the accumulating form (the
    second call on a handle, which finds the kept copy), and a second weight."""
    rng = np.random.default_rng(d_out + d_in + n + kind)
    w, sc = _weights(kind, d_out, d_in, rng)
    x16 = rng.standard_normal((n, d_in)).astype(np.float16)
    ref = O.gemm_f16(kind, w, sc, x16.astype(np.float32))
    xs, ys = d_in + 8, d_out + 5
    xpad = np.zeros((n, xs), np.float16); xpad[:, :d_in] = x16
    y0 = rng.standard_normal((n, ys)).astype(np.float32)
    with PooledAttn(SHAPES["qwen36_moe"], 64, n_layers=1, max_cols=1) as pa:
        wh = pa.weight(kind, w, sc)
        dx = pa.to_device(xpad.view(np.uint16)); dy = pa.to_device(y0)
        pa.gemm(wh, dx, xs, n, dy, ys); pa.sync()
        got = dy.download(np.float32, n * ys).reshape(n, ys)
        assert _rel(got[:, :d_out], ref) < 2e-5, "plain"
        assert np.array_equal(got[:, d_out:], y0[:, d_out:]), "the stride padding of y must stay untouched"
        pa.gemm(wh, dx, xs, n, dy, ys, acc=True); pa.sync()
        assert _rel(dy.download(np.float32, n * ys).reshape(n, ys)[:, :d_out], 2.0 * ref) < 2e-5, "accumulate"
        w2, sc2 = _weights(kind, d_out, d_in, rng)
        pa.gemm(pa.weight(kind, w2, sc2), dx, xs, n, dy, ys); pa.sync()
        assert _rel(dy.download(np.float32, n * ys).reshape(n, ys)[:, :d_out], O.gemm_f16(kind, w2, sc2, x16.astype(np.float32))) < 2e-5, "second weight"


# with the next list every instance of the few-column kernel that a 256-CU part takes (test_proj_rules.py asks the rule)
GEMM_FEW_SIZES = [(16, 32, 1), (17, 256, 2), (31, 288, 15), (4096, 4096, 16), (4100, 4128, 8), (4130, 8192, 9), (8200, 512, 17),
                  (8193, 2080, 32), (8192, 5120, 16), (4111, 6144, 31), (2048, 4096, 33), (600, 7968, 32),
                  (33, 4128, 5), (70, 2080, 19), (33, 256, 20), (40, 4608, 11), (48, 5120, 31),   # one row group
                  (5000, 2048, 12), (5000, 2080, 16), (5000, 2048, 24), (4111, 1056, 32),   # two of chunks of 8 blocks
                  (9216, 2048, 16), (8201, 1056, 13),                                    # four, one column block
                  (4111, 4128, 31), (8193, 4128, 9), (8200, 4128, 20), (8200, 5120, 32),   # Q4_0: two and four of chunks of 16
                  (5120, 6144, 1), (5119, 6144, 2), (1001, 8192, 4), (999, 7968, 3), (9216, 4064, 1), (3, 4128, 2), (6001, 4096, 2)]   # dot products


@pytest.mark.parametrize("kind", [PA_W_Q8_0, PA_W_Q4_0])
@pytest.mark.parametrize("d_out,d_in,n", GEMM_FEW_SIZES)
def test_gemm_few_columns(kind, d_out, d_in, n):
    """Up to 32 columns straight from the packed planes, on the matrix cores: one, two and four 16-row groups a workgroup (fewer and more of them
    than CUs, d_in either side of 4096, what fits the LDS), one and two column blocks, chunks of 8 and 16 blocks that d_in
    fills or not, ragged rows, and the first column counts of the next kernel; one to four columns over long rows on the VALU's dot
    products.  The sums are f32 in another order than the
    f64 oracle's: 2e-5 of the largest output is some 300 roundings at most."""
    rng = np.random.default_rng(d_out + 7 * d_in + n + kind)
    w, sc = _weights(kind, d_out, d_in, rng)
    x16 = rng.standard_normal((n, d_in)).astype(np.float16)
    ref = O.gemm_f16(kind, w, sc, x16.astype(np.float32))
    xs, ys = d_in + 8, d_out + 3
    xpad = np.full((n, xs), np.float16(np.nan)); xpad[:, :d_in] = x16
    y0 = rng.standard_normal((n, ys)).astype(np.float32)
    with PooledAttn(SHAPES["qwen36_moe"], 64, n_layers=1, max_cols=1) as pa:
        wh = pa.weight(kind, w, sc)
        dx = pa.to_device(xpad.view(np.uint16)); dy = pa.to_device(y0)
        pa.gemm(wh, dx, xs, n, dy, ys); pa.sync()
        got = dy.download(np.float32, n * ys).reshape(n, ys)
        assert _rel(got[:, :d_out], ref) < 2e-5, "plain"
        assert np.array_equal(got[:, d_out:], y0[:, d_out:]), "the stride padding of y must stay untouched"
        pa.gemm(wh, dx, xs, n, dy, ys, acc=True); pa.sync()
        assert _rel(dy.download(np.float32, n * ys).reshape(n, ys)[:, :d_out], 2.0 * ref) < 2e-5, "accumulate"


# one size and more for every tile that a 256-CU part takes (test_proj_rules.py asks the rule)
GEMM_TILE_SIZES = [(8074, 256, 454), (8824, 256, 451), (8594, 256, 528), (7884, 128, 834), (8208, 128, 900), (8972, 128, 1028),
                   (7342, 128, 1544), (8561, 128, 1544), (4090, 2048, 500), (2040, 384, 3000)]


@pytest.mark.parametrize("d_out,d_in,n", GEMM_TILE_SIZES)
def test_gemm_tile_shapes(d_out, d_in, n):
    """The larger tiles of wide chunks: sizes that take each of 128 columns x 128 / 160 / 192 / 256 / 320 / 384 / 448 rows, 256 x
    256 and 64 x 128 on a 256-CU part (and 128 x 256 again), one to sixteen stages, ragged on both axes.  Sums in f32 in
    another order than the f64 oracle's, products of f16 exact: 2e-5 of the largest output as above."""
    rng = np.random.default_rng(d_out + d_in + n)
    w, sc = _weights(PA_W_Q8_0, d_out, d_in, rng)
    x16 = rng.standard_normal((n, d_in)).astype(np.float16)
    ref = O.gemm_f16(PA_W_Q8_0, w, sc, x16.astype(np.float32))
    xs, ys = d_in + 8, d_out + 5
    xpad = np.full((n, xs), np.float16(np.nan)); xpad[:, :d_in] = x16
    y0 = rng.standard_normal((n, ys)).astype(np.float32)
    with PooledAttn(SHAPES["qwen36_moe"], 64, n_layers=1, max_cols=1) as pa:
        wh = pa.weight(PA_W_Q8_0, w, sc)
        dx = pa.to_device(xpad.view(np.uint16)); dy = pa.to_device(y0)
        pa.gemm(wh, dx, xs, n, dy, ys); pa.sync()
        got = dy.download(np.float32, n * ys).reshape(n, ys)
        assert _rel(got[:, :d_out], ref) < 2e-5, "plain"
        assert np.array_equal(got[:, d_out:], y0[:, d_out:]), "the stride padding of y must stay untouched"
        pa.gemm(wh, dx, xs, n, dy, ys, acc=True); pa.sync()
        assert _rel(dy.download(np.float32, n * ys).reshape(n, ys)[:, :d_out], 2.0 * ref) < 2e-5, "accumulate"


@pytest.mark.parametrize("d_out,d_in,n", [(9213, 128, 777), (8209, 256, 900), (446, 128, 25000), (4095, 256, 4095)])
def test_gemm_tile_rows_four_at_a_time(d_out, d_in, n):
    """Whole-sum tiles store four rows a lane, at any alignment of y: rows that are no multiple of four, columns back to back (a store past a column's last
    row would land in the next one) and nothing past the last.  The bounds as above."""
    rng = np.random.default_rng(d_out + n)
    w, sc = _weights(PA_W_Q8_0, d_out, d_in, rng)
    x16 = rng.standard_normal((n, d_in)).astype(np.float16)
    ref = O.gemm_f16(PA_W_Q8_0, w, sc, x16.astype(np.float32))
    with PooledAttn(SHAPES["qwen36_moe"], 64, n_layers=1, max_cols=1) as pa:
        wh = pa.weight(PA_W_Q8_0, w, sc)
        y0 = rng.standard_normal(n * d_out + 8).astype(np.float32)
        dx = pa.to_device(x16.view(np.uint16)); dy = pa.to_device(y0)
        for acc, scale in ((False, 1.0), (True, 2.0)):
            pa.gemm(wh, dx, d_in, n, dy, d_out, acc=acc); pa.sync()
            got = dy.download(np.float32, y0.size)
            assert _rel(got[:-8].reshape(n, d_out), scale * ref) < 2e-5, acc
            assert np.array_equal(got[-8:], y0[-8:]), "past the last column"


@pytest.mark.parametrize("kind", [PA_W_Q8_0, PA_W_Q4_0])
def test_gemm_weight_cache_budget(kind):
    """The kept f16 copy and the per-call staging hold the same values: a context with no budget (every call widens into
    the context's staging), one whose budget holds the first weight only, and the default give the same bits, also
    when the weights alternate through the one staging matrix."""
    d_out, d_in, n = 2100, 256, 4000
    rng = np.random.default_rng(kind)
    ws = [_weights(kind, d_out, d_in, rng) for _ in range(2)]
    x16 = rng.standard_normal((n, d_in)).astype(np.float16)
    outs = []
    for budget in (None, 0, 2112 * 256 * 2 + 64):
        with PooledAttn(SHAPES["qwen36_moe"], 64, n_layers=1, max_cols=1) as pa:
            if budget is not None:
                pa.set_weight_cache(budget)
            whs = [pa.weight(kind, w, sc) for w, sc in ws]
            dx = pa.to_device(x16.view(np.uint16)); dy = pa.alloc(n * d_out * 4)
            got = []
            for i in (0, 1, 0, 1):
                pa.gemm(whs[i], dx, d_in, n, dy, d_out); pa.sync()
                got.append(dy.download(np.float32, n * d_out))
            assert np.array_equal(got[0], got[2]) and np.array_equal(got[1], got[3])
            outs.append(got[:2])
    for o in outs[1:]:
        assert np.array_equal(o[0], outs[0][0]) and np.array_equal(o[1], outs[0][1])
    assert _rel(outs[0][0].reshape(n, d_out), O.gemm_f16(kind, ws[0][0], ws[0][1], x16.astype(np.float32))) < 2e-5


def test_rmsnorm_f16_columns():
    cfg = SHAPES["qwen36_moe"]
    dim, n = 2048, 37
    rng = np.random.default_rng(2)
    x = (rng.standard_normal((n, dim)) * rng.uniform(0.1, 10, (n, 1))).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(dim)).astype(np.float32)
    ref = np.stack([O.rmsnorm(x[c], nw, cfg["eps"]) for c in range(n)]).astype(np.float64)
    with PooledAttn(cfg, 64, n_layers=1, max_cols=1) as pa:
        dx = pa.to_device(x); dnw = pa.to_device(nw); do = pa.alloc(n * dim * 2)
        pa.rmsnorm_f16(dx, dim, dnw, dim, n, do, dim); pa.sync()
        got = do.download(np.uint16, n * dim).view(np.float16).astype(np.float64).reshape(n, dim)
    assert np.abs(got - ref).max() <= np.abs(ref).max() * 2.0 ** -10          # f16 rounding of an f32 result


@pytest.mark.parametrize("shape,dim,kind,base,n", [("qwen36_moe", 512, PA_W_Q4_0, 100, 64), ("qwen36_moe", 1024, PA_W_Q8_0, 0, 33),
                                                    ("qwen3_1p7b", 512, PA_W_Q4_0, 300, 160), ("qwen38_27b", 1024, PA_W_Q8_0, 77, 40)])
def test_attn_layer_prefill_matches_oracle(shape, dim, kind, base, n):
    cfg = SHAPES[shape]
    nH, nKV, hd = cfg["n_heads"], cfg["n_kv_heads"], cfg["head_dim"]
    qd, kvd = nH * hd, nKV * hd
    q_rows = qd * (2 if cfg["gate"] else 1)
    rng = np.random.default_rng(base + dim + n)
    w_qkv, s_qkv = _weights(kind, q_rows + 2 * kvd, dim, rng, scale=0.05)
    w_o, s_o = _weights(kind, dim, qd, rng, scale=0.005)              # keeps the residual O(1): the gate below is absolute
    x = rng.standard_normal((n, dim)).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(dim)).astype(np.float32)
    qw = (1 + 0.1 * rng.standard_normal(hd)).astype(np.float32); kw = (1 + 0.1 * rng.standard_normal(hd)).astype(np.float32)
    k16, v16 = oracle_cache(cfg, rng.standard_normal((base, kvd)).astype(np.float32), rng.standard_normal((base, kvd)).astype(np.float32), kw)
    x_ref, k_rows, v_rows = O.attn_layer_prefill(x, kind, w_qkv, s_qkv, kind, w_o, s_o, nw, qw, kw, k16, v16, base, cfg)
    xs = dim + 4
    xpad = np.zeros((n, xs), np.float32); xpad[:, :dim] = x
    with PooledAttn(cfg, base + n + 8, n_layers=1, max_cols=n) as pa:
        pa.layer_alloc(0)
        if base:
            pa.kv_write(0, 0, 0, k16); pa.kv_write(0, 1, 0, v16)
        wq = pa.weight(kind, w_qkv, s_qkv); wo = pa.weight(kind, w_o, s_o)
        dx = pa.to_device(xpad); dnw = pa.to_device(nw); dqw = pa.to_device(qw); dkw = pa.to_device(kw)
        pa.attn_layer_prefill(0, wq, wo, dnw, dqw, dkw, dx, xs, base, n); pa.sync()
        got = dx.download(np.float32, n * xs).reshape(n, xs)[:, :dim]
        kc = pa.kv_read(0, 0, base, n).view(np.float16).astype(np.float64); vc = pa.kv_read(0, 1, base, n).view(np.float16).astype(np.float64)
    assert_parity(got, x_ref, "layer prefill %s base %d n %d" % (shape, base, n))
    for a, b in ((kc, k_rows), (vc, v_rows)):
        ref = np.asarray(b).reshape(a.shape).view(np.float16).astype(np.float64)
        assert np.abs(a - ref).max() <= np.abs(ref).max() * 2.0 ** -9


@pytest.mark.parametrize("tile", [1, 0])                          # 1: always the matrix-core attention kernel; 0: the table
@pytest.mark.parametrize("shape,more,base,n", [
    ("qwen36_moe", {}, 0, 129),                                   # unsplit halves, last block ragged
    ("qwen36_moe", dict(kv_q8=True), 700, 70),                    # split over the context (merge kernel), int8 caches
    ("qwen38_27b", {}, 33, 65),                                   # six heads a kv head
    ("qwen3_1p7b", {}, 5, 200),                                   # rotation of the whole head (pairs 64 apart), no gate
    ("qwen3_1p7b", dict(qk_norm=False), 0, 97),
    ("qwen36_moe", dict(n_rot=256), 40, 48),                      # pairs 128 apart
    ("qwen36_moe", dict(n_rot=128, qk_norm=False, gate=False), 3, 61),
    ("qwen36_moe", dict(n_rot=48), 20, 50),
    ("qwen3_1p7b", dict(n_rot=32, gate=True), 0, 80),
    ("qwen36_moe", {}, 0, 5),                                     # a verify block: projections and attention of a few columns
    ("qwen36_moe", {}, 0, 660),                                   # 10560 (column, head) rows
    ("qwen3_1p7b", {}, 17, 700),
])
def test_layer_prefill_equals_its_stages(shape, more, base, n, tile):
    """The layer call leaves the bits of its stages called one by one: the residual, the cache rows, and the q and gate buffers,
    which hold the pre-step's results after either."""
    from pooled_amd.capi import PA_OUT_F16
    cfg = dict(SHAPES[shape], **more)
    nH, nKV, hd = cfg["n_heads"], cfg["n_kv_heads"], cfg["head_dim"]
    qd, kvd, dim = nH * hd, nKV * hd, 256
    q_rows = qd * (2 if cfg["gate"] else 1)
    rows = q_rows + 2 * kvd
    rng = np.random.default_rng(base * 1000 + n)
    w_qkv, s_qkv = _weights(PA_W_Q4_0, rows, dim, rng, scale=0.05)
    w_o, s_o = _weights(PA_W_Q4_0, dim, qd, rng, scale=0.005)
    nw = (1 + 0.1 * rng.standard_normal(dim)).astype(np.float32)
    hw = (1 + 0.1 * rng.standard_normal(hd)).astype(np.float32); hk = (1 + 0.1 * rng.standard_normal(hd)).astype(np.float32)
    x = rng.standard_normal((n, dim)).astype(np.float32)
    outs, caches, pre = [], [], []
    with PooledAttn(cfg, base + n + 1, n_layers=2, max_cols=max(base, n)) as pa:
        pa.set_prefill_tile(tile)
        stale = np.full(n * qd, np.nan, np.float32)
        wq = pa.weight(PA_W_Q4_0, w_qkv, s_qkv); wo = pa.weight(PA_W_Q4_0, w_o, s_o)
        dnw = pa.to_device(nw); dqw = pa.to_device(hw); dkw = pa.to_device(hk)
        kraw, vraw = (pa.to_device(rng.standard_normal((max(base, 1), kvd)).astype(np.float32)) for _ in range(2))
        for layer in (0, 1):
            pa.layer_alloc(layer)
            if base:
                pa.kv_store(layer, kraw, kvd, vraw, kvd, 0, base)
            dx = pa.to_device(x)
            for buf in (pa.q_buffer_ptr(), pa.gate_buffer_ptr()):
                pa.L.pa_upload(pa.ctx, buf, stale.ctypes.data, stale.nbytes)
            if layer == 0:
                pa.attn_layer_prefill(layer, wq, wo, dnw, dqw, dkw, dx, dim, base, n)
            else:
                dxn = pa.alloc(n * dim * 2); dqkv = pa.alloc(n * rows * 4); dat = pa.alloc(n * qd * 2)
                pa.rmsnorm_f16(dx, dim, dnw, dim, n, dxn, dim)
                pa.gemm(wq, dxn, dim, n, dqkv, rows)
                pa.L.pa_glue_kv(pa.ctx, layer, dqkv.ptr, rows, dqkv.ptr + q_rows * 4, rows, dqkv.ptr + (q_rows + kvd) * 4, rows, dqw.ptr, dkw.ptr, base, n)
                pa.attn("prefill", layer, None, 0, pa.gate_buffer_ptr() if cfg["gate"] else None, qd, base, n, dat, qd, PA_OUT_F16)
                pa.gemm(wo, dat, qd, n, dx, dim, acc=True)
            pa.sync()
            outs.append(dx.download(np.float32, n * dim))
            pre.append((pa.read_q_buffer(n), pa.read_gate_buffer(n) if cfg["gate"] else np.zeros(0)))
            caches.append([pa.kv_read(layer, w, base, n) for w in range(4 if cfg.get("kv_q8") else 2)])
    for a, b in zip(*caches):
        assert np.array_equal(np.asarray(a), np.asarray(b))
    assert np.isfinite(outs[0]).all() and np.array_equal(outs[0], outs[1])
    for a, b in zip(*pre):
        assert np.isfinite(a).all() and np.array_equal(a, b)


def test_layer_calls_on_int8_caches_equal_their_stages():
    """pa_attn_layer_decode / pa_attn_layer_prefill on int8 caches: the same bits as their stages called one by one
    (each stage has its own parity test)."""
    from pooled_amd.capi import PA_OUT_F16
    cfg = dict(SHAPES["qwen36_moe"], kv_q8=True)
    nH, nKV, hd = cfg["n_heads"], cfg["n_kv_heads"], cfg["head_dim"]
    qd, kvd, dim = nH * hd, nKV * hd, 512
    q_rows = 2 * qd
    rng = np.random.default_rng(21)
    w_qkv, s_qkv = _weights(PA_W_Q4_0, q_rows + 2 * kvd, dim, rng, scale=0.05)
    w_o, s_o = _weights(PA_W_Q4_0, dim, qd, rng, scale=0.005)
    nw = (1 + 0.1 * rng.standard_normal(dim)).astype(np.float32)
    hw = (1 + 0.1 * rng.standard_normal(hd)).astype(np.float32)
    base, n = 200, 24
    xs = rng.standard_normal((base + n + 1, dim)).astype(np.float32)
    with PooledAttn(cfg, base + n + 1, n_layers=2, max_cols=base) as pa:
        pa.layer_alloc(0); pa.layer_alloc(1)
        wq = pa.weight(PA_W_Q4_0, w_qkv, s_qkv); wo = pa.weight(PA_W_Q4_0, w_o, s_o)
        dnw = pa.to_device(nw); dhw = pa.to_device(hw)
        rows = q_rows + 2 * kvd
        for layer, staged in ((0, False), (1, True)):
            # a chunk of `base` tokens, then a chunk of n, then one token
            outs = []
            for b0, cnt in ((0, base), (base, n)):
                dx = pa.to_device(xs[b0:b0 + cnt])
                if not staged:
                    pa.attn_layer_prefill(layer, wq, wo, dnw, dhw, dhw, dx, dim, b0, cnt)
                else:
                    dxn = pa.alloc(cnt * dim * 2); dqkv = pa.alloc(cnt * rows * 4); dat = pa.alloc(cnt * qd * 2)
                    pa.rmsnorm_f16(dx, dim, dnw, dim, cnt, dxn, dim)
                    pa.gemm(wq, dxn, dim, cnt, dqkv, rows)
                    pa.L.pa_glue_kv(pa.ctx, layer, dqkv.ptr, rows, dqkv.ptr + q_rows * 4, rows, dqkv.ptr + (q_rows + kvd) * 4, rows, dhw.ptr, dhw.ptr, b0, cnt)
                    pa.attn("prefill", layer, None, 0, pa.gate_buffer_ptr(), qd, b0, cnt, dat, qd, PA_OUT_F16)
                    pa.gemm(wo, dat, qd, cnt, dx, dim, acc=True)
                pa.sync()
                outs.append(dx.download(np.float32, cnt * dim))
            dx = pa.to_device(xs[base + n])
            if not staged:
                pa.attn_layer_decode(layer, wq, wo, dnw, dhw, dhw, dx, base + n)
            else:
                dqkv = pa.alloc(rows * 4); dat = pa.alloc(qd * 4)
                pa.gemv_norm(wq, dx, dnw, dqkv)
                pa.L.pa_attn_decode_step(pa.ctx, layer, dqkv.ptr, dqkv.ptr + q_rows * 4, dqkv.ptr + (q_rows + kvd) * 4, dhw.ptr, dhw.ptr, base + n, dat.ptr, 0)
                pa.gemv(wo, dat, dx, acc=True)
            pa.sync()
            outs.append(dx.download(np.float32, dim))
            if not staged:
                first = outs
        for a, b in zip(first, outs):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
            assert np.all(np.isfinite(a))
        for w in range(4):
            assert np.array_equal(pa.kv_read(0, w, 0, base + n + 1), pa.kv_read(1, w, 0, base + n + 1))


# (n_heads, n_kv_heads, head_dim, gate), model width, columns, tile: every tile that ends with the pre-step, ragged in columns
HEADS_SIZES = [((24, 4, 256, True), 1024, 292, (1, 96, 256)), ((24, 4, 256, True), 1024, 270, (1, 128, 256)), ((32, 8, 128, True), 128, 662, (1, 128, 256)), ((32, 2, 256, True), 256, 403, (1, 160, 256)),
               ((32, 2, 256, True), 256, 514, (1, 192, 256)), ((32, 2, 256, True), 2048, 588, (1, 224, 256)), ((32, 2, 256, True), 1024, 588, (1, 256, 256)),
               ((32, 8, 128, True), 1024, 1550, (1, 320, 256)), ((16, 2, 256, True), 2048, 300, (2, 64, 256)), ((16, 8, 128, False), 256, 995, (2, 128, 128)),
               ((16, 8, 128, False), 128, 33, (4, 64, 128)), ((17, 17, 128, False), 128, 40, (4, 64, 128)), ((21, 7, 128, False), 128, 1550, (1, 128, 256))]


@pytest.mark.parametrize("more", [{}, dict(kv_q8=True), dict(qk_norm=False, n_rot=8), dict(n_rot=-1), dict(n_rot=-1, kv_q8=True, qk_norm=False)])
@pytest.mark.parametrize("heads,dim,n,tile", HEADS_SIZES)
def test_projection_that_ends_with_the_pre_step_equals_the_two(heads, dim, n, tile, more):
    """What the layer call's [q | k | v] projection leaves in the q and gate buffers and in the caches is, bit for bit, what pa_gemm and
    pa_glue_kv leave: the same sums in the same order, the same arithmetic behind them.  n_rot: a quarter of the head, the least that is
    served, and the whole head (whose rotation tables are past the LDS of the wider tiles); rows around the chunk stay as they were."""
    nH, nKV, hd, gate = heads
    cfg = dict(n_heads=nH, n_kv_heads=nKV, head_dim=hd, n_rot=hd // 4 if hd == 256 else 64, rope_theta=1e6, eps=1e-6, qk_norm=True, gate=gate)
    cfg.update(more)
    if cfg["n_rot"] < 0:
        cfg["n_rot"] = hd
    qd, kvd = nH * hd, nKV * hd
    q_rows = qd * (2 if gate else 1)
    rows, base = q_rows + 2 * kvd, 7
    rng = np.random.default_rng(n)
    w_qkv, s_qkv = _weights(PA_W_Q4_0, rows, dim, rng, scale=0.05)
    w_o, s_o = _weights(PA_W_Q4_0, dim, qd, rng, scale=0.005)
    nw = (1 + 0.1 * rng.standard_normal(dim)).astype(np.float32)
    hw = (1 + 0.1 * rng.standard_normal(hd)).astype(np.float32); hk = (1 + 0.1 * rng.standard_normal(hd)).astype(np.float32)
    x = rng.standard_normal((n, dim)).astype(np.float32)
    pre, caches = [], []
    with PooledAttn(cfg, base + n + 2, n_layers=2, max_cols=n) as pa:
        wq = pa.weight(PA_W_Q4_0, w_qkv, s_qkv); wo = pa.weight(PA_W_Q4_0, w_o, s_o)
        dnw = pa.to_device(nw); dqw = pa.to_device(hw); dkw = pa.to_device(hk)
        stale = np.full(n * qd, np.nan, np.float32)
        for layer in (0, 1):
            pa.layer_alloc(layer)
            dx = pa.to_device(x)
            for buf in (pa.q_buffer_ptr(), pa.gate_buffer_ptr()):
                pa.L.pa_upload(pa.ctx, buf, stale.ctypes.data, stale.nbytes)
            if layer == 0:
                pa.attn_layer_prefill(layer, wq, wo, dnw, dqw, dkw, dx, dim, base, n)
            else:
                dxn = pa.alloc(n * dim * 2); dqkv = pa.alloc(n * rows * 4)
                pa.rmsnorm_f16(dx, dim, dnw, dim, n, dxn, dim)
                pa.gemm(wq, dxn, dim, n, dqkv, rows)
                pa.L.pa_glue_kv(pa.ctx, layer, dqkv.ptr, rows, dqkv.ptr + q_rows * 4, rows, dqkv.ptr + (q_rows + kvd) * 4, rows, dqw.ptr, dkw.ptr, base, n)
            pa.sync()
            pre.append((pa.read_q_buffer(n), pa.read_gate_buffer(n) if gate else np.zeros(0)))
            caches.append([pa.kv_read(layer, w, 0, base + n + 2) for w in range(4 if cfg.get("kv_q8") else 2)])
    for a, b in zip(*pre):
        assert np.isfinite(a).all() and np.array_equal(a, b)
    for a, b in zip(*caches):
        assert np.array_equal(np.asarray(a), np.asarray(b))


@pytest.mark.parametrize("shape,more,kind", [("qwen3_1p7b", {}, PA_W_Q8_0), ("qwen36_moe", {}, PA_W_Q4_0), ("qwen36_moe", dict(kv_q8=True), PA_W_Q8_0),
                                             ("qwen3_1p7b", dict(gate=True, n_heads=10, n_kv_heads=2), PA_W_F32), ("qwen36_moe", dict(n_heads=13, n_kv_heads=13, gate=False), PA_W_Q4_0),
                                             ("qwen38_27b", {}, PA_W_Q4_0)])
@pytest.mark.parametrize("dim", [64, 2080])
def test_layer_decode_equals_its_stages(shape, more, kind, dim):
    """The layer call on short contexts, one workgroup a kv head up to 256 streamed rows and splits past them: the bits of pa_gemv_norm,
    pa_attn_decode_step and pa_gemv, with no streamed row, one, a whole number of tiles and of splits, one row more."""
    cfg = dict(SHAPES[shape], **more)
    nH, nKV, hd = cfg["n_heads"], cfg["n_kv_heads"], cfg["head_dim"]
    qd, kvd = nH * hd, nKV * hd
    q_rows = qd * (2 if cfg["gate"] else 1)
    rows = q_rows + 2 * kvd
    rng = np.random.default_rng(dim + qd)
    w_qkv, s_qkv = _weights(kind, rows, dim, rng, scale=0.05)
    w_o, s_o = _weights(kind, dim, qd, rng, scale=0.01)
    nw = (1 + 0.1 * rng.standard_normal(dim)).astype(np.float32)
    hw = (1 + 0.1 * rng.standard_normal(hd)).astype(np.float32)
    x = rng.standard_normal(dim).astype(np.float32)
    with PooledAttn(cfg, 640, n_layers=2, max_cols=640) as pa:
        wq = pa.weight(kind, w_qkv, s_qkv); wo = pa.weight(kind, w_o, s_o)
        dnw = pa.to_device(nw); dhw = pa.to_device(hw)
        kraw, vraw = (pa.to_device(rng.standard_normal((640, kvd)).astype(np.float32)) for _ in range(2))
        dqkv = pa.alloc(rows * 4); dat = pa.alloc(qd * 4)
        for layer in (0, 1):
            pa.layer_alloc(layer); pa.kv_store(layer, kraw, kvd, vraw, kvd, 0, 640)
        for splits in (0, 3):                                         # 3: the tile loop, several tiles a wave
            pa.set_decode_splits(splits)
            for pos in (0, 1, 127, 128, 129, 255, 256, 257, 384, 513, 639):
                dx, dy = pa.to_device(x), pa.to_device(x)
                pa.attn_layer_decode(0, wq, wo, dnw, dhw, dhw, dx, pos)
                pa.gemv_norm(wq, dy, dnw, dqkv)
                pa.L.pa_attn_decode_step(pa.ctx, 1, dqkv.ptr, dqkv.ptr + q_rows * 4, dqkv.ptr + (q_rows + kvd) * 4, dhw.ptr, dhw.ptr, pos, dat.ptr, 0)
                pa.gemv(wo, dat, dy, acc=True)
                pa.sync()
                a, b = dx.download(np.float32, dim), dy.download(np.float32, dim)
                assert np.isfinite(a).all() and np.array_equal(a.view(np.uint32), b.view(np.uint32)), "pos %d splits %d" % (pos, splits)

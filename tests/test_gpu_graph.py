"""The decode entry points under HIP graph capture (callers that replay a recorded token step instead of launching
it): after one eager warm-up call (which sizes the context's partial buffers) the fused one-token call and the
layer call record nothing but kernel launches, so a captured sequence can be replayed.  Every replay -- with eager
work and synchronisations of the library's own between the replays -- must reproduce the eager results bit for bit."""
import ctypes
import numpy as np
import pytest
from pooled_amd.capi import PooledAttn, PA_OUT_F32, PA_W_Q4_0
from helpers import SHAPES, assert_parity, random_cache
from oracle import attn_oracle as O
from oracle import c_oracle as C

pytestmark = pytest.mark.gpu
vp = ctypes.c_void_p


def _hip():
    h = ctypes.CDLL("libamdhip64.so")
    for name, args in (("hipStreamCreate", [ctypes.POINTER(vp)]), ("hipStreamDestroy", [vp]), ("hipStreamSynchronize", [vp]),
                       ("hipStreamBeginCapture", [vp, ctypes.c_int]), ("hipStreamEndCapture", [vp, ctypes.POINTER(vp)]),
                       ("hipGraphInstantiate", [ctypes.POINTER(vp), vp, vp, vp, ctypes.c_size_t]), ("hipGraphLaunch", [vp, vp]),
                       ("hipGraphExecDestroy", [vp]), ("hipGraphDestroy", [vp])):
        f = getattr(h, name); f.restype = ctypes.c_int; f.argtypes = args
    return h


def _ok(rc, what):
    assert rc == 0, "%s failed with HIP error %d" % (what, rc)


def test_decode_steps_replayed_from_a_graph():
    cfg = SHAPES["qwen36_moe"]
    nH, nKV, hd = cfg["n_heads"], cfg["n_kv_heads"], cfg["head_dim"]
    qd, kvd, dim = nH * hd, nKV * hd, 512
    base, steps = 3000, 4
    rng = np.random.default_rng(5)
    hip = _hip()
    stream = vp()
    _ok(hip.hipStreamCreate(ctypes.byref(stream)), "hipStreamCreate")
    with PooledAttn(cfg, base + steps + 1, n_layers=1, max_cols=1) as pa:
        pa._chk(pa.L.pa_set_stream(pa.ctx, stream))
        pa.layer_alloc(0)
        k0 = rng.standard_normal((base, kvd), dtype=np.float32).astype(np.float16).view(np.uint16)
        v0 = rng.standard_normal((base, kvd), dtype=np.float32).astype(np.float16).view(np.uint16)
        pa.kv_write(0, 0, 0, k0); pa.kv_write(0, 1, 0, v0)
        dq = [pa.to_device(rng.standard_normal(2 * qd, dtype=np.float32)) for _ in range(steps)]
        dk = [pa.to_device(rng.standard_normal(kvd, dtype=np.float32)) for _ in range(steps)]
        dv = [pa.to_device(rng.standard_normal(kvd, dtype=np.float32)) for _ in range(steps)]
        dw = pa.to_device((1 + 0.1 * rng.standard_normal(hd)).astype(np.float32))
        douts = [pa.alloc(qd * 4) for _ in range(steps)]
        # a layer call on top: residual in / out, Q4_0 projections
        sc = lambda r, c: np.asarray(rng.uniform(0.002, 0.004, (r, c // 32)), np.float16).view(np.uint16)
        wq = pa.weight(PA_W_Q4_0, rng.integers(0, 256, (2 * qd + 2 * kvd, dim // 2), dtype=np.uint8), sc(2 * qd + 2 * kvd, dim))
        wo = pa.weight(PA_W_Q4_0, rng.integers(0, 256, (dim, qd // 2), dtype=np.uint8), sc(dim, qd))
        x0 = rng.standard_normal(dim, dtype=np.float32)
        dx = pa.to_device(x0); dnw = pa.to_device(np.ones(dim, np.float32))

        def sequence():
            for i in range(steps):
                pa.attn_decode_step(0, dq[i], dk[i], dv[i], dw, dw, base + i, douts[i], PA_OUT_F32)
            pa.attn_layer_decode(0, wq, wo, dnw, dw, dw, dx, base + steps)

        def results():
            pa.sync()
            return [d.download(np.float32, qd).copy() for d in douts] + [dx.download(np.float32, dim).copy(),
                    pa.kv_read(0, 0, base, steps + 1).copy(), pa.kv_read(0, 1, base, steps + 1).copy()]

        sequence()                                        # eager: also the warm-up that sizes the context's buffers
        eager = results()
        assert all(np.all(np.isfinite(a)) for a in eager[:steps + 1])
        graph, gexec = vp(), vp()
        dx.upload(x0)
        _ok(hip.hipStreamBeginCapture(stream, 0), "hipStreamBeginCapture")
        sequence()
        _ok(hip.hipStreamEndCapture(stream, ctypes.byref(graph)), "hipStreamEndCapture")
        _ok(hip.hipGraphInstantiate(ctypes.byref(gexec), graph, None, None, 0), "hipGraphInstantiate")
        for rep in range(3):
            # eager work of the library's own between replays: wipe what the sequence writes, restore the residual
            pa.kv_write(0, 0, base, np.zeros((steps + 1, kvd), np.uint16)); pa.kv_write(0, 1, base, np.zeros((steps + 1, kvd), np.uint16))
            for d in douts:
                d.upload(np.zeros(qd, np.float32))
            dx.upload(x0)
            pa.sync()
            _ok(hip.hipGraphLaunch(gexec, stream), "hipGraphLaunch")
            _ok(hip.hipStreamSynchronize(stream), "hipStreamSynchronize")
            for a, b in zip(results(), eager):
                assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), "replay %d differs from the eager run" % rep
        _ok(hip.hipGraphExecDestroy(gexec), "hipGraphExecDestroy"); _ok(hip.hipGraphDestroy(graph), "hipGraphDestroy")
        pa._chk(pa.L.pa_set_stream(pa.ctx, None))
    _ok(hip.hipStreamDestroy(stream), "hipStreamDestroy")


def test_chunk_captured_before_any_eager_call_takes_a_plan_without_scratch():
    """A chunk whose cheapest plan needs partials that the context has not allocated yet: under capture it takes the
    cheapest plan that needs none, and every replay gives that plan's result; eager calls take the cheapest plan."""
    cfg = SHAPES["qwen38_27b"]
    nH, nKV, hd = cfg["n_heads"], cfg["n_kv_heads"], cfg["head_dim"]
    qd, base, n = nH * hd, 300, 144
    rng = np.random.default_rng(15)
    k16, v16 = random_cache(cfg, base + n, seed=16)
    q = rng.standard_normal((n, nH, hd), dtype=np.float32); gate = rng.standard_normal(q.shape, dtype=np.float32)
    ref = C.attention(q, k16, v16, base, gate=gate)
    hip = _hip()
    stream = vp()
    _ok(hip.hipStreamCreate(ctypes.byref(stream)), "hipStreamCreate")
    with PooledAttn(cfg, base + n, n_layers=1, max_cols=n) as pa:
        pa._chk(pa.L.pa_set_stream(pa.ctx, stream))
        pa.layer_alloc(0)
        pa.kv_write(0, 0, 0, k16); pa.kv_write(0, 1, 0, v16)
        assert pa.plan("prefill", base, n)["n_splits"] > 1
        dq, dg, dout = pa.to_device(q), pa.to_device(gate), pa.alloc(n * qd * 4)
        graph, gexec = vp(), vp()
        pa.sync()
        _ok(hip.hipStreamBeginCapture(stream, 0), "hipStreamBeginCapture")
        pa.attn("prefill", 0, dq, qd, dg, qd, base, n, dout, qd, PA_OUT_F32)
        _ok(hip.hipStreamEndCapture(stream, ctypes.byref(graph)), "hipStreamEndCapture")
        _ok(hip.hipGraphInstantiate(ctypes.byref(gexec), graph, None, None, 0), "hipGraphInstantiate")
        first = None
        for rep in range(3):
            dout.upload(np.zeros(n * qd, np.float32)); pa.sync()
            _ok(hip.hipGraphLaunch(gexec, stream), "hipGraphLaunch")
            _ok(hip.hipStreamSynchronize(stream), "hipStreamSynchronize")
            got = dout.download(np.float32, n * qd).copy().reshape(ref.shape)
            assert_parity(got, ref, "captured chunk, replay %d" % rep)
            first = got if first is None else first
            assert np.array_equal(got, first)
            assert_parity(pa.run_attn("prefill", 0, q, base, gate=gate), ref, "eager chunk between replays")
        _ok(hip.hipGraphExecDestroy(gexec), "hipGraphExecDestroy"); _ok(hip.hipGraphDestroy(graph), "hipGraphDestroy")
        pa._chk(pa.L.pa_set_stream(pa.ctx, None))
    _ok(hip.hipStreamDestroy(stream), "hipStreamDestroy")


@pytest.mark.parametrize("shape,kv_q8,base,n,tile,warm", [
    ("qwen36_moe", False, 2000, 64, 0, (900, 512)), ("qwen38_27b", False, 300, 4, 0, None), ("qwen36_moe", False, 5000, 1, 0, None), ("qwen36_moe", False, 2000, 64, 2, None),
    ("qwen38_27b", False, 300, 144, 1, None), ("qwen3_1p7b", True, 0, 40, 0, None), ("qwen36_moe", True, 3000, 256, 0, None), ("qwen36_moe", True, 90, 2, 0, None)])
def test_any_chunk_is_captured_with_the_scratch_there_is(shape, kv_q8, base, n, tile, warm):
    """A prefill call captured in a context that has allocated nothing for it, or behind an eager call of a larger chunk whose plan had no partials: it takes a plan that
    fits, and every replay gives the same result; eager calls between the replays take the cheapest plan and grow the scratch.  (An int8 chunk over at most 128 rows
    has one split whose workgroups do not write the output themselves; a few columns and the tile overrides have no estimates to choose by.)"""
    cfg = dict(SHAPES[shape], kv_q8=kv_q8)
    nH, nKV, hd = cfg["n_heads"], cfg["n_kv_heads"], cfg["head_dim"]
    qd, rows = nH * hd, max(base + n, sum(warm) if warm else 0)
    rng = np.random.default_rng(base + n)
    k, v = rng.standard_normal((2, rows, nKV, hd), dtype=np.float32)
    q = rng.standard_normal((n, nH, hd), dtype=np.float32); gate = rng.standard_normal(q.shape, dtype=np.float32) if cfg["gate"] else None
    if kv_q8:
        kq, ks = O.q8_quantize(k); vq, vs = O.q8_quantize(v)
        parts = [kq, vq, ks, vs]
        ref = O.attention_values(q, O.q8_dequantize(kq, ks)[:base + n], O.q8_dequantize(vq, vs)[:base + n], base, gate=gate)
    else:
        parts = [x.astype(np.float16).view(np.uint16) for x in (k, v)]
        ref = C.attention(q, parts[0][:base + n], parts[1][:base + n], base, gate=gate)
    hip = _hip()
    stream = vp()
    _ok(hip.hipStreamCreate(ctypes.byref(stream)), "hipStreamCreate")
    with PooledAttn(cfg, rows, n_layers=1, max_cols=max(n, warm[1] if warm else 0)) as pa:
        pa._chk(pa.L.pa_set_stream(pa.ctx, stream))
        pa.set_prefill_tile(tile)
        pa.layer_alloc(0)
        for w, x in enumerate(parts):
            pa.kv_write(0, w, 0, x)
        if warm:
            assert pa.plan("prefill", warm[0], warm[1])["n_splits"] == 1 and pa.plan("prefill", base, n)["n_splits"] > 1
            pa.run_attn("prefill", 0, rng.standard_normal((warm[1], nH, hd), dtype=np.float32), warm[0])
        dq, dg, dout = pa.to_device(q), pa.to_device(gate) if cfg["gate"] else None, pa.alloc(n * qd * 4)
        graph, gexec = vp(), vp()
        pa.sync()
        _ok(hip.hipStreamBeginCapture(stream, 0), "hipStreamBeginCapture")
        pa.attn("prefill", 0, dq, qd, dg, qd if dg else 0, base, n, dout, qd, PA_OUT_F32)
        _ok(hip.hipStreamEndCapture(stream, ctypes.byref(graph)), "hipStreamEndCapture")
        _ok(hip.hipGraphInstantiate(ctypes.byref(gexec), graph, None, None, 0), "hipGraphInstantiate")
        first = None
        for rep in range(3):
            dout.upload(np.zeros(n * qd, np.float32)); pa.sync()
            _ok(hip.hipGraphLaunch(gexec, stream), "hipGraphLaunch")
            _ok(hip.hipStreamSynchronize(stream), "hipStreamSynchronize")
            got = dout.download(np.float32, n * qd).copy().reshape(ref.shape)
            assert_parity(got, ref, "captured %s %d columns at %d, replay %d" % (shape, n, base, rep))
            first = got if first is None else first
            assert np.array_equal(got, first)
            assert_parity(pa.run_attn("prefill", 0, q, base, gate=gate), ref, "eager call between replays")
        _ok(hip.hipGraphExecDestroy(gexec), "hipGraphExecDestroy"); _ok(hip.hipGraphDestroy(graph), "hipGraphDestroy")
        pa._chk(pa.L.pa_set_stream(pa.ctx, None))
    _ok(hip.hipStreamDestroy(stream), "hipStreamDestroy")

"""What a user of the library has it do, as timed cases: tokens, verify blocks, prompt chunks and session switches of the
three model shapes of the tests and the benchmark, through pooled_amd.capi.

Interface: listed() and draw(rng) give cases (dicts of plain values), prepare(case, seed) the state a program holds before
the call, run(state) one pass, work(case) its unavoidable bytes and flops, tolerance(case) how far two correct results
may be apart.

A pass covers several attention layers, each with weights and caches of its own, as a model's token or chunk does: the
layers' data together exceed the last-level cache, or, for the smallest passes, are what such a program really touches
between two tokens.  All passes go to one stream, like the one command queue of an engine.
"""
import torch

from pooled_amd.capi import (PA_OUT_F16, PA_OUT_F32, PA_W_Q4_0, PA_W_Q8_0, PooledAttn)

# attention shapes and model widths: Qwen3-1.7B (28 attention layers), Qwen3.6-35B-MoE (10), Qwen3.8-27B (16)
SHAPES = {
    "qwen3_1p7b": dict(dim=2048, n_heads=16, n_kv_heads=8, head_dim=128, n_rot=128, rope_theta=1e6, eps=1e-6, qk_norm=True, gate=False),
    "qwen36_moe": dict(dim=2048, n_heads=16, n_kv_heads=2, head_dim=256, n_rot=64, rope_theta=1e7, eps=1e-6, qk_norm=True, gate=True),
    "qwen38_27b": dict(dim=5120, n_heads=24, n_kv_heads=4, head_dim=256, n_rot=64, rope_theta=1e7, eps=1e-6, qk_norm=True, gate=True),
}
MODEL_LAYERS = {"qwen3_1p7b": 28, "qwen36_moe": 10, "qwen38_27b": 16}
WEIGHT_KINDS = {"q4_0": PA_W_Q4_0, "q8_0": PA_W_Q8_0}

# columns a context is made for: its prompts are fed in chunks of this many (or wider, where the case says so)
BATCH_COLS = 2048

# path: "layer" = the whole attention half of a layer (norm, projections, pre-step, cache write, attention, gate, output
#       projection into the residual), "attn" = the attention block alone, between an engine's own projections,
#       "session" = switch from one saved session to another
# pos:  cache rows before the pass;  cols: tokens of the pass;  exact: verify columns bit-equal to one-token decodes
_DEFAULTS = dict(weights="q4_0", kv_q8=False, exact=False, cols=1)


def _case(name, path, shape, layers, pos, **more):
    return dict(_DEFAULTS, name=name, path=path, shape=shape, layers=layers, pos=pos, **more)


def listed():
    return [
        # the first tokens of a chat on the small dense model, all layers: many small launches, little data
        _case("token_dense_203", "layer", "qwen3_1p7b", 28, 203, weights="q8_0"),
        # a token at 32K context, all attention layers of the MoE model: the benchmark's headline context
        _case("token_moe_32k", "layer", "qwen36_moe", 10, 32768),
        # a token on int8 caches at an odd position, half of the 27B model's layers (a room worker's share)
        _case("token_27b_int8_20k", "layer", "qwen38_27b", 8, 20011, kv_q8=True),
        # a draft of four tokens checked in one pass through the layers
        _case("verify_moe_5_at_8k", "layer", "qwen36_moe", 10, 8191, cols=5),
        # an 8-token draft over a 64K context, attention alone (the benchmark's verify configuration)
        _case("verify_27b_8_at_64k", "attn", "qwen38_27b", 8, 65536, cols=8),
        # the same kind of draft for an engine that needs speculative decoding to repeat plain decoding bit for bit
        _case("verify_exact_moe_4_at_12k", "attn", "qwen36_moe", 10, 12001, cols=4, exact=True),
        # a full-width pass of an engine that feeds its prompts 16 columns at a time
        _case("chunk_moe_16_at_12k", "layer", "qwen36_moe", 10, 12345, cols=16),
        # a mid-size chunk of a short prompt (the benchmark's short prefill configuration), all layers
        _case("chunk_dense_512_at_1536", "layer", "qwen3_1p7b", 28, 1536, cols=512, weights="q8_0"),
        # a ragged rest of a prompt on int8 caches
        _case("chunk_27b_777_int8_at_5k", "layer", "qwen38_27b", 8, 5003, cols=777, kv_q8=True),
        # the first wide chunk of a long prompt
        _case("chunk_moe_4096_at_0", "layer", "qwen36_moe", 10, 0, cols=4096),
        # the last wide chunk of a 128K prompt, attention alone (the benchmark's long prefill configuration)
        _case("chunk_moe_4096_at_124k", "attn", "qwen36_moe", 1, 126976, cols=4096),
        # from one conversation to another: the running session saved, the other one restored
        _case("session_moe_9k", "session", "qwen36_moe", 10, 9001),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more case of the same ranges: every path, shape and option of the listed ones, sizes by their logarithm."""
    shape = rng.choice(sorted(SHAPES))
    far = {"qwen3_1p7b": 32768, "qwen36_moe": 126976, "qwen38_27b": 65536}[shape]
    kv_q8 = rng.random() < 0.25
    most = {"qwen3_1p7b": 12 if kv_q8 else 20, "qwen36_moe": 10, "qwen38_27b": 8}[shape]
    c = dict(_DEFAULTS, shape=shape, layers=rng.randint(4, most), weights=rng.choice(["q4_0", "q8_0"]), kv_q8=kv_q8)
    kind = rng.choice(["token", "token", "verify", "verify", "chunk", "chunk", "chunk", "session"])
    if kind == "token":
        return dict(c, path=rng.choice(["layer", "layer", "attn"]), pos=_log_int(rng, 16, min(far, 65536)))
    if kind == "verify":
        path = rng.choice(["layer", "attn"])
        return dict(c, path=path, pos=_log_int(rng, 128, min(far, 65536)), cols=rng.randint(2, 16), exact=path == "attn" and rng.random() < 0.4)
    if kind == "session":
        return dict(c, path="session", pos=_log_int(rng, 64, 32768))
    c = dict(c, path=rng.choice(["layer", "layer", "attn"]), cols=_log_int(rng, 17, 4096), pos=_log_int(rng, 16, far) - 16)
    # at most the work of the largest listed case, long chunks over fewer layers
    while c["layers"] > 1 and work(c)["flops"] > 4e12:
        c["layers"] -= 1
    while work(c)["flops"] > 8e12:
        c["pos"] = c["pos"] * 3 // 4
    return c


class _Buf:
    """A tensor where the binding takes one of its device buffers."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, tensor.data_ptr()


class _Context(PooledAttn):
    """A context that goes with its last reference, launching on the program's stream."""

    def __init__(self, *a, **k):
        super().__init__(*a, **k)
        self._chk(self.L.pa_set_stream(self.ctx, _stream().cuda_stream))

    def __del__(self):
        if getattr(self, "ctx", None):
            self.sync()
            self.close()


_streams = []


def _stream():
    if not _streams:
        _streams.append(torch.cuda.Stream())
    return _streams[0]


class _CacheMemory:
    """A cache tensor's device memory as torch sees it; keeps the context alive as long as a view of it lives."""

    def __init__(self, pa, layer, which, shape, typestr):
        self.pa = pa
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, data=(pa.L.pa_kv_device_ptr(pa.ctx, layer, which), False), version=2)


def _cache(pa, layer):
    """[nKV, max_seq + 32, ...] views of a layer's K and V (int8 caches: and of their scales), in the device's layout."""
    nkv, hd, rows = pa.cfg["n_kv_heads"], pa.cfg["head_dim"], pa.max_seq + 32
    parts = [(0, hd, "|i1"), (1, hd, "|i1"), (2, hd // 32, "<f4"), (3, hd // 32, "<f4")] if pa.cfg["kv_q8"] else [(0, hd, "<f2"), (1, hd, "<f2")]
    return [torch.as_tensor(_CacheMemory(pa, layer, which, (nkv, rows, n), t), device="cuda") for which, n, t in parts]


def _fill(pa, layer, rows, gen):
    """Cache rows [0, rows): unit-variance keys and values, as the norms in front of the cache leave them."""
    kvd = pa.kv_dim
    for r in range(0, rows, BATCH_COLS):
        n = min(BATCH_COLS, rows - r)
        k, v = torch.randn(2, n, kvd, device="cuda", generator=gen)
        torch.cuda.current_stream().synchronize()
        pa.kv_store(layer, _Buf(k), kvd, _Buf(v), kvd, r, n)
        pa.sync()


def _weight(pa, kind, d_out, d_in, gen):
    """Random quantised rows whose products keep the variance of what goes in."""
    spread = torch.rand(d_out, d_in // 32, device="cuda", generator=gen) + 0.5
    if kind == "q4_0":
        low, high = torch.randint(1, 16, (2, d_out, d_in // 2), device="cuda", dtype=torch.uint8, generator=gen)   # zero-mean: -7 .. 7
        w = low | high << 4
        s = spread / (4.5 * d_in ** 0.5)
    else:
        w = torch.randint(-127, 128, (d_out, d_in), device="cuda", dtype=torch.int8, generator=gen)
        s = spread / (73.3 * d_in ** 0.5)
    return pa.weight(WEIGHT_KINDS[kind], w.cpu().numpy(), s.half().cpu().numpy().view("uint16"))


def _config(case):
    cfg = {k: v for k, v in SHAPES[case["shape"]].items() if k != "dim"}
    return dict(cfg, kv_q8=case["kv_q8"], verify_exact=case["exact"])


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    rand = lambda *shape: torch.randn(*shape, device="cuda", generator=gen)  # noqa: E731
    cfg, L, pos, n = _config(case), case["layers"], case["pos"], case["cols"]
    nh, nkv, hd, dim = cfg["n_heads"], cfg["n_kv_heads"], cfg["head_dim"], SHAPES[case["shape"]]["dim"]
    rows = pos if case["path"] == "session" else pos + n
    pa = _Context(cfg, -(-rows // 4096) * 4096, n_layers=L, max_cols=max(n, BATCH_COLS))
    st = dict(case=case, pa=pa)
    for l in range(L):
        pa.layer_alloc(l)
        _fill(pa, l, pos, gen)
    caches = [t for l in range(L) for t in _cache(pa, l)]
    if case["path"] == "session":
        pa.slot_save(1, pos)                      # the other conversation waits in slot 1
        pa.sync()
        for l in range(L):
            _fill(pa, l, pos, gen)                # and this one runs
        pa.slot_save(0, pos)
        st.update(running=0, outputs=[t[:, :pos] for t in caches])
        pa.sync()
        return st
    norm = lambda m: [_Buf(1 + 0.1 * rand(m)) for _ in range(L)]  # noqa: E731
    st.update(qw=norm(hd), kw=norm(hd))
    new_rows = [t[:, pos:pos + n] for t in caches]
    if case["path"] == "layer":
        st.update(wqkv=[_weight(pa, case["weights"], pa.q_in_dim + 2 * pa.kv_dim, dim, gen) for _ in range(L)],
                  wo=[_weight(pa, case["weights"], dim, pa.q_dim, gen) for _ in range(L)],
                  norm=norm(dim), x0=_Buf(rand(n, dim)), x=_Buf(torch.empty(n, dim, device="cuda")))
        st["outputs"] = [st["x"].tensor] + new_rows
    else:
        # the engine's attention output: f32 behind a token or a draft, f16 behind a prompt chunk
        dtype = torch.float32 if n <= 16 else torch.float16
        st.update(q=[_Buf(rand(n, pa.q_in_dim)) for _ in range(L)], k=[_Buf(rand(n, pa.kv_dim)) for _ in range(L)],
                  v=[_Buf(rand(n, pa.kv_dim)) for _ in range(L)], out=[_Buf(torch.empty(n, pa.q_dim, device="cuda", dtype=dtype)) for _ in range(L)],
                  gate=pa.gate_buffer_ptr() if cfg["gate"] else None, out_dtype=PA_OUT_F32 if n <= 16 else PA_OUT_F16)
        st["outputs"] = [b.tensor for b in st["out"]] + new_rows
    torch.cuda.current_stream().synchronize()
    pa.sync()
    return st


def run(st):
    """One pass: the residual (or the attention outputs) and the cache rows that it wrote."""
    case, pa = st["case"], st["pa"]
    L, pos, n = case["layers"], case["pos"], case["cols"]
    if case["path"] == "session":
        pa.slot_save(st["running"], pos)
        st["running"] ^= 1
        pa.slot_load(st["running"])
    elif case["path"] == "layer":
        x, dim = st["x"], st["x0"].tensor.shape[1]
        pa.copy_d2d(x, st["x0"], n * dim * 4)
        for l in range(L):
            if n == 1:
                pa.attn_layer_decode(l, st["wqkv"][l], st["wo"][l], st["norm"][l], st["qw"][l], st["kw"][l], x, pos)
            else:
                pa.attn_layer_prefill(l, st["wqkv"][l], st["wo"][l], st["norm"][l], st["qw"][l], st["kw"][l], x, dim, pos, n)
    else:
        qd, qi, kvd = pa.q_dim, pa.q_in_dim, pa.kv_dim
        for l in range(L):
            q, k, v, qw, kw, out = st["q"][l], st["k"][l], st["v"][l], st["qw"][l], st["kw"][l], st["out"][l]
            if n == 1:
                pa.attn_decode_step(l, q, k, v, qw, kw, pos, out, st["out_dtype"])
            else:
                pa.glue_kv(l, q, qi, k, kvd, v, kvd, qw, kw, pos, n)
                pa.attn("decode" if n <= 16 else "prefill", l, None, 0, st["gate"], qd, pos, n, out, qd, st["out_dtype"])
    return st["outputs"]


def work(case):
    """Weights, visible cache rows, activations in and results out, each once; products of the projections and of the
    causal attention."""
    s = SHAPES[case["shape"]]
    nh, nkv, hd, dim = s["n_heads"], s["n_kv_heads"], s["head_dim"], s["dim"]
    L, pos, n = case["layers"], case["pos"], case["cols"]
    row = 2 * nkv * (hd + hd // 32 * 4 if case["kv_q8"] else 2 * hd)      # K and V of one position
    if case["path"] == "session":
        return dict(bytes=L * 4 * pos * row, flops=0)                      # one session read and written, and the other
    qd, qi, kvd = nh * hd, nh * hd * (2 if s["gate"] else 1), nkv * hd
    bytes_ = (pos + n) * row
    flops = 4.0 * nh * hd * (n * pos + n * (n + 1) / 2)
    if case["path"] == "layer":
        weights = (qi + 2 * kvd) * dim + dim * qd
        bytes_ += weights * (0.5625 if case["weights"] == "q4_0" else 1.0625)
        flops += 2.0 * n * weights
        return dict(bytes=int(L * bytes_ + 2 * n * dim * 4), flops=L * flops)
    bytes_ += n * (4 * (qi + 2 * kvd) + qd * (4 if n <= 16 else 2))
    return dict(bytes=int(L * bytes_), flops=L * flops)


def tolerance(case):
    """Copies are exact.  Elsewhere four times what the same passes differ by when the sums run in another order (other
    split counts, the other attention kernel, a chunk in two halves): at most 4e-4 of an output's norm, single values by
    6e-3 of it (f16 query, probability and output rounding), and 0.1 to 0.5 % of the int8 cache values of later layers one
    step apart."""
    if case["path"] == "session":
        return "exact"
    return {"rel": 1.6e-3, "max": 2.4e-2, "differ": 1e-2}

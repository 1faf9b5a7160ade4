"""No-GPU checks of which kernel instance a projection takes by its sizes: the library's own rules, asked on a 256-CU part, against
the sizes that the GPU tests run.  A change of a rule that leaves an instance without a tested size fails here."""
import ctypes
from pooled_amd import capi
from pooled_amd.capi import PA_W_Q4_0, PA_W_Q8_0
from test_gpu_proj import GEMM_FEW_SIZES, GEMM_TILE_SIZES, GEMV_RESIDENT_SIZES, GEMV_WIDE_SIZES, HEADS_SIZES

CUS = 256
u32 = ctypes.c_uint32


def _rule(name, *args):
    fn = getattr(capi.load(), name)
    fn.restype = u32
    return fn(*(a if isinstance(a, ctypes._SimpleCData) else u32(a) for a in args))


def _gemv(kind, d_out, d_in, norm):
    """(kind, blocks a lane, norm, rows a wave) past 4096 inputs"""
    return kind, 3 if d_in <= 6144 else 4, norm, _rule("pa_rule_gemv_wide_rows", ctypes.c_int(kind), d_out, d_in, ctypes.c_int(norm), ctypes.c_int(CUS))


def test_gemv_sizes_take_every_number_of_rows():
    forms = [(k, norm) for k in (PA_W_Q4_0, PA_W_Q8_0) for norm in (False, True)]
    got = {_gemv(k, d_out, d_in, norm) for k, norm in forms for d_out, d_in in GEMV_WIDE_SIZES}
    most = {(PA_W_Q4_0, 3, True): 7, (PA_W_Q4_0, 3, False): 7, (PA_W_Q4_0, 4, True): 4, (PA_W_Q4_0, 4, False): 4,
            (PA_W_Q8_0, 3, True): 5, (PA_W_Q8_0, 3, False): 2, (PA_W_Q8_0, 4, True): 2, (PA_W_Q8_0, 4, False): 2}
    assert got == {(k, b, norm, r) for (k, b, norm), m in most.items() for r in range(1, m + 1)}
    # a wave whose last rows are past the end, for every instance of two rows and more but one (three rows are taken at one d_out only)
    ragged = {_gemv(k, d_out, d_in, norm) for k, norm in forms for d_out, d_in in GEMV_WIDE_SIZES if d_out % _gemv(k, d_out, d_in, norm)[3]}
    assert all(b == 3 and r == 3 for _, b, _, r in {g for g in got if g[3] > 1} - ragged)
    # Q8_0: two rows without the norm, and on tall weights
    assert _gemv(PA_W_Q8_0, 14336, 5120, False)[3] == 2 and _gemv(PA_W_Q8_0, 14336, 5120, True)[3] == 2 and _gemv(PA_W_Q8_0, 7168, 5120, True)[3] == 4


def test_gemv_resident_sizes_take_every_form():
    def form(kind, d_out, d_in, norm):
        v = _rule("pa_rule_gemv_resident", ctypes.c_int(kind), d_out, d_in, ctypes.c_int(norm), ctypes.c_int(CUS))
        return (kind, 3 if d_in <= 6144 else 4, norm, v >> 16, v & 0xffff) if v else None
    forms = [(k, norm) for k in (PA_W_Q4_0, PA_W_Q8_0) for norm in (0, 1)]
    sizes = GEMV_RESIDENT_SIZES + GEMV_WIDE_SIZES
    tested = {form(k, d_out, d_in, norm) for k, norm in forms for d_out, d_in in sizes}
    reached = {form(k, d_out, d_in, norm) for k, norm in forms for d_out in range(1, 20000, 7) for d_in in (4128, 5152, 8192)}
    assert {f[3:] for f in reached - {None}} == {(1, r) for r in range(1, 9)} | {(2, r) for r in range(5, 9)}
    assert reached <= tested
    # the line without the norm: not at four rows a wave, nor at six to eight of one workgroup a CU
    assert [form(PA_W_Q4_0, d_out, 6144, 0) for d_out in (4096, 5121, 8192)] == [None] * 3 and form(PA_W_Q8_0, 3072, 6144, 0) is None
    assert form(PA_W_Q4_0, 5120, 6144, 0)[3:] == (1, 5) and form(PA_W_Q4_0, 14336, 5120, 1)[3:] == (2, 7)
    # ... nor at five for a handful of rows past 4096
    assert [form(k, d_out, 6144, 0) for k in (PA_W_Q4_0, PA_W_Q8_0) for d_out in (4097, 4112)] == [None] * 4 and form(PA_W_Q4_0, 4113, 4128, 0)[3:] == (1, 5)
    # Q4_0 rows of at most 5120 inputs: six to eight rows a wave not with the norm, two workgroups a CU of five not without
    assert [form(PA_W_Q4_0, 7168, d_in, 1) for d_in in (4128, 5120)] == [None] * 2 and form(PA_W_Q4_0, 7168, 5152, 1)[3:] == (1, 7) and form(PA_W_Q8_0, 7168, 4128, 1)[3:] == (1, 7)
    assert form(PA_W_Q4_0, 9000, 5088, 0) is None and form(PA_W_Q4_0, 9000, 5120, 0)[3:] == (2, 5) and form(PA_W_Q4_0, 9000, 4128, 1)[3:] == (2, 5)


def test_gemv_sizes_take_every_instance():
    """Every kernel instance that some size reaches (kind, blocks a lane, norm, rows a wave, requested at once), ragged last rows among them where it has more than one."""
    def instance(kind, d_out, d_in, norm):
        v = _rule("pa_rule_gemv_resident", ctypes.c_int(kind), d_out, d_in, ctypes.c_int(norm), ctypes.c_int(CUS)) & 0xffff
        rows = v or _gemv(kind, d_out, d_in, norm)[3]
        once = not v and _rule("pa_rule_gemv_at_once", ctypes.c_int(kind), d_out, d_in, ctypes.c_int(norm), rows, ctypes.c_int(CUS))
        return kind, 3 if d_in <= 6144 else 4, norm, rows, bool(once)
    forms = [(k, norm) for k in (PA_W_Q4_0, PA_W_Q8_0) for norm in (0, 1)]
    tested = {instance(k, d_out, d_in, norm) for k, norm in forms for d_out, d_in in GEMV_RESIDENT_SIZES + GEMV_WIDE_SIZES}
    reached = {instance(k, d_out, d_in, norm) for k, norm in forms for d_out in range(1, 36000, 7) for d_in in (4128, 5120, 5152, 6144, 6176, 8192)}
    assert reached <= tested, reached - tested
    assert {i[1:] for i in reached if i[4]} == {(3, 0, 4, True), (3, 0, 5, True), (4, 0, 4, True)}


def _few(kind, d_out, d_in, n):
    """(kind, row groups, column blocks, blocks of a chunk, d_in in whole chunks) of the few-column kernel, (kind, blocks a lane) of the
    dot-product one; None past their range"""
    if n > 32 or (n > 16 and kind != PA_W_Q4_0 and d_in > 4096):
        return None
    if _rule("pa_rule_gemm_few_dot", ctypes.c_int(kind), d_out, d_in, n, ctypes.c_int(CUS)):
        return kind, 2 if d_in <= 4096 else 4
    ch = 8 if d_in <= 4096 else 16
    rg = _rule("pa_rule_gemm_few_groups", ctypes.c_int(kind), d_out, d_in, n, ctypes.c_int(CUS))
    return kind, rg, 1 if n <= 16 else 2, ch, d_in % (32 * ch) == 0


def test_few_column_sizes_take_every_instance():
    kinds = (PA_W_Q4_0, PA_W_Q8_0)
    tested = {_few(k, *size) for k in kinds for size in GEMM_FEW_SIZES}
    reached = {_few(k, d_out, d_in, n) for k in kinds for d_out in (16, 4096, 4097, 5000, 8176, 8177, 9216, 20000) for d_in in range(32, 8193, 32)
               for n in (1, 2, 4, 8, 9, 16, 17, 32)}
    assert len(reached) > 40 and reached <= tested | {None}
    # the dot-product kernel takes up to four columns over rows of more than 2048 inputs, two of them past 2048 rows
    dot = {(k, d_out, d_in, n) for k in kinds for d_out in (16, 1000, 2048, 2049, 5120, 9216, 20000) for d_in in range(32, 8193, 32) for n in (1, 2, 3, 4, 5)
           if len(_few(k, d_out, d_in, n)) == 2}
    assert {n for _, _, _, n in dot} == {1, 2, 3, 4} and all(d_in > 2048 and (n <= 2 or d_out <= 2048) for _, d_out, d_in, n in dot)
    assert all((PA_W_Q8_0, 5120, 6144, n) in dot for n in (1, 2)) and not any((PA_W_Q4_0, 20000, 5120, n) in dot for n in (1, 2))


def _tile(d_out, d_in, n, x_stride=None):
    t = _rule("pa_rule_gemm_wide_tile", d_out, d_in, n, x_stride or d_in + 8, ctypes.c_int(CUS))
    return t >> 16, t & 0xffff


def test_tile_sizes_take_every_tile():
    assert [_tile(*size) for size in GEMM_TILE_SIZES] == [(128, 128), (128, 160), (128, 192), (128, 256), (128, 320), (128, 384), (128, 448),
                                                          (256, 256), (64, 128), (128, 256)]
    every = {_tile(d_out, d_in, n) for d_out in range(33, 16000, 331) for d_in in (128, 2048, 5120, 8192) for n in (17, 100, 400, 512, 900, 1544, 2500, 4096)}
    small = {(64, 64), (64, 32)}
    assert every <= {_tile(*size) for size in GEMM_TILE_SIZES} | small
    # both forms of the 64-column kernel, as the docstrings of the other GEMM tests have them
    assert [_tile(600, 128, 11000), _tile(2048, 4096, 600), _tile(130, 8192, 513)] == [(64, 64), (64, 64), (64, 32)]
    assert [_tile(9216 - 40, 2048, 4096 - 3), _tile(2048, 4096, 4000), _tile(4090, 256, 4096)] == [(128, 384), (128, 256), (256, 256)]
    assert [_tile(9216, 2048, 300), _tile(4096, 2048, 512)] == [(128, 128), (64, 128)]
    assert {_tile(2048, 4096, 129), _tile(130, 8192, 40), _tile(100, 384, 65), _tile(64, 128, 33), _tile(130, 8192, 17)} == {(64, 32)}
    # rows further apart than the larger tiles' 32-bit offsets reach
    assert _tile(9216, 2048, 4096, 1 << 22) == (128, 384) and _tile(9216, 2048, 4096, (1 << 22) + 8) == (64, 64)


def test_pre_step_sizes_take_every_tile():
    def tile(heads, dim, n):
        nH, nKV, hd, gate = heads
        v = _rule("pa_rule_gemm_heads", nH * hd * (2 if gate else 1) + 2 * nKV * hd, dim, n, nH, hd, ctypes.c_int(gate), ctypes.c_int(CUS))
        return v >> 28, v >> 16 & 0xfff, v & 0xffff
    assert [tile(*size[:3]) for size in HEADS_SIZES] == [size[3] for size in HEADS_SIZES]
    models = [((16, 8, 128, False), 2048), ((16, 2, 256, True), 2048), ((24, 4, 256, True), 5120)]
    every = {tile(heads, dim, n) for heads, d in models for dim in (d, 256, 1024, 8192) for n in range(33, 4097, 13)}
    assert every <= {size[3] for size in HEADS_SIZES} | {(0, 0, 0)}
    assert [tile(*models[0], 512), tile(*models[1], 4096), tile(*models[2], 777)] == [(4, 64, 128), (1, 320, 256), (1, 224, 256)]
    # 24 / 4-head shape: apart where the estimates tell nothing (up to 256 columns); past them 96 columns a tile only where that is a block of columns more
    assert {tile(*models[2], n) for n in range(200, 257)} == {(0, 0, 0)} and {tile(*models[2], n) for n in range(257, 289)} == {(1, 128, 256)}
    assert {tile(*models[2], n) for n in range(289, 385)} == {(1, 96, 256)}
    # a few columns, and sizes whose sums are split as no tile of whole heads splits them: apart
    assert [tile(*models[0], 100), tile(*models[1], 100), tile(*models[1], 256)] == [(0, 0, 0)] * 3

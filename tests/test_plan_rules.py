"""No-GPU checks of which kernel serves an attention call: the library's own plan rules, asked on a 256-CU part."""
import ctypes
import pytest
from pooled_amd import capi
from helpers import attn_rule, BLOCK, LOOP, MFMA, ONE_WG, SHAPES, SINGLE_ROUND


@pytest.mark.parametrize("kv_q8", [False, True])
@pytest.mark.parametrize("head_dim,most", [(256, 32), (128, 64)])
def test_one_column_never_goes_to_the_kernel_without_an_own_row(head_dim, most, kv_q8):
    """One column of any group size over any context, with and without a splits override: its own row is a partial of its own (slots = splits + 1), which the
    kernel of verify blocks does not make."""
    for n_kv in (1, 2, 8):
        for group in sorted({1, 8, 16, 17, 24, most // 2 + 1, most}):
            cfg = dict(n_heads=group * n_kv, n_kv_heads=n_kv, head_dim=head_dim, n_rot=64, rope_theta=1e6, eps=1e-6, kv_q8=kv_q8)
            for base in (0, 1, 127, 128, 129, 255, 256, 257, 1000, 2048, 4100, 8192, 10001, 16400, 20000, 32768, 65536, 120000):
                for splits in (0, 1, 2, 7, 64):
                    for kind in ("decode", "prefill"):
                        kernel, pl = attn_rule(cfg, kind, base, 1, splits)
                        assert kernel >= 0 and pl["slots"] == pl["n_splits"] + 1 and kernel != BLOCK, (cfg, base, splits, kind, pl)


@pytest.mark.parametrize("kv_q8", [False, True])
@pytest.mark.parametrize("n_heads,n_kv,head_dim", [(16, 2, 256), (24, 4, 256), (16, 8, 128), (64, 2, 256), (64, 1, 128), (8, 8, 128)])
def test_a_chunk_under_capture_has_a_plan_without_scratch(n_heads, n_kv, head_dim, kv_q8):
    """Prefill calls captured in a context that holds no scratch, from one column to thousands, with the tile override and a splits override too: none is left with a plan
    that would allocate.  (Always the matrix-core kernel over int8 rows needs its widened cache.)"""
    cfg = dict(n_heads=n_heads, n_kv_heads=n_kv, head_dim=head_dim, n_rot=64, rope_theta=1e6, eps=1e-6, kv_q8=kv_q8)
    for n in (1, 2, 4, 9, 16, 33, 40, 64, 100, 144, 300, 777, 2048):
        for base in (0, 20, 88, 200, 300, 900, 2000, 5000, 30000):
            for splits in (0, 3):
                for tile in (0, 1, 2):
                    kernel, pl = attn_rule(cfg, "cold", base, n, splits, tile)
                    if tile == 1 and kv_q8 and n * n_heads // n_kv > (32 if head_dim == 256 else 64):
                        continue
                    assert kernel >= 0 and pl["n_splits"] == 1, (cfg, base, n, splits, tile, kernel, pl)
                    rows = pl["split_len"]
                    assert kernel == ONE_WG or (rows >= base + n and kernel in (MFMA, LOOP))


@pytest.mark.parametrize("n_heads,n_kv,head_dim", [(16, 2, 256), (24, 4, 256), (16, 8, 128)])
def test_a_gather_over_a_short_list_keeps_splits_of_one_tile_a_wave(n_heads, n_kv, head_dim):
    """Gather calls always have partials and a merge: lists of up to 256 rows are splits of 128, one tile a wave, on the single-round kernel, as longer ones are
    (not the one split that a block of columns over as many rows takes to write its output itself)."""
    cfg = dict(n_heads=n_heads, n_kv_heads=n_kv, head_dim=head_dim, n_rot=64, rope_theta=1e6, eps=1e-6)
    for rows in (1, 31, 32, 33, 127, 128, 129, 200, 255, 256, 257, 400, 2051):
        kernel, pl = attn_rule(cfg, "gather", rows, 1)
        assert (kernel, pl["split_len"], pl["n_splits"], pl["slots"]) == (SINGLE_ROUND, 128, -(-rows // 128), -(-rows // 128)), (rows, pl)


@pytest.mark.parametrize("n_heads,n_kv,head_dim", [(16, 2, 256), (24, 4, 256), (16, 8, 128), (32, 4, 128)])
def test_a_few_columns_over_a_short_context_keep_a_tile_a_wave(n_heads, n_kv, head_dim):
    """Up to 256 rows no wave of a block of columns takes two tiles: one launch of four or eight waves, or, one row block at head_dim 256 past 128 rows, two splits."""
    cfg = dict(n_heads=n_heads, n_kv_heads=n_kv, head_dim=head_dim, n_rot=64, rope_theta=1e6, eps=1e-6)
    group = n_heads // n_kv
    for rows in (3, 32, 33, 127, 128, 129, 130, 200, 255, 256, 257):
        for kind, n in [("decode", 2), ("decode", 16 // group), ("prefill", 2), ("prefill", 16 // group), ("prefill", 32 // group)]:
            if n > rows or n < 2:
                continue
            kernel, pl = attn_rule(cfg, kind, rows - n, n)
            assert pl["row_blocks"] <= 2 and pl["waves"] * pl["n_splits"] * 32 >= rows, (kind, n, rows, pl)
            one = rows <= (128 if head_dim == 256 and n * group <= 16 else 256)
            assert (pl["n_splits"] == 1) == one and (kernel == LOOP) == one, (kind, n, rows, kernel, pl)
            assert not one or pl["waves"] == (8 if rows > 128 else 4)


@pytest.mark.parametrize("shape,n,base,splits,kernel", [
    # one column group: from two tiles a wave on (three row blocks and more: also where few workgroups are made), not with one at head_dim 256, nor on less than half the chip
    ("qwen36_moe", 4, 16377, 0, SINGLE_ROUND), ("qwen36_moe", 4, 16385, 0, BLOCK), ("qwen36_moe", 4, 60000, 0, BLOCK), ("qwen38_27b", 5, 8180, 0, SINGLE_ROUND), ("qwen38_27b", 5, 8190, 0, BLOCK),
    ("qwen3_1p7b", 12, 2030, 0, SINGLE_ROUND), ("qwen3_1p7b", 12, 2040, 0, BLOCK), ("qwen3_1p7b", 12, 4080, 0, BLOCK), ("qwen3_1p7b", 12, 4090, 0, SINGLE_ROUND), ("qwen3_1p7b", 12, 8170, 0, SINGLE_ROUND),
    ("qwen3_1p7b", 12, 8190, 0, BLOCK), ("qwen3_1p7b", 24, 200, 0, LOOP), ("qwen3_1p7b", 24, 250, 0, BLOCK),
    # several: two tiles a wave, or one on more than half the chip and not twice
    ("qwen36_moe", 8, 4080, 0, SINGLE_ROUND), ("qwen36_moe", 8, 4090, 0, BLOCK), ("qwen36_moe", 8, 8180, 0, BLOCK), ("qwen36_moe", 8, 8190, 0, BLOCK), ("qwen36_moe", 8, 16370, 0, BLOCK),
    ("qwen36_moe", 8, 16380, 0, LOOP), ("qwen36_moe", 8, 60000, 0, LOOP), ("qwen38_27b", 10, 8170, 0, BLOCK), ("qwen38_27b", 10, 8190, 0, LOOP),
    # one split, one row block, and overrides by the same lines
    ("qwen36_moe", 4, 100, 0, LOOP), ("qwen36_moe", 2, 40000, 0, LOOP), ("qwen36_moe", 4, 8000, 10, BLOCK), ("qwen36_moe", 8, 8000, 10, LOOP), ("qwen36_moe", 8, 8000, 32, BLOCK), ("qwen36_moe", 4, 8000, 1, LOOP)])
def test_which_kernel_serves_a_verify_block(shape, n, base, splits, kernel):
    """Both sides of each line between the single-round kernel, the tile loop and the kernel whose waves share one softmax."""
    got, pl = attn_rule(SHAPES[shape], "decode", base, n, splits)
    assert got == kernel, (got, pl)


@pytest.mark.parametrize("shape,q8,n,base,kernel", [
    ("qwen36_moe", False, 854, 10, LOOP), ("qwen36_moe", False, 807, 44, LOOP), ("qwen3_1p7b", False, 655, 1093, LOOP), ("qwen3_1p7b", False, 1463, 86, LOOP), ("qwen38_27b", False, 606, 275, LOOP),
    ("qwen38_27b", False, 660, 0, MFMA), ("qwen36_moe", False, 1024, 0, MFMA), ("qwen3_1p7b", False, 2048, 0, MFMA), ("qwen36_moe", True, 585, 844, MFMA), ("qwen36_moe", True, 446, 1265, MFMA)])
def test_a_chunk_runs_in_one_launch_where_it_is_close(shape, q8, n, base, kernel):
    """One launch is taken within 3 % of the matrix-core kernel's estimate on f16 rows, not on int8 rows, whose plans stay what they were that close."""
    got, pl = attn_rule(dict(SHAPES[shape], kv_q8=q8), "prefill", base, n)
    assert got == kernel and (kernel == MFMA or pl["n_splits"] == 1), (got, pl)


@pytest.mark.parametrize("shape,n,base,kernel", [
    ("qwen38_27b", 5, 9000, BLOCK), ("qwen38_27b", 5, 24560, BLOCK), ("qwen38_27b", 5, 24580, LOOP), ("qwen38_27b", 5, 60000, LOOP), ("qwen38_27b", 8, 65000, LOOP), ("qwen36_moe", 3, 49140, BLOCK),
    ("qwen36_moe", 3, 49160, LOOP), ("qwen36_moe", 16, 8000, BLOCK), ("qwen3_1p7b", 16, 30000, BLOCK), ("qwen3_1p7b", 32, 30000, BLOCK)])
def test_which_kernel_serves_a_verify_block_over_int8_rows(shape, n, base, kernel):
    """Int8 rows at head_dim 256 leave the kernel with one softmax a workgroup past three tiles a wave; at head_dim 128 they do not."""
    got, pl = attn_rule(dict(SHAPES[shape], kv_q8=True), "decode", base, n)
    assert got == kernel, (got, pl)


@pytest.mark.parametrize("n_cols,n_heads,head_dim,n_splits,wide", [(15, 16, 256, 4, 0), (16, 16, 256, 4, 1), (16, 24, 256, 7, 1), (16, 24, 256, 8, 1), (16, 24, 256, 9, 0), (16, 16, 256, 32, 0),
                                                                   (25, 16, 256, 9, 0), (26, 16, 256, 9, 1), (51, 16, 128, 9, 0), (52, 16, 128, 9, 1), (64, 16, 256, 32, 1), (64, 16, 256, 33, 0)])
def test_which_kernel_merges_the_splits(n_cols, n_heads, head_dim, n_splits, wide):
    """From 16 columns on one thread a (column, head, 4 dims) merges up to 32 splits, but past the eight of one round trip only with more than two fifths of the CUs' worth of workgroups."""
    assert capi.load().pa_rule_merge_wide(*(ctypes.c_uint32(v) for v in (n_cols, n_heads, head_dim, n_splits)), ctypes.c_int(256)) == wide

"""The rules that plan a prefill launch (keys split between waves on the 16-bit
matrix cores; fp32 matrix cores or one wave per row elsewhere): the lines they
draw, that they go by the ranges of the requests and not by how wide a table
the caller keeps, and what they answer and refuse. Runs on the CPU."""

import ctypes

import pytest

from inferkernellab_amd import _lib


def _args(batch, heads, kv, dim, width, table_blocks, dtype=_lib.IKL_BF16, cache=0, **kw):
    a = _lib.PagedPrefillArgs()
    a.batch, a.query_width, a.num_heads, a.num_kv_heads = batch, width, heads, kv
    a.head_dim, a.block_size, a.dtype, a.cache_dtype, a.path = dim, 16, dtype, cache, -1
    a.table_width, a.num_blocks = table_blocks, 1 << 20
    for name, value in kw.items():
        setattr(a, name, value)
    return a


def _plan(a, longest, start):
    return _lib.load().ikl_paged_prefill_plan(ctypes.byref(a), longest, start)


@pytest.mark.parametrize("batch,heads,kv,dim,width", [(8, 32, 8, 128, 512), (4, 32, 8, 128, 1024), (6, 32, 8, 128, 512),
                                                      (8, 32, 8, 64, 512), (4, 32, 8, 96, 1024)])
def test_a_wide_table_changes_no_plan(batch, heads, kv, dim, width):
    tight, wide = (_args(batch, heads, kv, dim, width, n) for n in (width // 16, 8192 // 16))
    lib = _lib.load()
    assert lib.ikl_paged_prefill_key_groups(ctypes.byref(wide)) == lib.ikl_paged_prefill_key_groups(ctypes.byref(tight))
    assert _plan(wide, width, 0) == _plan(tight, width, 0) == 0


FP8 = _lib.IKL_FP8_E4M3
# (batch, heads, kv heads, dim, cache, start, tokens, plan): the short side of
# each line, where splitting was measured slower, and the long side
LINES = [
    (4, 32, 8, 128, 0, 0, 64, 0), (2, 32, 8, 128, 0, 120, 8, 0), (1, 32, 32, 128, 0, 0, 96, 0),
    (8, 32, 8, 64, 0, 0, 64, 0), (2, 32, 8, 64, 0, 120, 8, 4), (8, 32, 8, 128, 0, 480, 32, 4),
    (1, 8, 2, 128, 0, 0, 256, 4), (1, 32, 32, 128, 0, 0, 192, 2),
    (8, 32, 8, 128, 0, 0, 128, 0), (8, 32, 8, 128, FP8, 0, 128, 0), (32, 32, 8, 128, 0, 480, 32, 0),
    (16, 32, 8, 64, 0, 0, 64, 0), (8, 8, 2, 128, 0, 0, 256, 2), (1, 32, 8, 128, 0, 0, 1024, 2),
    (8, 32, 32, 128, 0, 0, 256, 0), (64, 32, 8, 128, 0, 480, 32, 0), (16, 32, 32, 64, 0, 0, 128, 0),
    (32, 32, 8, 128, 0, 1984, 64, 0), (32, 32, 8, 96, 0, 1984, 64, 1), (2, 32, 8, 128, 0, 2048, 1024, 1),
    (2, 32, 8, 128, 0, 0, 1024, 1), (8, 16, 4, 128, 0, 0, 512, 1),
    (25, 32, 8, 128, 0, 128, 128, 0), (4, 32, 8, 128, 0, 2048, 1024, 0), (3, 32, 8, 64, 0, 1024, 1024, 0),
    (3, 32, 8, 128, 0, 2048, 1024, 1), (4, 32, 8, 128, FP8, 2048, 1024, 1), (4, 32, 8, 64, 0, 2048, 1024, 1),
    (4, 32, 8, 96, 0, 2048, 1024, 1), (62, 32, 1, 128, 0, 64, 64, 0),
    (16, 32, 32, 96, FP8, 0, 128, 0), (64, 32, 32, 32, FP8, 0, 64, 0), (4, 32, 8, 32, 0, 0, 2048, 1),
    (8, 32, 8, 96, FP8, 0, 4096, 1), (8, 32, 8, 96, 0, 0, 4096, 0), (8, 32, 8, 128, 0, 0, 4096, 0),
]


@pytest.mark.parametrize("batch,heads,kv,dim,cache,start,tokens,plan", LINES)
def test_lines_of_the_rule(batch, heads, kv, dim, cache, start, tokens, plan):
    a = _args(batch, heads, kv, dim, tokens, 4096, cache=cache)
    assert _plan(a, start + tokens, start) == plan


def test_unknown_ranges_count_as_the_query_width_from_position_0():
    for width in (8, 64, 300, 512, 2048):
        a = _args(2, 32, 8, 128, width, 512)
        assert _plan(a, 0, 0) == _plan(a, width, 0) == _lib.load().ikl_paged_prefill_key_groups(ctypes.byref(a))


ROWS = _lib.IKL_PREFILL_ROWS
# (batch, heads, kv heads, dim, dtype, start, tokens, plan), off the 16-bit
# matrix cores: one wave per row where it was measured the faster
OTHER_LINES = [
    (64, 32, 32, 64, _lib.IKL_F32, 0, 1, ROWS), (4, 32, 8, 64, _lib.IKL_F32, 0, 5, ROWS),
    (1, 32, 8, 256, _lib.IKL_F32, 0, 12, ROWS), (64, 32, 32, 256, _lib.IKL_F32, 2047, 1, ROWS),
    (64, 32, 32, 256, _lib.IKL_BF16, 255, 1, ROWS), (64, 8, 1, 80, _lib.IKL_BF16, 0, 5, ROWS),
    (1, 8, 2, 512, _lib.IKL_BF16, 0, 4096, ROWS),  # no wider kernel
    (4, 32, 8, 64, _lib.IKL_F32, 255, 1, 0), (16, 32, 32, 256, _lib.IKL_F32, 2047, 1, 0),
    (64, 32, 32, 128, _lib.IKL_F32, 255, 1, 0), (4, 32, 8, 64, _lib.IKL_F32, 0, 64, 0),
    (4, 32, 8, 64, _lib.IKL_F32, 0, 512, 0), (1, 8, 1, 80, _lib.IKL_BF16, 0, 33, 0),
    (64, 32, 8, 32, _lib.IKL_F32, 0, 17, 0),
]


@pytest.mark.parametrize("batch,heads,kv,dim,dtype,start,tokens,plan", OTHER_LINES)
def test_lines_between_the_fp32_matrix_cores_and_one_wave_per_row(batch, heads, kv, dim, dtype, start, tokens, plan):
    a = _args(batch, heads, kv, dim, tokens, 4096, dtype=dtype, path=_lib.IKL_PATH_SCALAR_GROUPED)
    assert _plan(a, start + tokens, start) == plan
    assert _lib.load().ikl_paged_prefill_key_groups(ctypes.byref(a)) == 0


def test_a_plan_of_the_other_path_is_refused():
    lib = _lib.load()
    ptr = ctypes.addressof(ctypes.create_string_buffer(64)) & ~15
    a = _args(4, 32, 8, 64, 1024, 64, dtype=_lib.IKL_F32)
    for name in ("query", "k_cache", "v_cache", "block_tables", "query_starts", "context_lens", "out"):
        setattr(a, name, ptr)
    for plan in (1, 2, 4):
        assert lib.ikl_paged_prefill_attention_planned(ctypes.byref(a), plan, None) == _lib.IKL_EINVAL
    a.dtype = _lib.IKL_BF16
    for plan in (-2, 3, 5, ROWS):
        assert lib.ikl_paged_prefill_attention_planned(ctypes.byref(a), plan, None) == _lib.IKL_EINVAL
    assert b"plan" in lib.ikl_last_error()


def test_invalid_ranges_are_refused():
    a = _args(1, 8, 2, 64, 16, 8)
    assert _plan(a, -1, 0) == _lib.IKL_EINVAL and _plan(a, 16, -1) == _lib.IKL_EINVAL
    assert _lib.load().ikl_paged_prefill_plan(None, 0, 0) == _lib.IKL_EINVAL


@pytest.mark.parametrize("name", ["batch", "query_width", "num_heads", "num_kv_heads", "head_dim", "block_size",
                                  "table_width"])
@pytest.mark.parametrize("value", [0, -16])
def test_invalid_sizes_are_refused(name, value):
    a = _args(1, 8, 2, 64, 16, 8)
    setattr(a, name, value)
    lib = _lib.load()
    assert _plan(a, 16, 0) == _lib.IKL_EINVAL
    assert lib.ikl_paged_prefill_key_groups(ctypes.byref(a)) == _lib.IKL_EINVAL

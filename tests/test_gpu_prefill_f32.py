"""Paged prefill on the fp32 matrix cores against the oracle, at the edges of
its tiles: 32-key tiles (chunks and prefixes ending on, before and after a
tile), 64-row workgroups (a group of 1, 3 and 8 heads per KV head), head dims
at and between the compiled widths, rows that are not aligned to four
elements, block sizes that do not divide a tile, 16-bit rows, and V values
that are not finite past a row's causal limit."""

import numpy as np
import pytest
import torch

from tests.helpers import ATOL, make_prefill_case, max_abs_err

pytestmark = pytest.mark.gpu


def _prepare(case, query, plan=0):
    from inferkernellab_amd import PreparedPagedPrefill

    prep = PreparedPagedPrefill(case.base.device_cache(), case.base.device_tables(), case.starts, case.ends,
                                num_heads=query.shape[1], query_width=query.shape[2], path="scalar_grouped")
    prep.plan = plan  # whichever the rule takes for these sizes
    assert prep.kernel_name() == ("paged_prefill_scalar_kernel" if plan else "paged_prefill_f32_kernel")
    return prep


EDGES = [
    (4, 4, 8, 4, "float32", [0, 0, 0], [31, 32, 33]),
    (6, 2, 20, 5, "float32", [0, 64], [65, 97]),
    (6, 2, 33, 16, "float32", [7, 31], [40, 33]),  # odd rows: never aligned to four
    (8, 1, 64, 16, "float32", [0, 1], [8, 2]),
    (8, 2, 64, 24, "float32", [0, 100], [257, 129]),
    (3, 1, 96, 16, "float32", [32], [96]),
    (4, 2, 100, 8, "float32", [0], [70]),
    (2, 2, 128, 16, "float32", [0, 63], [64, 65]),
    (4, 2, 192, 48, "float32", [5], [75]),
    (2, 1, 256, 16, "float32", [0], [66]),
    (8, 2, 80, 16, "bfloat16", [0, 40], [90, 75]),
    (4, 2, 34, 16, "float16", [0], [50]),  # 4-byte rows
    (4, 1, 128, 8, "float16", [16, 0], [81, 64]),
]


@pytest.mark.parametrize("plan", [0, 8])  # fp32 matrix cores, one wave per row
@pytest.mark.parametrize("heads,kv,dim,bs,dtype,starts,ends", EDGES)
def test_tile_edges(heads, kv, dim, bs, dtype, starts, ends, plan):
    case = make_prefill_case(starts=starts, ends=ends, num_heads=heads, num_kv_heads=kv, head_dim=dim, block_size=bs,
                             dtype=dtype, seed=heads + dim + bs, table_slack=1)
    q = case.device_query()
    got = _prepare(case, q, plan)(q)
    # fp32: a few ulp per product over <= 257 keys; 16-bit: the output's rounding
    assert max_abs_err(got, case.expected()) <= (1e-5 if dtype == "float32" else ATOL[dtype])


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_rows_off_the_quad_alignment(dtype):
    """Query and output rows that start 4 bytes off a quad."""
    case = make_prefill_case(starts=[0, 20], ends=[45, 60], num_heads=4, num_kv_heads=2, head_dim=64, block_size=8,
                             dtype=dtype, seed=3)
    q = case.device_query()
    off = 4 // q.element_size()
    wide = torch.zeros(*q.shape[:3], 64 + 2 * off, dtype=q.dtype, device="cuda")
    view = wide[..., off:off + 64]
    view.copy_(q)
    out = torch.full_like(wide, float("nan"))[..., off:off + 64]
    _prepare(case, q)(view, out=out)
    assert max_abs_err(out, case.expected()) <= (1e-5 if dtype == "float32" else ATOL[dtype])


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_values_past_the_causal_limit_do_not_reach_a_row(value):
    """One V element that is not finite: the rows at and past its position
    take it, the rows before it stay as they are without it."""
    pos, dim = 41, 64
    case = make_prefill_case(starts=[0], ends=[70], num_heads=4, num_kv_heads=2, head_dim=dim, block_size=16,
                             dtype="float32", seed=9)
    q = case.device_query()
    expected = case.expected()
    prep = _prepare(case, q)
    slot = case.base.oracle_cache.slot_mapping(case.base.tables[0], pos, 1)[0]
    prep.cache.v[0, slot // 16, slot % 16, 1, 5] = value
    got = prep(q).cpu().numpy()
    touched = np.zeros(expected.shape, bool)
    touched[0, 2:, pos:, 5] = True  # heads 2, 3 share KV head 1
    assert np.abs(got[~touched] - expected[~touched]).max() <= 1e-5
    assert not np.isfinite(got[touched]).any()

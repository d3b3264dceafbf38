"""The matrix-core prefill kernels at the edges of their plans, against the
oracle: one, two and four waves per row (launches of up to 64, 256 and 512
128-row workgroups with long contexts, and two rounds behind long prefixes)
and the kernel of launches past that or with short ones, and every plan on
every shape. Key counts end on, before and after a 32-key tile and a
group's last step, tables cross the kernels' 64-half windows, some entries
lie outside the cache, rows end inside a 32-row group, one request has a
single key and one pads most of its rows."""

import numpy as np
import pytest
import torch

from oracle import paged_oracle as po
from tests.helpers import ATOL, make_prefill_case, max_abs_err, randn_storage, storage_to_torch
from tests.test_gpu_fp8 import _device_fp8_cache, _fp8_case
from tests.test_gpu_prefill import _expected_dropping_blocks

pytestmark = pytest.mark.gpu


# (expected groups, heads, kv heads, head dim, block size, starts, ends)
PLANS = [
    (0, 8, 2, 128, 16, [0, 0, 31, 95], [1, 33, 64, 129]),
    (4, 8, 2, 128, 16, [0, 0, 31, 255], [1, 33, 64, 289]),
    (4, 4, 1, 64, 32, [1500, 0], [1511, 97]),
    (4, 6, 2, 96, 48, [130, 40], [161, 60]),
    (4, 8, 8, 32, 16, [0, 160], [70, 193]),
    (2, 32, 8, 128, 16, [0, 0, 64, 1100, 31], [65, 1, 96, 1165, 95]),
    (2, 16, 8, 64, 16, [0, 0, 0, 900, 0, 5, 0, 64, 0, 0], [80, 64, 33, 930, 31, 36, 1, 65, 2, 80]),
    (2, 24, 8, 96, 16, [0, 32, 64, 96, 128], [50, 64, 65, 97, 160]),
    (1, 32, 8, 128, 16, [0, 0, 31, 64, 1050], [225, 1, 64, 289, 1100]),
    (1, 32, 8, 64, 16, [0, 0, 31, 64, 0], [225, 1, 64, 289, 33]),
    (0, 32, 8, 32, 32, [0] * 9, [250, 249, 33, 32, 31, 1, 250, 64, 65]),
    (1, 32, 8, 32, 32, [1000] + [0] * 8, [1250, 249, 33, 32, 31, 1, 250, 64, 65]),
    (1, 32, 4, 128, 16, [1200] * 17, [1325] + [1201 + 7 * i for i in range(16)]),  # two rounds, long prefixes
    (0, 32, 4, 128, 16, [0, 17] * 9, [128, 100, 1, 33, 32, 31, 127, 97, 96, 95, 65, 64, 63, 20, 50, 77, 128, 120]),
    (0, 32, 4, 64, 32, [0] * 18, [128, 100, 1, 33, 32, 31, 127, 97, 96, 95, 65, 64, 63, 20, 50, 77, 128, 120]),
    (1, 32, 4, 96, 16, [1200] * 18, [1328] + [1201 + 7 * i for i in range(17)]),
    (0, 32, 4, 96, 16, [0] * 18, [128, 100, 1, 33, 32, 31, 127, 97, 96, 95, 65, 64, 63, 20, 50, 77, 128, 120]),
    (0, 32, 8, 64, 16, [400, 0, 500], [1100, 33, 601]),  # windows move
]


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("groups,heads,kv,dim,bs,starts,ends", PLANS)
def test_plan_edges(groups, heads, kv, dim, bs, starts, ends, dtype):
    from inferkernellab_amd import PreparedPagedPrefill

    case = make_prefill_case(starts=starts, ends=ends, num_heads=heads, num_kv_heads=kv, head_dim=dim, block_size=bs,
                             dtype=dtype, seed=heads + dim + len(ends))
    q = case.device_query()
    prep = PreparedPagedPrefill(case.base.device_cache(), case.base.device_tables(), starts, ends, num_heads=heads,
                                query_width=q.shape[2])
    assert prep.key_groups == groups
    out = torch.full_like(q, float("nan"))
    got = prep(q, out=out).float().cpu().numpy()
    assert not np.isnan(got).any()
    assert max_abs_err(got, case.expected(), dtype) < ATOL[dtype]


@pytest.mark.parametrize("groups,heads,kv,dim,bs,starts,ends", [p for p in PLANS if p[3] != 32])
def test_plan_edges_over_the_fp8_cache(groups, heads, kv, dim, bs, starts, ends):
    from inferkernellab_amd import PreparedPagedPrefill

    act = "bfloat16"
    base, packed = _fp8_case(batch=len(ends), heads=heads, kv=kv, dim=dim, bs=bs, lengths=ends, act=act,
                             seed=dim + bs)
    width = max(e - s for s, e in zip(starts, ends))
    q = randn_storage(torch.Generator().manual_seed(dim), (len(ends), heads, width, dim), act)
    prep = PreparedPagedPrefill(_device_fp8_cache(base, packed, act), base.device_tables(), starts, ends,
                                num_heads=heads, query_width=width)
    assert prep.key_groups == groups
    got = prep(storage_to_torch(q, act).cuda()).float().cpu().numpy()
    expected = po.paged_prefill_attention(po.to_f32(q, act), base.oracle_cache, base.tables, starts, ends)
    assert not np.isnan(got).any()
    assert max_abs_err(got, expected, act) < ATOL[act]


@pytest.mark.parametrize("groups,heads,kv,starts,ends,dropped", [
    (4, 8, 2, [0, 1200], [90, 1300], [{1, 5}, {3, 70, 80}]),
    (2, 32, 8, [0, 1100, 31, 0, 0], [65, 1165, 95, 64, 33], [{1}, {2, 66, 71}, {5}, set(), {1, 2}]),
    (1, 32, 8, [0, 1050, 0, 64, 31], [225, 1100, 30, 289, 64], [{1, 13}, {1, 64, 68}, set(), {17}, {3}]),
    (0, 32, 8, [400, 0, 500], [1100, 33, 601], [{1, 65, 68}, {1}, {30, 37}]),
])
def test_entries_outside_the_cache(groups, heads, kv, starts, ends, dropped):
    from inferkernellab_amd import PreparedPagedPrefill

    case = make_prefill_case(starts=starts, ends=ends, num_heads=heads, num_kv_heads=kv, head_dim=64, block_size=16,
                             dtype="bfloat16", seed=groups)
    tables = case.base.device_tables()
    for b, blocks in enumerate(dropped):
        for i, lb in enumerate(sorted(blocks)):
            tables[b, lb] = -1 if i % 2 == 0 else case.base.oracle_cache.num_blocks + 5
    q = case.device_query()
    prep = PreparedPagedPrefill(case.base.device_cache(), tables, starts, ends, num_heads=heads,
                                query_width=q.shape[2])
    assert prep.key_groups == groups
    assert max_abs_err(prep(q), _expected_dropping_blocks(case, dropped)) < ATOL["bfloat16"]


FORCED = [
    (8, 2, 16, [0, 0, 31, 95], [1, 33, 64, 129]),
    (6, 2, 48, [130, 40], [161, 60]),
    (8, 8, 32, [0, 160, 3], [70, 193, 4]),
    (8, 1, 16, [500, 0], [533, 64]),
]


@pytest.mark.parametrize("dim", [32, 64, 96, 128])
@pytest.mark.parametrize("cache", ["same", "fp8"])
@pytest.mark.parametrize("heads,kv,bs,starts,ends", FORCED)
def test_every_plan_gives_the_same_result(heads, kv, bs, starts, ends, cache, dim):
    from inferkernellab_amd import PreparedPagedPrefill

    act = "bfloat16"
    width = max(e - s for s, e in zip(starts, ends))
    if cache == "fp8":
        base, packed = _fp8_case(batch=len(ends), heads=heads, kv=kv, dim=dim, bs=bs, lengths=ends, act=act, seed=dim)
        device = _device_fp8_cache(base, packed, act)
        q = randn_storage(torch.Generator().manual_seed(dim), (len(ends), heads, width, dim), act)
        expected = po.paged_prefill_attention(po.to_f32(q, act), base.oracle_cache, base.tables, starts, ends)
        query, tables = storage_to_torch(q, act).cuda(), base.device_tables()
    else:
        case = make_prefill_case(starts=starts, ends=ends, num_heads=heads, num_kv_heads=kv, head_dim=dim,
                                 block_size=bs, dtype=act, seed=heads + dim)
        device, query, tables, expected = (case.base.device_cache(), case.device_query(), case.base.device_tables(),
                                           case.expected())
    prep = PreparedPagedPrefill(device, tables, starts, ends, num_heads=heads, query_width=width)
    for plan in (0, 1, 2, 4):
        prep.plan = plan
        got = prep(query, out=torch.full_like(query, float("nan"))).float().cpu().numpy()
        assert not np.isnan(got).any()
        assert max_abs_err(got, expected, act) < ATOL[act], plan

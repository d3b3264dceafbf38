"""The value checks of block tables and context lengths (one kernel, read
back through pinned host memory) against the rule they state, over the edges
of the kernel's segments (256 entries a wave, 64 lanes), tables longer and
taller than one workgroup takes, both index types, and strided tables."""

import pytest
import torch

pytestmark = pytest.mark.gpu

BLOCKS, BS = 4000, 16


def _expected(tables, lens, max_context):
    if bool((lens <= 0).any()):
        return "context lengths must be positive"
    if bool((lens > tables.shape[1] * BS).any()):
        return "context length exceeds block table capacity"
    if bool((tables < 0).any()) or bool((tables >= BLOCKS).any()):
        return "block table contains an invalid physical block id"
    if max_context and bool((lens > max_context).any()):
        return "context length exceeds max_context_len"
    return None


def _found(tables, lens, max_context):
    from inferkernellab_amd import ops
    from inferkernellab_amd.cache import CacheLayout

    check = ops._MetadataCheck(tables, lens, CacheLayout(1, BLOCKS, BS, 1, 64), max_context)
    try:
        check.wait()
    except ValueError as exc:
        return str(exc)
    return None


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("batch,width", [(1, 1), (3, 64), (2, 257), (600, 3), (5, 5000), (70, 1024)])
def test_every_finding_at_the_edges(batch, width, dtype):
    gen = torch.Generator().manual_seed(batch + width)
    tables = torch.randint(0, BLOCKS, (batch, width), generator=gen).to(dtype)
    lens = torch.randint(1, width * BS + 1, (batch,), generator=gen).to(dtype)
    cases = [(tables, lens, None), (tables, lens, int(lens.max())), (tables, lens, int(lens.max()) - 1 or None),
             (tables, lens, -1)]
    for b in {0, batch // 2, batch - 1}:
        for w in {0, 63, 64, 255, 256, width - 1}:
            if w < width:
                for bad in (-1, BLOCKS, 2**31 - 1):
                    t = tables.clone()
                    t[b, w] = bad
                    cases.append((t, lens, None))
        for bad in (0, -5, width * BS + 1):
            n = lens.clone()
            n[b] = bad
            cases.append((tables, n, None))
    both = tables.clone()
    both[-1, -1] = -1
    zero = lens.clone()
    zero[0] = 0
    cases.append((both, zero, 1))  # the first rule's message wins
    for t, n, m in cases:
        assert _found(t.cuda(), n.cuda(), m) == _expected(t, n, m)


def test_strided_tables_and_lengths():
    wide = torch.randint(0, BLOCKS, (12, 90), dtype=torch.int32)
    wide[:, 0], wide[:, -1], wide[1::2] = -1, BLOCKS, -7  # outside every view below
    dev = wide.cuda()
    lens = torch.full((2, 6), 40, dtype=torch.int64)
    lens[1] = -1
    assert _found(dev[::2, 1:-1], lens.cuda()[0], None) is None
    assert _found(dev[::2, 1:-1].t()[:6, :6].t(), lens.cuda().t().contiguous()[:, 0], None) is None
    assert _found(dev[:6, 1:-1], lens.cuda()[0], None) == "block table contains an invalid physical block id"


def test_operator_raises_before_it_attends_and_refuses_capture():
    from inferkernellab_amd import PagedKVCache, ops

    cache = PagedKVCache(8, 16, 2, 64, dtype=torch.float16, device="cuda")
    cache.k.zero_()
    cache.v.zero_()
    q = torch.zeros(2, 4, 64, dtype=torch.float16, device="cuda")
    tables = torch.tensor([[0, 1], [2, 3]], dtype=torch.int32, device="cuda")
    lens = torch.tensor([20, 33], dtype=torch.int32, device="cuda")
    for attend in (ops.paged_decode_attention_hip, ops.paged_decode_attention_hip_grouped):
        with pytest.raises(ValueError, match="context length exceeds block table capacity"):
            attend(q, cache, tables, lens)
    with pytest.raises(ValueError, match="context length exceeds block table capacity"):
        ops.paged_decode_attention_hip_grouped(q, cache, tables, lens, query_group_size=3)
    lens.fill_(20)
    assert bool((ops.paged_decode_attention_hip(q, cache, tables, lens) == 0).all())
    graph = torch.cuda.CUDAGraph()
    with pytest.raises(RuntimeError, match="under capture"):
        with torch.cuda.graph(graph):
            ops.paged_decode_attention_hip(q, cache, tables, lens)
    torch.cuda.synchronize()
    assert bool((ops.paged_decode_attention_hip(q, cache, tables, lens) == 0).all())

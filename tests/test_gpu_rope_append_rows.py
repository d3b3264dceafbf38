"""The fused RoPE append at the edges of its row packing: head dims between
the lane groups' powers of two, row counts that leave groups and workgroups
part filled, token counts on both sides of the bound (1024) up to which a
token spreads over several workgroups, with and without a query. Bit for bit
against torch's elementwise rotation, and into the FP8 cache against the torch
quantiser on the rotated rows."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rotate(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos.unsqueeze(1) + torch.cat((-x[..., half:], x[..., :half]), dim=-1) * sin.unsqueeze(1)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("dtype,dim,heads,kv,tokens", [
    (torch.bfloat16, 16, 3, 1, 5),
    (torch.bfloat16, 80, 4, 2, 33),
    (torch.float16, 144, 6, 3, 40),
    (torch.bfloat16, 272, 2, 1, 17),
    (torch.bfloat16, 512, 1, 1, 7),
    (torch.float32, 48, 2, 2, 9),
    (torch.float32, 128, 5, 5, 1024),
    (torch.bfloat16, 128, 32, 32, 3),
    (torch.bfloat16, 128, 32, 8, 1025),
    (torch.float16, 64, 0, 2, 20),
    # past the bounds (512 rows up to 64 dims, 1024 past that) up to which an
    # FP8 row has a workgroup of its own, and four rows a token
    (torch.bfloat16, 16, 3, 1, 110),
    (torch.bfloat16, 64, 4, 2, 64),
    (torch.bfloat16, 64, 4, 2, 65),
    (torch.bfloat16, 80, 4, 2, 130),
    (torch.float16, 144, 6, 3, 90),
    (torch.bfloat16, 272, 3, 1, 210),
    (torch.bfloat16, 512, 2, 2, 172),
    (torch.float32, 48, 2, 2, 90),
    (torch.float16, 128, 2, 1, 700),
    (torch.bfloat16, 128, 8, 2, 85),
    (torch.bfloat16, 128, 8, 2, 86),
])
def test_rows_and_groups(dtype, dim, heads, kv, tokens, fp8):
    from inferkernellab_amd import ops
    from inferkernellab_amd.cache import PagedKVCache, quantize_rows_e4m3

    gen = torch.Generator(device="cuda").manual_seed(dim + tokens)
    rand = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").to(dtype)  # noqa: E731
    q, k, v = rand(tokens, heads, dim) if heads else None, 5 * rand(tokens, kv, dim), rand(tokens, kv, dim)
    v[0] = 0  # a row without a maximum
    cos, sin = rand(tokens, dim), rand(tokens, dim)
    blocks = tokens // 16 + 2
    slots = torch.randperm(blocks * 16, generator=torch.Generator().manual_seed(1))[:tokens].to(torch.int64).cuda()
    slots[tokens // 2] = -1
    cache = PagedKVCache(blocks, 16, kv, dim, dtype=torch.float8_e4m3fn if fp8 else dtype,
                         act_dtype=dtype if fp8 else None, device="cuda")
    for t in (cache.k, cache.v):
        t.view(torch.uint8).fill_(0x11)
    out = torch.empty_like(q) if heads else None
    ops.rope_append_kv_hip(q, k, v, cos, sin, cache, slots, query_out=out)
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    if heads:
        assert torch.equal(out.view(bits), _rotate(q, cos, sin).view(bits))
    ok = slots >= 0
    at = slots[ok]
    for name, rows in (("k", _rotate(k, cos, sin)), ("v", v)):
        store = getattr(cache, name)[0]
        got = store.reshape(blocks * 16, kv, dim)
        untouched = torch.ones(blocks * 16, dtype=torch.bool, device="cuda")
        untouched[at] = False
        if not fp8:
            assert torch.equal(got[at].view(bits), rows[ok].view(bits))
            assert bool((got[untouched].contiguous().view(torch.uint8) == 0x11).all())
            continue
        codes, scales = quantize_rows_e4m3(rows[ok])
        assert torch.equal(got[at].view(torch.uint8), codes.view(torch.uint8))
        assert bool((got[untouched].contiguous().view(torch.uint8) == 0x11).all())
        scale = getattr(cache, name + "_scale")[0].transpose(1, 2).reshape(blocks * 16, kv)
        assert torch.equal(scale[at], scales)
        assert bool((scale[untouched] == 1).all())

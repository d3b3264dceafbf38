"""The Llama layer kernels against the modules they restate, computed in
float64 from the same 16-bit inputs with the modules' roundings: RMSNorm
(+ residual) over row widths at the edges of a workgroup's pieces, SiLU * up,
and the decode linears over row counts at the edges of their 16-row tiles,
contraction lengths at the edges of a wave's steps, and one to three weights
with each epilogue. A result may land on the other side of a rounding
boundary: the bound is one ulp of the dtype per rounding of the sequence, and
what the fp32 arithmetic between the roundings adds. In 16 bits that is rare,
so nearly all results are equal to the reference's: a rounding that a kernel
left out would change one in four."""

import pytest
import torch

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0**-7, torch.float16: 2.0**-10, torch.float32: 2.0**-23}
# Relative errors of the fp32 steps. The norm's factor: a thread's up to 32
# squares summed in a chain and 8 levels of additions, halved by the root, and
# rsqrtf to an ulp. SiLU: expf to an ulp, an addition and a division.
NORM_FACTOR = (32 + 8) / 2 * 2.0**-24 + 2.0**-23
SILU = 2.0**-23 + 2 * 2.0**-24


def _close(got, expected, bound):
    err = (got.double() - expected).abs()
    assert bool((err <= bound).all()), (float((err - bound).max()), float(err.max()))
    if got.dtype != torch.float32:
        off = int((got != expected.to(got.dtype)).sum())
        assert off <= max(1, 0.03 * got.numel()), (off, got.numel())


def _rounded(expected, dtype, roundings, arithmetic, factor):
    """Bound of `expected` = round(round(.) * factor): relative, and below the
    dtype's normal range the ulp of its smallest normal value."""
    return (roundings * ULP[dtype] + arithmetic) * expected.abs() + _subnormal(dtype, factor)


def _subnormal(dtype, factor):
    return ULP[dtype] * torch.finfo(dtype).tiny * (1 + factor.double().abs())


def _norm(x, w, eps):
    d = x.double()
    d = (d * torch.rsqrt(d.square().mean(-1, keepdim=True) + eps)).to(x.dtype)
    return w.double() * d.double()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,cols", [(1, 8), (3, 24), (16, 2048), (5, 2056), (17, 4096)])
@pytest.mark.parametrize("add", [False, True])
def test_add_rms_norm(dtype, rows, cols, add):
    from inferkernellab_amd import layer_ops as lo

    g = torch.Generator(device="cuda").manual_seed(rows + cols)
    x = torch.randn(rows, cols, device="cuda", generator=g).to(dtype)
    wide = torch.randn(rows, 2 * cols, device="cuda", generator=g).to(dtype)
    delta = wide[:, :cols] if add else None  # strided rows
    w = (1 + 0.1 * torch.randn(cols, device="cuda", generator=g)).to(dtype)
    with torch.no_grad():
        assert lo.norm_fits(w, x)
        total, out = lo.add_rms_norm(x, delta, w, 1e-6)
    expected = x + delta if add else x
    assert torch.equal(total, expected)
    want = _norm(expected, w, 1e-6)
    _close(out, want, _rounded(want, dtype, 2, NORM_FACTOR, w))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_add_rms_norm_takes_a_delta_at_any_address(dtype):
    from inferkernellab_amd import layer_ops as lo

    x = torch.randn(5, 64, device="cuda").to(dtype)
    delta = torch.randn(5 * 64 + 1, device="cuda").to(dtype)[1:].view(5, 64)
    w = torch.ones(64, device="cuda", dtype=dtype)
    assert delta.is_contiguous() and delta.data_ptr() % 16
    with torch.no_grad():
        total, out = lo.add_rms_norm(x, delta, w, 1e-6)
    assert torch.equal(total, x + delta)
    want = _norm(x + delta, w, 1e-6)
    _close(out, want, _rounded(want, dtype, 2, NORM_FACTOR, w))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [(8,), (3, 40), (257, 512)])
def test_silu_mul(dtype, shape):
    from inferkernellab_amd import layer_ops as lo

    g = torch.Generator(device="cuda").manual_seed(7)
    gate, up = (4 * torch.randn(2, *shape, device="cuda", generator=g)).to(dtype)
    gate.view(-1)[:4] = torch.tensor([float("-inf"), 100.0, -100.0, 0.0], device="cuda")
    up.view(-1)[0] = 1.0
    assert lo.silu_mul_fits(gate, up)
    got = lo.silu_mul(gate, up)
    d = gate.double()
    expected = (d / (1 + torch.exp(-d))).to(dtype).double() * up.double()
    assert bool(torch.isnan(got.view(-1)[0])) and bool(torch.isnan(expected.view(-1)[0]))  # -inf * 0
    want = expected.view(-1)[1:]
    # below -88.7 fp32's exponential overflows and SiLU is 0, as the module's:
    # at most 89 exp(-88.7) lost
    up = up.view(-1)[1:]
    lost = 89 * 2.0**-128 * up.double().abs()
    _close(got.view(-1)[1:], want, _rounded(want, dtype, 2, SILU, up) + lost)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 7, 15, 16])
@pytest.mark.parametrize("cols,outs", [(64, (16,)), (512, (48, 16, 32)), (576, (64, 16)), (2048, (256, 64, 64)),
                                       (2112, (32,)), (5632, (16,))])
def test_decode_linear(dtype, rows, cols, outs):
    from inferkernellab_amd import layer_ops as lo

    g = torch.Generator(device="cuda").manual_seed(rows + cols + len(outs))
    x = torch.randn(rows, 2 * cols, device="cuda", generator=g).to(dtype)[:, cols:]  # strided rows
    ws = [(torch.randn(n, cols, device="cuda", generator=g) * cols**-0.5).to(dtype) for n in outs]
    products = [x.double() @ w.double().t() for w in ws]  # of magnitude about 1
    # fp32 sums in any order: a few times 2^-24 of the terms' magnitudes
    sums = [2.0**-21 * (x.double().abs() @ w.double().abs().t()) for w in ws]
    got = lo.decode_linear(x, ws)
    for y, e, err in zip([got] if len(ws) == 1 else got, products, sums):
        _close(y, e, 0.5 * ULP[dtype] * e.abs() + err)
    p, up = products[0], torch.flip(products[0], (1,))
    slack = sums[0] + torch.flip(sums[0], (1,))
    res = torch.randn(rows, outs[0], device="cuda", generator=g).to(dtype)
    y = lo.decode_linear(x, ws[:1], residual=res)
    want = res.double() + p.to(dtype).double()
    _close(y, want, ULP[dtype] * (p.abs() + want.abs()) + sums[0])
    y = lo.decode_linear(x, [ws[0], torch.flip(ws[0], (0,)).contiguous()], silu=True)
    a, b = p.to(dtype).double(), up.to(dtype).double()
    sigma = 1 / (1 + torch.exp(-a))
    want = (a * sigma).to(dtype).double() * b
    # an ulp of a moves SiLU by |1 + a (1 - sigma)| of itself; then SiLU's own
    # rounding, b's and the product's
    moved = 3 + (1 + a * (1 - sigma)).abs()
    _close(y, want, _rounded(want, dtype, moved, SILU, b) + 2 * slack * (1 + b.abs()))


@pytest.mark.parametrize("rows", [1, 5, 16])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_operand_order_changes_no_value(dtype, rows):
    """norm -> gate * up -> down with the tensors between them in operand
    order, against the same kernels over plain rows: bit for bit."""
    from inferkernellab_amd import layer_ops as lo

    g = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, 576, device="cuda", generator=g).to(dtype)
    w = torch.randn(576, device="cuda", generator=g).to(dtype)
    gate, up = (0.05 * torch.randn(2, 704, 576, device="cuda", generator=g)).to(dtype)
    down = (0.05 * torch.randn(576, 704, device="cuda", generator=g)).to(dtype)
    _, a = lo.add_rms_norm(x, None, w, 1e-6)
    b = lo.decode_linear(a, (gate, up), silu=True)
    c = lo.decode_linear(b, (down,), residual=x)
    _, pa = lo.add_rms_norm(x, None, w, 1e-6, packed=True)
    pb = lo.decode_linear(pa, (gate, up), rows=rows, silu=True, packed=True)
    assert torch.equal(lo.decode_linear(pb, (down,), rows=rows, residual=x), c)
    assert torch.equal(lo.decode_linear(pa, (gate,), rows=rows), lo.decode_linear(a, (gate,)))


def test_what_the_kernels_do_not_restate_is_left_to_the_module():
    from inferkernellab_amd import layer_ops as lo

    x = torch.zeros(4, 128, dtype=torch.bfloat16, device="cuda")
    lin = torch.nn.Linear(128, 32, bias=False, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        assert lo.kernels_apply(x) and lo.linear_fits(lin, x)
        assert not lo.linear_fits(lin, torch.zeros(17, 128, dtype=torch.bfloat16, device="cuda"))
        assert not lo.linear_fits(lin, x.float()) and not lo.linear_fits(lin, x[:0])
        assert not lo.linear_fits(torch.nn.Linear(128, 24, bias=False, device="cuda", dtype=torch.bfloat16), x)
        assert not lo.linear_fits(torch.nn.Linear(128, 32, device="cuda", dtype=torch.bfloat16), x)
        with torch.autocast("cuda", dtype=torch.float16):
            assert not lo.kernels_apply(x)
        handle = lin.register_forward_hook(lambda *a: None)
        assert not lo.linear_fits(lin, x)
        handle.remove()
        torch.nn.utils.parametrizations.weight_norm(lin)
        assert not lo.linear_fits(lin, x)
    assert not lo.kernels_apply(x)  # autograd may record


def test_a_hooked_head_sees_all_rows_and_gives_the_same_tokens():
    """The runner computes logits of the chunks' last rows only; with a hook
    on the head, of all rows. Ragged prompts, two prefill batches."""
    from inferkernellab_amd.llama import LlamaConfig, LlamaPagedDecodeRunner, random_llama

    cfg = LlamaConfig(vocab_size=128, hidden_size=256, intermediate_size=512, num_hidden_layers=2,
                      num_attention_heads=4, num_key_value_heads=2)
    model = random_llama(cfg, seed=3, device="cuda", dtype=torch.float32)
    prompts = [list(range(1, 1 + n)) for n in (5, 17, 9, 30)]
    kw = dict(max_new_tokens=4, max_num_batched_tokens=32)
    plain = LlamaPagedDecodeRunner(model, prompts, **kw).run()
    rows = []
    handle = model.lm_head.register_forward_hook(lambda mod, args, out: rows.append(args[0].shape))
    hooked = LlamaPagedDecodeRunner(model, prompts, **kw).run()
    handle.remove()
    assert any(len(shape) == 3 for shape in rows)
    assert plain.generated_tokens == hooked.generated_tokens
    assert torch.allclose(plain.prompt_logits, hooked.prompt_logits, atol=1e-5, rtol=1e-5)
    assert len(plain.decode_logits) == len(hooked.decode_logits) == 4
    for a, b in zip(plain.decode_logits, hooked.decode_logits):
        assert a.shape == b.shape and not a.is_cuda and torch.allclose(a, b, atol=1e-5, rtol=1e-5)

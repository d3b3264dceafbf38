"""Which layers of a decode step the linear kernels restate: they read the
norms' output in the norm kernel's own layout, so a norm that runs as a module
(any type, any strides may come out of it) takes the whole layer to its
modules. No kernel stands in for a module while a mode watches torch's calls.
And which final norms and heads a prefill gives the chunks' last rows alone. The rules themselves run here, with the device condition stubbed."""

import pytest
import torch
from torch import nn

from inferkernellab_amd import layer_ops
from inferkernellab_amd.llama import LlamaConfig, LlamaPagedDecodeRunner, RMSNorm, random_llama


class _ColumnMajorNorm(RMSNorm):
    def forward(self, x):
        return super().forward(x).t().contiguous().t()


@pytest.fixture
def layer(monkeypatch):
    monkeypatch.setattr(layer_ops, "kernels_apply", lambda x: True)
    cfg = LlamaConfig(vocab_size=32, hidden_size=64, intermediate_size=128, num_hidden_layers=1,
                      num_attention_heads=2, num_key_value_heads=1)
    return random_llama(cfg, seed=0, device="cpu", dtype=torch.bfloat16).model.layers[0]


def _restated(layer, delta=None):
    hidden = torch.zeros(3, 64, dtype=torch.bfloat16)
    runner = LlamaPagedDecodeRunner.__new__(LlamaPagedDecodeRunner)
    return runner._decode_linears(layer, hidden, delta)


def test_plain_layer_is_restated(layer):
    assert _restated(layer)
    assert _restated(layer, torch.zeros(3, 64, dtype=torch.bfloat16))


@pytest.mark.parametrize("name", ["input_layernorm", "post_attention_layernorm"])
@pytest.mark.parametrize("change", ["subclass", "hook", "weight type"])
def test_norm_that_runs_as_a_module_keeps_the_layers_linears(layer, name, change):
    norm = getattr(layer, name)
    if change == "subclass":
        setattr(layer, name, _ColumnMajorNorm(64, 1e-6).to(torch.bfloat16))
    elif change == "hook":
        norm.register_forward_hook(lambda mod, args, out: out.half())
    else:
        norm.weight = nn.Parameter(norm.weight.detach().float())
    assert not _restated(layer)


def test_delta_that_promotes_the_residual_keeps_the_layers_linears(layer):
    assert not _restated(layer, torch.zeros(3, 64))


class _GpuLooking:
    """A plain tensor on a GPU, to the rule."""

    device, dtype = torch.device("cuda"), torch.bfloat16


def test_a_watched_call_is_left_to_the_module(monkeypatch):
    from torch.overrides import TorchFunctionMode
    from torch.utils.flop_counter import FlopCounterMode

    monkeypatch.setattr(layer_ops.torch, "Tensor", _GpuLooking)
    x = _GpuLooking()
    with torch.no_grad():
        assert layer_ops.kernels_apply(x)
        with torch.device("cpu"):  # a default device is no watcher
            assert layer_ops.kernels_apply(x)
        with TorchFunctionMode():
            assert not layer_ops.kernels_apply(x)
        with FlopCounterMode(display=False):
            assert not layer_ops.kernels_apply(x)
        assert layer_ops.kernels_apply(x)


class _RecordingNorm(RMSNorm):
    """A replaced final norm: what it computes may depend on all rows."""

    def forward(self, x):
        self.seen.append(x.shape)
        return super().forward(x)


def _last_logits(change):
    cfg = LlamaConfig(vocab_size=32, hidden_size=64, intermediate_size=128, num_hidden_layers=1,
                      num_attention_heads=2, num_key_value_heads=1)
    runner = LlamaPagedDecodeRunner.__new__(LlamaPagedDecodeRunner)
    runner.model = random_llama(cfg, seed=0, device="cpu", dtype=torch.float32)
    seen = []
    change(runner.model, seen)
    gen = torch.Generator().manual_seed(1)
    hidden, delta = torch.randn(2, 3, 5, 64, generator=gen)
    spans = [5, 1, 3]
    got = runner._last_logits(hidden, delta, spans)
    full = runner.model.lm_head(runner.model.model.norm(hidden + delta))
    assert torch.allclose(got, full[torch.arange(3), torch.tensor(spans) - 1], atol=1e-6)
    return seen[0]


def test_a_plain_final_norm_and_head_see_the_last_rows_alone():
    def watch(model, seen):
        weight = model.lm_head.weight

        class Watched(torch.Tensor):
            @classmethod
            def __torch_function__(cls, func, types, args=(), kwargs=None):
                if func is nn.functional.linear:
                    seen.append(args[0].shape)
                return super().__torch_function__(func, types, args, kwargs or {})

        model.lm_head.weight = nn.Parameter(weight.as_subclass(Watched), requires_grad=False)

    assert _last_logits(watch) == (3, 64)


@pytest.mark.parametrize("what", ["replaced norm", "hooked norm", "hooked head"])
def test_anything_else_after_the_layers_sees_all_rows(what):
    def change(model, seen):
        if what == "replaced norm":
            model.model.norm = _RecordingNorm(64, 1e-6)
            model.model.norm.seen = seen
        else:
            module = model.model.norm if what == "hooked norm" else model.lm_head
            module.register_forward_hook(lambda mod, args, out: seen.append(args[0].shape))

    assert _last_logits(change) == (3, 5, 64)


def test_the_transformers_norm_works_row_by_row():
    modeling = pytest.importorskip("transformers.models.llama.modeling_llama")
    from inferkernellab_amd.llama import _plain_row_norm

    norm = modeling.LlamaRMSNorm(64)
    assert _plain_row_norm(norm) and _plain_row_norm(RMSNorm(64, 1e-6))
    norm.register_forward_hook(lambda *a: None)
    assert not _plain_row_norm(norm) and not _plain_row_norm(nn.LayerNorm(64))

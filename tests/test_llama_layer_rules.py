"""Which layers of a decode step the linear kernels restate: they read the
norms' output in the norm kernel's own layout, so a norm that runs as a module
(any type, any strides may come out of it) takes the whole layer to its
modules. The rule itself runs here, with the device condition stubbed."""

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

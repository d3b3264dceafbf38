"""The host side of the value checks (enqueue, wait, pinned words) with the
library stubbed: which device is current at each call, and which words a check
may write."""

import contextlib
import types

import pytest
import torch

from inferkernellab_amd import ops

LAYOUT = types.SimpleNamespace(block_size=16, num_blocks=8)


class _Lib:
    """Records each call with the device current at it; `found` is what a
    check finds."""

    def __init__(self, found=0):
        self.found, self.calls, self.current = found, [], "cuda:0"

    def ikl_check_metadata(self, *args):
        self.calls.append(("check", self.current, args[-3]))
        return 1

    def ikl_check_metadata_wait(self, words, count, stream):
        self.calls.append(("wait", self.current, words))
        return self.found


class _Tensor:
    """What a check asks of a tensor, on the second GPU."""

    dtype, device, shape = torch.int32, torch.device("cuda:1"), (2, 3)

    def data_ptr(self):
        return 0

    def stride(self, i):
        return 1


@pytest.fixture
def lib(monkeypatch):
    stub = _Lib()

    @contextlib.contextmanager
    def on_device(device):
        before, stub.current = stub.current, str(device)
        yield
        stub.current = before

    monkeypatch.setattr(ops, "_require_backend", lambda: stub)
    monkeypatch.setattr(ops, "_on_device", on_device)
    monkeypatch.setattr(ops.torch.cuda, "current_stream", lambda d: types.SimpleNamespace(cuda_stream=0))
    real = torch.empty
    monkeypatch.setattr(ops.torch, "empty", lambda *a, pin_memory=False, **kw: real(*a, **kw))
    return stub


def _check():
    return ops._MetadataCheck(_Tensor(), _Tensor(), LAYOUT, None)


@pytest.mark.parametrize("found", [0, 1])
def test_a_check_is_waited_for_on_its_own_device(lib, found):
    lib.found = found
    with pytest.raises(ValueError) if found else contextlib.nullcontext():
        with _check():
            assert lib.current == "cuda:0"
    assert [c[:2] for c in lib.calls] == [("check", "cuda:1"), ("wait", "cuda:1")]

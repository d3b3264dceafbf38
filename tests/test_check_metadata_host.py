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


@pytest.fixture
def words(monkeypatch):
    """The module's word buffers, empty, as the test leaves them."""
    for name in ("_check_words_made", "_check_words_free"):
        monkeypatch.setattr(ops, name, [], raising=False)


def test_words_serve_the_next_check_once_they_were_waited_for(lib, words):
    for _ in range(3):
        _check().wait()
    assert len({c[2] for c in lib.calls}) == 1


def test_words_of_a_check_that_was_not_waited_for_are_left_alone(lib, words):
    """Its kernel may still write: an interrupt came between the two."""
    lost = _check()
    _check().wait()
    with _check():  # and a check that begins while another is in flight
        _check().wait()
    first = lib.calls[0][2]
    assert all(c[2] != first for c in lib.calls[1:])
    assert lost is not None and any(tensor.data_ptr() == first for tensor, _ in ops._check_words_made)


def test_words_of_a_failed_wait_are_kept_and_not_used_again(lib, words):
    lib.found = -3
    with pytest.raises(RuntimeError):
        _check().wait()
    failed = lib.calls[0][2]
    lib.found = 0
    _check().wait()
    assert lib.calls[-1][2] != failed
    assert any(tensor.data_ptr() == failed for tensor, _ in ops._check_words_made)


def test_words_of_a_refused_check_are_free_again(lib, words, monkeypatch):
    monkeypatch.setattr(lib, "ikl_check_metadata", lambda *a: -3)
    for _ in range(3):
        with pytest.raises(RuntimeError):
            _check()
    assert len(ops._check_words_made) == 1

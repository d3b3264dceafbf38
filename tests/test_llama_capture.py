"""Capturing a decode step when memory runs out: the capture is made again once
the allocator has given its cached blocks back, those of the failed capture
included, and any other error is the caller's. And that no graph is destroyed
during a capture, which would end the process: no garbage is collected in one,
and a run leaves no graph to the collector."""

import contextlib
import gc
import weakref

import pytest
import torch

from inferkernellab_amd.llama import LlamaConfig, LlamaPagedDecodeRunner, random_llama


@pytest.fixture
def device(monkeypatch):
    """A device without a GPU: graphs that record what happens to them."""
    log = []

    class Graph:
        def __init__(self):
            log.append(weakref.ref(self))

        def capture_begin(self):
            log.append("begin")

        def capture_end(self):
            log.append("end")

    monkeypatch.setattr(torch.cuda, "CUDAGraph", Graph)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda d: None)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d: (1 << 40, 1 << 40))
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "empty_cache",
                        lambda: log.append(("empty", [r() for r in log if isinstance(r, weakref.ref)])))
    return log


def _runner(errors):
    runner = LlamaPagedDecodeRunner.__new__(LlamaPagedDecodeRunner)
    runner.device = None
    errors = iter(errors)

    def body(st):
        kind, message = next(errors, (None, ""))
        if kind is not None:
            raise kind(message)

    runner._graph_body = body
    return runner


def test_a_capture_that_runs_out_of_memory_is_made_again(device):
    graph = _runner([(torch.OutOfMemoryError, "full")])._capture(None, None)
    steps = [x for x in device if not isinstance(x, weakref.ref)]
    assert steps == ["begin", "end", ("empty", [None]), "begin", "end"]  # the first graph is gone by then
    assert graph is not None


def test_a_second_failure_and_other_errors_are_raised(device):
    with pytest.raises(torch.OutOfMemoryError, match="again"):
        _runner([(torch.OutOfMemoryError, "full"), (torch.OutOfMemoryError, "again")])._capture(None, None)
    del device[:]
    with pytest.raises(ValueError, match="wrong"):
        _runner([(ValueError, "wrong")])._capture(None, None)
    assert [x for x in device if not isinstance(x, weakref.ref)] == ["begin", "end"]


@pytest.mark.parametrize("enabled", [True, False])
@pytest.mark.parametrize("error", [None, ValueError])
def test_no_garbage_is_collected_during_a_capture(device, enabled, error):
    class Cycle:
        def __init__(self):
            self.me = self

    before = gc.isenabled()
    (gc.enable if enabled else gc.disable)()
    try:
        runner, collected = _runner([]), []

        def body(st):
            dead = Cycle()
            weakref.finalize(dead, collected.append, 1)
            del dead
            garbage = [[] for _ in range(200_000)]  # far past the collector's thresholds
            assert garbage and not collected
            if error is not None:
                raise error("body")

        runner._graph_body = body
        with pytest.raises(error) if error else contextlib.nullcontext():
            runner._capture(None, None)
        assert gc.isenabled() == enabled
    finally:
        (gc.enable if before else gc.disable)()


@pytest.mark.gpu
def test_a_run_leaves_no_graph_behind(monkeypatch):
    cfg = LlamaConfig(vocab_size=128, hidden_size=256, intermediate_size=512, num_hidden_layers=1,
                      num_attention_heads=4, num_key_value_heads=2)
    runner = LlamaPagedDecodeRunner(random_llama(cfg, seed=3, device="cuda", dtype=torch.float32),
                                    [[1, 2, 3], [4, 5]], max_new_tokens=3)
    graphs, record = [], runner._record

    def recorded(st, side):
        graph = record(st, side)
        graphs.append(weakref.ref(graph))
        return graph

    monkeypatch.setattr(runner, "_record", recorded)
    gc.disable()
    try:
        result = runner.run()
        assert graphs and all(g() is None for g in graphs)
    finally:
        gc.enable()
    assert len(result.decode_logits) == 3


@pytest.mark.gpu
def test_a_run_goes_on_after_a_capture_that_ran_out_of_memory(monkeypatch):
    cfg = LlamaConfig(vocab_size=128, hidden_size=256, intermediate_size=512, num_hidden_layers=2,
                      num_attention_heads=4, num_key_value_heads=2)
    model = random_llama(cfg, seed=3, device="cuda", dtype=torch.float32)
    prompts = [list(range(1, 1 + n)) for n in (5, 17, 9)]
    want = LlamaPagedDecodeRunner(model, prompts, max_new_tokens=4).run()
    runner = LlamaPagedDecodeRunner(model, prompts, max_new_tokens=4)
    real, failures = runner._graph_body, []

    def body(st):
        real(st)
        if torch.cuda.is_current_stream_capturing() and not failures:
            failures.append(1)
            raise torch.OutOfMemoryError("full")

    monkeypatch.setattr(runner, "_graph_body", body)
    got = runner.run()
    assert failures and got.generated_tokens == want.generated_tokens
    for a, b in zip(got.decode_logits, want.decode_logits):
        assert torch.equal(a, b)

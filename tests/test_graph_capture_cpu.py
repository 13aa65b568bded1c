"""Nothing is collected while a decode bucket is captured."""

import contextlib
import gc
from types import SimpleNamespace

import pytest
import torch


class _Dead:
    """Stands for an engine that holds captured graphs and is part of a
    cycle; notes whether it goes while another graph is captured."""

    def __init__(self, capturing, seen):
        self.me, self.capturing, self.seen = self, capturing, seen

    def __del__(self):
        self.seen.append(bool(self.capturing))


@pytest.fixture
def runner(monkeypatch):
    from gllm_amd.runtime.graph_runner import GraphRunner
    capturing, seen = [], []

    @contextlib.contextmanager
    def graph(g, pool=None, stream=None):
        capturing.append(1)
        try:
            yield
        finally:
            capturing.pop()
    cuda = torch.cuda
    monkeypatch.setattr(cuda.graphs, "graph_pool_handle", lambda: None)
    monkeypatch.setattr(cuda, "Stream", lambda: None)
    monkeypatch.setattr(cuda, "stream",
                        lambda s: contextlib.nullcontext())
    monkeypatch.setattr(cuda, "current_stream", lambda: SimpleNamespace(
        wait_stream=lambda s: None))
    monkeypatch.setattr(cuda, "synchronize", lambda: None)
    monkeypatch.setattr(cuda, "CUDAGraph", SimpleNamespace)
    monkeypatch.setattr(cuda, "graph", graph)
    r = GraphRunner.__new__(GraphRunner)
    r.buckets, r.max_bs, r.dummy_page = [1, 2], 2, 3
    r.graphs, r.hidden_out, r.captured = {}, {}, False
    r.uses_mrope, r.ssm_slots_dev = False, None
    r.in_ids, r.positions, r.slots = (torch.zeros(2, dtype=torch.long)
                                      for _ in range(3))
    r.block_table = torch.zeros(2, 4, dtype=torch.int32)
    r.seq_lens = torch.ones(2, dtype=torch.int32)
    r.qsl = torch.arange(3, dtype=torch.int32)

    def model(ids, pos, fctx):
        for _ in range(50):          # enough to set the collector off
            [[] for _ in range(20)]
            if capturing:
                _Dead(capturing, seen)
        return ids, None
    r.runner = SimpleNamespace(
        config=SimpleNamespace(page_size=16), resolve_tokens=lambda t: t,
        model=model, k_caches=[], v_caches=[])
    r.test = SimpleNamespace(capturing=capturing, seen=seen)
    before = gc.get_threshold()
    gc.collect()
    gc.set_threshold(10, 1, 1)
    yield r
    gc.set_threshold(*before)
    gc.enable()


def test_collector_is_held_over_captures(runner):
    _Dead(runner.test.capturing, runner.test.seen)
    runner.capture_all()
    assert runner.captured and sorted(runner.graphs) == [1, 2]
    gc.collect()
    # the one from before and those of both captures
    assert runner.test.seen == [False] * 101
    assert gc.isenabled()


def test_collector_is_left_as_it_was(runner):
    gc.disable()
    runner.capture_all()
    assert not gc.isenabled()
    gc.enable()

    def fails(ids, pos, fctx):
        raise RuntimeError("capture")
    runner.runner.model = fails
    with pytest.raises(RuntimeError, match="capture"):
        runner.capture_all()
    assert gc.isenabled()

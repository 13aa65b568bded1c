"""The zeros that a forward's decode attention counts in: whose they are, and
for how long."""

from types import SimpleNamespace

import pytest
import torch

from gllm_amd.runtime.forward_context import ForwardContext


@pytest.fixture
def now(monkeypatch):
    state = SimpleNamespace(stream=1, capturing=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a:
                        SimpleNamespace(cuda_stream=state.stream))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing",
                        lambda: state.capturing)
    return state


def _context(**kw):
    one = torch.ones(3, dtype=torch.int32)
    return ForwardContext(
        num_tokens=3, positions=one, slot_mapping=one, block_table=one[None],
        seq_lens=one, query_start_loc=one, max_query_len=1, max_seq_len=1,
        k_caches=[], v_caches=[], **kw)


def test_layers_of_a_stream_share_them(now):
    f = _context()
    few = f.arrivals(2)
    many = f.arrivals(8)
    assert few.numel() >= 6 and many.numel() >= 24
    assert many.dtype == torch.int32 and not many.any()
    assert f.arrivals(2) is many and f.arrivals(8) is many


def test_streams_do_not(now):
    f = _context()
    first = f.arrivals(4)
    now.stream = 2
    assert f.arrivals(4) is not first
    now.stream = 1
    assert f.arrivals(4) is first


def test_a_capture_keeps_its_own(now):
    f = _context()
    eager = f.arrivals(4)
    now.capturing = True
    captured = f.arrivals(4)
    # (the context may go before the graph does, and its buffer with it)
    assert captured is not eager
    # (what a capture zeroes is not zero before its first replay)
    now.capturing = False
    assert f.arrivals(4) is eager
    now.stream, now.capturing = 2, True
    captured = f.arrivals(4)
    now.capturing = False
    assert f.arrivals(4) is not captured


def test_the_owner_of_a_graph_lends_them(now):
    zeros = torch.zeros(12, dtype=torch.int32)
    f = _context(arrived=zeros)
    now.capturing = True
    assert f.arrivals(4) is zeros and f.arrivals(2) is zeros
    # a layer with more heads leaves the others their buffer
    assert f.arrivals(8).numel() == 24
    assert f.arrivals(4) is zeros

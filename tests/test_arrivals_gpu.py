"""A captured step whose context is gone before the graph is replayed, and two
streams that share a context."""

import pytest
import torch

from test_qkv_decode_gpu import _step

pytestmark = pytest.mark.gpu

LENS = [2600, 1, 40, 1300, 33, 900]


def _context(s):
    from gllm_amd.runtime.forward_context import ForwardContext
    return ForwardContext(
        num_tokens=len(LENS), positions=s["positions"],
        slot_mapping=s["slots"], block_table=s["table"], seq_lens=s["lens"],
        query_start_loc=torch.arange(len(LENS) + 1, device="cuda"),
        max_query_len=1, max_seq_len=max(LENS), k_caches=[s["k"]],
        v_caches=[s["v"]])


def _attend(s, fctx):
    from gllm_amd import ops
    return ops.qkv_decode(
        s["parts"], s["bias"], s["positions"], s["cos_sin"], s["k"], s["v"],
        s["slots"], s["table"], s["lens"], fctx.arrivals(8), 32, 128 ** -0.5)


def test_graph_outlives_its_context():
    s = _step(len(LENS), 32, 8, 128, 128, 4, LENS)
    fctx = _context(s)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        want = _attend(s, fctx).clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        outs = [_attend(s, fctx) for _ in range(3)]
    assert torch.equal(_attend(s, fctx), want)   # before any replay
    del fctx
    for i in range(4):
        # whatever memory is free now is not zero
        with torch.cuda.stream(stream):
            junk = [torch.full((n,), 7, dtype=torch.int32, device="cuda")
                    for n in (48, 64, 128, 512, 4096)]
        for out in outs:
            out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for out in outs:
            assert torch.equal(out, want), i
        assert all((j == 7).all() for j in junk)


def test_two_streams():
    steps = [_step(len(LENS), 32, 8, 128, 128, 4, LENS, seed=i)
             for i in range(2)]
    fctx = _context(steps[0])
    want = [_attend(s, _context(s)) for s in steps]
    streams = [torch.cuda.Stream() for _ in steps]
    torch.cuda.synchronize()
    outs = [[], []]
    for _ in range(20):
        for i, stream in enumerate(streams):
            with torch.cuda.stream(stream):
                outs[i].append(_attend(steps[i], fctx))
    torch.cuda.synchronize()
    for got, one in zip(outs, want):
        assert all(torch.equal(g, one) for g in got)

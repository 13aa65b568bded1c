"""Decode attention straight from a projection's parts against the two
kernels that it stands for: the same sums in the same order, so the same
bits, in the caches too; rows that are not rounded may be split less, and
then each form's weights are rounded to bf16 against another maximum."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _step(B, Hq, Hkv, D, rot, S, lens, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rand(*shape):
        return torch.randn(*shape, device="cuda", generator=g)
    N = (Hq + 2 * Hkv) * D
    pages = [max(1, -(-n // 16)) for n in lens]
    table = torch.zeros(B, max(pages) + 3, dtype=torch.int32, device="cuda")
    free = torch.randperm(sum(pages) + 1, generator=g,
                          device="cuda").int()[1:]
    at = 0
    slots = []
    for b, n in enumerate(pages):
        table[b, :n] = free[at:at + n]
        at += n
        last = max(lens[b] - 1, 0)
        slots.append(int(table[b, last // 16]) * 16 + last % 16)
    ang = torch.arange(4096).double()[:, None] * 1e4 ** (
        -torch.arange(0, rot, 2).double() / rot)
    return dict(
        parts=rand(S, B, N) * S ** -0.5, bias=rand(N).bfloat16(),
        positions=torch.tensor([max(n - 1, 0) for n in lens], device="cuda"),
        cos_sin=torch.cat([ang.cos(), ang.sin()], -1).float().cuda(),
        k=rand(sum(pages) + 1, 16, Hkv, D).bfloat16(),
        v=rand(sum(pages) + 1, 16, Hkv, D).bfloat16(),
        slots=torch.tensor(slots, device="cuda"), table=table,
        lens=torch.tensor(lens, dtype=torch.int32, device="cuda"))


def _both(s, Hq, D, window, rounded, bias, arrived):
    from gllm_amd import ops
    scale = D ** -0.5
    bias = s["bias"] if bias else None
    k0, v0 = s["k"].clone(), s["v"].clone()
    q = ops.qkv_rope_cache(s["parts"], bias, s["positions"], s["cos_sin"],
                           k0, v0, s["slots"], Hq, rounded=rounded)
    want = ops.paged_attention(
        q.view(-1, Hq, D), k0, v0, s["table"], s["lens"], None, scale,
        sliding_window=window).flatten(1)
    k1, v1 = s["k"].clone(), s["v"].clone()
    # what the new token's slots hold beforehand must not matter
    k1.view(-1, *k1.shape[2:])[s["slots"]] = float("nan")
    v1.view(-1, *v1.shape[2:])[s["slots"]] = float("nan")
    got = ops.qkv_decode(s["parts"], bias, s["positions"], s["cos_sin"], k1,
                         v1, s["slots"], s["table"], s["lens"], arrived, Hq,
                         scale, window, rounded)
    return (got, k1, v1), (want, k0, v0)


CASES = [
    # B, Hq, Hkv, D, rot, S, lengths, window
    (1, 32, 8, 128, 128, 6, [600], 0),          # split, few splits live
    (1, 8, 8, 64, 64, 1, [1], 0),               # nothing but the new token
    (3, 40, 8, 128, 128, 4, [32, 33, 2000], 0),  # edges of a tile
    (5, 6, 3, 80, 40, 9, [31, 128, 129, 500, 64], 0),
    (4, 16, 1, 128, 64, 16, [700, 5, 64, 1000], 0),  # the widest group
    (64, 40, 8, 128, 128, 4, [512 + 16 * i for i in range(64)], 0),
    (40, 32, 8, 128, 128, 7, [1 + 97 * i for i in range(40)], 0),  # in order
    (9, 14, 2, 64, 64, 3, [300, 1, 17, 64, 65, 900, 2, 33, 500], 100),
    (2, 4, 4, 96, 96, 2, [48, 1025], 0),
    # tiles up to which a sequence is not split, and a split's at least
    (4, 8, 8, 64, 64, 2, [256, 257, 384, 4000], 0),
    (12, 16, 8, 128, 128, 2, [768, 769, 1536, 1537, 40, 3000] * 2, 0),
]


@pytest.mark.parametrize("rounded", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,D,rot,S,lens,window", CASES)
def test_as_two_kernels(B, Hq, Hkv, D, rot, S, lens, window, rounded):
    s = _step(B, Hq, Hkv, D, rot, S, lens)
    arrived = torch.zeros(B * Hkv, dtype=torch.int32, device="cuda")
    for bias in (True, False):
        got, want = _both(s, Hq, D, window, rounded, bias, arrived)
        for a, b in zip(got[0 if rounded else 1:], want[0 if rounded else 1:]):
            assert torch.equal(a, b)
        # weights and results of both forms, 2^-9 relative each
        err = (got[0].double() - want[0].double()).norm()
        assert err <= 2 ** -7 * want[0].double().norm()
        assert not arrived.any()


def test_replayed():
    """Captured with counters of its own, replayed between eager launches."""
    from gllm_amd import ops
    s = _step(6, 32, 8, 128, 128, 6, [600, 1, 40, 1300, 33, 256])
    arrived = torch.zeros(48, dtype=torch.int32, device="cuda")
    want, _ = _both(s, 32, 128, 0, False, True, arrived)

    def call():
        return ops.qkv_decode(s["parts"], s["bias"], s["positions"],
                              s["cos_sin"], s["k"], s["v"], s["slots"],
                              s["table"], s["lens"], arrived, 32, 128 ** -0.5)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = call()
    for _ in range(4):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want[0])
        assert not arrived.any()
        assert torch.equal(call(), want[0])


def test_refusals():
    from gllm_amd import ops
    s = _step(2, 8, 2, 64, 64, 2, [10, 20])
    assert ops.qkv_decode_ok(s["parts"], s["k"], 8)
    assert not ops.qkv_decode_ok(s["parts"], s["k"], 34)  # group of 17
    many = s["parts"].expand(2, 2, -1).repeat(1, 600, 1)
    assert not ops.qkv_decode_ok(many, s["k"], 8)  # more than four per CU
    args = [s["parts"], s["bias"], s["positions"], s["cos_sin"], s["k"],
            s["v"], s["slots"], s["table"], s["lens"]]
    few = torch.zeros(3, dtype=torch.int32, device="cuda")
    with pytest.raises(RuntimeError):
        ops.qkv_decode(*args, few, 8, 0.125)
    wide = torch.zeros(4, dtype=torch.int64, device="cuda")
    with pytest.raises(RuntimeError):
        ops.qkv_decode(*args, wide, 8, 0.125)

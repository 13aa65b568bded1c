"""Causal attention of prompt rows against fp64 at the edges of its row and
key tiles."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _attend(q, k, v, scale):
    """q [n, H, D] (the last n positions), k [m, G, D], v [m, G, E], fp64."""
    n, H, m, G = q.shape[0], q.shape[1], k.shape[0], k.shape[1]
    k, v = (t.repeat_interleave(H // G, 1) for t in (k, v))
    s = (q.transpose(0, 1) @ k.permute(1, 2, 0).contiguous()) * scale
    hide = torch.arange(m)[None] > torch.arange(m - n, m)[:, None]
    s = s.masked_fill(hide, -float("inf")).softmax(-1)
    return (s @ v.transpose(0, 1).contiguous()).transpose(0, 1)


def _check(out, ref):
    # bf16 weights of a convex sum (2^-9 each, fp32 sums) and the result
    err = (out.cpu().double() - ref).norm() / ref.norm()
    assert err < 3 * 2 ** -9, err
    assert torch.isfinite(out).all()


@pytest.mark.parametrize("rows,past,Hq,Hkv,D,page", [
    ([2], [0], 1, 1, 128, 16),                      # less than a group
    ([127, 128, 129], [0, 0, 0], 8, 8, 128, 16),    # edges of a row tile
    ([63, 64, 65, 31, 33], [0, 0, 0, 0, 0], 5, 1, 64, 16),
    ([300, 2, 16], [1, 64, 500], 16, 2, 128, 16),   # cached prefixes
    ([1, 1, 200], [700, 0, 0], 10, 2, 128, 48),     # rows that decode
    ([3] * 256, [0] * 256, 2, 1, 64, 16),           # one launch
    ([3] * 256 + [140], [5] * 257, 2, 1, 64, 1),    # two
    ([5] * 300 + [1] * 5, [2] * 305, 2, 1, 64, 16),  # a tile each, one launch
    ([128, 1, 127, 1], [0, 9, 70, 0], 4, 2, 128, 16),
    ([1100], [0], 3, 3, 128, 16),
])
@pytest.mark.parametrize("single", [False, True])
def test_paged(rows, past, Hq, Hkv, D, page, single):
    from gllm_amd import ops
    torch.manual_seed(len(rows) + Hq)
    lens = [a + b for a, b in zip(rows, past)]
    need = [-(-n // page) for n in lens]
    ids = torch.randperm(sum(need) + 3)
    table = torch.zeros(len(lens), max(need), dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = ids[at:at + n].int()
        at += n
    k = torch.randn(sum(need) + 3, page, Hkv, D).bfloat16()
    v = torch.randn_like(k)
    wide = torch.randn(sum(rows), (Hq + 2) * D).bfloat16()  # a row view
    qsl = torch.tensor([0] + rows).cumsum(0).int()
    ref = torch.cat([_attend(
        wide[qsl[i]:qsl[i + 1], :Hq * D].view(-1, Hq, D).double(),
        k[table[i].long()].reshape(-1, Hkv, D)[:n].double(),
        v[table[i].long()].reshape(-1, Hkv, D)[:n].double(), D ** -0.5)
        for i, n in enumerate(lens)])
    q = wide.cuda()[:, :Hq * D].view(-1, Hq, D)
    out = ops.paged_attention(
        q, k.cuda(), v.cuda(), table.cuda(),
        torch.tensor(lens, dtype=torch.int32).cuda(), qsl.cuda(), D ** -0.5,
        max(rows), single_rows=rows.count(1) if single else 0)
    _check(out.view(ref.shape), ref)


def test_scores_far_apart():
    """Maxima that grow by little and by much from tile to tile, and scores
    far below them."""
    from gllm_amd import ops
    torch.manual_seed(1)
    n, D = 400, 64
    k = torch.randn(n // 16, 16, 1, D)
    grow = torch.linspace(0.1, 40, n).view(-1, 16, 1, 1)
    k = (k * grow).bfloat16()
    v = torch.randn_like(k)
    q = torch.randn(n, 2, D).bfloat16()
    ref = _attend(q.double(), k.view(n, 1, D).double(),
                  v.view(n, 1, D).double(), 0.5)
    table = torch.arange(n // 16, dtype=torch.int32)[None].cuda()
    qsl = torch.tensor([0, n], dtype=torch.int32).cuda()
    out = ops.paged_attention(q.cuda(), k.cuda(), v.cuda(), table, qsl[1:],
                              qsl, 0.5, n)
    _check(out.view(ref.shape), ref)


@pytest.mark.parametrize("D", [64, 128])
def test_weights_are_summed_in_32_bits(D):
    """One key of weight 1 and value 1, the others of one weight w a row and
    value 0: the result is 1 / (1 + n w), off by its own rounding only."""
    from gllm_amd import ops
    rows, past = 500, 300
    n = rows + past
    k = torch.zeros(n // 16, 16, 1, D)
    k[0, 0, 0, 0] = 1.0
    v = torch.zeros_like(k)
    v[0, 0] = 1.0
    q = torch.zeros(rows, 1, D)
    q[:, 0, 0] = torch.linspace(0.5, 6, rows)
    q, k, v = q.bfloat16(), k.bfloat16(), v.bfloat16()
    ref = _attend(q.double(), k.view(n, 1, D).double(),
                  v.view(n, 1, D).double(), 1.0)
    table = torch.arange(n // 16, dtype=torch.int32)[None].cuda()
    out = ops.paged_attention(
        q.cuda(), k.cuda(), v.cuda(), table,
        torch.tensor([n], dtype=torch.int32).cuda(),
        torch.tensor([0, rows], dtype=torch.int32).cuda(), 1.0, rows)
    err = (out.view(ref.shape).cpu().double() / ref - 1).abs().max()
    # half a step of the 8 bits of a bf16; rounded weights add as much again
    assert err < 2 ** -8 * 1.01, err

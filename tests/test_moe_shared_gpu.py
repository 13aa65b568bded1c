"""A shared expert's products in the launches of the routed ones', against the
formula in 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,topk,H,I,S", [
    (1, 8, 2, 64, 64, 64),          # one row: most dies have no tile
    (3, 8, 2, 128, 64, 128),
    (33, 8, 2, 192, 192, 320),      # blocks of 32, one row beside them
    (48, 8, 2, 128, 320, 64),       # 12 rows an expert: 32
    (49, 8, 2, 2048, 192, 384),     # just over: 64
    (161, 8, 2, 320, 128, 256),     # 128
    (256, 4, 2, 256, 64, 64),
    (130, 64, 6, 128, 64, 128),
    (260, 2, 1, 128, 64, 64),       # 256: a block of rows and four rows
    (700, 4, 2, 128, 64, 192),      # a second product of thrice the K
    (513, 2, 2, 320, 448, 1088),    # columns that end inside a tile
    (2100, 8, 2, 1024, 512, 1024)])  # several tiles a workgroup
def test_moe_shared(T, E, topk, H, I, S):
    from gllm_amd import ops
    gen = torch.Generator().manual_seed(T + S)

    def rand(*shape):
        return (torch.randn(*shape, generator=gen)
                * shape[-1] ** -0.5).bfloat16()

    x = torch.randn(T, H, generator=gen).bfloat16()
    res = torch.randn(T, H, generator=gen).bfloat16()
    w13, w2, up, down = (rand(E, 2 * I, H), rand(E, H, I), rand(2 * S, H),
                         rand(H, S))
    ids = torch.stack([torch.randperm(E, generator=gen)[:topk]
                       for _ in range(T)]).int()
    ids[T // 2, 0] = -1             # a padding pair contributes nothing
    weights = torch.rand(T, topk, generator=gen) + 0.1
    norm_w = torch.rand(H, generator=gen) + 0.5
    dev = [t.cuda() for t in (x, w13, w2, weights, ids, up, down)]
    got_res = res.cuda()
    out = ops.fused_moe(*dev[:5], num_global_experts=E, add_norm=(
        None, got_res, norm_w.cuda(), 1e-6), shared_mlp=tuple(dev[5:]))

    def gated(v, a, b):
        g, u = (v @ a.double().t()).chunk(2, -1)
        h = torch.nn.functional.silu(g) * u
        return h @ b.double().t()

    xd = x.double()
    want = res.double() + gated(xd, up, down)
    for e in range(E):
        row, col = (ids == e).nonzero(as_tuple=True)
        if len(row):
            want.index_add_(0, row, gated(xd[row], w13[e], w2[e]) *
                            weights[row, col].double()[:, None])
    # each term is rounded to bf16 once inside and once as it is stored, and
    # the stored sum once more: some 2^-8 of the terms' sizes, which are at
    # most a few times the row's
    err = (got_res.cpu().double() - want).abs().max()
    assert err <= 4 * 2 ** -8 * want.abs().max()
    n = got_res.cpu().double()
    n = n * torch.rsqrt(n.square().mean(-1, keepdim=True) + 1e-6)
    n = n * norm_w.double()
    assert ((out.cpu().double() - n).abs() <= 2 ** -8 * n.abs() + 1e-5).all()

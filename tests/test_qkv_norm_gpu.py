"""Norm per head, rotation and cache rows of a merged q | k | v projection in one
kernel, against the formula in 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,Hq,Hkv,D,rot", [
    (1, 1, 1, 128, 32), (5, 16, 2, 128, 128), (130, 13, 2, 128, 32),
    (33, 4, 4, 64, 64), (7, 3, 1, 40, 32), (9, 2, 1, 16, 16)])
@pytest.mark.parametrize("wdtype", [torch.bfloat16, torch.float32])
def test_qkv_norm(T, Hq, Hkv, D, rot, wdtype):
    from gllm_amd import ops
    torch.manual_seed(T + D)
    H = Hq + 2 * Hkv
    src = torch.randn(T, H * D + 8).bfloat16().cuda()[:, :H * D]
    qw, kw = ((torch.rand(D) + 0.5).to(wdtype).cuda() for _ in range(2))
    pos = torch.randint(0, 300, (T,)).cuda()
    ang = torch.arange(300).double()[:, None] * 1e4 ** (
        -torch.arange(0, rot, 2).double() / rot)
    cs = torch.cat([ang.cos(), ang.sin()], -1).float().cuda()
    kc, vc = (torch.zeros(T // 16 + 2, 16, Hkv, D).bfloat16().cuda()
              for _ in range(2))
    slots = torch.randperm(kc.shape[0] * 16)[:T].cuda()
    assert ops.qkv_rope_cache_ok(kc, vc, cs, True)
    assert ops.qkv_norm_rope_cache_ok(src, qw, kw, kc, cs)
    q = ops.qkv_norm_rope_cache(src, qw, kw, 1e-6, pos, cs, kc, vc, slots, Hq)
    x = src.double().view(T, H, D)

    def want(x, w):
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6)
        x = (x * w.double()).bfloat16().double()
        c, s = cs[pos].double()[:, None].chunk(2, -1)
        a, b = x[..., :rot // 2], x[..., rot // 2:rot]
        return torch.cat([a * c - b * s, b * c + a * s, x[..., rot:]], -1)
    # the norm is rounded to bf16, now and then to its other neighbour, and the
    # result once more: 2^-8 each of the larger of a pair
    for got, ref in ((q.view(T, Hq, D), want(x[:, :Hq], qw)),
                     (kc.view(-1, Hkv, D)[slots],
                      want(x[:, Hq:Hq + Hkv], kw))):
        assert (got.double() - ref).abs().max() <= 2 ** -7 * ref.abs().max()
        assert (got.double() - ref).norm() <= 2 ** -8 * ref.norm()
    assert torch.equal(vc.view(-1, Hkv, D)[slots].double(), x[:, Hq + Hkv:])
    free = torch.ones(kc.shape[0] * 16, dtype=torch.bool, device="cuda")
    free[slots] = False
    assert not kc.view(-1, Hkv, D)[free].any()
    assert not vc.view(-1, Hkv, D)[free].any()

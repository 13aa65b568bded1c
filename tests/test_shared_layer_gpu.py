"""A layer's routed and shared experts with the sum and norm behind them: the
route that runs the shared products beside the routed ones against the layer's
own parts one after the other."""

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu


def layer(H, I, E, topk, n_shared):
    from gllm_amd.models.deepseek_v2 import DeepseekMoE
    cfg = SimpleNamespace(
        hidden_size=H, moe_intermediate_size=I, n_routed_experts=E,
        num_experts_per_tok=topk, n_shared_experts=n_shared)
    moe = DeepseekMoE(cfg, SimpleNamespace(use_ep=False),
                      dtype=torch.bfloat16).cuda()
    gen = torch.Generator(device="cuda").manual_seed(H + I)
    for p in moe.parameters():
        p.data.normal_(0, p.shape[-1] ** -0.5, generator=gen)
    return moe


@pytest.mark.parametrize("T,beside", [
    (5, True), (64, True), (160, True),
    (161, False), (256, False),    # blocks of 128 rows, a wider one beside
    (257, True), (500, True),
    (700, False),                  # of 256 rows, too few of them
    (1536, True), (1700, True),    # of 256
    (2101, False)])                # a round more
def test_layer(T, beside, monkeypatch):
    from gllm_amd import ops
    from gllm_amd.layers.layernorm import RMSNorm
    H = 2048
    moe = layer(H, 1024, 8, 2, 2)
    gen = torch.Generator(device="cuda").manual_seed(T)

    def rand():
        return torch.randn(T, H, device="cuda", generator=gen).bfloat16()

    x, res = rand(), rand()
    norm = RMSNorm(H).cuda()
    norm.weight.data.uniform_(0.5, 1.5, generator=gen)
    took = []
    rule = ops.moe_shared_beside
    monkeypatch.setattr(ops, "moe_shared_beside",
                        lambda *a: took.append(rule(*a)) or took[-1])
    got, got_res = moe.forward_add_norm(x, res.clone(), norm)
    assert took == [beside]
    want = (moe(x).double() + res.double())
    # the shared and the routed part are rounded once each here, the stored
    # sum once on both sides
    size = want.abs().max()
    assert (got_res.double() - want).abs().max() <= 2 ** -7 * size
    assert (got_res.double() - want).norm() <= 2 ** -8 * want.norm()
    n = got_res.double()
    n = n * torch.rsqrt(n.square().mean(-1, keepdim=True) + norm.eps)
    n = n * norm.weight.double()
    assert ((got.double() - n).abs() <= 2 ** -8 * n.abs() + 1e-5).all()
    # the same with the shared part by itself: up to 256 rows the same bits
    weights, ids = moe._route(moe.gate(x))
    apart, apart_res = moe.experts.routed_add_norm(
        x, weights, ids, moe.shared_experts(x), res.clone(), norm)
    assert took == [beside]
    if T <= 256 or not beside:
        assert torch.equal(got, apart) and torch.equal(got_res, apart_res)

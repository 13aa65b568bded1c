"""The kernel behind the experts gives the numbers of the three that it
stands for."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,topk,start,E", [
    (1, 8, 1, 0, 4), (3, 2048, 6, 0, 64), (130, 2056, 8, 0, 16),
    (5, 4096, 2, 0, 8), (7, 4104, 9, 8, 8),   # a rank's share of experts
    (2, 8192, 5, 0, 16)])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("wide", [False, True])
def test_same_numbers(T, H, topk, start, E, shared, wide):
    from gllm_amd import ops
    torch.manual_seed(T + H)
    dev, k = "cuda", ops._gpu_kernels()
    pairs = torch.randn(T * topk, H, device=dev).bfloat16()
    ids = torch.randint(-1, start + E + 1, (T, topk), device=dev).int()
    # rows of experts elsewhere were never written
    out_of = (ids.view(-1) < start) | (ids.view(-1) >= start + E)
    pairs[out_of] = float("nan")
    sh = torch.randn(T, H, device=dev).bfloat16() if shared else None
    res = torch.randn(T, H, device=dev).bfloat16()
    w = torch.rand(H, device=dev) + 0.5
    w = w if wide else w.bfloat16()
    ref = torch.empty(T, H, dtype=torch.bfloat16, device=dev)
    k.moe_sum(ref, pairs, ids, start, E, topk)
    if shared:
        ref = ref + sh
    ref, ref_res = ops.fused_add_rmsnorm(ref, res.clone(), w, 1e-6)
    got_res = res.clone()
    out = k.moe_sum_norm(pairs, ids, start, E, topk, sh, got_res, w, 1e-6)
    assert torch.equal(got_res, ref_res) and torch.equal(out, ref)

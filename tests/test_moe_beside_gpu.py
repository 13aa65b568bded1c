"""Shared experts beside the routed ones: the same bits as apart."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def operands(T, E, topk, H, I, S):
    gen = torch.Generator().manual_seed(T + S)

    def rand(*shape):
        return (torch.randn(*shape, generator=gen)
                * shape[-1] ** -0.5).bfloat16().cuda()

    x, res = rand(T, H) * H ** 0.5, rand(T, H) * H ** 0.5
    ids = torch.rand(T, E, generator=gen).topk(topk).indices.int().cuda()
    weights = (torch.rand(T, topk, generator=gen) + 0.1).cuda()
    norm_w = (torch.rand(H, generator=gen) + 0.5).cuda()
    return (x, rand(E, 2 * I, H), rand(E, H, I), weights, ids, rand(2 * S, H),
            rand(H, S), res, norm_w)


# Up to 256 rows the products apart have fp32 sums over shares of K that are
# added in the order of K, from one share (K of 256) to 11 (K of 2816).
@pytest.mark.parametrize("T,E,topk,H,I,S", [
    (1, 8, 2, 512, 1408, 2816),
    (16, 8, 2, 512, 128, 256),
    (17, 8, 2, 1024, 512, 1024),
    (33, 16, 4, 512, 704, 1088),     # 17 stages: the last share is shorter
    (64, 8, 2, 2048, 512, 960),
    (65, 8, 2, 2048, 512, 960),
    (128, 64, 6, 2048, 1408, 2816),
    (129, 8, 2, 768, 1088, 2112),
    (256, 16, 2, 2048, 768, 1536),
    (256, 32, 8, 4096, 512, 512)])    # blocks of 128 rows
def test_beside_is_apart(T, E, topk, H, I, S):
    from gllm_amd import ops
    x, w13, w2, weights, ids, up, down, res, norm_w = operands(
        T, E, topk, H, I, S)
    assert ops.moe_shared_beside(x, w13, w2, topk, up, down)
    got_res, want_res = res.clone(), res.clone()
    got = ops.fused_moe(x, w13, w2, weights, ids, add_norm=(
        None, got_res, norm_w, 1e-6), shared_mlp=(up, down))
    shared = ops.linear(ops.linear_silu(x, up), down)
    want = ops.fused_moe(x, w13, w2, weights, ids, add_norm=(
        shared, want_res, norm_w, 1e-6))
    assert torch.equal(got_res, want_res)
    assert torch.equal(got, want)


def test_where_there_are_no_wide_tiles():
    """Widths that 64 does not divide: the shared expert's products apart."""
    from gllm_amd import ops
    x, w13, w2, weights, ids, up, down, res, norm_w = operands(
        40, 8, 2, 72, 64, 128)
    assert not ops.moe_shared_beside(x, w13, w2, 2, up, down)
    got_res, want_res = res.clone(), res.clone()
    got = ops.fused_moe(x, w13, w2, weights, ids, add_norm=(
        None, got_res, norm_w, 1e-6), shared_mlp=(up, down))
    want = ops.fused_moe(x, w13, w2, weights, ids, add_norm=(
        ops.linear(ops.linear_silu(x, up), down), want_res, norm_w, 1e-6))
    assert torch.equal(got_res, want_res)
    assert torch.equal(got, want)


@pytest.mark.parametrize("block_m", [16, 48, 512])
def test_tables_of_another_block_are_refused(block_m):
    """(on the host, ahead of any launch)"""
    from gllm_amd import ops
    x, w13, w2, weights, ids, up, down, res, norm_w = operands(
        40, 8, 2, 128, 64, 128)
    tables = [torch.zeros(n, dtype=torch.int32, device="cuda")
              for n in (80 + 8 * block_m, 80 + 8, 1)]
    act = x.new_empty(80 + 8 * block_m, 64)
    with pytest.raises(RuntimeError, match="block_m"):
        ops._gpu_kernels().moe_gemm_tiled_shared(
            act, x, w13, *tables, None, 80, 2, block_m, 1, x, up)

"""Few-row products at the tiles and splits that the size of the weight picks:
a last tile that is not full, a last part that is shorter, rows at both ends of
a tile."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(M, N, K):
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    return x, w, x.double() @ w.double().t()


def _close(got, want):
    # one bf16 rounding of the result
    err = (got.double() - want).norm() / want.norm()
    assert err < 2 ** -8, err
    assert not torch.isnan(got).any()


@pytest.mark.parametrize("M,N,K", [
    (1, 4104, 1536), (16, 1000, 6528), (9, 4096, 4096), (16, 22784, 2048),
    (32, 5128, 4160), (17, 18952, 1152),
    (64, 5128, 4160), (33, 18952, 1152),
    (128, 5128, 4160), (65, 1032, 1088),
    (33, 4104, 4096), (24, 12296, 1024), (100, 2048, 2112), (72, 5128, 640),
    (160, 2056, 1088), (256, 2568, 704), (129, 4104, 2048),
    (129, 1032, 1088), (256, 4104, 3136), (200, 5128, 10304)])
def test_plain(M, N, K):
    from gllm_amd import ops
    x, w, ref = _operands(M, N, K)
    k = ops._gpu_kernels()
    _close(k.stream_gemm(x, w, None), ref)
    if N > 8192:
        return
    res = torch.randn(M, N, device="cuda").bfloat16()
    want = res.double() + ref
    k.stream_add_norm(x, w, res, torch.ones(N, device="cuda").bfloat16(), 1e-6)
    _close(res, want)


@pytest.mark.parametrize("M,N,K", [
    (1, 22016, 128), (16, 48000, 64), (11, 55312, 192), (16, 28672, 64),
    (32, 22032, 192), (17, 36016, 128), (64, 22032, 192), (33, 28688, 64),
    (128, 22032, 192), (65, 8208, 128)])
def test_gated(M, N, K):
    from gllm_amd import ops
    x, w, ref = _operands(M, N, K)
    g, u = ref.chunk(2, dim=-1)
    _close(ops._gpu_kernels().stream_gemm_gated(x, w),
           torch.nn.functional.silu(g) * u)

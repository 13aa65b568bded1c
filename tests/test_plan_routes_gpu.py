"""Few-row products at the sizes where the choice between one launch and split
parts turns, and where the number of parts does: the result against fp64, and
which of the two it was by the memory that it took."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(M, N, K):
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    return x, w


def _close(got, x, w):
    # (in pieces: fp64 weights are four times the size); one bf16 rounding of
    # the result
    for n in range(0, w.shape[0], 4096):
        want = x.double() @ w[n:n + 4096].double().t()
        err = (got[:, n:n + 4096].double() - want).norm() / want.norm()
        assert err < 2 ** -8, err


def _behind(call):
    """What a call allocates beside its result, in bytes."""
    call()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = call()
    torch.cuda.synchronize()
    return out, torch.cuda.max_memory_allocated() - before - out.nbytes


@pytest.mark.parametrize("M,N,K,whole", [
    (64, 12288, 2048, True), (33, 12296, 4096, True), (16, 16384, 1024, True),
    (1, 10248, 1024, True), (17, 20480, 1024, True), (64, 16384, 4096, True),
    (128, 14336, 1536, True), (96, 7176, 3072, True), (128, 8192, 512, True),
    (16, 38016, 1024, True), (48, 38024, 1024, True), (1, 28672, 4096, True),
    (64, 5120, 2048, False), (17, 16384, 12288, False),
    (192, 8192, 8192, False), (256, 7168, 11008, False),
    (64, 12288, 14336, False), (1, 4608, 8192, False)])
def test_one_launch_or_parts(M, N, K, whole):
    from gllm_amd import ops
    x, w = _operands(M, N, K)
    got, more = _behind(lambda: ops._gpu_kernels().stream_gemm(x, w, None))
    _close(got, x, w)
    # (two parts and more are fp32, four results' bytes; what else there is is
    # the allocator's rounding)
    assert (more < 4 * got.nbytes) == whole


@pytest.mark.parametrize("M,N,K,parts", [
    # a workgroup a CU: 256 / tiles of 128 columns
    (1, 5120, 5120, 6), (16, 4608, 3584, 7), (16, 3328, 5120, 9),
    (1, 4096, 4096, 8), (16, 3584, 8192, 9),
    # ... but no shares of 4 KB
    (64, 8192, 8192, 3), (32, 7168, 8192, 3), (1, 4096, 16384, 7),
    # ... and the columns that leave enough of them
    (32, 768, 27648, 16), (1, 512, 14336, 16)])
def test_parts(M, N, K, parts):
    from gllm_amd import ops
    x, w = _operands(M, N, K)
    got = ops._gpu_kernels().stream_parts(x, w)
    assert got.shape == (parts, M, N)
    _close(got.sum(0), x, w)


@pytest.mark.parametrize("M,N,K", [
    (64, 16384, 192), (128, 16384, 128), (128, 16400, 128), (33, 28672, 2048),
    (33, 28672, 192), (1, 24576, 2048), (16, 49152, 2048), (16, 49168, 128),
    (32, 33024, 128), (17, 36000, 128), (16, 36000, 128)])
def test_gated(M, N, K):
    from gllm_amd import ops
    x, w = _operands(M, N, K)
    g, u = (x.double() @ w.double().t()).chunk(2, dim=-1)
    want = torch.nn.functional.silu(g) * u
    got = ops._gpu_kernels().stream_gemm_gated(x, w)
    # one bf16 rounding of the result
    assert (got.double() - want).norm() < 2 ** -8 * want.norm()

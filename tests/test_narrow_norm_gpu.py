"""Sums of parts and their norm for rows of fewer columns than a workgroup
has threads for."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [8, 512, 1016, 1024, 2040, 2048, 2056])
@pytest.mark.parametrize("S", [1, 2, 9, 16])
def test_norm_of_narrow_rows(N, S):
    from gllm_amd import ops
    torch.manual_seed(N + S)
    part = torch.randn(S, 5, N, device="cuda")
    res = torch.randn(5, N, device="cuda").bfloat16()
    w = torch.rand(N, device="cuda") + 0.5
    want = res.double() + part.double().sum(0)
    got = ops._gpu_kernels().parts_add_norm(part, res, w, 1e-6, False)
    # the sum is rounded to bf16 once, and so is the norm of what was stored
    assert (res.double() - want).norm() < 2 ** -8 * want.norm()
    r = res.double()
    norm = r * (r.square().mean(1, keepdim=True) + 1e-6).rsqrt() * w.double()
    assert (got.double() - norm).norm() < 2 ** -8 * norm.norm()

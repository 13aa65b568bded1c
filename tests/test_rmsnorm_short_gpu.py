"""Norms of short rows (heads) at the edges of their lane groups."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,hidden", [
    (1, 8), (15, 64), (16, 128), (17, 128), (9, 136), (8, 256), (33, 264),
    (5, 512), (4, 520), (70000, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("wide", [False, True])
def test_rows(rows, hidden, dtype, wide):
    from gllm_amd import ops
    torch.manual_seed(rows + hidden)
    x = (torch.randn(rows, hidden, device="cuda") * 3).to(dtype)
    w = torch.rand(hidden, device="cuda") + 0.5
    w = w if wide else w.to(dtype)
    out = ops.rmsnorm(x, w, 1e-6)
    y = x.double()
    y = y * (y.square().mean(-1, keepdim=True) + 1e-6).rsqrt() * w.double()
    # one rounding to the type, fp32 before it
    eps = 2 ** -8 if dtype == torch.bfloat16 else 2 ** -11
    assert ((out.double() - y).abs() <= y.abs() * eps * 1.01 + 1e-6).all()
    if rows > 2:  # a row's infinities and NaN stay in it
        x[1, 0], x[2, 3] = float("inf"), float("nan")
        bad = ops.rmsnorm(x, w, 1e-6)
        keep = torch.ones(rows, dtype=torch.bool)
        keep[1] = keep[2] = False
        assert torch.equal(bad[keep], out[keep])
        assert bad[2].isnan().all()

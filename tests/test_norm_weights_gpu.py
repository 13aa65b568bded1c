"""RMS norms with the weight in its own type: fp32 parameters beside 16-bit
rows."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden", [8, 128, 2056, 5120])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("wide", [False, True])
def test_weight_types(hidden, dtype, wide):
    from gllm_amd import ops
    torch.manual_seed(hidden)
    x, res = [torch.randn(3, hidden, device="cuda").to(dtype)
              for _ in range(2)]
    w = (torch.rand(hidden, device="cuda") + 0.5)
    w = w if wide else w.to(dtype)

    def norm(t):
        t = t.double()
        return t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + 1e-6) \
            * w.double()

    # half a step of the result's type, and the sums in 32 bits
    eps = 2 ** -8 if dtype == torch.bfloat16 else 2 ** -11
    ref = norm(x)
    out = ops.rmsnorm(x, w, 1e-6).double()
    assert ((out - ref).abs() <= (eps + 1e-5) * ref.abs() + 1e-6).all()
    s = (x.float() + res.float()).to(dtype)
    out, stored = ops.fused_add_rmsnorm(x.clone(), res.clone(), w, 1e-6)
    assert torch.equal(stored, s)
    ref = norm(s)
    assert ((out.double() - ref).abs()
            <= (eps + 1e-5) * ref.abs() + 1e-6).all()


def test_a_third_type():
    from gllm_amd import ops
    x = torch.randn(2, 64, dtype=torch.bfloat16, device="cuda")
    w = torch.rand(64, device="cuda").half()
    assert torch.equal(ops.rmsnorm(x, w, 1e-6),
                       ops.rmsnorm(x, w.float(), 1e-6))

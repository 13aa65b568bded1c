"""Softmax and top-k of rows of few experts (one per lane) and of more."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,k", [(64, 6), (64, 64), (65, 6), (130, 64), (512, 8), (8, 2), (1, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_of_few_experts(E, k, dtype):
    from gllm_amd import ops
    torch.manual_seed(E + k)
    logits = torch.randn(50, E, device="cuda").to(dtype)
    logits[3] = 0.5                                 # equal ones
    logits[4, 1::2] = float("-inf")
    got, ids = ops.topk_softmax(logits, k, False)
    p = logits.double().softmax(-1)
    # (equal probabilities: the lower index first)
    want = torch.sort(p.float(), dim=1, descending=True, stable=True)
    if dtype == torch.float32 and k < 64:
        assert torch.equal(ids[3].long(), torch.arange(k, device="cuda"))
    assert ((got.double() - want.values[:, :k].double()).abs() <=
            1e-6 + 1e-5 * got.abs()).all()

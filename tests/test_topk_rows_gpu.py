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
    assert torch.equal(ids[3].long(), torch.arange(k, device="cuda"))
    assert (ids.sort(1).values.diff(dim=1) > 0).all()
    # a weight is that of its expert
    of_ids = p.gather(1, ids.long())
    assert ((got.double() - of_ids).abs() <= 1e-6 + 1e-5 * got.abs()).all()
    assert ((got.double() - want.values[:, :k].double()).abs() <=
            1e-6 + 1e-5 * got.abs()).all()


def _ties(E):
    """Rows whose largest values are equal in several blocks of 64."""
    torch.manual_seed(E)
    x = torch.randn(40, E, device="cuda").clamp(-2, 2).double()
    for r in range(40):
        x[r, torch.randperm(E, device="cuda")[:1 + r % 9]] = 3.0
    x[0, [e for e in (3, 67, 131) if e < E]] = 3.0
    return x.float()


@pytest.mark.parametrize("E,k", [(64, 6), (130, 8), (256, 8), (512, 12)])
def test_equal_ones_in_order(E, k):
    from gllm_amd import ops
    x = _ties(E)
    want = torch.sort(x, dim=1, descending=True, stable=True).indices[:, :k]
    assert torch.equal(ops.topk_softmax(x, k)[1].long(), want)
    assert torch.equal(ops.topk_then_softmax(x, k)[1].long(), want)
    assert torch.equal(ops.sigmoid_group_topk(x, None, k)[1].long(), want)

"""Greedy choice: the first of equals, NaN as the largest."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [1, 7, 64, 8191, 8192, 32776, 152064, 32001])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_matches_argmax(V, dtype):
    from gllm_amd import ops
    torch.manual_seed(V)
    x = torch.randn(6, V).to(dtype)      # (bf16: many equal values)
    x[1] = 0.
    x[1, V // 2:] = -0.                  # zeros of both signs are equal
    x[2] = float("-inf")
    x[3, V // 3] = x[3, V - 1] = float("inf")
    x[4, V - 1] = float("nan")
    x[5] = -x[5].abs() - 1
    # first index of the row's largest, a NaN above everything
    want = []
    for row in x.double():
        nan = row.isnan().nonzero()
        want.append(int(nan[0]) if len(nan)
                    else int((row == row.max()).nonzero()[0]))
    for rows in (x, x[:1], x[4:]):
        at = {6: 0, 1: 0, 2: 4}[rows.shape[0]]
        got = ops.greedy_argmax(rows.cuda()).tolist()
        assert got == want[at:at + rows.shape[0]]
    assert ops.greedy_argmax(x[:0].cuda()).shape == (0,)

"""The short convolution's ways of dealing rows to threads, at their borders."""

import pytest
import torch
from test_short_conv_gpu import oracle

pytestmark = pytest.mark.gpu


# Eight tokens a thread from 2^20 vectors of 8 channels on, else 4 or taps - 1;
# fp32 with 6 taps one below 160 rows, with more below 384.
@pytest.mark.parametrize("C,lens", [
    (2048, [0, 8, 2049, 0, 1, 7, 2024, 9, 0]),   # 2^20 and a little more
    (2048, [2040, 2055]),                        # just below
    (64, [0, 5, 6, 7, 0, 12, 14, 13, 80, 1, 20, 1]),    # 159 rows
    (64, [0, 5, 6, 7, 0, 12, 14, 13, 80, 1, 20, 2]),    # 160
    (64, [0, 383]), (64, [380, 0, 4]), (64, [0, 11, 1, 0])])
@pytest.mark.parametrize("taps", [1, 3, 4, 6, 7, 8])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_forms(C, lens, taps, dtype):
    from gllm_amd import ops
    T, B = sum(lens), len(lens)
    torch.manual_seed(T + taps)
    x, w = torch.randn(T, C).to(dtype), (torch.randn(C, taps) * 0.5).to(dtype)
    state = torch.randn(B + 1, C, max(taps - 1, 1)).to(dtype)
    slots, init = torch.randperm(B + 1)[:B], [i % 3 % 2 for i in range(B)]
    got_state = state.cuda()
    got = ops.causal_conv_silu(
        x.cuda(), w.cuda(), got_state, slots.cuda(),
        torch.tensor(init).int().cuda(),
        torch.tensor([0] + lens).cumsum(0).int().cuda(),
        max_query_len=max(lens)).cpu().double()
    want_state = state.clone()
    want = oracle(x, w, want_state, slots.tolist(), init, lens, None)
    # (the bounds of test_short_conv)
    step = 2 ** -8 if dtype == torch.bfloat16 else 2 ** -23
    assert ((got - want).abs() <= want.abs() * (step + 2 ** -20) + 2e-5).all()
    assert torch.equal(got_state.cpu(), want_state)

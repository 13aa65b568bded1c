"""The ragged short convolution, which rolls the state that it reads, against
sums in 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def oracle(x, w, state, slots, init, lens, bias):
    """fp64 on the CPU; ``state`` (of the inputs' type) rolls in place."""
    taps, out, t = w.shape[1], [], 0
    for slot, has, n in zip(slots, init, lens):
        past = state[slot] if has else torch.zeros_like(state[slot])
        past = past[:, :taps - 1].t()
        line = torch.cat([past, x[t:t + n]])
        y = sum(line[i:i + n].double() * w[:, i].double()
                for i in range(taps))
        if bias is not None:
            y = y + bias.double()
        out.append(y / (1 + torch.exp(-y)))
        if taps > 1:
            state[slot] = line[n:].t()
        t += n
    return torch.cat(out)


@pytest.mark.parametrize("lens,init", [
    ([1], [1]), ([3, 0, 0, 1, 2], [1, 1, 0, 1, 0]),
    ([0, 4, 5, 7, 8, 9, 1, 1, 16, 0], [1, 0] * 5),
    ([31] * 33, [1, 0, 1] * 11),
    ([2050, 1, 2049, 6, 13], [0, 1, 1, 0, 1])])   # eight rows a thread
@pytest.mark.parametrize("taps", [1, 2, 4, 5, 6, 8])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_short_conv(lens, init, taps, dtype):
    from gllm_amd import ops
    C, T, B = 2048 if sum(lens) > 4000 else 72, sum(lens), len(lens)
    torch.manual_seed(T + taps)
    wide = torch.randn(T, C + 8).to(dtype)
    x, w = wide[:, :C], (torch.randn(C, taps) * 0.5).to(dtype)
    bias = torch.randn(C).to(dtype) if taps % 2 else None
    state = torch.randn(B + 2, C, max(taps - 1, 1)).to(dtype)
    slots = (torch.randperm(B + 1) + 1)[:B]
    qsl = torch.tensor([0] + lens).cumsum(0).int()
    got_state = state.cuda()
    got = ops.causal_conv_silu(
        wide.cuda()[:, :C], w.cuda(), got_state, slots.cuda(),
        torch.tensor(init).int().cuda(), qsl.cuda(),
        max_query_len=max(lens),
        bias=None if bias is None else bias.cuda()).cpu().double()
    want_state = state.clone()
    want = oracle(x, w, want_state, slots.tolist(), init, lens, bias)
    # the result is rounded once; taps + 1 terms of at most ~10 are summed in
    # 32 bits and the silu has a relative error of some 2^-22
    step = 2 ** -8 if dtype == torch.bfloat16 else 2 ** -23
    assert ((got - want).abs() <= want.abs() * (step + 2 ** -20) + 2e-5).all()
    assert torch.equal(got_state.cpu(), want_state)

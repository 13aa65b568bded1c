"""The chunked gated-delta recurrence over ragged batches in an order of its
own: the longest sequence first, its operands in blocks of 16 rows."""

import pytest
import torch
from test_gdn_rows_gpu import D, SCALE, oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [
    [0, 31, 0, 0, 130, 1, 0],             # empty sequences between others
    [64, 64, 16, 128, 16],                # equal lengths, whole blocks
    [257],                                # one: half a batch has no partner
    [5, 90, 33, 70, 2, 150, 15],          # odd count, two a CU
    list(range(1, 72)),                   # a rank per sequence beyond a wave
    [1] * 515 + [66] + [3] * 20])         # ... and beyond a workgroup
@pytest.mark.parametrize("Hk,Hv", [(1, 1), (2, 4)])
def test_gdn_order(lens, Hk, Hv):
    from gllm_amd import ops
    torch.manual_seed(sum(lens) + Hv)
    T, B, C = sum(lens), len(lens), (2 * Hk + Hv) * D
    bf = dict(dtype=torch.bfloat16, device="cuda")
    conv, ba = torch.randn(T, C, **bf), torch.randn(T, 2 * Hv, **bf)
    A_log = torch.randn(Hv, device="cuda") * 0.5
    dt = torch.randn(Hv, device="cuda") * 0.5
    state = torch.randn(B, Hv, D, D, device="cuda") * 0.3
    init = [i % 2 for i in range(B)]
    slots = torch.randperm(B)
    qsl = torch.tensor([0] + lens).cumsum(0).int().cuda()
    s = state.clone()
    o = ops._gpu_kernels().gdn_varlen(
        conv, ba, A_log, dt, s, slots.cuda(), torch.tensor(init).int().cuda(),
        qsl, Hk, max(lens), SCALE).cpu().double().view(T, -1)
    # the oracle ends in a norm and a gate: undone by heads of their own rms
    want = state.cpu().double()
    one = torch.zeros(T, Hv * D, dtype=torch.float64)
    gated, _ = oracle(conv.cpu(), ba.cpu(), one + 1, A_log.cpu(), dt.cpu(),
                      torch.ones(D), want, slots.tolist(), init, lens, Hk, Hv)
    empty = [i for i, n in enumerate(lens) if not n]
    want[slots[empty]] = state.cpu().double()[slots[empty]]
    n = o.view(T, Hv, D)
    n = n * torch.rsqrt(n.pow(2).mean(-1, keepdim=True) + 1e-6)
    n = n.view(T, -1) * torch.nn.functional.silu(one + 1)
    # o is rounded to bf16 (half a step: 2^-9 to 2^-8 of a value), its head's
    # rms moves by less; sums of 32 bits stay within 1e-3 of that rms
    assert ((n - gated).abs() <= 2 ** -7 * gated.abs() + 1e-3).all()
    err = (s.cpu().double() - want).abs().max()
    assert err <= 1e-5 * want.abs().max().clamp(min=1)

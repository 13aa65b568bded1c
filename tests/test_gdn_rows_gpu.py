"""The gated-delta layer between its projections over a ragged batch
(``ops.gdn_rows``), against the recurrence token by token in 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
D, EPS, SCALE = 128, 1e-6, 128 ** -0.5


def oracle(conv, ba, z, A_log, dt, norm_w, state, slots, init, lens, Hk, Hv):
    """fp64 on the CPU from the convolved rows."""
    G = Hv // Hk
    conv, ba, z = conv.double(), ba.double(), z.double()
    q, k, v = conv.split([Hk * D, Hk * D, Hv * D], -1)

    def unit(x):
        x = x.view(-1, Hk, D)
        x = x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)
        return x.repeat_interleave(G, 1)

    q, k, v = unit(q) * SCALE, unit(k), v.view(-1, Hv, D)
    beta = torch.sigmoid(ba[:, :Hv])
    g = -A_log.double().exp() * torch.nn.functional.softplus(
        ba[:, Hv:] + dt.double())
    out, t = torch.zeros_like(v), 0
    for slot, has, n in zip(slots, init, lens):
        S = state[slot].double() if has else torch.zeros(
            Hv, D, D, dtype=torch.float64)
        for _ in range(n):
            S = S * g[t].exp()[:, None, None]
            u = beta[t][:, None] * (v[t] - (S * k[t][:, None, :]).sum(-1))
            S = S + u[:, :, None] * k[t][:, None, :]
            out[t] = (S * q[t][:, None, :]).sum(-1)
            t += 1
        state[slot] = S
    n = out * torch.rsqrt(out.pow(2).mean(-1, keepdim=True) + EPS)
    gate = (norm_w.double() * torch.nn.functional.silu(z.view_as(n)))
    return (n * gate).reshape(t, -1), gate.reshape(t, -1)


@pytest.mark.parametrize("lens,init", [
    ([1], [0]), ([1, 1, 1], [1, 1, 1]), ([1, 1], [1, 0]),
    ([63, 1, 64, 65, 2, 193], [0, 1, 1, 0, 0, 1]),
    ([15, 16, 17, 32, 33, 48, 49, 80], [1, 0] * 4),  # waves without rows
    ([17] * 40, [1, 0] * 20)])
@pytest.mark.parametrize("Hk,Hv", [(2, 4), (3, 3)])
def test_gdn_rows(lens, init, Hk, Hv):
    from gllm_amd import ops
    torch.manual_seed(sum(lens) + Hk)
    T, B, C = sum(lens), len(lens), (2 * Hk + Hv) * D
    bf = dict(dtype=torch.bfloat16, device="cuda")
    qkvz = torch.randn(T, C + Hv * D, **bf)
    ba = torch.randn(T, 2 * Hv, **bf)
    w = torch.randn(C, 4, **bf) * 0.5
    A_log = torch.randn(Hv, device="cuda") * 0.5
    dt = torch.randn(Hv, device="cuda") * 0.5
    norm_w = torch.rand(D, **bf) + 0.5
    conv_state = torch.randn(B + 2, C, 3, **bf)
    state = torch.randn(B + 2, Hv, D, D, device="cuda") * 0.3
    slots = (torch.randperm(B + 1) + 1).tolist()[:B]
    st, it = torch.tensor(slots).cuda(), torch.tensor(init).int().cuda()
    qsl = torch.tensor([0] + lens).cumsum(0).int().cuda()
    assert ops.gdn_rows_ok(qkvz, ba, w, conv_state, state, norm_w, D, D)
    conv = ops.causal_conv_silu(qkvz[:, :C], w, conv_state.clone(), st, it,
                                qsl, max_query_len=max(lens))
    ref_state = state.cpu().double()
    ref, gate = oracle(conv.cpu(), ba.cpu(), qkvz[:, C:].cpu(), A_log.cpu(),
                       dt.cpu(), norm_w.cpu(), ref_state, slots, init, lens,
                       Hk, Hv)
    carried = max(lens) == 1 and all(init)
    forms = [False, True] if carried else [False]
    for form in forms:
        s = state.clone()
        out = ops.gdn_rows(qkvz, ba, w, A_log, dt, norm_w, EPS,
                           conv_state.clone(), s, st, it, qsl, max(lens),
                           form, Hk, SCALE).cpu().double()
        # o and the result are rounded to bf16 (8 significant bits: half a
        # step is up to 2^-8 of the value, and the norm's mean moves by a
        # fraction of one); the recurrence in 32 bits stays within 1e-3 of
        # a head's rms
        bound = 2.25 * 2 ** -8 * ref.abs() + 1e-3 * gate.abs() + 1e-6
        over = (out - ref).abs() / bound
        assert over.max() <= 1, [(i, float(x)) for i, x in enumerate(
            over.view(T, Hv, D).amax((1, 2))) if x > 1]
        rows = torch.tensor(slots)
        # (three bf16 numbers hold an fp32 one to 2^-24: 32-bit sums)
        err = (s.cpu().double() - ref_state)[rows].abs().max()
        assert err <= 1e-5 * ref_state.abs().max().clamp(min=1)
        rest = torch.tensor([i for i in range(B + 2) if i not in slots])
        assert torch.equal(s.cpu()[rest], state.cpu()[rest])


def test_gdn_rows_refusals():
    """Other head sizes, types and misaligned rows stay off this path."""
    from gllm_amd import ops
    bf = dict(dtype=torch.bfloat16, device="cuda")
    a = (torch.zeros(2, 1024, **bf), torch.zeros(2, 4, **bf),
         torch.zeros(768, 4, **bf), torch.zeros(2, 768, 3, **bf),
         torch.zeros(2, 2, D, D, device="cuda"), torch.zeros(D, **bf))
    assert ops.gdn_rows_ok(*a, 128, 128)
    assert not ops.gdn_rows_ok(*a, 64, 128)
    assert not ops.gdn_rows_ok(a[0].half(), *a[1:], 128, 128)
    assert not ops.gdn_rows_ok(torch.zeros(2, 1028, **bf)[:, 4:], *a[1:],
                               128, 128)

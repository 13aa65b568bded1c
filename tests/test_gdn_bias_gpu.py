"""The gated-delta recurrence with its time bias in 16 bits: the same bits as
with these values in 32."""

import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


@pytest.mark.parametrize("lens,carried", [
    ([70, 1, 16, 130], False), ([1, 1, 1], True)])
@pytest.mark.parametrize("Hk,Hv", [(1, 1), (2, 6)])
def test_bias_of_16_bits(lens, carried, Hk, Hv):
    from gllm_amd import ops
    torch.manual_seed(Hv)
    T, B, C = sum(lens), len(lens), (2 * Hk + Hv) * D
    bf = dict(dtype=torch.bfloat16, device="cuda")
    qkvz, ba = torch.randn(T, C + Hv * D, **bf), torch.randn(T, 2 * Hv, **bf)
    w, norm_w = torch.randn(C, 4, **bf) * 0.5, torch.rand(D, **bf) + 0.5
    A_log = torch.randn(Hv, device="cuda") * 0.5
    dt = torch.randn(Hv, **bf) - 1
    conv_state = torch.randn(B, C, 3, **bf)
    state = torch.randn(B, Hv, D, D, device="cuda") * 0.3
    slots = torch.randperm(B).cuda()
    init = torch.ones(B, dtype=torch.int32, device="cuda")
    qsl = torch.tensor([0] + lens).cumsum(0).int().cuda()

    def run(bias):
        s, c = state.clone(), conv_state.clone()
        return ops.gdn_rows(qkvz, ba, w, A_log, bias, norm_w, 1e-6, c, s,
                            slots, init, qsl, max(lens), carried, Hk,
                            D ** -0.5), s
    (got, got_s), (want, want_s) = run(dt), run(dt.float())
    assert torch.equal(got, want) and torch.equal(got_s, want_s)
    other, _ = run(dt + 1)
    assert not torch.equal(other, want)

"""What the gated-delta recurrence works on is part of a profile run's peak."""

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


def peak(f):
    """What f asks for at its peak, in bytes."""
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_stats()["requested_bytes.all.current"]
    f()
    return torch.cuda.memory_stats()["requested_bytes.all.peak"] - before


@pytest.mark.parametrize("lens", [
    [1] * 500 + [300],      # a block of 16 rows for each
    [700, 33, 1, 90]])
def test_profile_run_covers_a_step(lens):
    from gllm_amd import ops
    from gllm_amd.models.hybrid_gdn import GatedDeltaNet
    from gllm_amd.runtime.forward_context import ForwardContext
    T, B, Hk, Hv = sum(lens), len(lens), 2, 4
    bf = dict(dtype=torch.bfloat16, device="cuda")
    conv = torch.randn(T, (2 * Hk + Hv) * D, **bf)
    ba = torch.randn(T, 2 * Hv, **bf)
    A_log, dt = torch.zeros(2, Hv, device="cuda").unbind()
    state = torch.zeros(B, Hv, D, D, device="cuda")
    slots = torch.arange(B, device="cuda")
    init = torch.ones(B, dtype=torch.int32, device="cuda")
    qsl = torch.tensor([0] + lens).cumsum(0).int().cuda()
    step = peak(lambda: ops._gpu_kernels().gdn_varlen(
        conv, ba, A_log, dt, state, slots, init, qsl, Hk, max(lens), 0.1))
    out = T * Hv * D * 2
    cfg = SimpleNamespace(
        hidden_size=64, linear_num_value_heads=Hv, linear_num_key_heads=Hk,
        linear_key_head_dim=D, linear_value_head_dim=D,
        linear_conv_kernel_dim=4, rms_norm_eps=1e-6)
    layer = GatedDeltaNet(cfg, 0, dtype=torch.bfloat16).cuda()
    none = torch.zeros(1, dtype=torch.int32, device="cuda")
    fctx = ForwardContext(
        num_tokens=8, positions=none, slot_mapping=none, block_table=none,
        seq_lens=none, query_start_loc=none, max_query_len=8, max_seq_len=8,
        k_caches=[], v_caches=[], is_profile_run=True, largest_batch=(T, B))
    hidden = torch.zeros(8, 64, **bf)
    profile = peak(lambda: layer.heads(hidden, fctx))
    assert profile == step - out     # all but the result
    blocks = sum(-(-n // 16) for n in lens)
    assert profile >= blocks * Hv * (3 * 2 * (16 * D + 16 * 64) + 4 * 16 * D)

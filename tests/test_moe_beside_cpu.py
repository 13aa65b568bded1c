"""Sizes of shared experts that may run beside the routed ones."""

import pytest
import torch


@pytest.mark.parametrize("K,width,beside", [
    (8192, 32768, True),
    (8192, 65472, True),      # 2 * width * K just below 2^30
    (8192, 65536, False),     # ... and 2^30: 32-bit offsets would not do
    (512, 524224, True),
    (512, 524288, False)])    # rows of a weight: below 2^20
def test_sizes_that_the_product_takes(monkeypatch, K, width, beside):
    from gllm_amd import ops

    class Host:
        stream_slice = staticmethod(lambda M, N, K: 64)

    monkeypatch.setattr(ops, "_gpu_kernels", lambda: Host)
    assert ops._shared_beside(8, 2, 4, K, width, width) == beside


@pytest.mark.parametrize("activation,shared,add_norm", [
    ("relu2", None, True), ("swiglu_clamp", None, True),
    ("silu_glu", None, False), ("silu_glu", 1, True)])
def test_a_shared_expert_is_not_dropped(activation, shared, add_norm):
    """What the launches beside cannot form is an error, not a result without
    the shared part (or with the wrong one)."""
    from gllm_amd import ops
    x, w = torch.zeros(2, 64), torch.zeros(2, 128, 64)
    norm = (None if shared is None else x, x, x[0], 1e-6)
    with pytest.raises(ValueError, match="shared_mlp"):
        ops.fused_moe(x, w, w[:, :64], torch.ones(2, 1),
                      torch.zeros(2, 1).int(), activation=activation,
                      act_args=(7.0, 1.7), add_norm=norm if add_norm else None,
                      shared_mlp=(w[0], w[0, :64]))

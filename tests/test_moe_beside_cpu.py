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


@pytest.mark.parametrize("sizes,beside", [
    # rows, top, experts, K, inter, width: each line of the rule
    ((256, 6, 64, 2048, 1408, 2816), True),
    ((256, 6, 64, 2048, 1408, 2880), False),    # more than two routed ones
    ((83, 4, 32, 2048, 3136, 3136), True),
    ((83, 4, 32, 2048, 3136, 3200), False),     # a longer chain of K
    ((160, 2, 8, 2048, 1024, 2048), True),
    ((161, 2, 8, 2048, 1024, 2048), False),     # blocks of 128 rows
    ((161, 2, 8, 2048, 1024, 1024), True),
    ((161, 2, 8, 2048, 1088, 1088), False),
    ((64, 6, 64, 2112, 1408, 2816), False),
    ((200, 2, 2, 2048, 1024, 1024), False),     # of 256
    ((257, 6, 64, 2048, 1408, 2816), True),
    ((1024, 6, 64, 2048, 1408, 2816), True),
    ((1025, 6, 64, 2048, 1408, 2816), False),
    ((1000, 6, 64, 2048, 1600, 2816), True),
    ((1000, 6, 64, 2048, 1664, 2816), False),
    ((1000, 6, 64, 2112, 1408, 2816), False),
    ((1000, 6, 64, 2048, 1408, 1984), False),   # less than 2^22 elements
    ((512, 2, 64, 2048, 1408, 2816), True),     # 352 tiles of 64 rows
    ((600, 2, 64, 2048, 1408, 2816), False),    # 440
    ((1535, 6, 32, 2048, 1408, 2816), False),
    ((1536, 6, 32, 2048, 1408, 2816), True),
    ((5120, 2, 4, 2048, 2048, 2048), True),
    ((5121, 2, 4, 2048, 2048, 2048), False),
    ((5120, 6, 32, 2048, 1408, 2816), False),   # no round less
    ((4096, 6, 64, 2048, 1408, 2816), True),
    ((4096, 6, 64, 2048, 1408, 2752), False),   # no multiple
    ((3072, 6, 16, 2048, 2112, 2112), True),
    ((3072, 7, 16, 2048, 2112, 2112), False),   # less than a sixth
    ((1870, 6, 64, 2048, 1408, 2816), False),   # 175 rows an expert
    ((1880, 6, 64, 2048, 1408, 2816), True)])
def test_lines_of_the_rule(monkeypatch, sizes, beside):
    from gllm_amd import ops

    class Host:
        stream_slice = staticmethod(lambda M, N, K: 64)

    monkeypatch.setattr(ops, "_gpu_kernels", lambda: Host)
    monkeypatch.setattr(ops, "_compute_units", lambda: 256)
    assert ops._shared_beside(*sizes) == beside

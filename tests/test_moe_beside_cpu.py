"""Sizes of shared experts that may run beside the routed ones."""

import pytest


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

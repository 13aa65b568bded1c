"""Where products go without a GPU: rows that the tile kernel would take
stay with the host's product."""

import torch


def test_long_contractions_on_the_host():
    from gllm_amd import ops
    torch.manual_seed(0)
    for dtype in (torch.float32, torch.bfloat16):
        x = torch.randn(300, 384, dtype=dtype)
        w = torch.randn(64, 384, dtype=dtype)
        assert torch.equal(ops.linear(x, w),
                           torch.nn.functional.linear(x, w))

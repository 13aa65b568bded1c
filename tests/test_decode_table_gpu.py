"""Forms of a block table that decode attention takes."""

import pytest
import torch

from test_qkv_decode_gpu import _step

pytestmark = pytest.mark.gpu


def test_table_of_one_column():
    """Its second stride says nothing."""
    from gllm_amd import ops
    s = _step(3, 8, 2, 64, 64, 2, [5, 16, 9])
    wide = s["table"][:, :1].t().contiguous().t()
    assert wide.stride(1) != 1
    out = [ops.qkv_decode(
        s["parts"], s["bias"], s["positions"], s["cos_sin"], s["k"], s["v"],
        s["slots"], t, s["lens"],
        torch.zeros(6, dtype=torch.int32, device="cuda"), 8, 0.125)
        for t in (s["table"], wide)]
    assert torch.equal(*out)

"""Latent attention of few rows with a workgroup a CU and with two."""

import pytest
import torch

from test_mla_gpu import _case, _ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q_lens,ctx,H", [
    # not split: 256 workgroups and one more
    ([2] * 256, [30 + i % 70 for i in range(256)], 8),
    ([2] * 257, [30 + i % 70 for i in range(257)], 8),
    ([3, 1, 2], [2000, 63, 129], 5),
    # in 32 splits: the same
    ([1] * 8, [300, 64, 1, 0, 95, 1000, 33, 700], 16),
    ([1] * 9, [300, 64, 1, 0, 95, 1000, 33, 700, 31], 16),
    ([1] * 9, [300, 64, 1, 0, 95, 1000, 33, 700, 31], 3)])
def test_latent(q_lens, ctx, H):
    from gllm_amd import ops
    args = _case(q_lens, ctx, H)
    ref = _ref(*args, 192 ** -0.5)
    q, cache, table, lens, qsl = (t.cuda() for t in args)
    out = ops.mla_paged_attention(q, cache, cache[..., :512], table, lens,
                                  qsl, 192 ** -0.5)
    # weights and the result are rounded to bf16 (2^-9 each)
    err = (out.cpu().double() - ref).norm() / ref.norm()
    assert err < 3 * 2 ** -9, err

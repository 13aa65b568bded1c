"""Decode attention finds its sequences by length: every sequence is served
once, whatever the lengths, counts of heads and splits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hkv,lens", [
    (1, 8, "ragged"), (2, 1, "ragged"), (63, 8, "ragged"), (65, 2, "equal"),
    (128, 8, "ragged"),     # the last count that is put in order
    (129, 8, "ragged"),     # as they come
    (300, 3, "ragged"), (1024, 1, "ragged"), (70, 8, "one long"),
    (96, 4, "zero")])
def test_every_sequence_once(B, Hkv, lens):
    from gllm_amd import ops
    from gllm_amd.ops import torch_ref
    torch.manual_seed(B + Hkv)
    G, D, page = 2, 64, 16
    n = torch.randint(1, 90, (B,))
    if lens == "equal":
        n[:] = 48
    elif lens == "one long":
        n[:] = 1
        n[B // 2] = 2000
    pages = [-(-int(x) // page) for x in n]
    table = torch.zeros(B, max(pages), dtype=torch.int32)
    ids = torch.randperm(sum(pages)).int()
    at = 0
    for i, c in enumerate(pages):
        table[i, :c] = ids[at:at + c]
        at += c
    k = torch.randn(sum(pages), page, Hkv, D, device="cuda").bfloat16()
    v = torch.randn_like(k)
    q = torch.randn(B, Hkv * G, D, device="cuda").bfloat16()
    table, sl = table.cuda(), n.int().cuda()
    qsl = torch.arange(B + 1, dtype=torch.int32, device="cuda")
    if lens == "zero":
        sl[::5] = 0         # rows of nothing: zeros
    out = ops.paged_attention(q, k, v, table, sl, qsl, D ** -0.5)
    ref = torch_ref.paged_attention(
        q.float().cpu(), k.float().cpu(), v.float().cpu(), table.cpu(),
        n.int(), qsl.cpu(), D ** -0.5).view(B, -1)
    if lens == "zero":
        ref[::5] = 0
    # bf16 weights of a convex sum of values, and the result's rounding
    assert (out.view(B, -1).cpu().float() - ref).abs().max() < 3 * 2 ** -7

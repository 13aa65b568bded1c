"""Decode attention finds its sequences by length: every sequence is served
once, whatever the lengths, counts of heads and splits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hkv,lens", [
    # short sequences come as they are
    (1, 8, "ragged"), (2, 1, "ragged"), (63, 8, "ragged"), (65, 2, "equal"),
    (128, 8, "ragged"), (129, 8, "ragged"), (300, 3, "ragged"),
    (1024, 1, "ragged"), (96, 4, "zero"),
    (70, 8, "one long")])
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


def _in_order(n, Hkv, D, pool):
    """The kernel's rule: its splits, and whether it puts sequences with the
    visible keys ``n`` in order."""
    B, splits = len(n), 1
    while splits < 16 and B * Hkv * splits < 512 and splits * 2 <= pool / 128:
        splits *= 2
    most = max(n)
    alike = sum(x > most - most // 8 for x in n)
    share = 700 if B <= 64 and B * Hkv * splits <= 512 else 1024
    return splits, (256 < B * Hkv * splits <= 1024 and 2 * alike < B
                    and most > share * 256 // (2 * D) * splits)


@pytest.mark.parametrize("B,Hkv,D,splits,lens,order", [
    (64, 8, 128, 1, "wide", True),
    (128, 8, 128, 1, "wide", True),     # the most workgroups
    (129, 8, 128, 1, "wide", False),
    (1024, 1, 128, 1, "wide", True),    # the most sequences
    (400, 2, 64, 1, "wide", True),
    (37, 8, 128, 2, "wide", True), (24, 8, 128, 4, "wide", True),
    (64, 8, 128, 1, "shorter", True), (65, 8, 128, 1, "shorter", False),
    (32, 8, 128, 2, "shorter", True),
    (96, 4, 128, 2, "zeros", True),
    (40, 8, 128, 2, "one long", True),
    (64, 8, 128, 1, "alike", False), (64, 8, 128, 1, "half alike", False),
    (63, 8, 128, 2, "windowed", False), (70, 8, 128, 1, "windowed", True),
    (72, 8, 128, 1, "mixed", True)])
def test_long_sequences(B, Hkv, D, splits, lens, order):
    """Every sequence once where lengths decide the order, in one split and
    in more, with empty rows, windows and portions of prompts between."""
    from gllm_amd import ops
    from gllm_amd.ops import torch_ref
    torch.manual_seed(B + Hkv)
    G, page = 2, 16
    most = (750 if lens == "shorter" else 1100) * splits * 128 // D
    n = torch.randint(1, most // 3, (B,))
    longs = torch.randperm(B)[:1 if lens == "one long" else max(2, B // 16)]
    n[longs] = torch.randint(most // 2, most, longs.shape)
    n[longs[0]] = most
    window = 1100 if lens == "windowed" else 0
    if lens == "alike":
        n = torch.randint(most * 15 // 16, most + 1, (B,))
    elif lens == "half alike":
        n[::2] = most
    elif lens == "windowed":
        n[longs] += 500
    rows = torch.ones(B, dtype=torch.long)
    if lens == "mixed":
        rows[::5] = 3
        n[::5] = torch.randint(3, most + 300, rows[::5].shape)
    zero = torch.zeros(B, dtype=torch.bool)
    if lens == "zeros":
        zero[1::3] = True
        zero[longs] = False
    pages = [-(-int(x) // page) for x in n]
    table = torch.zeros(B, max(pages), dtype=torch.int32)
    ids, at = torch.randperm(sum(pages)).int(), 0
    for i, c in enumerate(pages):
        table[i, :c] = ids[at:at + c]
        at += c
    seen = torch.where(zero | (rows > 1), 0, n)
    if window:
        seen = seen.clamp_max(window)
    assert _in_order(seen.tolist(), Hkv, D, sum(pages) * page) == (splits,
                                                                   order)
    k = torch.randn(sum(pages), page, Hkv, D, device="cuda").bfloat16()
    v = torch.randn_like(k)
    q = torch.randn(int(rows.sum()), Hkv * G, D, device="cuda").bfloat16()
    qsl = torch.cat([torch.zeros(1), rows.cumsum(0)]).int()
    sl = torch.where(zero, 0, n).int()
    out = ops.paged_attention(
        q, k, v, table.cuda(), sl.cuda(), qsl.cuda(), D ** -0.5,
        int(rows.max()), sliding_window=window,
        single_rows=int((rows == 1).sum()) if lens == "mixed" else 0)
    ref = torch_ref.paged_attention(
        q.float().cpu(), k.float().cpu(), v.float().cpu(), table, n.int(),
        qsl, D ** -0.5, sliding_window=window).view(q.shape[0], -1)
    ref[zero.repeat_interleave(rows)] = 0
    # bf16 weights of a convex sum of values, and the result's rounding
    assert (out.view(ref.shape).cpu().float() - ref).abs().max() < 3 * 2 ** -7

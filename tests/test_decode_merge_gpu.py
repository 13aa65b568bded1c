"""Merges of one to seventeen splits of decode attention."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,splits", [(64, 1), (33, 2), (17, 4), (9, 8),
                                      (3, 16)])
@pytest.mark.parametrize("opt", ["", "gate sink", "kept"])
def test_merges(B, splits, opt):
    """``splits``, and one more for the kept first keys."""
    from gllm_amd import ops
    torch.manual_seed(B)
    H, D, n = 8, 64, 3000
    lens = [1 + (n * (i + 1)) // B for i in range(B)]
    need = [-(-x // 16) for x in lens]
    pool = sum(need)
    assert splits * 64 <= pool * 16 // 2 or splits == 1
    table = torch.zeros(B, max(need), dtype=torch.int32)
    perm, at = torch.randperm(pool).int(), 0
    for b, p in enumerate(need):
        table[b, :p] = perm[at:at + p]
        at += p
    k, v = (torch.randn(pool, 16, H, D).bfloat16() for _ in range(2))
    q = torch.randn(B, H * D).bfloat16()
    gate = torch.randn(B, H * D).bfloat16() if "gate" in opt else None
    window, keep = (400, 33) if opt == "kept" else (0, 0)
    want = torch.empty(B, H, D, dtype=torch.float64)
    for b, m in enumerate(lens):
        ks, vs = (c[table[b, :need[b]].long()].flatten(0, 1)[:m].double()
                  for c in (k, v))
        s = torch.einsum("hd,nhd->hn", q[b].view(H, D).double(), ks) / 8
        if window:
            hide = torch.arange(m)
            s[:, (hide < m - window) & (hide >= keep)] = -float("inf")
        top = s.max(1, keepdim=True).values
        if "sink" in opt:
            top = top.clamp_min(0)
        p = (s - top).exp()
        total = p.sum(1, keepdim=True)
        if "sink" in opt:
            total = total + (-top).exp()
        want[b] = torch.einsum("hn,nhd->hd", p / total, vs)
    if gate is not None:
        want *= gate.view(B, H, D).double().sigmoid()
    out = torch.empty(B, H * D, dtype=torch.bfloat16, device="cuda")
    assert ops._seq_kernels().window_attention_decode(
        out, q.cuda(), gate.cuda() if gate is not None else None, k.cuda(),
        v.cuda(), table.cuda(),
        torch.tensor(lens, dtype=torch.int32, device="cuda"), 0.125, window,
        keep, "sink" in opt, None, 0.0, None, 0.0, 0)
    # weights and results are rounded to bf16 once each, 2^-9 relative
    err = (out.double().cpu().view_as(want) - want).norm() / want.norm()
    assert err < 2 ** -8, err

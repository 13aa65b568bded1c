"""Decode attention at the edges of its 32-key tiles and of its heads, against
fp64: whatever the caches hold behind a sequence takes no part."""

import pytest
import torch

pytestmark = pytest.mark.gpu

LENS = [1, 31, 32, 33, 64, 127, 128, 129, 160, 257, 640, 1025]


@pytest.mark.parametrize("window", [0, 100])
@pytest.mark.parametrize("Hq,Hkv,D,ps,copies", [
    (8, 8, 8, 16, 1), (6, 3, 40, 16, 1), (4, 4, 64, 1, 1), (5, 1, 72, 16, 1),
    (16, 1, 128, 7, 1), (40, 8, 128, 16, 1), (40, 8, 128, 16, 8),
    (14, 2, 64, 16, 30)])
def test_tiles(Hq, Hkv, D, ps, copies, window):
    from gllm_amd import ops
    torch.manual_seed(D + Hq)
    lens = LENS * copies
    B, pages = len(lens), [-(-n // ps) for n in lens]
    table = torch.zeros(B, max(pages), dtype=torch.int32)
    perm, at = torch.randperm(sum(pages)).int(), 0
    shape = (sum(pages), ps, Hkv, D)
    k = torch.full(shape, float("nan"), dtype=torch.bfloat16)
    v = torch.full(shape, float("nan"), dtype=torch.bfloat16)
    q = torch.randn(B, Hq, D).bfloat16()
    want = torch.empty(B, Hq, D, dtype=torch.float64)
    for b, (n, p) in enumerate(zip(lens, pages)):
        ids = perm[at:at + p]
        at += p
        table[b, :p] = ids
        ks, vs = (torch.randn(n, Hkv, D).bfloat16() for _ in range(2))
        rows = torch.arange(n)
        where = ids.long()[rows // ps], rows % ps
        k[where], v[where] = ks, vs
        lo = max(0, n - window) if window else 0
        G = Hq // Hkv
        s = torch.einsum("hd,nhd->hn", q[b].double(),
                         ks[lo:].double().repeat_interleave(G, 1)) * D ** -0.5
        want[b] = torch.einsum("hn,nhd->hd", s.softmax(-1),
                               vs[lo:].double().repeat_interleave(G, 1))
    got = ops.paged_attention(
        q.cuda(), k.cuda(), v.cuda(), table.cuda(),
        torch.tensor(lens, dtype=torch.int32, device="cuda"), None,
        D ** -0.5, sliding_window=window)
    # weights and results are rounded to bf16 once each, 2^-9 relative
    err = (got.double().cpu().view_as(want) - want).norm() / want.norm()
    assert err < 2 ** -8, err

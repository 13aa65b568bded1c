"""Cache rows and absorbed queries of latent attention on both sides of the line
from which on the rows are a launch of their own: the same bits as in batches
below it."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H", [(3072, 2), (3073, 2), (4096, 8), (4097, 9)])
@pytest.mark.parametrize("wdtype", [torch.bfloat16, torch.float32])
def test_rows(T, H, wdtype):
    from gllm_amd import ops
    gen = torch.Generator(device="cuda").manual_seed(T)

    def rand(*shape):
        return torch.randn(*shape, generator=gen, device="cuda").bfloat16()

    q, kv, w = rand(T, H * 192 + 8)[:, :H * 192], rand(T, 576), \
        rand(H * 256, 512)
    norm_w = rand(512).to(wdtype)
    pos = torch.randint(0, 999, (T,), generator=gen, device="cuda")
    cs = torch.randn(1000, 64, generator=gen, device="cuda")
    slots = torch.randperm(T + 40, generator=gen, device="cuda")[:T]

    def run(rows):
        cache = torch.zeros((T + 40) // 16 + 1, 16, 1, 576,
                            dtype=torch.bfloat16, device="cuda")
        out = [ops.mla_queries(q[a:b], kv[a:b], norm_w, 1e-6, pos[a:b], cs, w,
                               cache, slots[a:b]) for a, b in rows]
        return torch.cat(out), cache
    got, got_cache = run([(0, T)])
    want, want_cache = run([(a, min(a + 1024, T)) for a in range(0, T, 1024)])
    assert torch.equal(got, want) and torch.equal(got_cache, want_cache)

"""Softmax layers of the hybrid stack without an output gate: norm, rotation
and cache rows in one kernel against the kernels one after the other."""

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
PAGE = 16


def context(lens, past, kv, D, layers):
    from gllm_amd.runtime.forward_context import ForwardContext
    gen = torch.Generator().manual_seed(sum(lens))
    total = [a + b for a, b in zip(lens, past)]
    per = [-(-t // PAGE) for t in total]
    pages = torch.randperm(sum(per) + 2, generator=gen)
    table = torch.zeros(len(lens), max(per), dtype=torch.int32)
    slots, positions, at = [], [], 0
    for i, (n, p) in enumerate(zip(lens, past)):
        own = pages[at:at + per[i]]
        table[i, :per[i]] = own
        at += per[i]
        pos = torch.arange(p, p + n)
        positions.append(pos)
        slots.append(own[pos // PAGE] * PAGE + pos % PAGE)
    caches = [[torch.randn(len(pages), PAGE, kv, D, generator=gen).bfloat16()
               .cuda() for _ in range(layers)] for _ in range(2)]
    return ForwardContext(
        num_tokens=sum(lens), positions=torch.cat(positions).cuda(),
        slot_mapping=torch.cat(slots).cuda(), block_table=table.cuda(),
        seq_lens=torch.tensor(total).int().cuda(),
        query_start_loc=torch.tensor([0] + lens).cumsum(0).int().cuda(),
        max_query_len=max(lens), max_seq_len=max(total),
        k_caches=caches[0], v_caches=caches[1])


@pytest.mark.parametrize("lens,past", [
    ([1], [40]), ([1, 1, 1], [0, 15, 16]), ([33, 1, 70], [0, 50, 10])])
@pytest.mark.parametrize("heads,kv,D,part", [
    (8, 2, 128, 0.25), (4, 4, 128, 1.0), (4, 1, 64, 0.5)])
@pytest.mark.parametrize("bias", [False, True])
def test_heads(lens, past, heads, kv, D, part, bias, monkeypatch):
    from gllm_amd import ops
    from gllm_amd.models.hybrid_gdn import HybridFullAttention
    cfg = SimpleNamespace(
        hidden_size=256, num_attention_heads=heads, num_key_value_heads=kv,
        head_dim=D, partial_rotary_factor=part, max_position_embeddings=256,
        attention_bias=bias, rms_norm_eps=1e-6)
    layer = HybridFullAttention(cfg, 1, dtype=torch.bfloat16).cuda()
    gen = torch.Generator(device="cuda").manual_seed(heads + D)
    for p in layer.parameters():
        p.data.normal_(0, 0.3 if p.dim() == 1 else p.shape[-1] ** -0.5,
                       generator=gen)
    fctx = context(lens, past, kv, D, 2)
    hidden = torch.randn(sum(lens), 256, device="cuda",
                         generator=gen).bfloat16()
    start = [t.clone() for t in fctx.k_caches + fctx.v_caches]
    took = []
    op = ops.qkv_norm_rope_cache
    monkeypatch.setattr(ops, "qkv_norm_rope_cache",
                        lambda *a: took.append(1) or op(*a))
    got = layer.heads(fctx.positions, hidden, fctx)
    assert took == [1]
    got_cache = [t.clone() for t in fctx.k_caches + fctx.v_caches]
    for t, s in zip(fctx.k_caches + fctx.v_caches, start):
        t.copy_(s)
    monkeypatch.setattr(ops, "qkv_norm_rope_cache_ok", lambda *a: False)
    want = layer.heads(fctx.positions, hidden, fctx)
    assert took == [1]
    caches = fctx.k_caches + fctx.v_caches
    for i in (0, 2):       # another layer's
        assert torch.equal(caches[i], start[i])
        assert torch.equal(got_cache[i], start[i])
    for i in (1, 3):
        assert not torch.equal(got_cache[i], start[i])
        assert torch.equal(got_cache[i], caches[i])
    assert torch.equal(got, want)

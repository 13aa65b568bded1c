"""A latent attention layer over decode rows, portions behind a cached
prefix and whole prompts in one batch, in its two forms, against fp64."""

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV, PAGE, HIDDEN = "cuda", 16, 320


def _layer(heads):
    from gllm_amd.models.deepseek_v2 import MLAAttention
    with torch.device(DEV):
        layer = MLAAttention(SimpleNamespace(
            hidden_size=HIDDEN, num_attention_heads=heads,
            qk_nope_head_dim=128, qk_rope_head_dim=64, v_head_dim=128,
            kv_lora_rank=512, q_lora_rank=None,
            max_position_embeddings=4096), 0, dtype=torch.bfloat16)
    for p in layer.parameters():
        p.data.normal_(0, p.shape[-1] ** -0.5) if p.dim() > 1 \
            else p.data.uniform_(0.5, 1.5)
    return layer.to(DEV)


def _context(rows, past, cache, table, extra):
    from gllm_amd.runtime.forward_context import ForwardContext
    lens = [a + b for a, b in zip(rows, past)]
    pos = [torch.arange(a, b) for a, b in zip(past, lens)]
    slots = [table[i].long()[p // PAGE] * PAGE + p % PAGE
             for i, p in enumerate(pos)]
    qsl = torch.tensor([0] + rows).cumsum(0).tolist() + extra
    return ForwardContext(
        num_tokens=sum(rows), positions=torch.cat(pos).to(DEV),
        slot_mapping=torch.cat(slots).to(DEV), block_table=table.to(DEV),
        seq_lens=torch.tensor(lens, dtype=torch.int32, device=DEV),
        query_start_loc=torch.tensor(qsl, dtype=torch.int32, device=DEV),
        max_query_len=max(rows), max_seq_len=max(lens), k_caches=[cache],
        v_caches=[cache[..., :512]])


def _turn(x, ang):
    a, b = x[..., :32], x[..., 32:]
    return torch.cat([a * ang.cos() - b * ang.sin(),
                      b * ang.cos() + a * ang.sin()], -1)


@pytest.mark.parametrize("rows,past,heads,extra,first", [
    # decode rows, then prompts
    ([1] * 5 + [33, 128, 8], [600, 15, 16, 900, 70] + [0] * 3, 16, [], 5),
    ([1, 129], [512, 0], 1, [130, 200], 1),
    # portions behind cached prefixes stay absorbed
    ([1, 40, 3, 300, 260], [77, 130, 1, 0, 0], 64, [], 3),
    ([1, 70, 2100], [33, 64, 0], 16, [2171, 2172], 2),
    # nothing before the prompts
    ([8, 200, 64], [0, 0, 0], 16, [272, 300], 0),
    # all absorbed: a short batch, a last sequence that is no prompt
    ([1, 1, 20], [10, 20, 0], 16, [], 3), ([30, 1], [0, 40], 16, [99], 2),
])
def test_mixed_batch(rows, past, heads, extra, first):
    torch.manual_seed(sum(rows))
    layer = _layer(heads)
    lens = [a + b for a, b in zip(rows, past)]
    need = [-(-n // PAGE) for n in lens]
    table = torch.zeros(len(lens), max(need), dtype=torch.int32)
    ids, at = torch.randperm(sum(need) + 2).int(), 0
    for i, n in enumerate(need):
        table[i, :n] = ids[at:at + n]
        at += n
    cache = torch.randn(sum(need) + 2, PAGE, 1, 576, device=DEV).bfloat16()
    hidden = torch.randn(sum(rows), HIDDEN, device=DEV).bfloat16()
    outs, caches = [], []
    for absorbed in (False, True):
        caches.append(cache.clone())
        fctx = _context(rows, past, caches[-1], table, extra)
        assert fctx.per_head_from(heads) == first
        if absorbed:
            fctx._per_head_from = (heads, len(rows))
        with torch.no_grad():
            outs.append(layer.heads(fctx.positions, hidden, fctx))
    assert torch.equal(*caches)
    # queries and latents as the layer forms them; their products in fp64
    with torch.no_grad():
        q, kv = layer._queries_and_latents(hidden)
    for got, mod in ((q, layer.q_proj), (kv, layer.kv_a_proj_with_mqa)):
        want = hidden.double() @ mod.weight.double().t()
        assert (got.double() - want).norm() / want.norm() < 2 ** -8
    ang = fctx.positions.double().cpu()[:, None] * \
        1e4 ** (-torch.arange(32).double() / 32)
    q = q.double().cpu().view(-1, heads, 192)
    q = torch.cat([q[..., :128], _turn(q[..., 128:], ang[:, None])], -1)
    kv = kv.double().cpu()
    norm = layer.kv_a_layernorm
    lat = kv[:, :512] * (kv[:, :512].square().mean(-1, keepdim=True)
                         + norm.eps).rsqrt() * norm.weight.double().cpu()
    new = torch.cat([lat, _turn(kv[:, 512:], ang)], -1)
    flat = caches[0].view(-1, 576).double().cpu()
    got = flat[fctx.slot_mapping.cpu()]
    assert (got - new).norm() / new.norm() < 2 ** -8  # one rounding
    flat[fctx.slot_mapping.cpu()] = 0    # rows of no new token are kept
    old = cache.view(-1, 576).double().cpu()
    old[fctx.slot_mapping.cpu()] = 0
    assert torch.equal(flat, old)
    flat = caches[0].view(-1, 576).double().cpu()
    w = layer.kv_b_proj.weight.double().cpu()
    ref, at = [], 0
    for i, (n, m) in enumerate(zip(rows, lens)):
        p = torch.arange(m)
        c = flat[table[i].long()[p // PAGE] * PAGE + p % PAGE]
        per = (c[:, :512] @ w.t()).view(m, heads, 256)
        k = torch.cat([per[..., :128],
                       c[:, None, 512:].expand(m, heads, 64)], -1)
        s = q[at:at + n].transpose(0, 1) @ k.permute(1, 2, 0).contiguous()
        hide = torch.arange(m)[None] > torch.arange(m - n, m)[:, None]
        s = (s * layer.scale).masked_fill(hide, -float("inf")).softmax(-1)
        ref.append((s @ per[..., 128:].transpose(0, 1).contiguous())
                   .transpose(0, 1).reshape(n, -1))
        at += n
    ref = torch.cat(ref)
    starts = torch.tensor([0] + rows).cumsum(0)
    for out in outs:
        out = out.double().cpu()
        for a, b in zip(starts, starts[1:]):
            # bf16 queries, keys or latent queries, weights, values, result
            err = (out[a:b] - ref[a:b]).norm() / ref[a:b].norm()
            assert err < 4 * 2 ** -9, (a, err)


def test_one_product_for_two():
    """The rows that lie together give what the two products give."""
    layer = _layer(16)
    torch.manual_seed(0)
    for M in (1, 40, 300):
        x = torch.randn(M, HIDDEN, device=DEV).bfloat16()
        with torch.no_grad():
            q, kv = layer._queries_and_latents(x)
            parts = layer.q_proj(x), layer.kv_a_proj_with_mqa(x)
        assert q.stride(0) == kv.stride(0) == 16 * 192 + 576
        for a, b in zip((q, kv), parts):  # sums in another order
            assert (a.double() - b.double()).norm() / b.norm() < 2 ** -8
    for M, one in ((4352, True), (4353, False)):  # 255 tiles, 270
        x = torch.randn(M, HIDDEN, device=DEV).bfloat16()
        with torch.no_grad():
            q, kv = layer._queries_and_latents(x)
            parts = layer.q_proj(x), layer.kv_a_proj_with_mqa(x)
        assert q.is_contiguous() != one
        for a, b in zip((q, kv), parts):
            assert (a.double() - b.double()).norm() / b.norm() < 2 ** -8
    b = layer.kv_a_proj_with_mqa.weight
    b.data = b.data.clone()               # apart: two products
    with torch.no_grad():
        q, kv = layer._queries_and_latents(x)
    assert q.is_contiguous() and kv.is_contiguous()
    assert torch.equal(q, parts[0]) and torch.equal(kv, parts[1])

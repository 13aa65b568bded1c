"""What a latent layer hands to its two attention forms for a batch of
decode rows and whole prompts."""

from types import SimpleNamespace

import pytest
import torch

from gllm_amd import ops
from gllm_amd.models.deepseek_v2 import MLAAttention
from gllm_amd.runtime.forward_context import ForwardContext


def _layer(heads=1):
    return MLAAttention(SimpleNamespace(
        hidden_size=64, num_attention_heads=heads, qk_nope_head_dim=128,
        qk_rope_head_dim=64, v_head_dim=128, kv_lora_rank=512,
        q_lora_rank=None, max_position_embeddings=64), 0)


def _context(rows, past, extra=()):
    """``extra``: offsets behind those of the sequences."""
    lens = [a + b for a, b in zip(rows, past)]
    qsl = torch.tensor([0] + rows).cumsum(0).tolist() + list(extra)
    n = sum(rows)
    return ForwardContext(
        num_tokens=n, positions=torch.arange(n),
        slot_mapping=torch.arange(n),
        block_table=torch.zeros(len(rows), 8, dtype=torch.int32),
        seq_lens=torch.tensor(lens, dtype=torch.int32),
        query_start_loc=torch.tensor(qsl, dtype=torch.int32),
        max_query_len=max(rows), max_seq_len=max(lens),
        k_caches=[torch.zeros(8, 16, 1, 576)], v_caches=[None])


@pytest.mark.parametrize("extra", [(), (19, 19), (99,)])
def test_longer_offsets(monkeypatch, extra):
    """Offsets behind the last sequence's are no prompts."""
    rows, past = [1, 1, 8, 9], [5, 7, 0, 0]
    fctx, seen = _context(rows, past, extra), {}

    def prompts(q, kv, w, eps, pos, cos_sin, w_kvb, cache, slots, starts,
                longest, scale, out):
        seen.update(starts=starts.tolist(), longest=longest,
                    rows=(q.shape[0], kv.shape[0], pos.tolist(),
                          slots.tolist(), out.shape[0]))
        out.fill_(2.0)

    def latent(q, k, v, table, lens, starts, scale, seq_lens_cpu,
               query_start_loc_cpu):
        seen.update(front=(lens.tolist(), starts.tolist(), seq_lens_cpu,
                           query_start_loc_cpu, table.shape[0]))
        return q

    monkeypatch.setattr(ops, "mla_queries", lambda q, *a: q)
    monkeypatch.setattr(ops, "mla_paged_attention", latent)
    monkeypatch.setattr(ops, "mla_values",
                        lambda o, w: torch.ones(o.shape[0], 128))
    monkeypatch.setattr(ops, "mla_prompts", prompts)
    n = sum(rows)
    out = _layer()._with_prompts(2, fctx.positions, None, None,
                                 torch.zeros(n, 192), torch.zeros(n, 576),
                                 fctx)
    tail = list(range(2, n))
    assert seen == {"starts": [0, 8, 17], "longest": 9,
                    "rows": (17, 17, tail, tail, 17),
                    "front": ([6, 8], [0, 1, 2], [6, 8], [0, 1, 2], 2)}
    assert (out[:2] == 1).all() and (out[2:] == 2).all()


def test_converted_rows_are_freed():
    """q_proj's dense rows go with its conversion although kv_a_proj's, which
    stay, were laid behind them."""
    from gllm_amd.layers.quantization.int4 import convert_model_to_int4
    for quantized in (False, True):
        layer = _layer()
        if quantized:
            convert_model_to_int4(torch.nn.ModuleDict({"attn": layer}),
                                  {"quant_method": "gptq", "group_size": 64})
        w = layer.kv_a_proj_with_mqa.weight
        assert w.shape == (576, 64)
        own = w.numel() * w.element_size()
        assert w.untyped_storage().nbytes() == (
            own if quantized else own + 192 * 64 * 4)


@pytest.mark.parametrize("rows,past,heads,prompts,per_head", [
    ([8], [0], 16, 0, 0), ([7], [0], 16, 0, 1),
    ([1], [0], 16, 1, 1), ([1], [30], 16, 1, 1),     # decode rows
    ([2] * 300, [0] * 300, 16, 0, 300), ([8] * 64, [0] * 64, 16, 0, 0),
    ([9, 1], [0, 0], 16, 2, 2),            # a prompt of one row ends the tail
    ([40, 40], [0, 16], 16, 2, 2),         # so does a cached prefix
    ([1] * 16 + [32], [510] * 16 + [0], 16, 16, 17),  # 511 keys
    ([1] * 16 + [32], [511] + [9] * 15 + [0], 16, 16, 16),
    ([1] * 64 + [63], [200] * 64 + [0], 16, 64, 65),  # tiles of the mixed
    ([1] * 64 + [64], [200] * 64 + [0], 16, 64, 64),
    ([1] * 64 + [63], [200] * 64 + [0], 32, 64, 64),
    ([1, 256, 2047], [900, 2000, 0], 16, 2, 3),       # behind a portion
    ([1, 256, 2048], [900, 2000, 0], 16, 2, 2),
    ([1, 256, 256], [900, 2000, 0], 128, 2, 2),
    ([0, 12], [5, 0], 16, 1, 2),
])
def test_forms(rows, past, heads, prompts, per_head):
    """Where whole prompts begin, and from where on they attend per head."""
    for extra in ((), (sum(rows), 9 + sum(rows))):
        fctx = _context(rows, past, extra)
        assert fctx.prompts_from() == prompts
        assert fctx.per_head_from(heads) == per_head
        assert fctx.per_head_from(heads) == per_head  # (kept)
        assert _layer()._prompts_from(fctx) == fctx.per_head_from(1)

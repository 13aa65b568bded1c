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

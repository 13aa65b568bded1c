"""e4m3 rows from layer to layer: the hidden states of a block-quantized
decoder are the same bits whether the kernels that form rows leave them or
each product quantizes its own, and no product quantizes rows that were left."""

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu

HIDDEN, FF, HEADS, KV, DIM, PAGE = 256, 18432, 4, 2, 128, 16


def _model(qk_norm, plain):
    from gllm_amd.layers.quantization.fp8 import convert_linear_to_fp8
    from gllm_amd.models.llama_family import LlamaFamilyForCausalLM

    class Model(LlamaFamilyForCausalLM):
        pass
    Model.qk_norm, Model.qkv_bias = qk_norm, not qk_norm
    cfg = SimpleNamespace(
        hidden_size=HIDDEN, intermediate_size=FF, num_attention_heads=HEADS,
        num_key_value_heads=KV, head_dim=DIM, num_hidden_layers=2,
        vocab_size=128, rms_norm_eps=1e-6, max_position_embeddings=256)
    model = Model(cfg, SimpleNamespace(
        torch_dtype=lambda: torch.bfloat16,
        pp_layer_range=lambda rank, n: (0, n)))
    for layer in model.layers:
        for name, proj in (("qkv", layer.self_attn.qkv_proj),
                           ("o", layer.self_attn.o_proj),
                           ("gate_up", layer.mlp.gate_up_proj),
                           ("down", layer.mlp.down_proj)):
            if name != plain:
                convert_linear_to_fp8(proj, (128, 128))
    model.cuda()
    g = torch.Generator(device="cuda").manual_seed(1)
    for name, p in model.named_parameters():
        x = torch.randn(p.shape, device="cuda", generator=g)
        if p.dtype == torch.float8_e4m3fn:
            p.data.copy_((x * 60).to(p.dtype))
        elif name.endswith("weight_scale_inv"):
            p.data.copy_((x.abs() * 0.3 + 0.7) * (HIDDEN ** -0.5 / 60))
        elif "norm" in name:
            p.data.copy_(1 + 0.1 * x)
        else:
            p.data.copy_(x * p.shape[-1] ** -0.5)
    return model


def _context(B):
    from gllm_amd.runtime.forward_context import ForwardContext
    lens = [1 + 13 * i % 90 for i in range(B)]
    per = -(-max(lens) // PAGE)
    g = torch.Generator(device="cuda").manual_seed(2)
    caches = [[torch.randn(B * per, PAGE, KV, DIM, device="cuda",
                           generator=g).bfloat16() for _ in range(2)]
              for _ in range(2)]
    slots = [b * per * PAGE + n - 1 for b, n in enumerate(lens)]
    return ForwardContext(
        num_tokens=B,
        positions=torch.tensor([n - 1 for n in lens], device="cuda"),
        slot_mapping=torch.tensor(slots, device="cuda"),
        block_table=torch.arange(B * per, dtype=torch.int32,
                                 device="cuda").view(B, per),
        seq_lens=torch.tensor(lens, dtype=torch.int32, device="cuda"),
        query_start_loc=torch.arange(B + 1, dtype=torch.int32,
                                     device="cuda"),
        max_query_len=1, max_seq_len=max(lens), k_caches=caches[0],
        v_caches=caches[1])


def _run(model, B, monkeypatch, left):
    from gllm_amd import ops
    from gllm_amd.layers.linear import LinearBase
    made, quant = [], ops.per_token_group_quant_fp8

    def counted(x, *args, **kw):
        made.append(tuple(x.shape))
        return quant(x, *args, **kw)
    fctx = _context(B)
    with monkeypatch.context() as m, torch.no_grad():
        m.setattr(ops, "per_token_group_quant_fp8", counted)
        if not left:
            m.setattr(LinearBase, "takes_fp8", lambda self, rows: False)
        ids = torch.arange(B, device="cuda") % 128
        out, _ = model(ids, fctx.positions, fctx)
    return (out, *fctx.k_caches, *fctx.v_caches), made


@pytest.mark.parametrize("plain", [None, "qkv", "o", "gate_up", "down"])
@pytest.mark.parametrize("qk_norm", [False, True])
@pytest.mark.parametrize("B", [1, 64, 65])
def test_layers(B, qk_norm, plain, monkeypatch):
    model = _model(qk_norm, plain)
    want, every = _run(model, B, monkeypatch, False)
    got, made = _run(model, B, monkeypatch, True)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    assert not torch.isnan(got[0]).any()
    if B > 64:
        assert not every and not made  # (bf16 copies of the weights)
    else:
        assert len(every) == (8 if plain is None else 6)
    if plain is None and B == 64:
        # the first layer's input; behind a norm per head, the attention
        # kernel's results
        assert len(made) == (3 if qk_norm else 1)

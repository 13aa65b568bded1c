"""The rotation's base survives a config whose class keeps it in
rope_parameters only."""

import json

import pytest
import torch


@pytest.mark.parametrize("theta", [10000.0, 500000.0])
def test_rope_theta_reaches_the_rotation(tmp_path, theta):
    from gllm_amd.models import loader
    (tmp_path / "config.json").write_text(json.dumps(dict(
        model_type="llama", architectures=["LlamaForCausalLM"],
        hidden_size=64, num_attention_heads=4, num_key_value_heads=2,
        num_hidden_layers=1, intermediate_size=128, vocab_size=64,
        max_position_embeddings=128, rope_theta=theta)))
    cfg = loader.load_hf_config(str(tmp_path))
    assert cfg.rope_theta == theta
    from gllm_amd.models.llama_family import DenseAttention
    rope = DenseAttention(cfg, 0, qkv_bias=False, qk_norm=False).rotary_emb
    half = 16 // 2
    want = torch.cos(1.0 / theta ** (torch.arange(half).float() / half))
    assert torch.allclose(rope.cos_sin_cache[1, :half].float(), want,
                          atol=1e-6)

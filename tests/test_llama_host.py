"""Host-side checks of the decoder (no GPU needed)."""

import pytest
import torch

from beam_engine_amd.llama import LlamaConfig, LlamaDecoder


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_prefill_refuses_prompts_beyond_the_rope_tables(dtype):
    """Refused before anything is written: the page table is never touched."""
    cfg = LlamaConfig(vocab_size=32, hidden_size=64, intermediate_size=64, num_hidden_layers=1, num_attention_heads=1,
                      num_key_value_heads=1, head_dim=64, max_position_embeddings=16)
    m = LlamaDecoder(cfg, device="cpu", dtype=dtype)
    with pytest.raises(ValueError, match="17 tokens"):
        m.prefill(torch.zeros((1, 17), dtype=torch.int64), None, [[0, 1]])

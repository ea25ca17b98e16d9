"""A cache counts no rows that a kernel refused to write."""

import pytest
import torch

from mlx_sharding_amd import ops
from mlx_sharding_amd.models.deepseek_v2 import MLAAttention
from mlx_sharding_amd.config import ModelConfig
from mlx_sharding_amd.ops.kvcache import KVCache


class Refuses:
    """The extension, whose kernels check their operands and raise."""

    def __getattr__(self, name):
        def kernel(*args, **kwargs):
            raise RuntimeError(name)
        return kernel


@pytest.fixture(autouse=True)
def refused(monkeypatch):
    monkeypatch.setattr(ops, "hip_ext", Refuses)


def test_rotated_rows():
    cache = KVCache(2, 16, 16)
    q, k, v = (torch.randn(1, 3, h, 16).bfloat16() for h in (4, 2, 2))
    turn = torch.ones(3, 8)
    with pytest.raises(RuntimeError, match="rope_qkv"):
        cache.append_rope_qkv(q, k, v, turn, turn)
    assert cache.offset == 0 and cache.k.shape[2] == 0


@pytest.mark.parametrize("T", [1, 5])
def test_latent_rows(T):
    cfg = ModelConfig.from_dict({
        "model_type": "deepseek_v2", "hidden_size": 64, "num_attention_heads": 2,
        "kv_lora_rank": 32, "qk_nope_head_dim": 128, "qk_rope_head_dim": 64,
        "v_head_dim": 128})
    attn = MLAAttention(cfg, lambda p: None, "a")
    cache = KVCache(1, 32 + 64, 0)
    q, latent = torch.zeros(1, T, 2 * 192).bfloat16(), torch.zeros(1, T, 96).bfloat16()
    turn = torch.ones(T, 32)
    go = attn._one_token if T == 1 else attn._prompt
    with pytest.raises(RuntimeError, match="mla_prepare" if T == 1 else "mla_rows"):
        go(q, latent, turn, turn, cache)
    assert cache.offset == 0

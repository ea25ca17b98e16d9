"""Decoding steps of packed models where their words have no copy: on the CPU, and with
torch's own operators."""

import pytest
import torch

from mlx_sharding_amd import ops
from mlx_sharding_amd.config import ModelConfig, QuantConfig
from mlx_sharding_amd.models import get_model_class
from mlx_sharding_amd.models.base import Linear
from mlx_sharding_amd.models.fuse import fuse_model
from mlx_sharding_amd.ops import reference as ref


def packed(kind, bits, fused, device="cpu"):
    cfg = ModelConfig.from_dict({
        "model_type": kind, "hidden_size": 128, "num_hidden_layers": 2,
        "intermediate_size": 192, "num_attention_heads": 4, "num_key_value_heads": 2,
        "head_dim": 32, "vocab_size": 128, "rms_norm_eps": 1e-5, "sliding_window": 64,
        "query_pre_attn_scalar": 32, "quantization": {"group_size": 32, "bits": bits}})
    torch.manual_seed(bits)
    model = get_model_class(kind)(cfg, cfg.shard(0, 2),
                                  quant_for=lambda path: QuantConfig(32, bits))
    for p in model.parameters():
        if p.is_floating_point():
            p.data.normal_(0, 0.05)
    for m in model.modules():
        if isinstance(m, Linear) and m.quant is not None:
            w = torch.randn(m.out_features, m.in_features) * 0.1
            m.weight.data, m.scales.data, m.biases.data = ref.quantize(w.bfloat16(), 32, bits)
    model = model.to(device).eval()
    if fused:
        fuse_model(model)
    return model


def stepwise(model, tokens):
    """Logits of a prompt of all but three tokens and of these, one by one."""
    cache = model.make_cache(batch_size=tokens.shape[0])
    out = [model(tokens[:, :-3], cache)]
    out += [model(tokens[:, t: t + 1], cache) for t in range(tokens.shape[1] - 3, tokens.shape[1])]
    return torch.cat(out, 1).double()


@torch.no_grad()
@pytest.mark.parametrize("kind", ["llama", "qwen2", "gemma2"])
@pytest.mark.parametrize("bits,fused,batch", [(4, False, 1), (4, True, 3), (8, True, 1)])
def test_on_the_cpu(kind, bits, fused, batch):
    model = packed(kind, bits, fused)
    tokens = torch.randint(0, 128, (batch, 9))
    got = stepwise(model, tokens)
    want = model(tokens, model.make_cache(batch_size=batch)).double()
    # rows alone and together: some ten roundings to bf16 (2^-9 each) through two layers
    assert float((got - want).norm() / want.norm()) < 10 * 2.0 ** -9
    assert not any(hasattr(p, "_mlxs_dqw") for p in model.parameters())


@torch.no_grad()
@pytest.mark.parametrize("T", [1, 5])
def test_attention_alone(T):
    """A layer's attention that is given the norm of its rows, with projections of several
    columns together."""
    model = packed("llama", 4, True)
    layer = next(iter(model.model.layers.values()))
    x = torch.randn(1, T, 128).bfloat16()
    angle = torch.rand(T, 16)
    outs = [layer.self_attn(*args) for args in (
        (x, angle.cos(), angle.sin(), model.make_cache()[0], layer.input_layernorm),
        (layer.input_layernorm(x), angle.cos(), angle.sin(), model.make_cache()[0]))]
    assert torch.equal(*outs)


@pytest.mark.gpu
@torch.no_grad()
def test_with_torch_operators(monkeypatch):
    """Nothing is copied that these do not read."""
    monkeypatch.setenv("MLXS_AMD_FORCE_TORCH", "1")
    model = packed("llama", 4, True, "cuda")
    tokens = torch.randint(0, 128, (2, 9), device="cuda")
    stepwise(model, tokens)
    assert not any(hasattr(p, "_mlxs_dqw") for p in model.parameters())


@pytest.mark.skipif(ops._load_ext() is None, reason="extension is not built")
def test_words_of_the_host_are_refused():
    words = torch.zeros(8, 4, dtype=torch.int32)
    scales = torch.zeros(8, 1).bfloat16()
    with pytest.raises(RuntimeError, match="on GPU"):
        ops.hip_ext().dequant(words, scales, scales, 32, 32, 4)

"""Halves of a layer of 65 to 384 tokens in one call each, beside what they stand for."""

import types

import pytest
import torch
import torch.nn.functional as F

from mlx_sharding_amd import ops
from test_attend_few import cache_of, inputs, one_by_one

pytestmark = pytest.mark.gpu


@torch.no_grad()
@pytest.mark.parametrize("B,T", [(1, 65), (2, 60), (33, 2), (5, 51), (1, 384)])
@pytest.mark.parametrize("H,heads,kv,D", [(512, 8, 2, 64), (1024, 4, 4, 128), (2048, 32, 4, 64),
                                          (544, 2, 1, 256)])
@pytest.mark.parametrize("bias", [False, True])
def test_attention(B, T, H, heads, kv, D, bias):
    at = 7
    a = inputs(B, T, H, heads, kv, D, bias)
    here, there = cache_of(B, kv, D, at), cache_of(B, kv, D, at)
    args = [a[n] for n in ("x", "w", "b", "norm", "cos", "sin")]
    got = ops.attend_few(*args, here, a["wo"], a["bo"], a["res"], heads, D ** -0.5, 0.0, 0)
    fits = ops.one_round(a["x"], (a["w"].shape[0], H, None), (H, heads * D, None))
    assert ops.more_tokens(a["x"]) and (got is not None) == fits
    if got is None:
        assert B * T * a["w"].shape[0] > 384 * 1024 and here.offset == at
        return
    want = one_by_one(*args, there, a["wo"], a["bo"], a["res"], heads, D ** -0.5, 0.0, 0)
    # rows of the norm are rounded once, there before the product, here behind the norm's
    # weights: 2^-8 of each term, of H like ones in a sum
    for one, two in ((here.k, there.k), (here.v, there.v), (got, want)):
        assert one.shape == two.shape
        assert float((one.double() - two.double()).norm() / two.double().norm()) < 2.0 ** -7
    assert here.offset == there.offset == at + T


@torch.no_grad()
@pytest.mark.parametrize("M", [65, 129, 200, 384])
@pytest.mark.parametrize("H,I", [(512, 512), (2048, 5632), (1056, 800)])
@pytest.mark.parametrize("normed,added", [(True, True), (False, False), (True, False)])
def test_feed_forward(M, H, I, normed, added):
    g = torch.Generator("cuda").manual_seed(M + I)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()  # noqa: E731
    x, w_in, w_out = rand(M, H), rand(2 * I, H) / H ** 0.5, rand(H, I) / I ** 0.5
    norm = types.SimpleNamespace(weight=rand(H), eps=1e-5, weight_offset=0.5) if normed else None
    res = rand(M, H) if added else None
    got = ops.feed_few(x, w_in, w_out, "silu", norm, res)
    if got is None:
        assert not ops.one_round(x, (I, H, "silu"), (H, I, None))
        return
    a = x.double()
    if normed:
        a = (a * (a.square().mean(-1, keepdim=True) + 1e-5).rsqrt()
             * (norm.weight.double() + 0.5))
    gate, up = (a @ w_in.double().T).chunk(2, -1)
    want = (F.silu(gate) * up) @ w_out.double().T + (res.double() if added else 0.0)
    # rows, units and the result are rounded to bf16
    assert float((got.double() - want).norm() / want.norm()) < 3 * 2.0 ** -9 * 1.5


def test_layers():
    """A model's layers with and without a hook that has them call their modules."""
    from mlx_sharding_amd.config import ModelConfig
    from mlx_sharding_amd.models.fuse import fuse_model
    from mlx_sharding_amd.models.llama import LlamaStageModel
    cfg = ModelConfig.from_dict({
        "model_type": "llama", "hidden_size": 512, "intermediate_size": 1024,
        "num_hidden_layers": 2, "num_attention_heads": 8, "num_key_value_heads": 2,
        "vocab_size": 256, "rms_norm_eps": 1e-6})
    torch.manual_seed(3)
    with torch.device("cuda"):
        model = LlamaStageModel(cfg, cfg.shard(0, 2))
    for p in model.parameters():
        p.data.normal_(0, 0.05)
    model = model.eval().requires_grad_(False)
    fuse_model(model)
    for B, T in ((1, 70), (3, 40), (1, 385)):
        tokens = torch.randint(0, 256, (B, T), device="cuda")
        outs = []
        for hook in (False, True):
            held = [m.register_forward_hook(lambda *a: None) for layer in
                    model.model.layers.values() for m in (layer.self_attn, layer.mlp)
                    ] if hook else []
            with torch.no_grad():
                outs.append(model(tokens, model.make_cache(batch_size=B)).double())
            for h in held:
                h.remove()
        assert float((outs[0] - outs[1]).norm() / outs[1].norm()) < 0.02

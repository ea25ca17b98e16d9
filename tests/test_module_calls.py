"""Modules that something hooks into or replaces are called, however few tokens come."""

import pytest
import torch

from mlx_sharding_amd.config import ModelConfig
from mlx_sharding_amd.models import deepseek_v2, gemma2, get_model_class, llama
from mlx_sharding_amd.models.base import as_built
from mlx_sharding_amd.models.fuse import fuse_model
from mlx_sharding_amd.ops.kvcache import KVCache

BASE = {"hidden_size": 256, "num_attention_heads": 4, "num_key_value_heads": 2,
        "head_dim": 64, "intermediate_size": 512, "sliding_window": 4096,
        "query_pre_attn_scalar": 64}
LATENT = {"hidden_size": 256, "num_attention_heads": 16, "kv_lora_rank": 512,
          "qk_nope_head_dim": 128, "qk_rope_head_dim": 64, "v_head_dim": 128,
          "intermediate_size": 512, "moe_intermediate_size": 128,
          "num_experts_per_tok": 2, "n_shared_experts": 1}


def a_layer(kind, fused, device="cuda"):
    """(layer, its cache, dimensions that are turned)"""
    if kind in ("llama", "gemma2"):
        cfg = ModelConfig.from_dict({"model_type": kind, **BASE})
        with torch.device(device):
            layer = (llama.LlamaDecoderLayer(cfg, lambda p: None, "m")
                     if kind == "llama" else
                     gemma2.Gemma2DecoderLayer(cfg, lambda p: None, "m", 0))
        cache, rope = KVCache(2, 64, 64, device=device), 64
    else:
        raw = {"model_type": "deepseek_v2", **LATENT}
        if kind == "experts":
            raw.update(n_routed_experts=8, first_k_dense_replace=0)
        with torch.device(device):
            layer = deepseek_v2.DeepseekV2DecoderLayer(
                ModelConfig.from_dict(raw), lambda p: None, "m", 0)
        cache, rope = KVCache(1, 576, 0, device=device), 64
    torch.manual_seed(0)
    for name, p in layer.named_parameters():
        p.data.normal_(1.0 if "layernorm" in name else 0.0, 0.05)
    if fused:
        fuse_model(layer)
    return layer, cache, rope


def steps(layer, cache, rope, device="cuda"):
    """A prompt of many tokens, one of few, one token."""
    out = []
    for T in (140, 9, 1):
        torch.manual_seed(T)
        x = torch.randn(1, T, 256, device=device).bfloat16()
        angle = torch.rand(T, rope // 2, device=device)
        out.append(layer(x, torch.cos(angle), torch.sin(angle), cache))
    return out


KINDS = ["llama", "gemma2", "dense latent", "experts"]


@pytest.mark.gpu
@torch.no_grad()
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("kind", KINDS)
def test_hooks_see_few_tokens_as_many(kind, fused):
    """Each module is called with its input alone, as it is for many tokens."""
    plain = steps(*a_layer(kind, fused))
    layer, cache, rope = a_layer(kind, fused)
    calls = []

    def note(name):
        def hook(module, args, result):
            calls[-1][name] = len(args)
        return hook

    for name, m in layer.named_modules():
        if name:
            m.register_forward_hook(note(name))
    got = []
    for T in (140, 9, 1):
        torch.manual_seed(T)
        x = torch.randn(1, T, 256, device="cuda").bfloat16()
        angle = torch.rand(T, rope // 2, device="cuda")
        calls.append({})
        got.append(layer(x, torch.cos(angle), torch.sin(angle), cache))
    # up to 128 tokens' routed experts, and the projection of cached latents for one
    # token, have never been calls
    optional = {"mlp.switch_mlp", "self_attn.kv_b_proj"}
    names = set(calls[0]) - optional
    assert "self_attn.o_proj" in names and "mlp" in names
    for seen in calls[1:]:
        assert set(seen) - optional == names
        assert seen["mlp"] == 1 and seen["self_attn"] == 4
    for y, expect in zip(got, plain):
        assert (y.double() - expect.double()).norm() < 0.02 * expect.double().norm()


@pytest.mark.gpu
@torch.no_grad()
@pytest.mark.parametrize("kind", KINDS)
def test_replaced_modules_run(kind):
    """Projections and norms in a wrapper's place, without weights to read."""
    class Twice(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, x):
            return self.inner(x) * 2

    layer, cache, rope = a_layer(kind, True)
    layer.self_attn.o_proj = Twice(layer.self_attn.o_proj)
    layer.input_layernorm = Twice(layer.input_layernorm)
    if kind == "experts":
        layer.mlp.gate = Twice(layer.mlp.gate)
        layer.mlp.gate.weight = layer.mlp.gate.inner.weight
        layer.mlp.shared_experts.down_proj = Twice(layer.mlp.shared_experts.down_proj)
    else:
        layer.mlp.down_proj = Twice(layer.mlp.down_proj)
    same, theirs, _ = a_layer(kind, True)
    same.self_attn.o_proj.weight.mul_(2)
    norm = same.input_layernorm
    norm.weight.copy_(norm.weight * 2 + norm.weight_offset)
    if kind == "experts":
        same.mlp.gate.weight.mul_(2)
        same.mlp.shared_experts.down_proj.weight.mul_(2)
    else:
        same.mlp.down_proj.weight.mul_(2)
    for y, expect in zip(steps(layer, cache, rope), steps(same, theirs, rope)):
        assert (y.double() - expect.double()).norm() < 0.02 * expect.double().norm()


def test_as_built():
    layer, _, _ = a_layer("llama", False, "cpu")
    proj, norm = layer.self_attn.o_proj, layer.input_layernorm
    assert as_built(proj, norm, layer.mlp, layer.self_attn)
    assert not as_built(torch.nn.Linear(2, 2))
    for register in (proj.register_forward_hook, proj.register_forward_pre_hook,
                     proj.register_full_backward_hook,
                     torch.nn.modules.module.register_module_forward_hook):
        handle = register(lambda *a: None)
        assert not as_built(norm, proj)
        handle.remove()
        assert as_built(norm, proj)
    proj.forward = lambda x: x
    assert not as_built(norm, proj)


@torch.no_grad()
@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("kind", ["llama", "experts"])
def test_replaced_head_runs(kind, device):
    """A head of another class, which need not say what it takes and gives."""
    raw = ({"model_type": "llama", **BASE} if kind == "llama" else
           {"model_type": "deepseek_v2", **LATENT, "n_routed_experts": 8})
    config = ModelConfig.from_dict({**raw, "num_hidden_layers": 1, "vocab_size": 64})
    with torch.device(device):
        model = get_model_class(config.model_type)(config, config.shard(0, 1))
    torch.manual_seed(0)
    for name, p in model.named_parameters():
        p.data.normal_(1.0 if "norm" in name else 0.0, 0.05)
    tokens = torch.arange(5, device=device)[None]
    want = model(tokens).float()
    head, model.lm_head = model.lm_head, torch.nn.Identity()
    got = model(tokens)
    assert got.shape == (1, 5, 256)
    got = torch.nn.functional.linear(got, head.weight).float()
    # the normed row is rounded to bf16 on both sides, or its factor is applied behind
    assert (got - want).norm() < 8e-3 * want.norm()


@torch.no_grad()
@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("kind", ["llama", "gemma2"])
@pytest.mark.parametrize("T", [1, 9, 100])
def test_attention_alone_calls_its_output(kind, T, device):
    """An attention that is given the norm of its rows, with a hook on its output's
    projection, and with a module of another class there."""
    layer, cache, rope = a_layer(kind, True, device)
    attn, norm = layer.self_attn, layer.input_layernorm
    torch.manual_seed(T)
    x = torch.randn(1, T, 256, device=device).bfloat16()
    angle = torch.rand(T, rope // 2, device=device)

    def call():
        return attn(x, torch.cos(angle), torch.sin(angle), KVCache(2, 64, 64, device=device), norm)

    want = call().double()
    handle = attn.o_proj.register_forward_hook(lambda m, args, y: y * 2)
    hooked = call().double()
    handle.remove()
    attn.o_proj = Halved(attn.o_proj)
    for got in (hooked / 2, call().double() * 2):
        assert (got - want).norm() < 0.02 * want.norm()


class Halved(torch.nn.Module):
    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward(self, x):
        return self.inner(x) * 0.5


@torch.no_grad()
def test_replaced_shared_experts_are_not_read():
    layer, _, _ = a_layer("experts", True, "cpu")
    layer.mlp.shared_experts = Halved(layer.mlp.shared_experts)
    assert layer.mlp._beside(torch.zeros(1, 256, dtype=torch.bfloat16)) is None


@pytest.mark.gpu
@torch.no_grad()
def test_replaced_shared_experts_run():
    layer, cache, rope = a_layer("experts", True)
    layer.mlp.shared_experts = Halved(layer.mlp.shared_experts)
    same, theirs, _ = a_layer("experts", True)
    same.mlp.shared_experts.down_proj.weight.mul_(0.5)
    for y, expect in zip(steps(layer, cache, rope), steps(same, theirs, rope)):
        assert (y.double() - expect.double()).norm() < 0.02 * expect.double().norm()


class Rows:
    """A cache of a program's own: what a layer needs of one on the CPU."""
    graph_pos = None

    def __init__(self):
        self.offset, self.k, self.v = 0, [], []

    def update(self, k, v):
        self.offset += k.shape[2]
        self.k.append(k)
        self.v.append(v)
        return torch.cat(self.k, 2), torch.cat(self.v, 2)


class Noted(KVCache):
    def append_rope_qkv(self, q, *rest):
        self.seen = getattr(self, "seen", 0) + q.shape[1]
        return super().append_rope_qkv(q, *rest)


@torch.no_grad()
@pytest.mark.parametrize("kind", ["llama", "gemma2"])
def test_other_caches_on_the_cpu(kind):
    want = steps(*a_layer(kind, False, "cpu"), device="cpu")
    layer, _, rope = a_layer(kind, False, "cpu")
    for y, expect in zip(steps(layer, Rows(), rope, "cpu"), want):
        assert torch.equal(y, expect)


@pytest.mark.gpu
@torch.no_grad()
@pytest.mark.parametrize("kind", ["llama", "gemma2"])
def test_caches_with_methods_of_their_own(kind):
    layer, _, rope = a_layer(kind, True)
    cache = Noted(2, 64, 64, device="cuda")
    for y, expect in zip(steps(layer, cache, rope), steps(*a_layer(kind, True))):
        assert (y.double() - expect.double()).norm() < 0.02 * expect.double().norm()
    assert cache.seen == cache.offset == 150


@torch.no_grad()
@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("where", ["class", "instance"])
def test_rotations_of_a_models_own(where, device, monkeypatch):
    """A captured step's rotations are those that the model's rope_for gives."""
    def own(self, cache0, T, device):
        cos, sin, offset = llama.LlamaStageModel.rope_for(self, cache0, T, device)
        return cos + 1.0, sin, offset

    class Other(llama.LlamaStageModel):
        rope_for = own

    config = ModelConfig.from_dict({"model_type": "llama", **BASE,
                                    "num_hidden_layers": 1, "vocab_size": 64})
    cls = Other if where == "class" else llama.LlamaStageModel
    with torch.device(device):
        model = cls(config, config.shard(0, 1))
    if where == "instance":
        model.rope_for = own.__get__(model)
    if device == "cpu":      # as the kernel would, were it asked
        monkeypatch.setattr(llama.ops, "step_begin",
                            lambda x, table, scale, pos, cos, sin:
                            (table[x], cos[pos], sin[pos]))
    cache = model.make_cache()
    cache[0].ensure_capacity(16, 1)
    cache[0].graph_pos = torch.tensor([5], dtype=torch.int32, device=device)
    x = torch.tensor([[3]], device=device)
    h, cos, sin = model.begin(x, cache, model.model.embed_tokens)
    want = model.rope_for(cache[0], 1, torch.device(device))
    assert torch.equal(cos, want[0]) and torch.equal(sin, want[1])
    assert torch.equal(h, model.model.embed_tokens(x))

"""What a user of this framework has it do, as cases whose time is measured.

Three kinds of work, each through the entry points that the servers and the
benchmark use:

  prompt   one stage of a pipeline takes a prompt's hidden states (fresh cache,
           optionally in chunks) and hands on those of the next stage
  decode   one graph-captured decoding step of a model over cached sequences,
           with the logits a server samples from
  batches  a continuously batched service: prompts of many lengths arrive, are
           prefilled while others decode, and end

Models are the presets' own sizes.  A stage is one eighth (or quarter) of its
model, as on a node; the models of the other two kinds are cut to a few layers
with the vocabulary cut alike, so that the head keeps its share of the time.
Weights are random: norms around one, recurrences with slow and fast decays.
"""

from __future__ import annotations

import math
import random
from dataclasses import dataclass, field
from typing import Any, Dict, List

import torch

from mlx_sharding_amd.config import ModelConfig
from mlx_sharding_amd.models import get_model_class
from mlx_sharding_amd.models.base import RMSNorm
from mlx_sharding_amd.models.fuse import fuse_model
from mlx_sharding_amd.parallel.batching import BatchEngine, Portion
from mlx_sharding_amd.parallel.rccl import (CapturedDecode, PipelineWorker,
                                            split_layers)
from mlx_sharding_amd.utils.presets import PRESETS, get_preset

F64 = torch.float64

# preset -> (stages of its pipeline, layers and vocabulary where it is cut)
MODELS = {
    "llama-3-8b": (8, 4, 16032),
    "tinyllama-1.1b": (8, 3, 4000),
    "qwen2-7b": (8, 4, 21720),
    "gemma-2-9b": (8, 6, 32000),
    "deepseek-v2-lite": (8, 4, 12800),
    "tuvutar-2b": (4, 7, 8000),
    "dufinex-7b": (3, 8, 10000),
}


# -- cases ------------------------------------------------------------------

def listed() -> List[dict]:
    return [
        # one user's chat: every token waits for a whole step
        _decode("llama decode one sequence", "llama-3-8b", 1, 1023),
        # a busy server: 64 conversations of 2048 tokens
        _decode("llama decode 64 sequences", "llama-3-8b", 64, 2048),
        # a few long conversations, past the sliding window of half the layers
        _decode("gemma decode long", "gemma-2-9b", 5, 5003),
        # the serving benchmark: 4-bit weights, 64 sequences behind prompts of 512
        _decode("deepseek 4-bit decode 64", "deepseek-v2-lite", 64, 512, 4),
        # the same model for one user in a long conversation
        _decode("deepseek 4-bit decode one", "deepseek-v2-lite", 1, 3001, 4),
        # a question of a few words
        _prompt("tinyllama short prompt", "tinyllama-1.1b", 1, 57),
        # a document that fills the context
        _prompt("llama long prompt", "llama-3-8b", 1, 8192),
        # a long document in chunks, past the sliding window
        _prompt("gemma chunked prompt", "gemma-2-9b", 1, 6001, chunk=4096),
        # the serving benchmark's prompts
        _prompt("deepseek 4-bit 64 prompts", "deepseek-v2-lite", 64, 512, 4),
        # recurrent and latent-attention layers over long documents
        _prompt("tuvutar long prompts", "tuvutar-2b", 2, 4001),
        # services under mixed load
        _batches("tuvutar service", "tuvutar-2b", 12, 17, 1300, 6),
        _batches("dufinex service", "dufinex-7b", 16, 9, 900, 6),
    ]


def draw(rng: random.Random) -> dict:
    kind = rng.choice(("prompt", "decode", "batches"))
    if kind == "batches":
        shortest = _spread(rng, 5, 300)
        case = _batches("", rng.choice(("tuvutar-2b", "dufinex-7b")),
                        _spread(rng, 2, 24), shortest,
                        min(1200, shortest + _spread(rng, 10, 1100)),
                        rng.randint(2, 8))
    elif kind == "decode":
        model = rng.choice(("llama-3-8b", "tinyllama-1.1b", "qwen2-7b",
                            "gemma-2-9b", "deepseek-v2-lite"))
        batch = _spread(rng, 1, 64)
        case = _decode("", model, batch, _spread(rng, 16, min(8000, 98304 // batch)),
                       _bits(rng, model))
    else:
        model = rng.choice(("llama-3-8b", "tinyllama-1.1b", "qwen2-7b",
                            "gemma-2-9b", "deepseek-v2-lite", "tuvutar-2b",
                            "dufinex-7b"))
        tokens = _spread(rng, 20, 6000)
        case = _prompt("", model, rng.randint(1, max(1, min(32, 6000 // tokens))),
                       tokens, _bits(rng, model),
                       rng.choice((0, 0, 512, 1000, 2048)))
    del case["name"]
    return case


def _spread(rng: random.Random, lo: int, hi: int) -> int:
    """Evenly over the logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _bits(rng: random.Random, model: str) -> int:
    return rng.choice((4, 4, 8, 0)) if model.startswith("deepseek") else 0


def _decode(name, model, batch, cached, bits=0):
    return {"name": name, "kind": "decode", "model": model, "bits": bits,
            "batch": batch, "cached": cached}


def _prompt(name, model, batch, tokens, bits=0, chunk=0):
    return {"name": name, "kind": "prompt", "model": model, "bits": bits,
            "batch": batch, "tokens": tokens, "chunk": chunk}


def _batches(name, model, requests, shortest, longest, steps):
    return {"name": name, "kind": "batches", "model": model, "bits": 0,
            "requests": requests, "shortest": shortest, "longest": longest,
            "steps": steps}


def _lengths(case: dict) -> List[int]:
    """Prompt lengths of a service, spread evenly over their logarithm and
    in no order."""
    n, lo, hi = case["requests"], case["shortest"], case["longest"]
    found = [round(lo * (hi / lo) ** (i / (n - 1))) for i in range(n)]
    random.Random(n).shuffle(found)
    return found


# -- models -----------------------------------------------------------------

def _config(case: dict) -> ModelConfig:
    config = get_preset(case["model"], quant=bool(case["bits"]),
                        bits=case["bits"] or 4)
    if case["kind"] != "prompt":
        _, layers, vocab = MODELS[case["model"]]
        raw = config.raw
        if "layers" in raw:
            raw["layers"], raw["vocab"] = raw["layers"][:layers], vocab
        else:
            raw["num_hidden_layers"], raw["vocab_size"] = layers, vocab
    return config


def _stage(case: dict, config: ModelConfig, device: torch.device):
    """The case's model without values, on ``device``."""
    cls = get_model_class(config.model_type)
    n = config.num_hidden_layers
    first, end = 0, n
    if case["kind"] == "prompt":
        stages = MODELS[case["model"]][0]
        first, end = split_layers(n, stages, cls.allowed_cuts(config))[1]
    quant = config.quantization
    with torch.device(device):
        return cls(config, config.shard(first, end),
                   quant_for=(lambda prefix: quant) if quant else None)


@torch.no_grad()
def _model(case: dict, seed: int):
    """The case's model with the seed's weights."""
    device = torch.device("cuda", torch.cuda.current_device())
    model = _stage(case, _config(case), device)
    gen = torch.Generator(device).manual_seed(seed)
    for name, p in model.named_parameters():
        if not p.is_floating_point():
            p.data.copy_(torch.randint(0, 2 ** 32, p.shape, generator=gen,
                                       device=device).to(p.dtype))
            continue
        leaf = name.rsplit(".", 1)[-1]
        mean, std = {"scales": (0.0, 0.0025 if case["bits"] == 4 else 0.00016),
                     "biases": (0.0, 0.005), "A_log": (0.5, 0.7),
                     "dt_bias": (-3.0, 1.0), "sink": (0.0, 1.0),
                     "bias": (0.0, 0.1)}.get(leaf, (0.0, 0.02))
        if name.endswith(".conv.weight"):
            std = 0.5
        p.data.normal_(mean, std, generator=gen)
    for m in model.modules():
        if isinstance(m, RMSNorm):
            m.weight.data.normal_(1.0 - m.weight_offset, 0.1, generator=gen)
    if case["model"] == "dufinex-7b":
        _route_by_topic(model, seed)
    return model.eval()


def _topics(width: int, seed: int) -> torch.Tensor:
    gen = torch.Generator("cuda").manual_seed(seed + 4)
    return torch.randint(0, 2, (64, width), generator=gen, device="cuda") * 2.0 - 1.0


def _route_by_topic(model, seed: int):
    """Tokens of one topic share a direction and routers choose by it, as
    trained ones do.  Random routers choose between experts that are nearly
    tied, and as what experts give is normed here, a tie that falls the other
    way in bf16 changes a whole row."""
    topics = _topics(model.config.hidden_size, seed)
    gen = torch.Generator("cuda").manual_seed(seed + 5)
    for name, p in model.named_parameters():
        if name == "embed.weight":
            at = torch.arange(p.shape[0], device="cuda") % 64
            p.data.add_(0.02 * topics[at].to(p.dtype))
        elif name.endswith("router.weight"):
            # every expert has six topics, every topic six experts
            order = torch.randperm(64, generator=gen, device="cuda")
            choice = torch.zeros(64, 64, device="cuda")
            for j in range(6):
                choice[order.roll(j), torch.arange(64, device="cuda")] = 2.0 + 0.2 * j
            p.data.copy_(choice @ topics / topics.shape[1])


# -- what a user's program has in hand, and the pass ------------------------

@dataclass
class State:
    kind: str
    model: Any
    chunk: int = 0
    x: Any = None                 # prompt: hidden states
    graph: Any = None             # decode: the captured step
    tokens: Any = None            # ... and what it is given
    engine: Any = None            # batches
    prompts: List[List[int]] = field(default_factory=list)
    replies: List[List[int]] = field(default_factory=list)


def _hidden(case: dict, seed: int, width: int, dtype: torch.dtype) -> torch.Tensor:
    """Hidden states as a first stage hands them on."""
    gen = torch.Generator("cuda").manual_seed(seed + 1)
    x = torch.randn(case["batch"], case["tokens"], width, generator=gen,
                    device="cuda")
    if case["model"] == "dufinex-7b":
        x += _topics(width, seed)[torch.randint(
            0, 64, x.shape[:2], generator=gen, device="cuda")]
    return x.to(dtype)


def _cached(case: dict, seed: int, specs):
    """Per layer the rows cached so far: keys (rotated) and values, or a
    latent with its rotated part; all are of unit size, as behind norms."""
    gen = torch.Generator("cuda").manual_seed(seed + 2)
    new = lambda h, d: torch.randn(  # noqa: E731
        case["batch"], h, case["cached"], d, generator=gen, device="cuda",
        dtype=torch.bfloat16)
    return [(new(h, kd), new(h, vd)) for h, kd, vd in specs]


def _next_tokens(case: dict, seed: int) -> torch.Tensor:
    gen = torch.Generator("cuda").manual_seed(seed + 3)
    return torch.randint(0, MODELS[case["model"]][2], (case["batch"],),
                         generator=gen, device="cuda")


def _requests(case: dict, seed: int):
    """Prompts, and the tokens that follow each of them."""
    rng, vocab = random.Random(seed), MODELS[case["model"]][2]
    new = lambda n: [rng.randrange(vocab) for _ in range(n)]  # noqa: E731
    return ([new(n) for n in _lengths(case)],
            [new(case["steps"] + 1) for _ in range(case["requests"])])


def prepare(case: dict, seed: int) -> State:
    model = _model(case, seed)
    fuse_model(model)
    state = State(case["kind"], model)
    if case["kind"] == "prompt":
        state.chunk = case["chunk"] or case["tokens"]
        state.x = _hidden(case, seed, model.hop_width, model.hop_dtype)
    elif case["kind"] == "decode":
        batch, device = case["batch"], next(model.parameters()).device
        worker = PipelineWorker(model, 0, 1, device)
        worker.reset(1, batch)
        for cache, (k, v) in zip(worker.caches[0],
                                 _cached(case, seed, model.cache_specs())):
            cache.update(k, v)
        state.tokens = [_next_tokens(case, seed)]
        # room for a reply of 256 tokens
        state.graph = CapturedDecode(worker, batch, 1, case["cached"] + 256,
                                     return_logits=True)
    else:
        state.prompts, state.replies = _requests(case, seed)
        pages = sum(-(-(len(p) + case["steps"] + 2) // 64) for p in state.prompts)
        state.engine = BatchEngine(model, 64 * pages, case["requests"])
    return state


def run(state: State):
    if state.kind == "prompt":
        cache = state.model.make_cache(batch_size=state.x.shape[0])
        with torch.no_grad():
            return [state.model(x, cache) for x in state.x.split(state.chunk, 1)]
    if state.kind == "decode":
        state.graph.rearm()
        state.graph.seed(state.tokens)
        return state.graph.decode_step(state.tokens)
    engine, prompts, replies = state.engine, state.prompts, state.replies
    last = len(prompts) - 1
    whole = [Portion(i, p, [len(p) - 1]) for i, p in enumerate(prompts)]
    said = lambda i, j: Portion(i, [replies[i][j]], [0])  # noqa: E731
    # all prompts but one; that one while the others decode; all decode
    out = [engine.step(whole[:last]),
           engine.step([*(said(i, 0) for i in range(last)), whole[last]])]
    for j in range(1, len(replies[0])):
        out.append(engine.step([*(said(i, j) for i in range(last)),
                                said(last, j - 1)]))
    for i in range(last + 1):
        engine.end(i)
    return out


# -- what a pass cannot do without ------------------------------------------

def _counts(case: dict):
    """((bytes, values) of the matrices that every token meets, those of all
    routed experts, share of the experts that a token meets)."""
    config = _config(case)
    bits, dense, routed = case["bits"], [0, 0], [0, 0]
    model = _stage(case, config, torch.device("meta"))
    tied = case["kind"] != "prompt" and not any(
        "head" in n for n, _ in model.named_parameters())
    for name, p in model.named_parameters():
        if "embed" in name and not tied:
            continue            # rows are looked up
        to = routed if p.dim() == 3 else dense
        to[0] += p.numel() * p.element_size()
        if p.dim() > 1 and not name.endswith((".scales", ".biases")):
            to[1] += p.numel() * (1 if p.is_floating_point() else 32 // bits)
    raw, share = config.raw, 0.0
    if routed[1]:
        share = 6 / 64
        assert raw.get("n_routed_experts", 64) == 64
    return dense, routed, share, config


def _mixing(config: ModelConfig, first: int, end: int, lengths, new):
    """(bytes of cached rows and states read, flops) of the mixers where
    sequences of ``lengths`` tokens get their last ``new`` ones."""
    bytes_, flops, raw = 0.0, 0.0, config.raw
    for i in range(first, end):
        if "layers" in raw:
            mx, kind = raw["layers"][i]["mixer"], raw["layers"][i]["type"]
        elif "kv_lora_rank" in raw:
            mx, kind = {"heads": raw["num_attention_heads"], "dim": 128,
                        "rot_dim": 64, "vdim": 128, "kv_rank": 512}, "latent_attention"
        else:
            heads = raw["num_attention_heads"]
            dim = raw.get("head_dim") or raw["hidden_size"] // heads
            mx, kind = {"heads": heads, "kv_heads": raw["num_key_value_heads"],
                        "dim": dim, "vdim": dim}, "attention"
        window = raw.get("sliding_window", 0) if i % 2 == 0 else 0
        for n, m in zip(lengths, new):
            if "delta" in kind:
                state = mx["heads"] * mx["dim"] * mx["vdim"]
                bytes_ += 8 * state
                flops += 7 * state * m
                continue
            keys = min(n, window) if window else n
            pairs = m * keys - (0 if window and n > window else m * (m - 1) / 2)
            width = mx["dim"] + mx.get("rot_dim", 0) + mx["vdim"]
            row = (mx["kv_rank"] + mx["rot_dim"] if kind == "latent_attention"
                   else mx["kv_heads"] * width)
            bytes_ += 2 * row * keys
            flops += 2 * mx["heads"] * width * pairs
    return bytes_, flops


def work(case: dict) -> Dict[str, float]:
    dense, routed, share, config = _counts(case)
    width, vocab = config.hidden_size, config.vocab_size
    if case["kind"] == "prompt":
        cls = get_model_class(config.model_type)
        first, end = split_layers(config.num_hidden_layers, MODELS[case["model"]][0],
                                  cls.allowed_cuts(config))[1]
        B, T = case["batch"], case["tokens"]
        steps = [([T] * B, [T] * B)]
        ends = B * T * width * (8 if "layers" in config.raw else 4)
    else:
        first, end = 0, config.num_hidden_layers
        if case["kind"] == "decode":
            B = case["batch"]
            steps = [([case["cached"] + 1] * B, [1] * B)]
        else:
            n, R = _lengths(case), case["requests"]
            steps = [(n[:-1], n[:-1]),
                     ([x + 1 for x in n[:-1]] + n[-1:], [1] * (R - 1) + n[-1:])]
            steps += [([x + 1 + j for x in n], [1] * R)
                      for j in range(1, case["steps"] + 1)]
        ends = 0
    bytes_, flops = float(ends), 0.0
    head = 0 if case["kind"] == "prompt" else width * vocab
    for lengths, new in steps:
        N = sum(new)
        met = 1.0 - (1.0 - share) ** N if share else 0.0
        moved, mixed = _mixing(config, first, end, lengths, new)
        bytes_ += dense[0] + met * routed[0] + moved + 4 * len(new) * vocab * bool(head)
        flops += (2 * N * (dense[1] - head + share * routed[1])
                  + 2 * len(new) * head + mixed)
    return {"bytes": bytes_, "flops": flops}


def tolerance(case: dict):
    """About four times what bf16 passes are off from 64 bits (measured: 0.7 to
    1.3% of hidden states, 1.0 to 1.6% of logits behind captured steps, up to
    2.2% of logits behind whole prompts)."""
    return {"rel": {"prompt": 0.04, "decode": 0.06, "batches": 0.08}[case["kind"]]}


# -- the same in 64 bits ----------------------------------------------------

@torch.no_grad()
def exact(case: dict, seed: int):
    model = _model(case, seed)
    P = dict(model.named_parameters())
    first, end = model.shard.start_layer, model.shard.end_layer
    config, layers = model.config, range(first, end)
    forward = {"tuvutar": _tuvutar, "dufinex": _dufinex, "gemma2": _gemma,
               "deepseek_v2": _deepseek}.get(config.model_type, _llama)
    net = _Net(P, config.raw, case["bits"])
    if case["kind"] == "prompt":
        x = _hidden(case, seed, model.hop_width, model.hop_dtype).to(F64)
        y = torch.stack([forward(net, s, layers) for s in x])
        return list(y.split(case["chunk"] or case["tokens"], 1))
    if case["kind"] == "decode":
        rows = [(k.transpose(1, 2).to(F64), v.transpose(1, 2).to(F64))
                for k, v in _cached(case, seed, model.cache_specs())]
        tokens = _next_tokens(case, seed)
        return [_head(net, torch.cat([
            forward(net, _embed(net, t[None]), layers,
                    [(k[b], v[b]) for k, v in rows])
            for b, t in enumerate(tokens)]))]
    prompts, replies = _requests(case, seed)
    ends = []
    for p, r in zip(prompts, replies):
        x = forward(net, _embed(net, torch.tensor(p + r, device="cuda")), layers)
        ends.append(_head(net, x[len(p) - 1:]))
    last = len(prompts) - 1
    out = [torch.stack([e[0] for e in ends[:last]])]
    out.append(torch.stack([e[1] for e in ends[:last]] + [ends[last][0]]))
    for j in range(1, len(replies[0])):
        out.append(torch.stack([e[j + 1] for e in ends[:last]] + [ends[last][j]]))
    return out


class _Net:
    """Weights by name, in 64 bits."""

    def __init__(self, P, raw, bits):
        self.P, self.raw, self.bits = P, raw, bits
        self.kept: Dict[str, torch.Tensor] = {}

    def has(self, name):
        return name in self.P

    def mat(self, name, e=None):
        key = f"{name}.{e}"
        if key in self.kept:
            return self.kept[key]
        pick = lambda leaf: self.P[f"{name}.{leaf}"][... if e is None else e]  # noqa: E731
        w = pick("weight")
        if f"{name}.scales" in self.P:
            words = w.view(torch.int32).to(torch.int64)
            shifts = torch.arange(0, 32, self.bits, device=w.device)
            q = (words[..., None] >> shifts) & ((1 << self.bits) - 1)
            scales = pick("scales").to(F64)
            q = q.reshape(*scales.shape, -1).to(F64)
            w = (q * scales[..., None] + pick("biases").to(F64)[..., None]).flatten(-2)
        self.kept[key] = w.to(F64)
        return self.kept[key]

    def vec(self, name):
        return self.P[name].to(F64)

    def lin(self, name, x, e=None):
        y = x @ self.mat(name, e).T
        return y + self.vec(name + ".bias") if self.has(name + ".bias") else y


def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _unit(x):
    return x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)


def _silu(x):
    return x * torch.sigmoid(x)


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _embed(net, tokens):
    raw = net.raw
    if "layers" in raw:
        x = net.P["embed.weight"][tokens].to(F64)
        return x * raw.get("embedding", {}).get("scale", 1.0)
    x = net.P["model.embed_tokens.weight"][tokens].to(F64)
    if raw["model_type"] == "gemma2":  # the factor is a bf16 number
        x = x * torch.tensor(raw["hidden_size"] ** 0.5, dtype=torch.bfloat16).item()
    return x


def _head(net, x):
    raw = net.raw
    if "layers" in raw:
        tied = not net.has("head.weight")
        h = _rms(x, raw["norm"]["eps"]) * (net.vec("final.norm.weight") + (not tied))
        return h @ net.mat("embed" if tied else "head").T
    gemma = raw["model_type"] == "gemma2"
    h = _rms(x, raw["rms_norm_eps"]) * (net.vec("model.norm.weight") + gemma)
    if not gemma:
        return net.lin("lm_head", h)
    cap = raw["final_logit_softcapping"]
    return cap * torch.tanh(h @ net.mat("model.embed_tokens").T / cap)


def _attend(q, k, v, scale, cap=0.0, window=0, sink=None):
    """q [T, H, D], k [S, G, D], v [S, G, E]; the last T of S tokens ask."""
    T, H, S, G = q.shape[0], q.shape[1], k.shape[0], k.shape[1]
    at = torch.arange(S - T, S, device=q.device)[:, None]
    key = torch.arange(S, device=q.device)[None, :]
    hidden = key > at
    if window:
        hidden |= key <= at - window
    out = q.new_empty(T, H, v.shape[-1])
    for h in range(H):
        g = h // (H // G)
        s = (q[:, h] @ k[:, g].T).mul_(scale)
        if cap:
            s = s.div_(cap).tanh_().mul_(cap)
        s.masked_fill_(hidden, -math.inf)
        m = s.amax(-1, keepdim=True)
        extra = 0.0
        if sink is not None:
            m = torch.maximum(m, sink[h])
            extra = torch.exp(sink[h] - m)
        p = s.sub_(m).exp_()
        out[:, h] = (p @ v[:, g]) / (p.sum(-1, keepdim=True) + extra)
    return out


def _turn(x, first, freq, neighbours, factor=1.0):
    """Rotates x [T, H, D] by positions from ``first`` on."""
    at = torch.arange(first, first + x.shape[0], device=x.device, dtype=F64)
    angle = (at[:, None] * freq.to(x.device))[:, None]
    c, s = torch.cos(angle) * factor, torch.sin(angle) * factor
    if neighbours:
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)
    a, b = x.chunk(2, -1)
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _frequencies(dims, base):
    return base ** (-torch.arange(0, dims, 2, dtype=F64) / dims)


def _slowed(freq, dims, base, factor, original, fast, slow):
    """YaRN: slow turns are slowed down, fast ones are kept."""
    place = lambda turns: (dims * math.log(original / (2 * math.pi * turns))  # noqa: E731
                           / (2 * math.log(base)))
    lo = max(math.floor(place(fast)), 0)
    hi = min(math.ceil(place(slow)), dims - 1)
    ramp = ((torch.arange(dims // 2, dtype=F64) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return freq / factor * ramp + freq * (1 - ramp)


def _grouped(net, pre, x, past, window=0, cap=0.0, scale=None):
    raw = net.raw
    H, G = raw["num_attention_heads"], raw["num_key_value_heads"]
    D = raw.get("head_dim") or raw["hidden_size"] // H
    T, n = x.shape[0], 0 if past is None else past[0].shape[0]
    q, k, v = (net.lin(f"{pre}{a}_proj", x).view(T, -1, D) for a in "qkv")
    freq = _frequencies(D, raw["rope_theta"])
    q, k = _turn(q, n, freq, False), _turn(k, n, freq, False)
    if past is not None:
        k, v = torch.cat([past[0], k]), torch.cat([past[1], v])
    o = _attend(q, k, v, scale or D ** -0.5, cap, window)
    return net.lin(f"{pre}o_proj", o.reshape(T, -1))


def _gated(net, pre, x, act):
    return net.lin(pre + "down_proj", act(net.lin(pre + "gate_proj", x))
                   * net.lin(pre + "up_proj", x))


def _llama(net, x, layers, past=None):
    eps = net.raw["rms_norm_eps"]
    for j, i in enumerate(layers):
        p = f"model.layers.{i}."
        h = _rms(x, eps) * net.vec(p + "input_layernorm.weight")
        x = x + _grouped(net, p + "self_attn.", h, past and past[j])
        h = _rms(x, eps) * net.vec(p + "post_attention_layernorm.weight")
        x = x + _gated(net, p + "mlp.", h, _silu)
    return x


def _gemma(net, x, layers, past=None):
    raw = net.raw
    norm = lambda y, name: (_rms(y, raw["rms_norm_eps"])  # noqa: E731
                            * (1 + net.vec(name + "_layernorm.weight")))
    for j, i in enumerate(layers):
        p = f"model.layers.{i}."
        y = _grouped(net, p + "self_attn.", norm(x, p + "input"), past and past[j],
                     raw["sliding_window"] if i % 2 == 0 else 0,
                     raw["attn_logit_softcapping"],
                     raw["query_pre_attn_scalar"] ** -0.5)
        x = x + norm(y, p + "post_attention")
        y = _gated(net, p + "mlp.", norm(x, p + "pre_feedforward"), _gelu)
        x = x + norm(y, p + "post_feedforward")
    return x


def _routed(net, pre, h, scores, top, expert):
    """Sum over each row's ``top`` experts; expert(name, e, rows, weights)."""
    weight, chosen = torch.topk(scores, top, -1)
    y = torch.zeros_like(h)
    for e in range(scores.shape[1]):
        row, place = torch.nonzero(chosen == e, as_tuple=True)
        if len(row):
            y.index_add_(0, row, expert(e, h[row], weight[row, place][:, None]))
    return y


def _deepseek(net, x, layers, past=None):
    raw = net.raw
    eps, H, T = raw["rms_norm_eps"], raw["num_attention_heads"], x.shape[0]
    rank, rope = raw["kv_lora_rank"], raw["qk_rope_head_dim"]
    nope, vd = raw["qk_nope_head_dim"], raw["v_head_dim"]
    yarn = raw["rope_scaling"]
    freq = _slowed(_frequencies(rope, raw["rope_theta"]), rope, raw["rope_theta"],
                   yarn["factor"], yarn["original_max_position_embeddings"],
                   yarn["beta_fast"], yarn["beta_slow"])
    stretch = 0.1 * yarn["mscale_all_dim"] * math.log(yarn["factor"]) + 1.0
    scale = (nope + rope) ** -0.5 * stretch ** 2
    for j, i in enumerate(layers):
        p = f"model.layers.{i}."
        h = _rms(x, eps) * net.vec(p + "input_layernorm.weight")
        a = p + "self_attn."
        n = 0 if past is None else past[j][0].shape[0]
        q = net.lin(a + "q_proj", h).view(T, H, nope + rope)
        q = torch.cat([q[..., :nope], _turn(q[..., nope:], n, freq, True)], -1)
        c = net.lin(a + "kv_a_proj_with_mqa", h)
        pe = _turn(c[:, None, rank:], n, freq, True)
        c = _rms(c[:, :rank], eps) * net.vec(a + "kv_a_layernorm.weight")
        if past is not None:
            old = past[j][0]
            c = torch.cat([old[:, 0, :rank], c])
            pe = torch.cat([old[..., rank:], pe])
        kv = net.lin(a + "kv_b_proj", c).view(-1, H, nope + vd)
        k = torch.cat([kv[..., :nope], pe.expand(-1, H, -1)], -1)
        o = _attend(q, k, kv[..., nope:], scale)
        x = x + net.lin(a + "o_proj", o.reshape(T, -1))
        h = _rms(x, eps) * net.vec(p + "post_attention_layernorm.weight")
        m = p + "mlp."
        if not net.has(m + "gate.weight"):
            x = x + _gated(net, m, h, _silu)
            continue

        def expert(e, rows, weight, s=m + "switch_mlp."):
            u = _silu(net.lin(s + "gate_proj", rows, e)) * net.lin(s + "up_proj", rows, e)
            return weight * net.lin(s + "down_proj", u, e)

        scores = torch.softmax(net.lin(m + "gate", h), -1)
        y = _routed(net, m, h, scores, raw["num_experts_per_tok"], expert)
        x = x + y + _gated(net, m + "shared_experts.", h, _silu)
    return x


def _conv(net, name, x):
    """silu of a causal convolution; the last tap meets the current row."""
    taps = net.mat(name + ".conv")
    K, T = taps.shape[1], x.shape[0]
    x = torch.cat([x.new_zeros(K - 1, x.shape[1]), net.lin(name, x)
                   if x.shape[1] != taps.shape[0] else x])
    return _silu(sum(taps[:, j] * x[j: j + T] for j in range(K)))


def _lanes(net, pre, h, mx):
    """q, k (unit, repeated for the heads that share them) and v."""
    H, KH, D, V = (mx[n] for n in ("heads", "kv_heads", "dim", "vdim"))
    T = h.shape[0]
    q, k, v = (_conv(net, pre + a, net.lin(pre + a, h)) for a in "qkv")
    q = (_unit(q.view(T, KH, D)) * D ** -0.5).repeat_interleave(H // KH, 1)
    k = _unit(k.view(T, KH, D)).repeat_interleave(H // KH, 1)
    return q, k, v.view(T, H, V)


def _delta_rule(q, k, v, beta, g):
    """q, k [T, H, D], v [T, H, V], beta [T, H], g [T, H, D or 1]."""
    S = q.new_zeros(q.shape[1], q.shape[2], v.shape[2])
    out = torch.empty_like(v)
    for t in range(q.shape[0]):
        S = S * g[t][..., None]
        u = beta[t][:, None] * (v[t] - torch.bmm(k[t][:, None], S)[:, 0])
        S = torch.baddbmm(S, k[t][..., None], u[:, None])
        out[t] = torch.bmm(q[t][:, None], S)[:, 0]
    return out


def _tuvutar(net, x, layers):
    eps, T, kept = net.raw["norm"]["eps"], x.shape[0], {}
    norm = lambda y, name: _rms(y, eps) * (1 + net.vec(name + ".weight"))  # noqa: E731
    for i in layers:
        spec = net.raw["layers"][i]
        p, m, mx = f"l{i}.", f"l{i}.mix.", spec["mixer"]
        h = norm(x, p + "norm1")
        if spec["type"] == "delta":
            q, k, v = _lanes(net, m, h, mx)
            beta = torch.sigmoid(net.lin(m + "b", h))
            step = torch.nn.functional.softplus(net.lin(m + "a", h)
                                                + net.vec(m + "dt_bias"))
            g = torch.exp(-torch.exp(net.vec(m + "A_log")) * step)
            o = _rms(_delta_rule(q, k, v, beta, g[..., None]), eps)
            o = o * net.vec(m + "norm.weight") * _silu(net.lin(m + "g", h)).view_as(o)
        else:
            H, dim, rot, r = mx["heads"], mx["dim"], mx["rot_dim"], mx["kv_rank"]
            sc = mx["rot"]["scaling"]
            base = mx["rot"]["base"]
            freq = _slowed(_frequencies(rot, base), rot, base, sc["factor"],
                           sc["original"], sc["fast"], sc["slow"])
            grow = 0.1 * math.log(sc["factor"]) + 1.0
            src = mx.get("kv_from", i)
            if src == i:
                d = net.lin(m + "dkv", h)
                kept[i] = (_rms(d[:, :r], eps) * net.vec(m + "dkv.norm.weight"),
                           _turn(d[:, None, r:], 0, freq, True, grow))
            c, pe = kept[src]
            q = net.lin(m + "q", h).view(T, H, dim + rot)
            q = torch.cat([q[..., :dim], _turn(q[..., dim:], 0, freq, True, grow)], -1)
            k = torch.cat([net.lin(m + "uk", c).view(T, H, dim),
                           pe.expand(-1, H, -1)], -1)
            o = _attend(q, k, net.lin(m + "uv", c).view(T, H, -1), mx["scale"])
        x = x + norm(net.lin(m + "o", o.reshape(T, -1)), p + "norm1b")
        h, f = norm(x, p + "norm2"), p + "mlp."
        y = net.lin(f + "down", _gelu(net.lin(f + "gate", h)) * net.lin(f + "up", h))
        x = x + norm(y, p + "norm2b")
    return x


def _dufinex(net, x, layers):
    eps, T, kept = net.raw["norm"]["eps"], x.shape[0], {}
    norm = lambda y, name: _rms(y, eps) * net.vec(name + ".weight")  # noqa: E731

    def unit(g, u, limit):
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        return g * torch.sigmoid(1.702 * g) * (u + 1.0)

    for i in layers:
        spec = net.raw["layers"][i]
        p, m, mx, mlp = f"l{i}.", f"l{i}.mix.", spec["mixer"], spec["mlp"]
        H = mx["heads"]
        if spec["type"] == "attention":
            src = mx.get("kv_from", i)
            if src == i:
                G = mx["kv_heads"]
                kept[i] = (norm(net.lin(m + "k", x).view(T, G, -1), m + "k.norm"),
                           net.lin(m + "v", x).view(T, G, -1))
            q = norm(net.lin(m + "q", x).view(T, H, -1), m + "q.norm")
            o = _attend(q, *kept[src], mx["scale"], sink=net.vec(m + "sink"))
            o = o * torch.sigmoid(net.lin(m + "g", x))[..., None]
        else:
            q, k, v = _lanes(net, m, x, mx)
            beta = torch.sigmoid(net.lin(m + "b", x))
            step = torch.nn.functional.softplus(
                net.lin(m + "a2", net.lin(m + "a1", x)) + net.vec(m + "dt_bias"))
            rate = torch.exp(net.vec(m + "A_log"))[:, None]
            o = _delta_rule(q, k, v, beta, torch.exp(-rate * step.view(T, H, -1)))
            gate = torch.sigmoid(net.lin(m + "g2", net.lin(m + "g1", x)))
            o = norm(o, m + "norm") * gate.view_as(o)
        x = x + norm(net.lin(m + "o", o.reshape(T, -1)), p + "norm1")
        f = p + "mlp."
        if mlp["kind"] == "dense":
            y = net.lin(f + "down", unit(net.lin(f + "gate", x), net.lin(f + "up", x),
                                         mlp["limit"]))
        else:
            def expert(e, rows, weight, f=f, limit=mlp["expert"]["limit"]):
                rows = rows * weight
                return net.lin(f + "down", unit(net.lin(f + "gate", rows, e),
                                                net.lin(f + "up", rows, e), limit), e)

            scores = torch.sigmoid(net.lin(f + "router", x))
            y = _routed(net, f, x, scores, mlp["router"]["top"], expert)
        x = x + norm(y, p + "norm2")
    return x

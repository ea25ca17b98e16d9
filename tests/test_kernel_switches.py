"""Environment switches that name a kernel have it run for few tokens."""

import pytest
import torch

from mlx_sharding_amd import ops
from test_module_calls import a_layer, steps
from test_moe_rows import decoder_layer, one_position

pytestmark = pytest.mark.gpu


class Spied:
    """The extension, and which of its kernels were called."""

    def __init__(self, ext, seen):
        self.ext, self.seen = ext, seen

    def __getattr__(self, name):
        kernel = getattr(self.ext, name)

        def call(*args, **kwargs):
            result = kernel(*args, **kwargs)
            if result is not None:  # what linear_few_try does not take
                self.seen.append(name)
            return result
        return call


@pytest.fixture
def seen(monkeypatch):
    names = []
    monkeypatch.setattr(ops, "_EXT", Spied(ops.hip_ext(), names))
    return names


@torch.no_grad()
@pytest.mark.parametrize("kind", ["llama", "gemma2"])
def test_dense_gemv(kind, seen, monkeypatch):
    expect = steps(*a_layer(kind, True))
    assert "linear_few_try" in seen
    seen.clear()
    monkeypatch.setenv("MLXS_AMD_DENSE_GEMV", "1")
    for y, z in zip(steps(*a_layer(kind, True)), expect):
        assert (y.double() - z.double()).norm() < 0.02 * z.double().norm()
    # four products for each of the two short inputs
    assert seen.count("dense_gemv") == 8 and "linear_few_try" not in seen


@torch.no_grad()
def test_dense_gemv_of_shared_experts(seen, monkeypatch):
    layer, _, _ = a_layer("experts", True)
    x = torch.randn(1, 1, 256, device="cuda").bfloat16()
    norm = layer.post_attention_layernorm
    expect = layer.mlp.decode(x, None, norm).double()
    assert "moe_rows" in seen and "dense_gemv" not in seen
    seen.clear()
    monkeypatch.setenv("MLXS_AMD_DENSE_GEMV", "1")
    y = layer.mlp.decode(x, None, norm).double()
    assert seen.count("dense_gemv") == 2
    # units and their product are rounded to bf16 on both sides
    assert (y - expect).norm() < 8e-3 * expect.norm()


@torch.no_grad()
@pytest.mark.parametrize("bits", [0, 4])
def test_resident_experts(bits, seen, monkeypatch):
    """Routed experts of packed weights on their bf16 copies; bf16 ones have none."""
    layer, turn = decoder_layer(bits), one_position()
    x = torch.randn(8, 1, 512, device="cuda").bfloat16()
    expect = layer(x, *turn, None).double()
    assert "moe_rows" in seen
    seen.clear()
    monkeypatch.setenv("MLXS_AMD_MOE_RESIDENT", "1")
    y = layer(x, *turn, None).double()
    assert ("moe_gateup_grouped" if bits else "moe_rows") in seen
    assert bits == 0 or "moe_rows" not in seen
    # where two experts are nearly tied, bf16 scores may choose the other
    off = (y - expect).norm(dim=-1) / expect.norm(dim=-1)
    assert (off < 0.02).sum() >= 7

"""Weights that are fetched beside a step's attention: nothing but time depends on them."""

import pytest
import torch

from mlx_sharding_amd import ops
from test_attn_step import _caches, _token

pytestmark = pytest.mark.gpu


# one block a column of the grid and many, more rows than are fetched, ends of tiles and chunks
@pytest.mark.parametrize("captured", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,D,cached,O", [
    (1, 32, 8, 128, 700, 4096), (1, 32, 4, 64, 5, 2048), (1, 9, 9, 64, 100, 1), (3, 14, 2, 128, 64, 40),
    (16, 8, 1, 64, 900, 1000), (2, 28, 4, 128, 3000, 20000), (17, 16, 1, 64, 40, 512),
    (1, 16, 8, 256, 90, 640),
    # the fewest weights that are fetched, and one row less
    (1, 9, 9, 64, 100, 1366), (1, 9, 9, 64, 100, 1365), (3, 14, 2, 128, 64, 1001),
    (16, 8, 1, 64, 900, 3001)])
def test_same(B, Hq, Hkv, D, cached, O, captured):
    g = torch.Generator("cuda").manual_seed(cached)
    one, two = _caches(B, Hkv, D, cached, cached + 40, captured, g)
    w = torch.randn(O, Hq * D + 8, generator=g, device="cuda").bfloat16() / 64
    for ahead in (w[:, : Hq * D], w[:, : Hq * D].contiguous(), w[:, 8:]):
        kept = w.clone()
        (q, k, v), cos, sin = _token(B, Hq, Hkv, D, g)
        got = one.attend_step(q, k, v, cos, sin, 0.1, ahead=ahead)
        assert torch.equal(got, two.attend_step(q, k, v, cos, sin, 0.1))
        x = got.view(B, -1)
        want = x.double() @ ahead.double().T
        off = (x.double().abs() @ ahead.double().abs().T) * (Hq * D * 2.0 ** -24)
        y = ops.linear(x, ahead)
        assert ((y.double() - want).abs() <= off + want.abs() * 2.0 ** -8 + 1e-6).all()
        assert torch.equal(w, kept) and not one._tickets.any()
        # bits, as places behind the token hold no numbers
        assert torch.equal(one._k.view(torch.int16), two._k.view(torch.int16))
        if captured:
            for c in (one, two):
                c.graph_pos += 1


def test_other_weights():
    """Hints of other kinds are none."""
    g = torch.Generator("cuda").manual_seed(1)
    one, two = _caches(1, 8, 128, 50, 100, False, g)
    w = torch.randn(512, 4096, device="cuda").bfloat16()
    for ahead in (w.float(), w.cpu(), w[:, :4000], torch.nn.Parameter(w), w.t().contiguous().t(), w[0], w[:0],
                  torch.empty(512 * 4096 + 1, device="cuda").bfloat16()[1:].view(512, 4096)):
        (q, k, v), cos, sin = _token(1, 32, 8, 128, g)
        assert torch.equal(one.attend_step(q, k, v, cos, sin, 0.1, ahead=ahead),
                           two.attend_step(q, k, v, cos, sin, 0.1))


def test_mapped_weights():
    """Weights that are mapped, of which there is no one address."""
    g = torch.Generator("cuda").manual_seed(2)
    one, two = _caches(1, 8, 128, 50, 100, False, g)
    (q, k, v), cos, sin = _token(1, 32, 8, 128, g)
    want = two.attend_step(q, k, v, cos, sin, 0.1)
    several = torch.randn(2, 512, 4096, device="cuda").bfloat16()
    got = torch.vmap(lambda w: one.attend_step(q, k, v, cos, sin, 0.1, ahead=w) @ w.t())(
        several[:1])
    assert torch.equal(got[0], want @ several[0].t())

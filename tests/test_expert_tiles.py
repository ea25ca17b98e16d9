"""Clamped experts of many tokens on the persistent tiles, against 64-bit products."""

import pytest
import torch

from mlx_sharding_amd.ops import experts
from mlx_sharding_amd.ops.ragged import ClampedGLU, hip_ragged

pytestmark = pytest.mark.gpu

GLU = ClampedGLU(1.5, 1.702)
ON_INPUT = experts.Routing("softmax", True, True)


def _operands(N, sh, seed=0):
    g = torch.Generator().manual_seed(seed)
    new = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    up = (new(sh.experts, 2 * sh.ffp, sh.widthp) * 2 * sh.width ** -0.5).bfloat16()
    down = (new(sh.experts, sh.width, sh.ffp) * sh.ff ** -0.5).bfloat16()
    router = experts.pack((new(sh.total, sh.width) * 0.3).bfloat16(), sh.widthp)
    return new(N, sh.widthp).bfloat16(), router, up, down


def _exact(h, idx, weight, up, down, sh):
    """(outputs of the chosen experts in 64 bits, how far bf16 units and results may be
    off) for pairs [N, top]; those of identity experts are zero."""
    out = torch.zeros(*idx.shape, sh.width, dtype=torch.float64, device=h.device)
    bound = torch.zeros_like(out)
    for e in range(sh.experts):
        t, j = (idx == e).nonzero(as_tuple=True)
        p = (h[t].double() @ up[e].double().T) * weight[t, j, None].double()
        g, u = p[:, : sh.ffp].clamp(max=GLU.limit), p[:, sh.ffp:].clamp(-GLU.limit, GLU.limit)
        unit = g * torch.sigmoid(GLU.alpha * g) * (u + 1)
        w = down[e].double()
        out[t, j] = unit @ w.T
        # half a step of 2^-8 each; sums, exponentials and quotients in 32 bits
        bound[t, j] = 2.0 ** -8 * (out[t, j].abs() + unit.abs() @ w.abs().T) + 1e-5
    return out, bound


# a mean of 16 pairs and of one more, 127 and 128: the borders of the kernels; experts
# without pairs; contractions of two and more than four stages; output tiles' remainders;
# experts that hand a row on, whose pairs have no places
@pytest.mark.parametrize("routing", [ON_INPUT, experts.Routing("sigmoid", False, True)])
@pytest.mark.parametrize("N,width,ff,E,identity,top", [
    (128, 128, 2048, 8, 0, 1), (129, 128, 2048, 8, 0, 1), (1016, 128, 2048, 8, 0, 1),
    (1024, 128, 2048, 8, 0, 1), (300, 320, 192, 90, 0, 6), (2100, 192, 320, 64, 0, 4),
    (400, 128, 1024, 16, 5, 3), (900, 192, 2048, 8, 1, 2)])
def test_against_64_bits(N, width, ff, E, identity, top, routing):
    sh = experts.ExpertShape(width, ff, E, identity, top)
    mean = N * top / sh.total
    assert sh.tiles(N) == (0 if mean <= 16 else 128 if mean < 128 else 256)
    h, router, up, down = (t.cuda() for t in _operands(N, sh))
    if E == 90:
        h[:] = h[:1]            # all tokens choose alike
    idx, weight = hip_ragged().expert_route(
        h, router, None, sh.total, sh.experts, top, routing.score == "sigmoid",
        routing.normalize)[:2]
    # the choice: no other expert's logit is larger, but by the error of a sum of 32 bits
    z = h.double() @ experts.unpack(router, sh.total, sh.widthp).double().T
    assert bool((idx.sort(-1).values.diff(dim=-1) > 0).all())
    left = z.scatter(-1, idx.long(), float("-inf")).max(-1).values
    assert bool((left <= z.gather(-1, idx.long()).min(-1).values + 1e-4).all())
    # the rest has that choice on both sides
    got, where, rest = experts.expert_rows(h, router, None, up, down, sh, routing, GLU)
    assert rest is None and bool(((where < 0) == (idx >= E)).all())
    own = where[where >= 0].sort().values
    assert torch.equal(own, torch.arange(len(own), device="cuda", dtype=torch.int32))
    want, bound = _exact(h, idx, weight, up, down, sh)
    there = where >= 0
    rows = got[where[there].long()].double()
    assert bool(((rows - want[there]).abs() <= bound[there]).all())


def test_refusals():
    ext = hip_ragged()
    sh = experts.ExpertShape(128, 128, 4, 0, 1)
    h, router, up, down = (t.cuda() for t in _operands(64, sh))
    ints = lambda *s: torch.zeros(*s, dtype=torch.int32, device="cuda")  # noqa: E731
    one = torch.ones(64, device="cuda")
    # no tiles: nothing is read
    ext.expert_tiles(h, ints(64), ints(4, 3), ints(1), up, down, one, 128, 1.0, 1.0)
    for args in ((h[:, :64], ints(64), ints(4, 3), ints(1), up, down, one, 128),
                 (h, ints(64), ints(4, 3), ints(1), up, down, one, 64),
                 (h, ints(64), ints(4, 3), ints(1), up, down, one[:32], 128),
                 (h, ints(64), ints(4, 3), ints(1), up[:, :128], down, one, 128),
                 (h.float(), ints(64), ints(4, 3), ints(1), up, down, one, 128)):
        with pytest.raises(RuntimeError):
            ext.expert_tiles(*args, 1.0, 1.0)

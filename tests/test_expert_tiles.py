"""Clamped experts of many tokens on the persistent tiles, beside the CPU's."""

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


# a mean of 16 pairs and of one more, 127 and 128: the borders of the kernels; experts
# without pairs; contractions of two and more than four stages; output tiles' remainders
@pytest.mark.parametrize("N,width,ff,E,top", [
    (128, 128, 2048, 8, 1), (129, 128, 2048, 8, 1), (1016, 128, 2048, 8, 1),
    (1024, 128, 2048, 8, 1), (300, 320, 192, 90, 6), (2100, 192, 320, 64, 4)])
def test_beside_cpu(N, width, ff, E, top):
    sh = experts.ExpertShape(width, ff, E, 0, top)
    assert sh.tiles(N) == (0 if N == 128 else 128 if N * top < 128 * E else 256)
    h, router, up, down = _operands(N, sh)
    if E == 90:
        h[:] = h[:1]            # all tokens choose alike
    want, at, _ = experts.expert_rows(h, router, None, up, down, sh, ON_INPUT, GLU)
    got, where, weight = experts.expert_rows(h.cuda(), router.cuda(), None, up.cuda(),
                                             down.cuda(), sh, ON_INPUT, GLU)
    assert weight is None
    # a token's experts as a set: pairs of rows in the order of choice
    a = want[at.long()].double()
    b = got[where.long()].double().cpu()
    # two experts whose scores are nearly tied may change places: compare the sums
    a, b = a.sum(1), b.sum(1)
    off = (a - b).norm(dim=1) / a.norm(dim=1)
    # units and results rounded to bf16
    assert float(off.median()) < 4e-3 and float((off > 2e-2).double().mean()) < 0.01


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

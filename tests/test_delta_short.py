"""Short portions of the gated delta rule: heads of a group in pairs, an odd one
behind them, groups that are too long for pairs, states that the threads tile."""

import pytest
import torch

import tuvutar_cases as cases
from test_tuvutar import F32, Mixer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,D,V", [
    (2, 2, 128, 128), (4, 2, 128, 128), (3, 1, 128, 128), (5, 1, 128, 64), (4, 1, 16, 128),
    (6, 2, 64, 256), (3, 1, 48, 128)])
def test_groups(heads, kv_heads, D, V):
    layer = cases.delta(heads, kv_heads, D, V, 4)
    for dtype, tol in ((F32, 5e-5), (torch.bfloat16, 5e-2)):  # as for other sizes
        m = Mixer(layer, 48, dtype, "cuda")
        h = torch.randn(50, 48, generator=torch.Generator().manual_seed(heads + D))
        want = m.want(h)
        for sizes in ([1], [2, 5, 1], [16], [15, 3]):
            assert cases.error(m.run(h, sizes), want) < tol, (dtype, sizes)

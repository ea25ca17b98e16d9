"""The gated delta rule's long portions on the GPU beside the CPU's: convolutions of one to
eight taps (four have a kernel of their own), q/k heads of one and of several value heads,
numbers of chunks and heads that make no whole round of eight."""

import copy

import pytest
import torch

from mlx_sharding_amd.models.mixers import GatedDelta
from mlx_sharding_amd.ops.paged import PagedState, RaggedBatch

pytestmark = pytest.mark.gpu

LENS = (17, 33, 64, 131)


def _run(m, rows):
    """Each request in two long portions: the second reads the first one's history."""
    dev = rows[0].device
    lens = [len(r) for r in rows]
    state = PagedState([m.store_spec()], sum(-(-2 * n // 64) * 64 for n in lens),
                       len(lens), torch.float32, dev)
    held = [state.admit(i) for i in range(len(lens))]
    out = []
    for _ in range(2):
        for i, h in enumerate(held):
            state.reserve(i, h.length + lens[i])
        b = RaggedBatch([(h, n) for h, n in zip(held, lens)], dev)
        out.append(m(torch.cat(rows), b, state.layers[0]).cpu())
        for h, n in zip(held, lens):
            h.length += n
    return torch.cat(out)


@pytest.mark.parametrize("D,V", [(128, 128), (64, 32), (32, 63)])
@pytest.mark.parametrize("heads,kv", [(1, 1), (6, 2), (4, 4)])
@pytest.mark.parametrize("taps", [1, 3, 4, 5, 8])
def test_taps(taps, heads, kv, D, V):
    torch.manual_seed(taps + heads)
    m = GatedDelta(64, heads, kv, D, V, taps, 1e-6, dtype=torch.float32)
    for p in m.parameters():
        p.data.normal_(0, 0.3)
    rows = [torch.randn(n, 64) for n in LENS]
    on_gpu = copy.deepcopy(m).cuda()   # before the first call lays weights out
    with torch.no_grad():
        want = _run(m, rows)
        got = _run(on_gpu, [r.cuda() for r in rows])
    # sums of up to 128 terms in 24 bits, through two chunks' states
    assert float((got - want).norm() / want.norm()) < 1e-4

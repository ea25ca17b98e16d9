"""Feed-forwards of few rows in one call, and products whose contraction blocks share."""

import pytest
import torch
import torch.nn.functional as F

from mlx_sharding_amd import ops
from mlx_sharding_amd.models.base import RMSNorm

pytestmark = pytest.mark.gpu

UNITS = {"silu": F.silu, "gelu_tanh": lambda t: F.gelu(t, approximate="tanh")}


def _case(M, K, ff, O, normed, residual, seed=0):
    g = torch.Generator("cuda").manual_seed(seed)
    new = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    x = new(M, K).bfloat16()
    w_in = (new(2 * ff, K) * K ** -0.5).bfloat16()
    w_out = (new(O, ff) * ff ** -0.5).bfloat16()
    norm = None
    if normed:
        norm = RMSNorm(K, 1e-5, 1.0).cuda()
        norm.weight.data = (new(K) * 0.1).bfloat16()
    return x, w_in, w_out, norm, new(M, O).bfloat16() if residual else None


def _exact(x, w_in, w_out, norm, residual, act):
    h = x.double()
    if norm is not None:
        h = h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + norm.eps)
        h = h * (norm.weight.double() + norm.weight_offset)
    g, u = (h @ w_in.double().T).chunk(2, -1)
    y = (UNITS[act](g) * u) @ w_out.double().T
    return y if residual is None else y + residual.double()


# units and results are rounded to bf16 (2^-9 at most, .3 of that in the mean), normed
# inputs too: with three such roundings less than 4e-3 of the result's 2-norm
TOL = 4e-3


@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("K,ff,O,act", [
    (64, 32, 16, "silu"),             # the smallest contraction: not shared
    (256, 4128, 100, "silu"),         # columns that make no whole tile, a last short step
    (2048, 5632, 2048, "silu"),       # shared by two or four
    (512, 8224, 2816, "gelu_tanh"),   # shared by blocks of four tiles, above 16 rows
    (512, 8192, 2848, "gelu_tanh"),
    (512, 7264, 4608, "silu"),        # below 8192 columns: not shared
])
def test_feed_few(M, K, ff, O, act):
    for normed, residual in ((True, True), (False, False)):
        case = _case(M, K, ff, O, normed, residual)
        want = _exact(*case, act)
        got = ops.feed_few(*case[:3], act, *case[3:])
        assert got is not None and got.shape == (M, O)
        assert float((got.double() - want).norm() / want.norm()) < TOL
        # sums have one order whichever block comes last
        for _ in range(3):
            assert torch.equal(ops.feed_few(*case[:3], act, *case[3:]), got)


@pytest.mark.parametrize("M,ff,O", [
    (16, 4096, 2048), (1, 4096, 2048), (64, 2560, 2048), (64, 2528, 2048),
    (16, 4096, 2064), (9, 12288, 2064), (16, 12288, 3584), (16, 12256, 3584),
    (16, 12288, 3600), (17, 8192, 4096), (17, 8192, 4112)])
def test_where_shares_begin(M, ff, O):
    """The last sizes that blocks share, and the first that they do not."""
    case = _case(M, 64, ff, O, False, True)
    want, got = _exact(*case, "silu"), ops.feed_few(*case[:3], "silu", *case[3:])
    assert float((got.double() - want).norm() / want.norm()) < TOL
    assert torch.equal(ops.feed_few(*case[:3], "silu", *case[3:]), got)


def test_feed_few_captured():
    case = _case(12, 512, 8192, 2048, True, True)
    x = case[0]
    ops.feed_few(*case[:3], "silu", *case[3:])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = ops.feed_few(*case[:3], "silu", *case[3:])
        y = y + ops.feed_few(*case[:3], "silu", *case[3:])
    for i in range(4):
        x.copy_(torch.randn(x.shape, device="cuda"))
        one = ops.feed_few(*case[:3], "silu", *case[3:])  # eager work between replays
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, one + one)


def test_feed_few_on_streams():
    cases = [_case(12, 512, 8192, 2048, True, True, s) for s in range(4)]
    want = [ops.feed_few(*c[:3], "silu", *c[3:]) for c in cases]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in cases]
    for _ in range(10):
        got = []
        for c, s in zip(cases, streams):
            with torch.cuda.stream(s):
                got.append(ops.feed_few(*c[:3], "silu", *c[3:]))
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_feed_few_leaves_others():
    x, w_in, w_out, _, _ = _case(4, 64, 64, 32, False, False)
    assert ops.feed_few(x.float(), w_in, w_out, "silu") is None
    assert ops.feed_few(x, w_in[:100], w_out, "silu") is None
    assert ops.feed_few(x, w_in, w_out[:, :32], "silu") is None
    assert ops.feed_few(x, w_in, w_out.T.contiguous().T, "silu") is None
    assert ops.feed_few(x.repeat(20, 1), w_in, w_out, "silu") is None
    assert ops.feed_few(x.cpu(), w_in, w_out, "silu") is None

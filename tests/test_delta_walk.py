"""The walk over chunks of the gated delta rule: a block takes one column tile of a
(request, head) where there are few of them and two where there are many.  The tests
of single requests against the oracle cover the first; here many requests at once
have to give what each gives alone."""

import pytest
import torch

from mlx_sharding_amd.models.mixers import GatedDelta
from mlx_sharding_amd.ops import ragged
from mlx_sharding_amd.ops.paged import PagedState, RaggedBatch, StateSpec

pytestmark = pytest.mark.gpu

LENS = (34, 80, 81, 82, 145, 146, 217, 50, 338)


def _run(m, rows, dtype):
    """Each request in two portions, so that the states of the first are read back."""
    lens = [len(r) for r in rows]
    dev = rows[0].device
    state = PagedState([m.store_spec()], sum(-(-n // 64) * 64 for n in lens), len(lens),
                       dtype, dev)
    held = [state.admit(i) for i in range(len(lens))]
    out = []
    for part in (0, 1):
        take = [r[-17:] if part else r[:-17] for r in rows]
        for i, h in enumerate(held):
            state.reserve(i, h.length + len(take[i]))
        b = RaggedBatch([(h, len(t)) for h, t in zip(held, take)], dev)
        y = m(torch.cat(take), b, state.layers[0])
        out.append(y.split([len(t) for t in take]))
        for h, t in zip(held, take):
            h.length += len(t)
    return [torch.cat(x) for x in zip(*out)]


@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("heads", [4, 8])   # 36 and 72 (request, head): by eights or not
@pytest.mark.parametrize("D", [16, 32, 64, 96, 128])
def test_many_as_alone(D, heads, channel):
    dev = torch.device("cuda")
    torch.manual_seed(D + heads)
    with dev:
        m = GatedDelta(64, heads, heads // 2, D, 128, 4, 1e-6, dtype=torch.float32,
                       ranks=(32, 32) if channel else None,
                       gate="sigmoid" if channel else "silu")
    for name, p in m.named_parameters():
        p.data.normal_(0, 0.5 if "conv" in name else 0.1)
    m.A_log.data.normal_(0.5, 0.7)
    m.dt_bias.data.normal_(-3, 1)
    m.prepare()
    rows = [torch.randn(n, 64, device=dev) for n in LENS]
    many = _run(m, rows, torch.float32)
    for r, got in zip(rows, many):
        want, = _run(m, [r], torch.float32)
        # the projections may sum in another order: a few roundings of 2^-24 over 64
        # terms, carried through a state that forgets
        assert (got - want).abs().max() <= 1e-4 * want.abs().max()


@pytest.mark.parametrize("words", [0, 1])
def test_chunks_at_any_word(words, monkeypatch):
    """A batch's index arrays lie behind one another in one buffer: the list of chunks
    begins at any multiple of four bytes."""
    dev = torch.device("cuda")
    torch.manual_seed(words)
    with dev:
        m = GatedDelta(64, 4, 2, 64, 128, 4, 1e-6, dtype=torch.float32, ranks=None,
                       gate="silu")
    for p in m.parameters():
        p.data.normal_(0, 0.1)
    m.prepare()
    rows = [torch.randn(n, 64, device=dev) for n in LENS]
    want = _run(m, rows, torch.float32)
    init = RaggedBatch.__init__

    def moved(self, *args):
        init(self, *args)
        n = self.chunks.numel()
        room = torch.empty(n + 2, dtype=torch.int32, device=dev)[words: words + n]
        self.chunks = room.view(-1, 2).copy_(self.chunks)
        assert self.chunks.data_ptr() % 8 == 4 * words

    monkeypatch.setattr(RaggedBatch, "__init__", moved)
    for got, expect in zip(_run(m, rows, torch.float32), want):
        assert torch.equal(got, expect)


def _plain(D, channel, n, change):
    """One request of n tokens that forgets nothing, without a convolution: (outputs [n, V],
    values [n, V], state [D, V]).  Values of 64 and more go through silu as they are.
    change(v, beta): values, and what goes into their sigmoid."""
    dev, V = torch.device("cuda"), 128
    torch.manual_seed(D)
    sh = ragged.DeltaShape(1, 1, D, V, 1, (32, 32) if channel else None)
    state = PagedState([StateSpec(1, D, V, sh.channels, 0)], -(-n // 64) * 64, 1,
                       torch.float32, dev)
    held = state.admit(0)
    state.reserve(0, n)
    at = sh.columns
    y = torch.zeros(n, -(-(at[5] + 1) // 8) * 8, device=dev)
    y[:, : 2 * D].uniform_(0.5, 1.5)                     # q and k
    v, beta = y[:, at[2]: at[2] + V].uniform_(64, 128), y[:, at[5]].normal_()
    change(v, beta)
    gate = None
    if channel:  # decay inputs are 0, as they are in y
        gate = torch.zeros(n, D + V, device=dev)
        gate[:, D:] = 3.0
    else:
        y[:, at[3]: at[3] + V] = 3.0
    one = lambda *s: torch.ones(*s, device=dev)  # noqa: E731
    out = ragged.gated_delta(
        y, one(sh.channels, 1), one(1) * -200, one(D if channel else 1), one(V),
        state.layers[0], sh, 1e-6, RaggedBatch([(held, n)], dev), gate)
    return out, v, state.layers[0].state[held.slot][0]


@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("D", [8, 32, 64, 128])
def test_a_lone_product_is_rounded_once(D, channel):
    """The state of one token's key and value: half a last place off, and 2^-7 of that for
    sums of parts that were rounded before."""
    def only(v, beta):
        v[:, 0] = 64.0  # that times a key is exact
        beta.fill_(-200.0)
        beta[37] = 200.0

    _, v, S = _plain(D, channel, 100, only)
    key = S[:, :1].double() / 64
    assert bool((key > 0).all())
    want = key * v[37].double()
    assert ((S.double() - want).abs() / want).max() <= 2.0 ** -24 * (1 + 2.0 ** -7)


@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("token", [16, 20, 52, 127])
def test_what_is_no_number_stays_with_its_neighbours(token, channel):
    """Tokens before those 16 that a value without a number lies in do not see it."""
    def spoil(v, beta):
        v[token, 5] = float("nan")

    want = _plain(64, channel, 150, lambda v, beta: None)[0]
    got = _plain(64, channel, 150, spoil)[0]
    before = token // 16 * 16
    assert torch.equal(got[:before], want[:before])
    assert bool(got[token].isnan().any())

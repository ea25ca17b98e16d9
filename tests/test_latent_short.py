"""Latent attention of short portions over the cached rows themselves."""

from types import SimpleNamespace

import pytest
import torch

from mlx_sharding_amd.ops import hip_ext, ragged
from mlx_sharding_amd.ops.paged import PagedState, RaggedBatch, RowSpec

pytestmark = pytest.mark.gpu


# one key, a tile of 32 keys and a page of 64 less one, whole and more; slices of
# several tiles; tiles of 16 rows with remainders; rotated parts of one piece a
# thread, less, more and none; what lies behind a request's keys is not a number
@pytest.mark.parametrize("heads, rank, rot, dtype", [
    (16, 512, 64, torch.bfloat16), (3, 64, 32, torch.bfloat16),
    (5, 1024, 96, torch.bfloat16), (4, 128, 160, torch.float32),
    (6, 512, 0, torch.bfloat16), (3, 64, 0, torch.float32),
])
def test_against_64_bits(heads, rank, rot, dtype):
    dev = torch.device("cuda")
    torch.manual_seed(heads)
    sh = ragged.LatentShape(heads, 32, rot, 32, rank)
    kept, new = (0, 30, 31, 32, 62, 63, 500, 2500), (1, 1, 2, 1, 1, 9, 16, 1)
    room = sum(-(-(a + b) // 64) * 64 for a, b in zip(kept, new))
    state = PagedState([RowSpec(sh.width)], room, len(kept), dtype, dev)
    rows = state.layers[0].rows
    rows.fill_(float("nan"))
    held = [state.admit(i) for i in range(len(kept))]
    for i, h in enumerate(held):
        state.reserve(i, kept[i] + new[i])
        h.length = kept[i]
        for j in range(kept[i] + new[i]):
            rows[h.pages[j // 64] * 64 + j % 64] = torch.randn(sh.width, device=dev)
    batch = [(h, n) for h, n in zip(held, new)]
    q = torch.randn(sum(new), heads * sh.dq, device=dev).to(dtype)
    q_abs = torch.randn(heads, sum(new), sh.rankp, device=dev).to(dtype)
    scale = sh.width ** -0.5
    got = ragged.latent_attention_absorbed(
        q, q_abs, state.layers[0], sh, scale, RaggedBatch(batch, dev), len(new),
        max(new)).cpu().double()
    want = ragged.latent_attention_absorbed(
        q.cpu().float(), q_abs.cpu().float(),
        SimpleNamespace(rows=rows.cpu().float()), sh, scale,
        RaggedBatch(batch, torch.device("cpu")), len(new), max(new)).double()
    # bf16: the result's own rounding, and that of the weights' two parts; float:
    # sums of up to 2501 products of weights that add up to 1
    bound = 2.0 ** -8 * 1.05 if dtype == torch.bfloat16 else 2.0 ** -18
    assert (got - want).abs().max() <= bound * want.abs().max()


# one row, a tile of 16 with one less and one more, every count of tiles a block;
# contractions of one step, fewer than the waves, uneven among them, none; both layouts
@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 64, 131, 256])
@pytest.mark.parametrize("wide, out, dtype", [
    (32, 16, torch.bfloat16), (96, 80, torch.bfloat16), (512, 128, torch.bfloat16),
    (160, 64, torch.float32), (0, 64, torch.bfloat16),
])
def test_products_of_heads(n, wide, out, dtype):
    torch.manual_seed(n)
    x = torch.randn(n, 3, wide + 8, device="cuda").to(dtype)[..., :wide]
    w = torch.randn(3, out, wide, device="cuda").to(dtype)
    want = torch.einsum("nhk,hok->nho", x.cpu().double(), w.cpu().double())
    size = torch.einsum("nhk,hok->nho", x.cpu().double().abs(), w.cpu().double().abs())
    # the result's rounding (bf16 keeps 8 bits: half a last place is up to 2^-8 of the
    # value), and 32-bit sums of ``wide`` products
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    bound = unit * want.abs() + wide * 2.0 ** -24 * size
    got = ragged.latent_heads(x, w, False).cpu().double()
    assert ((got - want).abs() <= bound).all()
    assert torch.equal(ragged.latent_heads(
        x.transpose(0, 1).contiguous().transpose(0, 1), w, True).cpu().double(),
        got.transpose(0, 1))


# room for many more keys than there are, as in a captured step; slices shared by groups
# of threads, by halves of them and not at all; fewer slices than groups
@pytest.mark.parametrize("N", [1, 2, 3, 17])
@pytest.mark.parametrize("S, room", [(1, 4096), (33, 1024), (65, 65), (700, 1024),
                                     (2049, 4096)])
def test_slices_of_cached_latents(N, S, room):
    H, rank, rope, vdim, scale = 16, 512, 64, 128, 0.05
    torch.manual_seed(N + S)
    q = torch.randn(N, H, 1, rank + rope, device="cuda").bfloat16()
    cache = torch.full((N, 1, room, rank + rope), float("nan"), device="cuda").bfloat16()
    cache[:, :, :S] = torch.randn(N, 1, S, rank + rope, device="cuda").bfloat16()
    w = (torch.randn(H, vdim, rank, device="cuda") * 0.05).bfloat16()
    pos = torch.tensor([S - 1], dtype=torch.int32, device="cuda")
    got = hip_ext().mla_attend(q, cache, w, scale, pos, 1).double().view(N, H, vdim)
    keys = cache[:, 0, :S].double()
    p = torch.softmax(torch.einsum("nhd,nsd->nhs", q[:, :, 0].double(), keys) * scale, -1)
    latent = torch.einsum("nhs,nsr->nhr", p, keys[..., :rank])
    want = torch.einsum("nhr,hvr->nhv", latent, w.double())
    size = torch.einsum("nhr,hvr->nhv", latent.abs(), w.double().abs())
    # the latent's rounding to bf16, the result's, and 32-bit scores and sums
    bound = 2.0 ** -8 * (size + want.abs()) + 2.0 ** -16 * size
    assert ((got - want).abs() <= bound).all()


@pytest.mark.parametrize("room", [65, 4096])
def test_a_place_before_the_first_key(room):
    """No keys, few slices and many: no numbers."""
    q = torch.randn(2, 16, 1, 576, device="cuda").bfloat16()
    cache = torch.randn(2, 1, room, 576, device="cuda").bfloat16()
    w = torch.randn(16, 128, 512, device="cuda").bfloat16()
    pos = torch.tensor([-1], dtype=torch.int32, device="cuda")
    assert hip_ext().mla_attend(q, cache, w, 0.05, pos, 1).isnan().all()

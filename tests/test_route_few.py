"""The router's choice among up to 64 experts, a lane each, and above."""

import pytest
import torch

from mlx_sharding_amd.ops.experts import pack
from mlx_sharding_amd.ops.ragged import hip_ragged

pytestmark = pytest.mark.gpu


def picks(z, choice, score, top, normalize):
    """One after the other: the largest, the first of equals, never what is not above
    -inf, in whose place the last one comes."""
    idx, weight = [], []
    for c, s in zip(choice.clone(), score):
        row = []
        for _ in range(top):
            above = c > -torch.inf
            at = (int((c == c[above].max()).nonzero()[0]) if bool(above.any())
                  else len(c) - 1)
            c[at] = -torch.inf
            row.append(at)
        idx.append(row)
        w = s[row]
        weight.append(w / (w.sum() + 1e-20) if normalize else w)
    return torch.tensor(idx), torch.stack(weight)


@pytest.mark.parametrize("sigmoid,normalize", [(False, True), (True, False), (True, True)])
@pytest.mark.parametrize("total,experts,top", [(1, 1, 1), (5, 3, 5), (16, 16, 4), (63, 60, 8),
                                               (64, 64, 64), (65, 65, 6), (130, 128, 9)])
@pytest.mark.parametrize("N,K", [(1, 64), (17, 320), (32, 2048)])
def test_choice(N, K, total, experts, top, sigmoid, normalize):
    g = torch.Generator().manual_seed(total + N)
    # few whole numbers: logits are exact, and many are equal
    h = torch.randint(-1, 2, (N, K), generator=g).float()
    w = torch.zeros(total, K)
    w[:, :: max(1, K // 8)] = torch.randint(-1, 2, w[:, :: max(1, K // 8)].shape,
                                            generator=g).float()
    z = h @ w.T
    if total > 3:
        h[0] = 0.0
        z[0] = 0.0
    score = torch.sigmoid(z) if sigmoid else torch.softmax(z, -1)
    packed = pack(w.bfloat16(), K).cuda()
    some = torch.randint(0, 3, (total,), generator=g).float() * 4
    some[some == 8] = -torch.inf
    for correction in (None, some.bfloat16()):
        choice = z if correction is None else score + correction.float()
        idx, weight = picks(z, choice, score, top, normalize)
        got = hip_ragged().expert_route(
            h.bfloat16().cuda(), packed, None if correction is None else correction.cuda(),
            total, experts, top, sigmoid, normalize)
        if correction is not None and not sigmoid:
            # scores that differ by their rounding only: the same choice, not its order
            torch.testing.assert_close(choice.gather(1, got[0].cpu().long()),
                                       choice.gather(1, idx), rtol=1e-6, atol=1e-6)
        else:
            assert torch.equal(got[0].cpu().long(), idx)
            torch.testing.assert_close(got[1].cpu(), weight, rtol=2e-6, atol=1e-7)
        pairs = got[0].cpu().flatten()
        counts = torch.bincount(pairs[pairs < experts], minlength=experts)[:experts]
        assert torch.equal(got[3].cpu().sum(0).long(), counts)

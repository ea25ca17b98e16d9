"""Norm, residual and next norm in one kernel, against 64 bits."""

import types

import pytest
import torch

from mlx_sharding_amd import ops


def _norm(H, dev, eps, offset):
    n = types.SimpleNamespace(weight=torch.randn(H, device=dev).bfloat16(), eps=eps,
                              weight_offset=offset)

    class Norm:
        weight, eps, weight_offset = n.weight, n.eps, n.weight_offset

        def __call__(self, x):
            return ops.rms_norm(x, n.weight, n.eps, n.weight_offset)
    return Norm()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,H", [(1, 8), (5, 3584), (3, 2048), (7, 2056), (2, 8192),
                                    (300, 72)])
def test_against_64_bits(rows, H):
    torch.manual_seed(H)
    a, b = _norm(H, "cuda", 1e-6, 1.0), _norm(H, "cuda", 1e-5, 0.0)
    x, r = (torch.randn(rows, 1, H, device="cuda").bfloat16() for _ in "xr")
    rms = lambda t, n: (t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + n.eps)  # noqa: E731
                        * (n.weight.double() + n.weight_offset))
    want = r.double() + rms(x.double(), a)
    close = lambda got, t: bool(  # noqa: E731
        ((got.double() - t).abs() <= 2.0 ** -8 * t.abs() + 1e-5).all())
    assert close(ops.norm_add(x, a, r), want)
    h, y = ops.norm_add(x, a, r, b)
    assert close(h, want) and close(y, rms(h.double(), b))


@pytest.mark.gpu
def test_other_forms_run_apart():
    """Rows that are no whole vectors, strided ones and wide ones, as before."""
    for H, make in ((12, lambda t: t), (64, lambda t: t[:, ::2]), (8200, lambda t: t)):
        n = _norm(H, "cuda", 1e-6, 1.0)
        x, r = (make(torch.randn(2, 4, H, device="cuda").bfloat16()) for _ in "xr")
        h, y = ops.norm_add(x, n, r, n)
        assert torch.equal(h, r + n(x)) and torch.equal(y, n(h))


def test_cpu():
    n = _norm(16, "cpu", 1e-6, 1.0)
    x, r = (torch.randn(2, 16).bfloat16() for _ in "xr")
    assert torch.equal(ops.norm_add(x, n, r), r + n(x))

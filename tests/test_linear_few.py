"""The product for few rows and what goes with it, against 64 bits."""

import types

import pytest
import torch
import torch.nn.functional as F

from mlx_sharding_amd import ops


def taken(x, w):
    """Whether ops.linear runs x W^T on the kernel."""
    return ops._linear_few(x, w) is not None


def make(M, O, K, act, wide):
    g = torch.Generator().manual_seed(M + O + K)
    new = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()  # noqa: E731
    x = new(M, K + 8 * wide)[:, 8 * wide:]      # rows as slices of wider ones
    w = (torch.randn(O, K + 16 * wide, generator=g) * 0.05).bfloat16().cuda()[:, :K]
    norm = types.SimpleNamespace(weight=new(K), eps=1e-5, weight_offset=1.0)
    return x, w, norm, new(O), new(M, O // 2 if act else O)


@pytest.mark.gpu
@pytest.mark.parametrize("M,O,K", [
    (1, 2, 32), (3, 18, 96), (16, 34, 2080), (5, 4098, 64), (16, 8194, 160),
    (4, 8210, 32), (9, 4100, 256), (2, 16386, 96), (16, 16400, 1056),
    (8, 96, 14336), (7, 8200, 2016), (17, 2, 32), (33, 18, 96), (64, 34, 2080),
    (20, 4098, 64), (48, 8194, 160), (64, 8210, 288), (31, 16400, 1056),
    (12, 96, 8224), (40, 100, 9216)])
def test_edges(M, O, K):
    """Tiles of 16, 32 and 64 columns with remainders, contractions that are not
    whole chunks or stages, fewer steps than waves, 16 rows and more, 32 and more;
    norm, bias, unit, residual."""
    for act in (None, "silu", "gelu_tanh"):
        x, w, norm, bias, res = make(M, O, K, act, wide=K % 64 == 0)
        assert taken(x, w)
        for normed in (False, True):
            for rest in (False, True):
                b, r = (bias, res) if rest else (None, None)
                y = ops.project(x, w, b, norm=norm if normed else None, act=act,
                                residual=r).double()
                h, size = x.double(), x.double().abs()
                if normed:
                    f = torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + 1e-5)
                    h, size = ((t * f * (norm.weight.double() + 1.0)) for t in (h, size))
                z = h @ w.double().T
                # 32-bit sums, and rows rounded to bf16 behind the norm
                off = (size.abs() @ w.double().abs().T) * (
                    K * 2.0 ** -24 + (2.0 ** -8 if normed else 0.0))
                if rest:
                    z = z + bias.double()
                if act:
                    gate, up = z.chunk(2, -1)
                    og, ou = off.chunk(2, -1)
                    unit = F.silu if act == "silu" else lambda t: F.gelu(
                        t, approximate="tanh")
                    z = unit(gate) * up
                    # both units grow by at most 1.13 of their argument
                    off = 1.13 * og * (up.abs() + ou) + unit(gate).abs() * ou + 1e-6
                if rest:
                    z = z + res.double()
                bound = 2.0 ** -8 * z.abs() + off + 1e-6
                assert bool(((y - z).abs() <= bound).all()), (act, normed, rest)


@pytest.mark.gpu
def test_same_as_separate_kernels():
    """What the projection takes along, beside the kernels it stands for."""
    x, w, norm, bias, _ = make(16, 512, 256, None, wide=True)
    several = torch.cat([x] * 5)                  # too many rows: separate
    assert not taken(several, w)
    norm = types.SimpleNamespace(
        weight=norm.weight, eps=1e-5, weight_offset=1.0)
    one = ops.project(x, w, bias, act="silu")
    two = ops.project(several, w, bias, act="silu")[:16]
    assert (one.double() - two.double()).norm() < 0.01 * two.double().norm()


@pytest.mark.gpu
def test_other_forms_keep_the_library():
    """Calls that the kernel does not take run as before."""
    w = torch.randn(24, 64, device="cuda").bfloat16()
    x = torch.randn(2, 3, 64, device="cuda").bfloat16()
    expect = x.double() @ w.double().T
    close = lambda y: (y.double() - expect).norm() < 0.01 * expect.norm()  # noqa: E731
    assert close(ops.linear(x, w))
    at = torch.randn(6 * 64 + 1, device="cuda").bfloat16()  # rows off 16 bytes
    odd = at[1:].view(2, 3, 64)
    odd.copy_(x)
    assert not taken(odd, w) and close(ops.linear(odd, w))
    turned = w.t().contiguous().t()                 # columns side by side
    assert not taken(x, turned) and close(ops.linear(x, turned))
    assert ops.linear(x.float(), w.float()).dtype == torch.float32
    assert ops.linear(x[:, :0], w).shape == (2, 0, 24)
    # what is differentiated or mapped
    p = torch.nn.Parameter(w)
    ops.linear(x, p).float().sum().backward()
    assert p.grad is not None
    assert close(torch.vmap(lambda r: ops.linear(r, w))(x))
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        tangent = torch.autograd.forward_ad.unpack_dual(ops.linear(dual, w)).tangent
    assert tangent is not None


@pytest.mark.gpu
def test_other_forms_of_what_goes_along():
    """Biases and residuals in the forms that separate operators take, on their own
    and with a norm: strides, broadcasts, other types, gradients."""
    x, w, norm, b, r = make(6, 24, 64, None, wide=False)
    x, r = x.view(2, 3, 64), r.view(2, 3, 24)
    wide = torch.randn(24, 2, device="cuda").bfloat16()
    h = x.double()
    normed = h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + 1e-5) * (
        norm.weight.double() + 1.0)

    class Norm:
        weight, eps, weight_offset = norm.weight, norm.eps, norm.weight_offset

        def __call__(self, t):
            return ops.rms_norm(t, self.weight, self.eps, self.weight_offset)

    for bias in (None, wide[:, 1], b[:1].expand(24), b[:1], b[None]):
        off = 0.0 if bias is None else bias.double()
        expect = h @ w.double().T + off
        y = ops.linear(x, w, bias)
        assert y.shape == expect.shape
        assert (y.double() - expect).norm() < 0.01 * expect.norm()
        for res in (r, r[:1, :1], r[..., :1], r.float(), r[0], r.transpose(0, 1)
                    .contiguous().transpose(0, 1), wide[:, 1]):
            for n, rows in ((None, h), (Norm(), normed)):
                expect = rows @ w.double().T + off + res.double()
                y = ops.project(x, w, bias, norm=n, residual=res)
                assert y.shape == expect.shape
                assert y.dtype == torch.promote_types(x.dtype, res.dtype)
                assert (y.double() - expect).norm() < 0.01 * expect.norm()
    p = torch.nn.Parameter(r)
    ops.project(x, w, residual=p).float().sum().backward()
    assert bool((p.grad == 1).all())


@pytest.mark.gpu
def test_tracers_see_a_product():
    """What records operators records torch's own, and what it made runs on other
    rows."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils._python_dispatch import TorchDispatchMode
    from torch.utils.flop_counter import FlopCounterMode

    class Names(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    class Calls(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func.__name__)
            return func(*args, **(kwargs or {}))

    w = torch.randn(24, 64, device="cuda").bfloat16()
    x, other = (torch.randn(3, 64, device="cuda").bfloat16() for _ in range(2))
    res = torch.randn(3, 24, device="cuda").bfloat16()
    f = lambda t: ops.project(t, w, residual=res)  # noqa: E731
    expect = other.double() @ w.double().T + res.double()
    close = lambda y: (y.double() - expect).norm() < 0.01 * expect.norm()  # noqa: E731
    assert close(torch.jit.trace(f, (x,), check_trace=False)(other))
    assert close(make_fx(f)(x)(other))
    for mode, name in ((Names, "mm"), (Calls, "linear")):
        seen = []
        with mode():
            assert not ops.few_tokens(x)
            y = f(other)
        assert close(y) and any(name in s for s in seen), seen
    with FlopCounterMode(display=False) as count:
        f(x)
    assert count.get_total_flops() == 2 * 3 * 64 * 24
    with torch.device("cuda"):  # a mode, too, that records nothing
        assert ops.few_tokens(x) and close(f(other))


@pytest.mark.gpu
def test_compiled_in_one_graph():
    """What torch.compile reads, it reads to the end."""
    w = torch.randn(24, 64, device="cuda").bfloat16()
    x = torch.randn(3, 64, device="cuda").bfloat16()
    graphs = []

    def backend(graph, inputs):
        graphs.append([n.target for n in graph.graph.nodes if n.op == "call_function"])
        return graph.forward

    y = torch.compile(lambda t: ops.linear(t, w) * 2, backend=backend, fullgraph=True)(x)
    expect = x.double() @ w.double().T * 2
    assert len(graphs) == 1 and len(graphs[0]) == 2
    assert (y.double() - expect).norm() < 0.01 * expect.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [3, 200])
def test_autocast_names_the_type(rows):
    """Few rows have the type that many have."""
    w = torch.randn(24, 64, device="cuda").bfloat16()
    x = torch.randn(rows, 64, device="cuda").bfloat16()
    for kind in (torch.float16, torch.bfloat16):
        with torch.autocast("cuda", dtype=kind):
            y, expect = ops.linear(x, w), F.linear(x, w)
        assert y.dtype == expect.dtype == kind
        assert (y.double() - expect.double()).norm() < 0.01 * expect.double().norm()


def test_cpu_tensors_keep_torch():
    x, w = torch.randn(2, 64).bfloat16(), torch.randn(24, 64).bfloat16()
    assert not ops.few_tokens(x)
    assert torch.equal(ops.linear(x, w), F.linear(x, w))

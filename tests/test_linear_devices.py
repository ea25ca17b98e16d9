"""Products of few rows on devices that are not the current one, and on two."""

import ctypes

import pytest
import torch

from mlx_sharding_amd import ops

pytestmark = pytest.mark.gpu


class _Managed(ctypes.Structure):
    """A tensor as DLPack hands it over, without an owner."""
    _fields_ = [("data", ctypes.c_void_p), ("device_type", ctypes.c_int32),
                ("device_id", ctypes.c_int32), ("ndim", ctypes.c_int32),
                ("code", ctypes.c_uint8), ("bits", ctypes.c_uint8),
                ("lanes", ctypes.c_uint16), ("shape", ctypes.POINTER(ctypes.c_int64)),
                ("strides", ctypes.POINTER(ctypes.c_int64)),
                ("offset", ctypes.c_uint64), ("owner", ctypes.c_void_p),
                ("deleter", ctypes.c_void_p)]


def on_device(t: torch.Tensor, index: int, kept: list) -> torch.Tensor:
    """t's memory under another device's name; ``kept`` outlives the result."""
    rows = ctypes.c_int64 * t.dim()
    shape, strides = rows(*t.shape), rows(*t.stride())
    m = _Managed(t.data_ptr(), 10, index, t.dim(), 4, 16, 1, shape, strides, 0, None,
                 None)
    new = ctypes.pythonapi.PyCapsule_New
    new.restype = ctypes.py_object
    new.argtypes = [ctypes.c_void_p, ctypes.c_char_p, ctypes.c_void_p]
    kept += [t, shape, strides, m]
    return torch._C._from_dlpack(new(ctypes.addressof(m), b"dltensor", None))


def test_operands_on_two_devices_are_refused():
    """As the library's product refuses them.  One device is enough: the other
    operand has the name of another, and memory of this one."""
    kept = []
    x = torch.randn(4, 64, device="cuda").bfloat16()
    w = torch.randn(32, 64, device="cuda").bfloat16()
    b = torch.randn(32, device="cuda").bfloat16()
    far = torch.cuda.current_device() + 1
    assert on_device(w, far, kept).device.index == far
    with pytest.raises(RuntimeError):
        ops.linear(x, on_device(w, far, kept))
    with pytest.raises(RuntimeError):
        ops.linear(x, w, on_device(b, far, kept))
    with pytest.raises(RuntimeError):
        ops.project(x, w, residual=on_device(x[:, :32].contiguous(), far, kept))


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two GPUs")
def test_runs_where_its_operands_are():
    """Neither the current device nor another's stream: work queued on the operands'
    own current stream comes first."""
    x = torch.randn(4, 64, device="cuda:1").bfloat16()
    w = torch.randn(32, 64, device="cuda:1").bfloat16()
    torch.cuda.synchronize(1)
    with torch.cuda.device(1):
        stream = torch.cuda.Stream()
    with torch.cuda.stream(stream), torch.cuda.device(0):
        y = ops.linear(x, w)
        expect = torch.nn.functional.linear(x, w)
        assert torch.cuda.current_device() == 0
    stream.synchronize()
    assert y.device == x.device
    assert (y.double() - expect.double()).norm() < 0.01 * expect.double().norm()


def test_runs_on_the_current_stream():
    """A stream other than the default, and operands that it has yet to write."""
    x = torch.zeros(4, 4096, device="cuda").bfloat16()
    w = torch.randn(64, 4096, device="cuda").bfloat16()
    big = torch.randn(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        for _ in range(20):
            big = big @ big * 1e-3
        x.fill_(1.0)
        y = ops.linear(x, w)
    stream.synchronize()
    expect = x.double() @ w.double().T
    assert (y.double() - expect).norm() < 0.01 * expect.norm()

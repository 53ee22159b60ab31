"""The staging of the torch gradients in the modes a caller's program may be in:
inference mode on some calls only, another default device."""
import ctypes as C

import numpy as np
import pytest
import torch

from masterthesis_amd import autograd, capi


class _HostArray:
    def __init__(self, count, dtype):
        self.count, self.dtype = count, np.dtype(dtype)
        self.nbytes = count * self.dtype.itemsize
        self.data = np.zeros(count, dtype)
        self.ptr = capi.vp(self.data.ctypes.data)


class _HostContext:
    """A context whose device memory is host memory."""
    h = None
    _bufs = ()

    class L:
        @staticmethod
        def scafes_memcpy_h2d(h, dst, src, nbytes):
            C.memmove(dst, src, nbytes)
            return 0
        scafes_memcpy_d2h = scafes_memcpy_h2d

    def alloc(self, count, dtype):
        return _HostArray(count, dtype)


def _round_trip(f, a, dtype):
    return f.get(f.put("x", a, dtype), a.shape)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_inference_mode_on_one_call_only(dtype):
    a = np.random.default_rng(0).standard_normal((5, 4))
    f = autograd._DeviceFields(_HostContext())
    for first in (True, False):
        with torch.inference_mode(first):
            np.testing.assert_array_equal(_round_trip(f, a, dtype), a.astype(dtype))


def test_other_default_device():
    a = np.random.default_rng(1).standard_normal(7)
    with torch.device("meta"):  # a tensor made without a device would have no memory
        np.testing.assert_array_equal(_round_trip(autograd._DeviceFields(_HostContext()), a, np.float64), a)


@pytest.mark.gpu
def test_kappa_gradient_after_inference_mode(hip):
    n, steps = (9, 8, 7), 4
    shape = tuple(m + 2 for m in reversed(n))
    tau = 0.9 / sum(2 * 1.5 * (m - 1.0) ** 2 for m in n)
    g = torch.Generator().manual_seed(2)
    u0, kap, tgt = (torch.rand(shape, generator=g, dtype=torch.float64) for _ in range(3))
    kap = (1.0 + 0.4 * kap).requires_grad_(True)
    with capi.Context(0) as ctx:
        fn = autograd.KappaMisfit(ctx, n, tau, steps, dtype="f64")
        with torch.inference_mode():
            first = fn(kap, u0, tgt).item()
        J = fn(kap, u0, tgt)
        grad, = torch.autograd.grad(J, kap)
        assert J.item() == first and float(grad.abs().max()) > 0.0
        del fn

"""FP64 updates at the limits of the quotient by h^2: states with zeros,
subnormal and near-overflow values, infinities and NaN against the same sums
with IEEE divisions in numpy (bit for bit, NaN at the same nodes)."""
import ctypes as C

import numpy as np
import pytest

from masterthesis_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(hip):
    c = capi.Context(0)
    yield c
    c.close()


def _extreme(rng, shape, kind):
    u = rng.standard_normal(shape)
    if kind == "scales":  # every magnitude from subnormal to near overflow
        return u * 2.0 ** rng.integers(-1074, 1010, size=shape)
    if kind == "tiny":
        return u * 2.0 ** rng.integers(-1074, -880, size=shape)
    if kind == "zeros":
        u[rng.random(shape) < 0.9] = 0.0
        return u
    u[rng.random(shape) < 0.02] = np.inf
    u[rng.random(shape) < 0.02] = np.nan
    u[rng.random(shape) < 0.05] = 1.7e308
    return u


def _nb(a, axis):
    """centre, lower and upper neighbour on inner nodes"""
    c = tuple(slice(1, -1) for _ in a.shape)
    lo = tuple(slice(0, -2) if q == axis else slice(1, -1) for q in range(a.ndim))
    hi = tuple(slice(2, None) if q == axis else slice(1, -1) for q in range(a.ndim))
    return a[c], a[lo], a[hi]


def _heat(u, tau, h):
    v = u.copy()
    inner = tuple(slice(1, -1) for _ in u.shape)
    s = u[inner].copy()
    for p in range(u.ndim):
        c, w, e = _nb(u, u.ndim - 1 - p)
        s = s + (tau * ((w + e) - 2.0 * c)) / (h[p] * h[p])
    v[inner] = s
    return v


def _heatvar(u, k, tau, h):
    v = u.copy()
    inner = tuple(slice(1, -1) for _ in u.shape)
    s = u[inner].copy()
    for p in range(u.ndim):
        c, w, e = _nb(u, u.ndim - 1 - p)
        kc, kw, ke = _nb(k, u.ndim - 1 - p)
        s = s + (tau * (0.5 * (ke + kc) * (e - c) - 0.5 * (kc + kw) * (c - w))) / (h[p] * h[p])
    v[inner] = s
    return v


def _mem(a):
    return np.pad(a, 1)


@pytest.mark.parametrize("kind", ["scales", "tiny", "zeros", "nonfinite"])
@pytest.mark.parametrize("n", [(37,), (19, 23), (70, 9, 13)])
def test_heat_step_limits(ctx, kind, n):
    rng = np.random.default_rng(len(n))
    u = _extreme(rng, tuple(reversed(n)), kind)
    g = capi.geom(n)
    h = [g.h[p] for p in range(len(n))]
    tau = 0.9 / sum(2.0 / q ** 2 for q in h)
    p = capi.Heat7Params(tau=tau, coeff_a=1.0, rhoc_inv=1.0, border_mode=capi.BORDER_KEEP)
    a, b = ctx.upload(_mem(u)), ctx.upload(_mem(0 * u))
    capi.check(ctx.L.scafes_heat7_step_f64(ctx.h, C.byref(g), 1, a.ptr, b.ptr, None, None, None, C.byref(p)))
    got = b.read(_mem(u).shape)[tuple(slice(1, -1) for _ in n)]
    with np.errstate(all="ignore"):
        np.testing.assert_array_equal(got, _heat(u, tau, h))
    a.free()
    b.free()


@pytest.mark.parametrize("kind", ["scales", "tiny", "zeros", "nonfinite"])
@pytest.mark.parametrize("cfg", [-1, 3])
def test_heatvar_steps_limits(ctx, kind, cfg):
    n = (70, 11, 9)
    rng = np.random.default_rng(5)
    u = _extreme(rng, tuple(reversed(n)), kind)
    k = 1.0 + 0.5 * rng.random(u.shape)
    g = capi.geom(n)
    h = [g.h[p] for p in range(3)]
    tau = 0.9 / sum(2.0 * 1.5 / q ** 2 for q in h)
    a, b, kk = ctx.upload(_mem(u)), ctx.upload(_mem(u)), ctx.upload(_mem(k))
    which = C.c_int(0)
    capi.check(ctx.L.scafes_heat7var_run(ctx.h, C.byref(g), 1, capi.HEATVAR_F64, a.ptr, b.ptr, None, None, kk.ptr, tau,
                                         3, capi.BORDER_KEEP, 0.0, cfg, C.byref(which)))
    got = (b if which.value else a).read(_mem(u).shape)[1:-1, 1:-1, 1:-1]
    with np.errstate(all="ignore"):
        for _ in range(3):
            u = _heatvar(u, k, tau, h)
        np.testing.assert_array_equal(got, u)
    for d in (a, b, kk):
        d.free()

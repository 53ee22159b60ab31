"""Column tiles of the two-row var-kappa sweeps: the first tile has no columns to
give up before it and the last none after it."""
import ctypes as C

import numpy as np
import pytest

from masterthesis_amd import capi


@pytest.mark.parametrize("k", [3, 4])
def test_tiles_cover_the_row(k):
    f = capi.load()._ZN6scafes12pair_tiles_xEii
    f.restype, f.argtypes = C.c_int, [C.c_int, C.c_int]
    step = 64 - 2 * k
    for nx in range(3, 1500):
        t = f(nx, k)
        x0 = 1 if f(nx + 1, k) == t else 0  # columns before the row
        stored = []
        for x in range(t):
            first, last = k if x else x0, 63 - k if x < t - 1 else 63
            stored += [q for q in range(x * step - x0 + first, x * step - x0 + last + 1) if q < nx]
        assert stored == list(range(nx)), nx
    assert [f(nx, k) for nx in (60, 64, 65, 120)] == [1, 1, 2, 2]


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [capi.HEATVAR_F32, capi.HEATVAR_F32_KAHAN])
@pytest.mark.parametrize("nx", [59, 60, 61, 63, 64, 65, 66, 119, 120, 121, 122, 123, 176, 177, 180, 181])
@pytest.mark.parametrize("border", [capi.BORDER_KEEP, capi.BORDER_VALUE])
def test_row_ends_match_one_step_launches(hip, mode, nx, border):
    """Three and four steps per sweep against one per launch, NaN ghosts."""
    n, steps = (nx, 9, 6), 11
    rng = np.random.default_rng(nx)
    shape = tuple(m + 2 for m in reversed(n))
    u0, kap = (np.full(shape, np.nan, np.float32) for _ in range(2))
    u0[1:-1, 1:-1, 1:-1] = rng.standard_normal(shape)[1:-1, 1:-1, 1:-1]
    kap[1:-1, 1:-1, 1:-1] = rng.uniform(0.2, 1.5, shape)[1:-1, 1:-1, 1:-1]
    tau = 0.9 / sum(2 * 1.5 * (m - 1) ** 2 for m in n)
    g = capi.geom(n)
    out = []
    with capi.Context(0) as ctx:
        for cfg in (0, 25, 39, -1):
            b = [ctx.upload(x) for x in (u0, u0, 0 * u0, 0 * u0, kap)]
            which = C.c_int(0)
            capi.check(ctx.L.scafes_heat7var_run(ctx.h, C.byref(g), 1, mode, *[x.ptr for x in b], tau, steps, border,
                                                 0.25, cfg, C.byref(which)))
            w = which.value
            out.append([b[q + w].read(shape)[1:-1, 1:-1, 1:-1] for q in ((0, 2) if mode else (0,))])
            for x in b:
                x.free()
    assert np.isfinite(out[0][0]).all()
    for got in out[1:]:
        np.testing.assert_array_equal(got[0], out[0][0])
        if mode == capi.HEATVAR_F32_KAHAN:
            np.testing.assert_array_equal(got[1], out[0][1])

"""scafes_heat7_run_f64 leaves what single steps leave in both buffers."""
import ctypes as C

import numpy as np
import pytest

from masterthesis_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(33, 20, 17), (64, 64, 64), (70, 68, 66), (210, 200, 200), (40, 30), (50,)])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 9])
def test_both_buffers(hip, n, steps):
    rng = np.random.default_rng(steps)
    shape = tuple(m + 2 for m in reversed(n))
    node = tuple(slice(1, -1) for _ in n)
    u0 = np.full(shape, np.nan)
    u0[node] = rng.standard_normal(tuple(reversed(n)))
    g = capi.geom(n)
    tau = 0.9 / (sum(2 * (m - 1.0) ** 2 for m in n) + 1.0)
    p = capi.Heat7Params(tau=tau, coeff_a=1.0, rhoc_inv=1.0, perf_c=1.0, perf_w=1.0, has_perf=1,
                         border_mode=capi.BORDER_KEEP)
    with capi.Context(0) as ctx:
        a, b = ctx.upload(u0), ctx.upload(0 * u0)
        which = C.c_int(0)
        run = ctx.L.scafes_heat7_run_f64
        capi.check(run(ctx.h, C.byref(g), C.c_int(1), a.ptr, b.ptr, C.c_int(steps), C.byref(p), C.byref(which)))
        assert which.value == steps % 2
        got = [x.read(shape)[node] for x in ((b, a) if which.value else (a, b))]
        a.write(u0)
        x, y = a, b
        for _ in range(steps):
            capi.check(ctx.L.scafes_heat7_step_f64(ctx.h, C.byref(g), 1, x.ptr, y.ptr, None, None, None, C.byref(p)))
            x, y = y, x
        for u, want in zip(got, (x, y)):
            np.testing.assert_array_equal(u, want.read(shape)[node])

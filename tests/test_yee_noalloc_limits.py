"""The box sizes scafes_yee_run_noalloc takes: its scratch array of 2^17 energy
partials holds two per workgroup up to 1203 cells per axis with a second buffer
and 1023 without, whatever z chunks the launches take."""
import ctypes as C

import numpy as np
import pytest

from masterthesis_amd import capi

SLOTS = 1 << 17
CUS = 256


def _slots():
    f = capi.load()._ZN6scafes16yee_energy_slotsEiibi
    f.restype, f.argtypes = C.c_long, [C.c_int, C.c_int, C.c_bool, C.c_int]
    return f


@pytest.mark.parametrize("elem", [4, 8])
@pytest.mark.parametrize("second,last", [(True, 1203), (False, 1023)])
def test_partials_fit_up_to_the_documented_box(elem, second, last):
    f = _slots()
    assert [n for n in range(2, last + 1) if f(n, elem, second, CUS) > SLOTS] == []
    assert all(f(n, elem, second, CUS) > SLOTS for n in (last + 1, 1300, 2000))


@pytest.mark.gpu
@pytest.mark.parametrize("code,dt,ncell", [(capi.F32, np.float32, 960), (capi.F64, np.float64, 760)])
def test_large_box_with_second_buffer(hip, code, dt, ncell):
    """One fused step and one two-step sweep, both recorded, against the
    allocating entry point: the same energies."""
    nsteps = 3
    with capi.Context(0) as ctx:
        f, f2 = (ctx.alloc(6 * (ncell + 1) ** 3, dt) for _ in range(2))
        edev = ctx.alloc(nsteps, np.float64)
        which = C.c_int(0)
        capi.check(ctx.L.scafes_yee_init_pulse(ctx.h, ncell, code, f.ptr, 3.0))
        capi.check(ctx.L.scafes_yee_run_noalloc(ctx.h, ncell, code, 0.5, f.ptr, f2.ptr, nsteps, 1, edev.ptr,
                                                C.byref(which)))
        got = edev.read()
        want = np.zeros(nsteps)
        capi.check(ctx.L.scafes_yee_init_pulse(ctx.h, ncell, code, f.ptr, 3.0))
        capi.check(ctx.L.scafes_yee_run(ctx.h, ncell, code, 0.5, f.ptr, f2.ptr, nsteps, 1,
                                        want.ctypes.data_as(C.POINTER(C.c_double)), C.byref(which)))
    assert want[0] > 0.0
    np.testing.assert_array_equal(got, want)

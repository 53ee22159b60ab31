"""Two rows per thread, three and four steps per sweep (FP32 fields): bit-identical
to one-step launches, the same products being rounded in the same order, at the
edges of the 58- and 56-column tiles, of the row tiles and of the z chunks."""
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


def _run(ctx, n, mode, nsteps, cfg, border):
    g = capi.geom(n)
    rng = np.random.default_rng(sum(n))
    shape = tuple(m + 2 for m in reversed(n))
    u0 = rng.standard_normal(shape).astype(np.float32)
    kap = rng.uniform(0.2, 1.5, shape).astype(np.float32)
    tau = 0.9 / sum(2 * 1.5 * (m - 1) ** 2 for m in n)
    bufs = [ctx.upload(u0.ravel()), ctx.upload(u0.ravel()), ctx.upload(np.zeros(u0.size, np.float32)),
            ctx.upload(np.zeros(u0.size, np.float32)), ctx.upload(kap.ravel())]
    a, b, c1, c2, k = bufs
    which = C.c_int(0)
    capi.check(ctx.L.scafes_heat7var_run(ctx.h, C.byref(g), 1, mode, a.ptr, b.ptr, c1.ptr, c2.ptr, k.ptr, tau, nsteps,
                                         border, 0.25, cfg, C.byref(which)))
    out = [(b if which.value else a).read(), (c2 if which.value else c1).read()]
    for d in bufs:
        d.free()
    return out


def _multi_cfgs(L):
    out = []
    for cfg in range(L.scafes_heat7var_num_cfgs()):
        v = [C.c_int() for _ in range(5)]
        capi.check(L.scafes_heat7var_cfg_desc(cfg, *[C.byref(x) for x in v]))
        if v[4].value >= 3:
            out.append(cfg)
    return out


@pytest.mark.parametrize("mode", [capi.HEATVAR_F32, capi.HEATVAR_F32_KAHAN])
@pytest.mark.parametrize("n", [(3, 3, 3), (58, 12, 5), (59, 13, 3), (57, 26, 40), (56, 21, 7), (117, 53, 4)])
def test_every_tile_matches_one_step(ctx, n, mode):
    for border in (capi.BORDER_KEEP, capi.BORDER_VALUE):
        ref = _run(ctx, n, mode, 7, 0, border)
        for cfg in [-1] + _multi_cfgs(ctx.L):
            got = _run(ctx, n, mode, 7, cfg, border)
            for x, y in zip(got, ref):
                np.testing.assert_array_equal(x, y, err_msg=str(cfg))


@pytest.mark.parametrize("mode", [capi.HEATVAR_F32, capi.HEATVAR_F32_KAHAN])
@pytest.mark.parametrize("n,steps", [((131, 113, 107), 4), ((131, 113, 107), 6), ((131, 113, 107), 15),
                                     ((305, 271, 247), 4)])
def test_large_default_matches_one_step(ctx, n, steps, mode):
    """Grids past the size from which the default takes four steps a sweep
    (the last one past the size at which FP32 changes its tile)."""
    ref = _run(ctx, n, mode, steps, 0, capi.BORDER_KEEP)
    for x, y in zip(_run(ctx, n, mode, steps, -1, capi.BORDER_KEEP), ref):
        np.testing.assert_array_equal(x, y)
    g, buf, cnt = capi.geom(n), (C.c_int * 8)(), C.c_int(0)
    capi.check(ctx.L.scafes_heat7var_plan(ctx.h, C.byref(g), 1, mode, steps, buf, 8, C.byref(cnt)))
    assert list(buf[:cnt.value]) == {4: [4], 6: [3, 3], 15: [4, 4, 4, 3]}[steps]


@pytest.mark.parametrize("mode", [capi.HEATVAR_F32, capi.HEATVAR_F32_KAHAN])
def test_gradient_with_states_of_large_grid(ctx, mode):
    """State-writing sweeps on a grid whose plain sweeps take four steps: the
    gradient is the one of single checkpoints (every state recomputed)."""
    n, steps = (131, 113, 107), 11
    g = capi.geom(n)
    rng = np.random.default_rng(3)
    shape = tuple(m + 2 for m in reversed(n))
    u0 = rng.standard_normal(shape).astype(np.float32).ravel()
    kap = rng.uniform(0.2, 1.5, shape).astype(np.float32).ravel()
    tgt = rng.standard_normal(shape).astype(np.float32).ravel()
    tau = 0.9 / sum(2 * 1.5 * (m - 1) ** 2 for m in n)
    outs = []
    for snaps in (1, 16):
        d = [ctx.upload(x) for x in (u0, kap, tgt)]
        gr = ctx.alloc(u0.size, np.float64)
        J = C.c_double(0)
        capi.check(ctx.L.scafes_heat7var_gradient(ctx.h, C.byref(g), 1, mode, d[0].ptr, d[1].ptr, d[2].ptr, tau,
                                                  capi.BORDER_KEEP, 0.0, steps, snaps, gr.ptr, C.byref(J), None))
        outs.append((J.value, gr.read()))
        for x in d + [gr]:
            x.free()
    assert outs[0][0] == outs[1][0]
    np.testing.assert_array_equal(outs[0][1], outs[1][1])

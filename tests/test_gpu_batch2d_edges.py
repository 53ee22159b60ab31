"""Block edges of the batched 2-D ensemble: problem edges on both sides of every
register-block size, odd and even step counts, borders kept."""
import ctypes as C

import numpy as np
import pytest

from masterthesis_amd import capi

pytestmark = pytest.mark.gpu

SIZES = [2, 3, 31, 32, 33, 63, 64, 65, 96, 97, 127, 128, 129, 160, 161, 192, 193, 224, 225, 250, 255, 256]


@pytest.mark.parametrize("steps", [1, 2, 5])
@pytest.mark.parametrize("gradient", [False, True])
def test_block_edges(hip, steps, gradient):
    """u against float64 with the nonzero border untouched; each step rounds a
    value below 4 in at most four operations, so the bound is 4 x 4 x 2^-24 per
    step.  J and dJ/dkappa against the float64 states within that bound's
    effect on the sums."""
    rng = np.random.default_rng(steps)
    n = np.array(SIZES, np.int32)
    off = np.concatenate([[0], np.cumsum(n.astype(np.int64) ** 2)[:-1]])
    kappa = rng.uniform(0.1, 1.0, len(n)).astype(np.float32)
    tau = (0.9 / 4.0 / (n - 1.0) ** 2).astype(np.float32)
    u0 = rng.uniform(-1, 1, int((n.astype(np.int64) ** 2).sum())).astype(np.float32)
    tgt = rng.uniform(-1, 1, u0.size).astype(np.float32)
    with capi.Context(0) as ctx:
        d = [ctx.upload(a) for a in (n, off, kappa, tau, np.arange(len(n), dtype=np.int32)[::-1].copy(), u0, tgt)]
        J, G = ctx.alloc(len(n)), ctx.alloc(len(n))
        p = [x.ptr for x in d]
        capi.check(ctx.L.scafes_batch2d_run(ctx.h, len(n), p[0], p[1], p[2], p[3], p[4], p[5],
                                            p[6] if gradient else None, J.ptr if gradient else None,
                                            G.ptr if gradient else None, steps, 0))
        got, j, gr = d[5].read(), J.read(), G.read()
    tol = 16 * steps * 2.0 ** -24
    for q, m in enumerate(SIZES):
        sl = slice(int(off[q]), int(off[q]) + m * m)
        u = u0[sl].astype(np.float64).reshape(m, m)
        g = got[sl].reshape(m, m)
        k = float(tau[q]) * float(kappa[q]) * (m - 1.0) ** 2
        lap = np.zeros((0, 0))
        for _ in range(steps):
            lap = u[1:-1, :-2] + u[1:-1, 2:] + u[:-2, 1:-1] + u[2:, 1:-1] - 4 * u[1:-1, 1:-1]
            u[1:-1, 1:-1] += k * lap
        border = np.ones((m, m), bool)
        border[1:-1, 1:-1] = False
        assert np.array_equal(g[border], u0[sl].reshape(m, m)[border]), m
        np.testing.assert_allclose(g, u, rtol=0, atol=tol, err_msg=str(m))
        if gradient and m > 2:
            r = (u - tgt[sl].reshape(m, m))[1:-1, 1:-1]
            cells = (m - 2.0) ** 2
            assert abs(j[q] - 0.5 * (r * r).sum()) <= 4 * tol * cells, m
            scale = steps * float(tau[q]) * (m - 1.0) ** 2
            assert abs(gr[q] - scale * (r * lap).sum()) <= scale * 32 * tol * cells, m

"""Batched 2-D ensemble: barriers where waves of a workgroup run different loops,
and the edge of the workgroup."""
import os
import re

import numpy as np
import pytest

from masterthesis_amd import capi

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "masterthesis_amd", "csrc",
                   "batch2d.hip")


def test_no_block_barrier_in_the_loops_that_waves_choose_between():
    """__syncthreads wants every thread at the same call; the masked and the plain
    loop each have their own, so they use the wave-counting barrier instead, in
    equal numbers because both are one body."""
    src = open(SRC).read()
    body = re.search(r"auto steps = \[&\].*?\n    \};\n", src, re.S).group(0)
    assert "__syncthreads" not in body and body.count("wave_barrier()") == 2
    assert re.search(r"if \(plain\) steps\(false\);\s*else steps\(true\);", src)


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [np.inf, np.nan, 3e38])
@pytest.mark.parametrize("gradient", [False, True])
def test_border_untouched_by_the_far_side_of_a_block(hip, bad, gradient):
    """One step with a value that is not finite (or overflows in a sum) in the
    columns and rows at the inner side of the outermost blocks: none is next to a
    border node, so every border node keeps its value."""
    sizes = [65, 96, 97, 128, 160, 192, 224, 225, 255, 256]
    n = np.array(sizes, np.int32)
    off = np.concatenate([[0], np.cumsum(n.astype(np.int64) ** 2)[:-1]])
    rng = np.random.default_rng(3)
    kappa = rng.uniform(0.1, 1.0, len(n)).astype(np.float32)
    tau = (0.9 / 4.0 / (n - 1.0) ** 2).astype(np.float32)
    u0 = rng.uniform(-1, 1, int((n.astype(np.int64) ** 2).sum())).astype(np.float32)
    for q, m in enumerate(sizes):
        b = (m + 31) // 32
        u = u0[off[q]:off[q] + m * m].reshape(m, m)  # a view
        for at in (b - 1, 31 * b):
            if 2 <= at <= m - 3:
                u[at, 2:-2] = bad
                u[2:-2, at] = bad
    with capi.Context(0) as ctx:
        d = [ctx.upload(a) for a in (n, off, kappa, tau, np.arange(len(n), dtype=np.int32), u0, np.zeros_like(u0))]
        J, G = ctx.alloc(len(n)), ctx.alloc(len(n))
        p = [x.ptr for x in d]
        capi.check(ctx.L.scafes_batch2d_run(ctx.h, len(n), *p[:6], p[6] if gradient else None,
                                            J.ptr if gradient else None, G.ptr if gradient else None, 1, 0))
        got = d[5].read()
    for q, m in enumerate(sizes):
        border = np.ones((m, m), bool)
        border[1:-1, 1:-1] = False
        sl = slice(int(off[q]), int(off[q]) + m * m)
        np.testing.assert_array_equal(got[sl].reshape(m, m)[border], u0[sl].reshape(m, m)[border], err_msg=str(m))

"""The first work of a fresh context."""
import ctypes as C
import glob
import os
import re

import numpy as np
import pytest

from masterthesis_amd import capi

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "masterthesis_amd", "csrc")


def test_nothing_runs_on_the_null_stream():
    """Contexts work on non-blocking streams, which the null stream is not ordered with."""
    for path in glob.glob(os.path.join(CSRC, "*.hip")):
        src = re.sub(r"//[^\n]*", "", open(path).read())
        assert not re.search(r"\bhip(Memset|Memcpy)\s*\(", src), path


@pytest.mark.gpu
def test_reductions_right_after_creation(hip):
    """Reductions over one block, several (the block counter) and many."""
    for n in ((32, 24, 20), (4, 4, 4), (60, 60, 60), (64, 24, 20)) * 3:
        g = capi.geom(n)
        a = np.ones(tuple(m + 2 for m in reversed(n)))
        out = C.c_double(0)
        with capi.Context(0) as ctx:
            d = ctx.upload(a)
            for _ in range(2):
                capi.check(ctx.L.scafes_reduce(ctx.h, C.byref(g), capi.F64, d.ptr, 1, d.ptr, 1, capi.RED_SUM_PROD, 0,
                                               C.byref(out)))
                assert out.value == float(np.prod(n))

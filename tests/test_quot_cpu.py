"""The quotient by a divisor known in advance (csrc/exact_quot.hpp), restated
with the C library's fma: equal to the IEEE division for every divisor h^2 of
the grids and for dividends whose quotient lies next to a rounding boundary."""
import ctypes
import math
import os
import random
import subprocess

import numpy as np
import pytest

_m = ctypes.CDLL("libm.so.6")
_m.fma.restype = ctypes.c_double
_m.fma.argtypes = [ctypes.c_double] * 3
fma = _m.fma


def quot(x, d):
    z = 1.0 / d
    t = fma(-d, z, 1.0) / d
    q = fma(x, z, x * t)
    return fma(fma(-q, d, x), z, q)


def _dividends(rng, d):
    yield 0.0
    for _ in range(40):
        x = rng.uniform(-1.0, 1.0) * 2.0 ** rng.randint(-890, 900)
        yield x
        # a quotient next to the middle of two doubles: x = RN((q + ulp/2) d) +- a few ulps
        q = x / d
        if not math.isfinite(q):
            continue
        m, e = math.frexp(q)
        num = (int(m * 2 ** 53) * 2 + 1)
        dm, de = math.frexp(d)
        prod = num * int(dm * 2 ** 53)
        y = math.ldexp(float(prod), e + de - 54 - 53)
        for k in range(-2, 3):
            v = y
            for _ in range(abs(k)):
                v = math.nextafter(v, math.inf if k > 0 else -math.inf)
            yield v


@pytest.mark.parametrize("seed", range(4))
def test_quotient_equals_division(seed):
    rng = random.Random(seed)
    divisors = [(1.0 / (n - 1)) ** 2 for n in rng.sample(range(2, 2000), 60)]
    divisors += [rng.uniform(0.5, 1.0) * 2.0 ** rng.randint(-199, 59) for _ in range(60)]
    for d in divisors:
        for x in _dividends(rng, d):
            if x != 0.0 and not (2.0 ** -900 <= abs(x) <= 2.0 ** 900):
                continue
            want, got = x / d, quot(x, d)
            # an overflow leaves a NaN, which sends the kernel to the division
            assert got == want or (math.isinf(want) and math.isnan(got)), (x.hex(), d.hex())


DRIVER = r"""
#include <algorithm>
using std::min;
#include "exact_quot.hpp"
extern "C" void sums(const double* hh, int dim, long count, const double* v, const double* x, double* got,
                     double* want)
{
    const scafes::ByHH c = scafes::make_by_hh(hh);
    for (long i = 0; i < count; ++i) {
        const double* y = x + 3 * i;
        got[i] = scafes::add_by_hh(c, dim, v[i], y[0], y[1], y[2]);
        double r = v[i] + y[0] / hh[0];
        if (dim > 1) r += y[1] / hh[1];
        if (dim > 2) r += y[2] / hh[2];
        want[i] = r;
    }
}
"""


@pytest.fixture(scope="module")
def sums(tmp_path_factory):
    """The header's own sum, built for the CPU."""
    d = tmp_path_factory.mktemp("quot")
    (d / "q.cpp").write_text(DRIVER)
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "masterthesis_amd", "csrc")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-w", "-shared", "-fPIC",
                           "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + csrc, str(d / "q.cpp"), "-o",
                           str(d / "q.so")])
    p = np.ctypeslib.ndpointer(np.float64, flags="C")
    f = ctypes.CDLL(str(d / "q.so")).sums
    f.restype, f.argtypes = None, [p, ctypes.c_int, ctypes.c_long, p, p, p, p]
    return f


@pytest.mark.parametrize("dim", [1, 2, 3])
@pytest.mark.parametrize("hh", [(100.0, 0.3, 7.0), (2.0 ** -12, 2.0 ** 40 / 3, 1e-8), (1.1, 2.0 ** -200, 2.0 ** 60)])
def test_sum_equals_divisions_at_every_magnitude(sums, dim, hh):
    """Dividends from the smallest subnormal (those without a bit in the upper
    word among them) over the bound at 2^-900 to overflow, zeros mixed in."""
    rng = np.random.default_rng(dim)
    n = 200000
    x = np.ldexp(rng.uniform(-2, 2, (n, 3)), rng.integers(-1074, 1023, (n, 3)))
    low = np.ldexp(rng.integers(-2 ** 40, 2 ** 40, (n, 3)).astype(float) // 2.0 ** rng.integers(0, 40, (n, 3)), -1074)
    pick = rng.integers(0, 4, (n, 3))
    x = np.where(pick == 0, 0.0, np.where(pick == 1, low, x))
    x[: n // 4] = np.where(pick[: n // 4] == 0, 0.0, low[: n // 4])  # every dividend of the sum subnormal
    edge = 2.0 ** -900
    x[-6:, 0] = [edge, -edge, np.nextafter(edge, 0), np.nextafter(edge, 1), 5e-324, -0.0]
    v = np.where(rng.random(n) < 0.5, 0.0, np.ldexp(rng.uniform(-2, 2, n), rng.integers(-1074, -1000, n)))
    got, want = np.empty(n), np.empty(n)
    sums(np.array(hh), dim, n, v, np.ascontiguousarray(x), got, want)
    np.testing.assert_array_equal(got, want)

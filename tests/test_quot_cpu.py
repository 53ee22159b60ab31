"""The quotient by a divisor known in advance (csrc/exact_quot.hpp), restated
with the C library's fma: equal to the IEEE division for every divisor h^2 of
the grids and for dividends whose quotient lies next to a rounding boundary."""
import ctypes
import math
import random

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

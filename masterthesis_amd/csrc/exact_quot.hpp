// exact_quot.hpp -- the FP64 updates' sums v + x0/h0^2 + x1/h1^2 + x2/h2^2
// with correctly rounded quotients by divisors that are known before the
// launch: the CPU path divides, so the FP64 results must be RN(x / d).
//
// With z = RN(1/d) and the tail t = RN(1/d - z) (host),
//   q = fma(x, z, x*t)     x/d to half an ulp plus 2^-52 ulp: within one ulp
//   e = fma(-q, d, x)      exact remainder
//   fma(e, z, q)           RN(x/d)
// The last step is Markstein's theorem (Computation of elementary functions
// on the IBM RISC System/6000 processor, 1990; Muller et al., Handbook of
// Floating-Point Arithmetic, section on division with an FMA): z correctly
// rounded, q within one ulp, e exact, no underflow or overflow on the way,
// d's significand not all ones.  The remainder is exact while x is zero or
// |x| > 2^-900; a smaller x, and any overflow, infinity or NaN (each leaves a
// NaN in the sum), takes the divisions instead.  A divisor outside
// [2^-200, 2^60] gets a NaN reciprocal, so it always does.  Sums equal the
// divisions' bit for bit, but for the sign of a zero sum at most.
//
// Four full-rate instructions stand for the eleven of a division, one of them
// the quarter-rate reciprocal.  Measured on an MI355X, us, divisions ->
// quotients: var-kappa FP64 three-step sweep 512^3 1890 -> 1490; 50 steps at
// 201x150x131 1211 -> 996; one constant-coefficient step 300x200x200 (bound by
// memory) 60 -> 57; MRI step 120x120x50 15.6 -> 15.0.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <limits>

namespace scafes {

struct ByHH {
    double d[3], z[3], t[3];  // h_p^2, its reciprocal and the reciprocal's tail
};

inline ByHH make_by_hh(const double hh[3])
{
    ByHH r;
    for (int p = 0; p < 3; ++p) {
        const double d = hh[p];
        int e = 0;
        const double m = std::frexp(d, &e);
        const bool ok = d >= std::ldexp(1.0, -200) && d <= std::ldexp(1.0, 60) && m != 1.0 - std::ldexp(1.0, -53);
        r.d[p] = d;
        r.z[p] = ok ? 1.0 / d : std::numeric_limits<double>::quiet_NaN();
        r.t[p] = ok ? std::fma(-d, r.z[p], 1.0) / d : 0.0;
    }
    return r;
}

// Exponent and leading significand bits of |x| from the 64-bit pattern minus one:
// zero alone wraps to the largest value, so one comparison finds the nonzero
// values below a bound, subnormals without a bit in their upper word included
// (one 64-bit shift-and-add).
__device__ inline unsigned small_key(double x)
{
    return (unsigned)(((__builtin_bit_cast(unsigned long long, x) << 1) - 1ull) >> 32);
}

__device__ inline double quot(const ByHH& c, int p, double x)
{
    const double q = __builtin_fma(x, c.z[p], x * c.t[p]);
    return __builtin_fma(__builtin_fma(-q, c.d[p], x), c.z[p], q);
}

// v + x0/hh0 (+ x1/hh1 (+ x2/hh2)), added in this order.
__device__ inline double add_by_hh(const ByHH& c, int dim, double v, double x0, double x1, double x2)
{
    constexpr unsigned kSmall = (1023u - 900u) << 21;  // small_key(2^-900) + 1
    unsigned k = small_key(x0);
    double r = v + quot(c, 0, x0);
    if (dim > 1) {
        k = min(k, small_key(x1));
        r += quot(c, 1, x1);
    }
    if (dim > 2) {
        k = min(k, small_key(x2));
        r += quot(c, 2, x2);
    }
    if (__builtin_expect(k < kSmall || !(r == r), 0)) {
        r = v + x0 / c.d[0];
        if (dim > 1) r += x1 / c.d[1];
        if (dim > 2) r += x2 / c.d[2];
    }
    return r;
}

}  // namespace scafes

// heatvar_ops.hpp -- per-node arithmetic of the variable-kappa heat update
// and of its kappa adjoint, shared by the multi-step kernels (heatvar_tb2.hip,
// heatvar_adjk.hip); the one-step operators in stencil3d.hip use the same
// operation order.
#ifndef SCAFES_HEATVAR_OPS_HPP_
#define SCAFES_HEATVAR_OPS_HPP_

#include <hip/hip_runtime.h>

#include "exact_quot.hpp"

namespace scafes {

struct VarCoef {
    ByHH hh;                    // FP64 path (CPU operation order)
    double tau;
    float c0, c1, c2;           // 0.5*tau/h_p^2, FP32 paths
    double border_value;
    int border_mode;
};

// Face coefficient between the centre and one neighbour: 0.5*(k_nb + k_c)
// in the FP64 path (the CPU path's grouping), k_nb + k_c in FP32 (the 0.5 is
// folded into c_p).  IEEE addition is commutative, so the face shared by two
// nodes has one value.
template <typename T, int MODE>
__device__ inline T face(T a, T b)
{
    if constexpr (MODE == 0)
        return 0.5 * (a + b);
    else
        return a + b;
}

template <typename T>
struct Faces {
    T e, w, n, s, u, d;
};

// One explicit step at one interior node from its six face coefficients.
// MODE 0: FP64 in the CPU path's order; 1: FP32; 2: FP32 + Kahan (cin -> *cout).
template <typename T, int MODE>
__device__ inline T var_update(const VarCoef& cf, T uc, T uw, T ue, T us, T un, T ud, T uu, const Faces<T>& f, T cin,
                               T* cout)
{
    if constexpr (MODE == 0) {
        *cout = T(0);
        return (T)add_by_hh(cf.hh, 3, uc, cf.tau * (f.e * (ue - uc) - f.w * (uc - uw)),
                            cf.tau * (f.n * (un - uc) - f.s * (uc - us)),
                            cf.tau * (f.u * (uu - uc) - f.d * (uc - ud)));
    } else {
        float d = cf.c0 * __builtin_fmaf(f.e, ue - uc, -(f.w * (uc - uw)));
        d = __builtin_fmaf(cf.c1, __builtin_fmaf(f.n, un - uc, -(f.s * (uc - us))), d);
        d = __builtin_fmaf(cf.c2, __builtin_fmaf(f.u, uu - uc, -(f.d * (uc - ud))), d);
        if constexpr (MODE == 2) {
            const float y = d + cin;
            const float t = uc + y;
            *cout = y - (t - uc);
            return t;
        } else {
            *cout = 0.0f;
            return uc + d;
        }
    }
}

struct AdjVarCoef {
    VarCoef v;                // lam update (the forward step's arithmetic)
    float f0, f1, f2;         // 0.5 th_p, th_p = tau / h_p^2, rounded to FP32 (exactly half of th_p rounded)
};

// The two faces of an axis in FP32; a face outside the grid adds nothing.
__device__ inline float adj_face_sum_f(bool lo, bool hi, float lc, float lm, float lp, float uc, float um, float up)
{
    const float a = lo ? (lc - lm) * (um - uc) : 0.0f;
    const float b = hi ? (lc - lp) * (up - uc) : 0.0f;
    return a + b;
}

// Kappa-gradient term of one adjoint step at a node of a 3-D grid, FP32 fields,
//   t = sum_p th_p * sum_{nb = -+e_p in the grid} (lam_c - lam_nb)(u_nb - u_c);
// returns the increment 0.5 t the FP64 gradient adds, formed in FP32 with the
// coefficients 0.5 th_p rounded to FP32 and the axes joined with fmaf, which is
// 0.5 times the term formed with th_p rounded to FP32 (scaling by 2^-1 is exact
// at every rounding step away from the subnormal range), so no FP64 multiply is
// left per term.  The one-step operator in stencil3d.hip uses the same
// arithmetic, so every schedule gives the same gradient; FP64 fields take that
// one only.
__device__ inline double adj_term3(const AdjVarCoef& cf, bool xlo, bool xhi, bool ylo, bool yhi, bool zlo, bool zhi,
                                   float lc, float lw, float le, float ls, float ln, float ld, float lu, float uc,
                                   float uw, float ue, float us, float un, float ud, float uu)
{
    float t = cf.f0 * adj_face_sum_f(xlo, xhi, lc, lw, le, uc, uw, ue);
    t = __builtin_fmaf(cf.f1, adj_face_sum_f(ylo, yhi, lc, ls, ln, uc, us, un), t);
    t = __builtin_fmaf(cf.f2, adj_face_sum_f(zlo, zhi, lc, ld, lu, uc, ud, uu), t);
    return (double)t;
}

}  // namespace scafes
#endif

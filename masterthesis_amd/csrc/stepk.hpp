// stepk.hpp -- K = 2 or 3 steps of a one-field update per sweep (temporal
// blocking) on 3-D grids whose border nodes are kept or take a constant: the
// operators of stencil3d.hip (Op::inner), so the result is bit-identical to K
// one-step launches, the compensation included.
//
// A 64 x TY workgroup streams z planes; iteration k computes level 1 (after
// one step) at plane k and level L at plane k - (L - 1) from level L - 1's LDS
// plane of the iteration before (in-plane neighbours) and its register ring (z
// neighbours), one barrier per plane; level L is valid L - 1 nodes inside the
// tile, level K on the (64 - 2 (K-1)) x (TY - 2 (K-1)) output tile.  The
// centre-only fields of a node ride in register rings; a compensation passes
// from level to level.  The plane loop is unrolled by the ring size, so rings
// cost no moves; loads and stores are issued by every thread, unneeded ones at
// an out-of-range offset.  MO: the states after 1..K-1 steps are written too.
//
// Tile: FP32 64 x 16 (56 VGPRs: two 16-wave workgroups per CU; 64 x 12 took 92
// us per three-step sweep at 256^3 against 87), FP32 + Kahan and FP64 64 x 12.
// On grids that the 256 MB Infinity Cache holds the one-step rows read from
// it at more than twice the HBM rate and a sweep's recomputed rings cost about
// what it saves; beyond it, and where launches bound the time, sweeps win.
// Measured on an MI355X, us per step, one-step rows -> three-step sweeps: Pennes
// FP32 64^3 2.6 -> 2.5, 97x80x75 4.2 -> 3.2, 128^3 7.0 -> 6.8, 201x150x131 11.3 ->
// 9.1, 256^3 47 -> 29; with the states in between written 4.2 -> 3.6, 7.0 -> 7.9, 11.3
// -> 10.3, 47 -> 42; FP32 + Kahan 97x80x75 5.0 -> 3.5, 128^3 9.5 -> 7.3, 256^3 79 ->
// 43; FP64 128^3 12.5 -> 12.5, 201x150x131 20.5 -> 20.1, 256^3 106 -> 71; heat FP64
// 64^3 3.7 -> 3.6, 128^3 9.5 -> 10.9, 256^3 61 -> 47.  Under the Tumor border the
// sweep lost to the rows up to 201x150x131 (13.8 against 12.2 us).
#pragma once

#include "buffer_chunk.hpp"
#include "scafes_common.hpp"

namespace scafes {

// An update's inputs at one node, and what it leaves (value, compensation,
// gradient increment).
template <typename T>
struct St7 {
    T c, w, e, s, n, d, u;  // centre, x-, x+, y-, y+, z-, z+
};

template <typename T>
struct Res {
    T v, c;
    double g;
};

struct StepMid {
    void* v[2];  // states after one and two steps
    void* c[2];  // their compensations
};

constexpr int kStepZC = 32;

template <class Op, typename T, int TY, int K, bool MO>
__global__ __launch_bounds__(64 * TY) void stepk_kernel(Op op, Geo g, StepMid mid, int zc, int tiles_x, int tiles_y)
{
    using namespace chunk;
    static_assert(K == 2 || K == 3, "two or three steps");
    constexpr int TX = 64, D = 2, R = K - 1, OX = TX - 2 * R, OY = TY - 2 * R, H = 3, U = 6;
    constexpr bool KH = Op::kComp;
    constexpr int NC = Op::kNX - (KH ? 1 : 0), NCA = NC > 0 ? NC : 1;
    auto ring = [](int c) { return ((c % H) + H) % H; };
    __shared__ T s0[2][TY + 2][TX + 2];  // level-0 plane with ring
    __shared__ T sl[K - 1][2][TY][TX];   // levels 1..K-1
    const int tx = threadIdx.x;
    const int ty = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    const int lb = xcd_remap(blockIdx.x, gridDim.x);
    const int per_plane = tiles_x * tiles_y;
    const int tz = lb / per_plane;
    const int r = lb - tz * per_plane;
    const int tyi = r / tiles_x, txi = r - tyi * tiles_x;
    const int i = txi * OX - R + tx, j = tyi * OY - R + ty;
    const int ic = min(max(i, 0), g.nx - 1), jc = min(max(j, 0), g.ny - 1);
    const bool out = tx >= R && tx <= TX - 1 - R && i < g.nx && ty >= R && ty <= TY - 1 - R && j < g.ny;
    const bool inner_xy = (i >= g.nl0) & (i <= g.nx - 1 - g.nl0) & (j >= g.nl1) & (j <= g.ny - 1 - g.nl1);
    const int k0 = tz * zc, k1 = min(k0 + zc, g.nz);
    const int kstart = k0 - R, kend = k1 + R - 1;
    const bool hx = (tx == 0) || (tx == TX - 1), hy = (ty == 0) || (ty == TY - 1);
    const int hxi = (tx == 0) ? max(ic - 1, 0) : min(ic + 1, g.nx - 1);
    const int hyj = (ty == 0) ? max(jc - 1, 0) : min(jc + 1, g.ny - 1);
    // x ring: a lane off the ring reloads and rewrites its own centre value
    const int sxc = hx ? ((tx == 0) ? 0 : TX + 1) : tx + 1;
    const int syh = (ty == 0) ? 0 : TY + 1;
    // clamped LDS neighbours: only values that are discarded read a clamped slot
    const int txm = max(tx - 1, 0), txp = min(tx + 1, TX - 1);
    const int tym = max(ty - 1, 0), typ = min(ty + 1, TY - 1);
    constexpr uint32_t B = sizeof(T);
    const uint32_t oc = (uint32_t)(g.base + ic + g.e0 * jc) * B;
    const uint32_t ohx = hx ? (uint32_t)(g.base + hxi + g.e0 * jc) * B : oc;
    const uint32_t ohy = hy ? (uint32_t)(g.base + ic + g.e0 * hyj) * B : kSkip;
    const uint32_t oo = out ? oc : kSkip;
    const uint32_t pb = (uint32_t)(g.e01 * B);
    const int kbase = max(kstart - 1, 0);
    const size_t lift = (size_t)kbase * g.e01 * B;
    auto pl = [&](int kk) { return (uint32_t)(min(max(kk, kbase), g.nz - 1) - kbase) * pb; };
    const Rsrc ra = chunk_rsrc((const char*)op.a + lift), rout = chunk_rsrc((char*)op.out + lift);
    Rsrc rx[NCA], rci, rco, rm[2], rmc[2];
#pragma unroll
    for (int q = 0; q < NC; ++q) rx[q] = chunk_rsrc((const char*)op.x[q] + lift);
    if constexpr (KH) {
        rci = chunk_rsrc((const char*)op.x[NC] + lift);
        rco = chunk_rsrc((char*)op.cout + lift);
    }
    if constexpr (MO) {
#pragma unroll
        for (int q = 0; q < R; ++q) {
            rm[q] = chunk_rsrc((char*)mid.v[q] + lift);
            if constexpr (KH) rmc[q] = chunk_rsrc((char*)mid.c[q] + lift);
        }
    }

    T qa[D], qax[D], qay[D], qc[D], qx[NCA][D];
    auto fetch = [&](const int s, const int kk) {
        const uint32_t p = pl(kk);
        qa[s] = cload<T>(ra, oc, p);
        qax[s] = cload<T>(ra, ohx, p);
        qay[s] = cload<T>(ra, ohy, p);
#pragma unroll
        for (int q = 0; q < NC; ++q) qx[q][s] = cload<T>(rx[q], oc, p);
        if constexpr (KH) qc[s] = cload<T>(rci, oc, p);
    };
#pragma unroll
    for (int s = 0; s < D; ++s) fetch(s, kstart + s);
    // hist[l][ring(it)]: level l at the plane of iteration it; xh: the
    // centre-only fields; cp[l]: level l's compensation one iteration ago
    T hist[K][H], xh[NCA][H], cp[K];
#pragma unroll
    for (int l = 0; l < K; ++l) {
        cp[l] = T(0);
#pragma unroll
        for (int a = 0; a < H; ++a) hist[l][a] = T(0);
    }
#pragma unroll
    for (int q = 0; q < NCA; ++q)
#pragma unroll
        for (int a = 0; a < H; ++a) xh[q][a] = T(0);
    hist[0][ring(-1)] = cload<T>(ra, oc, pl(kstart - 1));
    for (int kb = kstart; kb <= kend; kb += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = kb + u;
            if (k > kend) return;  // uniform over the workgroup
            const int s = u % D, buf = u & 1, pbf = buf ^ 1;
            const T ac = qa[s], ap = qa[(s + 1) % D], am = hist[0][ring(u - 1)];
            hist[0][ring(u)] = ac;
#pragma unroll
            for (int q = 0; q < NC; ++q) xh[q][ring(u)] = qx[q][s];
            T cold[K];
#pragma unroll
            for (int l = 0; l < K; ++l) cold[l] = cp[l];
            if constexpr (KH) cold[0] = qc[s];
            s0[buf][ty + 1][tx + 1] = ac;
            s0[buf][ty + 1][sxc] = qax[s];
            if (hy) s0[buf][syh][tx + 1] = qay[s];
            fetch(s, k + D);
            __syncthreads();
#pragma unroll
            for (int L = 1; L <= K; ++L) {
                const int p = k - (L - 1);
                const bool plane_out = p >= k0 && p < k1;
                // computed at every position of the rows the level above reads
                // (wave-uniform), kept where the step does not update
                const bool inner = inner_xy && p >= g.nl2 && p <= g.nz - 1 - g.nl2;
                Res<T> res{};
                if (L == 1 || (ty >= L - 1 && ty <= TY - L && (L < K || plane_out))) {
                    St7<T> st;
                    if (L == 1)
                        st = St7<T>{ac, s0[buf][ty + 1][tx], s0[buf][ty + 1][tx + 2], s0[buf][ty][tx + 1],
                                    s0[buf][ty + 2][tx + 1], am, ap};
                    else
                        st = St7<T>{hist[L - 1][ring(u - 1)], sl[L - 2][pbf][ty][txm], sl[L - 2][pbf][ty][txp],
                                    sl[L - 2][pbf][tym][tx], sl[L - 2][pbf][typ][tx], hist[L - 1][ring(u - 2)],
                                    hist[L - 1][ring(u)]};
                    T xv[Op::kNX > 0 ? Op::kNX : 1];
#pragma unroll
                    for (int q = 0; q < NC; ++q) xv[q] = xh[q][ring(u - (L - 1))];
                    if constexpr (KH) xv[NC] = cold[L - 1];
                    op.inner(3, st, xv, res);
                    if (!inner) {
                        res.v = op.kept(st.c);
                        if constexpr (KH) res.c = xv[NC];
                    }
                }
                const uint32_t os = plane_out ? oo : kSkip;
                if (L < K) {
                    hist[L][ring(u)] = res.v;
                    sl[L - 1][buf][ty][tx] = res.v;
                    if constexpr (KH) cp[L] = res.c;
                    if constexpr (MO) {
                        cstore<T>(res.v, rm[L - 1], os, pl(p));
                        if constexpr (KH) cstore<T>(res.c, rmc[L - 1], os, pl(p));
                    }
                } else {
                    cstore<T>(res.v, rout, os, pl(p));
                    if constexpr (KH) cstore<T>(res.c, rco, os, pl(p));
                }
            }
        }
    }
}

// 3-D grids whose chunk offsets (the z chunk, the pipeline's planes and a
// plane) fit the 31-bit buffer range.
inline bool stepk_supported(const Geo& g, int elem_bytes)
{
    return g.dim == 3 &&
           ((long)(kStepZC + 8) * g.e01 + g.base + g.e01) * (long)elem_bytes < (long)chunk::kRecords;
}

template <class Op, typename T, int K, bool MO>
int stepk_launch(Ctx* c, const Op& op, const Geo& g, const StepMid& mid)
{
    constexpr int R = K - 1, TY = sizeof(T) == 4 && !Op::kComp ? 16 : 12;
    const int tiles_x = ceil_div(g.nx, 64 - 2 * R), tiles_y = ceil_div(g.ny, TY - 2 * R);
    const int zc = fit_chunk((long)tiles_x * tiles_y, g.nz, 2 * R + 1, kStepZC, sizeof(T) == 4 ? 2 : 1, c->cu_count);
    const long nb = (long)tiles_x * tiles_y * ceil_div(g.nz, zc);
    if (nb > 0x7fffffffL) return fail(SCAFES_ERR_ARG, "grid too large");
    stepk_kernel<Op, T, TY, K, MO><<<dim3((unsigned)nb), dim3(64, TY), 0, c->stream>>>(op, g, mid, zc, tiles_x,
                                                                                       tiles_y);
    SCAFES_HIP(hipGetLastError());
    return SCAFES_OK;
}

}  // namespace scafes

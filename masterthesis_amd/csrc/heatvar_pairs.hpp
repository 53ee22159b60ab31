// heatvar_pairs.hpp -- three or four time steps per HBM sweep of the
// variable-kappa heat update on 3-D grids, FP32 fields, two rows per thread;
// bit-identical to the one-step kernel.
//
// With one node per thread the sweeps of heatvar_tb2.hip issue about as many LDS
// cycles as vector cycles (16 reads and 8 writes of a wavefront per plane for
// three levels, two cycles each for the whole CU), and their 64x12 tile computes
// 1.6 nodes per stored one.  Here
//   - a wavefront is a 64-lane row pair: x neighbours come from the lanes beside
//     (DPP, one vector instruction, instead of an LDS read), so the tile gives up K
//     columns on each inner side and needs no x ring; rows of up to 64 nodes are one
//     tile (60 nodes as two: 24 steps at 60x512x512 FP32 674 us, as one 382);
//   - each product of a face and the difference across it is formed once and used by
//     both nodes (lane below, row below, plane before), which also drops the west,
//     south and lower faces and the second old plane of each level;
//   - LDS carries only the rows that the wavefronts above and below read: 8 reads and
//     10 writes per row pair and plane for three levels (48 before).
// 78-128 vector registers, no spills.  The faces and prefetch slots are rings
// indexed by the unrolled plane (four planes; six for three steps cost 15
// registers more).  Measured on an MI355X, us for 20 steps of FP32 + Kahan at 512^3
// 5620 -> 3460 (three steps of one sweep 800 -> 710, four 1084 -> 690); FP32 at
// 512^3, four steps, 637 (three) -> 511; 24 steps, FP32 + Kahan 128^3 188 -> 135, 256^3
// 943 -> 558, 97x80x75 93 -> 81.  What is left at 512^3 is the copy rate: 2.7 GB per
// sweep take 565 us.  FP64 keeps one node per thread: this form needs 174 registers
// (two wavefronts per SIMD) and took 353 us against 321 for 24 steps at 128^3 and 2541
// against 2509 at 300x320x280.
#pragma once

#include "heatvar_ops.hpp"
#include "plane_buffer.hpp"
#include "scafes_common.hpp"

namespace scafes {

// Planes of a workgroup's z chunk at most, and the grids from which four steps
// a sweep are the default (FP32 and FP32 + Kahan; us for 24 steps as three /
// four per sweep, FP32 + Kahan: 64^3 70 / 67, 97x80x75 81 / 78, 128^3 145 / 135,
// 256^3 720 / 558; 512^3, per step, 237 / 172).
constexpr int kPairZC = 128;
constexpr long kFourStepNodes = 1500000;

// The value of the neighbouring lane of the wavefront (0 past its ends).
template <int CTRL>
__device__ inline float lane_shift(float v)
{
    return __builtin_bit_cast(float,
                              __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
__device__ inline float lane_above(float v)
{
    return lane_shift<0x130>(v);  // wave_shl:1, lane + 1
}
__device__ inline float lane_below(float v)
{
    return lane_shift<0x138>(v);  // wave_shr:1, lane - 1
}

struct PairFaces {
    float e[2], n[3], u[2];  // x+ and z+ face of each row; y faces below, between and above them
};

// One step at two rows: v, their values; ys and yn, the rows below and above;
// up, the plane above; pz, the product of the lower z face (replaced by the
// upper one's).  The product of a face is the same for the nodes on both
// sides of it, so the x- one comes from the lane below, the z- one from the
// plane before and the one between the rows is formed once.  Rounding as in
// var_update.
template <int MODE>
__device__ inline void pair_update(const VarCoef& cf, const float (&v)[2], float ys, float yn, const float (&up)[2],
                                   const PairFaces& f, float (&pz)[2], const float (&cin)[2], float (&out)[2],
                                   float (&cout)[2])
{
    const float ds = v[0] - ys, dm = v[1] - v[0], dn = yn - v[1];
    const float dy[2] = {dm, dn}, py[2] = {f.n[0] * ds, f.n[1] * dm};
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const float dx = lane_above(v[r]) - v[r];
        const float dz = up[r] - v[r];
        const float pw = lane_below(f.e[r] * dx);
        float d = cf.c0 * __builtin_fmaf(f.e[r], dx, -pw);
        d = __builtin_fmaf(cf.c1, __builtin_fmaf(f.n[r + 1], dy[r], -py[r]), d);
        d = __builtin_fmaf(cf.c2, __builtin_fmaf(f.u[r], dz, -pz[r]), d);
        pz[r] = f.u[r] * dz;
        if constexpr (MODE == 2) {
            const float y = d + cin[r];
            const float t = v[r] + y;
            cout[r] = y - (t - v[r]);
            out[r] = t;
        } else {
            cout[r] = 0.0f;
            out[r] = v[r] + d;
        }
    }
}

template <int MODE, int TY, int K, int D, bool MO>
__global__ __launch_bounds__(64 * TY) void heatvar_pairs_kernel(Geo g, const float* __restrict__ u,
                                                                 const float* __restrict__ cin,
                                                                 const float* __restrict__ kap, float* __restrict__ uout,
                                                                 float* __restrict__ cout, float* __restrict__ u1o,
                                                                 float* __restrict__ u2o, float* __restrict__ u3o, VarCoef cf,
                                                                 int zc, int tiles_x, int tiles_y, int x0)
{
    static_assert(K == 3 || K == 4, "three or four steps");
    static_assert(D == 2 || D == 4, "the prefetch slots repeat within the unrolled planes");
    constexpr int NY = 2 * TY, OX = 64 - 2 * K, OY = NY - 2 * (K - 1), U = 4;
    constexpr bool KH = (MODE == 2);
    // level-0 and kappa planes with the y ring; row NY + 2 takes the writes of
    // the waves off the ring (never read)
    __shared__ float s0[2][NY + 3][64];
    __shared__ float sk[2][NY + 3][64];
    __shared__ float sl[K - 1][2][NY][64];  // levels 1..K-1
    const int tx = threadIdx.x;
    const int ty = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    const int lb = xcd_remap(blockIdx.x, gridDim.x);
    const int per_plane = tiles_x * tiles_y;
    const int tz = lb / per_plane;
    const int rr = lb - tz * per_plane;
    const int tyi = rr / tiles_x;
    const int txi = rr - tyi * tiles_x;
    // the first tile needs no columns before it and the last none after it: the
    // border nodes there take no neighbour values
    const int i = txi * OX - x0 + tx, j0 = tyi * OY - (K - 1) + 2 * ty;
    const int ic = min(max(i, 0), g.nx - 1);
    const bool inner_x = i >= g.nl0 && i <= g.nx - 1 - g.nl0;
    const bool col_out = (tx >= K || (txi == 0 && i >= 0)) && (tx <= 63 - K || txi == tiles_x - 1) && i < g.nx;
    const int k0 = tz * zc, k1 = min(k0 + zc, g.nz);
    const int kfirst = k0 - (K - 1);  // first plane with a level-1 value
    const int klast = k1 + K - 2;     // last iteration
    const int klo = g.nl2, khi = g.nz - 1 - g.nl2;
    constexpr uint32_t B = sizeof(float);
    const size_t pb = (size_t)g.e01 * B;
    const uint32_t range = (uint32_t)((g.base + g.e01) * B);
    uint32_t oc[2], oo[2];
    bool inner_xy[2];
    bool any_out = false;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int j = j0 + r, row = 2 * ty + r;
        const int jc = min(max(j, 0), g.ny - 1);
        oc[r] = (uint32_t)(g.base + ic + g.e0 * jc) * B;
        const bool row_out = row >= K - 1 && row <= NY - K && j < g.ny;
        any_out |= row_out;
        oo[r] = (row_out && col_out) ? oc[r] : range;
        inner_xy[r] = inner_x && j >= g.nl1 && j <= g.ny - 1 - g.nl1;
    }
    // the row below the tile is the first wave's, the row above it the last one's
    const bool hy = ty == 0 || ty == TY - 1;
    const int hyj = min(max(ty == 0 ? j0 - 1 : j0 + 2, 0), g.ny - 1);
    const uint32_t oh = hy ? (uint32_t)(g.base + ic + g.e0 * hyj) * B : range;
    const int sh = ty == 0 ? 0 : ty == TY - 1 ? NY + 1 : NY + 2;
    // level planes: clamped rows only feed values that are never stored
    const int rs = max(2 * ty - 1, 0), rn = min(2 * ty + 2, NY - 1);
    const char* ub = (const char*)u;
    const char* kb8 = (const char*)kap;
    const char* cb = (const char*)cin;
    auto plane = [&](int kk) { return (size_t)min(max(kk, 0), g.nz - 1) * pb; };

    float qa[D][2], qb[D][2], qc[D][2], qah[D], qbh[D];
#pragma unroll
    for (int s = 0; s < D; ++s) {
        qah[s] = qbh[s] = 0.0f;
        qa[s][0] = qa[s][1] = qb[s][0] = qb[s][1] = qc[s][0] = qc[s][1] = 0.0f;
    }
    // the same loads every plane; an unneeded one reads past the range
    auto fetch = [&](const int slot, const int kk) {
        const size_t o = plane(kk);
        const Rsrc ru = plane_rsrc(ub + o, range), rk = plane_rsrc(kb8 + o, range);
        const bool cen = kk <= klast + 1, mid = kk <= klast;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            qa[slot][r] = bload<float>(ru, cen ? oc[r] : range);
            qb[slot][r] = bload<float>(rk, cen ? oc[r] : range);
            if constexpr (KH) qc[slot][r] = bload<float>(plane_rsrc(cb + o, range), mid ? oc[r] : range);
        }
        qah[slot] = bload<float>(ru, mid ? oh : range);
        qbh[slot] = bload<float>(rk, mid ? oh : range);
    };
    float pz[K][2];  // product of the lower z face of each level's plane
    {
        const size_t o = plane(kfirst - 1);
        float am[2], bm[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            am[r] = bload<float>(plane_rsrc(ub + o, range), oc[r]);
            bm[r] = bload<float>(plane_rsrc(kb8 + o, range), oc[r]);
        }
#pragma unroll
        for (int s = 0; s < D; ++s) fetch(s, kfirst + s);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            pz[0][r] = face<float, MODE>(qb[0][r], bm[r]) * (qa[0][r] - am[r]);
#pragma unroll
            for (int l = 1; l < K; ++l) pz[l][r] = 0.0f;
        }
    }
    PairFaces fq[U] = {};           // faces of the last planes, a ring
    float lv[K][2] = {}, lc[K][2] = {};  // level l at its last plane, and its compensation
    const float bv = (float)cf.border_value;
    const bool keep = cf.border_mode != SCAFES_BORDER_VALUE;
    for (int kb = kfirst; kb <= klast; kb += U) {
#pragma unroll
        for (int uu = 0; uu < U; ++uu) {
            const int s = uu % D;
            const int k = kb + uu;
            if (k > klast) return;  // uniform over the workgroup
            const int buf = uu & 1, pbf = buf ^ 1;
            float ac[2], bc[2], c0[2], ap[2], bp[2];
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                ac[r] = qa[s][r];
                bc[r] = qb[s][r];
                c0[r] = qc[s][r];
                ap[r] = qa[(s + 1) % D][r];
                bp[r] = qb[(s + 1) % D][r];
                s0[buf][2 * ty + r + 1][tx] = ac[r];
                sk[buf][2 * ty + r + 1][tx] = bc[r];
            }
            s0[buf][sh][tx] = qah[s];
            sk[buf][sh][tx] = qbh[s];
            fetch(s, k + D);
            __syncthreads();
            PairFaces& f = fq[uu];
            f.n[0] = face<float, MODE>(bc[0], sk[buf][2 * ty][tx]);
            f.n[1] = face<float, MODE>(bc[1], bc[0]);
            f.n[2] = face<float, MODE>(sk[buf][2 * ty + 3][tx], bc[1]);
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                f.e[r] = face<float, MODE>(lane_above(bc[r]), bc[r]);
                f.u[r] = face<float, MODE>(bp[r], bc[r]);
            }
            // level l at plane k - l + 1 from level l - 1 there (one plane
            // old, its in-plane neighbours in LDS) and one plane above (new)
            float v[2] = {ac[0], ac[1]}, vc[2] = {c0[0], c0[1]}, up[2] = {ap[0], ap[1]};
#pragma unroll
            for (int l = 1; l <= K; ++l) {
                const int kl = k - l + 1;
                const bool inner_z = kl >= klo && kl <= khi;
                float o[2] = {0.0f, 0.0f}, oc2[2] = {0.0f, 0.0f};
                if (l < K || (any_out && kl >= k0 - 1)) {
                    const float ys = l == 1 ? s0[buf][2 * ty][tx] : sl[l >= 2 ? l - 2 : 0][pbf][rs][tx];
                    const float yn = l == 1 ? s0[buf][2 * ty + 3][tx] : sl[l >= 2 ? l - 2 : 0][pbf][rn][tx];
                    pair_update<MODE>(cf, v, ys, yn, up, fq[(uu + U - (l - 1)) % U], pz[l - 1], vc, o, oc2);
#pragma unroll
                    for (int r = 0; r < 2; ++r) {
                        if (!(inner_xy[r] & inner_z)) {
                            o[r] = keep ? v[r] : bv;
                            oc2[r] = keep ? vc[r] : 0.0f;
                        }
                    }
                }
                const size_t po = plane(kl);
                const bool in_z = kl >= k0 && kl < k1;
                if (l == K) {
#pragma unroll
                    for (int r = 0; r < 2; ++r) {
                        bstore<float>(o[r], plane_rsrc((const char*)uout + po, range), in_z ? oo[r] : range);
                        if constexpr (KH)
                            bstore<float>(oc2[r], plane_rsrc((const char*)cout + po, range), in_z ? oo[r] : range);
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < 2; ++r) {
                        sl[l - 1][buf][2 * ty + r][tx] = o[r];
                        if constexpr (MO) {
                            float* const uo = l == 1 ? u1o : l == 2 ? u2o : u3o;
                            bstore<float>(o[r], plane_rsrc((const char*)uo + po, range), in_z ? oo[r] : range);
                        }
                        // the next level's centre is this level's last plane, its upper neighbour the new one
                        v[r] = lv[l][r];
                        vc[r] = lc[l][r];
                        up[r] = o[r];
                        lv[l][r] = o[r];
                        lc[l][r] = oc2[r];
                    }
                }
            }
        }
    }
}

}  // namespace scafes

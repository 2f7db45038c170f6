// Residual and restriction of a small plane level in one launch:
// r_c = (1/8) P^T (r - A x), x_c = 0 (region::residual and
// region::restriction, region.cc:1009-1055, :1767-1812).
//
// On a small level the two launches are latency, and the residual between
// them is written and read for nothing.  A workgroup owns 4 x 4 coarse points
// of one coarse plane: the x window of its fine residuals (11 x 11 points of
// five planes) is staged in LDS, two waves compute the 9 x 9 residuals of each
// of the three fine planes -- coefficients in scalar registers, as in the
// marching residual -- and 48 threads sum one component of one coarse point
// each, in restrict_point's order.  Residuals on the tiles' seams are computed
// twice (1.9 times the work).  A 32 x 32 x 33 FP64 V-cycle with two restricted
// levels goes from 150 to 137 us.
#pragma once

#include "mg_halo.hpp"

namespace stzmg {

constexpr int kRR = 4;               // coarse points of a tile per side
constexpr int kRRThreads = 6 * 64;   // two waves per fine plane

// Grid: (ceil(mc / 4), ceil(nc / 4), oc).  PLANE operator, x and y periodic,
// fine m and n even and at least 8.  pk: rows of march_stride(KEY) values per
// plane, the last nine the centre block.
template <typename T, int KEY>
__global__ __launch_bounds__(kRRThreads) void k_resid_restrict(Dims F, Dims C, const T *__restrict__ x,
                                                               const T *__restrict__ r, const T *__restrict__ pk,
                                                               T *__restrict__ rc, T *__restrict__ xc) {
    constexpr int RX = 2 * kRR + 1, NP = RX * RX;     // residuals of a plane
    constexpr int WX = RX + 2, CSZ = WX * WX, PSZ = 3 * CSZ;
    static_assert(NP <= 128, "two waves per plane");
    __shared__ T lds[5 * PSZ];
    __shared__ T res[3][3][NP];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int I0 = blockIdx.x * kRR, J0 = blockIdx.y * kRR, K = blockIdx.z;
    const long mn = (long)F.m * F.n;
    // plane f of the walk, wrapped where z is periodic; outside a wall: -1
    auto plane = [&](int f) { return f < 0 ? (F.pz ? f + F.o : -1) : (f >= F.o ? (F.pz ? f - F.o : -1) : f); };

    // the window: fine points from (2 I0 - 2, 2 J0 - 2), planes 2 K - 2 ..
    constexpr int NE = 5 * PSZ, NI = (NE + kRRThreads - 1) / kRRThreads;
    T w[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int e = tid + kRRThreads * i < NE ? tid + kRRThreads * i : NE - 1;
        const int sl = e / CSZ, rem = e - sl * CSZ, yy = rem / WX, xx = rem - yy * WX, p = sl / 3, c = sl - 3 * p;
        const int k = plane(2 * K - 2 + p);
        w[i] = k < 0 ? T(0)
                     : x[c * F.N + mn * k + wrap1(2 * I0 - 2 + xx, F.m) + (long)F.m * wrap1(2 * J0 - 2 + yy, F.n)];
    }
    // this thread's residual: point t of plane 2 K - 1 + ez
    const int ez = wv / 2, t0 = (wv & 1) * 64 + lane, t = t0 < NP ? t0 : 0;
    const int ty = t / RX, tx = t - ty * RX;
    const int k = plane(2 * K - 1 + ez), kc = k < 0 ? 0 : k;
    const T *A = pk + (long)kc * kMarchStride<KEY>;
    T rv[3];
    {
        const long q = mn * kc + wrap1(2 * I0 - 1 + tx, F.m) + (long)F.m * wrap1(2 * J0 - 1 + ty, F.n);
#pragma unroll
        for (int c = 0; c < 3; c++) rv[c] = r[c * F.N + q];
    }
#pragma unroll
    for (int i = 0; i < NI; i++)
        if (tid + kRRThreads * i < NE) lds[tid + kRRThreads * i] = w[i];
    __syncthreads();

    if (k >= 0) {  // (a wave lies in one plane)
        const int at = (ez + 1) * PSZ + (ty + 1) * WX + tx + 1;
        const HaloNb<T, WX, CSZ, PSZ> ld[1] = {
            {lds, at - PSZ - WX - 1, at - PSZ - WX, at - PSZ - WX + 1}};
        T a[1][3] = {{0, 0, 0}};
        halo_acc<T, KEY, 0, 0, 1>(A, ld, a);
        halo_acc<T, KEY, 1, 0, 1>(A, ld, a);
        constexpr int off = halo_off(KEY, 27);
        const T *D = halo_row(A) + off;
        const T v0 = lds[at], v1 = lds[at + CSZ], v2 = lds[at + 2 * CSZ];
        a[0][0] += D[0] * v0 + D[1] * v1 + D[2] * v2;
        a[0][1] += D[3] * v0 + D[4] * v1 + D[5] * v2;
        a[0][2] += D[6] * v0 + D[7] * v1 + D[8] * v2;
        if (t0 < NP)
#pragma unroll
            for (int c = 0; c < 3; c++) res[ez][c][t] = rv[c] - a[0][c];
    }
    __syncthreads();

    if (tid < 3 * kRR * kRR) {
        const int c = tid / (kRR * kRR), q = tid % (kRR * kRR), qy = q / kRR, qx = q % kRR;
        const int I = I0 + qx, J = J0 + qy;
        if (I < C.m && J < C.n) {
            T s = 0;
#pragma unroll
            for (int ek = 0; ek < 3; ek++) {
                if (plane(2 * K - 1 + ek) < 0) continue;
                const T wk = ek == 1 ? T(1) : T(0.5);
#pragma unroll
                for (int ej = 0; ej < 3; ej++) {
                    const T wj = ej == 1 ? wk : T(0.5) * wk;
#pragma unroll
                    for (int ei = 0; ei < 3; ei++) {
                        const T wi = T(0.125) * (ei == 1 ? wj : T(0.5) * wj);
                        s += wi * res[ek][c][(2 * qy + ej) * RX + 2 * qx + ei];
                    }
                }
            }
            const long p = I + (long)C.m * (J + (long)C.n * K);
            rc[p + c * C.N] = s;
            xc[p + c * C.N] = 0;
        }
    }
}

}  // namespace stzmg

// Colour pass of block Gauss-Seidel for per-point operators, 16 lanes per
// point.
//
// A point's operator row is 1,944 bytes (FP64) of its own, and a colour pass
// reads each row once: the pass is bound by that stream.  With one thread per
// point a wave's loads touch 64 rows at a time, each line many times over, and
// a level of some ten thousand points gives 28 workgroups for 256 CUs
// (44 x 40 x 33: 16.8 us a pass, 0.8 TB/s of operator).  Here 16 lanes share a
// point, two blocks each: neighbouring lanes read neighbouring blocks, a wave
// four whole rows, and the pass has 16 times the threads.  The 16 partial
// sums are added with DPP row permutes and lanes 0 to 2 write one component
// each.
#pragma once

#include "mg_coarse.hpp"

namespace stzmg {

constexpr int kPointLanes = kBottomLanes;

// Grid: (ceil(16 cntx cnty / kThreads), cntz).
template <typename T>
__global__ __launch_bounds__(kThreads) void k_gs_points(Dims d, T *__restrict__ x, const T *__restrict__ r,
                                                        const T *__restrict__ ops, const T *__restrict__ inv, int cx,
                                                        int cy, int cz, int cntx, int cnty) {
    const int k = col_coord(blockIdx.y, cz, d.o);
    const long t = ((long)blockIdx.x * kThreads + threadIdx.x) / kPointLanes;
    const int sl = threadIdx.x % kPointLanes;
    const bool live = t < (long)cntx * cnty;
    // a row of lanes without a point repeats the last one and stores nothing
    const int tt = live ? (int)t : cntx * cnty - 1;
    const int jj = tt / cntx, ii = tt - jj * cntx;
    const int i = col_coord(ii, cx, d.m), j = col_coord(jj, cy, d.n);
    const long p = i + (long)d.m * (j + (long)d.n * k);
    const T *A = ops + p * kBlk;
    // lanes 0 to 2: right-hand side and the inverse row of their component,
    // in flight with the operator
    const int c = sl < 3 ? sl : 0;
    const T *B = inv + p * 9 + 3 * c;
    const T r0 = r[p], r1 = r[p + d.N], r2 = r[p + 2 * d.N], b0 = B[0], b1 = B[1], b2 = B[2];
    T a0 = 0, a1 = 0, a2 = 0;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int b = sl + kPointLanes * h;
        if (b >= 27 || b == 13) continue;
        const int ni = nb(i, b % 3 - 1, d.m, d.px), nj = nb(j, (b / 3) % 3 - 1, d.n, d.py),
                  nk = nb(k, b / 9 - 1, d.o, d.pz);
        if (ni < 0 || nj < 0 || nk < 0) continue;
        const long q = ni + (long)d.m * (nj + (long)d.n * nk);
        mv(A + 9 * b, x[q], x[q + d.N], x[q + 2 * d.N], a0, a1, a2);
    }
    const T e0 = r0 - row16_sum(a0), e1 = r1 - row16_sum(a1), e2 = r2 - row16_sum(a2);
    if (live && sl < 3) x[p + c * d.N] = b0 * e0 + b1 * e1 + b2 * e2;
}

}  // namespace stzmg

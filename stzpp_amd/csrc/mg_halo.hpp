// One launch per sweep for small plane levels: a whole 8-colour block
// Gauss-Seidel sweep with a recomputed halo.
//
// What bounds a small level is not memory or arithmetic but the chain of
// dependent launches: a launch of the marching sweep (mg_march.hpp) on a few
// thousand points is a fixed chain -- dispatch, staging round trip,
// coefficients, four barrier-separated sub-passes, store -- and a sweep takes
// two of them, or eight colour launches where no tile divides the plane.
// Here a workgroup owns TX x TY points of two planes, k0 (even, swept first)
// and k0 + 1, and computes everything its points depend on itself: the even
// planes k0 and k0 + 2 over a halo of 7, 6, 5, 4 points (the four in-plane
// colours), then the odd plane k0 + 1 over 3, 2, 1, 0, from a window of the
// five planes k0 - 1 .. k0 + 3 with a halo of 8 staged in LDS.  The points
// computed twice come from the same old values in the same order, so tiles
// agree; the sweep reads x and writes a second buffer.  The arithmetic grows
// 6.7-fold at 8 x 8 (3.6-fold at 16 x 16), which a level that leaves the
// chip idle does not notice.
//
// Within a plane the part of the stencil sum that no sub-pass changes -- the
// planes above and below, and the in-plane neighbours of colours swept later
// -- is taken before the sub-passes, so the serial chain of the four
// sub-passes holds 0, 2, 6 and 8 in-plane blocks instead of 8 each.
//
// Coefficients come from the marching sweep's packed per-plane table through
// the scalar cache.  A launch this short meets that cache cold, and every
// group of coefficients would wait for memory in turn: the three planes'
// tables are touched, one word per line, while the window is in flight.
//
// Any even m, n >= 8 (a tile that sticks out of the plane computes wrapped
// points and stores none of them), z periodic (even) or walled.
//
// Measured per sweep (MI355X, back to back on one stream; two marching
// launches before, or eight colour launches where no tile divides the
// plane): dense walled Galerkin level 16 x 16 x 17 FP64 18.1 -> 10.5 us,
// FP32 14.4 -> 9.5; 32 x 32 x 33 FP64 18.2 -> 12.0, FP32 14.8 -> 10.1;
// shear operator 32 x 32 x 33 FP64 12.9 -> 9.4, FP32 10.3 -> 7.5;
// 24 x 20 x 13 (colour launches) FP64 51 -> 11.0, FP32 50 -> 9.6.
#pragma once

#include "mg_march.hpp"

namespace stzmg {

// Block lists of a point of in-plane colour s = cx + 2 cy: kind 0 the blocks
// of the planes above and below, kind 1 + s the in-plane neighbours of a
// colour swept later (old values), kind 5 + s those swept before (new
// values); kinds 9 and 10 are two halves of kind 0.  Centrosymmetric keys list one block of each opposite pair (both
// neighbours have the same colour).
__host__ __device__ constexpr bool halo_in(int kind, int b) {
    const int di = b % 3 - 1, dj = (b / 3) % 3 - 1, dk = b / 9 - 1;
    if (kind == 0) return dk != 0;
    if (kind >= 9) return dk != 0 && ((b % 18 < 5) == (kind == 9));
    if (dk != 0 || (di == 0 && dj == 0)) return false;
    const int s = kind < 5 ? kind - 1 : kind - 5;
    const int c = s ^ ((di != 0) + 2 * (dj != 0));
    return kind < 5 ? c > s : c < s;
}
__host__ __device__ constexpr int halo_len(int key, int kind) {
    int n = 0;
    for (int b = 0; b < (march_sym(key) ? 13 : 27); b++) n += halo_in(kind, b);
    return n;
}
__host__ __device__ constexpr int halo_block(int key, int kind, int i) {
    for (int b = 0; b < (march_sym(key) ? 13 : 27); b++)
        if (halo_in(kind, b) && i-- == 0) return b;
    return 27;
}
// Offset of block b (27: the inverse centre block) in the packed row.
__host__ __device__ constexpr int halo_off(int key, int b) {
    int n = 0;
    for (int ph = 0; ph < 2; ph++)
        for (int q = 0; q < march_len(key, ph); q++) {
            if (march_block(key, ph, q) == b) return n;
            n += popc9(march_mask(key, march_block(key, ph, q)));
        }
    return n;
}
// Groups of at most G coefficients, as in march_group.
__host__ __device__ constexpr int halo_group(int key, int kind, int G, int i) {
    int g = 0, run = 0;
    for (int q = 0; q <= i; q++) {
        const int nz = popc9(march_mask(key, halo_block(key, kind, q)));
        if (run > 0 && run + nz > G) {
            g++;
            run = 0;
        }
        run += nz;
    }
    return g;
}
__host__ __device__ constexpr int halo_ngroups(int key, int kind, int G) {
    return halo_len(key, kind) ? halo_group(key, kind, G, halo_len(key, kind) - 1) + 1 : 0;
}
__host__ __device__ constexpr int halo_pos(int key, int kind, int G, int i) {
    const int g = halo_group(key, kind, G, i);
    int n = 0;
    for (int q = 0; q < i; q++)
        if (halo_group(key, kind, G, q) == g) n += popc9(march_mask(key, halo_block(key, kind, q)));
    return n;
}
__host__ __device__ constexpr int halo_gsize(int key, int kind, int G, int g) {
    int n = 0;
    for (int q = 0; q < halo_len(key, kind); q++)
        if (halo_group(key, kind, G, q) == g) n += popc9(march_mask(key, halo_block(key, kind, q)));
    return n;
}

// The same table row behind an offset the compiler cannot see is zero: loads
// of one phase are not merged with those of another and then held in
// registers (and spilled) across the phases between.
template <typename T>
__device__ __forceinline__ const T *halo_row(const T *A) {
    int z = 0;
    asm volatile("" : "+s"(z));
    return A + z;
}

// Group GR of list KIND in scalar registers.
template <typename T, int KEY, int KIND, int GR>
struct HaloGroup {
    static constexpr int G = MarchGroup<T>::G;
    static constexpr int N = halo_gsize(KEY, KIND, G, GR);
    T c[N > 0 ? N : 1];
    __device__ __forceinline__ void load(const T *A0) {
        if constexpr (N > 0) {
            const T *A = halo_row(A0);
            static_for<halo_len(KEY, KIND)>([&](auto i_) {
                constexpr int I = decltype(i_)::value;
                if constexpr (halo_group(KEY, KIND, G, I) == GR) {
                    constexpr int b = halo_block(KEY, KIND, I), q0 = halo_pos(KEY, KIND, G, I);
                    constexpr int off = halo_off(KEY, b);
                    static_for<popc9(march_mask(KEY, b))>([&](auto e) {
                        c[q0 + decltype(e)::value] = A[off + decltype(e)::value];
                    });
                }
            });
#pragma unroll
            for (int q = 0; q < N; q++) asm volatile("" : "+s"(c[q]));
        }
    }
    // a += its blocks times the neighbours of one point
    template <typename LD>
    __device__ __forceinline__ void add(const LD &ld, T (&a)[3]) const {
        if constexpr (N > 0) {
            static_for<halo_len(KEY, KIND)>([&](auto i_) {
                constexpr int I = decltype(i_)::value;
                if constexpr (halo_group(KEY, KIND, G, I) == GR) {
                    constexpr int b = halo_block(KEY, KIND, I), q = halo_pos(KEY, KIND, G, I);
                    constexpr unsigned m = march_mask(KEY, b), cols = pat_cols(m);
                    constexpr int di = b % 3 - 1, dj = (b / 3) % 3 - 1, dk = b / 9 - 1;
                    T v0 = 0, v1 = 0, v2 = 0;
                    if constexpr (march_sym(KEY)) {
                        if constexpr (cols & 1) v0 = ld(0, di, dj, dk) + ld(0, -di, -dj, -dk);
                        if constexpr (cols & 2) v1 = ld(1, di, dj, dk) + ld(1, -di, -dj, -dk);
                        if constexpr (cols & 4) v2 = ld(2, di, dj, dk) + ld(2, -di, -dj, -dk);
                    } else {
                        if constexpr (cols & 1) v0 = ld(0, di, dj, dk);
                        if constexpr (cols & 2) v1 = ld(1, di, dj, dk);
                        if constexpr (cols & 4) v2 = ld(2, di, dj, dk);
                    }
                    if constexpr (m & 0x001) a[0] += c[q + rank9(m, 0)] * v0;
                    if constexpr (m & 0x002) a[0] += c[q + rank9(m, 1)] * v1;
                    if constexpr (m & 0x004) a[0] += c[q + rank9(m, 2)] * v2;
                    if constexpr (m & 0x008) a[1] += c[q + rank9(m, 3)] * v0;
                    if constexpr (m & 0x010) a[1] += c[q + rank9(m, 4)] * v1;
                    if constexpr (m & 0x020) a[1] += c[q + rank9(m, 5)] * v2;
                    if constexpr (m & 0x040) a[2] += c[q + rank9(m, 6)] * v0;
                    if constexpr (m & 0x080) a[2] += c[q + rank9(m, 7)] * v1;
                    if constexpr (m & 0x100) a[2] += c[q + rank9(m, 8)] * v2;
                }
            });
            // complete before the next group is loaded (all groups at once
            // would not fit the scalar registers)
            asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]));
        }
    }
};

// a[p] += sum over the blocks of list KIND, from group FIRST on, of block
// times neighbour for NP points.  ld[p](c, di, dj, dk): component c of a
// neighbour of point p.
template <typename T, int KEY, int KIND, int FIRST, int NP, typename LD>
__device__ __forceinline__ void halo_acc(const T *A, const LD (&ld)[NP], T (&a)[NP][3]) {
    constexpr int NG = halo_ngroups(KEY, KIND, MarchGroup<T>::G);
    if constexpr (NG > FIRST)
        static_for<NG - FIRST>([&](auto g_) {
            HaloGroup<T, KEY, KIND, FIRST + decltype(g_)::value> g;
            g.load(A);
#pragma unroll
            for (int p = 0; p < NP; p++) g.add(ld[p], a[p]);
        });
}

// The update of one point of colour S in its plane: the blocks of the
// colours swept before, then the inverse centre block.  prepare() runs
// before the barrier that the update waits for, so the first group and the
// inverse are in registers when the neighbours' new values are.
template <typename T, int KEY, int S>
struct HaloUpdate {
    HaloGroup<T, KEY, 5 + S, 0> g0;
    T v[9];
    __device__ __forceinline__ void prepare(const T *A) {
        constexpr int off = halo_off(KEY, 27);
        const T *I = halo_row(A) + off;
#pragma unroll
        for (int e = 0; e < 9; e++) v[e] = I[e];
#pragma unroll
        for (int e = 0; e < 9; e++) asm volatile("" : "+s"(v[e]));
        g0.load(A);
    }
    template <typename LD>
    __device__ __forceinline__ void run(const T *A, const LD &ld, const T (&r)[3], T (&a)[3], T *out, int cs,
                                        bool own) {
        g0.add(ld, a);
        const LD l[1] = {ld};
        T b[1][3] = {{a[0], a[1], a[2]}};
        halo_acc<T, KEY, 5 + S, 1, 1>(A, l, b);
        const T e0 = r[0] - b[0][0], e1 = r[1] - b[0][1], e2 = r[2] - b[0][2];
        if (own) {
            out[0] = v[0] * e0 + v[1] * e1 + v[2] * e2;
            out[cs] = v[3] * e0 + v[4] * e1 + v[5] * e2;
            out[2 * cs] = v[6] * e0 + v[7] * e1 + v[8] * e2;
        }
    }
};

// Component c of a neighbour of one point, in the staged window: bases of
// the point's own column and of the columns left and right of it, one plane
// and one row below it, so that every neighbour lies at a compile-time
// distance >= 0.
template <typename T, int WX, int CSZ, int PSZ>
struct HaloNb {
    const T *lds;
    int bl, bc, br;
    static constexpr int low = PSZ + WX;
    __device__ __forceinline__ T operator()(int c, int di, int dj, int dk) const {
        const int b = di < 0 ? bl : (di > 0 ? br : bc);
        return lds[b + (low + dk * PSZ + c * CSZ + dj * WX)];
    }
};

// Points of in-plane colour s computed over a halo of H0 + 3 - s points
// around a TX x TY tile.
template <int TX, int TY, int H0>
struct HaloPass {
    static constexpr int h(int s) { return H0 + 3 - s; }
    static constexpr int xf(int s) { return -h(s) + (((s & 1) + h(s)) & 1); }
    static constexpr int yf(int s) { return -h(s) + (((s >> 1) + h(s)) & 1); }
    static constexpr int nx(int s) { return (TX + h(s) - 1 - xf(s)) / 2 + 1; }
    static constexpr int ny(int s) { return (TY + h(s) - 1 - yf(s)) / 2 + 1; }
    static constexpr int npts(int s) { return nx(s) * ny(s); }
};

// Threads: the even planes k0 and k0 + 2 take half the workgroup each; half
// of those threads own one point of colour 0 and one of colour 2, the others
// one of 1 and one of 3.
template <int TX, int TY>
constexpr int halo_threads() {
    return 4 * ((HaloPass<TX, TY, 4>::npts(0) + 63) / 64 * 64);
}

// Grid: (ceil(m / TX), ceil(n / TY), ceil(o / 2)).  PLANE operator, x and y
// periodic, m and n even and at least 8, o at least 4, any number (walls) or
// even (periodic).  Blocks that point across a wall add nothing.  pk: rows of march_stride(KEY) values per plane.  zero: x is
// zero whatever the buffer holds.  xc (may be null): the sweep starts from
// x + P xc, the coarse level's correction (dimensions C) added as the window
// arrives, in interp_point's order -- the correction costs no pass over x and
// no launch (5.3 us) of its own.
template <typename T, int KEY, int TX, int TY>
__global__ __launch_bounds__((halo_threads<TX, TY>())) __attribute__((amdgpu_waves_per_eu(4))) void k_gs_halo(Dims d, const T *__restrict__ x,
                                                                     T *__restrict__ xd, const T *__restrict__ r,
                                                                     const T *__restrict__ pk, int zero, Dims C,
                                                                     const T *__restrict__ xc) {
    constexpr int NT = halo_threads<TX, TY>(), NW = NT / 64;
    constexpr int H = 8;
    constexpr int WP = (TX + 2 * H) / 2;   // column pairs of the window
    constexpr int WY = TY + 2 * H;
    // row length in LDS: the even columns, then the odd ones; an odd length
    // spreads the rows of a colour (every second one) over the banks
    constexpr int WX = 2 * WP + 3;
    constexpr int CSZ = WX * WY, PSZ = 3 * CSZ;
    using P0 = HaloPass<TX, TY, 4>;
    using P1 = HaloPass<TX, TY, 0>;
    constexpr int LQ = (P1::npts(0) + 63) / 64;  // waves per colour of the odd plane
    static_assert(TX % 2 == 0 && TY % 2 == 0 && 8 * LQ <= NW, "tile shape");
    struct alignas(2 * sizeof(T)) Pair {
        T v[2];
    };
    __shared__ T lds[5 * PSZ];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int x0 = blockIdx.x * TX, y0 = blockIdx.y * TY, k0 = 2 * blockIdx.z;
    const long mn = (long)d.m * d.n;
    const bool odd = k0 + 1 < d.o;  // the plane k0 + 1 exists
    // window coordinate into [0, n): from -8 to n + 14, n >= 8
    auto wrap = [](int i, int n) { return i < 0 ? i + n : (i >= 2 * n ? i - 2 * n : (i >= n ? i - n : i)); };
    auto plane = [&](int k) { return k < 0 ? k + d.o : (k >= d.o ? k - d.o : k); };

    // ---- the window in flight ----
    constexpr int NE = WP * WY, NI = (NE + 63) / 64;  // column pairs of one component of one plane
    constexpr int NS = (15 + NW - 1) / NW;            // (plane, component) slabs per wave
    Pair w[NS][NI];
    unsigned go[NI];
    int lo[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int e = lane + 64 * i < NE ? lane + 64 * i : NE - 1;
        const int yy = e / WP, pc = e - yy * WP;
        go[i] = (unsigned)(sizeof(T) * (wrap(x0 - H + 2 * pc, d.m) + (long)d.m * wrap(y0 - H + yy, d.n)));
        lo[i] = yy * WX + pc;
    }
    static_for<NS>([&](auto j_) {
        constexpr int j = decltype(j_)::value;
        const int sl = wv + NW * j, p = sl / 3, c = sl - 3 * p, k = k0 - 1 + p;
        if (sl < 15 && !zero && (d.pz || (k >= 0 && k < d.o))) {
            const T *base = x + mn * plane(k) + c * d.N;
#pragma unroll
            for (int i = 0; i < NI; i++) w[j][i] = at_bytes(reinterpret_cast<const Pair *>(base), go[i]);
        } else {
#pragma unroll
            for (int i = 0; i < NI; i++) w[j][i] = Pair{{T(0), T(0)}};
        }
    });

    // ---- the coarse level's correction ----
    if (xc) {
        // coarse rows and columns of every column pair (x even): its even
        // point sits on column I, its odd point between I and I + 1
        int q00[NI], q01[NI], q10[NI], q11[NI];
        bool oy[NI];
        const int cmn = C.m * C.n;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int e = lane + 64 * i < NE ? lane + 64 * i : NE - 1;
            const int yy = e / WP, pc = e - yy * WP;
            const int I = wrap(x0 - H + 2 * pc, d.m) >> 1, fj = wrap(y0 - H + yy, d.n), J = fj >> 1;
            const int I1 = I + 1 < C.m ? I + 1 : 0, J1 = J + 1 < C.n ? J + 1 : 0;
            oy[i] = (fj & 1) != 0;
            q00[i] = I + C.m * J;
            q01[i] = I1 + C.m * J;
            q10[i] = I + C.m * J1;
            q11[i] = I1 + C.m * J1;
        }
        static_for<NS>([&](auto j_) {
            constexpr int j = decltype(j_)::value;
            const int sl = wv + NW * j, p = sl / 3, c = sl - 3 * p, k = k0 - 1 + p;
            if (sl < 15 && (d.pz || (k >= 0 && k < d.o))) {
                const int kw = plane(k), K = kw >> 1, nk = (kw & 1) + 1;
                const int K1 = K + 1 < C.o ? K + 1 : 0;
                const T wk = nk == 2 ? T(0.5) : T(1);
                T ev[NI], od[NI];
#pragma unroll
                for (int i = 0; i < NI; i++) ev[i] = od[i] = 0;
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    if (h >= nk) continue;
                    const T *b = xc + c * C.N + (long)cmn * (h ? K1 : K);
#pragma unroll
                    for (int i = 0; i < NI; i++) {
                        const T w0 = oy[i] ? T(0.5) * wk : wk, w1 = T(0.5) * w0;
                        const T a = b[q00[i]], e1 = b[q01[i]], f = b[q10[i]], g = b[q11[i]];
                        ev[i] += w0 * a;
                        od[i] += w1 * a;
                        od[i] += w1 * e1;
                        if (oy[i]) {
                            ev[i] += w0 * f;
                            od[i] += w1 * f;
                            od[i] += w1 * g;
                        }
                    }
                }
#pragma unroll
                for (int i = 0; i < NI; i++) {
                    w[j][i].v[0] += ev[i];
                    w[j][i].v[1] += od[i];
                }
            }
        });
    }

    // ---- this thread's points ----
    // even planes: plane k0 (first half of the workgroup) or k0 + 2, point
    // (tx, ty) of colour hf and of colour hf + 2
    const int pl = wv >= NW / 2 ? 1 : 0;                 // 0: plane k0, 1: plane k0 + 2
    const int hf = (wv / (NW / 4)) & 1;
    const int t0 = tid % (NT / 4);
    const int kA = plane(k0 + 2 * pl);
    // plane k0 + 2 serves plane k0 + 1 only; above a wall there is none (its
    // slot of the window stays zero)
    const bool live = pl == 0 || (odd && (d.pz || k0 + 2 < d.o));
    int cen[2];      // window index of the point in its plane, component 0
    bool own[2];
    T rr[2][3];
    static_for<2>([&](auto q_) {
        constexpr int q = decltype(q_)::value;
        const int s = hf + 2 * q;
        const int nx = hf ? P0::nx(1 + 2 * q) : P0::nx(2 * q), np = hf ? P0::npts(1 + 2 * q) : P0::npts(2 * q);
        const int xf = hf ? P0::xf(1 + 2 * q) : P0::xf(2 * q), yf = hf ? P0::yf(1 + 2 * q) : P0::yf(2 * q);
        own[q] = live && t0 < np;
        const int t = t0 < np ? t0 : 0;
        const int ty = hf ? t / P0::nx(1 + 2 * q) : t / P0::nx(2 * q), tx = t - ty * nx;
        const int xx = xf + 2 * tx + H, yy = yf + 2 * ty + H;
        cen[q] = yy * WX + (s & 1) * WP + (xx >> 1);
        const unsigned o =
            (unsigned)(sizeof(T) * (wrap(x0 + xx - H, d.m) + (long)d.m * wrap(y0 + yy - H, d.n)));
        if (live) {
#pragma unroll
            for (int c = 0; c < 3; c++) rr[q][c] = at_bytes(r + mn * kA + c * d.N, o);
        }
    });
    // odd plane: one point of colour s1; two waves (one of each half of the
    // workgroup) share it
    const int wh = wv % (NW / 2), s1 = wh / LQ, t1 = (wh % LQ) * 64 + lane;
    const bool first = s1 < 4 && wv < NW / 2, second = s1 < 4 && wv >= NW / 2;
    int cen1 = (H + 1) * WX + H / 2;
    bool own1 = false;
    T r1[3] = {0, 0, 0};
    if (odd && s1 < 4) {
        static_for<4>([&](auto s_) {
            constexpr int S = decltype(s_)::value;
            if (s1 == S) {
                own1 = t1 < P1::npts(S);
                const int t = own1 ? t1 : 0;
                const int ty = t / P1::nx(S), tx = t - ty * P1::nx(S);
                const int xx = P1::xf(S) + 2 * tx + H, yy = P1::yf(S) + 2 * ty + H;
                cen1 = yy * WX + (S & 1) * WP + (xx >> 1);
                const unsigned o =
                    (unsigned)(sizeof(T) * (wrap(x0 + xx - H, d.m) + (long)d.m * wrap(y0 + yy - H, d.n)));
#pragma unroll
                for (int c = 0; c < 3; c++) r1[c] = at_bytes(r + mn * (k0 + 1) + c * d.N, o);
            }
        });
    }

    // ---- the coefficient tables into the scalar cache ----
    const T *A0 = pk + (long)kA * kMarchStride<KEY>;
    const T *A1 = pk + (long)(odd ? k0 + 1 : k0) * kMarchStride<KEY>;
    {
        // every wave touches its share of the lines of the three rows
        constexpr int step = 64 / (int)sizeof(T), lines = (march_stride(KEY) + step - 1) / step;
        const int kB = plane(k0 + (odd ? 2 : 0));
        const T *R[3] = {halo_row(pk + (long)k0 * kMarchStride<KEY>), halo_row(pk + (long)kB * kMarchStride<KEY>),
                         halo_row(A1)};
        T touch = 0;
#pragma unroll
        for (int i = 0; i < (lines + NW - 1) / NW; i++) {
            const int q = wv + NW * i < lines ? wv + NW * i : lines - 1;
#pragma unroll
            for (int e = 0; e < 3; e++) touch += R[e][q * step];
        }
        asm volatile("" ::"v"(touch));
    }

    static_for<NS>([&](auto j_) {
        constexpr int j = decltype(j_)::value;
        const int sl = wv + NW * j;
        if (sl < 15) {
            T *dst = lds + (sl / 3) * PSZ + (sl % 3) * CSZ;
#pragma unroll
            for (int i = 0; i < NI; i++)
                if (NE % 64 == 0 || lane + 64 * i < NE) {
                    dst[lo[i]] = w[j][i].v[0];
                    dst[lo[i] + WP] = w[j][i].v[1];
                }
        }
    });
    __syncthreads();

    // neighbours of the point at window index cen: in a parity-split row the
    // columns x + 1 and x - 1 of an even column are the odd columns of the
    // same index and of the one before, those of an odd column the even
    // columns of the next index and of the same
    using Nb = HaloNb<T, WX, CSZ, PSZ>;
    auto nbs = [&](int at, int parity) {
        const int b = at - Nb::low;
        return Nb{lds, b + (parity ? -WP : WP - 1), b, b + (parity ? 1 - WP : WP)};
    };

    // ---- even planes ----
    {
        T a[2][3] = {{0, 0, 0}, {0, 0, 0}};
        const int at[2] = {cen[0] + (1 + 2 * pl) * PSZ, cen[1] + (1 + 2 * pl) * PSZ};
        const Nb ld[2] = {nbs(at[0], hf), nbs(at[1], hf)};
        if (live && !zero) {
            halo_acc<T, KEY, 0, 0, 2>(A0, ld, a);
            static_for<4>([&](auto s_) {
                constexpr int S = decltype(s_)::value, q = S >> 1;
                if (hf == (S & 1)) {
                    const Nb l[1] = {ld[q]};
                    T b[1][3] = {{a[q][0], a[q][1], a[q][2]}};
                    halo_acc<T, KEY, 1 + S, 0, 1>(A0, l, b);
#pragma unroll
                    for (int c = 0; c < 3; c++) a[q][c] = b[0][c];
                }
            });
        }
        static_for<4>([&](auto s_) {
            constexpr int S = decltype(s_)::value, q = S >> 1;
            if (hf == (S & 1) && live) {
                HaloUpdate<T, KEY, S> u;
                u.prepare(A0);
                __syncthreads();
                u.run(A0, ld[q], rr[q], a[q], lds + at[q], CSZ, own[q]);
            } else {
                __syncthreads();
            }
        });
        __syncthreads();
    }
    // the tile's points of slot p (plane k) to xd, one column pair per thread
    auto put = [&](int p, int k, int t) {
        constexpr int HXT = TX / 2;
        if (t < 3 * HXT * TY) {
            const int c = t / (HXT * TY), e = t - c * (HXT * TY), yy = e / HXT, pc = e - yy * HXT;
            if (x0 + 2 * pc < d.m && y0 + yy < d.n) {
                const T *s = lds + p * PSZ + c * CSZ + (yy + H) * WX + pc + H / 2;
                const unsigned o = (unsigned)(sizeof(T) * ((x0 + 2 * pc) + (long)d.m * (y0 + yy)));
                at_bytes(reinterpret_cast<Pair *>(xd + mn * k + c * d.N), o) = Pair{{s[0], s[WP]}};
            }
        }
    };
    static_assert(3 * (TX / 2) * TY <= NT / 2, "one column pair per thread of half the workgroup");
    if (!odd) {  // the whole workgroup
        put(1, k0, tid);
        return;
    }

    // ---- odd plane: the waves of a colour take one half of the sum over the
    // planes above and below, the same waves of the workgroup's second half
    // the other, passed on through slot 0 (plane k0 - 1 is no longer read) ----
    {
        const int at = cen1 + 2 * PSZ;
        const Nb ld = nbs(at, s1 & 1);
        const Nb l[1] = {ld};
        T a[1][3] = {{0, 0, 0}};
        T *half = lds + (s1 * LQ * 64 + t1);
        constexpr int HS = 4 * LQ * 64;
        static_assert(3 * HS <= PSZ, "partial sums in slot 0");
        if (second) {
            halo_acc<T, KEY, 10, 0, 1>(A1, l, a);
            static_for<4>([&](auto s_) {
                constexpr int S = decltype(s_)::value;
                if (s1 == S && !zero) halo_acc<T, KEY, 1 + S, 0, 1>(A1, l, a);
            });
#pragma unroll
            for (int c = 0; c < 3; c++) half[c * HS] = a[0][c];
        } else if (first) {
            halo_acc<T, KEY, 9, 0, 1>(A1, l, a);
        }
        if (wv < NW / 2) put(1, k0, tid);
        __syncthreads();
        if (first)
#pragma unroll
            for (int c = 0; c < 3; c++) a[0][c] += half[c * HS];
        static_for<4>([&](auto s_) {
            constexpr int S = decltype(s_)::value;
            if (first && s1 == S) {
                HaloUpdate<T, KEY, S> u;
                u.prepare(A1);
                if constexpr (S > 0) __syncthreads();
                u.run(A1, ld, r1, a[0], lds + at, CSZ, own1);
            } else {
                if constexpr (S > 0) __syncthreads();
            }
        });
        __syncthreads();
        put(2, k0 + 1, tid);
    }
}

}  // namespace stzmg

// Direct (explicit dynamics) step of shear_sim_3d (include/stz.h,
// stz_step_direct): step_forward, src/shear_sim_3d.cpp:206-213, with
// calc_updates :89-104, step_stress :774-896, step_chi :1193-1215,
// step_velocity :919-994, step_ref :997-1030 and merge_updates :154-162.
//
// Per step, on the handle's stream:
//   k_direct_plastic  STZ plasticity of every cell: adapt, the plastic chi
//                     change and this step's ad_Dpl (adapt / 2 / mu / dt sbar)
//   k_direct_cell     stress and chi: elastic, Truesdell, ENO2 advection and
//                     plastic terms; chi advection and dt chi_diffusion / c0
//                     with the reference's in-place ad_Dpl order (this step's
//                     value at -x/-y/-z inside the domain, last step's at
//                     +x/+y/+z and at periodic images, zero across a wall)
//   k_direct_vertex   velocity (dt/rho div sigma + dt kappa/rho Lap u -
//                     u.grad u) and reference map (- u.grad xi) at the
//                     vertices 0 < k < Nz; the plane k = 0 is left as it is
//                     (the reference skips zz = 0 when its x coordinate in
//                     the rank grid is 0, :101, i.e. always with one rank)
//   k_direct_plate    top plate velocity and reference map at t + dt
//                     (set_boundary_conditions, :2393-2466; with one rank in
//                     z the bottom branch is never taken)
// Ghosts are computed where they are read: periodic images (the reference
// map shifted by the domain length, :1470-1500), linear extrapolation of
// velocity across the walls (the top plate's image from the plate value,
// :2461-2463), and zero reference map beyond the walls (an extrapolated
// Field carries only the ten primary members, src/field.hh:49-112).
#include <hip/hip_runtime.h>

#include <cmath>
#include <utility>

#include "../../include/stz.h"

// Every product and sum rounds on its own, as the reference's host code
// does, so that the explicit step matches it bit for bit where no
// transcendental function enters.
#pragma clang fp contract(off)

#include "stz_advect.hpp"
#include "stz_internal.hpp"

using namespace stz;

namespace {

inline unsigned nbk(long n) { return (unsigned)((n + kT - 1) / kT); }

struct Dyn {
    double rho, kappa, U;
    double ax, ay, az, Lx, Ly, Lz;
};

static __global__ __launch_bounds__(kT) void k_direct_plastic(Grid g, Mat M, double dt,
                                                              const double *__restrict__ sig,
                                                              const double *__restrict__ chi,
                                                              double *__restrict__ adapt, double *__restrict__ dchi,
                                                              double *__restrict__ dpl_new,
                                                              int *__restrict__ counters) {
    const long c = xcd_block() * kT + threadIdx.x;
    if (c >= g.Nc) return;
    double s[6];
#pragma unroll
    for (int q = 0; q < 6; q++) s[q] = sig[q * g.Nc + c];
    const double sb = sbar_of(s);
    double a = 0, dc = 0, D = 0;
    if (sb > M.sy) {
        int n;
        a = adaptive(M, sb, chi[c], dt, dc, n);
        D = a / 2. / M.mu / dt * sb;
    }
    count_wave(counters, sb > M.sy);
    adapt[c] = a;
    dchi[c] = dc;
    dpl_new[c] = D;
}

// Stress and chi of every cell, marching a tile of kAX x kAY cells through a
// chunk of z planes with the window of k_advect_march (stz_advect.hpp: the
// seven fields of a plane with a halo of two in LDS, a column's planes
// k - 2 .. k + 2 in registers, two vertex planes in LDS).  One thread per cell
// reading its 13-point stencils through the caches waited on some 130 loads
// at three waves per SIMD: 192 x 192 x 96 cells took 486 us, this form 275 us
// (0.6 GB of compulsory traffic, about 100 us).  What is left is the wait for
// a plane's loads between two barriers at two workgroups per CU (242
// registers; bounded to three it spills 124).
template <bool PZ>
static __global__ __launch_bounds__(kT) void k_direct_cell(
    Grid g, Mat M, double dt, AdvTiles T, const double *__restrict__ vel, const double *__restrict__ sig,
    const double *__restrict__ chi, const double *__restrict__ adapt, const double *__restrict__ dchi,
    const double *__restrict__ dnew, const double *__restrict__ dold, double *__restrict__ sig_out,
    double *__restrict__ chi_out) {
    constexpr int NF = 7;
    __shared__ double sc[NF][kSY * kSX];
    __shared__ double sv[2][3][kVY * kVX];

    const long Lb = xcd_block();
    const int tx = (int)(Lb % T.ntx), ty = (int)((Lb / T.ntx) % T.nty), zc = (int)(Lb / ((long)T.ntx * T.nty));
    const int k0 = zc * T.kchunk;
    if (k0 >= g.Nz) return;
    const int k1 = k0 + T.kchunk < g.Nz ? k0 + T.kchunk : g.Nz;
    const int i0 = tx * kAX, j0 = ty * kAY;
    const int tid = threadIdx.x, lx = tid % kAX, ly = tid / kAX;
    const int i = i0 + lx, j = j0 + ly;
    const bool act = i < g.Nx && j < g.Ny;
    const int nx = g.Nx, ny = g.Ny, nz = g.Nz;
    const int nxy = nx * ny;
    const int col = wrapm(i, nx) + nx * wrapm(j, ny);  // load position of this lane
    const long nc = g.Nc, nv = g.Nv;  // component strides (cell and vertex indices fit in int)

    // The positions a lane stages are those of every plane: formed once.
    static_assert(kHalo <= 2 * kT && kVX * kVY <= 2 * kT, "two positions per lane");
    int hp[2], hs[2], vp[2];
#pragma unroll
    for (int e = 0; e < 2; e++) {
        const int h = tid + e * kT;
        int sx, sy;
        halo_pos(h < kHalo ? h : 0, sx, sy);
        hp[e] = wrapm(i0 + sx - 2, nx) + nx * wrapm(j0 + sy - 2, ny);
        hs[e] = sy * kSX + sx;
        const int vy = h / kVX, vx = h - vy * kVX;
        vp[e] = wrapm(i0 + vx, nx) + nx * wrapm(j0 + vy, ny);
    }
    auto stage_vertices = [&](int kv) {
        const int kw = PZ ? wrapc(kv, nz) : kv;
        double(*dst)[kVY * kVX] = sv[kv & 1];
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const int h = tid + e * kT;
            if (h < kVX * kVY) {
                const int q = vp[e] + nxy * kw;
#pragma unroll
                for (int d = 0; d < 3; d++) dst[d][h] = vel[d * nv + q];
            }
        }
    };
    // field q (0..5 stress components, 6 chi) at offset p
    auto F = [&](int q, int p) -> double { return q < 6 ? sig[q * nc + p] : chi[p]; };

    // z window of this thread's column: w[q][s] holds plane k - 2 + s.
    // Across a wall the ghost planes follow the reference's extrapolation
    // f(-1) = 2 f(0) - f(1), f(-2) = 2 f(-1) - f(0) and its mirror at the
    // top, each formed from the two planes next to it in the window.
    double w[NF][5];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int kk = k0 - 2 + s;
        if (PZ || (kk >= 0 && kk < nz)) {
            const int p = col + nxy * (PZ ? wrapc(kk, nz) : kk);
#pragma unroll
            for (int q = 0; q < NF; q++) w[q][s] = F(q, p);
        }
    }
    if (!PZ) {
        if (k0 + 1 >= nz) {
#pragma unroll
            for (int q = 0; q < NF; q++) w[q][3] = (w[q][2] + w[q][2]) - w[q][1];
        }
#pragma unroll
        for (int s = 1; s >= 0; s--)
            if (k0 - 2 + s < 0) {
#pragma unroll
                for (int q = 0; q < NF; q++) w[q][s] = (w[q][s + 1] + w[q][s + 1]) - w[q][s + 2];
            }
    }
    stage_vertices(k0);

    const double hx = g.dx / dt, hy = g.dy / dt, hz = g.dz / dt;
    const int me = (ly + 2) * kSX + lx + 2;
    for (int k = k0; k < k1; k++) {
        if (PZ || k + 2 < nz) {
            const int p = col + nxy * (PZ ? wrapc(k + 2, nz) : k + 2);
#pragma unroll
            for (int q = 0; q < NF; q++) w[q][4] = F(q, p);
        } else {
#pragma unroll
            for (int q = 0; q < NF; q++) w[q][4] = (w[q][3] + w[q][3]) - w[q][2];
        }
        __syncthreads();  // the previous plane's LDS reads are done
#pragma unroll
        for (int q = 0; q < NF; q++) sc[q][me] = w[q][2];
#pragma unroll
        for (int e = 0; e < 2; e++)
            if (tid + e * kT < kHalo) {
                const int p = hp[e] + nxy * k;
#pragma unroll
                for (int q = 0; q < NF; q++) sc[q][hs[e]] = F(q, p);
            }
        stage_vertices(k + 1);
        __syncthreads();

        if (act) {
            const int c = i + nx * j + nxy * k;
            auto S = [&](int q, int dx, int dy) -> double { return sc[q][me + dy * kSX + dx]; };
            // vertex d of (i + a, j + b, k + e)
            auto V = [&](int d, int a, int b, int e) -> double {
                return sv[(k + e) & 1][d][(ly + b) * kVX + lx + a];
            };
            // velocity gradient and cell velocity (vel_grad_o)
            double G[3][3], v[3];
            {
                const double gx = .25 * (1.0 / g.dx), gy = .25 * (1.0 / g.dy), gz = .25 * (1.0 / g.dz);
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    const double u000 = V(q, 0, 0, 0), u100 = V(q, 1, 0, 0);
                    const double u010 = V(q, 0, 1, 0), u110 = V(q, 1, 1, 0);
                    const double u001 = V(q, 0, 0, 1), u101 = V(q, 1, 0, 1);
                    const double u011 = V(q, 0, 1, 1), u111 = V(q, 1, 1, 1);
                    G[q][0] = gx * (u100 - u000 + u110 - u010 + u101 - u001 + u111 - u011);
                    G[q][1] = gy * (u010 - u000 + u110 - u100 + u011 - u001 + u111 - u101);
                    G[q][2] = gz * (u001 - u000 + u101 - u100 + u011 - u010 + u111 - u110);
                    v[q] = 0.125 * (u000 + u100 + u001 + u101 + u010 + u110 + u011 + u111);
                }
            }
            const double dtlamb = dt * M.lamb, twomudt = 2 * M.mu * dt, dtmu = dt * M.mu;
            double ug[7];
#pragma unroll
            for (int q = 0; q < 7; q++) {
                const double f0 = S(q, 0, 0);
                const double ddx = eno2(hx, v[0], S(q, 2, 0), S(q, 1, 0), f0, S(q, -1, 0), S(q, -2, 0));
                const double ddy = eno2(hy, v[1], S(q, 0, 2), S(q, 0, 1), f0, S(q, 0, -1), S(q, 0, -2));
                const double ddz = eno2(hz, v[2], w[q][4], w[q][3], f0, w[q][1], w[q][0]);
                ug[q] = v[0] * ddx + v[1] * ddy + v[2] * ddz;
            }
            const double s11 = S(0, 0, 0), s12 = S(1, 0, 0), s13 = S(2, 0, 0);
            const double s22 = S(3, 0, 0), s23 = S(4, 0, 0), s33 = S(5, 0, 0);
            const double du_dx = G[0][0], du_dy = G[0][1], du_dz = G[0][2];
            const double dv_dx = G[1][0], dv_dy = G[1][1], dv_dz = G[1][2];
            const double dw_dx = G[2][0], dw_dy = G[2][1], dw_dz = G[2][2];
            const double d_trace = (du_dx + dv_dy + dw_dz);
            const double t11 = s11 * (du_dx - dv_dy - dw_dz) + 2 * s13 * du_dz + 2 * s12 * du_dy;
            const double t12 = s23 * du_dz + s13 * dv_dz - s12 * dw_dz + s22 * du_dy + s11 * dv_dx;
            const double t13 = s33 * du_dz + s11 * dw_dx + s23 * du_dy + s12 * dw_dy - s13 * dv_dy;
            const double t22 = 2 * s23 * dv_dz + s22 * (dv_dy - du_dx - dw_dz) + 2 * s12 * dv_dx;
            const double t23 = s33 * dv_dz + s22 * dw_dy + s13 * dv_dx - s23 * du_dx + s12 * dw_dx;
            const double t33 = s33 * (dw_dz - dv_dy - du_dx) + 2 * s23 * dw_dy + 2 * s13 * dw_dx;
            double cs11 = dtlamb * d_trace + twomudt * du_dx - ug[0] + dt * t11;
            double cs22 = dtlamb * d_trace + twomudt * dv_dy - ug[3] + dt * t22;
            double cs33 = dtlamb * d_trace + twomudt * dw_dz - ug[5] + dt * t33;
            double cs12 = dtmu * (du_dy + dv_dx) - ug[1] + dt * t12;
            double cs13 = dtmu * (du_dz + dw_dx) - ug[2] + dt * t13;
            double cs23 = dtmu * (dv_dz + dw_dy) - ug[4] + dt * t23;
            const double a = adapt[c];
            if (a != 0.0) {
                const double sig_trace = s11 + s22 + s33, third = 1. / 3.;
                cs11 -= a * (s11 - third * sig_trace);
                cs12 -= a * (s12);
                cs13 -= a * (s13);
                cs22 -= a * (s22 - third * sig_trace);
                cs23 -= a * (s23);
                cs33 -= a * (s33 - third * sig_trace);
            }
            sig_out[c] = s11 + cs11;
            sig_out[g.Nc + c] = s12 + cs12;
            sig_out[2 * g.Nc + c] = s13 + cs13;
            sig_out[3 * g.Nc + c] = s22 + cs22;
            sig_out[4 * g.Nc + c] = s23 + cs23;
            sig_out[5 * g.Nc + c] = s33 + cs33;
            // chi diffusion (chi_diffusion, src/shear_sim_3d.cpp:1217-1237)
            const double Dc = dnew[c];
            const double Dxm = i > 0 ? dnew[c - 1] : dold[c + (nx - 1)];
            const double Dxp = dold[c + (i + 1 < nx ? 1 : 1 - nx)];
            const double Dym = j > 0 ? dnew[c - nx] : dold[c + (ny - 1) * nx];
            const double Dyp = dold[c + (j + 1 < ny ? nx : -(ny - 1) * nx)];
            double Dzm, Dzp;
            if (PZ) {
                Dzm = k > 0 ? dnew[c - nxy] : dold[c + (nz - 1) * nxy];
                Dzp = dold[c + (k + 1 < nz ? nxy : -(nz - 1) * nxy)];
            } else {
                Dzm = k > 0 ? dnew[c - nxy] : 0.0;
                Dzp = k < nz - 1 ? dold[c + nxy] : 0.0;
            }
            const double x0 = S(6, 0, 0);
            const double xxm = S(6, -1, 0), xxp = S(6, 1, 0);
            const double xym = S(6, 0, -1), xyp = S(6, 0, 1);
            const double xzm = w[6][1], xzp = w[6][3];
            const double ix = 1 / g.dx, iy = 1 / g.dy, iz = 1 / g.dz;
            const double ddx = .5 * ix * (Dxp - Dxm) * (.5 * ix * (xxp - xxm)) + Dc * (ix * ix * (xxp - 2 * x0 + xxm));
            const double ddy = .5 * iy * (Dyp - Dym) * (.5 * iy * (xyp - xym)) + Dc * (iy * iy * (xyp - 2 * x0 + xym));
            const double ddz = .5 * iz * (Dzp - Dzm) * (.5 * iz * (xzp - xzm)) + Dc * (iz * iz * (xzp - 2 * x0 + xzm));
            const double diff = M.diff_l * M.diff_l * (ddx + ddy + ddz);
            double cchi = dchi[c];
            cchi -= ug[6];
            cchi += dt * diff / M.c0;
            chi_out[c] = x0 + cchi;
        }
#pragma unroll
        for (int q = 0; q < NF; q++)
#pragma unroll
            for (int s = 0; s < 4; s++) w[q][s] = w[q][s + 1];
    }
}

// Velocity and reference map of every vertex, marching like k_direct_cell: the
// six fields of a plane with a halo of two in LDS, a column's planes
// k - 2 .. k + 2 in registers, the stress of cell planes k - 1 and k (one more
// cell at -x and -y) in LDS.  One thread per vertex took 514 us at
// 192 x 192 x 96 cells, this form 236 us; bound as k_direct_cell is.  The wall
// ghosts of the velocity are extrapolated from the two planes next to them
// (2 f(0) - f(1) at k = -1, its mirror at Nz + 1); the reference map is zero
// there and shifted by the domain length at the periodic images of a
// component's own axis.
template <bool PZ>
static __global__ __launch_bounds__(kT) void k_direct_vertex(Grid g, Dyn D, double dt, AdvTiles T,
                                                             const double *__restrict__ vel,
                                                             const double *__restrict__ sig,
                                                             const double *__restrict__ xi,
                                                             double *__restrict__ vel_out,
                                                             double *__restrict__ xi_out) {
    constexpr int NF = 6;
    __shared__ double sc[NF][kSY * kSX];
    __shared__ double st[2][6][kVY * kVX];

    const long Lb = xcd_block();
    const int tx = (int)(Lb % T.ntx), ty = (int)((Lb / T.ntx) % T.nty), zc = (int)(Lb / ((long)T.ntx * T.nty));
    const int nx = g.Nx, ny = g.Ny, nz = g.Nz, nzv = g.Nzv;
    const int k0 = zc * T.kchunk;
    if (k0 >= nzv) return;
    const int k1 = k0 + T.kchunk < nzv ? k0 + T.kchunk : nzv;
    const int i0 = tx * kAX, j0 = ty * kAY;
    const int tid = threadIdx.x, lx = tid % kAX, ly = tid / kAX;
    const int i = i0 + lx, j = j0 + ly;
    const bool act = i < nx && j < ny;
    const int nxy = nx * ny;
    const int col = wrapm(i, nx) + nx * wrapm(j, ny);  // load position of this lane
    const long nc = g.Nc, nv = g.Nv;  // component strides (cell and vertex indices fit in int)

    // fields 0..2 velocity, 3..5 reference map at offset p; (a, b) is the
    // position in the plane, whose periodic images shift the map
    auto F = [&](int q, int p) -> double { return q < 3 ? vel[q * nv + p] : xi[(q - 3) * nv + p]; };
    auto shift = [](double v, int a, int n, double len) {
        return a >= n ? v + len : (a < 0 ? v - len : v);
    };
    auto image = [&](int q, double v, int a, int b) {
        return q == 3 ? shift(v, a, nx, D.Lx) : (q == 4 ? shift(v, b, ny, D.Ly) : v);
    };
    // plane kk of field q in this lane's column
    auto Z = [&](int q, int kk) -> double {
        if (PZ) {
            const double v = F(q, col + nxy * wrapc(kk, nz));
            return q == 5 ? shift(v, kk, nz, D.Lz) : v;
        }
        return F(q, col + nxy * kk);
    };
    int hp[2], hs[2], vp[2];  // the positions a lane stages of every plane
    int ha[2], hb[2];         // and their place before wrapping
#pragma unroll
    for (int e = 0; e < 2; e++) {
        const int h = tid + e * kT;
        int sx, sy;
        halo_pos(h < kHalo ? h : 0, sx, sy);
        const int a = i0 + sx - 2, b = j0 + sy - 2;
        hp[e] = wrapm(a, nx) + nx * wrapm(b, ny);
        hs[e] = sy * kSX + sx;
        ha[e] = a;
        hb[e] = b;
        const int vy = h / kVX, vx = h - vy * kVX;
        vp[e] = wrapm(i0 + vx - 1, nx) + nx * wrapm(j0 + vy - 1, ny);
    }
    auto stage_stress = [&](int kc) {
        double(*dst)[kVY * kVX] = st[kc & 1];
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const int h = tid + e * kT;
            if (h < kVX * kVY) {
                const int p = vp[e] + nxy * kc;
#pragma unroll
                for (int q = 0; q < 6; q++) dst[q][h] = sig[q * nc + p];
            }
        }
    };

    double w[NF][5];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int kk = k0 - 2 + s;
        if (PZ || (kk >= 0 && kk < nzv)) {
#pragma unroll
            for (int q = 0; q < NF; q++) w[q][s] = Z(q, kk);
        } else {
#pragma unroll
            for (int q = 0; q < NF; q++) w[q][s] = 0.0;
        }
    }
    if (k0 > 0) stage_stress(k0 - 1);

    const double dx_inv = 1. / g.dx, dy_inv = 1. / g.dy, dz_inv = 1. / g.dz;
    const double dx_inv_sq = dx_inv * dx_inv, dy_inv_sq = dy_inv * dy_inv, dz_inv_sq = dz_inv * dz_inv;
    const double rho_inv = 1. / D.rho;
    const double dtrho_inv = dt * rho_inv, dtkaprho_inv = D.kappa * dtrho_inv;
    const double dxdt = g.dx / dt, dydt = g.dy / dt, dzdt = g.dz / dt;
    const int me = (ly + 2) * kSX + lx + 2, mv = (ly + 1) * kVX + lx + 1;
    for (int k = k0; k < k1; k++) {
        if (PZ || k + 2 < nzv) {
#pragma unroll
            for (int q = 0; q < NF; q++) w[q][4] = Z(q, k + 2);
        } else {
            // only plane Nz + 1, seen from Nz - 1, is used
#pragma unroll
            for (int q = 0; q < NF; q++) w[q][4] = q < 3 ? (w[q][3] + w[q][3]) - w[q][2] : 0.0;
        }
        if (!PZ && k == 1) {
#pragma unroll
            for (int q = 0; q < 3; q++) w[q][0] = (w[q][1] + w[q][1]) - w[q][2];
        }
        __syncthreads();  // the previous plane's LDS reads are done
#pragma unroll
        for (int q = 0; q < NF; q++) sc[q][me] = image(q, w[q][2], i, j);
#pragma unroll
        for (int e = 0; e < 2; e++)
            if (tid + e * kT < kHalo) {
                const int p = hp[e] + nxy * k;
#pragma unroll
                for (int q = 0; q < NF; q++) sc[q][hs[e]] = image(q, F(q, p), ha[e], hb[e]);
            }
        if (k < nz) stage_stress(k);
        __syncthreads();

        if (act) {
            const int p = i + nx * j + nxy * k;
            if (k == 0 || k >= nz) {
                // the plane zz = 0 and the top plate are not updated here
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    vel_out[q * nv + p] = w[q][2];
                    xi_out[q * nv + p] = w[3 + q][2];
                }
            } else {
                auto S = [&](int q, int dx, int dy) -> double { return sc[q][me + dy * kSX + dx]; };
                // backward staggered stress derivatives
                // (calculate_first_order_stresses,
                // src/shear_sim_3d.cpp:971-987): cells (i-1..i, j-1..j, k-1..k)
                const double(*hi)[kVY * kVX] = st[k & 1], (*lo)[kVY * kVX] = st[(k - 1) & 1];
                auto DX = [&](int q) {
                    const double *a = hi[q] + mv, *b = lo[q] + mv;
                    return .25 * dx_inv * (a[0] - a[-1] + a[-kVX] - a[-kVX - 1] + b[0] - b[-1] + b[-kVX] - b[-kVX - 1]);
                };
                auto DY = [&](int q) {
                    const double *a = hi[q] + mv, *b = lo[q] + mv;
                    return .25 * dy_inv * (a[0] - a[-kVX] + a[-1] - a[-kVX - 1] + b[0] - b[-kVX] + b[-1] - b[-kVX - 1]);
                };
                auto DZ = [&](int q) {
                    const double *a = hi[q] + mv, *b = lo[q] + mv;
                    return .25 * dz_inv * (a[0] - b[0] + a[-1] - b[-1] + a[-kVX] - b[-kVX] + a[-kVX - 1] - b[-kVX - 1]);
                };
                const double div[3] = {DX(0) + DY(1) + DZ(2), DX(1) + DY(3) + DZ(4), DX(2) + DY(4) + DZ(5)};
                const double u = w[0][2], v = w[1][2], ww = w[2][2];
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    const double f0 = w[q][2], z1p = w[q][3], z1m = w[q][1];
                    const double xp = S(q, 1, 0), xm = S(q, -1, 0), yp = S(q, 0, 1), ym = S(q, 0, -1);
                    const double gsq = dx_inv_sq * (xp - 2 * f0 + xm) + dy_inv_sq * (yp - 2 * f0 + ym) +
                                       dz_inv_sq * (z1p - 2 * f0 + z1m);
                    const double ddx = eno2(dxdt, u, S(q, 2, 0), xp, f0, xm, S(q, -2, 0));
                    const double ddy = eno2(dydt, v, S(q, 0, 2), yp, f0, ym, S(q, 0, -2));
                    const double ddz = eno2(dzdt, ww, w[q][4], z1p, f0, z1m, w[q][0]);
                    const double ugq = u * ddx + v * ddy + ww * ddz;
                    vel_out[q * nv + p] = f0 + (dtrho_inv * div[q] + dtkaprho_inv * gsq - ugq);
                    const int x = 3 + q;
                    const double x0 = w[x][2];
                    const double ex = eno2(dxdt, u, S(x, 2, 0), S(x, 1, 0), x0, S(x, -1, 0), S(x, -2, 0));
                    const double ey = eno2(dydt, v, S(x, 0, 2), S(x, 0, 1), x0, S(x, 0, -1), S(x, 0, -2));
                    const double ez = eno2(dzdt, ww, w[x][4], w[x][3], x0, w[x][1], w[x][0]);
                    xi_out[q * nv + p] = x0 + (0.0 - (u * ex + v * ey + ww * ez));
                }
            }
        }
#pragma unroll
        for (int q = 0; q < NF; q++)
#pragma unroll
            for (int s = 0; s < 4; s++) w[q][s] = w[q][s + 1];
    }
}

// Top plate at time t: velocity (U t, 0, 0) (U for t >= 1) and reference map
// (a_x + i dx + U t^2 / 2 or + U (t - 1/2), a_y + j dy, 0).
static __global__ __launch_bounds__(kT) void k_direct_plate(Grid g, Dyn D, double t, double *__restrict__ vel,
                                                            double *__restrict__ xi) {
    const long q = xcd_block() * kT + threadIdx.x;
    const long nxy = (long)g.Nx * g.Ny;
    if (g.pz || q >= nxy) return;
    const int i = (int)(q % g.Nx), j = (int)(q / g.Nx);
    const long p = q + nxy * g.Nz;
    vel[p] = t < 1 ? D.U * t : D.U;
    vel[g.Nv + p] = 0;
    vel[2 * g.Nv + p] = 0;
    xi[p] = D.ax + i * g.dx + (t < 1 ? D.U * t * t * .5 : D.U * (t - 0.5));
    xi[g.Nv + p] = D.ay + j * g.dy;
    xi[2 * g.Nv + p] = 0;
}

// The reference map at the grid positions (init_ref, src/shear_sim_3d.cpp:
// 1036-1057) below the top plate.
static __global__ __launch_bounds__(kT) void k_init_ref(Grid g, Dyn D, double *__restrict__ xi) {
    const long p = xcd_block() * kT + threadIdx.x;
    if (p >= g.Nv) return;
    const int i = (int)(p % g.Nx);
    const int j = (int)((p / g.Nx) % g.Ny);
    const int k = (int)(p / ((long)g.Nx * g.Ny));
    if (k >= g.Nz) return;
    xi[p] = D.ax + g.dx * i;
    xi[g.Nv + p] = D.ay + g.dy * j;
    xi[2 * g.Nv + p] = D.az + g.dz * k;
}

// Block partials of l2_comparison (src/shear_sim_3d.cpp:3122-3158) over the
// points p < Nx Ny (Nz + 1): vertex velocity with the trapezoid weight in z
// (1/2 on plane 0 and on plane Nz, the top plate or the periodic image of
// plane 0), and for p < Nc the cell's six stress and chi differences.
// part[q nblocks + block], q = velocity, stress, chi (unscaled sums).
static __global__ __launch_bounds__(kT) void k_l2_parts(Grid g, const double *__restrict__ ua,
                                                        const double *__restrict__ sa, const double *__restrict__ xa,
                                                        const double *__restrict__ ub, const double *__restrict__ sb,
                                                        const double *__restrict__ xb, double *__restrict__ part) {
    const long p = xcd_block() * kT + threadIdx.x;
    const long nxy = (long)g.Nx * g.Ny;
    double v[3] = {0, 0, 0};
    if (p < nxy * (g.Nz + 1)) {
        const int k = (int)(p / nxy);
        const long pv = (g.pz && k == g.Nz) ? p - nxy * g.Nz : p;
        const double du = ua[pv] - ub[pv], dv = ua[g.Nv + pv] - ub[g.Nv + pv];
        const double dw = ua[2 * g.Nv + pv] - ub[2 * g.Nv + pv];
        if (k < g.Nz) {
            v[0] = (du * du + dv * dv + dw * dw) * (k == 0 ? .5 : 1);
            double t = 0;
#pragma unroll
            for (int q = 0; q < 6; q++) {
                const double d = sa[q * g.Nc + p] - sb[q * g.Nc + p];
                t += d * d;
            }
            v[1] = t;
            const double dc = xa[p] - xb[p];
            v[2] = dc * dc;
        } else {
            v[0] = .5 * (du * du + dv * dv + dw * dw);
        }
    }
    __shared__ double red[3][kT / 64];
#pragma unroll
    for (int q = 0; q < 3; q++) {
        double t = v[q];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) t += __shfl_down(t, off, 64);
        if ((threadIdx.x & 63) == 0) red[q][threadIdx.x >> 6] = t;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        double t = 0;
        for (int w = 0; w < kT / 64; w++) t += red[threadIdx.x][w];
        part[(long)threadIdx.x * gridDim.x + blockIdx.x] = t;
    }
}

#define DHIP(s, call)                                                                          \
    do {                                                                                       \
        hipError_t e_ = (call);                                                                \
        if (e_ != hipSuccess)                                                                  \
            return stz_detail::fail((s), STZMG_ERR_HIP, "%s: %s", #call, hipGetErrorString(e_)); \
    } while (0)

Dyn dyn_of(const stz_t s) {
    const stz_params &p = s->p;
    return Dyn{p.rho, p.kappa, p.U, p.ax, p.ay, p.az, p.bx - p.ax, p.by - p.ay, p.bz - p.az};
}

// Workgroups of a marching kernel the device keeps resident at once: one
// round of the launch.
template <typename F>
int resident(F *kernel) {
    int dev = 0, ncu = 0, per = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || ncu < 1)
        ncu = 256;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, kT, 0) != hipSuccess || per < 1) per = 1;
    return ncu * per;
}

template <bool PZ>
void launch_cell_z(stz_t s, double dt) {
    const Grid &g = s->g;
    int &r = s->direct_resident[PZ ? 1 : 0];
    if (r <= 0) r = resident(&k_direct_cell<PZ>);
    const AdvTiles t = adv_tiles(g, r);
    hipLaunchKernelGGL((k_direct_cell<PZ>), dim3((unsigned)((long)t.ntx * t.nty * t.nzc)), dim3(kT), 0, s->stream, g,
                       s->M, dt, t, (const double *)s->vel, (const double *)s->sig, (const double *)s->chi,
                       (const double *)s->adapt, (const double *)s->dchi, (const double *)s->dpl2,
                       (const double *)s->dpl, s->sig2, s->chi2);
}
void launch_cell(stz_t s, double dt) {
    if (s->g.pz) launch_cell_z<true>(s, dt);
    else launch_cell_z<false>(s, dt);
}

template <bool PZ>
void launch_vertex_z(stz_t s, const Dyn &D, double dt) {
    Grid g = s->g;
    int &r = s->direct_resident[PZ ? 3 : 2];
    if (r <= 0) r = resident(&k_direct_vertex<PZ>);
    g.Nz = g.Nzv;  // the planes the tiles march through
    const AdvTiles t = adv_tiles(g, r);
    hipLaunchKernelGGL((k_direct_vertex<PZ>), dim3((unsigned)((long)t.ntx * t.nty * t.nzc)), dim3(kT), 0, s->stream,
                       s->g, D, dt, t, (const double *)s->vel, (const double *)s->sig, (const double *)s->xi, s->vel2,
                       s->xi2);
}
void launch_vertex(stz_t s, const Dyn &D, double dt) {
    if (s->g.pz) launch_vertex_z<true>(s, D, dt);
    else launch_vertex_z<false>(s, D, dt);
}

int ensure_ref_map(stz_t s) {
    if (s->xi) return 0;
    const Grid &g = s->g;
    DHIP(s, hipMalloc((void **)&s->xi, sizeof(double) * 3 * g.Nv));
    DHIP(s, hipMalloc((void **)&s->xi2, sizeof(double) * 3 * g.Nv));
    DHIP(s, hipMalloc((void **)&s->vel2, sizeof(double) * 3 * g.Nv));
    DHIP(s, hipMemsetAsync(s->xi, 0, sizeof(double) * 3 * g.Nv, s->stream));
    return 0;
}

int check_direct(stz_t s) {
    if (s->p.transform != STZ_T_NONE)
        return stz_detail::fail(s, STZMG_ERR_UNSUPPORTED, "the direct step is the untransformed shear_sim_3d one");
    if (!(s->p.rho > 0) || !(s->p.kappa >= 0))
        return stz_detail::fail(s, STZMG_ERR_ARG, "direct step needs rho > 0 and kappa >= 0");
    return 0;
}

}  // namespace

extern "C" {

double stz_direct_dt(stz_t s) {
    if (!s) return 0;
    // solve_direct (src/shear_sim_3d.cpp:166-172)
    const double dx = s->g.dx, kappa = s->p.kappa, tmult = s->p.tmult;
    const double cfl = dx / 4.;
    if (!(kappa > 0)) return cfl;
    const double visc = dx * dx / 3. / kappa / 2.;
    return (tmult * visc < cfl) ? tmult * visc : cfl;
}

int stz_init_ref(stz_t s) {
    if (!s) return STZMG_ERR_ARG;
    if (int rc = ensure_ref_map(s)) return rc;
    const Grid &g = s->g;
    const Dyn D = dyn_of(s);
    hipLaunchKernelGGL(k_init_ref, dim3(nbk(g.Nv)), dim3(kT), 0, s->stream, g, D, s->xi);
    hipLaunchKernelGGL(k_direct_plate, dim3(nbk((long)g.Nx * g.Ny)), dim3(kT), 0, s->stream, g, D, s->t, s->vel,
                       s->xi);
    DHIP(s, hipGetLastError());
    DHIP(s, hipStreamSynchronize(s->stream));
    return 0;
}

int stz_set_ref_map(stz_t s, const double *xi) {
    if (!s || !xi) return STZMG_ERR_ARG;
    if (int rc = ensure_ref_map(s)) return rc;
    const Grid &g = s->g;
    DHIP(s, s->ring.upload(s->stage, xi, sizeof(double) * 3 * g.Nv, s->stream));
    hipLaunchKernelGGL(k_aos2soa, dim3(nbk(g.Nv)), dim3(kT), 0, s->stream, (const double *)s->stage, s->xi, g.Nv, 3);
    DHIP(s, hipGetLastError());
    DHIP(s, hipStreamSynchronize(s->stream));
    return 0;
}

int stz_get_ref_map(stz_t s, double *xi) {
    if (!s || !xi) return STZMG_ERR_ARG;
    if (!s->xi) return stz_detail::fail(s, STZMG_ERR_STATE, "no reference map (stz_init_ref or stz_set_ref_map)");
    const Grid &g = s->g;
    hipLaunchKernelGGL(k_soa2aos, dim3(nbk(g.Nv)), dim3(kT), 0, s->stream, (const double *)s->xi, s->stage, g.Nv, 3);
    DHIP(s, hipGetLastError());
    DHIP(s, s->ring.download(xi, s->stage, sizeof(double) * 3 * g.Nv, s->stream));
    return 0;
}

int stz_step_direct(stz_t s, double dt, int nsteps, stz_step_stats *st) {
    if (!s || !(dt > 0) || nsteps < 0) return STZMG_ERR_ARG;
    if (int rc = check_direct(s)) return rc;
    if (int rc = ensure_ref_map(s)) return rc;
    const Grid &g = s->g;
    const Dyn D = dyn_of(s);
    stz_step_stats S{};
    for (int q = 0; q < nsteps; q++) {
        DHIP(s, hipMemsetAsync(s->counters, 0, sizeof(int) * kCountInts, s->stream));
        hipLaunchKernelGGL(k_direct_plastic, dim3(nbk(g.Nc)), dim3(kT), 0, s->stream, g, s->M, dt,
                           (const double *)s->sig, (const double *)s->chi, s->adapt, s->dchi, s->dpl2, s->counters);
        launch_cell(s, dt);
        launch_vertex(s, D, dt);
        DHIP(s, hipGetLastError());
        std::swap(s->sig, s->sig2);
        std::swap(s->chi, s->chi2);
        std::swap(s->dpl, s->dpl2);
        std::swap(s->vel, s->vel2);
        std::swap(s->xi, s->xi2);
        s->t += dt;
        hipLaunchKernelGGL(k_direct_plate, dim3(nbk((long)g.Nx * g.Ny)), dim3(kT), 0, s->stream, g, D, s->t, s->vel,
                           s->xi);
        DHIP(s, hipGetLastError());
        S.steps++;
    }
    // one synchronisation per call: the counters hold the last step's count
    int cnt[kCountInts];
    DHIP(s, hipMemcpyAsync(cnt, s->counters, sizeof(cnt), hipMemcpyDeviceToHost, s->stream));
    DHIP(s, hipStreamSynchronize(s->stream));
    S.yielded_cells = nsteps ? count_total(cnt) : 0;
    if (st) *st = S;
    return 0;
}

int stz_l2_comparison(stz_t a, stz_t b, double l2[3]) {
    if (!a || !b || !l2) return STZMG_ERR_ARG;
    const Grid &g = a->g;
    if (b->g.Nx != g.Nx || b->g.Ny != g.Ny || b->g.Nz != g.Nz || b->g.pz != g.pz)
        return stz_detail::fail(a, STZMG_ERR_ARG, "l2_comparison: the two simulations have different grids");
    // b's fields must be complete before a's stream reads them
    DHIP(a, hipStreamSynchronize(b->stream));
    const long np = (long)g.Nx * g.Ny * (g.Nz + 1);
    const unsigned nb = nbk(np);
    double *part = a->stage;  // 3 nb partials + 3 sums: within 6 max(Nc, Nv) doubles
    double *sums = part + 3 * (long)nb;
    hipLaunchKernelGGL(k_l2_parts, dim3(nb), dim3(kT), 0, a->stream, g, (const double *)a->vel,
                       (const double *)a->sig, (const double *)a->chi, (const double *)b->vel,
                       (const double *)b->sig, (const double *)b->chi, part);
    for (int q = 0; q < 3; q++)
        hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(kT), 0, a->stream, (const double *)(part + (long)q * nb),
                           (long)nb, sums + q);
    DHIP(a, hipGetLastError());
    double h[3];
    DHIP(a, hipMemcpyAsync(h, sums, sizeof(h), hipMemcpyDeviceToHost, a->stream));
    DHIP(a, hipStreamSynchronize(a->stream));
    // normalisation (:3152-3155) with a's grid, plate speed and chi_inf
    const stz_params &p = a->p;
    const double norm_val = g.dx * g.dy * g.dz / ((p.bx - p.ax) * (p.by - p.ay) * (p.bz - p.az));
    l2[0] = h[0] * norm_val / (p.U * p.U);
    l2[1] = h[1] * norm_val;
    l2[2] = h[2] * norm_val / (p.chi_inf * p.chi_inf);
    return 0;
}

int stz_direct_time_kernels(stz_t s, double dt, int reps, double ms[4]) {
    if (!s || !(dt > 0) || reps < 1 || !ms) return STZMG_ERR_ARG;
    if (int rc = check_direct(s)) return rc;
    if (int rc = ensure_ref_map(s)) return rc;
    const Grid &g = s->g;
    const Dyn D = dyn_of(s);
    hipEvent_t e0, e1;
    DHIP(s, hipEventCreate(&e0));
    DHIP(s, hipEventCreate(&e1));
    // Every kernel reads the current state and writes the second buffers (the
    // plate kernel rewrites the plate's values at the current time), so the
    // repeated launches leave the state as it was.
    auto launch = [&](int which) {
        if (which == 0)
            hipLaunchKernelGGL(k_direct_plastic, dim3(nbk(g.Nc)), dim3(kT), 0, s->stream, g, s->M, dt,
                               (const double *)s->sig, (const double *)s->chi, s->adapt, s->dchi, s->dpl2,
                               s->counters);
        else if (which == 1)
            launch_cell(s, dt);
        else if (which == 2)
            launch_vertex(s, D, dt);
        else
            hipLaunchKernelGGL(k_direct_plate, dim3(nbk((long)g.Nx * g.Ny)), dim3(kT), 0, s->stream, g, D, s->t,
                               s->vel, s->xi);
    };
    int rc = 0;
    for (int w = 0; w < 4 && !rc; w++) {
        launch(w);  // warm
        hipEventRecord(e0, s->stream);
        for (int r = 0; r < reps; r++) launch(w);
        hipEventRecord(e1, s->stream);
        hipError_t e = hipEventSynchronize(e1);
        if (e == hipSuccess) e = hipGetLastError();
        float t = 0;
        if (e == hipSuccess) e = hipEventElapsedTime(&t, e0, e1);
        if (e != hipSuccess) rc = stz_detail::fail(s, STZMG_ERR_HIP, "direct kernel timing: %s", hipGetErrorString(e));
        ms[w] = (double)t / reps;
    }
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    return rc;
}

}  // extern "C"

// Tile classes of the marching kernels and the list of their instances.
//
// k_gs_march and k_resid_march are compiled in the mg_sweep_*.hip and
// mg_resid_*.hip files, one share of the instances each, so that the
// library builds in parallel; every other file only declares them.
#pragma once

#include "mg_halo.hpp"
#include "mg_march.hpp"
#include "mg_resid.hpp"
#include "mg_restrict.hpp"

namespace stzmg {

// Tiles of the plane-marching residual (k_resid_march): 64 x 16 in FP32,
// 32 x 16 in FP64, 256 threads.
template <typename T>
struct ResidTile;
template <>
struct ResidTile<float> {
    static constexpr int TX = 64, TY = 16;
};
template <>
struct ResidTile<double> {
    static constexpr int TX = 32, TY = 16;
};

// Tile and workgroup size of the large fused-smoother class (k_gs_march):
// 64 x 16 with 512 threads in FP32 (three staged planes of 71 x 24 points,
// 61,344 B of LDS: two workgroups per CU) and 32 x 16 with 256 threads in
// FP64 (39 x 24 points, 67,392 B: two per CU).  Measured on the 256^3
// transformed-operator sweep (MI355X): FP32 64 x 16 / 512 threads 0.256 ms,
// 64 x 8 / 256 0.272 ms, 32 x 16 / 256 0.291 ms; FP64 32 x 16 0.519 ms,
// 32 x 8 0.666 ms.
#ifndef STZ_F32_TX
#define STZ_F32_TX 64
#endif
#ifndef STZ_F32_TY
#define STZ_F32_TY 16
#endif
#ifndef STZ_F32_NT
#define STZ_F32_NT 512
#endif
#ifndef STZ_F64_TX
#define STZ_F64_TX 32
#endif
#ifndef STZ_F64_TY
#define STZ_F64_TY 16
#endif
#ifndef STZ_F64_NT
#define STZ_F64_NT 256
#endif
template <typename T>
struct FusedTile;
template <>
struct FusedTile<float> {
    static constexpr int TX = STZ_F32_TX, TY = STZ_F32_TY, NT = STZ_F32_NT;
};
template <>
struct FusedTile<double> {
    static constexpr int TX = STZ_F64_TX, TY = STZ_F64_TY, NT = STZ_F64_NT;
};

// The small classes: 16 x 16 tiles with 128 threads and 8 x 8 tiles with one
// wave (sweep), 16 x 16 tiles (residual).
constexpr int kSmallTile = 16, kSmallThreads = 128;
constexpr int kTinyTile = 8, kTinyThreads = 64;
constexpr int kResidSmall = 16;
// Tile of the one-launch sweep (k_gs_halo).
constexpr int kHaloTile = 8;

#define STZ_SWEEP_SIG(T) \
    (Dims, const T *__restrict__, const T *__restrict__, T *__restrict__, const T *__restrict__, \
     const T *__restrict__, int, int, int)
#define STZ_SWEEP_INST(PRE, T, KEY)                                                                                   \
    PRE template __global__ void k_gs_march<T, KEY, FusedTile<T>::TX, FusedTile<T>::TY, FusedTile<T>::NT>             \
        STZ_SWEEP_SIG(T);                                                                                             \
    PRE template __global__ void k_gs_march<T, KEY, kSmallTile, kSmallTile, kSmallThreads> STZ_SWEEP_SIG(T);          \
    PRE template __global__ void k_gs_march<T, KEY, kTinyTile, kTinyTile, kTinyThreads> STZ_SWEEP_SIG(T);
#define STZ_SWEEP_PLAIN(PRE, T) \
    STZ_SWEEP_INST(PRE, T, 0) STZ_SWEEP_INST(PRE, T, 1) STZ_SWEEP_INST(PRE, T, 2) STZ_SWEEP_INST(PRE, T, 3)
#define STZ_SWEEP_SYM(PRE, T) \
    STZ_SWEEP_INST(PRE, T, 4) STZ_SWEEP_INST(PRE, T, 5) STZ_SWEEP_INST(PRE, T, 6) STZ_SWEEP_INST(PRE, T, 7)

#define STZ_HALO_SIG(T) \
    (Dims, const T *__restrict__, T *__restrict__, const T *__restrict__, const T *__restrict__, int, Dims, \
     const T *__restrict__)
#define STZ_RR_SIG(T) \
    (Dims, Dims, const T *__restrict__, const T *__restrict__, const T *__restrict__, T *__restrict__, T *__restrict__)
#define STZ_HALO_INST(PRE, T, KEY)                                                        \
    PRE template __global__ void k_gs_halo<T, KEY, kHaloTile, kHaloTile> STZ_HALO_SIG(T); \
    PRE template __global__ void k_resid_restrict<T, KEY> STZ_RR_SIG(T);
#define STZ_HALO_PLAIN(PRE, T) \
    STZ_HALO_INST(PRE, T, 0) STZ_HALO_INST(PRE, T, 1) STZ_HALO_INST(PRE, T, 2) STZ_HALO_INST(PRE, T, 3)
#define STZ_HALO_SYM(PRE, T) \
    STZ_HALO_INST(PRE, T, 4) STZ_HALO_INST(PRE, T, 5) STZ_HALO_INST(PRE, T, 6) STZ_HALO_INST(PRE, T, 7)

#define STZ_RESID_SIG(T) \
    (Dims, const T *__restrict__, const T *__restrict__, const T *__restrict__, T *__restrict__, double *__restrict__, \
     int, T *__restrict__)
#define STZ_RESID_ONE(PRE, T, KEY, NORM, APPLY, TX, TY) \
    PRE template __global__ void k_resid_march<T, KEY, NORM, APPLY, TX, TY, kThreads> STZ_RESID_SIG(T);
#define STZ_RESID_INST(PRE, T, KEY)                                                  \
    STZ_RESID_ONE(PRE, T, KEY, true, false, ResidTile<T>::TX, ResidTile<T>::TY)      \
    STZ_RESID_ONE(PRE, T, KEY, false, false, ResidTile<T>::TX, ResidTile<T>::TY)     \
    STZ_RESID_ONE(PRE, T, KEY, false, true, ResidTile<T>::TX, ResidTile<T>::TY)      \
    STZ_RESID_ONE(PRE, T, KEY, false, false, kResidSmall, kResidSmall)               \
    STZ_RESID_ONE(PRE, T, KEY, false, true, kResidSmall, kResidSmall)                \
    STZ_RESID_ONE(PRE, T, KEY, true, false, kResidSmall, kResidSmall)
#define STZ_RESID_ALL(PRE, T)                                                                                \
    STZ_RESID_INST(PRE, T, 0) STZ_RESID_INST(PRE, T, 1) STZ_RESID_INST(PRE, T, 2) STZ_RESID_INST(PRE, T, 3)  \
    STZ_RESID_INST(PRE, T, 4) STZ_RESID_INST(PRE, T, 5) STZ_RESID_INST(PRE, T, 6) STZ_RESID_INST(PRE, T, 7)

STZ_SWEEP_PLAIN(extern, float)
STZ_SWEEP_PLAIN(extern, double)
STZ_SWEEP_SYM(extern, float)
STZ_SWEEP_SYM(extern, double)
STZ_HALO_PLAIN(extern, float)
STZ_HALO_PLAIN(extern, double)
STZ_HALO_SYM(extern, float)
STZ_HALO_SYM(extern, double)
STZ_RESID_ALL(extern, float)
STZ_RESID_ALL(extern, double)

}  // namespace stzmg

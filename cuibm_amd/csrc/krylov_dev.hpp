// Device pieces shared by the BiCGSTAB kernels: block reductions, and the finish of a reduction
// inside the kernel that needs its result.
#pragma once
#include <hip/hip_runtime.h>

#include "krylov.hpp"

namespace cuibm {

// Sum over the wavefront in lane 0, in the order of a shfl_down tree (offsets 32, 16, 8, 4, 2, 1).
// The lanes come by register permutes (row shifts within 16 lanes, the gfx950 half and row swaps
// above) instead of through LDS: a reduction's tail is a chain of six of them.
template <int CTRL>
__device__ __forceinline__ double dpp_down(double v) {
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ double wave_sum(double v) {
    const auto h32 = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
    const auto l32 = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
    v += __hiloint2double((int)h32[1], (int)l32[1]);  // lanes 0..31: lane + 32
    const auto h16 = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
    const auto l16 = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
    v += __hiloint2double((int)h16[1], (int)l16[1]);  // lanes 0..15: lane + 16
    v += dpp_down<0x108>(v);                          // row_shl: lane + 8, 4, 2, 1 of the row
    v += dpp_down<0x104>(v);
    v += dpp_down<0x102>(v);
    v += dpp_down<0x101>(v);
    return v;
}

// reduce K values per thread across each group of BS threads of a block of TB; the group's first
// thread gets the sums
template <int K, int TB = BS>
__device__ __forceinline__ void block_sum(double (&v)[K]) {
    __shared__ double sh[K][TB / 64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, w0 = wid & ~3;
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = wave_sum(v[k]);
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < K; k++) sh[k][wid] = v[k];
    __syncthreads();
    if (threadIdx.x % BS == 0)
#pragma unroll
        for (int k = 0; k < K; k++) v[k] = (sh[k][w0] + sh[k][w0 + 1]) + (sh[k][w0 + 2] + sh[k][w0 + 3]);
}

// the thread's group of a reduction (see red_parts) in block blk, and its index in the group
template <int TB>
__device__ __forceinline__ int red_group(int blk) {
    return TB == BS ? blk : blk * (TB / BS) + (int)threadIdx.x / BS;
}
__device__ __forceinline__ int red_lane() { return threadIdx.x % BS; }

// the totals of NG groups of partials in every thread of a block of TB threads, added as
// k_bicg_finish's 1024 threads add them (a wavefront of a smaller block stands for several of its
// 16), so fused and separate finishes give the same bits. A small block has at most FUSE_PARTS.
template <int NG, int TB>
__device__ __forceinline__ void finish_sums(const FinArgs &f, double (&tot)[2]) {
    constexpr int PER = TB == RED_WIDE ? 1 : FUSE_PARTS / TB, NW = TB / 64;
    __shared__ double sh[NG][16];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    double v[NG][PER];
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int k = (int)threadIdx.x + TB * j;
            const double *p = f.part + (size_t)g * f.np;
            v[g][j] = k < f.np ? p[k] : 0.0;
            if (TB == RED_WIDE && k + RED_WIDE < f.np) v[g][j] += p[k + RED_WIDE];
        }
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const double t = wave_sum(v[g][j]);
            if (lane == 0) sh[g][wid + NW * j] = t;
        }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < NG; g++) {
        double t = 0;
#pragma unroll
        for (int w = 0; w < NW * PER; w++) t += sh[g][w];
        tot[g] = t;
    }
}

// The scalar updates of one iteration's reductions (see FinArgs). Each returns the value its
// consumer needs; `write` (one thread of the grid) stores what later kernels read. A slot that
// is written here is read by no other block of the same launch: rho and the stop code have one
// slot per parity of the iteration, the stop code of the half step one of its own.
__device__ __forceinline__ double fin_alpha(const double (&tot)[2], double *sc, int par, bool write) {
    const double alpha = sc[sc_rho(par)] / tot[0];
    if (write) sc[SC_ALPHA] = alpha;
    return alpha;
}
// the stop code of the half step: a breakdown, or the monitor's test on ||s||
__device__ __forceinline__ double fin_ss(const double (&tot)[2], double *sc, bool write) {
    double code = 0.0;
    if (!isfinite(tot[0]) || !isfinite(sc[SC_ALPHA])) code = STOP_BREAK_HALF;
    else if (sqrt(tot[0]) <= sc[SC_TOL]) code = STOP_HALF_PENDING;
    if (write) {
        sc[SC_SS] = tot[0];
        sc[SC_STOPS] = code;
    }
    return code;
}
__device__ __forceinline__ double fin_omega(const double (&tot)[2], double *sc, bool write) {
    const double w = tot[0] / tot[1];  // (AMs.s, AMs.AMs); a breakdown leaves omega = 0 so that x stays finite
    const double omega = isfinite(w) ? w : 0.0;
    if (write) sc[SC_OMEGA] = omega;
    return omega;
}
// (rs.r, r.r): the monitor's test on ||r||, the breakdown tests and the iteration limit
__device__ __forceinline__ double fin_beta(const double (&tot)[2], double *sc, int par, int maxit, bool write) {
    const double beta = (tot[0] / sc[sc_rho(par)]) * (sc[SC_ALPHA] / sc[SC_OMEGA]);
    if (write) {
        const double rn = sqrt(tot[1]), its = sc[SC_ITS] + 1.0;
        sc[SC_BETA] = beta;
        sc[sc_rho(par ^ 1)] = tot[0];
        sc[SC_RR] = tot[1];
        sc[SC_ITS] = its;
        double code = 0.0;
        if (rn <= sc[SC_TOL]) code = STOP_CONVERGED;
        else if (sc[SC_OMEGA] == 0.0 || tot[0] == 0.0 || !isfinite(beta) || !isfinite(rn)) code = STOP_BREAK_FULL;
        else if (its >= (double)maxit) code = STOP_MAXIT;
        sc[sc_stop(par ^ 1)] = code;
    }
    return beta;
}
// the next iteration's stop code after an iteration that began or ended stopped
__device__ __forceinline__ void pass_stop(double *sc, int par) {
    const double a = sc[sc_stop(par)], h = sc[SC_STOPS];
    sc[sc_stop(par ^ 1)] = a != 0.0 ? a : h == STOP_HALF_PENDING ? (double)STOP_HALF : h;
}

}  // namespace cuibm

// Vector, reduction and sparse-product kernels for the Krylov and AMG solvers.
//
// Reductions are deterministic: groups that depend on n alone (red_parts) strides over the
// vector, each block reduces its threads in a fixed tree (wavefront shuffles, then
// LDS across the 4 wavefronts of a 256-thread block) and writes one partial; the
// consumer, or a single-block kernel, then sums the partials in a fixed order. The result
// depends only on n, never on scheduling.
#include "batch.hpp"
#include "krylov.hpp"
#include "krylov_dev.hpp"
#include "kernels.hpp"

namespace cuibm {

template <class T>
__global__ void k_fill(T *x, T v, long n) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) x[i] = v;
}
__global__ void k_copy(double *__restrict__ y, const double *__restrict__ x, long n, const double *__restrict__ stop) {
    const double stopv = stop ? *stop : 0.0;  // read at once, tested after the first load
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        const double v = x[i];
        if (stopv != 0.0) return;
        y[i] = v;
    }
}
__global__ void k_to_float(float *__restrict__ y, const double *__restrict__ x, long n) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) y[i] = (float)x[i];
}
__global__ void k_to_double(double *__restrict__ y, const float *__restrict__ x, long n) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) y[i] = (double)x[i];
}

static int grid_for(long n) {
    const long b = (n + BS - 1) / BS;
    return (int)(b < 65536 ? b : 65536);
}

void launch_fill(double *x, double v, long n, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_fill<double>, dim3(grid_for(n)), dim3(BS), 0, s, x, v, n);
    CUIBM_LAUNCH_CHECK();
}
void launch_fill_i(int *x, int v, long n, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_fill<int>, dim3(grid_for(n)), dim3(BS), 0, s, x, v, n);
    CUIBM_LAUNCH_CHECK();
}
void launch_copy(double *y, const double *x, long n, hipStream_t s, const double *stop) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_copy, dim3(grid_for(n)), dim3(BS), 0, s, y, x, n, stop);
    CUIBM_LAUNCH_CHECK();
}
void launch_to_float(float *y, const double *x, long n, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_to_float, dim3(grid_for(n)), dim3(BS), 0, s, y, x, n);
    CUIBM_LAUNCH_CHECK();
}
void launch_to_double(double *y, const float *x, long n, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_to_double, dim3(grid_for(n)), dim3(BS), 0, s, y, x, n);
    CUIBM_LAUNCH_CHECK();
}

// ---- sparse matrix-vector products --------------------------------------------------

template <class V, class X>
__device__ __forceinline__ X row_dot(const int *__restrict__ rp, const int *__restrict__ ci, const V *__restrict__ v,
                                     const X *__restrict__ x, int i) {
    return (X)csr_row_sum<double>(ci, v, x, rp[i], rp[i + 1]);  // FP64 accumulation also for float operands
}

template <class V, class X>
__global__ void __launch_bounds__(BS) k_spmv(int n, const int *__restrict__ rp, const int *__restrict__ ci,
                                             const V *__restrict__ v, const X *__restrict__ x, X *__restrict__ y) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) y[i] = row_dot(rp, ci, v, x, i);
}

template <class V, class X>
void launch_spmv(const DCsr<V> &A, const X *x, X *y, hipStream_t s) {
    if (A.n <= 0) return;
    hipLaunchKernelGGL((k_spmv<V, X>), dim3(grid_for(A.n)), dim3(BS), 0, s, A.n, A.rp.p(), A.ci.p(), A.v.p(), x, y);
    CUIBM_LAUNCH_CHECK();
}
template void launch_spmv<double, double>(const DCsr<double> &, const double *, double *, hipStream_t);
template void launch_spmv<float, double>(const DCsr<float> &, const double *, double *, hipStream_t);

// y = A x with block partials of (y . a) and, when want_yy is set, (y . y). JAC: x = D^-1 p, formed
// at every gather, and written to Mp.
// Each block takes a contiguous chunk of rows, and the chunks of one XCD are contiguous too, so
// that the gathers of x from neighbouring rows stay in that XCD's L2.
template <bool JAC, int TB>
__global__ void __launch_bounds__(TB) k_spmv_dot(int n, const int *__restrict__ rp, const int *__restrict__ ci,
                                                 const double *__restrict__ val, const double *__restrict__ x,
                                                 const double *__restrict__ dinv, double *__restrict__ Mp,
                                                 double *__restrict__ y, const double *__restrict__ a, int want_yy,
                                                 FinArgs f, double *__restrict__ part, const double *__restrict__ stop) {
    const double stopv = stop ? *stop : 0.0;  // read at once, tested after the first row
    if (JAC && f.part) {
        double tot[2] = {0, 0};
        finish_sums<1, TB>(f, tot);
        if (stopv != 0.0) return;  // uniform, as every return before the last barrier
        if (fin_ss(tot, f.sc, blockIdx.x == 0 && threadIdx.x == 0) != 0.0) return;
    }
    double acc[2] = {0, 0};
    bool tested = false;
    const int np = red_parts(n), chunk = (n + np - 1) / np;
    // group v = x + 8 c takes chunk x np / 8 + c; the groups of a block share x, its XCD
    const int c = red_group<TB>(blockIdx.x / 8), v = c < np / 8 ? (int)(blockIdx.x % 8) + 8 * c : np;
    const int r0 = v < np ? ((int)(blockIdx.x % 8) * (np / 8) + c) * chunk : n, r1 = min(n, r0 + chunk);
    for (int i = r0 + red_lane(); i < r1; i += BS) {
        double yi;
        if (JAC) {
            yi = csr_lane_sum<double, 1>(ci, val, rp[i], rp[i + 1], [&](int c) { return dinv[c] * x[c]; });
        } else {
            yi = row_dot(rp, ci, val, x, i);
        }
        if (!tested) {
            if (stopv != 0.0) return;  // every thread returns here or below: no barrier is reached
            tested = true;
        }
        if (JAC) Mp[i] = dinv[i] * x[i];
        y[i] = yi;
        acc[0] += yi * a[i];
        acc[1] += yi * yi;
    }
    if (stopv != 0.0) return;
    block_sum<2, TB>(acc);
    if (red_lane() == 0 && v < np) {
        part[v] = acc[0];
        if (want_yy) part[np + v] = acc[1];
    }
}

void launch_spmv_dot(const DCsr<double> &A, const double *x, double *y, const double *a, bool want_yy, double *part,
                     hipStream_t s, const double *stop) {
    by_block(A.n, [&](auto tb) {
        hipLaunchKernelGGL((k_spmv_dot<false, tb>), dim3(red_grid(A.n)), dim3(tb), 0, s, A.n, A.rp.p(), A.ci.p(),
                           A.v.p(), x, nullptr, nullptr, y, a, (int)want_yy, FinArgs{}, part, stop);
    });
    CUIBM_LAUNCH_CHECK();
}

void launch_spmv_dot_jacobi(const DCsr<double> &A, const double *dinv, const double *p, double *Mp, double *y,
                            const double *a, bool want_yy, const FinArgs &f, double *part, hipStream_t s,
                            const double *stop) {
    by_block(A.n, [&](auto tb) {
        hipLaunchKernelGGL((k_spmv_dot<true, tb>), dim3(red_grid(A.n)), dim3(tb), 0, s, A.n, A.rp.p(), A.ci.p(),
                           A.v.p(), p, dinv, Mp, y, a, (int)want_yy, f, part, stop);
    });
    CUIBM_LAUNCH_CHECK();
}

// r = b - A x; also p = r and rs = r when given; partials of (r.r) and (b.b)
template <int TB>
__global__ void __launch_bounds__(TB) k_bicg_init(int n, const int *__restrict__ rp, const int *__restrict__ ci,
                                                  const double *__restrict__ val, const double *__restrict__ x,
                                                  const double *__restrict__ b, double *__restrict__ r,
                                                  double *__restrict__ p, double *__restrict__ rs,
                                                  double *__restrict__ part) {
    double acc[2] = {0, 0};
    const int np = red_parts(n), v = red_group<TB>(blockIdx.x);
    for (int i = v < np ? v * BS + red_lane() : n; i < n; i += np * BS) {
        const double bi = b[i];
        const double ri = bi - row_dot(rp, ci, val, x, i);
        r[i] = ri;
        p[i] = ri;
        rs[i] = ri;
        acc[0] += ri * ri;
        acc[1] += bi * bi;
    }
    block_sum<2, TB>(acc);
    if (red_lane() == 0 && v < np) {
        part[v] = acc[0];
        part[np + v] = acc[1];
    }
}

void launch_bicg_init(const DCsr<double> &A, const double *x, const double *b, double *r, double *p, double *rs,
                      double *part, hipStream_t s) {
    by_block(A.n, [&](auto tb) {
        hipLaunchKernelGGL(k_bicg_init<tb>, dim3(red_grid(A.n)), dim3(tb), 0, s, A.n, A.rp.p(), A.ci.p(), A.v.p(), x,
                           b, r, p, rs, part);
    });
    CUIBM_LAUNCH_CHECK();
}

// s = r - alpha AMp with partials of (s.s)
template <bool W, int TB>
__global__ void __launch_bounds__(TB) k_bicg_s(int n, const double *__restrict__ r, const double *__restrict__ AMp,
                                               double *__restrict__ s, FinArgs f, double *__restrict__ part,
                                               InputWeights w) {
    const int np = red_parts(n), v = red_group<TB>(blockIdx.x);
    int i = v < np ? v * BS + red_lane() : n;
    double rv = i < n ? r[i] : 0.0, av = i < n ? AMp[i] : 0.0;  // in flight during the finish
    const double stopv = f.sc[sc_stop(f.par)];
    double tot[2] = {0, 0};
    finish_sums<1, TB>(f, tot);
    if (stopv != 0.0) return;  // uniform, as every return before the last barrier
    const double alpha = fin_alpha(tot, f.sc, f.par, blockIdx.x == 0 && threadIdx.x == 0);
    double acc[2] = {0, 0};
    while (i < n) {
        const double si = rv - alpha * av;
        s[i] = si;
        acc[0] += si * si;
        if (W) acc[1] += (w.wx[i % w.nx] * w.wy[i / w.nx]) * si;
        i += np * BS;
        if (i < n) {
            rv = r[i];
            av = AMp[i];
        }
    }
    block_sum<2, TB>(acc);
    if (red_lane() == 0 && v < np) {
        part[v] = acc[0];
        if (W) w.part[v] = acc[1];
    }
}

void launch_bicg_s(int n, const double *r, const double *AMp, double *s_, const FinArgs &f, double *part,
                   hipStream_t s, const InputWeights *w) {
    const dim3 g(red_grid(n));
    by_block(n, [&](auto tb) {
        if (w) hipLaunchKernelGGL((k_bicg_s<true, tb>), g, dim3(tb), 0, s, n, r, AMp, s_, f, part, *w);
        else hipLaunchKernelGGL((k_bicg_s<false, tb>), g, dim3(tb), 0, s, n, r, AMp, s_, f, part, InputWeights{});
    });
    CUIBM_LAUNCH_CHECK();
}

// x += alpha Mp + omega Ms; r = s - omega AMs; partials of (rs.r) and (r.r). In the
// iteration that ended at its half step (STOP_HALF_PENDING) it applies the half-step update
// x += alpha Mp alone.
template <int TB>
__global__ void __launch_bounds__(TB) k_bicg_xr(int n, double *__restrict__ x, const double *__restrict__ Mp,
                                                const double *__restrict__ Ms, double *__restrict__ r,
                                                const double *__restrict__ s, const double *__restrict__ AMs,
                                                const double *__restrict__ rs, FinArgs f, double *__restrict__ part) {
    const int np = red_parts(n), v = red_group<TB>(blockIdx.x);
    int i = v < np ? v * BS + red_lane() : n;
    auto at = [&](const double *a) { return i < n ? a[i] : 0.0; };
    double xv = at(x), mp = at(Mp), ms = at(Ms), sv = at(s), am = at(AMs), rv = at(rs);  // in flight during the finish
    const double stopv = f.sc[sc_stop(f.par)], half_code = f.sc[SC_STOPS], alpha = f.sc[SC_ALPHA];
    const bool half = stopv == 0.0 && half_code == STOP_HALF_PENDING;
    const bool stopped = stopv != 0.0 || half_code != 0.0;
    double tot[2] = {0, 0};
    finish_sums<2, TB>(f, tot);
    const double omega = stopped ? 0.0 : fin_omega(tot, f.sc, blockIdx.x == 0 && threadIdx.x == 0);
    if (stopped && !half) return;  // uniform, as every return before the last barrier
    double acc[2] = {0, 0};
    while (i < n) {
        const double xh = xv + alpha * mp;
        if (half) {
            x[i] = xh;
        } else {
            const double ri = sv - omega * am;
            x[i] = xh + omega * ms;
            r[i] = ri;
            acc[0] += rv * ri;
            acc[1] += ri * ri;
        }
        i += np * BS;
        if (i < n) {
            xv = x[i];
            mp = Mp[i];
            ms = Ms[i];
            sv = s[i];
            am = AMs[i];
            rv = rs[i];
        }
    }
    if (half) return;
    block_sum<2, TB>(acc);
    if (red_lane() == 0 && v < np) {
        part[v] = acc[0];
        part[np + v] = acc[1];
    }
}

void launch_bicg_xr(int n, double *x, const double *Mp, const double *Ms, double *r, const double *s_,
                    const double *AMs, const double *rs, const FinArgs &f, double *part, hipStream_t s) {
    by_block(n, [&](auto tb) {
        hipLaunchKernelGGL(k_bicg_xr<tb>, dim3(red_grid(n)), dim3(tb), 0, s, n, x, Mp, Ms, r, s_, AMs, rs, f, part);
    });
    CUIBM_LAUNCH_CHECK();
}

// p = r + beta p - beta omega AMp; W: with the weighted partial sums of the new p
template <bool W, int TB>
__global__ void __launch_bounds__(TB) k_bicg_p(int n, double *__restrict__ p, const double *__restrict__ r,
                                               const double *__restrict__ AMp, FinArgs f, InputWeights w) {
    const int np = red_parts(n), v = red_group<TB>(blockIdx.x);
    int i = v < np ? v * BS + red_lane() : n;
    double pv = i < n ? p[i] : 0.0, rv = i < n ? r[i] : 0.0, av = i < n ? AMp[i] : 0.0;  // in flight during the finish
    const double omega = f.sc[SC_OMEGA];
    const bool one = blockIdx.x == 0 && threadIdx.x == 0;
    const bool stopped = f.sc[sc_stop(f.par)] != 0.0 || f.sc[SC_STOPS] != 0.0;
    double tot[2] = {0, 0};
    finish_sums<2, TB>(f, tot);
    if (stopped) {
        if (one) pass_stop(f.sc, f.par);
        return;  // uniform, as every return before the last barrier
    }
    const double beta = fin_beta(tot, f.sc, f.par, f.maxit, one);  // a p past the last iteration is not used
    double acc[1] = {0};
    while (i < n) {
        const double pi = rv + beta * pv - beta * omega * av;
        p[i] = pi;
        if (W) acc[0] += (w.wx[i % w.nx] * w.wy[i / w.nx]) * pi;
        i += np * BS;
        if (i < n) {
            pv = p[i];
            rv = r[i];
            av = AMp[i];
        }
    }
    if (!W) return;
    block_sum<1, TB>(acc);
    if (red_lane() == 0 && v < np) w.part[v] = acc[0];
}

void launch_bicg_p(int n, double *p, const double *r, const double *AMp, const FinArgs &f, hipStream_t s,
                   const InputWeights *w) {
    const dim3 g(red_grid(n));
    by_block(n, [&](auto tb) {
        if (w) hipLaunchKernelGGL((k_bicg_p<true, tb>), g, dim3(tb), 0, s, n, p, r, AMp, f, *w);
        else hipLaunchKernelGGL((k_bicg_p<false, tb>), g, dim3(tb), 0, s, n, p, r, AMp, f, InputWeights{});
    });
    CUIBM_LAUNCH_CHECK();
}

// the scalar updates and stopping tests of one finish of a batched case, from the summed
// partials tot
__device__ __forceinline__ void finish_update(int op, const double (&tot)[2], double *__restrict__ sc, double tol,
                                              int maxit) {
    switch (op) {
        case FIN_INIT:  // (r.r, b.b); a (re)start clears the stop code, the count goes on
            sc[SC_RR] = tot[0];
            sc[SC_RHO] = tot[0];
            sc[SC_BB] = tot[1];
            sc[SC_STOP] = 0.0;
            break;
        case FIN_ALPHA:  // rs.AMp
            sc[SC_ALPHA] = sc[SC_RHO] / tot[0];
            break;
        case FIN_SS:
            sc[SC_SS] = tot[0];
            if (!isfinite(tot[0]) || !isfinite(sc[SC_ALPHA])) {
                sc[SC_STOP] = STOP_BREAK_HALF;
            } else if (sqrt(tot[0]) <= tol) {
                sc[SC_STOP] = STOP_HALF_PENDING;
            }
            break;
        case FIN_OMEGA: {  // (AMs.s, AMs.AMs); a breakdown leaves omega = 0 so that x stays finite
            const double w = tot[0] / tot[1];
            sc[SC_OMEGA] = isfinite(w) ? w : 0.0;
            break;
        }
        case FIN_BETA: {  // (rs.r, r.r)
            sc[SC_BETA] = (tot[0] / sc[SC_RHO]) * (sc[SC_ALPHA] / sc[SC_OMEGA]);
            sc[SC_RHO] = tot[0];
            sc[SC_RR] = tot[1];
            sc[SC_ITS] = sc[SC_ITS] + 1.0;
            const double rn = sqrt(tot[1]);
            if (rn <= tol)
                sc[SC_STOP] = STOP_CONVERGED;
            else if (sc[SC_OMEGA] == 0.0 || sc[SC_RHO] == 0.0 || !isfinite(sc[SC_BETA]) || !isfinite(rn))
                sc[SC_STOP] = STOP_BREAK_FULL;
            else if (sc[SC_ITS] >= (double)maxit)
                sc[SC_STOP] = STOP_MAXIT;
            break;
        }
    }
}

// sum the partial groups and update the recurrence scalars (one block): of a (re)start, or, where
// the next launches have to know whether the half step ended the solve, FIN_SS
__global__ void __launch_bounds__(1024) k_bicg_finish(int op, FinArgs f, double rtol) {
    double *sc = f.sc;
    const double stopv = op == FIN_SS ? sc[sc_stop(f.par)] : 0.0;
    double tot[2] = {0, 0};
    finish_sums<2, 1024>(f, tot);
    if (threadIdx.x != 0) return;
    if (op == FIN_SS) {
        if (stopv != 0.0) sc[SC_STOPS] = stopv;  // what the second half reads
        else fin_ss(tot, sc, true);
        return;
    }
    sc[SC_RR] = tot[0];  // (r.r, b.b)
    sc[SC_RHO] = tot[0];
    sc[SC_STOPS] = 0.0;
    sc[SC_STOP] = 0.0;
    if (op == FIN_INIT) {
        sc[SC_BB] = tot[1];
        sc[SC_D0] = tot[0];
        sc[SC_ITS] = 0.0;
        sc[SC_TOL] = rtol * sqrt(tot[1]);
        if (sqrt(tot[0]) <= sc[SC_TOL]) sc[SC_STOP] = STOP_CONVERGED;
    }
}

void launch_bicg_finish(int op, const FinArgs &f, hipStream_t s, double rtol) {
    hipLaunchKernelGGL(k_bicg_finish, dim3(1), dim3(1024), 0, s, op, f, rtol);
    CUIBM_LAUNCH_CHECK();
}

// z = dinv * r (Jacobi)
__global__ void k_jacobi_apply(int n, const double *__restrict__ dinv, const double *__restrict__ r,
                               double *__restrict__ z, const double *__restrict__ stop) {
    const double stopv = stop ? *stop : 0.0;  // read at once, tested after the first loads
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const double v = dinv[i] * r[i];
        if (stopv != 0.0) return;
        z[i] = v;
    }
}

void launch_jacobi_apply(int n, const double *dinv, const double *r, double *z, hipStream_t s, const double *stop) {
    hipLaunchKernelGGL(k_jacobi_apply, dim3(grid_for(n)), dim3(BS), 0, s, n, dinv, r, z, stop);
    CUIBM_LAUNCH_CHECK();
}

// dinv = 1 / (sum of the diagonal entries of each row)
__global__ void k_diag_inv(int n, const int *__restrict__ rp, const int *__restrict__ ci, const double *__restrict__ v,
                           double *__restrict__ dinv) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        double d = 0;
        for (int k = rp[i]; k < rp[i + 1]; k++)
            if (ci[k] == i) d += v[k];
        dinv[i] = 1.0 / d;
    }
}

void launch_diag_inv(const DCsr<double> &A, double *dinv, hipStream_t s) {
    hipLaunchKernelGGL(k_diag_inv, dim3(grid_for(A.n)), dim3(BS), 0, s, A.n, A.rp.p(), A.ci.p(), A.v.p(), dinv);
    CUIBM_LAUNCH_CHECK();
}

// ---- lockstep batches: BiCGSTAB vector updates with per-case scalars ----
// Each block belongs to one case, so a stopped case's blocks return before any barrier.

struct BSeg {
    double *sc;
    long off;
    int n;
};
__device__ __forceinline__ BSeg bseg(int op, const BCase &C) {
    return op == BOP_VEL ? BSeg{C.scV, C.offUV, C.numUV} : BSeg{C.scP, C.offP, C.numP};
}

__global__ void __launch_bounds__(BS) k_b_bicg_s(int op, const BCase *__restrict__ tab, BMapDev m,
                                                 const double *__restrict__ r, const double *__restrict__ AMp,
                                                 double *__restrict__ s, double *__restrict__ part,
                                                 double *__restrict__ wpart) {
    const BCase &C = tab[m.cs[blockIdx.x]];
    const BSeg g = bseg(op, C);
    if (g.sc[SC_STOP] != 0.0) return;
    const double alpha = g.sc[SC_ALPHA];
    const int i = m.loc[blockIdx.x] * BS + threadIdx.x;
    double acc[2] = {0, 0};
    if (i < g.n) {
        const double si = r[g.off + i] - alpha * AMp[g.off + i];
        s[g.off + i] = si;
        acc[0] = si * si;
        if (wpart) acc[1] = (C.g.dx[i % C.g.nx] * C.g.dy[i / C.g.nx]) * si;
    }
    block_sum<2>(acc);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = acc[0];
        if (wpart) wpart[blockIdx.x] = acc[1];
    }
}

__global__ void __launch_bounds__(BS) k_b_bicg_xr(int op, const BCase *__restrict__ tab, BMapDev m,
                                                  double *__restrict__ x, const double *__restrict__ Mp,
                                                  const double *__restrict__ Ms, double *__restrict__ r,
                                                  const double *__restrict__ s, const double *__restrict__ AMs,
                                                  const double *__restrict__ rs, double *__restrict__ part) {
    const BSeg g = bseg(op, tab[m.cs[blockIdx.x]]);
    const double stopv = g.sc[SC_STOP];
    const bool half = stopv == STOP_HALF_PENDING;
    if (stopv != 0.0 && !half) return;
    const double alpha = g.sc[SC_ALPHA], omega = g.sc[SC_OMEGA];
    const int i = m.loc[blockIdx.x] * BS + threadIdx.x;
    double acc[2] = {0, 0};
    if (i < g.n) {
        const long j = g.off + i;
        const double xh = x[j] + alpha * Mp[j];
        if (half) {
            x[j] = xh;
        } else {
            const double ri = s[j] - omega * AMs[j];
            x[j] = xh + omega * Ms[j];
            r[j] = ri;
            acc[0] = rs[j] * ri;
            acc[1] = ri * ri;
        }
    }
    if (half) return;  // uniform per block
    block_sum<2>(acc);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = acc[0];
        part[m.nblk + blockIdx.x] = acc[1];
    }
}

__global__ void __launch_bounds__(BS) k_b_bicg_p(int op, const BCase *__restrict__ tab, BMapDev m,
                                                 double *__restrict__ p, const double *__restrict__ r,
                                                 const double *__restrict__ AMp, double *__restrict__ wpart) {
    const BCase &C = tab[m.cs[blockIdx.x]];
    const BSeg g = bseg(op, C);
    if (g.sc[SC_STOP] != 0.0) return;
    const double beta = g.sc[SC_BETA], omega = g.sc[SC_OMEGA];
    const int i = m.loc[blockIdx.x] * BS + threadIdx.x;
    double acc[1] = {0};
    if (i < g.n) {
        const long j = g.off + i;
        const double v = r[j] + beta * p[j] - beta * omega * AMp[j];
        p[j] = v;
        if (wpart) acc[0] = (C.g.dx[i % C.g.nx] * C.g.dy[i / C.g.nx]) * v;
    }
    if (!wpart) return;  // uniform
    block_sum<1>(acc);
    if (threadIdx.x == 0) wpart[blockIdx.x] = acc[0];
}

// one block per case: the case's block partials in a fixed order, then finish_update
__global__ void __launch_bounds__(BS) k_b_finish(int op, const BCase *__restrict__ tab, const int *__restrict__ first,
                                                 int nblk, const double *__restrict__ part, int fin, double rtol,
                                                 int maxit, const int *__restrict__ mask) {
    const int c = blockIdx.x;
    if (mask && !mask[c]) return;  // uniform per block
    double *sc = bseg(op, tab[c]).sc;
    if (fin == FIN_BETA && sc[SC_STOP] == STOP_HALF_PENDING) {  // the half-step update is done
        if (threadIdx.x == 0) sc[SC_STOP] = STOP_HALF;
        return;
    }
    if (fin != FIN_INIT && sc[SC_STOP] != 0.0) return;  // uniform per block
    const int ng = (fin == FIN_ALPHA || fin == FIN_SS) ? 1 : 2;  // FIN_RESTART: (r.r, b.b)
    const int b0 = first[c], b1 = first[c + 1];
    double v[2] = {0, 0};
    for (int g = 0; g < ng; g++)
        for (int k = b0 + (int)threadIdx.x; k < b1; k += BS) v[g] += part[g * nblk + k];
    block_sum<2>(v);
    if (threadIdx.x != 0) return;
    const double tot[2] = {v[0], v[1]};
    if (fin == FIN_INIT) {
        sc[SC_ITS] = 0.0;
        finish_update(fin, tot, sc, 0.0, maxit);
        sc[SC_TOL] = rtol * sqrt(sc[SC_BB]);
        if (sqrt(sc[SC_RR]) <= sc[SC_TOL]) sc[SC_STOP] = STOP_CONVERGED;  // converged at the start
    } else if (fin == FIN_RESTART) {  // new recurrences from the true residual
        sc[SC_RR] = tot[0];
        sc[SC_RHO] = tot[0];
        if (sqrt(tot[0]) <= sc[SC_TOL]) sc[SC_STOP] = STOP_CONVERGED;
    } else {
        finish_update(fin, tot, sc, sc[SC_TOL], maxit);
    }
}

void launch_b_bicg_s(int op, const BCase *tab, const BMapDev &m, const double *r, const double *AMp, double *s_,
                     double *part, double *wpart, hipStream_t s) {
    hipLaunchKernelGGL(k_b_bicg_s, dim3(m.nblk), dim3(BS), 0, s, op, tab, m, r, AMp, s_, part, wpart);
    CUIBM_LAUNCH_CHECK();
}

void launch_b_bicg_xr(int op, const BCase *tab, const BMapDev &m, double *x, const double *Mp, const double *Ms,
                      double *r, const double *s_, const double *AMs, const double *rs, double *part,
                      hipStream_t s) {
    hipLaunchKernelGGL(k_b_bicg_xr, dim3(m.nblk), dim3(BS), 0, s, op, tab, m, x, Mp, Ms, r, s_, AMs, rs, part);
    CUIBM_LAUNCH_CHECK();
}

void launch_b_bicg_p(int op, const BCase *tab, const BMapDev &m, double *p, const double *r, const double *AMp,
                     double *wpart, hipStream_t s) {
    hipLaunchKernelGGL(k_b_bicg_p, dim3(m.nblk), dim3(BS), 0, s, op, tab, m, p, r, AMp, wpart);
    CUIBM_LAUNCH_CHECK();
}

void launch_b_finish(int op, const BCase *tab, int ncases, const int *first, int nblk, const double *part, int fin,
                     double rtol, int maxit, hipStream_t s, const int *mask) {
    hipLaunchKernelGGL(k_b_finish, dim3(ncases), dim3(BS), 0, s, op, tab, first, nblk, part, fin, rtol, maxit, mask);
    CUIBM_LAUNCH_CHECK();
}

void launch_b_jacobi(long n, const double *dinv, const double *r, double *z, hipStream_t s) {
    hipLaunchKernelGGL(k_jacobi_apply, dim3(grid_for(n)), dim3(BS), 0, s, (int)n, dinv, r, z, nullptr);
    CUIBM_LAUNCH_CHECK();
}

}  // namespace cuibm

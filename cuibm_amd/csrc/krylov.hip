// Preconditioned BiCGSTAB replacing cusp::krylov::bicgstab + cusp::monitor
// (call sites NavierStokesSolver.cu:227-228 and :256-257 under src/solvers/NavierStokes/).
//
// Right-preconditioned BiCGSTAB (van der Vorst 1992) with the monitor rule
// ||r||_2 <= rtol ||b||_2 checked on r before every iteration and on s half-way
// through it; the iteration count counts full iterations. The recurrence scalars
// (rho, alpha, omega, beta) never leave the GPU: reductions finish in the kernel that needs
// the result, or in a one-block kernel, and update them in place; the stopping tests run
// there too, and the host reads the scalar block back once per batch of queued iterations.
//
// Breakdown (alpha or ||s|| not finite, omega = 0, rho = 0, beta not finite) restarts
// the recurrence from the true residual b - A x of the current iterate, keeping the
// iteration count; x never takes a non-finite update (omega falls back to 0). This
// never triggers in a run whose recurrence stays finite, so such runs follow the
// textbook iteration exactly; it matters for preconditioners that are not exactly
// linear (FP32 storage), where a breakdown would otherwise spin to maxit on NaN.
#include <cmath>

#include "krylov.hpp"

namespace cuibm {

JacobiPrecond::JacobiPrecond(const DCsr<double> &A, hipStream_t s) : n_(A.n) {
    own_.alloc(A.n);
    dinv_ = own_.p();
    launch_diag_inv(A, dinv_, s);
}

JacobiPrecond::JacobiPrecond(const DCsr<double> &A, double *dinv, hipStream_t s) : n_(A.n), dinv_(dinv) {
    launch_diag_inv(A, dinv_, s);
}

void JacobiPrecond::refresh(const DCsr<double> &A, hipStream_t s) {
    if (A.n != n_) throw Error("Jacobi refresh: matrix size changed", ERR_ARGUMENT);
    launch_diag_inv(A, dinv_, s);
}

void JacobiPrecond::apply(const double *r, double *z, hipStream_t s) {
    launch_jacobi_apply(n_, dinv_, r, z, s, stop_);
}

Bicgstab::Bicgstab(int n) : n_(n) {
    own_.alloc(workspace_doubles(n));
    double *ws = own_.p();
    const size_t st = stride(n);
    for (double **a : {&r_, &rs_, &p_, &Mp_, &AMp_, &s_, &Ms_, &AMs_}) {
        *a = ws;
        ws += st;
    }
    part_ = ws;
    sc_ = ws + 4 * (size_t)red_parts(n);
    CUIBM_HIP(hipHostMalloc((void **)&host_sc_, SC_COUNT * sizeof(double), hipHostMallocDefault));
    pinned_ = true;
}

Bicgstab::Bicgstab(int n, double *ws, double *host_sc) : n_(n), host_sc_(host_sc) {
    const size_t st = stride(n);
    for (double **a : {&r_, &rs_, &p_, &Mp_, &AMp_, &s_, &Ms_, &AMs_}) {
        *a = ws;
        ws += st;
    }
    part_ = ws;
    sc_ = ws + 4 * (size_t)red_parts(n);
}

Bicgstab::~Bicgstab() {
    if (pinned_ && host_sc_) (void)hipHostFree(host_sc_);
}

SolveStat Bicgstab::solve(const LinOp &A, double *x, const double *b, Preconditioner &M, double rtol,
                          int maxit, hipStream_t s) {
    if (A.n() != n_) throw Error("BiCGSTAB workspace size mismatch", ERR_ARGUMENT);
    const int n = n_, np = red_parts(n);
    // a reduction is finished by the kernel that uses it (FinArgs), from the half of the partials
    // that this kernel does not write
    double *sc = sc_, *part0 = part_, *part1 = part_ + 2 * (size_t)np;
    const double *diag = M.diagonal();
    int par = 0;  // parity of the iteration since the last (re)start
    auto args = [&](const double *part) { return FinArgs{part, np, sc, par, maxit}; };
    SolveStat st;
    auto fetch = [&]() {  // the scalar block: one small copy, one sync
        CUIBM_HIP(hipMemcpyAsync(host_sc_, sc, SC_COUNT * sizeof(double), hipMemcpyDeviceToHost, s));
        CUIBM_HIP(hipStreamSynchronize(s));
    };
    auto start = [&](int op) {  // r = b - A x, rs = p = r; clears the stop codes
        par = 0;
        A.init(x, b, r_, p_, rs_, part0, s);
        launch_bicg_finish(op, args(part0), s, rtol);
    };
    // the first half of iteration k (through s, and the test on ||s|| if `test`), then the second
    // half. A preconditioner that forms weighted sums of its input gets them from the kernels
    // that produce s and p (for the p of a (re)start, it forms them itself).
    const InputWeights iw = M.input_weights();
    const InputWeights *wp = iw.part ? &iw : nullptr;
    bool p_weighted = false;
    auto half1 = [&](bool test) {
        const double *stop = sc + sc_stop(par);
        A.set_stop(stop);
        M.set_stop(stop);
        if (diag) {
            A.spmv_dot_jacobi(diag, p_, Mp_, AMp_, rs_, false, FinArgs{}, part0, s);
        } else {
            if (wp && p_weighted) M.apply_weighted(p_, Mp_, s);
            else M.apply(p_, Mp_, s);
            A.spmv_dot(Mp_, AMp_, rs_, false, part0, s);
        }
        launch_bicg_s(n, r_, AMp_, s_, args(part0), part1, s, wp);
        if (test) launch_bicg_finish(FIN_SS, args(part1), s);
    };
    auto half2 = [&](bool tested) {
        const double *stop = sc + (tested ? (int)SC_STOPS : sc_stop(par));  // FIN_SS hands the other on
        A.set_stop(stop);
        M.set_stop(stop);
        if (diag) {
            A.spmv_dot_jacobi(diag, s_, Ms_, AMs_, s_, true, tested ? FinArgs{} : args(part1), part0, s);
        } else {
            if (wp) M.apply_weighted(s_, Ms_, s);
            else M.apply(s_, Ms_, s);
            A.spmv_dot(Ms_, AMs_, s_, true, part0, s);
        }
        launch_bicg_xr(n, x, Mp_, Ms_, r_, s_, AMs_, rs_, args(part0), part1, s);
        launch_bicg_p(n, p_, r_, AMp_, args(part1), s, wp);
        p_weighted = wp != nullptr;
        par ^= 1;
    };
    const bool test_early = !diag;  // ||s|| is tested before the second half (else in its product)
    start(FIN_INIT);
    double tol = 0, rn = 0, rn0 = 0, rn_ref = 0;
    // with an earlier solve to go by, iterations are queued before the first read-back
    bool known = false;
    auto first_known = [&]() {
        tol = host_sc_[SC_TOL];
        rn0 = rn_ref = std::sqrt(host_sc_[SC_D0]);
        known = true;
    };
    if (exact_ || last_its_ < 0 || maxit <= 0) {
        fetch();
        first_known();
        rn = rn0;
    }
    int it = 0, restarts = 0;
    // The recurrence residual r can drift from b - A x through rounding when a solve runs
    // many iterations with large updates (seen with the FP32 V-cycle at tolerances near
    // 1e-12: after thousands of iterations r claimed 5e-11 of ||b|| while b - A x was
    // larger than b). A solve that converged after kVerifyIts iterations or a restart
    // therefore forms b - A x once; more than kDriftFactor times the tolerance restarts
    // the iteration from it (counted as a restart), at most kMaxChecks times.
    int checks = 0;
    const double reliable = M.restart_reduction();  // rn_ref: the true residual at the last (re)start
    auto restart = [&]() {
        start(FIN_RESTART);
        fetch();
        p_weighted = false;
        return std::sqrt(host_sc_[SC_RR]);
    };
    for (;;) {
        while (!known || (!(rn <= tol) && it < maxit)) {
            // iterations to queue before the next read-back: a fraction of the estimate from
            // the residual reduction so far (or of the last solve), so that few launches
            // fall past the end; one in exact mode
            int batch = 1;
            // a solve that will likely leave at its first half step is read back there
            const bool stepwise = exact_ || (!known && last_its_ == 0);
            if (!exact_) {
                double left = 0;
                if (!known) {
                    left = last_its_;
                } else {
                    double rate = rate_;
                    if (it > 0 && rn < rn0) rate = std::pow(rn / rn0, 1.0 / it);
                    if (rate > 0 && rate < 1) left = std::log(tol / rn) / std::log(rate);
                }
                batch = (int)std::max(1.0, std::min(16.0, std::floor(0.7 * left)));
                batch = std::min(batch, maxit - it);
            }
            int code = 0;
            for (int j = 0; j < batch; j++) {
                half1(test_early || stepwise);
                if (stepwise) {  // no launch past a half-step exit or breakdown
                    fetch();
                    const int h = (int)host_sc_[SC_STOPS], c = (int)host_sc_[sc_stop(par)];
                    if (c == 0 && h == STOP_HALF_PENDING) {  // the half-step update alone
                        launch_bicg_xr(n, x, Mp_, Ms_, r_, s_, AMs_, rs_, args(part0), part1, s);
                        code = STOP_HALF;
                    } else if (c != 0 || h != 0) {
                        code = c != 0 ? c : h;
                    }
                    if (code != 0) break;
                }
                half2(test_early || stepwise);
            }
            if (code == 0) {
                fetch();
                code = (int)host_sc_[sc_stop(par)];
            }
            if (!known) first_known();
            it = (int)host_sc_[SC_ITS];
            if (code == STOP_HALF) {
                rn = std::sqrt(host_sc_[SC_SS]);
                break;
            }
            rn = std::sqrt(host_sc_[SC_RR]);
            if (code == STOP_BREAK_HALF || code == STOP_BREAK_FULL) {
                if (++restarts > kMaxRestarts) break;
                rn = rn_ref = restart();  // x is untouched by a half-step breakdown
            } else if (reliable > 0 && code == 0 && rn < reliable * rn_ref) {
                if (++restarts > kMaxRestarts) break;
                rn = rn_ref = restart();  // reliable update: the true residual, new search directions
            }
        }
        if (!(rn <= tol) || (it < kVerifyIts && restarts == 0) || checks >= kMaxChecks) break;
        checks++;
        const double tr = restart();
        if (tr <= kDriftFactor * tol) break;
        rn = rn_ref = tr;
        if (++restarts > kMaxRestarts) break;
    }
    if (it > 0 && rn > 0 && rn0 > 0 && rn < rn0) rate_ = std::pow(rn / rn0, 1.0 / it);
    last_its_ = it;
    A.set_stop(nullptr);
    M.set_stop(nullptr);
    st.restarts = restarts;
    st.iterations = it;
    st.residual = rn;
    st.tolerance = tol;
    st.converged = rn <= tol;
    return st;
}

}  // namespace cuibm

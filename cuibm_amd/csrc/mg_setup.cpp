// Host set-up of the tensor multigrid (mg.hpp): the grid's levels, the 1-D couplings and the
// 1-D eigenvectors of the directly solved level.
#include <algorithm>
#include <cmath>

#include "mg.hpp"

namespace cuibm {

namespace {

// aggregate of each cell: a cell and its successor merge while their joint width is at most t
std::vector<int> merge_pairs(const std::vector<double> &w, double t) {
    std::vector<int> a(w.size());
    int k = 0;
    for (size_t j = 0; j < w.size(); k++) {
        a[j] = k;
        if (j + 1 < w.size() && w[j] + w[j + 1] <= t * (1 + 1e-7)) a[++j] = k;
        j++;
    }
    return a;
}

std::vector<double> merged(const std::vector<double> &w, const std::vector<int> &a) {
    std::vector<double> c(a.back() + 1, 0.0);
    for (size_t j = 0; j < w.size(); j++) c[a[j]] += w[j];
    return c;
}

std::vector<double> centres(const std::vector<double> &w) {
    std::vector<double> x(w.size());
    double s = 0;
    for (size_t j = 0; j < w.size(); j++) {
        x[j] = s + 0.5 * w[j];
        s += w[j];
    }
    return x;
}

// linear interpolation at the fine centres between aggregate centres: value (1 - t) e[a] + t e[o]
void interpolation(const std::vector<double> &w, const std::vector<int> &a, const std::vector<double> &wc,
                   std::vector<int> &o, std::vector<double> &t) {
    const std::vector<double> x = centres(w), xc = centres(wc);
    const int nc = (int)wc.size();
    o.resize(w.size());
    t.resize(w.size());
    for (size_t j = 0; j < w.size(); j++) {
        const int k = a[j];
        o[j] = x[j] >= xc[k] ? std::min(k + 1, nc - 1) : std::max(k - 1, 0);
        t[j] = o[j] == k ? 0.0 : std::fabs(x[j] - xc[k]) / std::fabs(xc[o[j]] - xc[k]);
    }
}

}  // namespace

std::vector<MgHostLevel> mg_levels(const std::vector<double> &dx, const std::vector<double> &dy, int cap, long most) {
    std::vector<MgHostLevel> lv(1);
    lv[0].dx = dx;
    lv[0].dy = dy;
    for (;;) {
        MgHostLevel &L = lv.back();
        const size_t nx = L.dx.size(), ny = L.dy.size();
        if (nx <= (size_t)cap && ny <= (size_t)cap && (most <= 0 || (long)(nx * ny) <= most)) return lv;
        // at least a quarter of the cells go at every level
        double t = MG_WIDTH * std::min(*std::min_element(L.dx.begin(), L.dx.end()),
                                       *std::min_element(L.dy.begin(), L.dy.end()));
        for (;; t *= 1.1) {
            L.ax = merge_pairs(L.dx, t);
            L.ay = merge_pairs(L.dy, t);
            if ((double)(L.ax.back() + 1) * (L.ay.back() + 1) <= 0.75 * (double)nx * (double)ny) break;
        }
        MgHostLevel C;
        C.dx = merged(L.dx, L.ax);
        C.dy = merged(L.dy, L.ay);
        interpolation(L.dx, L.ax, C.dx, L.ox, L.tx);
        interpolation(L.dy, L.ay, C.dy, L.oy, L.ty);
        lv.push_back(std::move(C));
    }
}

bool mg_axis(const std::vector<double> &w) {
    return !w.empty() && std::all_of(w.begin(), w.end(), [&](double v) {
        return std::isfinite(v) && v != 0 && std::signbit(v) == std::signbit(w[0]);
    });
}

void axis_couplings(const std::vector<double> &w, double dt, std::vector<double> &next, std::vector<double> &prev) {
    const size_t n = w.size();
    next.assign(n, 0.0);
    prev.assign(n, 0.0);
    for (size_t j = 0; j + 1 < n; j++) {
        next[j] = dt / (w[j] * (w[j] + w[j + 1]) * 0.5);
        prev[j + 1] = dt / (w[j + 1] * (w[j + 1] + w[j]) * 0.5);
    }
}

// Implicitly shifted QR with Wilkinson's shift (Golub & Van Loan, Matrix Computations, 8.3):
// each sweep chases a bulge down the unreduced block with Givens rotations, which are
// accumulated into the rows of q.
void tridiagonal_eigen(std::vector<double> d, std::vector<double> e, std::vector<double> &lam, std::vector<double> &q) {
    const int n = (int)d.size();
    q.assign((size_t)n * n, 0.0);
    for (int i = 0; i < n; i++) q[(size_t)i * n + i] = 1.0;
    auto small = [&](int k) { return std::fabs(e[k]) <= 1e-16 * (std::fabs(d[k]) + std::fabs(d[k + 1])); };
    int hi = n - 1;
    for (long sweeps = 0; hi > 0;) {
        if (small(hi - 1)) {
            e[hi - 1] = 0;
            hi--;
            continue;
        }
        if (++sweeps > 60L * n) throw Error("tridiagonal eigenproblem did not converge", ERR_GENERIC);
        int lo = hi - 1;
        while (lo > 0 && !small(lo - 1)) lo--;
        if (lo > 0) e[lo - 1] = 0;
        const double h = 0.5 * (d[hi - 1] - d[hi]), b2 = e[hi - 1] * e[hi - 1];
        const double shift = d[hi] - b2 / (h + std::copysign(std::hypot(h, e[hi - 1]), h));
        double x = d[lo] - shift, z = e[lo];
        for (int k = lo; k < hi; k++) {
            const double r = std::hypot(x, z), c = r > 0 ? x / r : 1.0, s = r > 0 ? z / r : 0.0;
            if (k > lo) e[k - 1] = r;
            const double p = d[k], m = e[k], u = d[k + 1];
            d[k] = c * c * p + 2 * c * s * m + s * s * u;
            d[k + 1] = s * s * p - 2 * c * s * m + c * c * u;
            e[k] = c * s * (u - p) + (c * c - s * s) * m;
            if (k + 1 < hi) {
                x = e[k];
                z = s * e[k + 1];
                e[k + 1] = c * e[k + 1];
            }
            double *qa = &q[(size_t)k * n], *qb = qa + n;
            for (int i = 0; i < n; i++) {
                const double va = qa[i], vb = qb[i];
                qa[i] = c * va + s * vb;
                qb[i] = c * vb - s * va;
            }
        }
    }
    lam = std::move(d);
}

AxisModes axis_modes(const std::vector<double> &w, double dt) {
    AxisModes M;
    const int n = M.n = (int)w.size(), p = M.pad = (n + 15) / 16 * 16;
    std::vector<double> next, prev, d(n), e(std::max(n - 1, 0)), q;
    axis_couplings(w, dt, next, prev);
    for (int i = 0; i < n; i++) d[i] = next[i] + prev[i];
    for (int i = 0; i + 1 < n; i++) e[i] = -std::sqrt(next[i] * prev[i + 1]);
    tridiagonal_eigen(d, e, M.lam, q);
    M.zero = (int)(std::min_element(M.lam.begin(), M.lam.end()) - M.lam.begin());
    M.F.assign((size_t)p * p, 0.0);
    M.B.assign((size_t)p * p, 0.0);
    for (int k = 0; k < n; k++)
        for (int i = 0; i < n; i++) {
            const double r = std::sqrt(w[i]), v = q[(size_t)k * n + i];
            M.F[(size_t)k * p + i] = v * r;
            M.B[(size_t)i * p + k] = v / r;
        }
    M.lam.resize(p, 1.0);
    return M;
}

}  // namespace cuibm

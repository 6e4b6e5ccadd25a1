"""One BiCGSTAB iteration with the multigrid levels (mg.hip) against the same iteration on the
host, whose cycle is written from the description of the levels (mg.hpp) with numpy: the grids by
cell width, three sweeps down and up, volume averages, linear interpolation, the pseudo-inverse
of the coarsest level and the constant mode around it. A weight, neighbour or aggregate that is
wrong anywhere on the grid changes the iterate, whatever it does to the rate of convergence.

Bar: the iterate is mostly the lowest modes, whose coefficients on the directly solved level of N
cells are 1/sqrt(N) of a random right-hand side, formed by sums whose rounding is a few units of the
level's precision of the whole: 16 eps sqrt(N). Both sides' eigenvalues are off by a few FP64 eps
of the largest, which the lowest nonzero one divides: 16 eps64 max(lambda) / min(lambda) of the
axes. (The reciprocal of a diagonal is a sweep's weight: 1e-14 of it at most in FP64 levels.)"""
import math

import numpy as np
import pytest
import scipy.linalg
import scipy.sparse as sp

import cuibm_amd
from helpers import rel_l2
from test_gpu_mg import write_case

pytestmark = pytest.mark.gpu

SWEEPS = [1.0 / (1.1 + 0.9 * math.cos(math.pi * (2 * k + 1) / 6)) for k in range(3)]  # on [0.2, 2]


def pairs(w, t):
    a, j = [], 0
    while j < len(w):
        a.append(a[-1] + 1 if a else 0)
        if j + 1 < len(w) and w[j] + w[j + 1] <= t * (1 + 1e-7):
            a.append(a[-1])
            j += 1
        j += 1
    return np.array(a)


class Axis:
    def __init__(self, w, dt):
        n = len(w)
        self.w = w
        self.up, self.dn = np.zeros(n), np.zeros(n)  # couplings to the next and the previous cell
        self.up[:-1] = dt / (w[:-1] * (w[:-1] + w[1:]) * 0.5)
        self.dn[1:] = dt / (w[1:] * (w[1:] + w[:-1]) * 0.5)

    def coarsen(self, a):
        self.agg = a
        wc = np.bincount(a, self.w)
        centre, cc = np.cumsum(self.w) - 0.5 * self.w, np.cumsum(wc) - 0.5 * wc
        n, m = len(a), len(wc)
        R, P = np.zeros((m, n)), np.zeros((n, m))
        for j in range(n):
            R[a[j], j] = self.w[j] / wc[a[j]]
            o = min(a[j] + 1, m - 1) if centre[j] >= cc[a[j]] else max(a[j] - 1, 0)
            t = 0.0 if o == a[j] else abs(centre[j] - cc[a[j]]) / abs(cc[o] - cc[a[j]])
            P[j, a[j]] += 1 - t
            P[j, o] += t
        self.R, self.P = sp.csr_matrix(R), sp.csr_matrix(P)
        return wc

    def modes(self):
        d, e = self.up + self.dn, -np.sqrt(self.up[:-1] * self.dn[1:])
        lam, q = scipy.linalg.eigh_tridiagonal(d, e) if len(d) > 1 else (np.zeros(1), np.ones((1, 1)))
        r = np.sqrt(self.w)
        return lam, q.T * r, q / r[:, None]


class Level:
    def __init__(self, dx, dy, dt):
        self.x, self.y = Axis(dx, dt), Axis(dy, dt)
        self.d = (self.x.up + self.x.dn)[None, :] + (self.y.up + self.y.dn)[:, None]

    def apply(self, v):
        s = self.d * v
        s[:, :-1] -= self.x.up[:-1] * v[:, 1:]
        s[:, 1:] -= self.x.dn[1:] * v[:, :-1]
        s[:-1] -= self.y.up[:-1, None] * v[1:]
        s[1:] -= self.y.dn[1:, None] * v[:-1]
        return s


def hierarchy(dx, dy, dt, most):
    levels = [Level(dx, dy, dt)]
    while max(len(dx), len(dy)) > 224 or (most and len(dx) * len(dy) > most):
        t = 6.0 * min(dx.min(), dy.min())
        while True:
            ax, ay = pairs(dx, t), pairs(dy, t)
            if (ax[-1] + 1) * (ay[-1] + 1) <= 0.75 * len(dx) * len(dy):
                break
            t *= 1.1
        dx, dy = levels[-1].x.coarsen(ax), levels[-1].y.coarsen(ay)
        levels.append(Level(dx, dy, dt))
    return levels


def cycle(levels, b):
    L = levels[0]
    if len(levels) == 1:
        (lx, fx, bx), (ly, fy, by) = L.x.modes(), L.y.modes()
        lam = ly[:, None] + lx[None, :]
        lam[0, 0] = np.inf  # the constant (both eigenvalues ascend from zero)
        return by @ ((fy @ b @ fx.T) / lam) @ bx.T
    v = np.zeros_like(b)
    for w in SWEEPS:
        v += w / L.d * (b - L.apply(v))
    r = b - L.apply(v)
    v += L.y.P @ cycle(levels[1:], L.y.R @ r @ L.x.R.T) @ L.x.P.T
    for w in SWEEPS[::-1]:
        v += w / L.d * (b - L.apply(v))
    return v


def first_iterate(A, M, b):
    p = M(b)
    q = A @ p
    alpha = (b @ b) / (b @ q)
    s = b - alpha * q
    t = M(s)
    u = A @ t
    return alpha * p + (u @ s) / (u @ u) * t


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("nx,ny,solver,h,ratio,most", [
    (342, 333, "NAVIER_STOKES_SOLVER", None, None, 0), (57 * 7, 58 * 6, "NAVIER_STOKES_SOLVER", None, None, 0),
    (9, 1200, "NAVIER_STOKES_SOLVER", None, None, 0), (130, 120, "NAVIER_STOKES_SOLVER", None, None, 400),
    (0, 0, "LUO", 0.012, 1.0137, 0), (0, 0, "LUO", 0.008, 1.035, 0), (0, 0, "LUO", 0.008, 1.035, 3000)])
def test_first_iterate(tmp_path, nx, ny, solver, h, ratio, most, precision):
    folder = write_case(tmp_path, nx, ny, solver, ratio, h)
    f = tmp_path / "simParams.yaml"
    f.write_text(f.read_text().replace("maxIterations: 200", "maxIterations: 1"))
    args = ["-amgCoarseMax", most] if most else []
    with cuibm_amd.Solver(folder, "-amgPrecision", precision, *args, diagnostics=False) as s:
        s.initialise()
        dx, dy = s.get("dx"), s.get("dy")
        nx, ny = len(dx), len(dy)
        A = sp.csr_matrix((s.get("LHS2_val"), s.get("LHS2_col"), s.get("LHS2_rowptr")), shape=(nx * ny, nx * ny))
        levels = hierarchy(dx, dy, 0.01, most)
        assert s.info()["amg_levels"] == len(levels) > 1
        b = np.random.default_rng(3).standard_normal(nx * ny)
        s.set("rhs2", b)
        s.set("p", np.zeros(nx * ny))
        with pytest.raises(cuibm_amd.CuibmError) as e:
            s.phase("solvePoisson")
        assert e.value.code == -4  # not converged after the one iteration
        p = s.get("p")

    a = A @ np.ones(nx * ny)
    a[np.abs(a) < 0.1 * A.diagonal()] = 0.0  # nonzero at the pinned cells alone
    area = np.outer(dy, dx).ravel()

    def M(r):
        c = (area @ r) / (area @ a)
        return cycle(levels, (r - c * a).reshape(ny, nx)).ravel() + c

    d = rel_l2(p, first_iterate(A, M, b))
    N = levels[-1].d.size
    lam = [ax.modes()[0] for ax in (levels[-1].x, levels[-1].y)]
    spread = max(v[-1] for v in lam) / min(v[1] for v in lam if len(v) > 1)
    bar = 16 * (np.finfo(np.float64 if precision == 64 else np.float32).eps * math.sqrt(N)
                + np.finfo(np.float64).eps * spread)
    print(f"{nx} x {ny} precision {precision}: {len(levels)} levels, difference {d:.2e} (bar {bar:.2e})", flush=True)
    assert d <= bar

"""The work that users of this framework have it do, as cases to be timed.

Three families, all through the public entry points of ``cuibm_amd``:

- ``steps``: a solver of one case folder advances a given flow state by a few time steps and
  hands back the fields and the drag, as a program does that restarts a flow and saves it
  every few steps. The plain cavity, the Luo external, the modified Fadlun and the Luo
  embedded method, FP64 and mixed precision.
- ``whole``: whole calls that set themselves up and run: a body in prescribed motion (its
  hierarchy is set up again every step), an ensemble of cases in lockstep, the gradient of
  the mean drag by the discrete adjoint (forward and backward).
- ``csr``: BiCGSTAB with smoothed aggregation (or without) on a matrix of the caller's.

Grids go from 32 x 32 (launches and waits count) to 1024 x 1024 (memory counts); the sizes
are those of the package's own case folders, and odd and uneven ones beside them.
"""
import math
import os
import tempfile

import numpy as np

import cuibm_amd
from cuibm_amd import ensemble
from cuibm_amd.adjoint import RotatingCylinder, mean_drag

STATE = ("u", "uhat", "N", "p", "xp")  # what one time step leaves for the next


def listed():
    return [
        # the smallest run: a lid-driven cavity of the package; latency and launches alone
        {"name": "cavity32", "family": "steps", "folder": "lidDrivenCavityRe100_32", "nx": 32, "ny": 32, "steps": 10},
        # an ordinary cavity (the package's 128 x 128 validation case)
        {"name": "cavity128", "family": "steps", "folder": "lidDrivenCavityRe100_128", "nx": 128, "ny": 128,
         "steps": 10},
        # an odd, uneven cavity with cells that are not square
        {"name": "cavity301x173", "family": "steps", "kind": "plain", "nx": 301, "ny": 173, "steps": 10},
        # the Re = 40 cylinder (Luo external) at its configured tolerances, FP64
        {"name": "luo336", "family": "steps", "folder": "cylinderRe40_luo", "nx": 336, "ny": 336, "steps": 10},
        # the Re = 550 cylinder at 1024 x 1024 with the FP32 V-cycle, the benchmark's form
        {"name": "luo1024_mixed", "family": "steps", "folder": "cylinderRe550_1024_luo", "nx": 1024, "ny": 1024,
         "steps": 10, "precision": 32, "dt": 0.00125},
        # the same in FP64, the benchmark's other form
        {"name": "luo1024_fp64", "family": "steps", "folder": "cylinderRe550_1024_luo", "nx": 1024, "ny": 1024,
         "steps": 10, "precision": 64, "dt": 0.00125},
        # modified Fadlun at 890 x 890, one of the published whole runs (tolerance 1e-5)
        {"name": "fadlun890", "family": "steps", "folder": "cylinderRe40_890_fadlun", "nx": 890, "ny": 890,
         "steps": 20},
        # Luo embedded at 462 x 462, another of them: the body's rows are part of both matrices.
        # (At its configured 1e-5 two correct solves differ by percents in the pressure.)
        {"name": "embedded462", "family": "steps", "folder": "cylinderRe40_462_embedded", "nx": 462, "ny": 462,
         "steps": 10, "solve": 1e-7},
        # a cylinder oscillating in a stream, embedded: a whole short run, set-up and all, with
        # the matrices and the hierarchy set up again after every move
        {"name": "osc_embedded224", "family": "whole", "what": "moving", "folder": "oscFlowRe100_embedded",
         "cells": 224 * 224, "steps": 20, "solve": 1e-7},
        # an ensemble of impulsively started cylinders of uneven size, in lockstep
        {"name": "lockstep8", "family": "whole", "what": "ensemble", "cases": 8, "least": 160, "most": 300,
         "precision": 32, "steps": 50, "cells": 8 * 230 * 230},
        # the gradient of the mean drag at the size of the rotating-cylinder study
        {"name": "adjoint498", "family": "whole", "what": "adjoint", "folder": "rotatingCylinderRe100_luo",
         "cells": 498 * 498, "steps": 6, "every": 3},
        # a caller's own pressure matrix through the linear-algebra entry point
        {"name": "csr400x357", "family": "csr", "nx": 400, "ny": 357, "precond": "SMOOTHED_AGGREGATION",
         "precision": 64, "rtol": 1e-8},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    pick = rng.random()
    if pick < 0.25:  # cavities from the smallest up, uneven, either Poisson form
        nx, ny = int(_log(rng, 24, 600)), int(_log(rng, 24, 600))
        return {"family": "steps", "kind": "plain", "nx": nx, "ny": ny, "steps": rng.randint(4, 10),
                "precision": rng.choice([64, 64, 32])}
    if pick < 0.75:  # cylinders on stretched grids of about 90 to 1000 cells an edge
        kind = rng.choice(["luo", "luo", "luo", "fadlun", "embedded"])
        while True:
            h = _log(rng, 0.006, 0.06) if kind != "embedded" else _log(rng, 0.02, 0.06)
            ratio = round(rng.uniform(1.008, 1.04), 4)
            nx = ensemble.core_cells(h) + 2 * ensemble.cells_stretched(ratio, h, 14.4)
            if 90 <= nx <= 1000:
                break
        return {"family": "steps", "kind": kind, "h": h, "ratio": ratio, "nx": nx, "ny": nx,
                "steps": rng.randint(4, 10), "precision": rng.choice([64, 32]) if kind == "luo" else 64,
                "rtol": rng.choice([1e-8, 1e-9])}
    if pick < 0.82:
        least = rng.randint(160, 200)
        return {"family": "whole", "what": "ensemble", "cases": rng.randint(3, 8), "least": least,
                "most": least + rng.randint(20, 130), "precision": rng.choice([64, 32]),
                "steps": rng.randint(10, 40), "cells": 6 * (least + 60) ** 2}
    if pick < 0.9:
        while True:
            h, ratio = _log(rng, 0.015, 0.05), round(rng.uniform(1.015, 1.04), 4)
            nx = ensemble.core_cells(h) + 2 * ensemble.cells_stretched(ratio, h, 14.4)
            if 160 <= nx <= 360:
                break
        return {"family": "whole", "what": "adjoint", "kind": "luo", "h": h, "ratio": ratio, "cells": nx * nx,
                "steps": rng.randint(8, 12), "every": rng.randint(2, 6), "rtol": 1e-12}
    return {"family": "csr", "nx": int(_log(rng, 40, 500)), "ny": int(_log(rng, 40, 500)),
            "precond": rng.choice(["SMOOTHED_AGGREGATION", "SMOOTHED_AGGREGATION", "DIAGONAL"]),
            "precision": rng.choice([64, 32, 3264]), "rtol": 1e-8}


# ---- case folders -----------------------------------------------------------------------

SOLVERS = {"plain": "NAVIER_STOKES_SOLVER", "luo": "LUO", "fadlun": "FADLUN", "embedded": "OSC_CYLINDER"}


def _sides(x_plus, values):
    text = "  boundaryConditions:\n"
    for loc in ("xMinus", "xPlus", "yMinus", "yPlus"):
        kind = x_plus if loc == "xPlus" else "DIRICHLET"
        text += f"    - location: {loc}\n      u: [{kind}, {values[loc]}]\n      v: [{kind}, 0.0]\n"
    return text


def _write_folder(case, folder):
    """The four input files of a drawn case."""
    kind, rtol = case["kind"], case.get("rtol", 1e-8)
    if kind == "plain":
        # n cells of one size on [0, 1]: the grid rule takes int(1 / mid_h) of them
        axis = lambda name, n: (f"- direction: {name}\n  start: 0.0\n  mid_h: {1.0 / (n + 0.5)!r}\n  subDomains:\n"
                                "    - end: 1.0\n      stretchRatio: 1.0\n")
        domain = axis("x", case["nx"]) + "\n" + axis("y", case["ny"])
        flow = ("- type: flow\n  nu: 0.01\n  initialVelocity: [0.0, 0.0]\n"
                + _sides("DIRICHLET", {"xMinus": 0.0, "xPlus": 0.0, "yMinus": 0.0, "yPlus": 1.0}))
        dt = 0.3 / max(case["nx"], case["ny"])
    else:
        h, ratio = case["h"], case["ratio"]
        axis = lambda name, n: (f"- direction: {name}\n  start: -15.0\n  mid_h: {h!r}\n  subDomains:\n"
                                f"    - end: -0.6\n      stretchRatio: {ratio!r}\n"
                                "    - end: 0.6\n      stretchRatio: 1.0\n"
                                f"    - end: 15.0\n      stretchRatio: {ratio!r}\n")
        domain = axis("x", 0) + "\n" + axis("y", 0)
        flow = ("- type: flow\n  nu: 0.025\n  initialVelocity: [1.0, 0.0]\n"
                + _sides("CONVECTIVE", {"xMinus": 1.0, "xPlus": 1.0, "yMinus": 1.0, "yPlus": 1.0}))
        dt = (0.1 if kind != "luo" else 0.3) * h
        points = int(math.pi / h) // 2 * 2
        with open(os.path.join(folder, "bodies.yaml"), "w") as f:
            f.write(f"- type: circle\n  circleOptions: [0.0, 0.0, 0.5, {points}, false]\n")
    solve = lambda system, m: (f"    - system: {system}\n      solver: BICGSTAB\n      preconditioner: {m}\n"
                               f"      tolerance: {rtol}\n      maxIterations: 20000\n")
    sim = (f"- type: simulation\n  dt: {dt!r}\n  nt: 1000\n  nsave: 1000\n  scaleCV: 2.0\n"
           f"  SolverType: {SOLVERS[kind]}\n  linearSolvers:\n"
           + solve("velocity", "DIAGONAL") + solve("Poisson", "SMOOTHED_AGGREGATION"))
    for name, text in (("domain.yaml", domain), ("flow.yaml", flow), ("simParams.yaml", sim)):
        with open(os.path.join(folder, name), "w") as f:
            f.write(text)


def _perturbation(seed):
    r = np.random.default_rng(seed)
    return float(r.uniform(0.01, 0.05)), float(r.uniform(0.01, 0.05))


def _solver(case, folder, seed):
    """The case's solver, initialised from a perturbed field."""
    up, vp = _perturbation(seed)
    args = ["-uPerturb", up, "-vPerturb", vp]
    if "precision" in case:
        args += ["-amgPrecision", case["precision"]]
    if "solve" in case:
        args += ["-velocityTol", case["solve"], "-poissonTol", case["solve"]]
    if "dt" in case:
        args += ["-dt", case["dt"]]
    s = cuibm_amd.Solver(folder, *args, diagnostics=False)
    s.initialise()
    return s


class _Matrix:
    """What cuibm_amd.Csr asks of a matrix."""

    def __init__(self, n, indptr, indices, data):
        self.shape, self.indptr, self.indices, self.data = (n, n), indptr, indices, data

    def tocsr(self):
        return self

    def sort_indices(self):
        pass


def _widths(n, seed):
    """Cell widths of one axis: a finer core, as the stretched grids have."""
    r = np.random.default_rng(seed)
    t = np.linspace(-1.0, 1.0, n)
    w = 0.2 + t ** 2 * r.uniform(1.0, 3.0)
    return w / w.sum()


def _pressure_matrix(wx, wy):
    """Neumann Laplacian per cell volume on a stretched grid, cell 0's diagonal doubled."""
    nx, ny = wx.size, wy.size
    ex, ey = 2.0 / (wx[:-1] + wx[1:]), 2.0 / (wy[:-1] + wy[1:])
    cE, cW = np.append(ex, 0) / wx, np.append(0, ex) / wx
    cN, cS = np.append(ey, 0) / wy, np.append(0, ey) / wy
    I, J = np.tile(np.arange(nx), ny), np.repeat(np.arange(ny), nx)
    ip = J * nx + I
    diag = cE[I] + cW[I] + cN[J] + cS[J]
    diag[0] *= 2
    cols = np.stack([ip - nx, ip - 1, ip, ip + 1, ip + nx], 1)
    vals = np.stack([-cS[J], -cW[I], diag, -cE[I], -cN[J]], 1)
    keep = np.stack([J > 0, I > 0, I >= 0, I < nx - 1, J < ny - 1], 1)
    rp = np.concatenate([[0], np.cumsum(keep.sum(1))])
    return _Matrix(nx * ny, rp.astype(np.int32), cols[keep].astype(np.int32), vals[keep])


def prepare(case, seed):
    if case["family"] == "csr":
        wx, wy = _widths(case["nx"], seed), _widths(case["ny"], seed + 1)
        A = cuibm_amd.Csr(_pressure_matrix(wx, wy))
        b = np.random.default_rng(seed).standard_normal(A.n)
        if case["precond"] == "SMOOTHED_AGGREGATION":
            A.vcycle(b, case["precision"])  # lays out the hierarchy, which such a program keeps
        return {"case": case, "A": A, "b": b}
    st = {"case": case, "seed": seed}
    if case.get("what") == "ensemble":
        st["tmp"] = tempfile.TemporaryDirectory()
        st["folders"], _ = ensemble.write_cases(st["tmp"].name, n=case["cases"], seed=seed, steps=case["steps"],
                                                edges=(case["least"], case["most"]))
        return st
    if "folder" in case:
        folder = os.path.join(cuibm_amd.CASES, case["folder"])
    else:
        st["tmp"] = tempfile.TemporaryDirectory()
        folder = st["tmp"].name
        _write_folder(case, folder)
    if case.get("what") == "moving":
        return {**st, "folder": folder}
    if case.get("what") == "adjoint":
        k = case["steps"]
        st["problem"] = RotatingCylinder(folder, nsteps=k, n0=max(1, k // 2), n1=k, every=case["every"])
        st["blow"] = np.random.default_rng(seed).normal(0.0, 0.01, st["problem"].npts)
        return st
    s = _solver(case, folder, seed)
    if "bodies.yaml" in os.listdir(folder):
        s.step_time(3)  # past the first, impulsive steps
    st["solver"] = s
    st["fields"] = {n: s.get(n) for n in STATE}
    return st


def _flow(s):
    """Velocity and pressure; the pressure of an incompressible flow is known up to a constant
    (one raised diagonal entry pins it, weakly), so a program looks at it about its mean."""
    p = s.get("p")
    return {"u": s.get("u"), "p": p - p.mean()}


def run(state):
    case = state["case"]
    if case["family"] == "csr":
        x, its, resid, ok = state["A"].bicgstab(state["b"], precond=case["precond"], rtol=case["rtol"], maxit=20000,
                                                amg_precision=case["precision"])
        return {"x": x, "ok": ok}
    if case["family"] == "steps":
        s = state["solver"]
        for n, a in state["fields"].items():
            s.set(n, a)
        s.step_time(case["steps"])
        return _flow(s)
    if case["what"] == "moving":
        with _solver(case, state["folder"], state["seed"]) as s:
            s.step_time(case["steps"])
            return {**_flow(s), "cd": 2.0 * s.info()["forceX"]}
    if case["what"] == "ensemble":
        r = cuibm_amd.ensemble_run(state["folders"], "-amgPrecision", case["precision"], steps=case["steps"],
                                   workers=8, lockstep=True)
        return {"cells": r["cells"], "cd": r["cd"]}
    import torch

    alpha = torch.tensor(0.5, dtype=torch.float64, requires_grad=True)
    blow = torch.tensor(state["blow"], dtype=torch.float64, requires_grad=True)
    drag = mean_drag(alpha, blow, state["problem"])
    drag.backward()
    return {"drag": drag.detach(), "d_alpha": alpha.grad, "d_blow": blow.grad}


def work(case):
    """A step reads and writes u, the last N and p once; the arithmetic is that of the two
    right-hand sides, the projection and one product with each operator. The gradient takes
    a forward and a backward pass. A solve reads the matrix and b and writes x."""
    if case["family"] == "csr":
        n = case["nx"] * case["ny"]
        return {"bytes": 5 * n * 12.0 + 4.0 * n + 16.0 * n, "flops": 10.0 * n}
    cells = case["nx"] * case["ny"] if case["family"] == "steps" else case["cells"]
    passes = case["steps"] * (2 if case.get("what") == "adjoint" else 1)
    return {"bytes": passes * cells * 8.0 * (4 * 2 + 2), "flops": passes * cells * 170.0}


def tolerance(case):
    """About four times the largest difference measured between the solves with another
    coarsest level of the hierarchy and with another precision of it: where a solve stops
    within its residual tolerance is what separates two correct runs, and the pressure of the
    embedded method feels it most."""
    if case["family"] == "csr":
        return {"rel": 4e-8, "max": 6e-8}
    if case.get("what") == "ensemble":
        return {"rel": 1e-8, "max": 2e-8}
    if case.get("what") == "adjoint":
        return {"rel": 2e-11, "max": 2e-11}
    if case.get("solve") == 1e-7:  # the embedded folders
        return {"rel": 2.5e-3, "max": 1e-2}
    if case.get("folder") == "cylinderRe40_890_fadlun":  # solved to 1e-5
        return {"rel": 1.5e-3, "max": 8e-3}
    if case.get("folder") == "cylinderRe550_1024_luo" or case.get("rtol") == 1e-9:
        return {"rel": 2.5e-6, "max": 2.5e-5}
    if case.get("kind") == "plain" or case["folder" if "folder" in case else "kind"].startswith("lidDriven"):
        return {"rel": 2e-6, "max": 1e-5}
    return {"rel": 2.5e-5, "max": 1.6e-4}


# ---- 64-bit answers in plain numpy --------------------------------------------------------


class _Separable:
    """(Tx (+) Ty) x = b for x[J, I], Tx and Ty tridiagonal (diagonal, lower, upper), by the
    eigenvectors of both after a diagonal scaling that makes them symmetric; optionally with
    the diagonal of a few cells raised (Woodbury)."""

    def __init__(self, tx, ty, raised=()):
        (self.lx, self.qx, self.sx), (self.ly, self.qy, self.sy) = self._axis(*tx), self._axis(*ty)
        lam = self.ly[:, None] + self.lx[None, :]
        # the constant of the unraised Neumann operator: one of its cells' raises is added back
        # through a shift that Woodbury takes away again
        self.shift = np.zeros_like(lam)
        if raised:
            k = np.unravel_index(np.argmin(np.abs(lam)), lam.shape)
            self.shift[k] = np.abs(lam).max() * 1e-3
        self.inv = 1.0 / (lam + self.shift)
        self.raised = list(raised)
        if self.raised:
            # A = A0 + sum_c d_c e_c e_c^T, A0 = (shifted operator) - s v w^T
            shape = lam.shape
            k = np.unravel_index(np.argmax(self.shift), shape)
            v = np.outer(self.qy[:, k[0]] / self.sy, self.qx[:, k[1]] / self.sx)
            w = np.outer(self.qy[:, k[0]] * self.sy, self.qx[:, k[1]] * self.sx)
            U, V = [], []
            for (J, I), d in self.raised:
                e = np.zeros(shape)
                e[J, I] = 1.0
                U.append(d * e)
                V.append(e)
            U.append(-self.shift[k] * v)
            V.append(w)
            self.V = np.stack([a.ravel() for a in V])
            self.AU = np.stack([self._plain(a).ravel() for a in U], 1)
            self.cap = np.eye(len(U)) + self.V @ self.AU

    @staticmethod
    def _axis(d, lo, up):
        n = d.size
        s = np.ones(n)
        s[1:] = np.exp(np.cumsum(0.5 * (np.log(-up) - np.log(-lo))))  # S T S^-1 is symmetric
        T = np.diag(d)
        i = np.arange(n - 1)
        T[i, i + 1] = T[i + 1, i] = -np.sqrt(up * lo)
        lam, q = np.linalg.eigh(T)
        return lam, q, s

    def _plain(self, b):
        t = self.qy.T @ (b * self.sy[:, None] * self.sx[None, :]) @ self.qx
        return (self.qy @ (t * self.inv) @ self.qx.T) / (self.sy[:, None] * self.sx[None, :])

    def solve(self, b):
        x = self._plain(b)
        if self.raised:
            x = x - (self.AU @ np.linalg.solve(self.cap, self.V @ x.ravel())).reshape(b.shape)
        return x


def _neumann(w, dt):
    """Diagonal, lower and upper entries of -dt d2/dx2 per cell, no flux through the ends."""
    e = dt * 2.0 / (w[:-1] + w[1:])
    up, lo = -e / w[:-1], -e / w[1:]
    return -np.append(up, 0) - np.append(0, lo), lo, up


def _cavity(case, up, vp, dt, steps, nu=0.01):
    """`steps` steps of the lid-driven cavity on cells of one size per axis: Adams-Bashforth
    convection, Crank-Nicolson diffusion, pressure projection."""
    nx, ny = case["nx"], case["ny"]
    hx, hy = 1.0 / nx, 1.0 / ny
    xc, yc, xf, yf = (np.arange(nx) + 0.5) * hx, (np.arange(ny) + 0.5) * hy, np.arange(1, nx) * hx, np.arange(1, ny) * hy
    ax = lambda x, lo, hi: (2 * x - hi - lo) / (hi - lo)
    X = lambda x: ax(x, xc[0], xc[-1])
    Y = lambda y: ax(y, yc[0], yc[-1])
    u = up * np.outer(np.sin(np.pi * Y(yc)), np.cos(0.5 * np.pi * X(xf)))
    v = vp * np.outer(np.cos(0.5 * np.pi * Y(yf)), np.sin(np.pi * X(xc)))
    lid, a = 1.0, 0.5 * dt * nu

    def tri(n, h, walls):  # 1/2 of the identity and the diffusion along one axis
        d = np.full(n, 0.5 + 2 * a / h ** 2)
        if not walls:  # the velocity along the wall: half a cell off it
            d[0] = d[-1] = 0.5 + 2 * a / h ** 2
        return d, np.full(n - 1, -a / h ** 2), np.full(n - 1, -a / h ** 2)

    su = _Separable(tri(nx - 1, hx, True), tri(ny, hy, False))
    sv = _Separable(tri(nx, hx, False), tri(ny - 1, hy, True))
    tx, ty = _neumann(np.full(nx, hx), dt), _neumann(np.full(ny, hy), dt)
    cells = [(0, 0)]
    c = (ny // 2, nx // 2)
    if 0 < c[0] < ny - 1 and 0 < c[1] < nx - 1:
        cells.append(c)
    sp = _Separable(tx, ty, [((J, I), tx[0][I] + ty[0][J]) for J, I in cells])
    N = [np.zeros_like(u), np.zeros_like(v)]
    for _ in range(steps):
        # neighbours, the walls' values beyond the last node; 2 wall - inside along a wall
        ue, uw = np.pad(u[:, 1:], ((0, 0), (0, 1))), np.pad(u[:, :-1], ((0, 0), (1, 0)))
        un, us = np.vstack([u[1:], 2 * lid - u[-1:]]), np.vstack([-u[:1], u[:-1]])
        vn, vs = np.pad(v[1:], ((0, 1), (0, 0))), np.pad(v[:-1], ((1, 0), (0, 0)))
        ve, vw = np.hstack([v[:, 1:], -v[:, -1:]]), np.hstack([-v[:, :1], v[:, :-1]])
        vf = np.pad(v, ((1, 1), (0, 0)))  # v on every horizontal face
        uf = np.pad(u, ((0, 0), (1, 1)))
        vu = 0.25 * (vf[1:, :-1] + vf[1:, 1:] + vf[:-1, :-1] + vf[:-1, 1:])
        uv = 0.25 * (uf[:-1, 1:] + uf[1:, 1:] + uf[:-1, :-1] + uf[1:, :-1])
        new = [u * (ue - uw) / (2 * hx) + vu * (un - us) / (2 * hy), uv * (ve - vw) / (2 * hx) + v * (vn - vs) / (2 * hy)]
        lu = nu * ((ue - 2 * u + uw) / hx ** 2 + (un - 2 * u + us) / hy ** 2)
        lv = nu * ((ve - 2 * v + vw) / hx ** 2 + (vn - 2 * v + vs) / hy ** 2)
        ru = u + dt * (0.5 * N[0] - 1.5 * new[0] + 0.5 * lu)
        rv = v + dt * (0.5 * N[1] - 1.5 * new[1] + 0.5 * lv)
        ru[-1] += (2 * lid - u[-1]) * a / hy ** 2
        ru[0] += -u[0] * a / hy ** 2
        rv[:, -1] += -v[:, -1] * a / hx ** 2
        rv[:, 0] += -v[:, 0] * a / hx ** 2
        N = new
        uh, vh = su.solve(ru), sv.solve(rv)
        uf, vf = np.pad(uh, ((0, 0), (1, 1))), np.pad(vh, ((1, 1), (0, 0)))
        p = sp.solve(-(uf[:, 1:] - uf[:, :-1]) / hx - (vf[1:] - vf[:-1]) / hy)
        u, v = uh - dt * (p[:, 1:] - p[:, :-1]) / hx, vh - dt * (p[1:] - p[:-1]) / hy
    return {"u": np.concatenate([u.ravel(), v.ravel()]), "p": p.ravel() - p.mean()}


def exact(case, seed):
    """The cavities and the caller's matrix; a flow around a body has no short plain form (the
    tagging of the nodes alone would take longer than the limit in plain Python)."""
    if case["family"] == "csr":
        wx, wy = _widths(case["nx"], seed), _widths(case["ny"], seed + 1)
        b = np.random.default_rng(seed).standard_normal(case["nx"] * case["ny"]).reshape(case["ny"], case["nx"])
        tx, ty = _neumann(wx, 1.0), _neumann(wy, 1.0)
        s = _Separable(tx, ty, [((0, 0), tx[0][0] + ty[0][0])])
        return {"x": s.solve(b).ravel(), "ok": None}
    if case["family"] == "steps" and (case.get("kind") == "plain" or case.get("folder", "").startswith("lidDriven")):
        up, vp = _perturbation(seed)
        dt = 0.3 / max(case["nx"], case["ny"]) if "kind" in case else 0.01
        return _cavity(case, up, vp, dt, case["steps"])
    return None

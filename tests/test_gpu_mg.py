"""The multigrid levels of the stencil-form Poisson operator (mg.hip: FP32 levels, and FP64
solves to 1e-9 or less) at the sizes where their kernels can go wrong: strips of 57 and 58
columns and chunks of 4 and 8 rows that end inside or just past the grid, axes that never
coarsen, aggregates across chunk and strip edges, the smallest and the largest directly solved
grid, one and two pins, FP32 and FP64 levels.

Each solve is checked on the assembled CSR matrix: the residual of the returned p must be the
one the solve claims, at most rtol ||b|| and the recurrence's rounding, and the solve must take
no more iterations than the levels are worth: none where the grid is solved directly (the
first half step already converges), otherwise at most 10, a factor of 10 per iteration over
the ten digits asked for (they give 20 to 100). test_gpu_mg_cycle.py
compares the values of an iteration."""
import math

import numpy as np
import pytest
import scipy.sparse as sp

import cuibm_amd
import pyoracle as po
from cuibm_amd import ensemble as ens
from helpers import case, rel_l2

pytestmark = pytest.mark.gpu


def write_case(d, nx, ny, solver, ratio=None, h=None, ends=(1.0, 1.0)):
    """a cavity of nx x ny equal cells from 0 to `ends` (solver NAVIER_STOKES_SOLVER), or a
    cylinder on a grid stretched by `ratio` from spacing h"""
    if ratio is None:
        axis = lambda n, m, e: (f"- direction: {n}\n  start: 0.0\n  mid_h: {e / (m + 0.5)!r}\n  subDomains:\n"
                                f"    - end: {e!r}\n      stretchRatio: 1.0\n")
        dom = axis("x", nx, ends[0]) + axis("y", ny, ends[1])
    else:
        axis = lambda n: (f"- direction: {n}\n  start: -15.0\n  mid_h: {h!r}\n  subDomains:\n    - end: -0.6\n"
                          f"      stretchRatio: {ratio!r}\n    - end: 0.6\n      stretchRatio: 1.0\n"
                          f"    - end: 15.0\n      stretchRatio: {ratio!r}\n")
        dom = axis("x") + axis("y")
        (d / "bodies.yaml").write_text(f"- type: circle\n  circleOptions: [0.0, 0.0, 0.5, {int(math.pi / h)}, false]\n")
    (d / "domain.yaml").write_text(dom)
    flow = "- type: flow\n  nu: 0.01\n  initialVelocity: [0.0, 0.0]\n  boundaryConditions:\n"
    for loc in ("xMinus", "xPlus", "yMinus", "yPlus"):
        flow += f"    - location: {loc}\n      u: [DIRICHLET, 0.0]\n      v: [DIRICHLET, 0.0]\n"
    (d / "flow.yaml").write_text(flow)
    solve = lambda n, m: (f"    - system: {n}\n      solver: BICGSTAB\n      preconditioner: {m}\n"
                          "      tolerance: 1e-10\n      maxIterations: 200\n")
    (d / "simParams.yaml").write_text(f"- type: simulation\n  dt: 0.01\n  nt: 10\n  nsave: 10\n  scaleCV: 2.0\n"
                                      f"  SolverType: {solver}\n  linearSolvers:\n" + solve("velocity", "DIAGONAL")
                                      + solve("Poisson", "SMOOTHED_AGGREGATION"))
    return str(d)


def check(folder, precision, most, *args):
    rtol = 1e-10
    with cuibm_amd.Solver(folder, "-amgPrecision", precision, *args, diagnostics=False) as s:
        s.initialise()
        i = s.info()
        nx, ny = int(i["nx"]), int(i["ny"])
        A = sp.csr_matrix((s.get("LHS2_val"), s.get("LHS2_col"), s.get("LHS2_rowptr")), shape=(nx * ny, nx * ny))
        for seed in range(2):
            b = np.random.default_rng(seed).standard_normal(nx * ny)
            s.set("rhs2", b)
            s.set("p", np.zeros(nx * ny))
            s.phase("solvePoisson")
            p, it = s.get("p"), s.info()["iter2"]
            res = np.linalg.norm(b - A @ p) / np.linalg.norm(b)
            print(f"{nx} x {ny} precision {precision}: levels {i['amg_levels']:.0f} iterations {it:.0f} residual {res:.2e}",
                  flush=True)
            # the recurrence's rounding: a few eps ||A|| ||p|| in every update
            floor = 16 * np.finfo(float).eps * 2 * A.diagonal().max() * np.linalg.norm(p) / np.linalg.norm(b)
            assert res <= rtol + floor
            assert it <= most


# (a grid solved directly is solved in FP64 in either precision)
@pytest.mark.parametrize("nx,ny,precision", [(51, 50, 32), (57, 64, 32), (320, 17, 32), (301, 173, 32),
                                             (101, 100, 64), (320, 320, 64)])
def test_direct_grids(tmp_path, nx, ny, precision):
    check(write_case(tmp_path, nx, ny, "NAVIER_STOKES_SOLVER"), precision, 0)


# axes that run downwards (negative cell widths): the operator, and the iterations, are those of
# the axes turned round
@pytest.mark.parametrize("ends", [(-1.0, 1.0), (1.0, -1.0), (-1.0, -1.0)])
@pytest.mark.parametrize("nx,ny,precision,most", [(101, 100, 64, 0), (57, 64, 32, 0), (342, 333, 64, 10),
                                                  (321, 17, 32, 16)])
def test_axes_that_run_downwards(tmp_path, nx, ny, precision, most, ends):
    check(write_case(tmp_path, nx, ny, "NAVIER_STOKES_SOLVER", ends=ends), precision, most)


# FP32 levels restart after every three digits, and each restart finds the modes of the cavity's
# two pins anew (two iterations of three restarts more)
@pytest.mark.parametrize("nx,ny", [(321, 17), (9, 400), (342, 333), (57 * 7, 58 * 6), (513, 345), (1030, 225)])
def test_fp32_levels_of_uniform_grids(tmp_path, nx, ny):
    check(write_case(tmp_path, nx, ny, "NAVIER_STOKES_SOLVER"), 32, 16)


@pytest.mark.parametrize("nx,ny", [(321, 33), (9, 1200), (342, 333), (57 * 7, 58 * 6), (513, 345), (1030, 225)])
def test_fp64_levels_of_uniform_grids(tmp_path, nx, ny):
    check(write_case(tmp_path, nx, ny, "NAVIER_STOKES_SOLVER"), 64, 10)


@pytest.mark.parametrize("precision", [64, 32, 3264])
@pytest.mark.parametrize("h,ratio", [(0.021, 1.021), (0.012, 1.0137), (0.008, 1.035)])
def test_levels_of_stretched_grids(tmp_path, h, ratio, precision):
    check(write_case(tmp_path, 0, 0, "LUO", ratio, h), precision, 10)


def test_coarsest_level_as_asked_for(tmp_path):
    """-amgCoarseMax bounds the directly solved level"""
    check(write_case(tmp_path, 130, 120, "NAVIER_STOKES_SOLVER"), 64, 10, "-amgCoarseMax", 400)
    check(case("cylinderRe40_luo"), 64, 10, "-poissonTol", "1e-10", "-amgCoarseMax", 3000)


def test_coarsest_level_does_not_choose_the_kind():
    """4489 unknowns to 1e-12 in FP64 keep the stored hierarchy with a small -amgCoarseMax too: the
    oracle's iterations (33 to 5 with the multigrid levels), to the one that rounding may move"""
    tol = {"velocityTol": 1e-12, "poissonTol": 1e-12}
    po.set_amg_coarse_max(400)
    try:
        o = po.Oracle(po.read_case(case("cylinderRe40_small_luo"), tol))
        o.step(3)
    finally:
        po.set_amg_coarse_max(0)
    with cuibm_amd.Solver(case("cylinderRe40_small_luo"), "-velocityTol", "1e-12", "-poissonTol", "1e-12",
                          "-amgCoarseMax", "400", diagnostics=False) as g:
        g.initialise()
        g.step_time(3)
        d = rel_l2(g.get("p"), o.get("p"))
        print("p", d, "iterations", g.info()["iter2"], o.info()["iter2"], flush=True)
        assert abs(g.info()["iter2"] - o.info()["iter2"]) <= 1
        assert d <= 1e-10


def test_lockstep_of_both_kinds(tmp_path):
    """an FP64 batch at 1e-10 of a grid small enough for a stored hierarchy and of larger ones:
    drag within 1e-8 of the cases alone"""
    paths, cases = ens.write_cases(str(tmp_path), n=4, seed=12, steps=20, edges=(80, 150))
    sizes = [c[0] ** 2 for c in cases]
    assert min(sizes) <= 10000 < max(sizes)
    tight = ["-amgPrecision", "64", "-velocityTol", "1e-10", "-poissonTol", "1e-10"]
    r = cuibm_amd.ensemble_run(paths, *tight, steps=20, workers=4, lockstep=True)
    for k, path in enumerate(paths):
        with cuibm_amd.Solver(path, *tight, diagnostics=False) as s:
            s.initialise()
            s.step_time(20)
            assert abs(r["cd"][k] - 2 * s.info()["forceX"]) <= 1e-8

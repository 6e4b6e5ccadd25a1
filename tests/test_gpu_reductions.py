"""The reductions of BiCGSTAB at the sizes where their partial sums can go wrong: fewer unknowns
than a group's 256, the last group of a grid full and one past it, both sides of the line where a
block holds one group and four (512 partial sums), and both sides of the most partial sums (2048),
where the groups take more than one stride. Three iterations on a diagonally dominant matrix
against the same recurrence with numpy's products.

Bar: a sum of n products regrouped differs by at most ~ 2 log2(n) eps sum|a_i b_i| (both sides sum
pairwise above runs of 8 to 300), so a quotient's relative error is that times w, how far the
products lie from their Cauchy-Schwarz bound (measured on the reference's own, 7 to 600 here);
three iterations multiply at most six such quotients."""
import math

import numpy as np
import pytest
import scipy.sparse as sp

import cuibm_amd
from helpers import rel_l2

pytestmark = pytest.mark.gpu


def three_iterations(A, b, dinv):
    worst = 1.0

    def dot(u, v):
        nonlocal worst
        d = float(np.dot(u, v))
        worst = max(worst, np.linalg.norm(u) * np.linalg.norm(v) / abs(d))
        return d

    x = np.zeros_like(b)
    r = b.copy()
    p, rs = r.copy(), r.copy()
    rho = dot(rs, r)
    for _ in range(3):
        Mp = dinv * p
        AMp = A @ Mp
        alpha = rho / dot(rs, AMp)
        s = r - alpha * AMp
        Ms = dinv * s
        AMs = A @ Ms
        omega = dot(AMs, s) / dot(AMs, AMs)
        x += alpha * Mp + omega * Ms
        r = s - omega * AMs
        rho2 = dot(rs, r)
        beta = rho2 / rho * alpha / omega
        rho = rho2
        p = r + beta * (p - omega * AMp)
    return x, worst


@pytest.mark.parametrize("precond", ["NONE", "DIAGONAL"])
@pytest.mark.parametrize("n", [5, 255, 2047, 2048, 2049, 131071, 131072, 131073, 262144, 524287, 524288, 700001])
def test_three_iterations(n, precond):
    d = 2.5 + 0.5 * np.cos(np.arange(n) / 7.0)
    A = sp.diags([np.full(n - 1, -1.0), d, np.full(n - 1, -0.7)], [-1, 0, 1]).tocsr()
    b = 1.0 + 0.5 * np.sin(np.arange(n) / 11.0)
    dinv = 1.0 / d if precond == "DIAGONAL" else np.ones(n)
    xr, worst = three_iterations(A, b, dinv)
    g = cuibm_amd.Csr(A)
    x, its, _, ok = g.bicgstab(b, precond=precond, rtol=1e-300, maxit=3)
    print(n, precond, "its", its, "x diff", rel_l2(x, xr), "worst quotient", worst, flush=True)
    assert its == 3 and not ok
    assert rel_l2(x, xr) < 6 * worst * 2 * math.log2(n) * np.finfo(float).eps
    if n <= 2**18:  # the fixed scratch array
        y, _, _, _ = g.bicgstab_noalloc(b, precond=precond, rtol=1e-300, maxit=3)
        assert np.array_equal(x, y)

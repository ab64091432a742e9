"""The small levels of the aligned hierarchy's V-cycle in one launch
(k_small_cycle): solves on grids whose coarse levels it takes over -- one, two
and three of them, the largest first levels (13 x 9 x 11, a
lane per cell of a colour; 17^3, past it), sides of 3 to 33 cells,
even coarsest sides -- converge at the rate of the hierarchy to the solution
of a dense solve of the operator that find_AX gives. Bars: the relative
residual 1e-12 within 14 V-cycles (the aligned hierarchy reduces it by 0.1
per cycle on these problems), and the solution's error at most cond(A) times
that residual."""
import numpy as np
import pytest

from mps3d_amd import FieldSolver, ghosted
from mps3d_amd import workloads as W

pytestmark = pytest.mark.gpu

GRIDS = [(5, 5, 5), (9, 9, 9), (7, 5, 9), (11, 7, 5), (13, 9, 7), (5, 9, 17), (17, 5, 5)]


def operator(s, n):
    """The dense matrix of the operator, 27 probes (cells of equal index mod 3)."""
    N = int(np.prod(n))
    idx = np.indices(n).reshape(3, -1, order="F")
    A = np.zeros((N, N))
    lin = np.arange(N).reshape(n, order="F")
    for r in range(27):
        sel = (idx[0] % 3 == r % 3) & (idx[1] % 3 == r // 3 % 3) & (idx[2] % 3 == r // 9)
        e = np.where(sel, 1.0, 0.0).reshape(n, order="F")
        ax = s.find_AX(ghosted(e))[0]
        for q in np.nonzero(sel)[0]:
            i, j, k = idx[:, q]
            for di, dj, dk in ((0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1)):
                a, b, c = i + di, j + dj, k + dk
                if 0 <= a < n[0] and 0 <= b < n[1] and 0 <= c < n[2]:
                    A[lin[a, b, c], q] = ax[a, b, c]
    return A


@pytest.mark.parametrize("n", GRIDS)
@pytest.mark.parametrize("form", ["diffusion", "sg", "sg_transpose", "fp32dc", "fmg"])
def test_solution_is_the_dense_solve(gpu, n, form):
    c = W.varcoef_poisson(n)
    c.length = tuple(0.02 * m / max(n) for m in n)
    kw = {"fp32dc": dict(precision="fp32dc"), "fmg": dict(start="fmg")}.get(form, {})
    sg = form.startswith("sg")
    if sg:
        c.dcoeff = np.full(n, 100.0, order="F")
        c.velx, c.vely, c.velz = (np.full(n, v, order="F") for v in (1e4, -2e4, 3e4))
        c.timederiv, c.dt = True, 1e-7
        kw = dict(flux="sg")
    b = np.random.default_rng(1).standard_normal(n)
    with FieldSolver(c.n, c.length, hierarchy="aligned", arith="fast", tol=1e-12, tol_kind="rel", max_cycles=14,
                     **kw) as s:
        s.set_case(c)
        x = ghosted(np.zeros(n))
        A = operator(s, n)
        if form == "sg_transpose":
            A = A.T
            k, r, st = s.solve_transpose(b, x)
        else:
            k, r, _, st = s.solve_rhs(b, x)
    assert st == 0, (k, r)
    ref = np.linalg.solve(A, b.ravel(order="F"))
    err = np.linalg.norm(x[1:-1, 1:-1, 1:-1].ravel(order="F") - ref) / np.linalg.norm(ref)
    assert err <= 1e-12 * np.linalg.cond(A)


@pytest.mark.parametrize("n", [(33, 33, 33), (33, 17, 25), (25, 33, 17), (25, 17, 21)])
@pytest.mark.parametrize("prec", ["fp64", "fp32dc"])
def test_the_largest_levels_converge_at_the_hierarchy_rate(gpu, n, prec):
    c = W.varcoef_poisson(n)
    c.length = tuple(0.02 * m / max(n) for m in n)
    with FieldSolver(c.n, c.length, hierarchy="aligned", arith="fast", precision=prec, tol=1e-12, tol_kind="rel",
                     max_cycles=14) as s:
        s.set_case(c)
        x = ghosted(np.zeros(n))
        _, r, _, st = s.solve(x)
    assert st == 0, r

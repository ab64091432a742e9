"""The coarsest level's dense inverse (k_dense_inverse_regs, and the paths for
larger grids) on grids that are their own coarsest level: the solve is then
x = A^-1 b, compared with numpy's dense solve of the matrix that find_AX
gives. Bar: 8 n eps cond(A) relative, the forward error of an inverse formed
by elimination with partial pivoting and applied by one product, with a
factor for its constants. Sizes: one cell, the edges of each register
layout, and above the largest. A singular operator is refused where an
elimination in FP64, operation by operation, meets a zero pivot, and accepted
where its rounding leaves one that is not zero. On the reference hierarchy
with Scharfetter-Gummel rows the inverse is of those rows, with their drift
and reaction."""
import numpy as np
import pytest

from mps3d_amd import FieldSolver, _lib as M, ghosted
from mps3d_amd import workloads as W

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (3, 3, 3), (4, 4, 2), (3, 11, 1), (4, 4, 4), (5, 13, 1), (8, 4, 4), (3, 43, 1), (7, 5, 6), (8, 7, 4),
         (15, 15, 1)]


def dense(s, n):
    N = int(np.prod(n))
    A = np.empty((N, N))
    for q in range(N):
        e = np.zeros(N)
        e[q] = 1.0
        A[:, q] = s.find_AX(ghosted(e.reshape(n, order="F")))[0].ravel(order="F")
    return A


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("form", ["aligned_sg", "aligned_cdr", "aligned_diffusion", "ref_fast"])
def test_coarsest_solve_is_the_dense_solve(gpu, n, form):
    c = W.random_cdr(n, seed=17 + sum(n))
    if form == "aligned_diffusion":
        c.velx = c.vely = c.velz = None
    # a reaction of either sign as large as the diffusive rows: the diagonal
    # does not dominate, so rows are exchanged
    c.reac = 400.0 * c.reac
    kw = {"ref_fast": dict(hierarchy="ref", p=n, arith="fast"),
          "aligned_sg": dict(hierarchy="aligned", flux="sg", arith="fast")}.get(form, dict(hierarchy="aligned", arith="fast"))
    if form == "ref_fast":
        c.velx = c.vely = c.velz = None
    b = np.random.default_rng(2).standard_normal(n)
    with FieldSolver(c.n, c.length, tol=1e-8, tol_kind="rel", max_cycles=1, **kw) as s:
        s.set_case(c)
        A = dense(s, n)
        x = ghosted(np.zeros(n))
        s.solve_rhs(b, x)
    ref = np.linalg.solve(A, b.ravel(order="F"))
    err = np.linalg.norm(x[1:-1, 1:-1, 1:-1].ravel(order="F") - ref) / np.linalg.norm(ref)
    assert err <= 8 * b.size * np.finfo(float).eps * np.linalg.cond(A)


@pytest.mark.parametrize("n", [(3, 3, 3), (8, 7, 4), (15, 15, 1)])
def test_a_singular_coarsest_operator_is_refused(gpu, n):
    with FieldSolver(n, hierarchy="aligned", arith="fast") as s:
        s.set_bc(("ZGRD",) * 6)
        with pytest.raises(M.MpsError, match="singular"):
            s.set_coeffs(np.zeros(n))


def eliminates(A):
    """Whether Gauss-Jordan elimination with partial pivoting meets no zero pivot."""
    A = A.copy()
    for c in range(len(A)):
        p = c + int(np.argmax(np.abs(A[c:, c])))
        if not abs(A[p, c]) > 0.0:
            return False
        A[[c, p]] = A[[p, c]]
        A[c] *= 1.0 / A[c, c]
        for r in np.nonzero(A[:, c])[0]:
            if r != c:
                A[r] -= A[r, c] * A[c]
    return True


def no_flux_rows(n, length):
    """The operator with D = 1 and no flux through any face, as find_AX sums it."""
    N = int(np.prod(n))
    A = np.zeros((N, N))
    for r, p in enumerate(np.ndindex(n[::-1])):
        for d in (2, 1, 0):
            w = (0.5 * (1.0 + 1.0)) / (length / n[2 - d]) * (1.0 / (length / n[2 - d]))
            for s in (-1, 1):
                if 0 <= p[d] + s < n[2 - d]:
                    A[r, r + s * int(np.prod(n[:2 - d]))] = -w
                    A[r, r] += w
    return A


def test_a_singular_operator_is_judged_by_its_rounding(gpu):
    wrong, refused = [], 0
    for n in ((i, j, k) for i in range(1, 7) for j in range(1, 7) for k in range(1, 7)):
        # (grids that are their own coarsest level)
        if np.prod(n) > 100 or min(n) > 3 and all(v % 2 for v in n):
            continue
        want = eliminates(no_flux_rows(n, 0.02))
        refused += not want
        with FieldSolver(n, (0.02,) * 3, hierarchy="aligned", arith="fast") as s:
            s.set_bc(("ZGRD",) * 6)
            try:
                s.set_coeffs(np.ones(n))
                got = True
            except M.MpsError as e:
                got = "singular" not in str(e)
        if got != want:
            wrong.append(n)
    assert refused > 0 and wrong == []


@pytest.mark.parametrize("n,p", [((16, 16, 16), (1, 1, 1)), ((24, 24, 24), (3, 3, 3)), ((16, 16, 16), (4, 4, 4)),
                                 ((56, 56, 40), (7, 7, 5))])
@pytest.mark.parametrize("prec", ["fp64", "fp32dc"])
@pytest.mark.parametrize("timederiv", [False, True])
def test_reference_hierarchy_with_drift_in_fast_arithmetic(gpu, n, p, prec, timederiv):
    # coarsest grids of 1, 27, 64 and 245 cells; the cycle in exact arithmetic, whose
    # coarse solve is GMRES, sets the count (one more is allowed)
    drift = [np.full(n, v, order="F") for v in (1e4, -2e4, 3e4)]
    reac = np.full(n, -1e6, order="F")
    b = np.asfortranarray(np.random.default_rng(3).standard_normal(n))
    count = {}
    for arith in ("exact", "fast"):
        with FieldSolver(n, (0.02,) * 3, p=p, hierarchy="ref", flux="sg", arith=arith, precision=prec, tol=1e-10,
                         tol_kind="rel", max_cycles=30) as s:
            s.set_bc(("ZGRD",) * 4 + ("DIRC",) * 2, (0.0,) * 4 + (1.0, 2.0))
            s.set_coeffs(np.full(n, 100.0, order="F"), *drift, reac, b, timederiv, 1e-7)
            x, y = ghosted(np.zeros(n)), ghosted(np.zeros(n))
            k, _, _, st = s.solve(x)
            g, _, gst = s.gmres(b, y, m=30, restarts=1, tol=1e-10)
            assert st == 0 and gst == 0, (arith, k, g)
            count[arith] = k, g
    assert all(f <= e + 1 for f, e in zip(count["fast"], count["exact"])), count

"""The small levels of the aligned hierarchy's V-cycle in one launch
(k_small_cycle).

Solves on grids of two and three levels (of GRIDS only 9^3 has a small level
above its coarsest) converge to the solution of a dense solve of the operator
that find_AX gives; bars: the relative residual 1e-12 within 14 V-cycles (the
aligned hierarchy reduces it by 0.1 per cycle on these problems), and the
solution's error at most cond(A) times that residual.

One V-cycle, forward and transposed, is a V-cycle on the host from the same
rows, transfers, smoothing and coarsest solve, on grids that reach each form
of the launch (CYCLES)."""
import numpy as np
import pytest
import scipy.sparse as sp

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


# levels, and what the launch takes of them
CYCLES = [
    (9, 9, 9),      # 9^3, 5^3 over 3^3
    (17, 17, 17),   # below 17^3: the same
    (33, 33, 33),   # below 17^3 again, from one level higher
    (25, 17, 21),   # 13 x 9 x 11, 693 cells of a colour (1024 lanes), over 7 x 5 x 6, 210 rows in two rounds of loads
    (33, 17, 21),   # 17 x 9 x 11, 891 cells of a colour, over 9 x 5 x 6, 270 rows inverted on the host
    (13, 9, 17),    # 7 x 5 x 9 over 4 x 3 x 5
    (17, 9, 33),    # 9 x 5 x 17 over 5 x 3 x 9, 135 rows
    (25, 25, 25),   # 7^3 over 4^3 below 13^3, which does not fit in FP64
    (9, 21, 13),    # 5 x 11 x 7 over 3 x 6 x 4
]


def bernoulli(x):
    return 1.0 if x == 0.0 else x / np.expm1(x)


def host_levels(n, h0, D, vel, dirc, shift):
    """Per level (sizes, matrix, restriction onto it, prolongation from it):
    the rows for constant D and velocity are sums of one-dimensional ones."""
    out, H, W, P = [], list(h0), None, None
    n = list(n)
    while True:
        A = 0
        for d in range(3):
            m = n[d]
            a = np.full(m, 1.0 / H[d])
            a[0] = a[-1] = 1.0 / (0.5 * H[d] + 0.5 * h0[d])
            Dh = D if vel[d] == 0.0 else 2.0 * D * D / (D + D + 1e-10)
            Pe = vel[d] * H[d] / Dh
            wl, wr = Dh / H[d] * bernoulli(-Pe), -Dh / H[d] * bernoulli(Pe)
            T = np.zeros((m, m))
            for i in range(m - 1):   # face i | i + 1
                T[i, i] += wl * a[i]
                T[i, i + 1] += wr * a[i]
                T[i + 1, i + 1] -= wr * a[i + 1]
                T[i + 1, i] -= wl * a[i + 1]
            if d == 2 and dirc:
                T[0, 0] += 2.0 * D / h0[d] * a[0]
                T[-1, -1] += 2.0 * D / h0[d] * a[-1]
            eye = [sp.identity(v) for v in n]
            eye[d] = sp.csr_matrix(T)
            A = A + sp.kron(eye[2], sp.kron(eye[1], eye[0]))
        out.append((tuple(n), (A + shift * sp.identity(int(np.prod(n)))).tocsr(), W, P))
        if min(n) <= 3 or any(v % 2 == 0 for v in n):
            return out
        w1, p1 = [], []
        for d in range(3):
            m, mc = n[d], (n[d] + 1) // 2
            vol = np.full(m, H[d])
            vol[0] = vol[-1] = 0.5 * H[d] + 0.5 * h0[d]
            w, p = np.zeros((mc, m)), np.zeros((m, mc))
            for c in range(mc):
                for f, part in ((2 * c - 1, 0.5), (2 * c, 1.0), (2 * c + 1, 0.5)):
                    if 0 <= f < m:
                        w[c, f] = part * vol[f]
            w /= w.sum(axis=1, keepdims=True)
            for f in range(m):
                p[f, f // 2] += 0.5
                p[f, (f + 1) // 2] += 0.5
            w1.append(sp.csr_matrix(w))
            p1.append(sp.csr_matrix(p))
            n[d], H[d] = mc, 2.0 * H[d]
        W = sp.kron(w1[2], sp.kron(w1[1], w1[0])).tocsr()
        P = sp.kron(p1[2], sp.kron(p1[1], p1[0])).tocsr()


def host_cycle(levels, l, u, b, nu, omega):
    """Red-black sweeps, full weighting, the coarser correction, trilinear
    interpolation, sweeps; a dense solve on the coarsest."""
    n, A, _, _ = levels[l]
    if l == len(levels) - 1:
        return np.linalg.solve(A.toarray(), b)
    i, j, k = (q.ravel(order="F") for q in np.indices(n))
    dg = A.diagonal()

    def smooth(u, times):
        for _ in range(times):
            for colour in (0, 1):
                own = (i + j + k) % 2 == colour
                u = u + np.where(own, omega[l] * (b - A @ u) / dg, 0.0)
        return u

    u = smooth(u, nu[0])
    r = levels[l + 1][2] @ (b - A @ u)
    u = u + levels[l + 1][3] @ host_cycle(levels, l + 1, np.zeros_like(r), r, nu, omega)
    return smooth(u, nu[1])


def plain_omega(levels, omega, size):
    """omega on the finest levels, 1 on those that sweep plainly: the coarsest
    ones, at most four, that fit 64 KB with their ghosts, right-hand sides,
    residuals and rows."""
    out, words, q = [omega] * len(levels), 0, len(levels) - 1
    while q >= 1:
        n = levels[q][0]
        words += int(np.prod([v + 2 for v in n])) + 9 * int(np.prod(n))
        if words * size > 64 * 1024 or len(levels) - q > 4:
            break
        out[q] = 1.0
        q -= 1
    return out if q < len(levels) - 2 else [omega] * len(levels)


@pytest.mark.parametrize("n", CYCLES)
@pytest.mark.parametrize("form,nu", [("diffusion", (2, 2)), ("diffusion", (1, 2)), ("diffusion", (3, 1)),
                                     ("sg", (2, 2)), ("sg", (1, 1)), ("sg_transpose", (2, 2)),
                                     ("sg_transpose", (1, 3)), ("relaxed", (2, 2)), ("fp32dc", (2, 2))])
def test_one_cycle_is_the_hosts(gpu, n, form, nu):
    # bars: the coarsest solve's, 8 n eps cond of the coarsest matrix, times 4
    # a level, by which the finest matrix's condition and so the cancellation
    # in its residuals is larger; an FP32 cycle loses cond eps32, here at most
    # 1e4 of 6e-8
    length = tuple(0.02 * v / max(n) for v in n)
    h0 = [a / v for a, v in zip(length, n)]
    drift = form.startswith("sg")
    D, vel = (100.0, (1e4, -2e4, 3e4)) if drift else (1.0, (0.0,) * 3)
    shift = 1e7 if drift else 0.0
    levels = host_levels(n, h0, D, vel, not drift, shift)
    g = np.random.default_rng(sum(n))
    b, u0 = g.standard_normal(n) / h0[0] ** 2, g.standard_normal(n)
    kw = dict(flux="sg") if drift else {}
    if form == "fp32dc":
        kw = dict(precision="fp32dc", dc_inner=1, omega=1.0)
    with FieldSolver(n, length, hierarchy="aligned", arith="fast", nu1=nu[0], nu2=nu[1], max_cycles=1, tol=0.0,
                     tol_kind="rel", **kw) as s:
        s.set_bc(("FLUX",) * 6 if drift else ("ZGRD",) * 4 + ("DIRC",) * 2, (0.0,) * 6)
        full = [np.full(n, v, order="F") for v in (D,) + vel]
        s.set_coeffs(full[0], *(full[1:] if drift else (None,) * 3), None, None, drift, 1.0 / shift if drift else 1.0)
        x = ghosted(u0)
        probe = g.standard_normal(n)
        ax = (s.apply_transpose if form == "sg_transpose" else lambda q: s.find_AX(q)[0])(ghosted(probe))
        if form == "sg_transpose":
            s.solve_transpose(np.asfortranarray(b), x)
        elif form in ("relaxed", "fp32dc"):
            s.solve_rhs(np.asfortranarray(b), x)
        else:
            s.perform_vcycle(x, np.asfortranarray(b))
    if form == "sg_transpose":
        levels = [(m, A.T.tocsr(), W, P) for m, A, W, P in levels]
    flat = lambda a: np.asarray(a).ravel(order="F")  # noqa: E731
    want = levels[0][1] @ flat(probe)
    assert np.linalg.norm(flat(ax) - want) <= 1e-12 * np.linalg.norm(want)
    omega = plain_omega(levels, 1.15, 8) if form == "relaxed" else [1.0] * len(levels)
    if form == "fp32dc":
        defect = flat(b) - levels[0][1] @ flat(u0)
        ref = flat(u0) + host_cycle(levels, 0, np.zeros(defect.size), defect, nu, omega)
    else:
        ref = host_cycle(levels, 0, flat(u0), flat(b), nu, omega)
    coarse = levels[-1][1].toarray()
    bar = 1e-3 if form == "fp32dc" else 8 * len(coarse) * np.finfo(float).eps * np.linalg.cond(coarse) * \
        4.0 ** (len(levels) - 1)
    assert np.linalg.norm(flat(x[1:-1, 1:-1, 1:-1]) - ref) <= bar * np.linalg.norm(ref)

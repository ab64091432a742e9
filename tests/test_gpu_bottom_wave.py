"""The coarse GMRES of at most 64 cells in one wavefront (k_bottom_wave)
through mps_gmres(precond=0): bit for bit the oracle's performgmres (every
operation is an IEEE addition, multiplication, division or square root in the
reference's order), from one cell to the 64 of a full wavefront and one case
above it (k_bottom), with fewer and more Krylov vectors than cells, restarts
and rows with and without convection and reaction; and, for explicit
(Scharfetter-Gummel) rows, a restatement of the same algorithm on the dense
matrix that find_AX gives."""
import math

import numpy as np
import pytest

from mps3d_amd import FieldSolver, ghosted
from mps3d_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [((1, 1, 1), 1, 1), ((2, 1, 1), 2, 1), ((7, 1, 1), 7, 1), ((3, 5, 1), 15, 1), ((2, 2, 4), 16, 1),
         ((1, 17, 1), 17, 1), ((4, 4, 2), 32, 1), ((3, 11, 1), 33, 1), ((3, 3, 7), 63, 1), ((4, 4, 4), 64, 1),
         ((64, 1, 1), 64, 1), ((4, 5, 3), 7, 5), ((4, 4, 4), 1, 3), ((2, 3, 1), 64, 1), ((13, 5, 1), 65, 1)]


@pytest.mark.parametrize("n,m,restarts", CASES)
@pytest.mark.parametrize("form", ["cdr", "diffusion", "no_reaction"])
def test_one_wave_gmres_equals_the_oracle(gpu, n, m, restarts, form):
    c = W.random_cdr(n, seed=31 + sum(n))
    if form == "diffusion":
        c.velx = c.vely = c.velz = None
    if form != "cdr":
        c.reac = None
    rng = np.random.default_rng(5)
    b, x0 = rng.standard_normal(n), rng.standard_normal(n)
    P = O.Problem(c.n, c.length, (1, 1, 1), c.bc_codes, c.bc_vals, c.dcoeff, c.velx, c.vely, c.velz, c.reac, c.source,
                  c.timederiv, c.dt)
    ref = O.gmres(P, b, ghosted(x0), m, restarts, 1e-15)
    with FieldSolver(c.n, c.length) as s:
        s.set_case(c)
        x = ghosted(x0)
        s.gmres(b, x, m=m, restarts=restarts, tol=1e-15, precond=0)
    assert np.array_equal(x[1:-1, 1:-1, 1:-1], ref[1:-1, 1:-1, 1:-1])


def gmres_dense(A, n, b, x0, m, tol):
    """One restart of performgmres with gseidel_precond on explicit rows."""
    nx, ny, nz = n
    cells = [(i, j, k) for k in range(nz) for j in range(ny) for i in range(nx)]
    nb = [[q + d if 0 <= c[a] + s < n[a] else None for a, d in ((0, 1), (1, nx), (2, nx * ny)) for d, s in ((-d, -1), (d, 1))]
          for q, c in enumerate(cells)]
    N = len(cells)

    def off(v, q):
        o = 0.0
        for r in nb[q]:
            if r is not None:
                o = o + A[q, r] * v[r]
        return o

    def apply(v):
        return [A[q, q] * v[q] + off(v, q) for q in range(N)]

    def precond(v):
        out = [0.0] * N
        for colour in (1, 0):   # cell (1, 1, 1) is red
            for q, c in enumerate(cells):
                if (sum(c) + 3) % 2 == colour:
                    out[q] = (v[q] - off(out, q)) / A[q, q]
        return out

    def dot(a, c):
        t = 0.0
        for p, r in zip(a, c):
            t = t + p * r
        return t

    r = precond([p - q for p, q in zip(b, apply(x0))])
    beta = math.sqrt(dot(r, r))
    V, H, cs, be = [[p / beta for p in r]], [], [], [beta]
    for kd in range(m):
        w = precond(apply(V[kd]))
        h = [dot(w, v) for v in V]
        for hv, v in zip(h, V):
            w = [p - hv * q for p, q in zip(w, v)]
        hn = math.sqrt(dot(w, w))
        assert hn > 1e-25
        V.append([p / hn for p in w])
        h.append(hn)
        for i, (c, s) in enumerate(cs):
            h[i], h[i + 1] = c * h[i] + s * h[i + 1], -s * h[i] + c * h[i + 1]
        d = math.sqrt(h[kd] * h[kd] + h[kd + 1] * h[kd + 1])
        c, s = h[kd] / d, h[kd + 1] / d
        h[kd] = c * h[kd] + s * h[kd + 1]
        cs.append((c, s))
        be[kd], nxt = c * be[kd], -s * be[kd]
        be.append(nxt)
        H.append(h)
    y = [0.0] * m
    for i in range(m - 1, -1, -1):
        t = be[i]
        for j in range(i + 1, m):
            t = t - H[j][i] * y[j]
        y[i] = t / H[i][i]
    x = list(x0)
    for j in range(m):
        x = [p + y[j] * q for p, q in zip(x, V[j])]
    return x


@pytest.mark.parametrize("n,m", [((4, 3, 2), 24), ((4, 4, 4), 30)])
def test_one_wave_gmres_on_explicit_rows(gpu, n, m):
    c = W.random_cdr(n, seed=3)
    rng = np.random.default_rng(6)
    b, x0 = rng.standard_normal(n), rng.standard_normal(n)
    N = b.size
    with FieldSolver(c.n, c.length, flux="sg") as s:
        s.set_case(c)
        A = np.empty((N, N))
        for q in range(N):
            e = np.zeros(N)
            e[q] = 1.0
            A[:, q] = s.find_AX(ghosted(e.reshape(n, order="F")))[0].ravel(order="F")
        x = ghosted(x0)
        s.gmres(b, x, m=m, restarts=1, tol=1e-15, precond=0)
    ref = gmres_dense(A, n, b.ravel(order="F").tolist(), x0.ravel(order="F").tolist(), m, 1e-15)
    assert np.array_equal(x[1:-1, 1:-1, 1:-1].ravel(order="F"), np.array(ref))

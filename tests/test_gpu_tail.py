"""The small levels of the reference hierarchy's V-cycle in two launches
(k_tail_down, k_tail_up): solutions after whole cycles bit for bit the
oracle's perform_vcycle where the arithmetic is exact (every operation in
the reference's order), with and without convection and reaction, with
Dirichlet faces in the prolongation's ghost rule, for levels from two cells a
side to the largest that the launches take over (16^3) and grids one level
above it, coarsest grids of odd sizes, and grids whose finest level is
already small. Fast rows and explicit (Scharfetter-Gummel) rows against the
exact cycle of the same operator: residual histories within 1e-6 of the
initial residual (rows that differ by rounding, or by the harmonic mean's
1e-10 guard, in a contracting cycle)."""
import numpy as np
import pytest

from mps3d_amd import FieldSolver
from mps3d_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

GRIDS = [((2, 2, 2), (1, 1, 1)), ((4, 8, 2), (1, 2, 1)), ((8, 8, 8), (1, 1, 1)), ((12, 8, 20), (3, 2, 5)),
         ((16, 16, 16), (2, 2, 2)), ((16, 16, 16), (1, 1, 1)), ((24, 16, 8), (3, 2, 1)), ((32, 16, 16), (2, 1, 1)),
         ((32, 32, 16), (2, 4, 1)), ((4, 4, 256), (1, 1, 64))]
CODES = ("DIRC", "FLUX", "ZGRD", "DIRC", "DIRC", "ZGRD")


@pytest.mark.parametrize("n,p", GRIDS)
@pytest.mark.parametrize("form", ["cdr", "convection", "reaction", "diffusion"])
def test_exact_cycles_equal_the_oracle(gpu, n, p, form):
    c = W.random_cdr(n, seed=5 + sum(n), codes=CODES)
    if form in ("reaction", "diffusion"):
        c.velx = c.vely = c.velz = None
    if form in ("convection", "diffusion"):
        c.reac = None
    P = O.Problem(c.n, c.length, p, c.bc_codes, c.bc_vals, c.dcoeff, c.velx, c.vely, c.velz, c.reac, c.source,
                  c.timederiv, c.dt)
    ref, _ = O.solve(P, P.zeros(), 3, 0.0)
    with FieldSolver(c.n, c.length, p, max_cycles=3, tol=0.0) as s:
        s.set_case(c)
        u = np.zeros(s.shape, order="F")
        s.solve(u)
    assert np.array_equal(u[1:-1, 1:-1, 1:-1], ref[1:-1, 1:-1, 1:-1])


@pytest.mark.parametrize("n,p", GRIDS[2:])
@pytest.mark.parametrize("form", ["fast", "fast_reaction", "sg", "fp32dc"])
def test_fast_and_explicit_rows_follow_the_exact_cycle(gpu, n, p, form):
    c = W.random_cdr(n, seed=9 + sum(n), codes=CODES)
    c.velx = c.vely = c.velz = None
    c.dcoeff = np.ones(n)
    c.reac = -np.abs(c.reac) if form == "fast_reaction" else None
    kw = {"sg": dict(flux="sg"), "fp32dc": dict(arith="fast", precision="fp32dc", dc_inner=1)}.get(form, dict(arith="fast"))
    hist = []
    for k in (dict(), kw):
        with FieldSolver(c.n, c.length, p, max_cycles=3, tol=0.0, tol_kind="rel", **k) as s:
            s.set_case(c)
            u = np.zeros(s.shape, order="F")
            hist.append(s.solve(u)[2])
    # (FP32 cycles: 1e-5 of the residual they start from)
    assert np.max(np.abs(hist[0] - hist[1])) <= (1e-4 if form == "fp32dc" else 1e-6)

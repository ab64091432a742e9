"""FGMRES preconditioned by one V-cycle on the device: its Gram-Schmidt passes
keep the products with the first four vectors in registers and take further
ones in passes of their own, so solves of one to some ten steps and restarts
after one to six are run, in every operator form and precision, from a zero
guess and from another, to the residual of the operator that find_AX gives.
Bar: the tolerance asked for, with a margin of 1 % for the two residuals'
rounding (1e-16 relative to |A||x| against tolerances of 1e-9 |b|)."""
import numpy as np
import pytest
import torch

from mps3d_amd import FieldSolver, ghosted
from mps3d_amd import workloads as W

pytestmark = pytest.mark.gpu


def solver(n, form, prec, hier):
    c = W.varcoef_poisson(n)
    c.length = tuple(0.02 * m / max(n) for m in n)
    kw = {}
    if form != "diffusion":
        c.dcoeff = np.full(n, 100.0, order="F")
        c.velx, c.vely, c.velz = (np.full(n, v, order="F") for v in (1e4, -2e4, 3e4))
        c.timederiv, c.dt = True, 1e-6
    if form == "sg":
        kw["flux"] = "sg"
    if form == "reac":
        c.velx = c.vely = c.velz = None
        c.reac = np.full(n, -3.0e4, order="F")
    s = FieldSolver(c.n, c.length, hierarchy=hier, precision=prec, arith="fast" if prec == "fp32dc" else "exact",
                    **kw)
    s.set_case(c)
    s.set_bc(c.bc_codes, (0.0,) * 6)
    return s


@pytest.mark.parametrize("n", [(16, 16, 16), (17, 9, 33), (64, 32, 32), (65, 33, 65)])
@pytest.mark.parametrize("form", ["diffusion", "upwind", "sg", "reac"])
@pytest.mark.parametrize("prec", ["fp64", "fp32dc"])
def test_residual_meets_the_tolerance(gpu, n, form, prec):
    hier = "aligned" if n[0] % 2 else "ref"
    if hier == "aligned" and form == "upwind":
        pytest.skip("the aligned hierarchy discretises convection by Scharfetter-Gummel fluxes")
    b = np.random.default_rng(7).standard_normal(n)
    bd = torch.from_numpy(np.ascontiguousarray(b.T)).cuda()
    counts = []
    with solver(n, form, prec, hier) as s:
        for tol, m in ((1e-3, 30), (1e-9, 30), (1e-9, 6), (1e-6, 1), (1e-9, 2)):
            for guess in (0.0, 1.0):
                x = torch.full(tuple(v + 2 for v in n)[::-1], 0.0, dtype=torch.float64, device="cuda")
                x[1:-1, 1:-1, 1:-1] = 1e-4 * guess
                k, r, st = s.gmres(bd, x, m=m, restarts=60, tol=tol)
                assert st == 0, (tol, m, k, r)
                xn = x[1:-1, 1:-1, 1:-1].cpu().numpy().T
                ax = s.find_AX(ghosted(xn))[0]
                assert np.linalg.norm(b - ax) <= 1.01 * tol * np.linalg.norm(b)
                counts.append(k)
        x.zero_()
        assert s.gmres(torch.zeros_like(bd), x, tol=1e-9) == (0, 0.0, 0)
    assert min(counts) <= 4 < max(counts) or prec == "fp64"

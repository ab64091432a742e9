"""The coarsest inverse on the context's second stream: set-ups and solves
queued back to back, with new velocities each time, give what the same calls
give with the device idle between them, bit for bit; coarsest grids of 48 to
210 cells, on both sides of the 64 from which the second stream is used."""
import pytest
import torch

from mps3d_amd import FieldSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(25, 17, 21), (65, 33, 49), (13, 15, 11)])
@pytest.mark.parametrize("prec", ["fp64", "fp32dc"])
def test_back_to_back_setups(gpu, n, prec):
    shape = tuple(v + 2 for v in n)[::-1]
    g = torch.Generator(device="cuda").manual_seed(11)
    new = lambda s=1.0: s * (torch.rand(shape, generator=g, dtype=torch.float64, device="cuda") - 0.5)  # noqa: E731
    D = torch.full(shape, 100.0, dtype=torch.float64, device="cuda")
    sets = [[new(1e5) for _ in range(3)] + [new()] for _ in range(6)]
    out = []
    with FieldSolver(n, tuple(0.02 * v / max(n) for v in n), hierarchy="aligned", flux="sg", precision=prec,
                     max_cycles=2, tol=0.0) as s:
        s.set_bc(("ZGRD",) * 4 + ("DIRC",) * 2, (0.0,) * 6)
        for idle in (False, True):
            for vx, vy, vz, b in sets:
                s.set_coeffs(D, vx, vy, vz, None, b, True, 1e-9)
                if idle:
                    torch.cuda.synchronize()
                x = torch.zeros(shape, dtype=torch.float64, device="cuda")
                s.solve(x)
                out.append(x.clone())
    assert all(torch.equal(a, b) for a, b in zip(out[:6], out[6:]))


@pytest.mark.parametrize("n,cells", [((25, 25, 25), 64), ((33, 17, 41), 90), ((33, 17, 65), 135), ((49, 33, 25), 140)])
@pytest.mark.parametrize("prec", ["fp64", "fp32dc"])
def test_coarsest_grids_of(gpu, n, cells, prec):
    c = n
    while min(c) > 3 and all(v % 2 for v in c):
        c = tuple((v + 1) // 2 for v in c)
    assert c[0] * c[1] * c[2] == cells
    test_back_to_back_setups(gpu, n, prec)

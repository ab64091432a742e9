"""Rows of calls ordered after torch's stream once (FieldSolver.chained): the
same results as the calls one by one, on torch's default stream and on one of
its own, with torch work still queued before the row; afterwards, and after
an error in a row, calls are ordered one by one again."""
import pytest
import torch

from mps3d_amd import FieldSolver
from mps3d_amd import _lib as M

pytestmark = pytest.mark.gpu
F64 = torch.float64


def rows(s, n, chained, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    new = lambda: torch.rand(tuple(v + 2 for v in n)[::-1], generator=g, dtype=F64, device="cuda")  # noqa: E731
    x = torch.ones((2048, 2048), dtype=torch.float32, device="cuda")
    d, src, u = new(), new(), new()
    for _ in range(20):
        x = (x @ x) / 2048.0   # (stays one; keeps the stream busy before the fields are written)
    d = 1.0 + d + 0.0 * x[0, 0].to(F64)
    src.mul_(2.0)

    def calls():
        s.set_coeffs(d, None, None, None, None, src, False, 1.0)
        s.solve(u)
        s.fill_ghosts(u)

    if chained:
        with s.chained():
            calls()
    else:
        calls()
    return u * 2.0


@pytest.mark.parametrize("n", [(8, 8, 8), (32, 16, 32), (64, 64, 64)])
@pytest.mark.parametrize("own", [False, True])
def test_a_row_is_its_calls(gpu, n, own):
    st = torch.cuda.Stream() if own else torch.cuda.current_stream()
    with FieldSolver(n, (1.0, 1.0, 1.0), max_cycles=3, tol=0.0) as s, torch.cuda.stream(st):
        s.set_bc(("DIRC",) * 6, (0.0, 1.0, 0.0, 0.0, 0.0, 2.0))
        for seed in range(3):
            a, b = rows(s, n, False, seed), rows(s, n, True, seed)
            assert torch.equal(a, b)


def test_an_error_ends_the_row(gpu):
    n = (8, 8, 8)
    with FieldSolver(n, (1.0, 1.0, 1.0), max_cycles=3, tol=0.0) as s:
        s.set_bc(("DIRC",) * 6, (0.0,) * 6)
        with pytest.raises(M.MpsError):
            with s.chained():
                s.set_coeffs(None, None, None, None, None, None, True, 0.0)   # a time derivative without a step
        assert not s._chained and not s._torch_call
        a, b = rows(s, n, True, 5), rows(s, n, False, 5)
        assert torch.equal(a, b)

"""Rows of calls ordered after torch's stream once (FieldSolver.chained): the
same results as the calls one by one, on torch's default stream and on one of
its own, with torch work still queued before the row; afterwards, and after
an error in a row, calls are ordered one by one again. Boundary values given as
numbers, or as device faces written in the row, come after the row's earlier
calls."""
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


def busy(s):
    """Work of some milliseconds on the context's own stream: the calls of a
    row queued after it have not run when the next call of the row begins."""
    with torch.cuda.stream(torch.cuda.ExternalStream(s.lib.mps_stream(s._h))):
        x = torch.ones((2048, 2048), dtype=torch.float32, device="cuda")
        for _ in range(40):
            x = (x @ x) / 2048.0
    return x


PLATES = ("ZGRD",) * 4 + ("DIRC", "DIRC")


@pytest.mark.parametrize("own", [False, True])
def test_host_faces_come_after_the_calls_before_them(gpu, own):
    # ghosts of DIRC faces are 2 g - u: each fill takes the faces set before it
    n = (17, 9, 9)
    st = torch.cuda.Stream() if own else torch.cuda.current_stream()
    with FieldSolver(n, (1.0, 1.0, 1.0), hierarchy="aligned") as s, torch.cuda.stream(st):
        u = [torch.zeros(tuple(v + 2 for v in n)[::-1], dtype=F64, device="cuda") for _ in range(4)]
        s.set_bc(PLATES, (0.0,) * 4 + (1.0, 2.0))
        keep = []
        torch.cuda.synchronize()
        with s.chained():
            for q, t in enumerate(u):
                keep.append(busy(s))
                s.fill_ghosts(t)
                s.set_bc(PLATES, (0.0,) * 4 + (float(q + 2), 2.0 * (q + 2)))
        torch.cuda.synchronize()
        for q, t in enumerate(u):
            assert torch.all(t[0, 1:-1, 1:-1] == 2.0 * (q + 1)) and torch.all(t[-1, 1:-1, 1:-1] == 4.0 * (q + 1))


@pytest.mark.parametrize("hierarchy,precision", [("aligned", "fp64"), ("ref", "fp64"), ("ref", "fp32dc")])
def test_a_face_written_in_the_row_reaches_a_mixed_set(gpu, hierarchy, precision):
    # the thermal outflow of a FLUX face beside five numbers, ghosts and right-
    # hand side from it, as the same calls one by one give them
    n = (17, 9, 9) if hierarchy == "aligned" else (16, 8, 8)
    codes = ("ZGRD",) * 4 + ("DIRC", "FLUX")
    g = torch.Generator(device="cuda").manual_seed(4)
    ne, te = (0.5 + torch.rand(tuple(v + 2 for v in n)[::-1], generator=g, dtype=F64, device="cuda") for _ in range(2))
    out = []
    with FieldSolver(n, (1.0, 1.0, 1.0), hierarchy=hierarchy, precision=precision, max_cycles=3, tol=0.0) as s:
        s.set_bc(codes)
        s.set_coeffs(torch.ones_like(ne))
        for chained in (False, True):
            face, u, keep = torch.zeros((n[1], n[0]), dtype=F64, device="cuda"), torch.zeros_like(ne), None
            torch.cuda.synchronize()
            if chained:
                with s.chained():
                    keep = busy(s)
                    s.eden_faces(codes, ne, te, 1e-3, [None] * 5 + [face])
                    s.set_bc(codes, [0.0] * 4 + [3.0, face])
                    s.solve(u)
                    s.fill_ghosts(u)
            else:
                s.eden_faces(codes, ne, te, 1e-3, [None] * 5 + [face])
                s.set_bc(codes, [0.0] * 4 + [3.0, face])
                s.solve(u)
                s.fill_ghosts(u)
            out.append((face, u, torch.from_numpy(s.find_bvec())))
            del keep
    assert float(out[0][0].abs().min()) > 0.0
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.parametrize("chem", ["ion_elec", "h2_o2"])
def test_a_plasma_step_launches_nothing_of_torchs_in_its_rows(gpu, chem):
    # nothing but views, also where faces and densities are strided; and the
    # same fields as from contiguous ones
    from torch.utils._python_dispatch import TorchDispatchMode

    from mps3d_amd import chemistry, plasma
    deck, make = {"ion_elec": (plasma.ION_ELEC_DECK, chemistry.ion_elec),
                  "h2_o2": (plasma.H2_O2_DECK, chemistry.h2_o2)}[chem]

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            if any(s is not None and s._chained for s in contexts) and not func.is_view:
                seen.append(str(func))
            return func(*args, **(kwargs or {}))

    out, seen = [], []
    for strided in (False, True):
        run = plasma.PlasmaRun(dict(deck, n=(16, 16, 16), p=(2, 2, 1)), make())
        contexts = [run.pois, run.ener, run.elec, run.ion, run.neut]
        if strided:
            for faces in [run.faces["pot"]] + run.faces["ion"]:
                for k in range(6):
                    if not (faces is not run.faces["pot"] and run.codes["spec"][k] == "FLUX"):
                        faces[k] = faces[k].t().contiguous().t()
            wide = torch.zeros((2 * run.numden.shape[0],) + run.numden.shape[1:], dtype=F64, device="cuda")
            wide[::2] = run.numden
            run.numden = wide[::2]
        with Watch():
            for _ in range(2):
                run.step()
        out.append([run.numden.clone(), run.phi_s.clone(), run.E.clone(), run.Te.clone(), run.eps_s.clone()])
        run.close()
    assert seen == []
    for a, b in zip(*out):
        assert torch.equal(a, b)

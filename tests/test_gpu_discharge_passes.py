"""The library's field passes of a discharge step (mps_pad_fields,
mps_charge_rhs, mps_discharge_rhs) against the step built from tensor
operations: the right-hand sides and velocities that reach each solve. The
passes do the same operations in the same order without contraction, so the
bar is 1e-14 relative to the largest value (exp may differ by an ulp), and
bitwise for the padded fields. Where a step may not take the passes it does
not: gradients wanted, replaced methods, rates of the caller's, other
layouts. Operators of the caller's are called as they are where a step is
built from tensor operations."""
import pytest
import torch

from mps3d_amd import autograd as AG
from mps3d_amd import discharge as DS

pytestmark = pytest.mark.gpu
F64 = torch.float64


class Torch(DS.Discharge):
    """A subclass: its steps are built from tensor operations."""


def record(model):
    """Replaces the operators' solves; returns what they are given."""
    seen = []

    class Op:
        def __init__(self, scale):
            self.scale = scale

        def configure(self, vel=None, rhs=None, scale=1.0):
            vg = [] if vel is None else AG.pad_fields(vel, scale)
            seen.append([rhs.clone()] + [v.clone() for v in vg])
            self.rhs = rhs

        def solve(self, x0=None):
            return AG.pad(self.scale * self.rhs)

        advance = AG.Operator.advance

        def close(self):
            pass

    model.poisson = Op(1e-9 * model.h ** 2)
    model.ops = [Op(0.9 * model.dt) for _ in model.species]
    if model.energy:
        model.energy_op = Op(0.9 * model.dt)
    return seen


def build(cls, form, n):
    sp = [DS.Species("e", -1, 20.0, 100.0, mass=DS.M_E), DS.Species("A+", 1, 0.2, 0.01),
          DS.Species("A-", -1, 0.2, 0.01, electrode="ZGRD"), DS.Species("A*", 0, 0.0, 0.01)]
    re = [DS.Reaction(("e", "gas"), ("e", "e", "A+"), DS.arrhenius(1e-13, 15.0), energy=15.0),
          DS.Reaction(("A-", "A*"), ("e",), 1e-16), DS.Reaction(("gas",), ("A*",), 2.0),
          DS.Reaction(("e", "A+", "gas"), ("A*",), DS.arrhenius(3e-30, 1.0), energy=-2.0)]
    if form == "one":
        sp, re = sp[1:2], []
    el = DS.split_electrodes(n, n, "cuda") if form != "energy" else DS.plate_electrodes(n, n, "cuda")
    eps = 1.0 + torch.rand((n,) * 3, dtype=F64, generator=torch.Generator().manual_seed(3))
    return cls(n, 0.02, sp, re, el, energy=form == "energy", eps_r=eps)


def state(model, n):
    g = torch.Generator().manual_seed(n)
    f = [(1e12 + 1e16 * torch.rand((n,) * 3, dtype=F64, generator=g)).cuda() for _ in range(len(model.species) + 1)]
    return tuple(f[:-1]), (3.0 * f[-1] if model.energy else None)


@pytest.mark.parametrize("n", [4, 6, 17, 64, 65, 70])
@pytest.mark.parametrize("form", ["energy", "local", "one"])
def test_passes_equal_the_tensor_operations(gpu, n, form):
    out = []
    V = torch.tensor([800.0, -300.0], dtype=F64, device="cuda")
    for cls in (DS.Discharge, Torch):
        m = build(cls, form, n)
        solvers = [o for o in [m.poisson, *m.ops, getattr(m, "energy_op", None)] if o is not None]
        seen = record(m)
        dens, neps = state(m, n)
        assert (m._native(dens, neps, V) is not None) == (cls is DS.Discharge)
        for _ in range(2):
            new, neps = m.step(dens, neps, V)
            dens = tuple(d.clone() for d in new)
        out.append(seen)
        for o in solvers:
            o.close()
    assert len(out[0]) == len(out[1])
    for a, b in zip(*out):
        assert len(a) == len(b)
        for x, y in zip(a, b):
            assert float((x - y).abs().max()) <= 1e-14 * float(y.abs().max())


@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 4, 5), (2, 9, 63), (5, 3, 64), (4, 8, 131)])
def test_pad_fields(gpu, shape):
    f = [torch.randn(shape, dtype=F64, device="cuda") for _ in range(4)]
    for k in (1, 3, 4):
        for s in (1.0, -0.3):
            for got, t in zip(AG.pad_fields(f[:k], s), f[:k]):
                assert torch.equal(got, AG.pad(s * t))
    t = torch.randn(shape[::-1], dtype=F64, device="cuda").permute(2, 1, 0)   # not contiguous: tensor operations
    assert torch.equal(AG.pad_fields([t])[0], AG.pad(t))
    assert AG.pad_fields([f[0].float()])[0].dtype == torch.float32


def test_steps_that_stay_tensor_operations(gpu):
    m = build(DS.Discharge, "energy", 6)
    dens, neps = state(m, 6)
    V = torch.tensor([800.0], dtype=F64, device="cuda")
    assert m._native(dens, neps, V) is not None
    Vg = V.clone().requires_grad_()
    assert m._native(dens, neps, Vg) is None
    assert m._native((dens[0].clone().requires_grad_(),) + dens[1:], neps, V) is None
    with torch.no_grad():
        assert m._native(dens, neps, Vg) is not None
    assert m._native((dens[0].permute(2, 1, 0),) + dens[1:], neps, V) is None
    with torch.autograd.forward_ad.dual_level():
        assert m._native(dens, neps, V) is None
    m.solve_species = lambda k, rhs, vel, x0: rhs
    assert m._native(dens, neps, V) is None
    del m.solve_species
    m.reactions[0].rate = lambda eps: 1e-13 * torch.exp(-15.0 / eps)
    assert m._native(dens, neps, V) is None
    m.close()


def recorder(seen, factor):
    """configure and solve as LinearSolve calls them, with nothing else."""
    def configure(self, vel=None, rhs=None):
        seen.append([rhs.clone()] + [v.clone() for v in vel or ()])
        self.given = rhs

    def solve(self, x0=None):
        return AG.pad(factor * self.given)

    return configure, solve


@pytest.mark.parametrize("how", ["object", "subclass", "instance", "class"])
@pytest.mark.parametrize("form", ["energy", "local"])
def test_operators_of_the_callers(gpu, how, form, monkeypatch):
    n, out = 8, []
    V = torch.tensor([800.0, -300.0], dtype=F64, device="cuda")
    for cls in (DS.Discharge, Torch):
        m = build(cls, form, n)
        seen = []
        configure, solve = recorder(seen, 0.9 * m.dt)
        body = {"configure": configure, "solve": solve}
        ops = m.ops + ([m.energy_op] if m.energy else [])
        if how == "object":
            m.ops = [type("Op", (), body)() for _ in m.ops]
            if m.energy:
                m.energy_op = type("Op", (), body)()
        with monkeypatch.context() as mp:
            for op in ops:
                if how == "subclass":
                    op.__class__ = type("Op", (AG.Operator,), body)
                elif how == "instance":
                    op.configure, op.solve = configure.__get__(op), solve.__get__(op)
            if how == "class":
                for k, f in body.items():
                    mp.setattr(AG.Operator, k, f)
                m.poisson.__class__ = type("Op", (AG.Operator,), dict(body, solve=recorder(seen, 1e-9 * m.h ** 2)[1]))
            dens, neps = state(m, n)
            m.step(dens, neps, V)
        out.append(seen)
        for op in ops + [m.poisson]:
            op.close()
    assert len(out[0]) == len(out[1]) == len(ops) + (how == "class")
    # (where the potential is not replaced the velocities hold a solve to 1e-10)
    bar = 1e-14 if how == "class" else 1e-8
    for a, b in zip(*out):
        assert len(a) == len(b)
        for x, y in zip(a, b):
            assert float((x - y).abs().max()) <= bar * float(y.abs().max())


def test_methods_replaced_on_the_class(gpu, monkeypatch):
    m = build(DS.Discharge, "energy", 6)
    dens, neps = state(m, 6)
    V = torch.tensor([800.0], dtype=F64, device="cuda")
    for cls, name in [(DS.Discharge, k) for k in ("potential", "efield", "mean_energy", "rates", "thermal_outflow",
                                                  "solve_species", "solve_energy")] + [(DS.Reaction, "coefficient")]:
        with monkeypatch.context() as mp:
            old = getattr(cls, name)
            mp.setattr(cls, name, lambda *a, _f=old: _f(*a))
            assert m._native(dens, neps, V) is None, name
        assert m._native(dens, neps, V) is not None
    m.close()


def test_the_local_field_constants_are_read_where_they_are_used(gpu):
    # with the energy equation the mean energy takes none of them
    out = []
    for lfa in ((1.0, 5e4), None):
        m = build(DS.Discharge, "energy", 8)
        m.eps_lfa = lfa
        dens, neps = state(m, 8)
        out.append(m.step(dens, neps, torch.tensor([800.0], dtype=F64, device="cuda")))
        m.close()
    (a, ea), (b, eb) = out
    assert all(torch.equal(x, y) for x, y in zip(a + (ea,), b + (eb,)))


def gradients(m, n, V, every, extra=()):
    """A run of five steps: its end and the gradients of a sum over it."""
    dens, neps = state(m, n)
    dens = tuple(d.requires_grad_() for d in dens)
    m._phi = None
    out, end = m.run(V, 5, (dens, neps), checkpoint_every=every)
    out = out + ((end,) if m.energy else ())
    g = torch.Generator(device="cuda").manual_seed(2)
    J = sum((t * torch.rand(t.shape, generator=g, dtype=F64, device="cuda")).sum() for t in out)
    J = J + 1e-3 * float(J.detach()) / 1e6 * (m.potential_of((out[:len(dens)], None), V) ** 2).mean()
    return [t.detach() for t in out], torch.autograd.grad(J, [V, *dens, *extra])


@pytest.mark.parametrize("form", ["energy", "local"])
@pytest.mark.parametrize("every", [1, 2, 5])
def test_checkpointed_gradients(gpu, form, every, monkeypatch):
    # segments of native steps give the gradients of the steps kept whole. The
    # solves reach 1e-10 of their right-hand sides, so both hold to 1e-8 and
    # their gradients to some ten times that
    n, native = 8, []
    m = build(DS.Discharge, form, n)
    V = torch.tensor([800.0, -300.0], dtype=F64, device="cuda", requires_grad=True)
    step = DS.Discharge._native_step
    monkeypatch.setattr(DS.Discharge, "_native_step", lambda self, *a: native.append(1) or step(self, *a))
    end, want = gradients(m, n, V, 0)
    assert not native
    got_end, got = gradients(m, n, V, every)
    assert len(native) == 5
    for a, b in zip(list(got) + got_end, list(want) + end):
        assert float((a - b).abs().max()) <= 1e-7 * float(b.abs().max())
    m.close()


def test_what_else_wants_a_gradient_keeps_it(gpu):
    # a tensor that the electrodes' faces hold, a permittivity, a rate: their
    # segments are checkpointed as they are, and V may be a list
    n = 8
    V = torch.tensor([800.0, -300.0], dtype=F64, device="cuda", requires_grad=True)
    for what in ("faces", "rate", "eps_r"):
        m = build(DS.Discharge, "local", n)
        p = torch.ones((), dtype=F64, device="cuda", requires_grad=True)
        faces, rate, eps = m.faces, m.reactions[0].rate, m.eps_r
        if what == "faces":
            m.faces = lambda V_: tuple(p * f for f in faces(V_))
        elif what == "rate":
            m.reactions[0].rate = lambda e: p * rate(e)
        else:
            m.eps_r = p * eps
        assert not m._closed(V, state(m, n)[0])
        if what == "eps_r":
            m.eps_r = eps   # (its gradient would run through the potential's right-hand side only)
            m.close()
            continue
        _, want = gradients(m, n, V, 0, (p,))
        _, got = gradients(m, n, V, 2, (p,))
        for a, b in zip(got, want):
            assert float((a - b).abs().max()) <= 1e-7 * float(b.abs().max())
        m.close()
    m = build(DS.Discharge, "local", n)
    assert m._closed(V, state(m, n)[0])
    assert not m._closed([V[0], V[1]], state(m, n)[0])
    m.solve_poisson = lambda rhs: DS.Discharge.solve_poisson(m, rhs)
    assert not m._closed(V, state(m, n)[0])
    m.close()


def test_function_modes_see_the_tensor_operations(gpu):
    # as dispatch modes do; a default device is no such mode
    from torch.overrides import TorchFunctionMode

    class Hot(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            out = func(*args, **(kwargs or {}))
            return 2.0 * out if func is torch.exp else out

    out, V = [], torch.tensor([800.0], dtype=F64, device="cuda")
    for cls in (DS.Discharge, Torch):
        m = build(cls, "energy", 8)
        dens, neps = state(m, 8)
        with torch.device("cuda"):
            assert (m._native(dens, neps, V) is not None) == (cls is DS.Discharge)
        with Hot():
            native = m._native(dens, neps, V)
            new, end = m.step(dens, neps, V)
        out.append(new + (end,))
        m.close()
        assert native is None
    for a, b in zip(*out):
        assert torch.equal(a, b)

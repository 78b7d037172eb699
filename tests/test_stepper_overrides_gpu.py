"""Subclasses (and objects) that bring their own addlinearterm, substepsol or
update: the explicit steppers call them, and agree with the library's own
passes where they only pass on to them."""

import numpy as np
import pytest
import torch

import fourierflows_hip as ff
from fourierflows_hip import timesteppers as tst

pytestmark = pytest.mark.gpu

EPS = {np.float32: 2.0**-24, np.float64: 2.0**-53}
CALLS = {"RK4": {"addlinearterm": 4, "substepsol": 3, "update": 1},
         "FilteredRK4": {"addlinearterm": 4, "substepsol": 3, "update": 1},
         "AB3": {"addlinearterm": 1}, "FilteredAB3": {"addlinearterm": 1},
         "LSRK54": {"addlinearterm": 5}, "FilteredLSRK54": {"addlinearterm": 5}}


def _problem(stepper, T):
    g = ff.TwoDGrid(ff.HIP(), nx=32, Lx=2 * np.pi, ny=24, Ly=2 * np.pi, T=T)
    w = torch.zeros(24, 32, dtype=torch.float32 if T == np.float32 else torch.float64, device="cuda")

    def calcN(N, sol, t, clock, vars, params, grid):
        ff.ldiv(w, grid.rfftplan, sol)
        w.mul_(w)
        ff.mul(N, grid.rfftplan, w)

    p = ff.Problem(ff.Equation(-1e-2 * g.Krsq_host, calcN, g), stepper, 2.0**-10, g)
    rng = np.random.default_rng(1)
    w0 = torch.tensor(rng.standard_normal((24, 32))).to(w.dtype).cuda()
    ff.mul(p.sol, g.rfftplan, w0)
    return p


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("on", ["subclass", "object", "class"])
@pytest.mark.parametrize("stepper", list(CALLS))
def test_overrides_are_called(stepper, on, T, monkeypatch):
    p, q = _problem(stepper, T), _problem(stepper, T)
    ff.stepforward(q, 5)
    calls = {}

    def counting(name):
        inherited = getattr(tst.RK4TimeStepper, name)

        def fn(self, *args):
            calls[name] = calls.get(name, 0) + 1
            return inherited(self, *args)

        return fn

    fns = {name: counting(name) for name in ("addlinearterm", "substepsol", "update")}
    ts = p.timestepper
    if on == "subclass":
        ts.__class__ = type("Mine", (type(ts),), fns)
    elif on == "object":
        for name, fn in fns.items():
            setattr(ts, name, fn.__get__(ts))
    else:
        for name, fn in fns.items():
            monkeypatch.setattr(tst.RK4TimeStepper, name, fn)
    ff.stepforward(p, 5)
    assert calls == {k: 5 * n for k, n in CALLS[stepper].items()}
    # the same sums of at most six terms, rounded at the same places
    a, b = p.sol.to(torch.complex128), q.sol.to(torch.complex128)
    assert float(torch.linalg.vector_norm(a - b)) <= 5 * 5 * 16 * EPS[T] * float(torch.linalg.vector_norm(b))
    assert p.clock.t == q.clock.t and p.clock.step == q.clock.step == 5


def test_an_override_acts(monkeypatch):
    class Damped(tst.FilteredRK4TimeStepper):
        def update(self, sol, dt):
            super().update(sol, dt)
            sol.mul_(0.5)

    p, q = _problem("FilteredRK4", np.float64), _problem("FilteredRK4", np.float64)
    p.timestepper.__class__ = Damped
    ff.stepforward(p, 1)
    ff.stepforward(q, 1)
    assert float(torch.linalg.vector_norm(p.sol - 0.5 * q.sol)) <= 80 * 2.0**-53 * float(torch.linalg.vector_norm(q.sol))

"""An L that is not finite at modes outside the kept band, where the state is
zero: 0 L is NaN there on every path."""

import numpy as np
import pytest
import torch

import fourierflows_hip as ff

pytestmark = pytest.mark.gpu


def _finite(t):
    return torch.isfinite(t.real) & torch.isfinite(t.imag)


def _run(make, monkeypatch):
    out = []
    for plans in (False, True):
        if plans:
            monkeypatch.setenv("FFHIP_DISABLE_FUSED", "1")
        else:
            monkeypatch.delenv("FFHIP_DISABLE_FUSED", raising=False)
        p = make()
        ff.stepforward(p, 2)
        out.append(_finite(p.sol))
    return out


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("stepper", ["RK4", "FilteredRK4", "AB3", "LSRK54", "ForwardEuler"])
@pytest.mark.parametrize("nx", [64, 48])
def test_vorticity(nx, stepper, T, monkeypatch):
    def make():
        g = ff.TwoDGrid(ff.HIP(), nx=nx, Lx=2 * np.pi, T=T)
        L = -1e-3 * g.Krsq_host
        L[nx // 2, 2], L[1, nx // 2] = -np.inf, np.nan
        p = ff.Problem(ff.Equation(L, ff.VorticityOperator(g), g), stepper, 2.0**-8, g)
        p.sol.copy_(ff.vorticity_ic(g, seed=1))
        ff.dealias(p.sol, g)
        return p

    got, want = _run(make, monkeypatch)
    assert not bool(got[nx // 2, 2]) and not bool(got[1, nx // 2])
    assert torch.equal(got, want)


@pytest.mark.parametrize("T", [np.float32, np.float64])
def test_tracer(T, monkeypatch):
    def make():
        g = ff.ThreeDGrid(ff.HIP(), nx=24, Lx=2 * np.pi, T=T)
        L = -1e-2 * g.Krsq_host
        L[12, 2, 3], L[1, 2, 12] = np.inf, np.nan
        p = ff.Problem(ff.Equation(L, ff.TracerOperator(g), g), "RK4", 2.0**-8, g)
        p.sol[1, 2, 3] = 1 + 2j
        return p

    got, want = _run(make, monkeypatch)
    assert not bool(got[12, 2, 3]) and not bool(got[1, 2, 12])
    assert torch.equal(got, want)

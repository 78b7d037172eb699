"""An infinity or NaN in one mode of the ABC-flow tracer: the stencil over
modes leaves what the transforms leave, and the runs after it are clean."""

import numpy as np
import pytest
import torch

import fourierflows_hip as ff

pytestmark = pytest.mark.gpu


def _problem(T, monkeypatch, transforms):
    if transforms:
        monkeypatch.setenv("FFHIP_DISABLE_FUSED", "1")
    else:
        monkeypatch.delenv("FFHIP_DISABLE_FUSED", raising=False)
    g = ff.ThreeDGrid(ff.HIP(), nx=24, ny=20, nz=32, Lx=2 * np.pi, x0=0.3, y0=-1.0, z0=0.0, T=T)
    op = ff.TracerOperator(g, 1.0, 0.7, -0.4)
    return ff.Problem(ff.Equation(-0.01 * g.Krsq_host, op, g), "RK4", 2.0**-8, g)


def _finite(t):
    return torch.isfinite(t.real) & torch.isfinite(t.imag)


# (m, l, kx): the mean, the kx = 0 plane, the inside and the edge of the band, outside it
MODES = [(0, 0, 0), (3, -2, 0), (2, 1, 5), (-10, 6, 7), (0, 0, 12), (16, 3, 2)]


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("value", [complex("nan+nanj"), complex("inf"), complex(1, float("inf"))])
@pytest.mark.parametrize("mode", MODES)
def test_non_finite_mode(T, value, mode, monkeypatch):
    ps, pt = _problem(T, monkeypatch, False), _problem(T, monkeypatch, True)
    rng = np.random.default_rng(1)
    z = torch.tensor(rng.standard_normal(ps.sol.shape) + 1j * rng.standard_normal(ps.sol.shape)).to(ps.sol.dtype).cuda()
    bad = z.clone()
    bad[mode] = value
    N, clean = {}, {}
    for p in (ps, pt):
        p.sol.copy_(z)
        ff.stepforward(p, 2)
        clean[p] = p.sol.clone()
        N[p] = torch.zeros_like(z)
    for nsteps in (1, 3):
        for p in (ps, pt):
            p.eqn.calcN(N[p], bad, 0.0)
            p.sol.copy_(bad)
            ff.stepforward(p, nsteps)
        assert torch.equal(_finite(N[ps]), _finite(N[pt]))
        assert torch.equal(_finite(ps.sol), _finite(pt.sol))
        assert mode == (0, 0, 0) or not bool(_finite(ps.sol)[mode])
        for p in (ps, pt):  # nothing of it stays
            p.sol.copy_(z)
            ff.stepforward(p, 2)
            assert torch.equal(p.sol, clean[p])
            p.eqn.calcN(N[p], z, 0.0)
            assert bool(_finite(N[p]).all())


@pytest.mark.parametrize("T", [np.float32, np.float64])
def test_mode_that_overflows_during_a_run(T, monkeypatch):
    """A state that is finite at the start and not at a later step."""
    top = float(np.finfo(T).max)
    out = []
    for transforms in (False, True):
        p = _problem(T, monkeypatch, transforms)
        p.sol.zero_()
        p.sol[2, 1, 5] = top / 8
        p.clock.dt = type(p.clock.dt)(64)
        ff.stepforward(p, 6)
        out.append(_finite(p.sol))
    assert not bool(out[0][2, 1, 5])
    assert torch.equal(out[0], out[1])

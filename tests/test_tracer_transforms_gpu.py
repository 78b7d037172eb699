"""The fused RK4 tracer on a box that is no multiple of 2 pi, where the
transforms run (on multiples of 2 pi the stencil over modes does): against the
oracle and the plan-based path, forward and as the map whose transpose the
fused adjoint is."""

import numpy as np
import pytest
import torch

from oracle import grids as og
from oracle import ics as oics
from oracle import physics as oph
from oracle import timesteppers as ots

import fourierflows_hip as ff
from fourierflows_hip import _lib

pytestmark = pytest.mark.gpu

L = 1.5 * 2 * np.pi
EPS = {np.float32: 2.0**-24, np.float64: 2.0**-53}


def _problem(n, T, monkeypatch, transforms="fused", **kw):
    if transforms == "plans":
        monkeypatch.setenv("FFHIP_DISABLE_FUSED", "1")
    p = ff.TracerProblem(n=n, L=L, T=T, **kw)
    monkeypatch.delenv("FFHIP_DISABLE_FUSED", raising=False)
    assert p.eqn.calcN.fused == (transforms == "fused")
    return p


def _run(p, nsteps, fused):
    """Steps p and checks which kernels that took."""
    _lib.profile_start()
    ff.stepforward(p, nsteps)
    names = {k["name"] for k in _lib.profile_stop()["kernels"]}
    assert not any(n.startswith("tracer_modes") for n in names)
    assert ({"tracer_y_inverse", "tracer_x", "tracer_y_forward", "tracer_z_stage4"} <= names) == fused


def _tol(n, T, nsteps, dt):
    """Relative L2: the four transforms of a stage at 8 eps per halving of the
    length each, times dt |u| kmax (|u| <= 2 sqrt(3)), on both sides, and four
    roundings of the state per step."""
    kmax = 2 * np.pi / L * n / 3 * np.sqrt(3)
    return 2 * nsteps * EPS[T] * (4 * 4 * 8 * 3 * np.log2(n) * dt * 3.5 * kmax + 8)


def test_oracle(monkeypatch):
    n, kappa, dt, steps = 64, 2e-3, 0.01, 8
    p = _problem(n, np.float64, monkeypatch, kappa=kappa, dt=dt)
    o = og.ThreeDGrid(n, L, x0=0, y0=0, z0=0)
    params = oph.TracerParams(kappa=kappa)
    rng = np.random.default_rng(4)
    c0 = o.mul(oics.tracer_ic(o, seed=5, ngauss=6, sigma=0.5))
    c0 += 1e-3 * (rng.standard_normal(c0.shape) + 1j * rng.standard_normal(c0.shape))  # aliased modes too
    c0[..., 0] = c0[..., 0].real
    want = ots.Problem(ots.Equation(oph.tracer_linear(o, kappa), oph.tracer_calcN, o), "RK4", dt, o,
                       oph.TracerVars(o, params), params)
    want.sol[...] = c0
    want.stepforward(steps)
    p.sol.copy_(torch.tensor(c0))
    _run(p, 3, True)
    _run(p, steps - 3, True)
    d = p.sol.cpu().numpy() - want.sol
    assert np.linalg.norm(d) <= _tol(n, np.float64, steps, dt) * np.linalg.norm(want.sol)


@pytest.mark.parametrize("n,T", [(64, np.float32), (128, np.float64), (256, np.float32)])
def test_plans(n, T, monkeypatch):
    dt, steps = 0.0025, 10
    ps = [_problem(n, T, monkeypatch, t, kappa=1e-3, dt=dt) for t in ("fused", "plans")]
    g = ps[0].grid
    s = torch.zeros_like(ps[0].sol)
    ff.mul(s, g.rfftplan, ff.tracer_ic(g, seed=2, ngauss=16, sigma=0.3))
    ff.dealias(s, g)
    for p, fused in zip(ps, (True, False)):
        p.sol.copy_(s)
        _run(p, steps, fused)
    a, b = (p.sol.to(torch.complex128) for p in ps)
    assert float(torch.linalg.vector_norm(a - b)) <= _tol(n, T, steps, dt) * float(torch.linalg.vector_norm(b))


def test_adjoint_is_the_transpose(monkeypatch):
    nsteps = 5
    p = _problem(64, np.float64, monkeypatch, kappa=1e-2, dt=0.01)
    gen = torch.Generator(device="cuda").manual_seed(11)
    d = torch.randn(p.sol.shape, generator=gen, device="cuda", dtype=torch.complex128)
    lam = torch.randn(p.sol.shape, generator=gen, device="cuda", dtype=torch.complex128)
    ff.dealias(d, p.grid)
    p.sol.copy_(d)
    _run(p, nsteps, True)
    out = torch.zeros_like(lam)
    _lib.call("ffhip_op_rk4_adjoint", p.eqn.calcN.handle, p.timestepper.handle, lam.data_ptr(), out.data_ptr(),
              p.clock.dt, nsteps, torch.cuda.current_stream().cuda_stream)

    def dot(a, b):
        return float(torch.sum(a.real * b.real + a.imag * b.imag))

    size = float(torch.linalg.vector_norm(d) * torch.linalg.vector_norm(out))
    assert abs(dot(p.sol, lam) - dot(d, out)) <= 2 * _tol(64, np.float64, nsteps, 0.01) * size

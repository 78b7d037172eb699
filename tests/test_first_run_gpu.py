"""The first run of a stepper, which makes its working arrays: on a stream of
the caller's own, and inside a caller's capture, where nothing may be
allocated."""

import ctypes as C

import numpy as np
import pytest
import torch

import fourierflows_hip as ff
from fourierflows_hip import _lib

pytestmark = pytest.mark.gpu


def _problem(nx, stepper, T):
    p = ff.TwoDVorticityProblem(nx=nx, nu=1e-3, dt=2.0**-8, stepper=stepper, T=T)
    p.sol.copy_(ff.vorticity_ic(p.grid, seed=3))
    return p


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("stepper", ["FilteredRK4", "AB3", "LSRK54", "ETDRK4"])
@pytest.mark.parametrize("nx", [64, 96, 512])
def test_first_run_on_a_side_stream(nx, stepper, T):
    p, q = _problem(nx, stepper, T), _problem(nx, stepper, T)
    ff.stepforward(p, 5)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ff.stepforward(q, 5)
    s.synchronize()
    assert torch.equal(p.sol, q.sol)


@pytest.mark.parametrize("stepper", ["RK4", "FilteredRK4", "FilteredLSRK54"])
@pytest.mark.parametrize("nx", [64, 48])
def test_first_explicit_run_under_capture(nx, stepper, monkeypatch):
    """With the stepper's scratch there, the first run of an operator can be
    captured: it replays to what the plan-based path computes."""
    monkeypatch.setenv("FFHIP_DISABLE_FUSED", "1")
    want = _problem(nx, stepper, np.float64)
    monkeypatch.delenv("FFHIP_DISABLE_FUSED")
    p = _problem(nx, stepper, np.float64)
    z = p.sol.clone()
    ff.stepforward(want, 4)
    N = torch.zeros_like(z)
    arr = C.c_void_p()
    for which in range(5):
        _lib.call("ffhip_rk4_scratch", p.timestepper.handle, which, C.byref(arr))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        p.sol.copy_(z)
        ff.stepforward(p, 4)
    for _ in range(3):
        p.sol.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(p.sol, want.sol)
        p.eqn.calcN(N, z, 0.0)  # eager work between the replays
    # and an eager run takes the fused passes afterwards
    p.sol.copy_(z)
    p.clock.step = 0
    ff.stepforward(p, 4)
    assert float(torch.linalg.vector_norm(p.sol - want.sol)) <= 1e-12 * float(torch.linalg.vector_norm(want.sol))

"""The array-kappa diffusion calcN writes its arrays in place: saved tensors
see that, and tensors that carry tangents take the array operations."""

import numpy as np
import pytest
import torch
import torch.autograd.forward_ad as fwd

import fourierflows_hip as ff

pytestmark = pytest.mark.gpu


def _problem(nx=64):
    p = ff.Diffusion.Problem(nx=nx, Lx=2 * np.pi, kappa=np.linspace(0.5, 1, nx), dt=1e-4, stepper="RK4")
    p.sol.copy_(torch.fft.rfft(torch.randn(nx, dtype=torch.float64, device="cuda")))
    return p


def test_written_arrays_count_as_written():
    p = _problem()
    N = torch.zeros_like(p.sol)
    before = [t._version for t in (p.vars.cx, p.vars.cxh, N)]
    assert ff.Diffusion._one_kernel(N, p.sol, p.vars, p.params, p.grid)
    assert all(t._version > v for t, v in zip((p.vars.cx, p.vars.cxh, N), before))
    x = torch.ones_like(N, requires_grad=True)
    y = (x * N).abs().sum()  # saves N
    p.eqn.calcN(N, p.sol, 0.0, p.clock, p.vars, p.params, p.grid)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward()


def test_tangents_take_the_array_operations():
    p = _problem()
    N = torch.zeros_like(p.sol)
    kernel = ff.Diffusion._one_kernel
    with fwd.dual_level():
        assert kernel(N, p.sol, p.vars, p.params, p.grid)  # none of them carries a tangent
        for name in ("sol", "kappa"):
            sol, kappa = p.sol, p.params.kappa
            if name == "sol":
                sol = fwd.make_dual(sol, torch.ones_like(sol))
            else:
                p.params.kappa = fwd.make_dual(kappa, torch.ones_like(kappa))
            assert not kernel(N, sol, p.vars, p.params, p.grid)
            p.params.kappa = kappa
    assert kernel(N, p.sol, p.vars, p.params, p.grid)


def test_inference_tensors():
    with torch.inference_mode():
        p = _problem()
        ff.stepforward(p, 2)
        q = _problem()
        q.sol.copy_(p.sol)
        N, M = torch.zeros_like(p.sol), torch.zeros_like(p.sol)
        p.eqn.calcN(N, p.sol, 0.0, p.clock, p.vars, p.params, p.grid)
        q.eqn.calcN(M, q.sol, 0.0, q.clock, q.vars, q.params, q.grid)
        assert torch.equal(N, M)

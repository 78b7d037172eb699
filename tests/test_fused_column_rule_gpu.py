"""FP64 columns of 512 points on both sides of the widths at which the column
stages leave the three-team kernels, against the plan-based path."""

import numpy as np
import pytest
import torch

import fourierflows_hip as ff

pytestmark = pytest.mark.gpu

EPS = 2.0**-53


# tiles of four kept columns: 240, 241, and (a quarter of the modes aliased) 384
@pytest.mark.parametrize("stepper", ["ETDRK4", "RK4"])
@pytest.mark.parametrize("nx,af", [(2880, 1 / 3), (2886, 1 / 3), (4096, 0.25)])
def test_matches_plans(nx, af, stepper, monkeypatch):
    ny, dt, steps = 512, 2.0**-13, 2
    out = []
    for plans in (False, True):
        if plans:
            monkeypatch.setenv("FFHIP_DISABLE_FUSED", "1")
        else:
            monkeypatch.delenv("FFHIP_DISABLE_FUSED", raising=False)
        p = ff.TwoDVorticityProblem(nx=nx, ny=ny, Ly=2 * np.pi, nu=1e-4, dt=dt, stepper=stepper, aliased_fraction=af)
        z = torch.zeros(ny, nx, dtype=torch.float64, device="cuda")
        rng = np.random.default_rng(1)
        x, y = (2 * np.pi * torch.arange(n, dtype=torch.float64, device="cuda") / n for n in (nx, ny))
        for k in range(1, 9):
            for l in range(-8, 9):
                z += rng.standard_normal() * torch.cos(k * x[None, :] + l * y[:, None] + 6 * rng.random()) / 12
        ff.mul(p.sol, p.grid.rfftplan, z)
        ff.stepforward(p, steps)
        out.append(p.sol.clone())
    # five transforms of 4 eps per halving of the length in each of eight
    # stages, on both sides, times dt kmax |u| < 1
    tol = 2 * 4 * steps * 5 * 4 * EPS * np.log2(nx * ny)
    assert float(torch.linalg.vector_norm(out[0] - out[1])) <= tol * float(torch.linalg.vector_norm(out[1]))

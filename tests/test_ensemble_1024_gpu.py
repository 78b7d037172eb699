"""Untuned ensembles with members of 1024 points: the variant they take, and
their steps against the single-grid kernels."""

import numpy as np
import pytest
import torch

import fourierflows_hip as ff

pytestmark = pytest.mark.gpu

EPS = {np.float32: 2.0**-24, np.float64: 2.0**-53}


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("sizes", [[(1024, 64)], [(64, 1024), (128, 128)], [(1024, 128), (64, 64), (512, 256)]])
def test_untuned(sizes, T):
    nu, dt, steps = 1e-3, 2.0**-10, 12
    ens = ff.VorticityEnsemble([{"nx": nx, "ny": ny, "nu": nu} for nx, ny in sizes], dt, T=T)
    threads, masks, _ = ens.info()
    assert threads == 256 and masks == 0  # 8 points per thread
    single = []
    for s, (nx, ny) in zip(ens.sols, sizes):
        p = ff.TwoDVorticityProblem(nx=nx, ny=ny, Ly=2 * np.pi, nu=nu, dt=dt, T=T)
        rng = np.random.default_rng(nx + ny)
        for k in range(1, 5):
            for l in range(-4, 5):
                p.sol[l, k] = nx * ny / 50 * complex(*rng.standard_normal(2))
        s.copy_(p.sol)
        ff.stepforward(p, steps)
        single.append(p.sol)
    ens.run(steps)
    for s, want, (nx, ny) in zip(ens.sols, single, sizes):
        # five transforms of 4 eps per halving of the length in each of four
        # stages a step, on both sides, times dt kmax |u| < 1
        tol = 2 * 4 * steps * 5 * 4 * EPS[T] * np.log2(nx * ny)
        a, b = s.to(torch.complex128), want.to(torch.complex128)
        assert float(torch.linalg.vector_norm(a - b)) <= tol * float(torch.linalg.vector_norm(b))

"""Gradients on the grids whose passes run three thread teams, and on those
beside them, against the adjoint of the oracle in 64 bits."""

import numpy as np
import pytest
import torch

from oracle import adjoint as oa
from oracle import grids as og
from oracle import physics as oph

import fourierflows_hip as ff

pytestmark = pytest.mark.gpu

EPS = {np.float32: 2.0**-24, np.float64: 2.0**-53}
F32, F64 = np.float32, np.float64


# rows and columns of every three-team length in both precisions, columns on
# both sides of the count up to which they run so (rows too), FP64 rows of 1024 that store
# the stage fields, and rows of many lines
@pytest.mark.parametrize("nx,ny,T", [(64, 256, F32), (256, 64, F32), (256, 256, F32), (256, 256, F64), (128, 64, F32),
                                     (64, 128, F32), (512, 512, F32), (1024, 512, F32), (2048, 512, F32),
                                     (1024, 64, F64), (512, 1024, F32), (512, 2048, F64), (2048, 128, F64)])
def test_gradient(nx, ny, T):
    nu, dt, nsteps, ncheck = 1e-3, 1e-3, 4, 2
    p = ff.TwoDVorticityProblem(nx=nx, ny=ny, nu=nu, dt=dt, T=T)
    g = p.grid
    o = og.TwoDGrid(nx, 2 * np.pi, ny, 2 * np.pi, x0=0, y0=0)
    rng = np.random.default_rng(nx + ny)
    x, y = o.x[None, :], o.y[:, None]
    z0, zobs = (sum(rng.standard_normal() * np.cos(k * x + l * y + 6 * rng.random())
                    for k in range(5) for l in range(-4, 5) if k or l > 0).astype(T) for _ in range(2))
    J, grad = ff.adjoint.misfit_gradient(p, torch.tensor(z0).cuda(), torch.tensor(zobs).cuda(), nsteps, ncheck)
    adj = oa.ETDRK4Adjoint(o, oph.vorticity_linear(o, nu=nu), dt)
    Jr, gr = adj.gradient(z0.astype(F64), zobs.astype(F64), nsteps, ncheck)
    # L2: in each of four stages a step, forward and back, ten transforms of 4
    # eps per halving of the length at most; the misfit is a sum of squares
    tol = 2 * 4 * nsteps * 10 * 4 * EPS[T] * np.log2(nx * ny)
    assert abs(J - Jr) <= 2 * tol * Jr
    assert np.linalg.norm(grad.cpu().numpy() - gr) <= tol * np.linalg.norm(gr)

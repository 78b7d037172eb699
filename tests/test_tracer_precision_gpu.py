"""N of the FP32 tracer on the stencil over modes: as exact as its one rounding."""

import numpy as np
import pytest
import torch

from oracle import grids as og
from oracle import physics as oph

import fourierflows_hip as ff

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("A,B,C,x0s", [(1, 1, 1, (0, 0, 0)), (1.1, 0.7, -0.4, (0.3, -1.1, 2.0)),
                                       (1 / 3, 1e-3, 7.7, (0.1, 0.2, 0.3))])
@pytest.mark.parametrize("n", [24, 64])
def test_rounded_once(n, A, B, C, x0s):
    g = ff.ThreeDGrid(ff.HIP(), nx=n, Lx=2 * np.pi, x0=x0s[0], y0=x0s[1], z0=x0s[2], T=np.float32)
    o = og.ThreeDGrid(n, 2 * np.pi, x0=x0s[0], y0=x0s[1], z0=x0s[2])
    sol = torch.tensor(o.mul(np.random.default_rng(n).standard_normal((n, n, n)))).to(torch.complex64).cuda()
    N = torch.empty_like(sol)
    ff.TracerOperator(g, A, B, C)(N, sol, 0.0)
    params = oph.TracerParams(A, B, C)
    want = np.zeros(N.shape, dtype=np.complex128)
    oph.tracer_calcN(want, sol.cpu().numpy().astype(np.complex128), 0.0, None, oph.TracerVars(o, params), params, o)
    # each component rounded once: 2^-24 of it at most
    assert np.linalg.norm(N.cpu().numpy() - want) <= 2.0**-24 * np.linalg.norm(want)

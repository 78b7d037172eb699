"""Rows of 8 complex points (16 reals), on both sides of the row counts at which
the kernels change, against NumPy in 64 bits."""

import numpy as np
import pytest
import torch

import fourierflows_hip as ff

pytestmark = pytest.mark.gpu

EPS = {np.float32: 2.0**-24, np.float64: 2.0**-53}


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("kind,nx", [("rfft", 16), ("fft", 8)])
@pytest.mark.parametrize("rows", [1, 63, 1000, (1 << 15) - 1, 1 << 15, (1 << 17) - 1, 1 << 17])
def test_rows(rows, kind, nx, T):
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((rows, nx))
    if kind == "fft":
        x = x + 1j * rng.standard_normal((rows, nx))
    x = x.astype(T if kind == "rfft" else np.result_type(T, np.complex64))
    want = (np.fft.rfft if kind == "rfft" else np.fft.fft)(x.astype(np.result_type(x, np.float64)), axis=1)
    plan = ff.Plan((nx,), T, kind, rows)
    xd = torch.tensor(x).cuda()
    X = torch.empty(want.shape, dtype=torch.complex64 if T == np.float32 else torch.complex128, device="cuda")
    back = torch.empty_like(xd)
    ff.mul(X, plan, xd)
    ff.ldiv(back, plan, X)
    tol = 4 * EPS[T] * np.log2(nx)  # L2: 4 eps per halving of the length at most
    assert np.linalg.norm(X.cpu().numpy().reshape(want.shape) - want) <= tol * np.linalg.norm(want)
    assert np.linalg.norm(back.cpu().numpy() - x) <= 2 * tol * np.linalg.norm(x)

"""Column passes over many slabs of few columns: transforms of both kinds
against NumPy in 64 bits."""

import numpy as np
import pytest
import torch

import fourierflows_hip as ff

pytestmark = pytest.mark.gpu

EPS = {np.float32: 2.0**-24, np.float64: 2.0**-53}


# slabs of one workgroup and of part of one, of a few, of seven, eight and more,
# with a batch of fields and as the planes of a 3D field; columns of 64 to 512
# points on both sides of 2048 in all
@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["rfft", "fft"])
@pytest.mark.parametrize("ns,batch", [((2, 16), 33), ((16, 16), 300), ((12, 20), 65), ((6, 96), 17), ((96, 96), 9),
                                      ((222, 48), 5), ((256, 30), 6), ((500, 12), 3), ((10, 14, 50), 1),
                                      ((16, 20, 9), 4), ((62, 64), 65), ((62, 128), 63), ((62, 512), 64),
                                      ((126, 256), 33)])
def test_transforms(ns, batch, kind, T):
    rng = np.random.default_rng(batch)
    shape = (batch,) + tuple(reversed(ns))
    x = rng.standard_normal(shape)
    if kind == "fft":
        x = x + 1j * rng.standard_normal(shape)
    x = x.astype(T if kind == "rfft" else np.result_type(T, np.complex64))
    axes = tuple(range(1, len(shape)))
    want = (np.fft.rfftn if kind == "rfft" else np.fft.fftn)(x.astype(np.result_type(x, np.float64)), axes=axes)
    plan = ff.Plan(ns, T, kind, batch)
    X = torch.empty(want.shape, dtype=torch.complex64 if T == np.float32 else torch.complex128, device="cuda")
    xd = torch.tensor(x).cuda()
    ff.mul(X, plan, xd)
    # L2: 4 eps per halving of the length at most (a direct prime factor below 64 counts as six)
    tol = 4 * EPS[T] * (np.log2(np.prod(ns)) + 6)
    assert np.linalg.norm(X.cpu().numpy() - want) <= tol * np.linalg.norm(want)
    back = torch.empty_like(xd)
    ff.ldiv(back, plan, X)
    assert np.linalg.norm(back.cpu().numpy() - x) <= 2 * tol * np.linalg.norm(x)

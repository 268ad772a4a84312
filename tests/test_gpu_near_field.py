"""The near field alone: in a tree of level 1 every leaf is a neighbour of
every other, so the matvec is the direct sum, in whichever way the leaf's size
and the columns choose.

Both sides sum the same products in FP64 in different orders: 2 (N + 32) 2^-53
sum |K w| bounds the difference (32 covers a value's own rounding).  The mixed
modes evaluate leaves of more than 16 points in FP32: 16 roundings of 2^-24
per value (r^2, its root, a Gaussian's argument of up to 8.4 and its
exponential) bound theirs."""
import numpy as np
import pytest

import pbbfmm3d_amd as pbb
from tests._helpers import gpu_matvec

pytestmark = pytest.mark.gpu

KERNELS = {"lap": (pbb.laplacian(), lambda r2: 1 / np.sqrt(r2)),
           "gauss": (pbb.gaussian(0.6), lambda r2: np.exp(-r2 / 0.36))}
# points of the 8 leaves: the edges of the leaf classes, of the 64-target
# passes (33..64 left, up to 32 left) and of the 32- and 64-source chunks
LEAVES = [(1, 0, 0, 0, 0, 0, 0, 0), (1, 2, 3, 4, 5, 8, 9, 16), (16, 17, 32, 33, 64, 0, 1, 2), (65, 96, 97, 128, 129, 200, 7, 31)]


def _case(name, leaves, ncols):
    kernel, f = KERNELS[name]
    rng = np.random.default_rng(sum(leaves) + ncols)
    x = [0.02 + 0.46 * rng.random((n, 3)) + 0.5 * np.array([b >> 2, b >> 1 & 1, b & 1]) for b, n in enumerate(leaves)]
    x[0][0] = 0.0  # the box of all points is the unit cube where its two corners are taken
    x[7][:1] = 1.0
    x = np.concatenate(x)
    w = rng.standard_normal((ncols, len(x)))
    r2 = ((x[None] - x[:, None]) ** 2).sum(-1)
    with np.errstate(divide="ignore"):
        k = f(r2)
    k[np.isinf(k)] = 0.0
    plan = pbb.Plan(pbb.Operators(kernel, 1.0, 1, 4, 1e-5), x)
    return plan, w, w @ k.T, np.abs(w) @ k.T


@pytest.mark.parametrize("ncols", [1, 2, 3, 5, 8, 9, 16, 17, 32, 35])
@pytest.mark.parametrize("leaves", LEAVES)
@pytest.mark.parametrize("name", list(KERNELS))
def test_level_one_is_the_direct_sum(gpu, name, leaves, ncols):
    plan, w, want, mag = _case(name, leaves, ncols)
    n = w.shape[1]
    got = gpu_matvec(plan, w, ncols).reshape(ncols, n)
    assert (np.abs(got - want) <= 2 * (n + 32) * 2.0**-53 * mag).all()


@pytest.mark.parametrize("ncols", [1, 8, 17, 35])
@pytest.mark.parametrize("name", list(KERNELS))
def test_mixed_modes(gpu, name, ncols):
    import torch
    plan, w, want, mag = _case(name, LEAVES[3], ncols)
    got = plan.matvec(torch.tensor(w, device="cuda"), precision=pbb.capi.PREC_MIXED_F16X2).cpu().numpy()
    assert (np.abs(got - want) <= 16 * 2.0**-24 * mag).all()

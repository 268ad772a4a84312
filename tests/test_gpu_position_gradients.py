"""The near part of the position gradients: in a tree of level 1 every leaf is
a neighbour of every other, so the gradient of psi^T A sigma is the direct
sum, in whichever way the leaf's size and the columns choose.

Both sides form s = sum_c psi_ic sigma_jc + sigma_ic psi_jc (2 C products) and
sum s K' d over N points in FP64 in different orders:
2 (N + 2 C + 64) 2^-53 sum |psi sigma| |K' d| bounds the difference (64 covers
K', with a Gaussian's argument of up to 8.4)."""
import numpy as np
import pytest

import pbbfmm3d_amd as pbb

pytestmark = pytest.mark.gpu

# K' : the gradient in the target is K' (source - target)
KERNELS = {"lap": (pbb.laplacian(), lambda r2: r2**-1.5),
           "soft": (pbb.soft_laplacian(1e-4), lambda r2: (r2 + 1e-4) ** -1.5),
           "gauss": (pbb.gaussian(0.6), lambda r2: 2 / 0.36 * np.exp(-r2 / 0.36))}
# points of the 8 leaves: the edges of the leaf classes, of the 32-target
# blocks and of the 16- and 64-source chunks
LEAVES = [(1, 0, 0, 0, 0, 0, 0, 1), (1, 2, 3, 4, 5, 8, 9, 16), (16, 17, 32, 33, 64, 0, 1, 2), (65, 96, 97, 128, 129, 200, 7, 31)]


@pytest.mark.parametrize("ncols", [1, 4, 5, 16, 17, 35])
@pytest.mark.parametrize("leaves", LEAVES)
@pytest.mark.parametrize("name", list(KERNELS))
def test_level_one_is_the_direct_gradient(gpu, name, leaves, ncols):
    import torch
    kernel, f = KERNELS[name]
    rng = np.random.default_rng(sum(leaves) + ncols)
    x = [0.02 + 0.46 * rng.random((n, 3)) + 0.5 * np.array([b >> 2, b >> 1 & 1, b & 1]) for b, n in enumerate(leaves)]
    x[0][0] = 0.0  # the box of all points is the unit cube
    x[7][0] = 1.0
    x = np.concatenate(x)
    n = len(x)
    sig, psi = rng.standard_normal((2, ncols, n))
    plan = pbb.Plan(pbb.Operators(kernel, 1.0, 1, 4, 1e-5), x)
    got = plan.grad_positions(torch.tensor(sig, device="cuda"), torch.tensor(psi, device="cuda")).cpu().numpy()
    d = x[None] - x[:, None]
    r2 = (d**2).sum(-1)
    with np.errstate(divide="ignore"):
        k = f(r2)
    k[r2 == 0] = 0.0
    s, mag = psi.T @ sig + sig.T @ psi, np.abs(psi).T @ np.abs(sig) + np.abs(sig).T @ np.abs(psi)
    want = ((s * k)[..., None] * d).sum(1)
    bound = ((mag * np.abs(k))[..., None] * np.abs(d)).sum(1)
    assert (np.abs(got - want) <= 2 * (n + 2 * ncols + 64) * 2.0**-53 * bound).all()

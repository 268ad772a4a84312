"""The direct sum against NumPy in FP64, at the edges of its workgroups (64
targets), waves (16 shares of a source slice), slices and column groups.

Both sides sum Ns products in FP64 in different orders: each is within
(Ns + c) units of 2^-53 of sum |K w|, where c covers a value's own rounding
(r^2, square root, division; an exponential carries its argument's, up to 10
here): 2 (Ns + 32) 2^-53 sum |K w| bounds the difference."""
import numpy as np
import pytest

import pbbfmm3d_amd as pbb
from tests._helpers import gpu_direct

pytestmark = pytest.mark.gpu

KERNELS = {
    "lap": (pbb.laplacian(), lambda r2: 1 / np.sqrt(r2)),
    "r2": (pbb.oneoverr2(), lambda r2: 1 / r2),
    "soft": (pbb.soft_laplacian(1e-4), lambda r2: 1 / np.sqrt(r2 + 1e-4)),
    "gauss": (pbb.gaussian(0.6), lambda r2: np.exp(-r2 / 0.36)),
    "exp": (pbb.exponential(0.3), lambda r2: np.exp(-np.sqrt(r2) / 0.3)),
}


def _want(f, t, s, w):
    r2 = ((s[None] - t[:, None]) ** 2).sum(-1)
    with np.errstate(divide="ignore"):
        k = f(r2)
    k[np.isinf(k)] = 0.0
    return (k @ w.T).T, (np.abs(k) @ np.abs(w).T).T


@pytest.mark.parametrize("name", list(KERNELS))
@pytest.mark.parametrize("nt,ns,ncols", [(1, 1, 1), (63, 15, 2), (64, 16, 4), (65, 17, 5), (3, 1023, 16),
                                         (130, 1024, 17), (200, 1537, 33), (700, 5000, 3)])
def test_against_numpy(gpu, name, nt, ns, ncols):
    kernel, f = KERNELS[name]
    rng = np.random.default_rng(nt + ns)
    t, s, w = rng.random((nt, 3)), rng.random((ns, 3)), rng.standard_normal((ncols, ns))
    s[: min(nt, ns) // 2] = t[: min(nt, ns) // 2]  # coincident points: 1/r is 0 there
    got = gpu_direct(kernel, t, s, w.reshape(-1), ncols).reshape(ncols, nt)
    want, mag = _want(f, t, s, w)
    assert (np.abs(got - want) <= 2 * (ns + 32) * 2.0**-53 * mag).all()


@pytest.mark.parametrize("r", [0.0, 1e-158, 1e-150, 1e-100, 1e-20, 1.0, 1e20, 1e100, 1e150, 1e160, np.inf, np.nan])
@pytest.mark.parametrize("name", ["lap", "soft"])
def test_range_of_the_inverse_root(gpu, name, r):
    """One pair on an axis over the range of FP64, down to squares below the
    normal numbers (4 units in the last place)."""
    kernel, f = KERNELS[name]
    got = gpu_direct(kernel, np.zeros((1, 3)), np.array([[r, 0.0, 0.0]]), np.ones(1), 1)[0]
    with np.errstate(divide="ignore", over="ignore"):
        want = f(np.float64(r) ** 2)
    want = 0.0 if np.isinf(want) else want
    assert np.isnan(got) if np.isnan(want) else abs(got - want) <= 4 * 2.0**-52 * abs(want)


def test_more_targets_than_one_launch_holds(gpu):
    """2^28 + 65 targets at 16 threads each: more than the 2^32 - 1 threads of
    a launch, and the remainders of a workgroup and of a range of targets."""
    import ctypes as C

    import torch
    from pbbfmm3d_amd import _capi as capi
    nt = 2**28 + 65
    print(f"case nt={nt}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(7)
    t = torch.rand(nt, 3, dtype=torch.float64, device="cuda", generator=g)
    s = torch.tensor([[0.25, 0.5, 0.75], [0.5, -1.0, 2.0]], dtype=torch.float64, device="cuda")
    w = torch.tensor([[1.0, -3.0]], dtype=torch.float64, device="cuda")
    out = torch.full((nt,), -1.0, dtype=torch.float64, device="cuda")
    d = pbb.quadric().desc()
    capi.check(capi.lib().pbb_direct_sum(C.byref(d), t.data_ptr(), nt, s.data_ptr(), 2, w.data_ptr(), 1,
                                         out.data_ptr(), None))
    torch.cuda.synchronize()
    for i in range(0, nt, 2**25):
        x = t[i:i + 2**25]
        k = [1 + ((x - s[j]) ** 2).sum(1) for j in (0, 1)]
        bound = 2 * (2 + 32) * 2.0**-53 * (k[0] + 3 * k[1])
        assert bool(((out[i:i + 2**25] - (k[0] - 3 * k[1])).abs() <= bound).all())

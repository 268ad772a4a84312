"""One very full leaf beside many of 33 points and more: the near field and
the gradients run as many passes of 64 targets as there are, whatever the
largest leaf holds.

The kernel 1 + r^2 is a polynomial, which the interpolation of order 4 gives
exactly, so matvec and gradients are moments of the points.  Both sides sum N
products in FP64 in different orders, and the far field keeps its operators to
1e-13 of their norm: (2 (N + 32) 2^-53 + 1e-12) sum |K w| bounds the
difference, and the same of sum |grad K| (|psi sigma| terms) the gradients'."""
import numpy as np
import pytest

import pbbfmm3d_amd as pbb

pytestmark = pytest.mark.gpu


def _points(level, per_leaf, extra, seed):
    """per_leaf points in every leaf of the unit cube, extra more in one."""
    rng = np.random.default_rng(seed)
    m = 1 << level
    cell = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 1, 3)
    x = (cell + 0.01 + 0.98 * rng.random((m**3, per_leaf, 3))) / m
    x[0, 0], x[-1, 0] = 0.0, 1.0  # the box of all points is the unit cube
    more = (cell[m**3 // 2 + 5] + 0.01 + 0.98 * rng.random((extra, 3))) / m
    return np.concatenate([x.reshape(-1, 3), more])


def _check(plan, xyz, ncols, seed):
    import torch
    n = len(xyz)
    x = torch.tensor(xyz, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.randn(ncols, n, dtype=torch.float64, device="cuda", generator=g)
    psi = torch.randn(ncols, n, dtype=torch.float64, device="cuda", generator=g)
    tol = 2 * (n + 32) * 2.0**-53 + 1e-12

    def sums(v):  # sum_j v_j (1 + |x_i - x_j|^2), per column
        return v.sum(1, keepdim=True) * (1 + (x * x).sum(1)) - 2 * (v @ x) @ x.T + (v @ (x * x).sum(1))[:, None]

    def grad(a, b):  # sum_c a_i sum_j 2 (x_i - x_j) b_j
        return 2 * ((a.T @ b.sum(1))[:, None] * x - a.T @ (b @ x))

    mag = 4 * w.abs().sum(1, keepdim=True)
    out = plan.matvec(w)
    assert bool(((out - sums(w)).abs() <= tol * mag).all())
    gx = plan.grad_positions(w, psi)
    gmag = 4 * (psi.abs().T @ w.abs().sum(1) + w.abs().T @ psi.abs().sum(1))
    assert bool(((gx - grad(psi, w) - grad(w, psi)).abs() <= tol * gmag[:, None]).all())
    return out, gx


# as many passes for every leaf as for the largest would be 67.6M workgroups
# of 64 threads, more than a launch holds
@pytest.mark.parametrize("ncols", [1, 9])
def test_one_leaf_of_132k_points(gpu, ncols):
    xyz = _points(5, 33, 132000, seed=410)
    print(f"case N={len(xyz)} ncols={ncols}", flush=True)
    plan = pbb.Plan(pbb.Operators(pbb.quadric(), 1.0, 5, 4, 1e-14), xyz)
    assert plan.info()["max_leaf_points"] == 132033
    _check(plan, xyz, ncols, seed=411)


@pytest.mark.parametrize("per_leaf,extra", [(31, 33), (33, 31), (40, 24), (40, 25), (1, 700), (64, 64), (65, 1)])
@pytest.mark.parametrize("ncols", [3, 17])
def test_passes_of_both_trees(gpu, per_leaf, extra, ncols):
    import torch
    xyz = _points(2, per_leaf, extra, seed=412)
    ops = pbb.Operators(pbb.quadric(), 1.0, 2, 4, 1e-14)
    a = _check(pbb.Plan(ops, xyz), xyz, ncols, seed=413)
    b = _check(pbb.Plan(ops, xyz, host_tree=True), xyz, ncols, seed=413)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])

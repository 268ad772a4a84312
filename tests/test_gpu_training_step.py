"""Both gradients of a training step from one transposed pass, with the
forward's leaf expansions kept or recomputed, against the separate calls
(pbb_plan_matvec_transpose, pbb_plan_grad_positions) on the same plan."""
import numpy as np
import pytest

import pbbfmm3d_amd as pbb
from pbbfmm3d_amd import _capi as capi
from tests._helpers import uniform_points

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float((a - b).norm() / b.norm())


# (N, level, order, columns): levels without and with a far field, orders on
# both sides of the direct passes' 4..8, one column and column blocks
@pytest.mark.parametrize("N,level,n,ncols", [(700, 1, 4, 2), (3001, 2, 3, 3), (4999, 3, 4, 1), (5000, 3, 5, 9),
                                             (2500, 3, 8, 2), (2000, 2, 9, 2)])
@pytest.mark.parametrize("prec", [capi.PREC_FP64, capi.PREC_MIXED_F16X2])
def test_gradients_from_one_transposed_pass(gpu, N, level, n, ncols, prec):
    import torch
    print(f"case N={N} level={level} order={n} ncols={ncols} precision={prec}", flush=True)
    if prec != capi.PREC_FP64 and not 4 <= n <= 8:
        pytest.skip("the mixed modes are tested at the direct orders")
    xyz = uniform_points(N, seed=90 + n)
    rng = np.random.default_rng(91)
    ops = pbb.Operators(pbb.gaussian(0.3), 1.0, level, n, 1e-7)
    plan, ref = pbb.Plan(ops, xyz), pbb.Plan(ops, xyz)
    sig = torch.tensor(rng.standard_normal((ncols, N)), device="cuda")
    psi = torch.tensor(rng.standard_normal((ncols, N)), device="cuda")
    out0, gw0 = ref.matvec(sig, precision=prec), ref.matvec_transpose(psi, precision=prec)
    gx0 = ref.grad_positions(sig, psi, precision=prec)
    out, kept = plan._matvec_keep(sig, prec)
    assert (kept is not None) == (prec == capi.PREC_FP64 and level >= 2)
    # the same sums in another order (transfers in place of direct passes);
    # the mixed modes' plain pass rounds its expansions to FP32 besides
    tol = 1e-12 if prec == capi.PREC_FP64 else 1e-5
    assert _rel(out, out0) < tol
    plan.matvec_transpose(psi, precision=prec)  # (the workspace between forward and gradient)
    for k in ([kept, None] if kept is not None else [None]):
        gw, gx = plan._gradients(sig, k, psi, prec, weights=True)
        assert _rel(gw, gw0) < tol and _rel(gx, gx0) < 1e-12
        none, gx = plan._gradients(sig, k, psi, prec, weights=False)
        assert none is None and _rel(gx, gx0) < 1e-12


def test_backward_of_two_forwards(gpu):
    """Two forwards of one plan before their backwards, and weights without
    or with a gradient: each backward uses its own forward's expansions."""
    import torch
    N, nc = 4000, 3
    xyz0 = uniform_points(N, seed=95)
    ops = pbb.Operators(pbb.soft_laplacian(1e-6), 1.0, 3, 5, 1e-7)
    plan = pbb.Plan(ops, xyz0)
    rng = np.random.default_rng(96)
    w = [torch.tensor(rng.standard_normal((nc, N)), device="cuda") for _ in range(2)]
    xyz = torch.tensor(xyz0, device="cuda", requires_grad=True)
    outs = [pbb.fmm_matvec(xyz, w[0], ops, plan=plan), pbb.fmm_matvec(xyz, w[1].requires_grad_(True), ops, plan=plan)]
    psi = [torch.tensor(rng.standard_normal((nc, N)), device="cuda") for _ in range(2)]
    for k in (0, 1):
        g = torch.autograd.grad(outs[k], (xyz, w[1])[:1 + k], psi[k])
        assert _rel(g[0], plan.grad_positions(w[k].detach(), psi[k])) < 1e-12
        if k:
            assert _rel(g[1], plan.matvec_transpose(psi[1])) < 1e-12

"""The FP64 M2L in the reflection-adapted bases against the M2L of the sets'
own factors, on the same plan and weights.

The plan's first matvec makes the adapted sets; the allocation-free matvec
before it still runs the own factors.  An adapted set is kept only when it
gives its operators back to 1e-13 of their norm, so the two matvecs differ by
rounding: 1e-11 bounds 1e-13 times the ratio of the operators' stacked norm
(where near and far directions add up) to an output's far field."""
import ctypes as C

import numpy as np
import pytest

import pbbfmm3d_amd as pbb
from pbbfmm3d_amd import _capi as capi
from pbbfmm3d_amd.FMMTree import myKernel
from tests._helpers import clustered_points, uniform_points

pytestmark = pytest.mark.gpu

# (kernel, order, eps): ranks from 22 to 313 and every row configuration;
# 1/r at order 5 and exp(-r) at order 6 cut a degenerate cluster, the Gaussian
# at order 6 has directions at the rounding level from level 4 down
KERNELS = {
    "aniso4": (myKernel.device_kernel, 4, 1e-5),
    "lap3": (pbb.laplacian(), 3, 1e-4),
    "lap4": (pbb.laplacian(), 4, 1e-5),
    "lap5": (pbb.laplacian(), 5, 1e-7),
    "exp5": (pbb.exponential(0.5), 5, 1e-7),
    "gauss5": (pbb.gaussian(0.3), 5, 1e-7),
    "exp6": (pbb.exponential(0.5), 6, 1e-7),
    "lap6": (pbb.laplacian(), 6, 1e-8),
    "gauss6": (pbb.gaussian(0.3), 6, 1e-8),
    "lap7": (pbb.laplacian(), 7, 1e-12),
}


def _noalloc(torch, plan, w):
    out = torch.zeros((w.shape[0], plan.ntargets), dtype=torch.float64, device=w.device)
    st = torch.cuda.current_stream().cuda_stream
    capi.check(capi.lib().pbb_plan_matvec_noalloc(plan._h, C.c_void_p(w.data_ptr()), w.shape[0],
                                                  C.c_void_p(out.data_ptr()), capi.PREC_FP64, C.c_void_p(st)))
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("name,level,points,n,ncols", [
    ("aniso4", 3, "uniform", 1500, 120),
    ("lap3", 3, "uniform", 2000, 7),
    ("lap4", 2, "uniform", 70, 1),
    ("lap4", 4, "clustered", 3001, 3),
    ("lap5", 4, "uniform", 4000, 1),
    ("lap5", 3, "uniform", 1111, 33),
    ("exp5", 4, "clustered", 1500, 5),
    ("gauss5", 4, "uniform", 600, 9),
    ("exp6", 3, "uniform", 801, 17),
    ("lap6", 4, "clustered", 1200, 2),
    ("gauss6", 5, "clustered", 900, 2),
    ("lap7", 3, "uniform", 900, 1),
])
def test_adapted_sets_equal_own_factors(gpu, name, level, points, n, ncols):
    import torch
    kernel, order, eps = KERNELS[name]
    print(f"case {name} level={level} {points} n={n} ncols={ncols}", flush=True)
    xyz = (uniform_points if points == "uniform" else clustered_points)(n, seed=300 + n)
    plan = pbb.Plan(pbb.Operators(kernel, 1.0, level, order, eps), xyz)
    g = torch.Generator(device="cuda").manual_seed(n)
    w = torch.randn(ncols, n, dtype=torch.float64, device="cuda", generator=g)
    own = _noalloc(torch, plan, w)
    got = plan.matvec(w)
    assert torch.equal(got, plan.matvec(w))
    rel = float((got - own).norm() / own.norm())
    print(f"  difference {rel:.2e}", flush=True)
    assert not torch.equal(got, own)  # the adapted sets ran
    assert rel <= 1e-11
    # column chunks of a small workspace give the same columns
    plan.set_workspace_limit(1)
    assert torch.equal(plan.matvec(w), got)


def test_separate_sources_and_transpose(gpu):
    import torch
    kernel, order, eps = KERNELS["exp5"]
    ops = pbb.Operators(kernel, 1.0, 4, order, eps)
    plan = pbb.Plan(ops, uniform_points(1301, seed=310), sources=clustered_points(777, seed=311))
    g = torch.Generator(device="cuda").manual_seed(312)
    w = torch.randn(3, 777, dtype=torch.float64, device="cuda", generator=g)
    y = torch.randn(3, 1301, dtype=torch.float64, device="cuda", generator=g)
    own = _noalloc(torch, plan, w)
    got = plan.matvec(w)
    assert float((got - own).norm() / own.norm()) <= 1e-11
    # <A w, y> = <w, A^T y>: the transposed operators find their own bases
    a, b = float((got * y).sum()), float((w * plan.matvec_transpose(y)).sum())
    assert abs(a - b) <= 1e-11 * float(got.norm() * y.norm())


def test_operators_without_the_symmetry_keep_their_factors(gpu):
    # one block of a homogeneous set perturbed: no orbit of its operators
    # holds, so the matvec is the own factors' bit for bit
    import torch
    kernel, order, eps = KERNELS["lap4"]
    ops = pbb.Operators(kernel, 1.0, 3, order, eps)
    U, VT, E, _, _ = ops.export()
    E = E.copy()
    blk = ops.rank_f * ops.rank_s
    E[17 * blk:18 * blk] *= 1.0 + 1e-6
    bent = pbb.Operators.from_arrays(kernel, 1.0, 3, order, eps, ops.rank_f, ops.rank_s, ops.nsets, U, VT, E)
    plan = pbb.Plan(bent, uniform_points(1500, seed=320))
    g = torch.Generator(device="cuda").manual_seed(321)
    w = torch.randn(2, 1500, dtype=torch.float64, device="cuda", generator=g)
    own = _noalloc(torch, plan, w)
    assert torch.equal(plan.matvec(w), own)


def test_tuner_times_the_own_factors(gpu):
    # FP64 tiles serve the sets' own factors, so the tuner runs these: it
    # leaves the adapted sets unmade, and the allocation-free matvec the same
    import torch
    kernel, order, eps = KERNELS["lap5"]
    plan = pbb.Plan(pbb.Operators(kernel, 1.0, 3, order, eps), uniform_points(3000, seed=330))
    g = torch.Generator(device="cuda").manual_seed(331)
    w = torch.randn(4, 3000, dtype=torch.float64, device="cuda", generator=g)
    own = _noalloc(torch, plan, w)
    plan.tune_m2l(w)
    plan.set_m2l_tile(0)
    assert torch.equal(_noalloc(torch, plan, w), own)
    assert not torch.equal(plan.matvec(w), own)


def test_small_ranks_of_many_columns_run_the_own_factors(gpu):
    # ranks below 16 in 7 parity classes: the own factors above 64 columns, the
    # whole call's (column chunks give the same bits)
    import torch
    ops = pbb.Operators(pbb.laplacian(), 1.0, 3, 4, 1e-2)
    assert ops.rank_f == ops.rank_s == 7
    plan = pbb.Plan(ops, uniform_points(1500, seed=340))
    g = torch.Generator(device="cuda").manual_seed(341)
    w = torch.randn(65, 1500, dtype=torch.float64, device="cuda", generator=g)
    own = _noalloc(torch, plan, w)
    adapted = plan.matvec(w[:64].contiguous())
    assert not torch.equal(adapted, own[:64])
    assert float((adapted - own[:64]).norm() / own.norm()) <= 1e-11
    assert torch.equal(plan.matvec(w), own)
    assert torch.equal(_noalloc(torch, plan, w), own)
    plan.set_workspace_limit(1)
    assert torch.equal(plan.matvec(w), own)

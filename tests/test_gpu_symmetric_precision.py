"""The reflection-adapted operators carry no more than rounding: the matvec in
them against the one of the sets' own factors on the same plan.

Weights are positive, so nothing cancels and an error of the operators shows
in the outputs.  The way into the adapted bases and out of them are products of
at most n^3 terms each, whose roundings add up as their square root: 8 products
(the blocks, their average, VT', U' and the two passes) of sqrt(n^3) units of
2^-53 bound the difference.  Operators rebuilt through the singular vectors'
transpose miss this by their loss of orthogonality (1e-14 at order 4, 2e-13 at
order 6)."""
import ctypes as C

import pytest

import pbbfmm3d_amd as pbb
from pbbfmm3d_amd import _capi as capi
from tests._helpers import uniform_points

pytestmark = pytest.mark.gpu

KERNELS = {"const": pbb.constant(), "quadric": pbb.quadric(), "r2": pbb.r2_homogeneous(), "lap": pbb.laplacian(),
           "gauss": pbb.gaussian(0.3), "exp": pbb.exponential(0.5)}


@pytest.mark.parametrize("name,order,eps,level", [
    ("const", 4, 1e-6, 3), ("quadric", 3, 1e-6, 3), ("quadric", 4, 1e-6, 4), ("r2", 4, 1e-6, 3), ("quadric", 6, 1e-6, 3),
    ("lap", 4, 1e-5, 3), ("lap", 5, 1e-7, 3), ("lap", 6, 1e-8, 3), ("lap", 8, 1e-6, 2), ("gauss", 6, 1e-8, 4),
    ("exp", 6, 1e-7, 3),
])
def test_adapted_sets_are_exact_to_rounding(gpu, name, order, eps, level):
    import torch
    print(f"case {name} order={order} eps={eps} level={level}", flush=True)
    n = 3000
    plan = pbb.Plan(pbb.Operators(KERNELS[name], 1.0, level, order, eps), uniform_points(n, seed=500 + order))
    g = torch.Generator(device="cuda").manual_seed(order)
    w = torch.rand(2, n, dtype=torch.float64, device="cuda", generator=g)
    own = torch.zeros_like(w)  # the allocation-free matvec before the first plain one runs the own factors
    capi.check(capi.lib().pbb_plan_matvec_noalloc(plan._h, C.c_void_p(w.data_ptr()), 2, C.c_void_p(own.data_ptr()),
                                                  capi.PREC_FP64, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    got = plan.matvec(w)
    assert not torch.equal(got, own)  # the adapted sets ran
    rel = float((got - own).norm() / own.norm())
    print(f"  difference {rel:.2e}", flush=True)
    assert rel <= 8 * order ** 1.5 * 2.0**-53

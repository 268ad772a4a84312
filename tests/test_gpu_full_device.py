"""Calls on a device with no room for the padded rows of the reflection-adapted
sets: passes that cannot run in column chunks take the sets' own factors.  And
without the memory to make the sets, a matvec runs the own factors until a later
one has it."""
import contextlib
import ctypes as C

import pytest

import pbbfmm3d_amd as pbb
from pbbfmm3d_amd import _capi as capi
from tests._helpers import uniform_points

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def _filled(left=None):
    """64 MB less free than `left` bytes, by default what workspaces leave to
    the caller, a sixteenth of the device (every allocation of the tests still
    succeeds)."""
    import torch
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    held = []
    for _ in range(4):  # (the free memory reported after an allocation of this size is not exact)
        free, total = torch.cuda.mem_get_info()
        more = free - (left or max(1 << 30, total // 16)) + (64 << 20)
        if more > 0:
            held.append(torch.empty(max(more, 32 << 20), dtype=torch.uint8, device="cuda"))
    try:
        yield
    finally:
        torch.cuda.synchronize()
        held.clear()
        torch.cuda.empty_cache()


def test_gradients_take_the_unpadded_workspace(gpu):
    import torch
    n, nc = 100000, 32
    xyz = uniform_points(n, seed=600)
    ops = pbb.Operators(pbb.laplacian(), 1.0, 5, 5, 1e-9)
    plan = pbb.Plan(ops, xyz)
    g = torch.Generator(device="cuda").manual_seed(601)
    w, psi = (torch.randn(nc, n, dtype=torch.float64, device="cuda", generator=g) for _ in range(2))
    plan.grad_positions(w[:1].contiguous(), psi[:1].contiguous())  # both operator sets and their adapted sets
    print(f"case N={n} ncols={nc} rank={ops.rank_f}", flush=True)
    with _filled():
        before = torch.cuda.mem_get_info()[0]
        got = plan.grad_positions(w, psi)
        torch.cuda.synchronize()
        grown = before - torch.cuda.mem_get_info()[0]
    boxes = plan.info()["boxes"]
    # S, P and Pf of every box, the sorted weights thrice, the leaf expansions and weights that the gradient saves
    own = 8 * nc * (sum(boxes[2:]) * (125 + 2 * ops.rank_f) + 3 * n + boxes[5] * 125 + n)
    assert grown <= own + (256 << 20)
    ref = pbb.Plan(ops, xyz).grad_positions(w, psi)
    assert float((got - ref).norm() / ref.norm()) <= 1e-11


def test_batch_takes_the_own_factors(gpu):
    import torch
    n, nc = 2500, 3
    ops = pbb.Operators(pbb.laplacian(), 1.0, 3, 5, 1e-7)
    plan = pbb.Plan(ops, uniform_points(n, seed=610))
    g = torch.Generator(device="cuda").manual_seed(611)
    w = torch.randn(nc, n, dtype=torch.float64, device="cuda", generator=g)
    own, out = torch.zeros_like(w), torch.zeros_like(w)
    # the allocation-free matvec runs the own factors before the first plain one
    capi.check(capi.lib().pbb_plan_matvec_noalloc(plan._h, C.c_void_p(w.data_ptr()), nc, C.c_void_p(own.data_ptr()),
                                                  capi.PREC_FP64, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    adapted = plan.matvec(w)
    assert not torch.equal(adapted, own)
    with _filled():
        pbb.Batch([plan], [w], [out], nc).launch()
        torch.cuda.synchronize()
    assert torch.equal(out, own)
    pbb.Batch([plan], [w], [out], nc).launch()  # and with the memory free again
    torch.cuda.synchronize()
    assert torch.equal(out, adapted)


def test_sets_are_made_when_there_is_memory(gpu):
    import torch
    n, nc = 2500, 3
    ops = pbb.Operators(pbb.laplacian(), 1.0, 3, 5, 1e-7)
    plan = pbb.Plan(ops, uniform_points(n, seed=620))
    g = torch.Generator(device="cuda").manual_seed(621)
    w = torch.randn(nc, n, dtype=torch.float64, device="cuda", generator=g)
    own = torch.zeros_like(w)
    capi.check(capi.lib().pbb_plan_matvec_noalloc(plan._h, C.c_void_p(w.data_ptr()), nc, C.c_void_p(own.data_ptr()),
                                                  capi.PREC_FP64, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    with _filled(1 << 30):
        for _ in range(4):  # (as often as a call likes)
            assert torch.equal(plan.matvec(w), own)
    got = plan.matvec(w)
    assert not torch.equal(got, own)
    assert float((got - own).norm() / own.norm()) <= 1e-11

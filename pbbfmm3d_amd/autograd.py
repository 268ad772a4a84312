"""torch.autograd.Function over the FMM matvec.

``fmm_matvec(xyz, weights, ops)`` returns A~(xyz) @ weights (weights as
(ncols, N) or (N,)); its backward gives
  d/dweights  through the transposed FMM (pbb_plan_matvec_transpose), and
  d/dxyz      through pbb_plan_gradients (derivatives of the Chebyshev
              interpolants and of the P2P kernel; box membership and the
              bbox centre are held fixed, as they are piecewise constant).
Both together take one transposed pass; a forward in FP64 whose points need
a gradient saves its leaf expansions for it where the device has the memory
beside them (otherwise the backward runs the forward's far field again).  The
two forwards sum in different orders: on a device that is nearly full, equal
calls can differ in their last bits, and a checkpointed step (which compares
what its two forwards saved) can find different ones.
The tree is built from xyz at every forward call, unless a plan is given:
then its points are moved to xyz (pbb_plan_update_points, which fails if a
point leaves its leaf box) and its tree is reused.  Weights of any floating
dtype (FP32 included) are handed to the kernels as FP64, the output has the
weights' dtype and every gradient the dtype of its input; the arithmetic is
the precision mode's.
"""
from __future__ import annotations

import torch

from . import _capi as capi
from .core import Operators, Plan


class FMMMatvec(torch.autograd.Function):
    @staticmethod
    def forward(ctx, xyz, weights, ops: Operators, precision: int, plan, keep: bool = False):
        pts = xyz.detach().to(torch.float64).cpu().numpy()
        if plan is None:
            plan = Plan(ops, pts)
        else:
            if plan.ops is not ops:
                raise ValueError("the plan was built with other operators")
            plan.update_points(pts)
        w64 = weights.detach().to(device="cuda", dtype=torch.float64).contiguous()
        kept = None
        if keep:
            out, kept = plan._matvec_keep(w64, precision)
        else:
            out = plan.matvec(w64, precision=precision)
        ctx.plan = plan
        ctx.precision = precision
        ctx.xyz_meta = (xyz.dtype, xyz.device)
        ctx.save_for_backward(w64, kept)
        return out.to(weights.dtype)

    @staticmethod
    def backward(ctx, grad_out):
        w64, kept = ctx.saved_tensors
        g64 = grad_out.detach().to(device="cuda", dtype=torch.float64).contiguous()
        gx = gw = None
        if ctx.needs_input_grad[0]:
            dt, dev = ctx.xyz_meta
            gw, gx = ctx.plan._gradients(w64, kept, g64, ctx.precision, weights=ctx.needs_input_grad[1])
            gx = gx.to(device=dev, dtype=dt)
        elif ctx.needs_input_grad[1]:
            gw = ctx.plan.matvec_transpose(g64, precision=ctx.precision)
        if gw is not None:
            gw = gw.to(grad_out.dtype)
        return gx, gw, None, None, None, None


def fmm_matvec(xyz: torch.Tensor, weights: torch.Tensor, ops: Operators,
               precision: int = capi.PREC_FP64, plan: Plan = None) -> torch.Tensor:
    """A~(xyz) @ weights with gradients for both arguments.  plan: a plan of
    ops whose tree is reused (its points are moved to xyz); it holds the
    points of its last forward, so run a backward before the next forward
    with the same plan."""
    keep = torch.is_grad_enabled() and xyz.requires_grad
    return FMMMatvec.apply(xyz, weights, ops, precision, plan, keep)

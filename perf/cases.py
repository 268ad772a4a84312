"""Workloads of the FMM, from the smallest call to the largest, through the
public entry points: the one-shot host call, the plan's matvec, iterative
solver products, training steps, graph batches and the direct sum.

A case is a dict of plain values.  prepare(case, seed) makes what a program
holds before the call (points, weights, operators, plan), run(state) is one
pass, exact(case, seed) the same results as dense FP64 sums over all pairs,
work(case) the bytes and flops of a pass.
"""
import functools
import math

import numpy as np
import torch

import pbbfmm3d_amd as pbb
from pbbfmm3d_amd import _capi as capi
from pbbfmm3d_amd.FMMCompute import Compute, convert_to_vecOfdouble, convert_to_vecOfvec3, vecOfdouble, vecOfvec3
from pbbfmm3d_amd.FMMTree import myKernel

PRECISION = {"fp64": capi.PREC_FP64, "f16x2": capi.PREC_MIXED_F16X2}


def listed():
    return [
        # one product of a Krylov solver with the FMM operator on the host
        # vectors of scipy's solvers (the reference's GMRES example input):
        # the smallest call, repeated hundreds of times a solve
        dict(name="gmres_5k", kind="gmres", n=5000, points="uniform", kernel="laplacian", level=3, order=4, eps=1e-5,
             ncols=1, precision="fp64"),
        # the reference's plain call: tree, matvec and copies in one go
        dict(name="host_call_20k", kind="host", n=20000, points="uniform", kernel="laplacian", level=4, order=4,
             eps=1e-5, ncols=1, precision="fp64"),
        # the randomized eigensolver of the Python front end: an anisotropic
        # covariance against a block of 120 columns
        dict(name="compute_10k_120col", kind="compute", n=10000, points="uniform", kernel="aniso", level=3, order=4,
             eps=1e-5, ncols=120, precision="fp64"),
        # prediction at other places than the data: separate targets and
        # sources, odd sizes, a covariance kernel
        dict(name="targets_78k_sources_30k", kind="matvec", n=77777, nsources=30011, points="uniform",
             kernel="exponential", level=4, order=5, eps=1e-7, ncols=3, precision="fp64"),
        # the drop-in call at a million points, host buffers in and out
        dict(name="host_call_1m_8col", kind="host", n=1000000, points="uniform", kernel="laplacian", level=6, order=5,
             eps=1e-7, ncols=8, precision="fp64"),
        # the same problem on a tree that is kept, weights on the GPU
        dict(name="matvec_1m_8col", kind="matvec", n=1000000, points="uniform", kernel="laplacian", level=6, order=5,
             eps=1e-7, ncols=8, precision="fp64"),
        # a clustered cloud against a block of weights (the benchmark's
        # recipe at a quarter of its points), plain FP64 ...
        dict(name="clustered_1m_32col", kind="matvec", n=1000000, points="clustered", kernel="gaussian", level=6,
             order=6, eps=1e-8, ncols=32, precision="fp64"),
        # ... and in the mixed-precision mode it is meant for
        dict(name="clustered_1m_32col_f16x2", kind="matvec", n=1000000, points="clustered", kernel="gaussian",
             level=6, order=6, eps=1e-8, ncols=32, precision="f16x2"),
        # a training step of FP32 weights and FP64 positions on a fixed tree:
        # forward, adjoint and position gradients
        dict(name="train_500k_4col", kind="train", n=500000, points="uniform", kernel="soft_laplacian", level=6,
             order=5, eps=1e-7, ncols=4, precision="fp64", fixed_tree=True),
        # a training step of a smaller clustered cloud in the mixed mode,
        # the tree built for the positions of the step
        dict(name="train_60k_16col_f16x2", kind="train", n=60000, points="clustered", kernel="gaussian", level=5,
             order=6, eps=1e-8, ncols=16, precision="f16x2", fixed_tree=False),
        # many uneven clouds in one graph launch, forward and adjoint each
        dict(name="batch_24_clouds", kind="batch", n=200000, clouds=24, points="uniform", kernel="exponential",
             level=0, order=0, eps=1e-7, ncols=16, precision="fp64"),
        # the exact sum that approximations are checked against
        dict(name="direct_50k", kind="direct", n=50000, points="uniform", kernel="laplacian", level=0, order=0,
             eps=0.0, ncols=1, precision="fp64"),
    ]


def _level_for(n, points_per_leaf=60.0, deepest=6):
    """About 60 points a leaf, as the clouds of a batch choose their trees."""
    return int(min(deepest, max(3, round(math.log(n / points_per_leaf) / math.log(8.0)))))


def draw(rng):
    def size(lo, hi):  # log-uniform, odd
        return int(math.exp(rng.uniform(math.log(lo), math.log(hi)))) | 1

    kind = rng.choice(["gmres", "host", "compute", "matvec", "matvec", "matvec", "train", "train", "batch", "direct"])
    case = dict(kind=kind, points=rng.choice(["uniform", "uniform", "clustered"]), precision="fp64")
    if kind == "gmres":
        n = size(2000, 100000)
        case.update(n=n, kernel=rng.choice(["laplacian", "exponential"]), order=rng.choice([4, 5]), eps=1e-5, ncols=1)
    elif kind == "host":
        n = size(5000, 400000)
        case.update(n=n, kernel=rng.choice(["laplacian", "gaussian"]), order=rng.choice([4, 5, 6]), eps=1e-6,
                    ncols=rng.choice([1, 2, 5, 8]), precision=rng.choice(["fp64", "fp64", "f16x2"]))
    elif kind == "compute":
        n = size(3000, 40000)
        case.update(n=n, kernel="aniso", order=rng.choice([4, 5]), eps=1e-5, ncols=rng.randint(1, 120))
    elif kind == "matvec":
        n = size(3000, 500000)
        case.update(n=n, kernel=rng.choice(["laplacian", "gaussian", "exponential", "soft_laplacian"]),
                    order=rng.choice([4, 5, 6, 6]), eps=rng.choice([1e-5, 1e-7, 1e-8]),
                    ncols=rng.choice([1, 3, 8, 16, 17, 32]), precision=rng.choice(["fp64", "fp64", "f16x2"]))
        if rng.random() < 0.25:
            case["nsources"] = size(3000, 200000)
    elif kind == "train":
        n = size(5000, 300000)
        case.update(n=n, kernel=rng.choice(["soft_laplacian", "gaussian", "exponential"]), order=rng.choice([4, 5, 6]),
                    eps=1e-7, ncols=rng.choice([1, 2, 4, 16]), precision=rng.choice(["fp64", "f16x2"]),
                    fixed_tree=rng.random() < 0.5)
    elif kind == "batch":
        n = size(20000, 200000)
        case.update(n=n, clouds=rng.randint(5, 24), kernel=rng.choice(["exponential", "gaussian"]), order=0, eps=1e-7,
                    ncols=rng.choice([1, 4, 16]), precision=rng.choice(["fp64", "f16x2"]))
    else:
        n = size(3000, 60000)
        case.update(n=n, kernel=rng.choice(["laplacian", "gaussian"]), order=0, eps=0.0, ncols=1)
    # clustered clouds take two levels more, as the benchmark's does
    deeper = 2 if case["points"] == "clustered" else 0
    case["level"] = 0 if kind in ("batch", "direct") else min(6, _level_for(n) + deeper)
    return case


# ---- inputs ------------------------------------------------------------------
ANISO = (0.75, 1 / 100.0, 1 / 100.0, 1 / 2.25)  # FMMTree.myKernel


def _kernel(name):
    return {"laplacian": pbb.laplacian(), "gaussian": pbb.gaussian(0.3), "exponential": pbb.exponential(0.5),
            "soft_laplacian": pbb.soft_laplacian(1e-6), "aniso": myKernel.device_kernel}[name]


@functools.lru_cache(maxsize=None)
def _operators(kernel, level, order, eps):
    """A program makes a kernel's operators once and uses them for all its
    point sets (the reference keeps them in cache files)."""
    return pbb.Operators(_kernel(kernel), 1.0, level, order, eps)


@functools.lru_cache(maxsize=None)
def _tree(level, order, eps):
    return myKernel(1, level, order, eps, 1).buildFMMTree()


def _cloud(points, n, rng):
    """Uniform, or 8 Gaussian clusters over a fifth of uniform background,
    clipped to the unit cube."""
    if points == "uniform":
        return rng.random((n, 3))
    nb = n // 5
    centres = rng.uniform(0.2, 0.8, (8, 3))
    x = centres[rng.integers(0, 8, n - nb)] + 0.05 * rng.standard_normal((n - nb, 3))
    return np.clip(np.concatenate([x, rng.random((nb, 3))]), 0.0, 1.0)


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _randn(shape, seed, dtype=torch.float64):
    """Standard normal values on the GPU, the same for a seed."""
    g = torch.Generator(device=_device()).manual_seed(seed)
    return torch.randn(shape, dtype=dtype, device=_device(), generator=g)


def _inputs(case, seed):
    """Points (numpy) and weights of a case from the seed: numpy where the
    call takes host data, tensors on the GPU elsewhere."""
    rng = np.random.default_rng([17, seed])
    kind, n, nc = case["kind"], case["n"], case["ncols"]
    if kind == "batch":
        # one cloud of the given size, the others log-uniform below it
        sizes = np.exp(np.random.default_rng(n).uniform(math.log(2e3), math.log(n), case["clouds"] - 1))
        sizes = sorted([n] + [int(v) for v in sizes])
        xyz = [_cloud(case["points"], m, rng) for m in sizes]
        w = [_randn((nc, m), 1000 * seed + 2 * k) for k, m in enumerate(sizes)]
        psi = [_randn((nc, m), 1000 * seed + 2 * k + 1) for k, m in enumerate(sizes)]
        return {"xyz": xyz, "w": w, "psi": psi}
    xyz = _cloud(case["points"], n, rng)
    if kind in ("gmres", "direct", "host", "compute"):
        return {"xyz": xyz, "w": rng.uniform(-1.0, 1.0, (nc, n))}
    if kind == "train":
        return {"xyz": xyz, "w": _randn((nc, n), 2 * seed, torch.float32),
                "b": _randn((nc, n), 2 * seed + 1, torch.float32)}
    src = _cloud(case["points"], case["nsources"], rng) if case.get("nsources") else None
    return {"xyz": xyz, "src": src, "w": _randn((nc, n if src is None else len(src)), 2 * seed)}


def prepare(case, seed):
    I = _inputs(case, seed)
    kind, nc, prec = case["kind"], case["ncols"], PRECISION[case["precision"]]
    s = {"kind": kind, "ncols": nc, "precision": prec}
    if kind == "direct":
        s["op"] = pbb.MatrixDirect(_kernel(case["kernel"]), I["xyz"], shift=0.0)
        s["x"] = I["w"][0]
        return s
    if kind == "compute":
        s["tree"] = _tree(case["level"], case["order"], case["eps"])
        s["points"], s["weights"] = vecOfvec3(), vecOfdouble()
        convert_to_vecOfvec3(I["xyz"], s["points"])
        convert_to_vecOfdouble(I["w"].reshape(-1), s["weights"])
        return s
    if kind == "batch":
        plans, entries, w = [], [], []
        for k, x in enumerate(I["xyz"]):
            ops = _operators(case["kernel"], _level_for(len(x)), 4 + k % 3, case["eps"])
            plan = pbb.Plan(ops, x)
            plans += [plan, plan]
            w += [I["w"][k], I["psi"][k]]
        s["out"] = [torch.zeros_like(v) for v in w]
        s["batch"] = pbb.Batch(plans, w, s["out"], nc, precision=prec, transpose=[False, True] * len(I["xyz"]))
        return s
    s["ops"] = _operators(case["kernel"], case["level"], case["order"], case["eps"])
    if kind == "gmres":
        s["op"] = pbb.MatrixFMM(s["ops"], I["xyz"], shift=0.0)
        s["x"] = I["w"][0]
    elif kind == "host":
        s["xyz"], s["w"] = I["xyz"], I["w"].reshape(-1)
    elif kind == "train":
        s["xyz"] = torch.tensor(I["xyz"], dtype=torch.float64, device="cuda", requires_grad=True)
        s["w"] = I["w"].requires_grad_(True)
        s["b"] = I["b"]
        s["plan"] = pbb.Plan(s["ops"], I["xyz"]) if case["fixed_tree"] else None
    else:
        s["plan"] = pbb.Plan(s["ops"], I["xyz"], sources=I["src"])
        s["w"] = I["w"]
    return s


def run(state):
    kind = state["kind"]
    if kind in ("gmres", "direct"):
        return state["op"].matvec(state["x"])
    if kind == "host":
        return pbb.matvec_host(state["ops"], state["xyz"], state["w"], state["ncols"], precision=state["precision"])
    if kind == "compute":
        out = vecOfdouble(len(state["points"]) * state["ncols"])
        Compute(state["tree"], state["points"], state["points"], state["weights"], state["ncols"], out)
        return out.data
    if kind == "batch":
        state["batch"].launch()
        return state["out"]
    if kind == "train":  # loss 1/2 |A(x) w - b|^2
        out = pbb.fmm_matvec(state["xyz"], state["w"], state["ops"], precision=state["precision"], plan=state["plan"])
        loss = 0.5 * (out - state["b"]).square().sum()
        gx, gw = torch.autograd.grad(loss, (state["xyz"], state["w"]))
        return {"out": out.detach(), "grad_points": gx, "grad_weights": gw}
    return state["plan"].matvec(state["w"], precision=state["precision"])


# ---- the same results as dense sums --------------------------------------------
def _dense(name, t, s):
    """K(t_i, s_j) in FP64, zero where the kernel is infinite, and for the
    kernels of training steps f with grad K = f (t_i - s_j)."""
    scale = ANISO[1:] if name == "aniso" else (1.0, 1.0, 1.0)
    r = sum(c * (t[:, k, None] - s[None, :, k]) ** 2 for k, c in enumerate(scale)).sqrt()
    if name == "aniso":
        return ANISO[0] * torch.exp(-r), None
    if name == "laplacian":
        k = 1.0 / r
        return torch.where(torch.isinf(k), torch.zeros((), dtype=k.dtype, device=k.device), k), None
    if name == "gaussian":
        k = torch.exp(-r * r / 0.09)
        return k, lambda: (-2.0 / 0.09) * k
    if name == "exponential":
        k = torch.exp(-r / 0.5)
        return k, lambda: torch.where(r > 0, -2.0 * k / r, torch.zeros((), dtype=k.dtype, device=k.device))
    k = 1.0 / torch.sqrt(r * r + 1e-6)
    return k, lambda: -(k * k * k)


def _blocks(nt, ns):
    step = max(1, min(nt, int(2e8 if torch.cuda.is_available() else 4e6) // ns))
    return [(i, min(nt, i + step)) for i in range(0, nt, step)]


def _dense_sum(name, tgt, src, w):
    """(ncols, targets) = w K^T for (ncols, sources) weights."""
    out = torch.empty((w.shape[0], tgt.shape[0]), dtype=torch.float64, device=w.device)
    for i, j in _blocks(tgt.shape[0], src.shape[0]):
        out[:, i:j] = (_dense(name, tgt[i:j], src)[0] @ w.T.contiguous()).T
    return out


def exact(case, seed):
    kind, name = case["kind"], case["kernel"]
    n = case["n"]
    I = _inputs(case, seed)
    if kind == "batch":
        pairs = 2.0 * sum(float(len(x)) ** 2 for x in I["xyz"])
    else:
        pairs = float(n) * (case.get("nsources") or n) * (3 if kind == "train" else 1)
    if pairs > (2.5e11 if torch.cuda.is_available() else 1e9):
        return None
    def put(a):
        return torch.as_tensor(a, dtype=torch.float64, device=_device())

    if kind == "batch":
        res = []
        for x, w, p in zip(I["xyz"], I["w"], I["psi"]):
            x = put(x)
            res += [_dense_sum(name, x, x, w), _dense_sum(name, x, x, p)]
        return res
    x, w = put(I["xyz"]), put(I["w"])
    if kind == "train":
        b = put(I["b"])
        r = _dense_sum(name, x, x, w) - b
        gw = _dense_sum(name, x, x, r)
        gx = torch.empty_like(x)
        for i, j in _blocks(n, 2 * n):
            f = _dense(name, x[i:j], x)[1]()
            f *= r[:, i:j].T @ w + w[:, i:j].T @ r
            gx[i:j] = x[i:j] * f.sum(1, keepdim=True) - f @ x
        return {"out": r + b, "grad_points": gx, "grad_weights": gw}
    src = put(I["src"]) if I.get("src") is not None else x
    out = _dense_sum(name, x, src, w)
    if kind == "matvec":
        return out
    return out.reshape(-1).cpu().numpy()


# ---- the work of a pass ---------------------------------------------------------
def _window(grid, lo, hi):
    """Sums of a cubic grid over the offsets lo..hi of every cell and axis."""
    for ax in range(3):
        z = np.zeros_like(np.take(grid, [0], ax))
        c = np.cumsum(np.concatenate([z, grid], ax), ax)
        m = grid.shape[ax]
        a, b = np.clip(np.arange(m) + lo, 0, m), np.clip(np.arange(m) + hi + 1, 0, m)
        grid = np.take(c, b, ax) - np.take(c, a, ax)
    return grid


def _fmm_work(xyz, nt, kernel, level, order, eps, nc, precision, gradient=False):
    """Flops of one FMM pass over the points: P2M and L2P once per point, M2M
    and L2L once per box, the low-rank far field per box pair and the near
    field per point pair."""
    ops = _tree(level, order, eps).operators() if kernel == "aniso" else _operators(kernel, level, order, eps)
    ranks = [(ops.rank_f, ops.rank_s)] * ops.nsets
    if precision != "fp64":
        ranks = [(min(a, ops.rank_f), min(b, ops.rank_s)) for a, b, _ in ops.mixed_ranks()]
    n3, eval_flops = order ** 3, 10
    centre = 0.5 * (xyz[:nt].min(0) + xyz[:nt].max(0))
    m = 1 << level
    cell = np.clip(np.floor((xyz - centre + 0.5) * m).astype(np.int64), 0, m - 1)
    count = np.bincount((cell[:, 0] * m + cell[:, 1]) * m + cell[:, 2], minlength=m ** 3).reshape(m, m, m)
    near = float((count * _window(count, -1, 1)).sum())
    flops = near * (eval_flops + 2 * nc) + 4.0 * len(xyz) * n3 * nc
    if gradient:
        flops += near * (eval_flops + 8 * nc) + 12.0 * len(xyz) * n3 * nc
    for l in range(level, 1, -1):
        kf, ks = ranks[l - 2 if ops.nsets > 1 else 0]
        occ = (count > 0).astype(np.int64)
        # far sources of a box: the children of its parent's neighbours less its own neighbours
        up = occ.reshape(m // 2, 2, m // 2, 2, m // 2, 2).sum((1, 3, 5))
        fam = np.repeat(np.repeat(np.repeat(_window(up, -1, 1), 2, 0), 2, 1), 2, 2)
        pairs = float((occ * (fam - _window(occ, -1, 1))).sum())
        flops += pairs * 2.0 * kf * ks * nc + float(occ.sum()) * nc * (2.0 * n3 * (kf + ks) + 12.0 * order * n3)
        count = count.reshape(m // 2, 2, m // 2, 2, m // 2, 2).sum((1, 3, 5))
        m //= 2
    return flops


def work(case):
    I = _inputs(case, 0)
    kind, nc, n = case["kind"], case["ncols"], case["n"]
    if kind == "direct":
        return {"bytes": 24.0 * n + 16.0 * n * nc, "flops": float(n) * n * (9 + 2 * nc)}
    if kind == "batch":
        flops = 2 * sum(_fmm_work(x, len(x), case["kernel"], _level_for(len(x)), 4 + k % 3, case["eps"], nc,
                                  case["precision"]) for k, x in enumerate(I["xyz"]))
        return {"bytes": sum(len(x) for x in I["xyz"]) * (24.0 + 32.0 * nc), "flops": flops}
    xyz = I["xyz"] if I.get("src") is None else np.concatenate([I["xyz"], I["src"]])
    args = (xyz, n, case["kernel"], case["level"], case["order"], case["eps"], nc, case["precision"])
    if kind == "train":  # forward, adjoint and the gradient's near and far parts
        return {"bytes": n * (48.0 + 16.0 * nc), "flops": _fmm_work(*args) + _fmm_work(*args, gradient=True)}
    ns = case.get("nsources") or n
    return {"bytes": 24.0 * len(xyz) + 8.0 * nc * (n + ns), "flops": _fmm_work(*args)}

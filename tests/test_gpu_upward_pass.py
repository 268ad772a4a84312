"""The direct upward pass on the matrix cores, through whole FP64 matvecs
against the oracle: every order, one and several column blocks of a wave and
columns divided over the waves, boxes of one point, of 16 and 32 points and
their neighbours, and a box of more points than a work item holds."""
import numpy as np
import pytest

import pbbfmm3d_amd as pbb
from oracle import oracle as orc
from tests._helpers import oracle_ops_from

pytestmark = pytest.mark.gpu

# columns: 1 and 2 column blocks of 16 at the low orders, a partial last block,
# a wave's all blocks, one more, and ranges divided over 3 and 4 waves
CASES = [(4, 1), (4, 5), (4, 17), (4, 33), (5, 3), (5, 4), (5, 10), (5, 31), (6, 2), (6, 9), (6, 32), (7, 1), (7, 5),
         (7, 15), (8, 2), (8, 5), (8, 13)]


def _points(counts, big, rng):
    """counts[k] points in the k-th cell of a 4 x 4 x 4 grid, `big` more in
    the last one, and the unit cube's corners (the grid's place)."""
    xyz = [np.array([[0.0, 0, 0], [1.0, 1, 1]])]
    for k, m in enumerate(counts):
        c = np.array([k // 16, k // 4 % 4, k % 4])
        xyz.append((c + rng.uniform(0.05, 0.95, (m + (big if k == 63 else 0), 3))) / 4)
    return np.concatenate(xyz)


@pytest.mark.parametrize("n,ncols", CASES)
def test_upward_pass(gpu, n, ncols):
    import torch
    print(f"case order={n} ncols={ncols}", flush=True)
    rng = np.random.default_rng(100 * n + ncols)
    counts = np.resize([1, 3, 4, 5, 15, 16, 17, 31, 32, 33, 0, 65], 64)
    xyz = _points(counts, 2100 if ncols < 6 else 0, rng)
    N = len(xyz)
    w = rng.uniform(-1.0, 1.0, N * ncols)
    for level in (2, 3):  # few and many points a box
        ops = pbb.Operators(pbb.gaussian(0.3), 1.0, level, n, 1e-5)
        oops = oracle_ops_from(ops, pbb.gaussian(0.3))
        got = pbb.Plan(ops, xyz).matvec(torch.tensor(w.reshape(ncols, N), device="cuda")).cpu().numpy().reshape(-1)
        assert orc.rel_err(got, orc.matvec(oops, xyz, w, ncols)) <= 1e-10

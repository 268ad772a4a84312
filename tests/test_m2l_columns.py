"""Columns of an FP64 pass whose proxies are more than the 32-bit offsets of
the reflection-adapted M2L reach (64 GB a level)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "host.hpp"
int main(int argc, char **argv)
{
    for (int i = 1; i + 2 < argc; i += 3) {
        const long long nb = atoll(argv[i]), nk = atoll(argv[i + 2]);
        const int c = pbb::sym_columns(nb, atoi(argv[i + 1]), nk);
        std::printf("%d %d\n", c, (int)pbb::sym_level_fits(nb, c, nk));
    }
}
"""
# (boxes, columns, nk): a full level 7 with 64 proxies and 64 columns is 64 GiB
# and one box; the largest trees at the largest ranks
CASES = [(4096, 1, 8), (262144, 8, 104), (2**21, 63, 64), (2**21 - 1, 64, 64), (2**21, 64, 64), (2**21, 41, 104),
         (2**21, 170, 48), (2**24, 120, 104), (2**24, 7, 1024), (2**27 - 1, 1, 64), (2**27, 1, 64), (2**27, 5, 512)]


def test_columns_of_a_pass(tmp_path):
    (tmp_path / "c.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "c")
    subprocess.run(["g++", "-std=c++17", f"-I{ROOT}/pbbfmm3d_amd/csrc", f"-I{ROOT}/include", str(tmp_path / "c.cpp"),
                    "-o", exe], check=True)
    out = subprocess.run([exe] + [str(v) for c in CASES for v in c], check=True, capture_output=True, text=True).stdout
    for (nb, ncols, nk), line in zip(CASES, out.splitlines()):
        c, fits = map(int, line.split())
        reach = lambda k: (nb + 1) * k * nk // 2 < 2**32  # noqa: E731 (units of 16 bytes)
        want = ncols
        while want > 1 and not reach(want):
            want = (want + 1) // 2
        assert (c, fits) == (want, int(reach(want))), (nb, ncols, nk)


@pytest.mark.gpu
def test_level_of_more_than_64_gb(gpu):
    """2.1M leaves, 64 columns, 64 proxies each: 64 GiB and one box.  The
    columns are those of calls of one column's workspace, bit for bit."""
    import numpy as np
    import torch

    import pbbfmm3d_amd as pbb
    m = 128
    print(f"case level 7, {m**3} leaves, 64 columns", flush=True)
    cell = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
    xyz = (cell + 0.1 + 0.8 * np.random.default_rng(77).random((m**3, 3))) / m
    xyz[0], xyz[-1] = 0.0, 1.0
    ops = pbb.Operators(pbb.laplacian(), 1.0, 7, 4, 1e-9)
    assert ops.rank_s == 64
    plan = pbb.Plan(ops, xyz)
    assert plan.info()["boxes"][7] == m**3
    g = torch.Generator(device="cuda").manual_seed(78)
    w = torch.randn(64, m**3, dtype=torch.float64, device="cuda", generator=g)
    out = plan.matvec(w)
    plan.set_workspace_limit(20 << 30)
    assert torch.equal(plan.matvec(w), out)

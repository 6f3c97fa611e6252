"""The caching pool: its rules on the CPU (csrc/pool.hpp, plain host code:
reuse by size, the bound and what it evicts, room made when memory runs out,
several threads at once), and the call that empties it on the GPU."""
import os
import subprocess

import numpy as np
import pytest

import idrs_amd
from idrs_amd import problems as P

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pool_rules(tmp_path):
    exe = str(tmp_path / "pool_test")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "idrs-package_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "pool_test.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr


@pytest.mark.gpu
def test_release_pool(gpu):
    import torch

    crs, _ = P.convection_diffusion_3d(40, 8.0, reaction=1.0)
    A = idrs_amd.Matrix(idrs_amd.crs_format(crs.n, crs.n, crs.row_ptr, crs.col_ind, rval=crs.val))
    b = np.random.default_rng(0).uniform(-1, 1, crs.n)
    first = idrs_amd.idrs(A, b, 4, tolerance=1e-9)
    before = torch.cuda.mem_get_info()[0]
    freed = idrs_amd.release_pool()
    assert freed >= 8 * crs.n * 16        # G, U, P, r, t and the vectors of the call
    assert torch.cuda.mem_get_info()[0] >= before and idrs_amd.release_pool() == 0
    again = idrs_amd.idrs(A, b, 4, tolerance=1e-9)
    assert first.flag == again.flag == 0 and np.array_equal(first.x, again.x)

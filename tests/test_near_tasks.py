"""The near field's waves (near_tasks) on the CPU: every (point, lane) pair of every
near box in one wave, from one box of a few points, which starts at 64 lanes a
point, to leaves that take one lane; built apart from the near lists, which stored
products and points share without them."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "elfmmlib3d_amd", "csrc")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("nt") / "near_tasks.so")
    srcs = [os.path.join(ROOT, "tests", "csrc", "near_tasks.cpp")] + [
        os.path.join(CSRC, f) for f in ("elfmm_tree.cpp", "elfmm_plan.cpp", "elfmm_ops.cpp", "elfmm_pool.cpp")]
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-pthread", "-o", out, *srcs], check=True)
    return C.CDLL(out)


@pytest.mark.parametrize("n,nt,nbox", [(1, 0, 40), (3, 1, 40), (65, 63, 40), (1000, 10, 3), (3000, 5000, 120), (20000, 0, 60)])
@pytest.mark.parametrize("src_eval", [0, 1])
def test_every_lane_once(lib, n, nt, nbox, src_eval):
    rng = np.random.default_rng(n + nt)
    s, t = rng.random((n, 3)) ** 2, rng.random((max(nt, 1), 3))
    waves = lib.near_tasks_check(s.ctypes.data_as(C.c_void_p), n, t.ctypes.data_as(C.c_void_p), nt, nbox, src_eval)
    assert waves > 0 or not (src_eval or nt)

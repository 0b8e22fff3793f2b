"""What the M2L, M2M and L2L kernels multiply by (records of rotation, shift
along z and rotation back; dense matrices for M2L of the lower orders) on the
host against the addition theorems in long double: every octant, and the list-2
offsets, of every order in use.

Tolerance: three products of at most 40 terms of orthogonal or one-signed rows
on doubles, 3 x 40 x 1.1e-16, and the phases' rounding, p x 1.1e-16: 2e-14."""
import ctypes as C
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "elfmmlib3d_amd", "csrc")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("tr") / "translations.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-pthread", "-o", out,
                    os.path.join(ROOT, "tests", "csrc", "translations.cpp")] +
                   [os.path.join(CSRC, f"elfmm_{n}.cpp") for n in ("ops", "tree", "plan", "pool")], check=True)
    lib = C.CDLL(out)
    lib.translation_error.restype = C.c_double
    return lib


@pytest.mark.parametrize("iprec,p", [(-2, 2), (-1, 5), (0, 9), (1, 14), (2, 26), (3, 39)])
def test_translations(lib, iprec, p):
    order, seen = C.c_int(), set()
    for kind, count in ((0, 8), (1, 8), (2, 343)):
        for k in range(count):
            if kind == 2 and p > 14 and k % 7 not in (k // 7 % 7, 3):
                continue                                  # a third of the offsets at the high orders
            assert lib.translation_error(iprec, p, kind, k, k, C.byref(order)) <= 2e-14, (kind, k)
            seen.add(order.value)
    assert -1 in seen and p in seen

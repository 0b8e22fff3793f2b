"""P2M and P2L through triangle moments (elfmm_moments.h) built for the host, a
thread per lane, against the node sums in long double: every launch shape (the
orders of iprec 0 to 3), leaves of one triangle, of a chunk, one more and
several chunks, and a source list of more boxes than one pass takes (64).

Tolerance: a coefficient of degree l is a sum of up to 12 x 100 terms carried
through l <= 40 recurrence steps, each rounding once or twice: 1e-12 per degree
bounds 40 x 12 x 2.2e-16 x 10 for sums whose terms do not all share a sign."""
import ctypes as C
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("mom") / "moments.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-pthread", "-w", "-o", out,
                    os.path.join(ROOT, "tests", "csrc", "moments_host.cpp")], check=True)
    lib = C.CDLL(out)
    lib.moments_host.restype = C.c_double
    lib.moment_parts_host.restype = C.c_double
    return lib


@pytest.mark.parametrize("p,nq,chunk", [(9, 6, 10), (14, 12, 8), (26, 12, 9), (39, 12, 12)])
@pytest.mark.parametrize("irr", [0, 1])
def test_moments(lib, p, nq, chunk, irr):
    counts = (C.c_int * 4)(1, chunk, chunk + 1, 2 * chunk + 3)
    assert 0 <= lib.moments_host(p, nq, irr, counts, 3, 7 * p + irr) <= 1e-12


def test_long_source_list(lib):
    counts = (C.c_int * 4)(1, 0, 2, 1)
    assert 0 <= lib.moments_host(14, 12, 1, counts, 67, 5) <= 1e-12


def test_other_orders_have_no_shape(lib):
    counts = (C.c_int * 4)(1, 1, 1, 1)
    for p, nq in ((5, 3), (2, 1), (44, 12), (26, 6)):
        assert lib.moments_host(p, nq, 0, counts, 1, 1) < 0


@pytest.mark.parametrize("p,nq,count,nparts", [(9, 6, 1, 1), (9, 6, 23, 3), (14, 12, 37, 2), (26, 12, 36, 2),
                                               (26, 12, 19, 1), (39, 12, 27, 5)])
def test_parts_and_mindlin_moments(lib, p, nq, count, nparts):
    """A box cut into parts whose coefficients are added, and the moments as they
    are (the Mindlin P2M), in parts too: the same sums, the same tolerance."""
    assert 0 <= lib.moment_parts_host(p, nq, count, nparts, 3 * p + count) <= 1e-12

"""The near-field kernel's pair code (elfmm_near.h) built for the host, against
the direct sum's pair code (elfmm_math.h) and the reference's pair routines
(fixture `pairs`): points beside, above, in the plane of and on the lines of
the edges of a triangle, its own centroid, each layer, with and without strain.

Tolerances: the closed forms lose eps * (R/L)^k between the edges at distance R
from a triangle of size L (k = 2 in the displacement of a double layer, 3 in its
strain); at the distances of a near list, R/L <= 8, that is 8^3 eps times the
few tens of terms: 1e-11 of the largest value for both codes together."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT, load_golden

CSRC = os.path.join(ROOT, "tests", "csrc")


@pytest.fixture(scope="module")
def nf(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("np") / "near_pair.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-o", out, os.path.join(CSRC, "near_pair.cpp")],
                   check=True)
    return C.CDLL(out)


def P(a):
    return np.ascontiguousarray(a, dtype=np.float64).ctypes.data_as(C.c_void_p)


def pair(nf, name, tri, s, d, x, iself, lam, mu, *flags):
    out = np.zeros(9)
    getattr(nf, name)(P(tri), P(s), P(d), P(x), int(iself), C.c_double(lam), C.c_double(mu), *flags, P(out))
    return out


def sym6(s):
    return np.array([s[0, 0], s[1, 1], s[2, 2], s[0, 1], s[0, 2], s[1, 2]])


def test_matches_reference(nf):
    g = load_golden("pairs")
    for t in range(len(g["ifself"])):
        for sl, dl, kp, ks in ((1, 0, "pt_sl", "st_sl"), (0, 1, "pt_dl", "st_dl")):
            out = pair(nf, "near_host_pair", g["tri"][t], g["sigma"][t], g["sigma"][t], g["target"][t],
                       g["ifself"][t], float(g["lam"][t]), float(g["mu"][t]), sl, dl, 1)
            ref = np.concatenate([g[kp][t], sym6(g[ks][t])])
            assert np.abs(out - ref).max() <= 1e-11 * max(1.0, np.abs(ref).max()), (t, sl)


def points(tri, rng):
    """(point, own centroid) around a triangle."""
    e = tri[1] - tri[0]
    L = np.linalg.norm(e)
    nrm = np.cross(e, tri[2] - tri[0])
    nrm /= np.linalg.norm(nrm)
    c = tri.mean(0)
    yield c, 1
    yield c + 1e-3 * L * nrm, 0
    yield c - 0.3 * L * nrm, 0
    for r in (0.6, 2.0, 8.0):
        v = rng.normal(size=3)
        yield c + r * L * v / np.linalg.norm(v), 0
    for k in range(3):                                   # beyond both ends of each edge: on its line, in the plane
        a, b = tri[k], tri[(k + 1) % 3]
        yield b + 0.7 * (b - a), 0
        yield a - 0.7 * (b - a) + 1e-9 * L * nrm, 0
        yield (a + b) / 2 + 1e-4 * L * nrm, 0             # over the middle of the edge
        yield (a + b) / 2 + 0.2 * ((a + b) / 2 - c), 0    # in the plane, beside it
        yield a + 0.05 * (a - c), 0                       # next to a vertex, foot points outside two edges


@pytest.mark.parametrize("sl,dl", [(1, 0), (0, 1), (1, 1)])
def test_matches_direct_pair(nf, sl, dl):
    rng = np.random.default_rng(7 + 2 * sl + dl)
    for t in range(40):
        tri = np.array([[0, 0, 0], [1, 0, 0], [0.4, 0.9, 0]]) + 0.15 * rng.normal(size=(3, 3))
        tri = tri * 10.0 ** rng.uniform(-3, 3) + rng.normal(size=3)
        for x, iself in points(tri, rng):
            s, d = rng.normal(size=3), rng.normal(size=3)
            lam, mu = rng.uniform(0.3, 3), rng.uniform(0.3, 3)
            old = pair(nf, "near_host_old", tri, s, d, x, iself, lam, mu, sl, dl)
            new = pair(nf, "near_host_pair", tri, s, d, x, iself, lam, mu, sl, dl, 1)
            for c in (slice(0, 3), slice(3, 9)):
                assert np.abs(new - old)[c].max() <= 1e-11 * np.abs(old[c]).max(), (t, x, iself)
            disp = pair(nf, "near_host_pair", tri, s, d, x, iself, lam, mu, sl, dl, 0)
            assert np.abs(disp - new)[:3].max() <= 1e-14 * np.abs(new[:3]).max()
            assert not disp[3:].any()


@pytest.mark.parametrize("sl,dl", [(1, 0), (0, 1)])
def test_distant_points_keep_their_digits(nf, tmp_path, sl, dl):
    """Far from a triangle (a leaf of few triangles beside large ones) the sums over
    its edges lose R/L of the digits and no more: 20 roundings a term, some tens of
    terms, 1e-13 R/L, against the direct sum's code in long double."""
    out = str(tmp_path / "near_long.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-o", out, os.path.join(CSRC, "near_pair_long.cpp")],
                   check=True)
    exact = C.CDLL(out)
    rng = np.random.default_rng(3 + sl)
    for r in (1.5, 8.0, 60.0, 1000.0):
        for t in range(50):
            tri = np.array([[0, 0, 0], [1, 0, 0], [0.4, 0.9, 0]]) + 0.2 * rng.normal(size=(3, 3))
            v = rng.normal(size=3)
            x = tri.mean(0) + r * v / np.linalg.norm(v)
            s, d = rng.normal(size=(2, 3))
            ref = pair(exact, "near_long", tri, s, d, x, 0, 1.1, 0.7, sl, dl)
            new = pair(nf, "near_host_pair", tri, s, d, x, 0, 1.1, 0.7, sl, dl, 1)
            for c in (slice(0, 3), slice(3, 9)):
                assert np.linalg.norm((new - ref)[c]) <= 1e-13 * r * np.linalg.norm(ref[c]), (r, t)

"""The point near field at the edges of its work split (lanes per point 64 down
to 1, workgroups of 256 lanes, source tiles of 256), through the direct sum,
against the Kelvin point kernels in numpy.

Tolerance: a sum of n terms of both signs in double, each within a few units
in the last place: n * 8 * 2.2e-16 * sum|terms| / |sum| bounds it by 1e-12 of
the largest value for n <= 700 random terms."""
import numpy as np
import pytest

import elfmmlib3d_amd as E

pytestmark = pytest.mark.gpu


def kelvin(x, src, skip_self, f, s, d, lam, mu):
    c1 = (lam + mu) / (lam + 2 * mu)
    c2 = 1 - c1
    R = x[:, None] - src[None]
    r2 = (R ** 2).sum(-1)
    if skip_self:
        np.fill_diagonal(r2, np.inf)
    i1 = 1 / np.sqrt(r2)
    i3, i5, i7 = i1 ** 3, i1 ** 5, i1 ** 7
    eye = np.eye(3)
    dot = lambda v: np.einsum("ijc,jc->ij", R, v)
    u = np.zeros(x.shape)
    g = np.zeros((x.shape[0], 3, 3))
    if f is not None:
        fR = dot(f)
        u += (np.einsum("ij,jc->ic", (2 - c1) * i1, f) + c1 * np.einsum("ij,ijc->ic", fR * i3, R)) / (2 * mu)
        g += (-(2 - c1) * np.einsum("ij,jc,ijd->icd", i3, f, R) + c1 * np.einsum("ij,ijc,jd->icd", i3, R, f)
              + c1 * np.einsum("ij,cd->icd", fR * i3, eye)
              - 3 * c1 * np.einsum("ij,ijc,ijd->icd", fR * i5, R, R)) / (2 * mu)
    if s is not None:
        sR, dR, sd = dot(s), dot(d), (s * d).sum(1)
        u += c2 * (np.einsum("ij,jc->ic", dR * i3, s) + np.einsum("ij,jc->ic", sR * i3, d)
                   - np.einsum("ij,ijc->ic", sd * i3, R)) + 3 * c1 * np.einsum("ij,ijc->ic", sR * dR * i5, R)
        a = (np.einsum("ij,jc,jd->icd", i3, s, d) + np.einsum("ij,jc,jd->icd", i3, d, s)
             - np.einsum("ij,cd->icd", sd * i3, eye))
        a -= 3 * (np.einsum("ij,jc,ijd->icd", dR * i5, s, R) + np.einsum("ij,jc,ijd->icd", sR * i5, d, R)
                  - np.einsum("ij,ijc,ijd->icd", sd * i5, R, R))
        b = (np.einsum("ij,ijc,jd->icd", dR * i5, R, s) + np.einsum("ij,ijc,jd->icd", sR * i5, R, d)
             + np.einsum("ij,cd->icd", sR * dR * i5, eye) - 5 * np.einsum("ij,ijc,ijd->icd", sR * dR * i7, R, R))
        g += c2 * a + 3 * c1 * b
    return u, (g + np.swapaxes(g, 1, 2)) / 2


@pytest.mark.parametrize("n,m", [(1, 3), (2, 0), (63, 1), (64, 65), (195, 0), (255, 258), (257, 31), (700, 513)])
@pytest.mark.parametrize("layers", ["s", "d", "sd"])
def test_point_direct_split(n, m, layers):
    rng = np.random.default_rng(1000 * n + m)
    src, tg = rng.uniform(0, 1, (n, 3)), rng.uniform(0, 1, (m, 3))
    f = rng.uniform(-1, 1, (n, 3)) if "s" in layers else None
    s = rng.uniform(-1, 1, (n, 3)) if "d" in layers else None
    d = rng.normal(size=(n, 3)) if "d" in layers else None
    lam, mu = 1.7, 0.6
    pt, st, ptt, stt = E.el3dpartdirecttarg(lam, mu, src, f, s, d, tg)
    for x, skip, p, e in ((src, True, pt, st), (tg, False, ptt, stt)):
        if not len(x):
            continue
        u, h = kelvin(x, src, skip, f, s, d, lam, mu)
        assert np.abs(p - u).max() <= 1e-12 * max(np.abs(u).max(), 1e-300)
        assert np.abs(e - h).max() <= 1e-12 * max(np.abs(h).max(), 1e-300)
    # displacement alone runs without the strain sums
    p0 = E.el3dpartdirecttarg(lam, mu, src, f, s, d, tg, 1, 0, 1, 0)
    assert np.abs(p0[0] - pt).max() <= 1e-13 * max(np.abs(pt).max(), 1e-300)
    if m:
        assert np.abs(p0[2] - ptt).max() <= 1e-13 * np.abs(ptt).max()

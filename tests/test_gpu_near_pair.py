"""The near-field kernel (k_near) on the GPU: its pair code, whose reciprocals and
roots are the hardware's estimates and one step there, against the direct sum's on
single triangles; and near lists of more than 64 boxes, the most it takes at a
time, against the call that stores the interactions, which walks them otherwise."""
import numpy as np
import pytest
import torch

from conftest import rel
from test_gpu_replay import soup
from test_near_pair_host import points

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sl,dl", [(1, 0), (0, 1), (1, 1)])
def test_pairs(gpu_lib, sl, dl):
    """One triangle and targets beside, above, in the plane of and on the lines of
    its edges, one box: near field alone. Tolerance: the closed forms lose up to 8^3
    eps at R/L = 8 times a few tens of terms in either code, 1e-11 of the value."""
    E = gpu_lib
    rng = np.random.default_rng(7 + 2 * sl + dl)
    for t in range(40):
        tri = np.array([[0, 0, 0], [1, 0, 0], [0.4, 0.9, 0]]) + 0.15 * rng.normal(size=(3, 3))
        tri = tri * 10.0 ** rng.uniform(-3, 3) + rng.normal(size=3)
        nrm = np.cross(tri[1] - tri[0], tri[2] - tri[0])
        x = np.array([p for p, own in points(tri, rng) if not own])
        s, d = rng.normal(size=(2, 1, 3))
        geo = (*rng.uniform(0.3, 3, 2), tri[None], nrm[None] / np.linalg.norm(nrm), tri.mean(0)[None], s if sl else None,
               d if dl else None, x)
        ier, pt, st, ptt, stt = E.elfmm3dtriatarg(3, *geo)
        assert ier == 0
        pd, sd, ptd, std = E.el3dtriadirecttarg(*geo)
        ier, p0, _, pt0, _ = E.elfmm3dtriatarg(3, *geo, 1, 0, 1, 0)     # without the strain's sums
        assert ier == 0
        for a, b in ((pt, pd), (st, sd), (ptt, ptd), (stt, std), (p0, pd), (pt0, ptd)):
            a, b = a.reshape(len(a), -1), b.reshape(len(b), -1)
            assert (np.abs(a - b).max(1) <= 1e-11 * np.abs(b).max(1)).all(), t


@pytest.mark.parametrize("layers", [(1, 0), (0, 1), (1, 1)])
def test_long_lists(gpu_lib, layers):
    """A finely divided wall beside a nearly empty half, whose leaves touch hundreds
    of boxes; the points of the empty half. Tolerance: R/L up to 17 between them and
    the wall, 17^3 eps in either pair code times some tens of terms, times 10 for the
    slimmest of the random triangles: 1e-9; a box left out is a part in a hundred."""
    E = gpu_lib
    rng = np.random.default_rng(13)
    c = np.concatenate([np.stack([np.full(24000, 0.502), *rng.random((2, 24000))], 1), rng.random((40, 3)) * [0.45, 1, 1],
                        [[0, 0, 0], [1, 1, 1]]])
    tri, nrm, src = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in soup(c, 0.02, rng))
    n, wsave = len(src), np.zeros(8)
    z = lambda *s: torch.zeros(s, dtype=torch.float64, device="cuda")
    s, d = (torch.from_numpy(rng.normal(size=(n, 3))).cuda() if on else None for on in layers)
    pt, st, p2, s2 = z(n, 3), z(n, 3, 3), z(n, 3), z(n, 3, 3)
    for icomp, a, b in ((1, pt, st), (2, p2, s2)):
        assert E.elfmm3dtriatargiter_dev(-2, 1.3, 0.8, tri, nrm, src, s, d, None, a, b, None, None, icomp, wsave)[0] == 0
    assert E.iter_release(wsave) == 1
    for a, b in ((pt, p2), (st, s2)):
        assert rel(a[24000:].cpu().numpy(), b[24000:].cpu().numpy()) < 1e-9

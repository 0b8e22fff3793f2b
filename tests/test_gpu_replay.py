"""The replay of the stored near field (k_near_replay) against the products
without a store, where its tasks can go wrong: 1 to 17 points a leaf (tasks of
4, 2 or 1, chunks of 16), lists of a few slots, and 1, 3, 5 and 9 density sets
(4 or 8 a pass); and lists of more boxes than fit at once (512) against the
call that stores, which sums the fields it stores by another walk.

Tolerance: the same pairs' fields from another expression of the kernel
(integrals of the unit densities), summed in another order: a few hundred
roundings of 1.1e-16 each against the norm of the result, below 1e-12."""
import numpy as np
import pytest
import torch

from conftest import rel

pytestmark = pytest.mark.gpu


def soup(centres, size, rng):
    tri = centres[:, None, :] + size * rng.normal(size=(len(centres), 3, 3))
    nrm = np.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])
    return tri, nrm / np.linalg.norm(nrm, axis=1, keepdims=True), tri.mean(1)


def wall(rng):
    """A finely divided wall beside a nearly empty half: the empty half's leaves
    touch more than 512 boxes."""
    c = np.concatenate([np.stack([np.full(24000, 0.502), *rng.random((2, 24000))], 1), rng.random((40, 3)) * [0.45, 1, 1],
                        [[0, 0, 0], [1, 1, 1]]])
    return soup(c, 1e-4, rng)


def scattered(n):
    return lambda rng: soup(rng.random((n, 3)) ** 2, 0.01, rng)


@pytest.mark.parametrize("mesh,iprec", [(scattered(1), -2), (scattered(67), -2), (scattered(700), -1), (scattered(1500), 1)])
@pytest.mark.parametrize("layers", [(1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("fields", [(1, 0), (0, 1), (1, 1)])
def test_replay(gpu_lib, mesh, iprec, layers, fields):
    E = gpu_lib
    rng = np.random.default_rng(11)
    tri, nrm, src = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in mesh(rng))
    n, wsave = len(src), np.zeros(8)
    z = lambda on, *s: torch.zeros(s, dtype=torch.float64, device="cuda") if on else None
    den = lambda on, r: torch.from_numpy(rng.normal(size=(r, n, 3))).cuda() if on else None
    one = lambda d, r: None if d is None else d[r].contiguous()
    first = den(layers[0], 1), den(layers[1], 1)
    pt, st = z(fields[0], n, 3), z(fields[1], n, 3, 3)
    product = lambda s, d, icomp: E.elfmm3dtriatargiter_dev(iprec, 1.3, 0.8, tri, nrm, src, s, d, None, pt, st, None, None,
                                                            icomp, wsave)[0]
    assert product(one(first[0], 0), one(first[1], 0), 2) == 0
    for sets in (1, 3, 5, 9):
        s, d = den(layers[0], sets), den(layers[1], sets)
        P, Q = z(fields[0], sets, n, 3), z(fields[1], sets, n, 3, 3)
        if sets == 1:
            assert product(one(s, 0), one(d, 0), 3) == 0
            P, Q = (None if a is None else a.clone()[None] for a in (pt, st))
        else:
            assert E.triatargiter_multi_dev(iprec, 1.3, 0.8, tri, nrm, src, s, d, None, P, Q, None, None, wsave) == 0
        for r in {0, sets - 1}:
            assert product(one(s, r), one(d, r), 1) == 0
            for a, b in ((P, pt), (Q, st)):
                if a is not None:
                    assert rel(a[r].cpu().numpy(), b.cpu().numpy()) < 1e-12
    assert E.iter_release(wsave) == 1


@pytest.mark.parametrize("layers", [(1, 0), (0, 1), (1, 1)])
def test_long_lists(gpu_lib, layers):
    """Tolerance: the same stored values and densities, at most 10^4 terms a point in
    another order, far fields' atomics too: 1e-12 as above."""
    E = gpu_lib
    rng = np.random.default_rng(12)
    tri, nrm, src = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in wall(rng))
    n, wsave = len(src), np.zeros(8)
    z = lambda *s: torch.zeros(s, dtype=torch.float64, device="cuda")
    s, d = (torch.from_numpy(rng.normal(size=(3, n, 3))).cuda() if on else None for on in layers)
    s0, d0 = (None if a is None else a[2].contiguous() for a in (s, d))
    pt, st, p3, s3, pm, sm = z(n, 3), z(n, 3, 3), z(n, 3), z(n, 3, 3), z(3, n, 3), z(3, n, 3, 3)
    for icomp, a, b in ((2, pt, st), (3, p3, s3)):
        assert E.elfmm3dtriatargiter_dev(-2, 1.3, 0.8, tri, nrm, src, s0, d0, None, a, b, None, None, icomp, wsave)[0] == 0
    assert E.triatargiter_multi_dev(-2, 1.3, 0.8, tri, nrm, src, s, d, None, pm, sm, None, None, wsave) == 0
    for got in ((p3, s3), (pm[2], sm[2])):
        for a, b in zip(got, (pt, st)):
            assert rel(a.cpu().numpy(), b.cpu().numpy()) < 1e-12
    assert E.iter_release(wsave) == 1

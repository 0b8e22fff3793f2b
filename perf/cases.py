"""Performance cases: the calls a user of elfmmlib3d_amd makes, over the range of
sizes, precisions and layers they are made at.

Kinds (the "kind" of a case):

tri     elfmm3dtriatarg_dev, one free-space apply of triangle layers on a closed
        surface (an icosphere, turned at random): a boundary-element matvec or
        a field evaluation, inputs resident on the GPU.
host    elfmm3dtriatarg, the same with host arrays in and out: the drop-in call
        of a Fortran, C or numpy program.
fault   elfmm3dtriatarg_dev on planar faults in z < 0 (double layer: slip).
points  elfmm3dparttarg_dev, point sources.
iter    elfmm3dtriatargiter_dev, icomp 3: one product of an iterative solve, the
        near field stored beforehand (icomp 2) and replayed with new densities.
half    the half-space product of a fault model: the direct arrival
        (elfmm3dtriatargiter_dev, icomp 3) plus the image part
        (elhfmm3dtriatargiter_dev, icomp 3) at the centroids.
batch   MeshBatch.apply, many meshes in one call (the forest schedule).

Geometry, densities and targets come from the seed alone. lam, mu vary with the
case. Every call in a case computes all the outputs it names.
"""
import math

import numpy as np
import torch

import elfmmlib3d_amd as E

DEV = "cuda"


def listed():
    return [
        # a handful of elements: launches and host latency are all there is
        dict(name="tri_tiny", kind="tri", split=3, targets=37, iprec=2, sl=True, dl=True, strain=True),
        # the reference's example size, called as its users call it
        dict(name="host_c1", kind="host", split=12, targets=1000, iprec=2, sl=True, dl=True, strain=True),
        # the benchmark's mesh: both layers on the surface and at targets around it
        dict(name="tri_c2", kind="tri", split=64, targets=100000, iprec=2, sl=True, dl=True, strain=True),
        # a single-layer potential at three digits, no strain
        dict(name="tri_sl", kind="tri", split=37, targets=20011, iprec=1, sl=True, dl=False, strain=False),
        # nine digits
        dict(name="tri_p3", kind="tri", split=32, targets=20480, iprec=3, sl=True, dl=True, strain=True),
        # slip on faults, stresses on the faults themselves
        dict(name="fault_dl", kind="fault", triangles=20000, iprec=1, sl=False, dl=True, strain=True),
        # particles: the sample and the large run of the benchmark, and a small one with targets
        dict(name="points_100k", kind="points", n=100000, targets=0, iprec=2, sl=True, dl=True, strain=True),
        dict(name="points_1m", kind="points", n=1000000, targets=0, iprec=2, sl=True, dl=True, strain=True),
        dict(name="points_small", kind="points", n=3001, targets=703, iprec=1, sl=False, dl=True, strain=True),
        # one product of a solve on a closed surface
        dict(name="iter_48", kind="iter", split=48, iprec=2, sl=True, dl=True, strain=False),
        # one product of a fault model below a free surface
        dict(name="half_20k", kind="half", triangles=20000, iprec=2, sl=False, dl=True, strain=True),
        # several meshes at once
        dict(name="batch_24", kind="batch", meshes=24, largest=8000, iprec=2, sl=True, dl=True, strain=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tri", "tri", "host", "fault", "points", "points", "iter", "half", "batch"])
    iprec = rng.choice([0, 1, 1, 2, 2, 2, 3])
    sl, dl = rng.choice([(True, True), (True, True), (True, False), (False, True)])
    c = dict(kind=kind, iprec=iprec, sl=sl, dl=dl, strain=rng.random() < 0.7)
    big = iprec < 3
    if kind == "tri":
        c.update(split=_log(rng, 3, 64 if big else 32), targets=_log(rng, 1, 100000 if big else 20480))
    elif kind == "host":
        c.update(split=_log(rng, 3, 32), targets=_log(rng, 1, 20000))
    elif kind == "fault":
        c.update(triangles=_log(rng, 200, 60000 if big else 20000), sl=False, dl=True)
    elif kind == "points":
        c.update(n=_log(rng, 300, 600000 if big else 100000), targets=rng.choice([0, _log(rng, 10, 50000)]))
    elif kind == "iter":
        c.update(split=_log(rng, 6, 48 if big else 32))
    elif kind == "half":
        c.update(triangles=_log(rng, 500, 20000), sl=False, dl=True, iprec=rng.choice([0, 1, 2]))
    else:
        c.update(meshes=rng.randint(3, 30), largest=_log(rng, 600, 8000), iprec=rng.choice([1, 2]))
    return c


# ---- geometry (numpy, a few tens of milliseconds at the largest size) -------

def _sphere(split, rng, radius=1.0, center=(0.0, 0.0, 0.0)):
    """Flat triangles of an icosphere, each icosahedron face cut into split x
    split triangles and projected, turned at random."""
    from elfmmlib3d_amd.mesh import icosahedron
    v, f = icosahedron()
    i, j = np.meshgrid(np.arange(split), np.arange(split), indexing="ij")
    up = i + j < split
    dn = i + j < split - 1
    cells = [np.stack([np.stack([i[up] + a, j[up] + b], -1) for a, b in ((0, 0), (1, 0), (0, 1))], 1),
             np.stack([np.stack([i[dn] + a, j[dn] + b], -1) for a, b in ((1, 0), (1, 1), (0, 1))], 1)]
    ij = np.concatenate(cells).astype(float) / split
    A, B, C = v[f[:, 0]], v[f[:, 1]], v[f[:, 2]]
    p = A[:, None, None] + (B - A)[:, None, None] * ij[None, :, :, :1] + (C - A)[:, None, None] * ij[None, :, :, 1:]
    p /= np.linalg.norm(p, axis=-1, keepdims=True)
    q, r = np.linalg.qr(rng.normal(size=(3, 3)))
    q = q * np.sign(np.diag(r))
    if np.linalg.det(q) < 0:
        q[:, 0] = -q[:, 0]
    return np.ascontiguousarray((p.reshape(-1, 3, 3) @ q.T) * radius + np.asarray(center))


def _faults(total, rng):
    """Eight rectangular faults in z < 0, cut into about total right triangles
    (their lengths and widths are always the same: the count does not change)."""
    k = 8
    size = np.random.default_rng(33)
    L, W = size.uniform(2.0, 10.0, k), size.uniform(1.0, 5.0, k)
    dip, strike = np.deg2rad(rng.uniform(15.0, 90.0, k)), rng.uniform(0, 2 * np.pi, k)
    top, cx, cy = rng.uniform(0.0, 3.0, k), rng.uniform(-10, 10, k), rng.uniform(-10, 10, k)
    h = math.sqrt(2.0 * float(np.sum(L * W)) / total)
    out = []
    for a in range(k):
        nl, nw = max(1, round(L[a] / h)), max(1, round(W[a] / h))
        s = np.array([np.cos(strike[a]), np.sin(strike[a]), 0.0])
        d = np.array([-np.sin(strike[a]) * np.cos(dip[a]), np.cos(strike[a]) * np.cos(dip[a]), -np.sin(dip[a])])
        o = np.array([cx[a], cy[a], -top[a] - 1e-3]) - s * L[a] / 2
        i, j = (x.reshape(-1, 1) for x in np.meshgrid(np.arange(nl), np.arange(nw), indexing="ij"))
        P = lambda u, w: o + s * (L[a] * (i + u) / nl) + d * (W[a] * (j + w) / nw)
        p00, p10, p01, p11 = P(0, 0), P(1, 0), P(0, 1), P(1, 1)
        out += [np.stack([p00, p10, p11], 1), np.stack([p00, p11, p01], 1)]
    return np.ascontiguousarray(np.concatenate(out))


def _normals(tri):
    n = np.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 1])
    return n / np.linalg.norm(n, axis=1)[:, None]


def _cube_targets(m, rng):
    """m points uniform in [-2, 2]^3 outside the unit ball."""
    out = np.empty((0, 3))
    while out.shape[0] < m:
        p = rng.uniform(-2, 2, (2 * m + 8, 3))
        out = np.concatenate([out, p[np.linalg.norm(p, axis=1) > 1.0]])
    return np.ascontiguousarray(out[:m])


def _problem(case, seed):
    """Everything a case's call takes, as host arrays (None where off)."""
    rng = np.random.default_rng(seed)
    c = dict(case)
    d = dict(lam=float(rng.uniform(0.5, 2.0)), mu=float(rng.uniform(0.5, 2.0)), tg=None)
    if c["kind"] == "points":
        n = c["n"]
        d["src"] = rng.uniform(0, 1, (n, 3))
        dv = rng.normal(size=(n, 3))
        d["dv"] = dv / np.linalg.norm(dv, axis=1)[:, None] if c["dl"] else None
        if c["targets"]:
            d["tg"] = rng.uniform(0, 1, (c["targets"], 3))
    elif c["kind"] == "batch":
        d["meshes"] = []
        for cnt in np.geomspace(c["largest"], 200, c["meshes"]):
            split = max(1, int(round(math.sqrt(cnt / 20.0))))
            d["meshes"].append(_sphere(split, rng, rng.uniform(0.5, 3.0), rng.uniform(-20, 20, 3)))
        n = sum(t.shape[0] for t in d["meshes"])
    else:
        tri = _faults(c["triangles"], rng) if c["kind"] in ("fault", "half") else _sphere(c["split"], rng)
        n = tri.shape[0]
        d["tri"], d["nrm"], d["src"] = tri, _normals(tri), np.ascontiguousarray(tri.mean(1))
        if c["kind"] in ("tri", "host"):
            d["tg"] = _cube_targets(c["targets"], rng)
    d["sl"] = rng.uniform(-1, 1, (n, 3)) if c["sl"] else None
    d["dl"] = rng.uniform(-1, 1, (n, 3)) if c["dl"] else None
    d["n"], d["m"] = n, 0 if d["tg"] is None else d["tg"].shape[0]
    return d


# ---- the calls --------------------------------------------------------------

class _Store:
    """A device store of near-field interactions, named by its wsave."""

    def __init__(self):
        self.wsave = np.zeros(8)

    def __del__(self):
        try:
            E.iter_release(self.wsave)
        except Exception:
            pass


def _dev(a):
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _check(ier):
    if ier != 0:
        raise RuntimeError("ier=%d" % ier)


def prepare(case, seed):
    d = _problem(case, seed)
    s = dict(case=dict(case), lam=d["lam"], mu=d["mu"], n=d["n"], m=d["m"])
    if case["kind"] == "host":
        s.update((k, d[k]) for k in ("tri", "nrm", "src", "sl", "dl", "tg"))
        return s
    out = lambda k, on: torch.empty((k, 3), dtype=torch.float64, device=DEV) if on else None
    st = lambda k, on: torch.empty((k, 3, 3), dtype=torch.float64, device=DEV) if on and case["strain"] else None
    s.update(sl=_dev(d["sl"]), dl=_dev(d["dl"]))
    if case["kind"] == "batch":
        ms = [(_dev(t), _dev(_normals(t)), _dev(t.mean(1)), None) for t in d["meshes"]]
        s["batch"] = E.MeshBatch(case["iprec"], s["lam"], s["mu"], ms, ifsingle=case["sl"], ifdouble=case["dl"],
                                 ifptfrc=True, ifstrain=case["strain"], ifptfrctarg=False, ifstraintarg=False,
                                 width=-100)
        return s
    s.update((k, _dev(d.get(k))) for k in ("tri", "nrm", "src", "dv", "tg"))
    n, m = s["n"], s["m"]
    s.update(pt=out(n, True), st=st(n, True), ptt=out(m, m), stt=st(m, m))
    if case["kind"] in ("iter", "half"):
        # the solve's first product, with other densities, keeps the near field
        first = lambda x: None if x is None else x.flip(0).contiguous()
        first_sl, first_dl = first(s["sl"]), first(s["dl"])
        if case["kind"] == "iter":
            s["store"] = _Store()
            _check(E.elfmm3dtriatargiter_dev(case["iprec"], s["lam"], s["mu"], s["tri"], s["nrm"], s["src"], first_sl,
                                             first_dl, None, s["pt"], s["st"], None, None, 2, s["store"].wsave)[0])
        else:
            s.update(store=_Store(), image=_Store(), pti=out(n, True), sti=st(n, True))
            _check(E.elfmm3dtriatargiter_dev(case["iprec"], s["lam"], s["mu"], s["tri"], s["nrm"], s["src"], first_sl,
                                             first_dl, None, s["pt"], s["st"], None, None, 2, s["store"].wsave)[0])
            _check(E.elhfmm3dtriatargiter_dev(case["iprec"], s["lam"], s["mu"], s["tri"], s["nrm"], s["src"], first_sl,
                                              first_dl, s["src"], s["pti"], s["sti"], 2, s["image"].wsave)[0])
    return s


def run(s):
    c = s["case"]
    kind, ip, lam, mu = c["kind"], c["iprec"], s["lam"], s["mu"]
    if kind in ("tri", "fault"):
        _check(E.elfmm3dtriatarg_dev(ip, lam, mu, s["tri"], s["nrm"], s["src"], s["sl"], s["dl"], s["tg"], s["pt"],
                                     s["st"], s["ptt"], s["stt"]))
        return [s["pt"], s["st"], s["ptt"], s["stt"]]
    if kind == "host":
        ier, pt, st, ptt, stt = E.elfmm3dtriatarg(ip, lam, mu, s["tri"], s["nrm"], s["src"], s["sl"], s["dl"], s["tg"],
                                                  1, int(c["strain"]), 1, int(c["strain"]))
        _check(ier)
        return [pt, st if c["strain"] else None, ptt, stt if c["strain"] else None]
    if kind == "points":
        _check(E.elfmm3dparttarg_dev(ip, lam, mu, s["src"], s["sl"], s["dl"], s["dv"], s["tg"], s["pt"], s["st"],
                                     s["ptt"], s["stt"]))
        return [s["pt"], s["st"], s["ptt"], s["stt"]]
    if kind == "iter":
        _check(E.elfmm3dtriatargiter_dev(ip, lam, mu, s["tri"], s["nrm"], s["src"], s["sl"], s["dl"], None, s["pt"],
                                         s["st"], None, None, 3, s["store"].wsave)[0])
        return [s["pt"], s["st"]]
    if kind == "half":
        _check(E.elfmm3dtriatargiter_dev(ip, lam, mu, s["tri"], s["nrm"], s["src"], s["sl"], s["dl"], None, s["pt"],
                                         s["st"], None, None, 3, s["store"].wsave)[0])
        _check(E.elhfmm3dtriatargiter_dev(ip, lam, mu, s["tri"], s["nrm"], s["src"], s["sl"], s["dl"], s["src"],
                                          s["pti"], s["sti"], 3, s["image"].wsave)[0])
        return [s["pt"], s["st"], s["pti"], s["sti"]]
    return s["batch"].apply(s["sl"], s["dl"])


# ---- what a pass cannot do without ------------------------------------------

def _sizes(case):
    """(elements, further evaluation points)."""
    if case["kind"] == "points":
        return case["n"], case["targets"]
    if case["kind"] == "batch":
        c = case["largest"]
        return int(c + (case["meshes"] - 1) * (c - 200) / math.log(c / 200.0)), 0
    if case["kind"] in ("fault", "half"):
        return case["triangles"], 0
    return 20 * case["split"] ** 2, case.get("targets", 0)


def work(case):
    """Bytes: inputs, outputs and, in the stored products, the stored
    interactions. Flops: the near pairs (about 500 operations for a triangle
    pair, 100 for a point pair, at the leaf sizes of the method) and the far
    field, which grows with the square of the expansion order."""
    n, m = _sizes(case)
    pts = n + m
    nl = int(case["sl"]) + int(case["dl"])
    comps = 3 + (9 if case["strain"] else 0)
    point = case["kind"] == "points"
    per = (3 + 3 * nl + 3 * int(case["dl"])) if point else (15 + 3 * nl)
    passes = 2 if case["kind"] == "half" else 1
    io = passes * 8.0 * (n * per + m * 3 + pts * comps)
    order = {0: 9, 1: 14, 2: 26, 3: 39}[case["iprec"]]
    stored = case["kind"] in ("iter", "half")
    near = min(n, {0: 60, 1: 90, 2: 140, 3: 200}[case["iprec"]] * (40 if point else 4 if stored else 1))
    far = 1500.0 * order ** 2 * (0.1 if point else 1.0) if n > 1000 else 0.0
    if stored:
        words = nl * 3 * (3 + (6 if case["strain"] else 0))
        return {"bytes": io + 8.0 * near * words * n, "flops": passes * pts * far + 2.0 * near * words * n}
    return {"bytes": io, "flops": pts * (far + near * (100.0 if point else 500.0 * nl))}


# ---- values in 64 bits ------------------------------------------------------
# Direct sums over all pairs in plain torch: the point kernels as they are
# written, and for a flat triangle the integrals over its edges.

def _kelvin_points(x, self0, d, mu, c1, strain):
    """Displacement and strain at points x of all point sources; self0: x are
    the sources themselves starting there (their own pair left out). With
    R = x - y: single layer ((2 - c1) f / r + c1 R (R.f) / r^3) / (2 mu), double
    layer c2 (s (R.n) + n (R.s) - R (n.s)) / r^3 + 3 c1 R (R.s) (R.n) / r^5."""
    src, c2 = _dev(d["src"]), 1.0 - c1
    one = torch.zeros_like(src)
    f = one if d["sl"] is None else _dev(d["sl"]) / (2 * mu)
    s = one if d["dl"] is None else _dev(d["dl"])
    n = one if d["dl"] is None else _dev(d["dv"])
    ns = (n * s).sum(1)
    f, s, n, y = f.T.contiguous(), s.T.contiguous(), n.T.contiguous(), src.T.contiguous()
    U = torch.zeros((x.shape[0], 3), dtype=torch.float64, device=DEV)
    H = torch.zeros((x.shape[0], 3, 3), dtype=torch.float64, device=DEV)
    step = max(1, 4_000_000 // src.shape[0])
    for a in range(0, x.shape[0], step):
        X = x[a:a + step]
        R = [X[:, c:c + 1] - y[c] for c in range(3)]
        r2 = R[0] * R[0] + R[1] * R[1] + R[2] * R[2]
        if self0 is not None:
            k = torch.arange(X.shape[0], device=DEV)
            r2[k, self0 + a + k] = math.inf
        i1 = r2.rsqrt()
        i2 = i1 * i1
        i3 = i1 * i2
        i5 = i3 * i2
        dot = lambda v: R[0] * v[0] + R[1] * v[1] + R[2] * v[2]
        fR = dot(f) if d["sl"] is not None else 0.0
        sR, nR = (dot(s), dot(n)) if d["dl"] is not None else (0.0, 0.0)
        sn5 = (3 * c1) * sR * nR * i5
        along = c1 * fR * i3 - c2 * ns * i3 + sn5                              # of R in u, of the unit tensor in the gradient
        for c in range(3):
            u = along * R[c]
            if d["sl"] is not None:
                u = u + ((2 - c1) * f[c]) * i1
            if d["dl"] is not None:
                u = u + (c2 * i3) * (s[c] * nR + n[c] * sR)
            U[a:a + step, c] = u.sum(1)
        if not strain:
            continue
        RR = (3 * i5) * (c2 * ns - c1 * fR) - (5 * i2) * sn5                   # of R R
        b = 3 * (c1 - c2) * i5
        p = [0.0] * 3                                                          # of R, symmetrised
        for c in range(3):
            if d["sl"] is not None:
                p[c] = p[c] + ((2 * c1 - 2) * f[c]) * i3
            if d["dl"] is not None:
                p[c] = p[c] + b * (s[c] * nR + n[c] * sR)
        for i in range(3):
            for j in range(i, 3):
                g = RR * R[i] * R[j] + (R[i] * p[j] + R[j] * p[i]) / 2
                if d["dl"] is not None:
                    g = g + (c2 * (s[i] * n[j] + n[i] * s[j])) * i3
                if i == j:
                    g = g + along
                H[a:a + step, i, j] = H[a:a + step, j, i] = g.sum(1)
    return U, H


def _triangles(x, self0, tri, sl, dl, lam, mu, strain):
    """Displacement and strain at points x of the layers on flat triangles."""
    c1 = (lam + mu) / (lam + 2 * mu)
    tri = _dev(tri)
    e1 = tri[:, 1] - tri[:, 0]
    e1 = e1 / e1.norm(dim=1, keepdim=True)
    e3 = torch.linalg.cross(e1, tri[:, 2] - tri[:, 0])
    e3 = e3 / e3.norm(dim=1, keepdim=True)
    F = torch.stack([e1, torch.linalg.cross(e3, e1), e3], 1)             # rows: the local axes
    loc = lambda s: None if s is None else torch.einsum("nij,nj->ni", F, _dev(s))
    sl, dl = loc(sl), loc(dl)
    V = torch.einsum("nij,nkj->nki", F, tri - tri[:, :1])                  # local vertices
    n = tri.shape[0]
    U = torch.zeros((x.shape[0], 3), dtype=torch.float64, device=DEV)
    H = torch.zeros((x.shape[0], 3, 3), dtype=torch.float64, device=DEV)
    step = max(1, 10_000_000 // n)
    for a in range(0, x.shape[0], step):
        X = torch.einsum("nij,pnj->ipn", F, x[a:a + step, None] - tri[None, :, 0])
        x0, y0, z0 = X[0], X[1], X[2].clone()
        if self0 is not None:
            k = torch.arange(x0.shape[0], device=DEV)
            z0[k, self0 + a + k] = 0.0
        w = -z0
        zero = torch.zeros_like(x0)
        T = {}

        def add(key, v):
            T[key] = T[key] + v if key in T else v

        F0 = zero
        for e in range(3):
            p, q = V[:, e], V[:, (e + 1) % 3]
            t = q - p
            L = t.norm(dim=1)
            sx, sy = t[:, 0] / L, t[:, 1] / L
            t1 = (p[:, 0] - x0) * sx + (p[:, 1] - y0) * sy
            de = (p[:, 0] - x0) * sy - (p[:, 1] - y0) * sx
            t2 = t1 + L
            r2 = de * de + w * w
            rho = r2.sqrt()
            ra, rb = (t1 * t1 + r2).sqrt(), (t2 * t2 + r2).sqrt()
            # int t^m / (t^2 + rho^2)^(q/2) over the edge
            lo, hi = torch.where(t2 <= 0, -t2, t1), torch.where(t2 <= 0, -t1, t2)
            rl, rh = torch.where(t2 <= 0, rb, ra), torch.where(t2 <= 0, ra, rb)
            k01 = torch.where(lo >= 0, torch.log((hi + rh) / (lo + rl)), torch.asinh(hi / rho) - torch.asinh(lo / rho))
            k11 = (t2 - t1) * (t2 + t1) / (ra + rb)
            # t / (rho^2 r) = 1/rho^2 - 1 / (r (r + t)), the two forms by side
            k03 = torch.where(lo >= 0, 1 / (rl * (rl + lo)) - 1 / (rh * (rh + hi)), (hi / rh - lo / rl) / r2)
            k13 = k11 / (ra * rb)
            k23 = k01 - r2 * k03
            nx, ny = sy, -sx
            s, v, nn = (sx, sy, None), (de * nx, de * ny, w), (nx, ny)
            F0 = F0 + de * k01
            m1 = [(0 if s[i] is None else s[i] * k11) + v[i] * k01 for i in range(3)]

            def m2(i, j, a2, a1, a0):
                r = v[i] * v[j] * a0
                if s[i] is not None:
                    r = r + s[i] * v[j] * a1
                if s[j] is not None:
                    r = r + v[i] * s[j] * a1
                if s[i] is not None and s[j] is not None:
                    r = r + s[i] * s[j] * a2
                return r

            for ax in range(2):
                add("r%d" % ax, nn[ax] * k01)
                for i in range(3):
                    add("b%d%d" % (ax, i), nn[ax] * m1[i])
                    for j in range(i, 3):
                        d2 = -m2(i, j, k23, k13, k03)
                        if i == j:
                            d2 = d2 + k01
                        add("c%d%d%d" % (ax, i, j), nn[ax] * d2)
            if dl is not None and strain:
                # int t^m / (t^2 + rho^2)^(5/2)
                k05 = (2 * k03 + (t2 / rb ** 3 - t1 / ra ** 3)) / (3 * r2)
                far = (lo > 0) & (r2 < 0.04 * lo * lo)
                if bool(far.any()):
                    # beside the edge's own line: series in (rho / t)^2
                    ser, cof = zero, 1.0
                    lo_, hi_ = torch.where(far, lo, zero + 1), torch.where(far, hi, zero + 2)
                    for k_ in range(24):
                        ser = ser + cof * r2 ** k_ * (lo_ ** (-4 - 2 * k_) - hi_ ** (-4 - 2 * k_)) / (4 + 2 * k_)
                        cof *= -(2.5 + k_) / (k_ + 1)
                    k05 = torch.where(far, ser, k05)
                k15 = (1 / ra ** 3 - 1 / rb ** 3) / 3
                k25 = k03 - r2 * k05
                u3 = [(0 if s[i] is None else s[i] * k13) + v[i] * k03 for i in range(3)]
                for ax in range(2):
                    for i in range(3):
                        add("q%d%d" % (ax, i), -nn[ax] * u3[i])
                        for j in range(i, 3):
                            d3 = 3 * w * m2(i, j, k25, k15, k05)               # d_i d_j d_z r on the edge
                            if i == j:
                                d3 = d3 - u3[2]
                            if j == 2:
                                d3 = d3 - u3[i]
                            if i == 2:
                                d3 = d3 - u3[j]
                            add("d%d%d%d" % (ax, i, j), nn[ax] * d3)
        # the solid angle, zero in the triangle's own plane
        P = [torch.stack([V[:, i, 0] - x0, V[:, i, 1] - y0, -z0]) for i in range(3)]
        l = [p.norm(dim=0) for p in P]
        dot = lambda i, j: (P[i] * P[j]).sum(0)
        den = l[0] * l[1] * l[2] + dot(0, 1) * l[2] + dot(0, 2) * l[1] + dot(1, 2) * l[0]
        wz = torch.where(z0 == 0, zero, 2 * torch.atan2(z0 * V[:, 1, 0] * V[:, 2, 1], den))
        F0 = F0 - z0 * wz
        r1 = [T["r0"], T["r1"], wz]

        def order(pre, idx):
            """A table entry with at least one in-plane index: that index leads."""
            idx = sorted(idx)
            return T["%s%d%s" % (pre, idx[0], "".join(map(str, idx[1:])))]

        def b2(i, j):
            return 2 * F0 - T["b00"] - T["b11"] if i == j == 2 else order("b", (i, j))

        def b3(i, j, k):
            return 2 * wz - order("c", (0, 0, 2)) - order("c", (1, 1, 2)) if i == j == k == 2 else order("c", (i, j, k))

        disp = [zero, zero, zero]
        G = {(i, j): zero for i in range(3) for j in range(i, 3)}
        if sl is not None:
            for i in range(3):
                disp[i] = disp[i] + 2 * sl[:, i] * F0 - c1 * sum(sl[:, k] * b2(i, k) for k in range(3))
            if strain:
                for i, j in G:
                    G[i, j] = G[i, j] + c1 * sum(sl[:, k] * b3(i, j, k) for k in range(3)) - sl[:, i] * r1[j] - sl[:, j] * r1[i]
        if dl is not None:
            sr = sum(dl[:, k] * r1[k] for k in range(3))
            for i in range(3):
                disp[i] = disp[i] + lam * dl[:, 2] * (2 - 2 * c1) * r1[i] + mu * (
                    -2 * c1 * sum(dl[:, k] * b3(i, k, 2) for k in range(3)) + 2 * dl[:, i] * wz + (2 * sr if i == 2 else 0))
            if strain:
                def r2_(i, j):
                    return -T["q00"] - T["q11"] if i == j == 2 else order("q", (i, j))

                def b4(i, j, k):                                               # d_i d_j d_k d_z r
                    if i == j == k == 2:
                        return 2 * r2_(2, 2) - order("d", (0, 0, 2)) - order("d", (1, 1, 2))
                    return order("d", (i, j, k))

                sv = [sum(dl[:, k] * r2_(i, k) for k in range(3)) for i in range(3)]
                for i, j in G:
                    g = lam * dl[:, 2] * (2 - 2 * c1) * r2_(i, j) + mu * (
                        -2 * c1 * sum(dl[:, k] * b4(i, j, k) for k in range(3)) + dl[:, i] * r2_(2, j) + dl[:, j] * r2_(2, i) +
                        (sv[j] if i == 2 else 0) + (sv[i] if j == 2 else 0))
                    G[i, j] = G[i, j] - g
        U[a:a + step] = sum(disp[i] @ F[:, i] for i in range(3)) / (2 * mu)
        if strain:
            for (i, j), g in G.items():
                M = F[:, i, :, None] * F[:, j, None, :]
                M = M if i == j else M + M.mT
                H[a:a + step] += (g @ M.reshape(n, 9)).reshape(-1, 3, 3) / (2 * mu)
    return U, H


def exact(case, seed):
    """Direct sums of all pairs; None where they are too many, and for the
    image part of the half space."""
    n, m = _sizes(case)
    pairs = case["meshes"] * case["largest"] ** 2 / 3 if case["kind"] == "batch" else (n + m) * n
    if pairs > (1.5e10 if case["kind"] == "points" else 2.5e9):
        return None
    d = _problem(case, seed)
    lam, mu, strain = d["lam"], d["mu"], case["strain"]
    c1 = (lam + mu) / (lam + 2 * mu)
    keep = lambda r: [r[0], r[1] if strain else None]
    if case["kind"] == "batch":
        at, us, hs = 0, [], []
        for t in d["meshes"]:
            k = slice(at, at + t.shape[0])
            at += t.shape[0]
            cut = lambda v: None if v is None else v[k]
            u, h = _triangles(_dev(t.mean(1)), 0, t, cut(d["sl"]), cut(d["dl"]), lam, mu, strain)
            us.append(u)
            hs.append(h)
        return [torch.cat(us), torch.cat(hs) if strain else None, None, None]
    if case["kind"] == "points":
        one = lambda x, s0: keep(_kelvin_points(_dev(x), s0, d, mu, c1, strain))
    else:
        one = lambda x, s0: keep(_triangles(_dev(x), s0, d["tri"], d["sl"], d["dl"], lam, mu, strain))
    r = one(d["src"], 0)
    if case["kind"] == "iter":
        return r
    if case["kind"] == "half":
        return r + [None, None]
    return r + (one(d["tg"], None) if d["m"] else [None, None])

"""Workloads of the pair counters, for timing them and for checking their results.

Each case is one call (or one training / fitting step) that a program using
this package makes, with the sizes of the package's benchmark and example
configurations: catalogues of 1e3 to 2e6 points in a periodic box of side
250-1000 Mpc/h (or an unperiodic survey volume with a random catalogue),
clustered like an NFW halo catalogue or uniform like a random one, 10-30
radial edges, (rp, pi) grids up to 16 x 41, and batches of up to 64 mocks.

``listed()`` gives the fixed cases, ``draw(rng)`` one more of the same ranges,
``prepare`` the inputs on the GPU, ``run`` one pass through the public entry
points, ``work`` the bytes and operations a pass cannot do without, and
``exact`` the floating-point results in plain 64-bit torch (a padded-grid
neighbour search that shares no code with the package).
"""
import math

import numpy as np
import torch

from halotools_amd import batch, mocks
from halotools_amd.autodiff import marked_npairs_3d_product
from halotools_amd.mock_observables import (marked_npairs_3d, marked_npairs_xy_z, npairs_3d, npairs_jackknife_3d,
                                            npairs_per_object_3d, npairs_projected, npairs_xy_z, tpcf, wp)


def listed():
    return [
        # the smallest calls: a 20k x 20k cross count in a 250 Mpc/h box (one snapshot of a small
        # simulation, cross-correlated with a tracer sample); latency, launches and host work count
        dict(name="npairs_3d cross 20k", kind="npairs_3d", n1=20000, n2=20000, L=250.0, rmin=0.1, rmax=20.0, nbins=15,
             clustered=False),
        # the headline workload: auto-count of a ~1M-galaxy clustered catalogue, 20 log edges to 50 Mpc/h
        dict(name="npairs_3d auto 1M", kind="npairs_3d", n1=999637, n2=0, L=1000.0, rmin=0.1, rmax=50.0, nbins=20,
             clustered=True),
        # an unperiodic survey: Landy-Szalay xi(r) from a data catalogue and a 4x random catalogue (DD, DR, RR)
        dict(name="tpcf survey LS", kind="tpcf", n1=60007, n2=240011, L=400.0, rmin=1.0, rmax=25.0, nbins=16,
             clustered=True),
        # redshift-space counts xi(rp, pi) of a random-like 2M sample: 16 x 41 edges
        dict(name="npairs_xy_z auto 2M", kind="npairs_xy_z", n1=2000000, n2=0, L=1000.0, rmin=0.1, rmax=30.0, nbins=16,
             pimax=40.0, npi=41, clustered=False),
        # the projected correlation function of a periodic box, analytic randoms
        dict(name="wp 500k", kind="wp", n1=500009, n2=0, L=500.0, rmin=0.1, rmax=30.0, nbins=16, pimax=40.0,
             clustered=True),
        # galaxy-matter like cross count: a sparse tracer against a dense particle sample, to pi_max
        dict(name="npairs_projected cross", kind="npairs_projected", n1=150001, n2=1000003, L=1000.0, rmin=0.1,
             rmax=30.0, nbins=16, pimax=40.0, clustered=True),
        # model fitting by autograd: product marks of 1M halos, forward and backward to two HOD parameters
        dict(name="marked product grad 1M", kind="marked_grad", n1=1000000, n2=0, L=1000.0, rmin=0.1, rmax=50.0,
             nbins=20, clustered=False),
        # a marked correlation with one of the general marking functions (two marks per point, compared pairwise)
        dict(name="marked_3d generic 200k", kind="marked_3d", n1=200003, n2=0, L=500.0, rmin=0.1, rmax=30.0, nbins=14,
             wfunc=5, clustered=True),
        # marked counts on an (rp, pi) grid
        dict(name="marked_xy_z 1M", kind="marked_xy_z", n1=1000000, n2=0, L=1000.0, rmin=0.1, rmax=30.0, nbins=16,
             pimax=40.0, npi=41, wfunc=1, clustered=False),
        # per-galaxy neighbour counts (environment measures) of the clustered catalogue
        dict(name="npairs_per_object 1M", kind="per_object", n1=999637, n2=0, L=1000.0, rmin=0.1, rmax=50.0, nbins=20,
             clustered=True),
        # jackknife tables of the clustered catalogue, 125 spatial subvolumes
        dict(name="npairs_jackknife 1M", kind="jackknife", n1=999637, n2=0, L=1000.0, rmin=0.1, rmax=50.0, nbins=20,
             side=5, clustered=True),
        # the largest: one fitting step over 64 mocks of 5e4 to 2e6 points (counts, marked sums, gradients)
        dict(name="batch step 64 mocks", kind="batch", mocks=64, nmin=50000, nmax=2000000, L=1000.0, rmin=0.1,
             rmax=50.0, nbins=20),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["npairs_3d", "npairs_3d", "tpcf", "npairs_xy_z", "wp", "npairs_projected", "marked_grad",
                       "marked_3d", "marked_xy_z", "per_object", "jackknife", "batch"])
    L = rng.choice([250.0, 400.0, 500.0, 750.0, 1000.0])
    c = dict(kind=kind, L=L, rmin=rng.choice([0.1, 0.2, 0.5]), nbins=rng.randint(10, 30),
             clustered=rng.random() < 0.5)
    # search lengths of 2-8 % of the box, at most 50 Mpc/h
    c["rmax"] = round(min(50.0, L * math.exp(rng.uniform(math.log(0.02), math.log(0.08)))), 3)
    # at most ~2e9 ordered pairs inside the search length
    cap = math.sqrt(2e9 / (4.0 / 3.0 * math.pi * (c["rmax"] / L) ** 3))  # uniform density
    hi = min(2.0e6 if kind in ("npairs_3d", "npairs_xy_z") else 1.0e6, cap)
    c["n1"] = _logint(rng, 1e3, hi)
    c["n2"] = 0
    if kind == "npairs_3d" and rng.random() < 0.4:
        c["n2"] = _logint(rng, 1e3, hi)
    if kind == "npairs_projected":
        c["n2"] = _logint(rng, 1e3, hi)
    if kind == "tpcf":
        c["n1"] = _logint(rng, 5e3, min(1e5, cap / 4))
        c["n2"] = int(c["n1"] * rng.uniform(3.0, 5.0))
        # the innermost bins of the random catalogue must hold pairs (the estimator divides by them)
        c["nbins"] = min(c["nbins"], 14)
        c["rmin"] = round(c["rmax"] * 0.25, 3)
    if kind in ("npairs_xy_z", "wp", "npairs_projected", "marked_xy_z"):
        c["rmax"] = round(min(c["rmax"], 30.0), 3)
        c["pimax"] = float(rng.choice([20, 25, 40]))
    if kind in ("npairs_xy_z", "marked_xy_z"):
        c["npi"] = int(c["pimax"]) + 1
        c["nbins"] = rng.randint(8, 16)
    if kind in ("marked_3d", "marked_xy_z"):
        c["wfunc"] = rng.choice([1, 2, 5, 9])
    if kind == "jackknife":
        c["side"] = rng.randint(2, 5)
    if kind == "batch":
        del c["clustered"], c["n1"], c["n2"]
        c["L"], c["rmax"] = 1000.0, round(rng.uniform(20.0, 50.0), 3)
        c["mocks"] = rng.randint(2, 24)
        c["nmin"] = _logint(rng, 2e4, 1e5)
        c["nmax"] = _logint(rng, 2e5, 1e6)
    return c


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + 12345)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, dtype=torch.float64, device="cuda")


def _g_nfw(y):
    return torch.log1p(y) - y / (1.0 + y)


def _points(n, L, clustered, g):
    """Uniform points, or a fifth of them uniform centres with the rest as NFW satellites (c = 5, r <= 0.5 Mpc/h)."""
    if not clustered:
        return _rand(g, n, 3) * L
    nc = max(1, n // 5)
    ns = n - nc
    centres = _rand(g, nc, 3) * L
    host = torch.randint(0, nc, (ns,), generator=g, device="cuda")
    target = _rand(g, ns) * (math.log1p(5.0) - 5.0 / 6.0)
    lo = torch.zeros(ns, dtype=torch.float64, device="cuda")
    hi = torch.ones_like(lo)
    for _ in range(40):
        mid = 0.5 * (lo + hi)
        below = _g_nfw(5.0 * mid) < target
        lo = torch.where(below, mid, lo)
        hi = torch.where(below, hi, mid)
    r = 0.25 * (lo + hi)
    v = torch.randn(ns, 3, generator=g, dtype=torch.float64, device="cuda")
    v /= v.norm(dim=1, keepdim=True)
    pts = torch.cat([centres, centres[host] + r[:, None] * v])
    return torch.remainder(pts, L).contiguous()


def _rbins(case):
    return np.logspace(math.log10(case["rmin"]), math.log10(case["rmax"]), case["nbins"])


def _pibins(case):
    return np.linspace(0.0, case["pimax"], case["npi"])


def _mock_sizes(case):
    M = case["mocks"]
    q = (np.arange(M) + 0.5) / M
    n = np.round(case["nmin"] * (case["nmax"] / case["nmin"]) ** q).astype(int) | 1
    return [int(v) for v in n[np.random.default_rng(M).permutation(M)]]  # uneven sizes in no order


def prepare(case, seed):
    g = _gen(seed)
    kind, L = case["kind"], case["L"]
    s = dict(case=case, rbins=_rbins(case))
    if kind == "batch":
        sizes = _mock_sizes(case)
        n = sum(sizes)
        b = batch.MockBatch(_rand(g, n, 3) * L, L, s["rbins"], sizes=sizes)
        logm = 11.0 + 4.0 * _rand(g, n)
        logMmin = 11.5 + _rand(g, len(sizes))
        c = torch.randn(case["nbins"], generator=g, dtype=torch.float64, device="cuda")
        s.update(logm=logm, logMmin=logMmin, c=c, sizes=sizes, points=b.rows)
        # a fitting loop builds the step once and replays its graph with new parameters
        s["step"] = batch.HODBatchStep(b, logm, logMmin, 0.3, c).capture()
        return s
    s["p1"] = _points(case["n1"], L, case["clustered"], g)
    s["p2"] = s["p1"]
    if case["n2"]:
        # the second sample: randoms of a survey, or another tracer of the box
        s["p2"] = _points(case["n2"], L, False, g)
    if "npi" in case:
        s["pibins"] = _pibins(case)
    if kind == "marked_grad":
        s["logm"] = 11.0 + 4.0 * _rand(g, case["n1"])
        s["c"] = torch.randn(case["nbins"], generator=g, dtype=torch.float64, device="cuda")
        s["theta"] = torch.tensor([12.0, 0.3], dtype=torch.float64, device="cuda", requires_grad=True)
    if kind in ("marked_3d", "marked_xy_z"):
        nw = 1 if case["wfunc"] in (1, 2) else 2
        s["w"] = _rand(g, case["n1"], nw)
    if kind == "jackknife":
        k = case["side"]
        sub = torch.clamp((s["p1"] / L * k).long(), max=k - 1)
        s["tags"] = (1 + (sub[:, 0] * k + sub[:, 1]) * k + sub[:, 2]).to(torch.int32)
    return s


def run(s):
    case = s["case"]
    kind, L = case["kind"], case["L"]
    if kind == "batch":
        counts, W, loss, grad = s["step"].replay()
        return dict(counts=counts, W=W, loss=loss, grad=grad)
    p1, p2, rb = s["p1"], s["p2"], s["rbins"]
    if kind == "npairs_3d":
        return npairs_3d(p1, p2, rb, period=L)
    if kind == "tpcf":
        return tpcf(p1, rb, randoms=p2, estimator="Landy-Szalay")
    if kind == "npairs_xy_z":
        return npairs_xy_z(p1, p2, rb, s["pibins"], period=L)
    if kind == "wp":
        return wp(p1, rb, case["pimax"], period=L)
    if kind == "npairs_projected":
        return npairs_projected(p1, p2, rb, case["pimax"], period=L)
    if kind == "marked_grad":
        theta = s["theta"]
        theta.grad = None
        w = mocks.zheng07_ncen(s["logm"], theta[0], theta[1])
        W = marked_npairs_3d_product(p1, p1, rb, w, w, period=L)
        (W * s["c"]).sum().backward()
        return dict(W=W.detach(), grad=theta.grad)
    if kind == "marked_3d":
        return marked_npairs_3d(p1, p1, rb, case["wfunc"], period=L, weights1=s["w"], weights2=s["w"])
    if kind == "marked_xy_z":
        return marked_npairs_xy_z(p1, p1, rb, s["pibins"], weight_func_id=case["wfunc"], period=L, weights1=s["w"],
                                  weights2=s["w"])
    if kind == "per_object":
        return npairs_per_object_3d(p1, p1, rb, period=L)
    if kind == "jackknife":
        return npairs_jackknife_3d(p1, p1, rb, s["tags"], s["tags"], case["side"] ** 3, period=L)
    raise ValueError(kind)


# ------------------------------------------------------------------ necessary work
def _volume(case):
    if "pimax" in case:
        return math.pi * case["rmax"] ** 2 * 2.0 * case["pimax"]
    return 4.0 / 3.0 * math.pi * case["rmax"] ** 3


def work(case):
    """Each input and output once; 8 flops (3 sub, 3 mul, 2 add) for every pair inside the search
    length, an auto-count's pairs once for both orders (uniform density; clumps add little)."""
    kind, f = case["kind"], _volume(case) / case["L"] ** 3
    K = case["nbins"] * case.get("npi", 1)
    if kind == "batch":
        n = _mock_sizes(case)
        # distances, and the two product terms with their sums per pair
        pairs = 0.5 * f * sum(float(v) * v for v in n)
        return dict(bytes=float(sum(n)) * 40.0 + 8.0 * len(n) * (3 * K + 3), flops=pairs * 14.0)
    n1, n2 = float(case["n1"]), float(case["n2"])
    if kind == "tpcf":
        return dict(bytes=24.0 * (n1 + n2) + 8.0 * K, flops=8.0 * f * (0.5 * n1 * n1 + n1 * n2 + 0.5 * n2 * n2))
    pairs = f * (n1 * n2 if n2 else 0.5 * n1 * n1)
    b, per_pair = 24.0 * (n1 + n2) + 8.0 * K, 8.0
    if kind == "marked_grad":
        b, per_pair = b + 16.0 * n1, 12.0
    elif kind in ("marked_3d", "marked_xy_z"):
        b, per_pair = b + 8.0 * n1 * (1 if case["wfunc"] in (1, 2) else 2), 10.0
    elif kind == "per_object":
        b += 8.0 * n1 * K
    elif kind == "jackknife":
        b, per_pair = b + 4.0 * n1 + 8.0 * K * (case["side"] ** 3 + 1), 9.0
    return dict(bytes=b, flops=per_pair * pairs)


# ------------------------------------------------------------------ 64-bit results
def _grid(p, n, cell, rim):
    """Point indices by cell of an n[0] x n[1] x n[2] grid, padded with -1 (rim: an empty layer of cells around)."""
    dev = p.device
    i = torch.stack([torch.clamp((p[:, d] / cell[d]).floor().long(), 0, n[d] - 1) + rim for d in range(3)])
    m = [v + 2 * rim for v in n]
    key = (i[0] * m[1] + i[1]) * m[2] + i[2]
    order = torch.argsort(key, stable=True)
    cnt = torch.bincount(key, minlength=m[0] * m[1] * m[2])
    first = torch.cumsum(cnt, 0) - cnt
    grid = torch.full((len(cnt), int(cnt.max())), -1, dtype=torch.long, device=dev)
    sk = key[order]
    grid[sk, torch.arange(len(order), device=dev) - first[sk]] = order
    return grid, m


def _pairs(p1, p2, L, reach, most=20_000_000):
    """Ordered pairs (i, j, dx, dy, dz) that can lie within `reach` (x, y, z lengths); L: periodic box side, or None."""
    if L is None:
        low = torch.minimum(p1.min(0).values, p2.min(0).values)
        p1, p2 = p1 - low, p2 - low
        side = [max(float(torch.maximum(p1.max(0).values, p2.max(0).values)[d]), reach[d]) * 1.000001 for d in range(3)]
    else:
        side = [L, L, L]
    n = [max(3 if L is not None else 1, int(side[d] / reach[d])) for d in range(3)]
    n = [min(v, 64) for v in n]
    rim = 0 if L is not None else 1
    cell = [side[d] / n[d] for d in range(3)]
    g1, m = _grid(p1, n, cell, rim)
    g2, _ = _grid(p2, n, cell, rim)
    full = torch.nonzero(g1[:, 0] >= 0)[:, 0]
    chunk = max(1, most // (g1.shape[1] * g2.shape[1]))
    for a in range(0, len(full), chunk):
        c1 = full[a:a + chunk]
        ix, iy, iz = c1 // (m[1] * m[2]), (c1 // m[2]) % m[1], c1 % m[2]
        i = g1[c1]
        q1 = p1[i.clamp(min=0)]
        for o in range(27):
            o3 = (o // 9 - 1, (o // 3) % 3 - 1, o % 3 - 1)
            c2 = (((ix + o3[0]) % m[0]) * m[1] + (iy + o3[1]) % m[1]) * m[2] + (iz + o3[2]) % m[2]
            j = g2[c2]
            d = []
            q2 = p2[j.clamp(min=0)]
            for k in range(3):
                x = (q1[:, :, None, k] - q2[:, None, :, k]).abs()
                d.append(torch.minimum(x, L - x) if L is not None else x)
            ok = (i >= 0)[:, :, None] & (j >= 0)[:, None, :]
            for k in range(3):
                ok &= d[k] <= reach[k]
            at = ok.nonzero(as_tuple=True)
            yield i[at[0], at[1]], j[at[0], at[2]], d[0][at], d[1][at], d[2][at]


_SPREAD = 512


def _hist(idx, w, nb, acc):
    """acc += sums of w (or counts) by idx, spread over columns so that the adds rarely meet."""
    col = torch.arange(len(idx), device=idx.device) % _SPREAD
    acc.index_add_(0, idx * _SPREAD + col, w if w is not None else torch.ones(len(idx), dtype=torch.float64,
                                                                             device=idx.device))


def _bins(r2, edges2):
    return torch.bucketize(r2, edges2)  # edges[k-1] < r2 <= edges[k]


def _acc(nb):
    return torch.zeros((nb + 1) * _SPREAD, dtype=torch.float64, device="cuda")


def _mark(wfunc, a, b):
    if wfunc == 1:
        return a[:, 0] * b[:, 0]
    if wfunc == 2:
        return a[:, 0] + b[:, 0]
    if wfunc == 5:
        return torch.where(b[:, 0] > a[:, 0], a[:, 1] * b[:, 1], torch.zeros_like(a[:, 0]))
    if wfunc == 9:
        return torch.where((a[:, 0] - b[:, 0]).abs() < a[:, 1], b[:, 1], torch.zeros_like(a[:, 0]))
    raise ValueError(wfunc)


def _counts_1d(p1, p2, L, rb, pimax=None):
    reach = (rb[-1],) * 3 if pimax is None else (rb[-1], rb[-1], pimax)
    e = torch.tensor(rb * rb, device="cuda")
    acc = _acc(len(rb))
    for i, j, dx, dy, dz in _pairs(p1, p2, L, reach):
        _hist(_bins(dx * dx + dy * dy + (dz * dz if pimax is None else 0.0), e), None, len(rb), acc)
    return acc.view(-1, _SPREAD).sum(1)[:-1].cumsum(0)


def exact(case, seed):
    kind, L = case["kind"], case["L"]
    if kind in ("npairs_3d", "npairs_xy_z", "npairs_projected", "per_object"):
        return None  # whole numbers
    if kind == "batch":
        if 13.0 * work(case)["flops"] / 14.0 > 6e10:
            return None  # minutes
        return _exact_batch(case, seed)
    s = prepare(case, seed)
    p1, p2, rb = s["p1"], s["p2"], s["rbins"]
    K = len(rb)
    e = torch.tensor(rb * rb, device="cuda")
    if kind == "tpcf":
        n, nr = float(len(p1)), float(len(p2))
        dd, dr, rr = [_counts_1d(a, b, None, rb).diff() for a, b in ((p1, p1), (p1, p2), (p2, p2))]
        return (dd / rr) * (nr * nr / (n * n)) - (2.0 * dr / rr) * (nr / n) + 1.0
    if kind == "wp":
        dd = _counts_1d(p1, p1, L, rb, case["pimax"])
        # the reference's innermost pi edge is 0: pairs at dz = 0 exactly (each point with itself) are outside the bin
        dd = dd - len(p1)
        n = float(len(p1))
        vol = math.pi * np.diff(rb ** 2) * 2.0 * case["pimax"]
        rr = torch.tensor(vol * n * n / L ** 3, device="cuda")
        return (dd.diff() / rr - 1.0) * 2.0 * case["pimax"]
    if kind == "marked_grad":
        c = s["c"]
        u = (s["logm"] - 12.0) / 0.3
        w = 0.5 * (1.0 + torch.erf(u))
        acc = _acc(K)
        v = torch.zeros(len(p1), dtype=torch.float64, device="cuda")
        tail = torch.cat([c.flip(0).cumsum(0).flip(0), c.new_zeros(1)])
        for i, j, dx, dy, dz in _pairs(p1, p1, L, (rb[-1],) * 3):
            k = _bins(dx * dx + dy * dy + dz * dz, e)
            _hist(k, w[i] * w[j], K, acc)
            v.index_add_(0, i, w[j] * tail[k])
        W = acc.view(-1, _SPREAD).sum(1)[:-1].cumsum(0)
        dw = torch.exp(-u * u) / math.sqrt(math.pi)
        grad = torch.stack([(2.0 * v * dw * (-1.0 / 0.3)).sum(), (2.0 * v * dw * (-u / 0.3)).sum()])
        return dict(W=W, grad=grad)
    if kind == "marked_3d":
        acc = _acc(K)
        for i, j, dx, dy, dz in _pairs(p1, p1, L, (rb[-1],) * 3):
            _hist(_bins(dx * dx + dy * dy + dz * dz, e), _mark(case["wfunc"], s["w"][i], s["w"][j]), K, acc)
        return acc.view(-1, _SPREAD).sum(1)[:-1].cumsum(0)
    if kind == "marked_xy_z":
        pb = s["pibins"]
        q = torch.tensor(pb * pb, device="cuda")
        P = len(pb)
        acc = _acc((K + 1) * (P + 1) - 1)
        for i, j, dx, dy, dz in _pairs(p1, p1, L, (rb[-1], rb[-1], pb[-1])):
            k = _bins(dx * dx + dy * dy, e) * (P + 1) + _bins(dz * dz, q)
            _hist(k, _mark(case["wfunc"], s["w"][i], s["w"][j]), 0, acc)
        t = acc.view(-1, _SPREAD).sum(1).view(K + 1, P + 1)[:K, :P]
        return t.cumsum(0).cumsum(1)
    if kind == "jackknife":
        S = case["side"] ** 3
        acc = _acc((S + 1) * (K + 1) - 1)
        t = s["tags"].long()
        for i, j, dx, dy, dz in _pairs(p1, p1, L, (rb[-1],) * 3):
            # each ordered pair takes half of its weight from the subsample of either point
            _hist(t[i] * (K + 1) + _bins(dx * dx + dy * dy + dz * dz, e), None, 0, acc)
        h = acc.view(-1, _SPREAD).sum(1).view(S + 1, K + 1)[:, :K].cumsum(1)
        total = h.sum(0, keepdim=True)
        return torch.cat([total, total - h[1:]])
    return None


def _exact_batch(case, seed):
    s = prepare(case, seed)
    L, rb, c = case["L"], s["rbins"], s["c"]
    K = len(rb)
    e = torch.tensor(rb * rb, device="cuda")
    W, grad, at = [], [], 0
    for m, n in enumerate(s["sizes"]):
        p = s["points"][at:at + n]
        u = (s["logm"][at:at + n] - s["logMmin"][m]) / 0.3
        at += n
        w, t = 0.5 * (1.0 + torch.erf(u)), -torch.exp(-u * u) / (math.sqrt(math.pi) * 0.3)
        a, d = _acc(K), _acc(K)
        for i, j, dx, dy, dz in _pairs(p, p, L, (rb[-1],) * 3):
            k = _bins(dx * dx + dy * dy + dz * dz, e)
            _hist(k, w[i] * w[j], K, a)
            _hist(k, t[i] * w[j] + w[i] * t[j], K, d)
        a, d = [x.view(-1, _SPREAD).sum(1)[:-1].cumsum(0) for x in (a, d)]
        W.append(a)
        grad.append((d * c).sum())
    W = torch.stack(W)
    return dict(counts=None, W=W, loss=(W * c).sum(1), grad=torch.stack(grad))

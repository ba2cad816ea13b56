"""Matrix-core pair kernels at the sizes where they can go wrong: sub-groups of
16, groups of 64, dealt parts of 128, split groups, pairs at and next to bin
edges, coincident points, periodic images; against the oracle (counts bit-exact,
sums to 1e-12, the bound of the other kernels: FP64 sums of up to ~1e6 positive
terms in another order) and against the general kernels."""
import numpy as np
import pytest

from oracle import mesh as ORC
from tests.test_gpu_autodiff import _seam_pair

pytestmark = pytest.mark.gpu

L = 100.0
RB = np.logspace(-1, np.log10(20.0), 12)
PI = np.array([0.0, 2.0, 7.5, 20.0])


@pytest.fixture(scope="module")
def mo(gpu):
    import halotools_amd.mock_observables as mo
    return mo


def _points(n, kind, seed):
    rng = np.random.default_rng([7, n, seed])
    p = rng.uniform(0, L, (n, 3))
    if kind == "clumps":   # pairs far below the first edge, and exact duplicates
        p = np.mod(p[rng.integers(0, max(1, n // 6), n)] + rng.normal(size=(n, 3)) * 0.01, L)
        p[n // 2:n // 2 + n // 10] = p[:n // 10]
    elif kind == "lattice":  # separations exactly on and next to edges
        p = rng.integers(0, 40, (n, 3)) * 2.5
    elif kind == "seam":   # everything next to the box faces and corners
        p = np.mod(rng.normal(size=(n, 3)) * 3.0, L)
    elif kind == "slab":   # wide, flat groups
        p[:, 2] = rng.uniform(0, 0.01, n)
    return p


CASES = [(n, 0, k) for n in (1, 2, 15, 16, 17, 63, 64, 65, 128, 129, 200, 1000) for k in ("uniform", "clumps")] + \
        [(3000, 0, k) for k in ("uniform", "clumps", "lattice", "seam", "slab")] + \
        [(1, 64, "uniform"), (17, 1, "seam"), (65, 2000, "uniform"), (2000, 65, "clumps"), (1500, 1500, "lattice"),
         (20000, 9000, "uniform")]


@pytest.mark.parametrize("period", [L, None], ids=["box", "open"])
@pytest.mark.parametrize("n1,n2,kind", CASES)
def test_counts(mo, n1, n2, kind, period):
    p1 = _points(n1, kind, 0)
    p2 = p1 if n2 == 0 else _points(n2, kind, 1)
    rb = np.array([2.5, 5.0, 7.5, 10.0, 12.5]) if kind == "lattice" else RB
    kw = dict(period=period)
    got = mo.npairs_3d(p1, p2, rb, **kw)
    assert np.array_equal(got, ORC.npairs_3d(p1, p2, rb, **kw))
    assert np.array_equal(mo.npairs_xy_z(p1, p2, rb, PI, **kw), ORC.npairs_xy_z(p1, p2, rb, PI, **kw))
    assert np.array_equal(mo.npairs_projected(p1, p2, rb, 7.5, **kw), ORC.npairs_projected(p1, p2, rb, 7.5, **kw))
    assert np.array_equal(mo.npairs_per_object_3d(p1, p2, rb, **kw), ORC.npairs_per_object_3d(p1, p2, rb, **kw))


@pytest.mark.parametrize("wfunc,nw", [(1, 1), (2, 1), (5, 2), (9, 2), (12, 4), (17, 5)])
@pytest.mark.parametrize("n1,n2,kind", [(65, 0, "clumps"), (129, 40, "uniform"), (1000, 0, "seam"),
                                        (1500, 700, "lattice")])
def test_sums(mo, n1, n2, kind, wfunc, nw):
    p1 = _points(n1, kind, 0)
    p2 = p1 if n2 == 0 else _points(n2, kind, 1)
    rb = np.array([2.5, 5.0, 7.5, 10.0, 12.5]) if kind == "lattice" else RB
    rng = np.random.default_rng(3)
    w1 = rng.uniform(0.1, 1, (len(p1), nw))
    w2 = w1 if n2 == 0 else rng.uniform(0.1, 1, (len(p2), nw))
    if nw == 5:
        w1[:, 4] = np.round(w1[:, 4] * 3)
        w2[:, 4] = np.round(w2[:, 4] * 3)
    kw = dict(period=L, weights1=w1, weights2=w2, weight_func_id=wfunc)
    np.testing.assert_allclose(mo.marked_npairs_3d(p1, p2, rb, **kw), ORC.marked_npairs_3d(p1, p2, rb, **kw),
                               rtol=1e-12, atol=1e-300)
    if wfunc < 16:
        np.testing.assert_allclose(mo.marked_npairs_xy_z(p1, p2, rb, PI, **kw),
                                   ORC.marked_npairs_xy_z(p1, p2, rb, PI, **kw), rtol=1e-12, atol=1e-300)


@pytest.mark.parametrize("layout", ["rows", "columns", "f32", "sliced"])
def test_layouts_and_general_kernels_agree(mo, gpu, layout, monkeypatch):
    import torch
    p = torch.as_tensor(_points(5000, "clumps", 2), device=gpu)
    if layout == "columns":
        p = p.t().contiguous().t()
    elif layout == "f32":
        p = p.to(torch.float32).clamp(0, float(np.nextafter(np.float32(L), np.float32(0))))
    elif layout == "sliced":
        p = torch.cat([p, p], dim=1)[::2, 1:4]
    got = [mo.npairs_3d(p, p, RB, period=L), mo.npairs_xy_z(p, p, RB, PI, period=L),
           mo.npairs_per_object_3d(p, p, RB, period=L), mo.npairs_projected(p, p, RB, 3.0, period=L)]
    monkeypatch.setenv("HALOPAIR_NO_TILES", "1")
    ref = [mo.npairs_3d(p, p, RB, period=L), mo.npairs_xy_z(p, p, RB, PI, period=L),
           mo.npairs_per_object_3d(p, p, RB, period=L), mo.npairs_projected(p, p, RB, 3.0, period=L)]
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


@pytest.mark.parametrize("same", [True, False])
def test_jacobian_rows_and_seam_corrections(gpu, same, monkeypatch):
    # weights that are small integers: both kernels' row sums are exact, so the rows agree bit for bit
    import torch

    from halotools_amd import _device as D
    from halotools_amd import _engine as E
    rng = np.random.default_rng(5)
    p1 = _points(1200, "lattice", 0) + 0.1 * rng.integers(0, 2, (1200, 3))
    p2 = _points(700, "lattice", 1)
    t1, t2 = [torch.as_tensor(np.mod(p, L), device=gpu) for p in (p1, p2)]
    w1 = torch.as_tensor(rng.integers(1, 9, (1200, 1)).astype(float), device=gpu)
    w2 = torch.as_tensor(rng.integers(1, 9, (700, 1)).astype(float), device=gpu)
    r2 = np.array([2.4, 2.5, 5.0, 7.5, 12.4]) ** 2
    mock = dict(n1=1200, n2=700, period=[L] * 3, pbc=True)

    def run():
        res = D.run(E.HP_MARKED_NPAIRS_3D, [mock], t1.unbind(1), (t1 if same else t2).unbind(1), r2, same=same, w1=w1,
                    w2=None if same else w2, nw=1, wfunc=1, want_counts=False, want_sums=True, rows1=True, rows2=True,
                    also_counts=True, device=gpu)
        return res.rows1, res.rows2, res.sums, res.counts
    got = run()
    monkeypatch.setenv("HALOPAIR_NO_TILES", "1")
    for a, b in zip(got, run()):
        assert torch.equal(a, b)


@pytest.mark.parametrize("tags", ["one", "slabs", "random"])
@pytest.mark.parametrize("n", [1, 64, 65, 700])
def test_jackknife_tables(mo, n, tags):
    rng = np.random.default_rng(n)
    p = rng.uniform(0, 1, (n, 3))
    r = 0.1
    if n > 20:
        x, y, r = _seam_pair()  # its two orders fall into different bins
        p[3], p[17] = [x, 0.5, 0.5], [y, 0.5, 0.5]
    ns = {"one": 1, "slabs": 4, "random": 40}[tags]
    t = {"one": np.ones(n, int), "slabs": 1 + np.minimum((p[:, 0] * 4).astype(int), 3),
         "random": rng.integers(1, ns + 1, n)}[tags]
    rb = np.array([0.5 * r, r, 0.2])
    got = mo.npairs_jackknife_3d(p, p, rb, t, t, ns, period=1.0)
    assert np.array_equal(got, ORC.npairs_jackknife(p, p, rb, t, t, ns, period=1.0))
    w = rng.uniform(0.1, 1, n)
    got = mo.npairs_jackknife_3d(p, p, rb, t, t, ns, period=1.0, weights1=w, weights2=w)
    ref = ORC.npairs_jackknife(p, p, rb, t, t, ns, period=1.0, weights1=w, weights2=w)
    np.testing.assert_allclose(got, ref, rtol=0, atol=1e-12 * ref.max())


@pytest.mark.parametrize("n1,n2", [(1023, 1025), (1024, 1), (1, 65536), (65535, 1024), (65536, 65536), (65537, 3000),
                                   (131072, 131073), (196609, 65536), (262144, 5000), (262145, 262144),
                                   (300000, 1), (63, 300001), (2000, 131072), (196608, 300000), (300000, 1500)])
def test_small_builds_agree_with_general(mo, gpu, n1, n2, monkeypatch):
    # edges of the sort tiles and of the range that the small build takes; two samples of
    # unlike sizes, half of the first in one spot (one digit holds whole tiles)
    import torch
    p1, p2 = _points(n1, "uniform", 3), _points(n2, "seam", 4)
    p1[: n1 // 2] = p1[0]
    w1, w2 = np.arange(1.0, n1 + 1) % 7 + 1, np.arange(1.0, n2 + 1) % 5 + 1
    t1, t2, u1, u2 = [torch.as_tensor(a, device=gpu) for a in (p1, p2, w1, w2)]
    rb = RB[:6]   # (sums of small whole numbers: exact in any order)

    def run():
        return (mo.npairs_3d(t1, t2, rb, period=L), mo.npairs_per_object_3d(t1, t2, rb, period=L),
                mo.marked_npairs_3d(t1, t2, rb, period=L, weights1=u1, weights2=u2, weight_func_id=1),
                mo.npairs_projected(t1, t1, rb, 2.0, period=L) if n1 < 2000 else mo.npairs_3d(t2, t2, rb, period=L))
    got = run()
    monkeypatch.setenv("HALOPAIR_NO_TILES", "1")
    for a, b in zip(got, run()):
        assert torch.equal(torch.as_tensor(a), torch.as_tensor(b))


@pytest.mark.parametrize("n1,n2", [(800001, 0), (650000, 70001)])
def test_queued_items_agree_with_general(mo, gpu, n1, n2, monkeypatch):
    # more lane groups than two per resident wave: waves take them from queues
    import torch
    g = torch.Generator(device=gpu).manual_seed(n1)
    t1 = torch.rand((n1, 3), dtype=torch.float64, device=gpu, generator=g) * 400.0
    t1[: n1 // 8] = 200.0 + 0.01 * (t1[: n1 // 8] - 200.0)   # items of very unlike cost
    t2 = t1 if n2 == 0 else torch.rand((n2, 3), dtype=torch.float64, device=gpu, generator=g) * 400.0
    u1 = torch.randint(1, 9, (n1,), device=gpu, generator=g).double()
    u2 = u1 if n2 == 0 else torch.randint(1, 9, (n2,), device=gpu, generator=g).double()
    rb, pi, kw = np.array([0.02, 0.1, 1.0, 4.0]), np.array([0.0, 0.5, 3.0]), dict(period=400.0)

    def run():
        return (mo.npairs_3d(t1, t2, rb, **kw), mo.npairs_xy_z(t1, t2, rb, pi, **kw),
                mo.npairs_per_object_3d(t1, t2, rb, **kw), mo.npairs_projected(t1, t2, rb, 3.0, **kw),
                mo.marked_npairs_3d(t1, t2, rb, weights1=u1, weights2=u2, weight_func_id=1, **kw))
    got = run()
    monkeypatch.setenv("HALOPAIR_NO_TILES", "1")
    for a, b in zip(got, run()):
        assert torch.equal(torch.as_tensor(a), torch.as_tensor(b))


@pytest.mark.parametrize("tiles", [True, False])
@pytest.mark.parametrize("seam", [True, False])
def test_seam_check(gpu, seam, tiles, monkeypatch):
    # the status bit tells whether rows2 would differ, and the gradient has it either way
    import torch

    from halotools_amd import _device as D
    from halotools_amd import _engine as E
    from halotools_amd.autodiff import marked_npairs_3d_product
    if not tiles:
        monkeypatch.setenv("HALOPAIR_NO_TILES", "1")
    xi, xj, r = _seam_pair()
    pts = np.random.default_rng(3).uniform(0, 1, (700, 3))
    if seam:
        pts[10], pts[20] = [xi, 0.5, 0.5], [xj, 0.5, 0.5]
    rb = np.array([0.5 * r, r, 0.2])
    t = torch.as_tensor(pts, device=gpu)
    w = torch.randint(1, 9, (700,), device=gpu).double().requires_grad_(True)
    args = dict(same=True, w1=w.detach().reshape(-1, 1), nw=1, wfunc=1, want_counts=False, want_sums=True, device=gpu)
    mock = [dict(n1=700, n2=700, period=[1.0] * 3, pbc=True)]
    chk = D.run(E.HP_MARKED_NPAIRS_3D, mock, t.unbind(1), t.unbind(1), rb * rb, rows1=True, seam_check=True, **args)
    full = D.run(E.HP_MARKED_NPAIRS_3D, mock, t.unbind(1), t.unbind(1), rb * rb, rows1=True, rows2=True, **args)
    assert (int(chk.status.item()) & 0xFFFFFFFF) == (4 if seam else 0)
    assert torch.equal(chk.rows1, full.rows1) and torch.equal(full.rows1, full.rows2) == (not seam)
    c = torch.tensor([1.0, 2.0, 4.0], dtype=torch.float64, device=gpu)
    (marked_npairs_3d_product(t, t, rb, w, w, period=1.0) * c).sum().backward()
    G = torch.tensor([7.0, 6.0, 4.0], dtype=torch.float64, device=gpu)
    assert torch.equal(w.grad, ((full.rows1 + full.rows2) * G).sum(dim=1))
    with pytest.raises(E.EngineError):
        D.run(E.HP_MARKED_NPAIRS_3D, mock, t.unbind(1), t.unbind(1), rb * rb, rows1=True, rows2=True, seam_check=True, **args)


@pytest.mark.parametrize("tags", ["slabs", "random"])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 0.0])
def test_jackknife_weights_that_are_not_finite(mo, value, tags, monkeypatch):
    # a pair's weight is the product of its two: bins without a pair of the infinite point stay finite
    # (sums of small whole numbers: the finite ones are exact)
    rng = np.random.default_rng(31)
    n, ns = 500, 4
    p = rng.uniform(0, 1, (n, 3))
    t = 1 + np.minimum((p[:, 0] * ns).astype(int), ns - 1) if tags == "slabs" else rng.integers(1, ns + 1, n)
    w = rng.integers(1, 5, n).astype(float)
    w[40] = value
    w[7] = 0.0
    rb = np.array([0.01, 0.02, 0.05, 0.1, 0.2])
    kw = dict(period=1.0, weights1=w, weights2=w)
    got = mo.npairs_jackknife_3d(p, p, rb, t, t, ns, **kw)
    monkeypatch.setenv("HALOPAIR_NO_TILES", "1")
    ref = mo.npairs_jackknife_3d(p, p, rb, t, t, ns, **kw)
    assert np.array_equal(got, ref, equal_nan=True)


def _seconds(f, reps=9):
    import time

    import torch
    times = []
    for _ in range(reps + 2):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        f()
        torch.cuda.synchronize()
        times.append(time.perf_counter() - t0)
    return float(np.median(times[2:]))


@pytest.mark.parametrize("ns", [1, 8, 511, 512, 513, 1024, 1025, 5000])
def test_many_subsamples(mo, ns, monkeypatch):
    # the table's total over parts of the subsamples (whole numbers: exact in any order)
    rng = np.random.default_rng(ns)
    p = rng.uniform(0, 1, (700, 3))
    t = rng.integers(1, ns + 1, 700)
    w = rng.integers(1, 5, 700).astype(float)
    rb = np.linspace(0.01, 0.2, 33)
    run = lambda: [mo.npairs_jackknife_3d(p, p, rb, t, t, ns, period=1.0, **kw)
                   for kw in ({}, dict(weights1=w, weights2=w))]
    got = run()
    monkeypatch.setenv("HALOPAIR_NO_TILES", "1")
    for a, b in zip(got, run()):
        assert np.array_equal(a, b)


def test_many_subsamples_cost_no_more_than_in_the_general_kernels(mo, gpu, monkeypatch):
    # 300 points, 65536 subsamples: the tables' total and output are the work (2.7 times the
    # general kernels' call with the total in one workgroup, 0.4 times in parts)
    import torch
    p = torch.rand((300, 3), dtype=torch.float64, device=gpu)
    t = torch.randint(1, 65537, (300,), device=gpu)
    rb = np.logspace(-2, -1, 15)
    run = lambda: mo.npairs_jackknife_3d(p, p, rb, t, t, 65536, period=1.0)
    tiles = _seconds(run)
    monkeypatch.setenv("HALOPAIR_NO_TILES", "1")
    assert tiles < 1.4 * _seconds(run)


@pytest.mark.parametrize("n1,n2", [(1, 0), (15, 0), (16, 0), (17, 0), (63, 0), (64, 0), (65, 0), (129, 0), (1000, 0),
                                   (1, 64), (17, 1), (65, 200), (200, 65), (64, 1000)])
@pytest.mark.parametrize("kind", ["uniform", "clumps", "lattice", "seam"])
def test_forward_mode_agrees_with_general(gpu, n1, n2, kind, monkeypatch):
    # weights and tangents that are small whole numbers: every term and its halves are exact
    import torch

    from halotools_amd import _device as D
    from halotools_amd import _engine as E
    same = n2 == 0
    rng = np.random.default_rng([n1, n2])
    p = [torch.as_tensor(_points(n, kind, i), device=gpu) for i, n in enumerate((n1, n2 or n1))]
    w = [torch.as_tensor(rng.integers(-8, 9, (len(x), 2)).astype(float), device=gpu) for x in p]
    rb = np.array([2.5, 5.0, 7.5, 10.0, 12.5]) if kind == "lattice" else RB

    def run():
        res = D.run(E.HP_MARKED_NPAIRS_3D, [dict(n1=n1, n2=n2 or n1, period=[L] * 3, pbc=True)], p[0].unbind(1),
                    p[0 if same else 1].unbind(1), rb * rb, same=same, w1=w[0], w2=None if same else w[1], nw=2,
                    wfunc=1, want_counts=False, want_sums=True, also_counts=True, tangent=True, device=gpu)
        return res.counts, res.sums, res.tangents
    got = run()
    monkeypatch.setenv("HALOPAIR_NO_TILES", "1")
    for a, b in zip(got, run()):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n1,n2", [(800001, 0), (650000, 600001)])
def test_queued_items_of_every_mode_agree_with_general(mo, gpu, n1, n2, monkeypatch):
    # the passes that test_queued_items_agree_with_general leaves out: one-column (rp, pi) cells, generic
    # marks, Jacobian rows and their swapped pass (a queue set of its own), jackknife rows
    import torch

    from halotools_amd import _device as D
    from halotools_amd import _engine as E
    g = torch.Generator(device=gpu).manual_seed(n1)
    box = 400.0
    t1 = torch.rand((n1, 3), dtype=torch.float64, device=gpu, generator=g) * box
    t1[: n1 // 8] = 200.0 + 0.01 * (t1[: n1 // 8] - 200.0)   # items of very unlike cost
    t2 = t1 if n2 == 0 else torch.rand((n2, 3), dtype=torch.float64, device=gpu, generator=g) * box
    u1 = torch.randint(1, 9, (n1, 2), device=gpu, generator=g).double()
    u2 = u1 if n2 == 0 else torch.randint(1, 9, (n2, 2), device=gpu, generator=g).double()
    s1, s2 = u1[:, 0].contiguous(), u2[:, 0].contiguous()
    rb, kw = np.array([0.02, 0.1, 1.0, 4.0]), dict(period=box)
    wide, pi = np.linspace(0.05, 3.0, 17), np.linspace(0.0, 3.0, 17)
    marks = lambda a, b, i: dict(weights1=a, weights2=b, weight_func_id=i, **kw)
    tags = 1 + torch.clamp((t1[:, 0] / box * 5).long(), max=4)

    def run():
        out = [mo.npairs_xy_z(t1, t2, wide, pi, **kw), mo.marked_npairs_xy_z(t1, t2, wide, pi, **marks(s1, s2, 1)),
               mo.marked_npairs_xy_z(t1, t2, rb, pi[:3], **marks(u1, u2, 5)),
               mo.marked_npairs_3d(t1, t2, rb, **marks(u1, u2, 9)), mo.marked_npairs_3d(t1, t2, rb, **marks(s1, s2, 2))]
        res = D.run(E.HP_MARKED_NPAIRS_3D, [dict(n1=n1, n2=n2 or n1, period=[box] * 3, pbc=True)], t1.unbind(1),
                    t2.unbind(1), rb * rb, same=n2 == 0, w1=s1.reshape(-1, 1),
                    w2=None if n2 == 0 else s2.reshape(-1, 1), nw=1, wfunc=1, want_counts=False, want_sums=True,
                    rows1=True, rows2=True, also_counts=True, device=gpu)
        out += [res.sums, res.counts, res.rows1, res.rows2]
        if n2 == 0:
            out += [mo.npairs_jackknife_3d(t1, t1, rb, tags, tags, 5, **kw),
                    mo.npairs_jackknife_3d(t1, t1, rb, tags, tags, 5, weights1=s1, weights2=s1, **kw)]
        return out
    got = run()
    monkeypatch.setenv("HALOPAIR_NO_TILES", "1")
    for a, b in zip(got, run()):
        assert torch.equal(torch.as_tensor(a), torch.as_tensor(b))


@pytest.mark.parametrize("clustered", [False, True])
def test_jackknife_rows_by_their_subsamples_own_counts(mo, gpu, clustered):
    # each subsample's row against the cross-counts of its points with all points, in both
    # orders (row 0 is the rows' sum, so the rows' sum says nothing about them)
    import torch
    g = torch.Generator(device=gpu).manual_seed(3)
    n, box = 800001, 400.0
    t = torch.rand((n, 3), dtype=torch.float64, device=gpu, generator=g) * box
    if clustered:
        t[: n // 8] = 200.0 + 0.01 * (t[: n // 8] - 200.0)
    sub = torch.clamp((t / box * 5).long(), max=4)
    tags = 1 + (sub[:, 0] * 5 + sub[:, 1]) * 5 + sub[:, 2]
    rb = np.array([0.02, 0.1, 1.0, 4.0])
    jk = mo.npairs_jackknife_3d(t, t, rb, tags, tags, 125, period=box)
    assert torch.equal(jk[0], mo.npairs_3d(t, t, rb, period=box).double())
    for s in (1, 2, 31, 63, 94, 125):
        own = t[tags == s]
        both = mo.npairs_3d(own, t, rb, period=box) + mo.npairs_3d(t, own, rb, period=box)
        assert torch.equal(jk[0] - jk[s], 0.5 * both.double()), s


@pytest.mark.parametrize("layout", ["columns", "f32", "rows"])
@pytest.mark.parametrize("n1,n2", [(196609, 0), (270001, 262145), (300000, 1000)])
def test_large_builds_of_one_mock(mo, gpu, n1, n2, layout, monkeypatch):
    # one mock beyond the small builds: packed rows of columns, both sort tiles (a stable
    # sort: the same rows, hence the same bits), against the general kernels
    import torch
    t = [torch.as_tensor(_points(n, "seam" if i else "uniform", 5), device=gpu) for i, n in enumerate((n1, n2 or 1))]
    if layout == "columns":
        t = [x.t().contiguous().t() for x in t]
    elif layout == "f32":
        t = [x.to(torch.float32).clamp(0, float(np.nextafter(np.float32(L), np.float32(0)))) for x in t]
    p, q = t[0], t[1] if n2 else t[0]
    w = [torch.rand((len(x),), dtype=torch.float64, device=gpu, generator=torch.Generator(device=gpu).manual_seed(9))
         for x in t]
    rb = RB[:6]

    def run():
        return (mo.npairs_3d(p, q, rb, period=L), mo.npairs_per_object_3d(p, q, rb, period=L),
                mo.marked_npairs_3d(p, q, rb, period=L, weights1=w[0], weights2=w[1 if n2 else 0], weight_func_id=1))
    monkeypatch.setenv("HALOPAIR_SORT_TILE", "2048")
    small = run()
    monkeypatch.setenv("HALOPAIR_SORT_TILE", "8192")
    large = run()
    for a, b in zip(small, large):
        assert torch.equal(torch.as_tensor(a), torch.as_tensor(b))
    monkeypatch.setenv("HALOPAIR_NO_TILES", "1")
    ref = run()
    assert torch.equal(small[0], ref[0]) and torch.equal(small[1], ref[1])
    np.testing.assert_allclose(torch.as_tensor(small[2]).cpu(), torch.as_tensor(ref[2]).cpu(), rtol=1e-12)


@pytest.mark.parametrize("box", [(200.0, 30.0, 25.0), (25.0, 200.0, 30.0), (30.0, 25.0, 600.0), (300.0, 280.0, 24.0)])
@pytest.mark.parametrize("n1,n2", [(2000, 0), (300, 5000)])
def test_elongated_boxes(mo, n1, n2, box):
    # the curve's cubes have as many along each side of the box as along the others
    rng = np.random.default_rng([n1, int(box[0])])
    p1 = rng.uniform(0, 1, (n1, 3)) * box
    p2 = p1 if n2 == 0 else rng.uniform(0, 1, (n2, 3)) * box
    rb, kw = np.logspace(-1, np.log10(7.9), 10), dict(period=list(box))
    assert np.array_equal(mo.npairs_3d(p1, p2, rb, **kw), ORC.npairs_3d(p1, p2, rb, **kw))
    assert np.array_equal(mo.npairs_xy_z(p1, p2, rb, PI[:3], **kw), ORC.npairs_xy_z(p1, p2, rb, PI[:3], **kw))
    assert np.array_equal(mo.npairs_per_object_3d(p1, p2, rb, **kw), ORC.npairs_per_object_3d(p1, p2, rb, **kw))

"""Inputs at the edges of what the entry points take: far queries, queries next
to sources, values that are no numbers, radii below zero, more queries than 32
bits count, calls recorded into a graph."""
import ctypes
import threading

import numpy as np
import pytest
import torch

import oracle as O
from dwg_amd import gpu, shapes

pytestmark = pytest.mark.gpu

SIGMA = 10.0


def test_knn_far_query_beside_a_cell_boundary(ctx):
    # A point just below a cell's lower boundary that its rounded difference to
    # the grid's corner puts into that cell, and a query so far away that its
    # differences to the point and to the boundary round to neighbouring floats:
    # the cell's box lies farther than the point, which ties with others of
    # higher index for the last place.  n, the extent and two points a cell make
    # the cells 1/64 wide.
    f = np.float32
    rng = np.random.default_rng(3)
    p = np.nextafter(f(0.53125), f(0))
    rows = [(p, 0, 0), (0.535, 0, 0), (0.5, 0, 0), (0.505, 0, 0), (-1, -1, -1), (-0.999, -1, -1)]
    cells = rng.choice(24 * 62 * 62, 16384 - 4, replace=False)
    x, y, z = cells % 24 + 104, cells // 24 % 62 + 65, cells // (24 * 62) + 65
    c = np.stack([x, y, z], 1) / 64 - 1
    far_end = [(1, 0.3, 0.3), (1, 0.301, 0.301)]
    P = np.concatenate([np.array(rows), c + 0.3 / 64, c + 0.7 / 64, far_end]).astype(np.float32)
    Q = np.array([[-524288.0625, 0, 0]], np.float32)
    got, d2 = gpu.KnnIndex(ctx, P, k_hint=1).query(Q, 3, d2=True)
    ref, rd2 = O.knn_brute(P, Q, 3, return_d2=True)
    assert sorted(ref[0]) == [0, 4, 5]
    np.testing.assert_array_equal(got.cpu().numpy(), ref)
    np.testing.assert_array_equal(d2.cpu().numpy(), rd2)


def _factors(rho, screened):
    """g and |g'| of w = g(ρ) d·b, b already divided by 4π, in FP64."""
    s = SIGMA if screened else 0.0
    eps = (1e-7 if screened else 1e-8) / (4 * np.pi)
    e = np.exp(s * rho)
    den = e * rho ** 3 + eps
    return (s * rho + 1) / den, (e * rho ** 2 * (s * s * rho * rho + 3 * s * rho + 3) - s * eps) / den ** 2


# one tile, several in one chain's place (split over waves), a leaf of the tree
# in the walk of one query and of many (which share it)
@pytest.mark.parametrize("where,n,nq", [("direct", 64, 1), ("direct", 1024, 1), ("tree", 64, 5), ("tree", 64, 786_432)])
@pytest.mark.parametrize("screened", [False, True])
def test_gradient_component_is_rounded_at_its_own_size(ctx, where, n, nq, screened):
    # Each tile: one source whose component is the tile's sum P, then 63 whose
    # two products are 0.55 and 0.45 units in the last place of P.  Formed first, a
    # component is 0.1 units, and its addition rounds by half a unit at most; the
    # products added one by one round to a whole unit and to none.
    r = 0.5
    g, gp = _factors(r, screened)
    cos = np.sqrt(0.45 / 0.55 * g / (gp * r))
    big = 1.25 / g  # P = 1.25
    small = 0.55 * 2.0 ** -23 / g
    tiles = n // 64
    P = np.tile([r * cos, r * np.sqrt(1 - cos * cos), 0.0], (n, 1)).astype(np.float32)
    A = np.full(n, small * 4 * np.pi, np.float32)
    P[::64] = 0.0, -r, 0.0
    A[::64] = big * 4 * np.pi
    N = np.tile(np.float32([1, 0, 0]), (n, 1))
    Q = torch.zeros((nq, 3), device="cuda")
    if where == "direct":
        _, got = ctx.gwn_direct(P, N, A, Q, sigma=SIGMA, screened=screened, kahan=True, grad=True)
    else:
        tree = gpu.Octree(ctx, P.astype(np.float64), A.astype(np.float64), max_depth=10, leaf_size=64)
        assert tree.info()["nodes"] == 1
        tree.update(N, A)
        _, got = tree.eval_grad(Q, 2.3, sigma=SIGMA, screened=screened)
    got = got.cpu().numpy()[:, 0].astype(np.float64)
    d = P.astype(np.float64)
    rr = np.linalg.norm(d, axis=1)
    g, gp = _factors(rr, screened)
    b = A.astype(np.float64) / (4 * np.pi)
    want = (gp / rr * d[:, 0] * b * d[:, 0] - g * b).sum()
    # units of 2^-23: the factors of P (32·2^-24 of it, as the sums' own test
    # derives), half a unit an addition, one for the sums of the tiles
    assert np.abs(got - want).max() <= tiles * (16 * 1.25 + 63 * 0.5 + 1) * 2.0 ** -23


def test_plain_gradient_rounds_the_smaller_product(ctx):
    # Of a component c·d − g·b the product g·b is rounded before they meet.  The
    # factors are read from the results: with a moment along x and x and z offsets
    # that are powers of two, w is g and the z component c, each times a power; the
    # moments (1, b, −b·dy/dz) leave d·b, and so both, as they are.
    rng = np.random.default_rng(11)
    f = np.float32
    A, inv4pi = f(4 * np.pi), f(1 / (4 * np.pi))
    moment = lambda v: f(f(A * v) * inv4pi)  # as the sources are packed
    assert moment(f(1)) == 1
    dx = f(2.0) ** np.arange(-2, 2, dtype=f)
    checked = 0
    for _ in range(2000):
        dy, by = f(rng.integers(257, 1024) / 1024), f(rng.integers(257, 1024) / 1024)
        bz = -dy * by
        if moment(by) != by or moment(bz) != bz:
            continue
        q = np.stack([-dx, np.full(4, -dy), np.full(4, f(-1))], 1)
        run = lambda n: [x.cpu().numpy() for x in ctx.gwn_direct(np.zeros((1, 3), f), np.array([n], f), np.array([A]),
                                                                 q, screened=False, kahan=False, grad=True)]
        w, grad = run((1, 0, 0))
        g, c = w / dx, grad[:, 2]
        w2, got = run((1, by, bz))
        np.testing.assert_array_equal(w2, w)
        want = c.astype(np.float64) * np.float64(dy) - (g * by).astype(np.float64)
        np.testing.assert_array_equal(got[:, 1], want.astype(f))
        checked += 4
        if checked >= 400:
            break
    assert checked >= 200


# one chain and split over the sources
@pytest.mark.parametrize("n", [1, 300])
@pytest.mark.parametrize("grad,kahan", [(False, True), (True, True), (True, False)])
def test_screened_factors_take_the_distance_by_its_root(ctx, n, grad, kahan):
    # d·b = 1 at distances whose squares are the 4,096 numbers above 1: their roots
    # are half as many numbers (the root's error of a unit adds one at either end),
    # and so are the factors g = w
    f = np.float32
    m = 4096
    dy = np.sqrt(np.arange(1, m + 1) * 2.0 ** -23).astype(f)
    r2 = (1.0 + dy.astype(np.float64) ** 2).astype(f)
    assert len(np.unique(r2)) == m and r2[-1] - 1 == f(m * 2.0 ** -23)
    P, N, A = np.zeros((n, 3), f), np.zeros((n, 3), f), np.full(n, f(4 * np.pi))
    P[:, 0] = N[0, 0] = 1
    Q = np.zeros((m, 3), f)
    Q[:, 1] = -dy
    w = ctx.gwn_direct(P, N, A, Q, sigma=SIGMA, screened=True, kahan=kahan, grad=grad)
    w = (w[0] if grad else w).cpu().numpy()
    assert len(np.unique(w)) <= m // 2 + 3


# one chain and split over the sources
@pytest.mark.parametrize("n,nq", [(100, 7), (700, 300)])
@pytest.mark.parametrize("kahan,near64", [(False, False), (True, False), (True, True)])
def test_screened_direct_sums_leave_out_what_is_no_number(ctx, n, nq, kahan, near64):
    # a term whose distance is no number is 0, as one at the query itself: the
    # sums are those of sources without it, and a query that is no number gets 0
    P, N = shapes.sphere(n, 5)
    rng = np.random.default_rng(n)
    A = rng.uniform(1e-4, 3e-3, n).astype(np.float32)
    Q = np.concatenate([rng.uniform(-1.3, 1.3, (nq - nq // 4, 3)), P[: nq // 4]]).astype(np.float32)
    P, N, bad = P.astype(np.float32), N.astype(np.float32), np.arange(3, n, 41)
    P0, N0 = P.copy(), N.copy()
    P0[bad], N0[bad] = 0.25, 0.0  # the same places in the chain, no contribution
    P[bad, rng.integers(0, 3, len(bad))] = np.nan
    Qn = Q.copy()
    Qn[::5, 1] = np.nan
    kw = dict(sigma=SIGMA, screened=True, kahan=kahan, near64=near64)
    for grad in (False, True):
        want = ctx.gwn_direct(P0, N0, A, Q, grad=grad, **kw)
        got = ctx.gwn_direct(P, N, A, Qn, grad=grad, **kw)
        for w, v in zip(want if grad else (want,), got if grad else (got,)):
            w = w.cpu().numpy().copy()
            w[::5] = 0.0
            np.testing.assert_array_equal(v.cpu().numpy(), w)


# a walk a query (64 and 8 lanes) and walks shared by 64
@pytest.mark.parametrize("nq", [500, 50_000, 786_500])
def test_screened_tree_gradient_of_a_query_that_is_no_number(ctx, nq):
    n = 2000
    P, N = shapes.sphere(n, 5)
    rng = np.random.default_rng(nq)
    tree = gpu.Octree(ctx, P.astype(np.float64), None, max_depth=10)
    A = np.full(n, 2e-6, np.float32)
    tree.update(N, A)
    Q = rng.uniform(-1.3, 1.3, (nq, 3)).astype(np.float32)
    Q = torch.from_numpy(Q[np.lexsort((Q * 20).astype(int).T)]).cuda()  # in order, with or without the others
    w0, g0 = tree.eval_grad(Q, 2.3, sigma=SIGMA)
    Q[100:200:7, 2] = float("nan")
    w, g = tree.eval_grad(Q, 2.3, sigma=SIGMA)
    w0[100:200:7] = 0.0
    g0[100:200:7] = 0.0
    assert torch.equal(w, w0) and torch.equal(g, g0)


@pytest.mark.parametrize("n", [1, 60, 3000, 100_000])
@pytest.mark.parametrize("grad", [False, True])
def test_points_share_walks_by_the_size_of_the_tree(ctx, n, grad):
    # the last number of points that walk alone and the first that share walks,
    # in order and not: each the sums of few points, by a walk of 64 lanes
    P, N = shapes.sphere(n, 7)
    rng = np.random.default_rng(n)
    tree = gpu.Octree(ctx, P.astype(np.float64), None, max_depth=10)
    tree.update(N.astype(np.float32), np.full(n, 0.5 / n, np.float32))
    first = int(62000 * n ** (1 / 6) if grad else 82000 * n ** (1 / 12))
    Q = rng.uniform(-1.2, 1.2, (first + 1, 3)).astype(np.float32)
    sub = rng.permutation(first - 1)[:2000]
    few = tree.eval_grad(Q[sub], 2.3, sigma=SIGMA) if grad else (tree.eval(Q[sub], 2.3, sigma=SIGMA),)
    for ordered in (False, True):
        at = np.lexsort((Q * 20).astype(int).T) if ordered else np.arange(len(Q))
        back = torch.from_numpy(np.argsort(at)[sub]).cuda()
        for nq in (first - 1, first, first + 1):
            q = torch.from_numpy(Q[at]).cuda()
            keep = back < nq
            got = tree.eval_grad(q[:nq], 2.3, sigma=SIGMA) if grad else (tree.eval(q[:nq], 2.3, sigma=SIGMA),)
            for g, f, tol in zip(got, few, (1e-5, 1e-4)):  # the tree's bounds against FP64
                assert (g[back[keep]] - f[keep]).abs().max() <= tol * f.abs().max()


@pytest.mark.parametrize("n", [199, 200, 3000])
@pytest.mark.parametrize("kind", ["equal", "far", "mixed"])
def test_points_in_few_places_share_walks(ctx, n, kind):
    # many points in one bucket of the order, or beyond the cube, among others
    P, N = shapes.sphere(n, 7)
    rng = np.random.default_rng(n)
    tree = gpu.Octree(ctx, P.astype(np.float64), None, max_depth=10)
    tree.update(N.astype(np.float32), np.full(n, 0.5 / n, np.float32))
    nq = 200_001
    Q = rng.uniform(-1.2, 1.2, (nq, 3)).astype(np.float32)
    at = rng.uniform(size=nq)
    if kind != "far":
        Q[at < 0.4] = 0.3, -0.2, 1.01
    if kind != "equal":
        Q[at > 0.7] *= 40
        Q[at > 0.98, rng.integers(0, 3)] = np.inf
    sub = rng.permutation(nq)[:3000]
    few, got = tree.eval(Q[sub], 2.3, sigma=SIGMA), tree.eval(Q, 2.3, sigma=SIGMA)[torch.from_numpy(sub).cuda()]
    ok = torch.from_numpy(np.isfinite(Q[sub]).all(1)).cuda()
    assert (got[ok] - few[ok]).abs().max() <= 1e-5 * few[ok].abs().max()  # the tree's bound against FP64


@pytest.mark.parametrize("res,h", [((8, 4, 8), 0.05), ((33, 29, 31), 0.08), ((51, 53, 55), 0.02), ((401, 399, 1), 0.003),
                                   ((190, 181, 183), 0.005), ((195, 191, 185), 0.005), ((801, 803, 3), 0.003),
                                   ((3, 500, 600), 0.004)])
@pytest.mark.parametrize("screened,bf16,radii", [(True, False, False), (True, True, True), (False, False, False),
                                                 (False, True, False)])
def test_compensated_grid_walk_equals_the_point_walk(ctx, res, h, screened, bf16, radii):
    # with compensation too a grid value is the explicit point's bit for bit, by
    # whichever walk the grid's size picks
    P, N = shapes.union(3000, 8, 11)
    P = np.concatenate([P, P[:40], P[:3] + 1e-6]).astype(np.float64)
    N = np.concatenate([N, N[:40], N[:3]]).astype(np.float32)
    A = np.full(len(P), 2e-6, np.float32)
    R = np.linspace(0.0, 0.05, len(P), dtype=np.float32) if radii else None
    tree = gpu.Octree(ctx, P, None, max_depth=10)
    tree.update(N, A, R)
    c = P.mean(0)
    grid = gpu.make_grid([c[d] - 0.5 * h * (res[d] - 1) for d in range(3)], h, res)
    ax = [(np.arange(res[d]) * np.float64(grid.h) + grid.origin[d]).astype(np.float32) for d in range(3)]
    z, y, x = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    Q = torch.from_numpy(np.stack([x, y, z], -1).reshape(-1, 3).astype(np.float32)).cuda()
    kw = dict(sigma=SIGMA, screened=screened, bf16=bf16, kahan=True)
    got = tree.eval_grid(grid, 2.3, **kw).cpu().numpy()
    many = Q if len(Q) > 200_000 else Q.repeat(200_000 // len(Q) + 1, 1)
    want = tree.eval(many, 2.3, **kw).cpu().numpy()[:len(Q)]
    np.testing.assert_array_equal(got, want)
    assert tree.grid_terms(grid) == int(tree.terms(Q).sum())


@pytest.mark.parametrize("leaf_size", [1, 8])
def test_radii_below_zero_screen_nothing(ctx, leaf_size):
    # ρ = max(s, r) is r for a radius of 0, below 0 and no number alike, in every
    # walk and the direct sums
    n = 3000
    P, N = shapes.sphere(n, 4)
    rng = np.random.default_rng(n)
    A = rng.uniform(1e-6, 4e-6, n).astype(np.float32)
    R = rng.uniform(0.001, 0.05, n).astype(np.float32)
    off = rng.uniform(size=n) < 0.5
    P = P.astype(np.float32)
    Q = (P[rng.integers(0, n, 786_500)] + rng.normal(0, 0.01, (786_500, 3))).astype(np.float32)
    grid = gpu.make_grid([-1.1] * 3, 0.05, [45] * 3)

    def results(bad):
        r = R.copy()
        r[off] = np.where(np.arange(off.sum()) % 3 == 0, np.float32(bad), r[off] * np.float32(0 if bad == 0 else -1))
        tree = gpu.Octree(ctx, P.astype(np.float64), None, max_depth=6, leaf_size=leaf_size)
        tree.update(N, A, r)
        for near64 in (False, True):
            yield tree.eval(Q[:500], 2.3, sigma=SIGMA, near64=near64)
            yield tree.eval(Q[:200_000], 2.3, sigma=SIGMA, near64=near64)
            yield ctx.gwn_direct(P, N, A, Q[:3000], sigma=SIGMA, screened=True, radii=r, near64=near64)
        yield tree.eval_grid(grid, 2.3, sigma=SIGMA)
        for nq in (500, 50_000, 786_500):
            yield from tree.eval_grad(Q[:nq], 2.3, sigma=SIGMA)

    for want, got in zip(results(0.0), results(float("nan"))):
        assert bool(torch.isfinite(want).all()) and torch.equal(got, want)


def test_knn_query_that_is_no_number(ctx):
    # at no distance from any point, it has no neighbours, in a small query set as
    # in a tiled one
    P, _ = shapes.sphere(40_000, 3)
    P = P.astype(np.float32)
    idx = gpu.KnnIndex(ctx, P, k_hint=8)
    rng = np.random.default_rng(1)
    for nq in (100, 60_000):
        Q = rng.uniform(-1.2, 1.2, (nq, 3)).astype(np.float32)
        Q[5::7, rng.integers(0, 3)] = np.nan
        got, d2 = (t.cpu().numpy() for t in idx.query(Q, 8, d2=True))
        assert (got[5::7] == -1).all() and np.isinf(d2[5::7]).all()
        sub = [0, 1, 2, 3, 4, 6, 7, 8, 9, 10, 11, 13]
        np.testing.assert_array_equal(got[sub], O.knn_brute(P, Q[sub], 8))
    # nor is a point that is no number anyone's neighbour, one cell or several
    for scale in (0.0, 1.0):
        P = np.float32(scale) * rng.uniform(-1, 1, (40, 3)).astype(np.float32)
        P[::4, 1] = np.nan
        for nq in (5, 20_000):
            got = gpu.KnnIndex(ctx, P, k_hint=8).query(rng.uniform(-1, 1, (nq, 3)).astype(np.float32), 32)
            got = np.sort(got.cpu().numpy(), axis=1)
            assert (got[:, :2] == -1).all() and (got[:, 2:] == np.flatnonzero(np.arange(40) % 4)).all()


def test_index_whose_boxes_another_stream_builds(ctx):
    # the first far walk of many queries builds the boxes that small query sets
    # then take too, here on another stream and thread
    rng = np.random.default_rng(2)
    P, _ = shapes.sphere(30_000, 4)
    P = (0.5 * P).astype(np.float32)
    far = rng.uniform(-1, 1, (100_000, 3)).astype(np.float32)
    Q = rng.uniform(-1, 1, (500, 3)).astype(np.float32)
    want, want_far = O.knn_brute(P, Q, 15), O.knn_brute(P, far[:300], 15)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        other = gpu.Context(0)
        q = torch.from_numpy(Q).cuda()
    for _ in range(5):
        index = gpu.KnnIndex(ctx, P, k_hint=15)
        here = gpu.KnnIndex.__new__(gpu.KnnIndex)  # the same index by the other context
        here.ctx, here.pts, here.n, here.h = other, index.pts, index.n, index.h
        torch.cuda.synchronize()
        got = []
        walk = threading.Thread(target=lambda: got.append(index.query(far, 15)))
        walk.start()
        with torch.cuda.stream(stream):
            small = [here.query(q, 15) for _ in range(20)]
        walk.join()
        torch.cuda.synchronize()
        here.h = None
        for s in small:
            np.testing.assert_array_equal(s.cpu().numpy(), want)
        np.testing.assert_array_equal(got[0].cpu().numpy()[:300], want_far)
    other.close()


def test_more_queries_than_32_bits_count(ctx):
    # all but a few at one place; the sums at the others, and beside them, are
    # those of a call with few queries
    nq = 2 ** 31 + 77
    if torch.cuda.mem_get_info()[0] < 16 * nq + 2 ** 32:
        pytest.skip("the queries and their sums take 35 GB")
    P, N = shapes.sphere(3, 4)
    tree = gpu.Octree(ctx, P.astype(np.float64), None, max_depth=4)
    tree.update(N, np.full(3, 1e-3, np.float32))
    Q = torch.zeros((nq, 3), device="cuda")
    at = torch.tensor([0, 5, 2 ** 24 - 1, 2 ** 24, 2 ** 31 - 1, 2 ** 31, nq - 1], device="cuda")
    Q[at] = torch.rand((len(at), 3), device="cuda")
    at = torch.cat([at, at[1:] - 2])
    few = Q[at].repeat(30_000, 1)  # enough to share walks as the many do
    want = tree.eval(few, 2.3, sigma=SIGMA)[:len(at)].clone()
    got = tree.eval(Q, 2.3, sigma=SIGMA)
    assert torch.equal(got[at], want)
    del got
    want, wantg = (t[:len(at)].clone() for t in tree.eval_grad(few[:786_500], 2.3, sigma=SIGMA))
    w = torch.empty(nq, device="cuda")
    ctx.check(ctx.L.dwg_gwn_tree_grad(ctx.h, tree.h, ctypes.c_void_p(Q.data_ptr()), nq, 2.3, SIGMA, 1,
                                      ctypes.c_void_p(w.data_ptr()), None))
    ok = (w[at] - want).abs() <= 1e-5 * want.abs().max()
    assert bool(ok.all())
    del w, Q, few
    torch.cuda.empty_cache()


def test_scratch_of_many_queries_is_bounded():
    c = gpu.Context(0)
    P, N = shapes.sphere(100, 4)
    tree = gpu.Octree(c, P.astype(np.float64), None, max_depth=6)
    tree.update(N, np.full(100, 1e-3, np.float32))
    Q = torch.rand((40_000_000, 3), device="cuda")
    out = torch.empty(len(Q), device="cuda")
    tree.eval(Q[:300_000], 2.3, sigma=SIGMA, out=out)
    gpu.cache_release()
    before = torch.cuda.mem_get_info()[0]
    tree.eval(Q, 2.3, sigma=SIGMA, out=out)
    torch.cuda.synchronize()
    assert before - torch.cuda.mem_get_info()[0] <= 256 << 20
    want = tree.eval(Q[-200_000:], 2.3, sigma=SIGMA)
    assert torch.equal(out[-200_000:], want)
    del tree
    c.close()


@pytest.mark.parametrize("kind,nq", [("tree", 200_000), ("tree_grad", 786_500), ("direct", 1000)])
def test_sums_recorded_into_a_graph(kind, nq):
    # a recorded call takes no scratch that it has to allocate, and none that a
    # later call may give back: replayed after other work it gives the eager sums
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        c = gpu.Context(0)
        P, N = shapes.sphere(3000, 4)
        A = np.full(len(P), 1e-3, np.float32)
        P, N, A = (torch.from_numpy(a.astype(np.float32)).cuda() for a in (P, N, A))
        tree = gpu.Octree(c, P.cpu().numpy().astype(np.float64), None, max_depth=8)
        tree.update(N, A)
        Q = torch.rand((nq, 3), device="cuda") * 2 - 1
        more = torch.rand((4 * nq + 300_000, 3), device="cuda") * 2 - 1
        w, g = torch.empty(nq, device="cuda"), torch.empty((nq, 3), device="cuda")
        p = [ctypes.c_void_p(t.data_ptr()) for t in (P, N, A, Q, w, g)]

        def call(q, n, ow, og):
            if kind == "tree":
                rc = c.L.dwg_gwn_tree(c.h, tree.h, q, n, 2.3, SIGMA, 1, ow)
            elif kind == "tree_grad":
                rc = c.L.dwg_gwn_tree_grad(c.h, tree.h, q, n, 2.3, SIGMA, 1, ow, og)
            else:
                rc = c.L.dwg_gwn_direct(c.h, p[0], p[1], p[2], None, len(P), q, n, SIGMA, 1, ow, og)
            c.check(rc)

        def eager(q):
            ow, og = torch.empty(len(q), device="cuda"), torch.empty((len(q), 3), device="cuda")
            call(*(ctypes.c_void_p(t.data_ptr()) for t in (q,)), len(q),
                 *(ctypes.c_void_p(t.data_ptr()) for t in (ow, og)))
            return ow, og

        # the far radii of these flags, and the packed sources' buffers
        eager(more[:100] if kind != "direct" else more)
        s.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            call(p[3], nq, p[4], p[5])
        for i in range(3):
            Q.copy_(torch.rand((nq, 3), device="cuda") * 2 - 1)
            eager(more[: (i + 1) * len(more) // 3])  # scratch grows
            w.fill_(-1)
            graph.replay()
            s.synchronize()
            ow, og = eager(Q)
            assert torch.equal(w, ow)
            if kind != "tree":
                assert torch.equal(g, og)
        s.synchronize()
        del tree
        c.close()


# 240 runs of 64 cubes, 256, 2032 and 2048: by 4, 8 and 16 cubes along z a wave
@pytest.mark.parametrize("res", [(65, 121, 257), (65, 129, 250), (65, 1017, 243), (65, 1025, 257)])
def test_any_order_marching_cubes_by_runs(ctx, res):
    # the rows of the ordered pass, bit for bit
    x, y, z = (torch.arange(r, device="cuda", dtype=torch.float32) for r in res)
    f = (torch.sin(0.3 * x)[None, None] + torch.sin(0.2 * y)[None, :, None] + torch.sin(0.25 * z)[:, None, None]).ravel()
    grid = gpu.make_grid([-1.1, -0.9, -1.0], 0.05, res)
    _, cent, nrm = gpu.marching_cubes(ctx, f, grid, 0.5)
    c1, n1 = gpu.marching_cubes_any_order(ctx, f, grid, 0.5, capacity=len(cent))
    rows = [torch.cat([c, m], 1).cpu().numpy().view(np.uint32) for c, m in ((cent, nrm), (c1, n1))]
    assert len(rows[0]) > 100_000 and np.array_equal(*(r[np.lexsort(r.T[::-1])] for r in rows))


# 4096 tiles of 2048 numbers, of which every block adds up those before its own,
# and one more, with a scan of their sums; tiles that are whole and not
@pytest.mark.parametrize("n", [4096 * 2048 - 3, 4096 * 2048, 4096 * 2048 + 1])
def test_learned_start_of_a_large_cloud(ctx, n):
    """The subsample that a large cloud's patches are taken from (flags, scan,
    gather) against the same from numpy."""
    rng = np.random.default_rng(n)
    P = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    stride = np.uint32(-(-n // 50_000))
    h = np.arange(n, dtype=np.uint32) * np.uint32(0x9E3779B1)
    h ^= h >> np.uint32(16)
    h *= np.uint32(0x85EBCA6B)
    h ^= h >> np.uint32(13)
    sub = torch.from_numpy(P[h % stride == 0]).cuda()
    net = gpu.Mlp(ctx, 0)
    q = torch.from_numpy(P).cuda()
    got = net.init_normals(q, np.zeros(3))
    sel = torch.from_numpy(rng.integers(0, n, 20_000)).cuda()
    want = net.forward(net.patches_from(gpu.KnnIndex(ctx, sub, 17), q[sel]))
    assert torch.equal(got[sel].abs(), want.abs())  # (turned away from the centre)

"""The variants a call is dispatched to by its sizes, each at the edges of its
range, against the FP64 references."""
import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from dwg_amd import _lib, gpu, shapes
from mc_order import to_brick_order
from oracle import mlp as M

pytestmark = pytest.mark.gpu

EPS_PLAIN, EPS_SCREENED, SCREEN, SIGMA = 1e-8, 1e-7, 0.0015, 10.0


def _direct64(P, N, A, Q, screened):
    """w, ∇w and the sums of the terms' magnitudes, all pairs in FP64."""
    d = P[None].astype(float) - Q[:, None].astype(float)
    b = N.astype(float) * A.astype(float)[:, None]
    r = np.sqrt((d * d).sum(-1))
    dot = (d * b).sum(-1)
    if screened:
        rho = np.maximum(r, float(np.float32(SCREEN)))
        e = np.exp(SIGMA * rho) * 4 * np.pi
        den = e * rho ** 3 + EPS_SCREENED
        g = (SIGMA * rho + 1) / den
        gp = (SIGMA * EPS_SCREENED - e * rho ** 2 * (SIGMA ** 2 * rho ** 2 + 3 * SIGMA * rho + 3)) / den ** 2
        c = np.where(r >= rho, -dot * gp / r, 0.0)
    else:
        den = 4 * np.pi * r ** 3 + EPS_PLAIN
        g = 1 / den
        c = 12 * np.pi * r * dot * g * g
    grad = c[..., None] * d - g[..., None] * b
    mag = (np.abs(c)[..., None] * np.abs(d) + np.abs(g)[..., None] * np.abs(b)).sum(1)
    rb = r * np.sqrt((b * b).sum(-1))[None]
    return (g * dot).sum(1), grad.sum(1), (g * rb).sum(1), mag


# one wave of queries or less, a query past a wave, few sources (no split),
# the first split sizes, ragged last runs and tiles, many splits
@pytest.mark.parametrize("n,nq", [(1, 1), (127, 64), (255, 65), (256, 1), (257, 63), (1000, 1000), (8191, 130),
                                  (8193, 64), (70_001, 33)])
@pytest.mark.parametrize("screened", [False, True])
@pytest.mark.parametrize("kahan", [False, True])
def test_direct_sums_split_over_sources(ctx, n, nq, screened, kahan):
    P, N = shapes.sphere(n, 5)
    rng = np.random.default_rng(n + nq)
    A = rng.uniform(1e-4, 3e-3, n).astype(np.float32)
    Q = rng.uniform(-1.3, 1.3, (nq, 3)).astype(np.float32)
    w, g = ctx.gwn_direct(P, N, A, Q, sigma=SIGMA, screened=screened, kahan=kahan, grad=True)
    w1 = ctx.gwn_direct(P, N, A, Q, sigma=SIGMA, screened=screened, kahan=kahan)
    w, g, w1 = (t.cpu().numpy().astype(float) for t in (w, g, w1))
    rw, rg, mw, mg = _direct64(P, N, A, Q, screened)
    # a term: the rounding of d (up to 3 ulp of r), of r³ and of the factors,
    # 1-ulp sqrt, exp2 and reciprocal: under 32·2^-24 of |d||b|g; the chain of
    # 64 terms in FP32 adds at most 64·2^-24 of their magnitudes, without
    # compensation the tiles' partial sums as many again per tile
    tiles = 0 if kahan else (n + 63) // 64
    tol = (32 + 64 + tiles) * 2.0 ** -24
    assert (np.abs(w - rw) <= tol * mw + 1e-30).all()
    assert (np.abs(w1 - rw) <= tol * mw + 1e-30).all()
    assert (np.abs(g - rg) <= 2 * tol * mg + 1e-30).all()


# each point alone, parts and whole bricks cut by every face of the grid, a
# single point, a flat grid, grids far from and across the cloud, and a cloud far
# from the origin (large residuals of the rounded centres)
@pytest.mark.parametrize("res,h,shift", [((8, 4, 8), 0.05, 0.0), ((9, 5, 7), 0.002, 0.0), ((1, 1, 1), 0.1, 0.0),
                                         ((33, 29, 31), 0.08, 0.0), ((23, 3, 17), 0.3, 0.0),
                                         ((25, 26, 9), 0.05, 100.0), ((51, 53, 55), 0.02, 0.0),
                                         ((401, 399, 1), 0.003, 0.0), ((65, 66, 67), 0.02, 100.0),
                                         ((190, 181, 183), 0.005, 0.0), ((195, 191, 185), 0.005, 0.0)])
@pytest.mark.parametrize("screened,bf16,radii", [(True, False, False), (True, True, True), (False, False, False),
                                                 (False, True, False)])
def test_grid_walk_equals_the_point_walk(ctx, res, h, shift, screened, bf16, radii):
    # the brick's whole-box decisions are each point's own, so a grid value is
    # the explicit point's bit for bit where that takes the same terms in the
    # same order: in the shared walk of many points (here the grid's, repeated)
    P, N = shapes.union(3000, 8, 11)
    P = np.concatenate([P, P[:40], P[:3] + 1e-6]).astype(np.float64) + shift  # leaves of several points
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
    kw = dict(sigma=SIGMA, screened=screened, bf16=bf16)
    got = tree.eval_grid(grid, 2.3, **kw).cpu().numpy()
    many = Q if len(Q) > 200_000 else Q.repeat(200_000 // len(Q) + 1, 1)
    want = tree.eval(many, 2.3, **kw).cpu().numpy()[:len(Q)]
    np.testing.assert_array_equal(got, want)


# (points, queries): fewer points than k, one query, one cell's worth, a
# query set at each end of the sizes searched one query at a time and of the
# tiled ones (dense and not), and of those whose open queries are put in order
# (half of them, enough to share walks first)
@pytest.mark.parametrize("n,nq,k", [(1, 3, 4), (5, 1, 10), (40, 64, 32), (3000, 1, 1), (3000, 257, 32),
                                    (20_000, 16_383, 15), (2500, 16_384, 15), (33_000, 32_767, 8),
                                    (33_000, 32_768, 10), (2000, 40_000, 17), (9000, 262_143, 15),
                                    (9000, 262_144, 15)])
@pytest.mark.parametrize("skipped", [0.0, 0.5, 0.999])
def test_knn_by_query_count(ctx, n, nq, k, skipped):
    rng = np.random.default_rng(n + nq)
    P, _ = shapes.sphere(n, 3)
    P = (P + rng.normal(0, 0.002, P.shape)).astype(np.float32)
    P[: n // 8] = P[0]  # one cell holds an eighth of the points, all at one place
    Q = np.concatenate([P[rng.integers(0, n, nq - nq // 2)] + rng.normal(0, 0.01, (nq - nq // 2, 3)),
                        rng.uniform(-1.6, 1.6, (nq // 2, 3))]).astype(np.float32)
    skip = (rng.uniform(size=n) < skipped).astype(np.uint8)
    skip[-1] = 0
    idx = gpu.KnnIndex(ctx, P, k_hint=k)
    got, d2 = idx.query(Q, k, d2=True, skip=torch.from_numpy(skip) if skipped else None)
    sub = rng.permutation(nq)[:3000]  # the reference is brute force
    ref, rd2 = O.knn_brute(P, Q[sub], k, skip=skip if skipped else None, return_d2=True)
    np.testing.assert_array_equal(got.cpu().numpy()[sub], ref)
    # the oracle gives no distance where there is no neighbour, the library ∞
    np.testing.assert_array_equal(d2.cpu().numpy()[sub], np.where(ref < 0, np.inf, rd2))


@pytest.mark.parametrize("n,k", [(20, 32), (1331, 1), (1331, 7), (9261, 15), (9261, 32)])
def test_knn_ties_at_the_last_neighbour(ctx, n, k):
    # points of a lattice, the queries on them, between them and far off: the
    # k-th distance is that of several points, of which those of least index
    # stay (and all points where there are fewer than k)
    side = round(n ** (1 / 3)) if n > 20 else 3
    z, y, x = np.meshgrid(*(np.arange(side),) * 3, indexing="ij")
    P = np.stack([x, y, z], -1).reshape(-1, 3)[:n].astype(np.float32) / 16
    rng = np.random.default_rng(n + k)
    P = P[rng.permutation(n)]
    Q = np.concatenate([P, P + np.float32(1 / 32), P * np.float32([1, 1, 0]) + np.float32([0, 0, 8])])
    got, d2 = gpu.KnnIndex(ctx, P, k_hint=k).query(Q[:6000], k, d2=True)
    ref, rd2 = O.knn_brute(P, Q[:6000], k, return_d2=True)
    np.testing.assert_array_equal(got.cpu().numpy(), ref)
    np.testing.assert_array_equal(d2.cpu().numpy(), np.where(ref < 0, np.inf, rd2))


@pytest.mark.parametrize("nq", [31_000, 60_000, 70_000])
def test_knn_far_walk_hands_over(ctx, nq):
    # far queries near the centre of a sphere of 30,000 points: every point is
    # about as near as any other, so shared walks (of the last size) run out of
    # pops and their queries search alone
    rng = np.random.default_rng(5)
    P, _ = shapes.sphere(30_000, 4)
    P = (0.5 * P + rng.normal(0, 1e-4, P.shape)).astype(np.float32)
    Q = rng.normal(0, 0.02, (nq, 3)).astype(np.float32)
    idx = gpu.KnnIndex(ctx, P, k_hint=15)
    got, d2 = idx.query(Q, 15, d2=True)
    sub = rng.permutation(len(Q))[:3000]
    ref, rd2 = O.knn_brute(P, Q[sub], 15, return_d2=True)
    np.testing.assert_array_equal(got.cpu().numpy()[sub], ref)
    np.testing.assert_array_equal(d2.cpu().numpy()[sub], rd2)


# one query, the last set searched with 64 lanes a query, the first with 8, the
# first that share walks in order (unordered and ordered), and trees of one
# leaf, of one level and with leaves of several points
@pytest.mark.parametrize("n,nq,ordered", [(1, 5, False), (2, 1, False), (3000, 1, False), (3000, 39_999, False),
                                          (3000, 40_001, False), (3000, 196_607, False), (3000, 196_611, False),
                                          (3000, 196_611, True), (3000, 786_435, False)])
@pytest.mark.parametrize("screened,radii,bf16", [(True, False, False), (True, True, False), (False, False, False),
                                                 (True, False, True), (False, False, True)])
def test_tree_sums_by_query_count(ctx, n, nq, ordered, screened, radii, bf16):
    P, N = shapes.sphere(n, 7)
    rng = np.random.default_rng(n + nq)
    P = (0.5 * P + rng.normal(0, 0.002, P.shape)).astype(np.float32).astype(np.float64)
    P[: n // 10] = P[0]  # a leaf of several points
    A = rng.uniform(1e-6, 4e-6, n).astype(np.float32)
    R = rng.uniform(0.0015, 0.015, n).astype(np.float32) if radii else None
    Q = np.concatenate([P[rng.integers(0, n, nq // 2)] + rng.normal(0, 0.01, (nq // 2, 3)),
                        rng.uniform(-0.8, 0.8, (nq - nq // 2, 3))]).astype(np.float32)
    if ordered:
        Q = Q[np.lexsort((Q * 40).astype(int).T)]
    tree = gpu.Octree(ctx, P, A.astype(np.float64), max_depth=10)
    tree.update(N, A, R)
    o = O.Octree(P, 10, 1)
    o.precompute(N.astype(np.float64), A.astype(np.float64))
    sub = rng.permutation(nq)[:1500]
    kind = "screened" if screened else "plain"
    rad = None if R is None else R.astype(np.float64)
    ref = o.eval(Q[sub].astype(np.float64), 2.3, kind=kind, sigma=SIGMA, radii=rad)
    w = tree.eval(Q, 2.3, sigma=SIGMA, screened=screened, bf16=bf16).cpu().numpy()[sub]
    if bf16:
        # the rounded moments are the same for every walk: against the shared
        # walk of many points (the queries compared, repeated)
        many = torch.from_numpy(np.tile(Q[sub], (200_000 // len(sub) + 1, 1)))
        ref = tree.eval(many, 2.3, sigma=SIGMA, screened=screened, bf16=True).cpu().numpy()[:len(sub)]
    # FP32 terms: 1e-5 of max|w|, the bound the precision sweep holds
    assert np.abs(w - ref).max() <= 1e-5 * np.abs(ref).max()
    if bf16:
        return
    wg, g = (t.cpu().numpy()[sub] for t in tree.eval_grad(Q, 2.3, sigma=SIGMA, screened=screened))
    assert np.abs(wg - ref).max() <= 1e-5 * np.abs(ref).max()
    rw, rg = o.eval_grad(Q[sub].astype(np.float64), 2.3, kind=kind, sigma=SIGMA, radii=rad)
    assert np.abs(g - rg).max() <= 1e-4 * np.abs(rg).max()  # the tree gradient's bound


# one row, a block of rows but one, one past it, past one split of the rows,
# past a multiple of it, and enough splits to take more rows each
@pytest.mark.parametrize("batch", [1, 31, 33, 257, 2049, 70_001])
@pytest.mark.parametrize("line", [False, True])
def test_training_gradient_by_batch(ctx, batch, line):
    rng = np.random.default_rng(batch)
    theta = np.concatenate([(rng.uniform(-1, 1, s) / np.sqrt(s[1] if len(s) == 2 else 64)).ravel()
                            for s in M.SIZES]).astype(np.float32)
    net = gpu.Mlp(ctx, 0)
    net.set_params(theta)
    X = M.to_bf16(rng.normal(size=(batch, 48)).astype(np.float32))
    T = rng.normal(size=(batch, 3)) + [1.0, 0.5, 0.0]
    T /= np.linalg.norm(T, axis=1, keepdims=True)
    xb = torch.from_numpy(M.bf16_bits(X).view(np.int16)).cuda()
    loss = net.loss_grad(xb, torch.from_numpy(T.astype(np.float32)), line=line)
    g = net.grad().astype(np.float64)
    W = [torch.from_numpy(M.to_bf16(a.astype(np.float32)).astype(np.float64) if a.ndim == 2 else a.astype(np.float64))
         .requires_grad_(True) for a in M.unpack(theta)]
    h = torch.from_numpy(X.astype(np.float64))
    for w, b in ((W[0], W[1]), (W[2], W[3])):
        h = torch.nn.functional.gelu(h @ w.T + b, approximate="tanh")
    y = h @ W[4].T + W[5]
    c = (y / y.norm(dim=1, keepdim=True) * torch.from_numpy(T)).sum(1)
    ref = (1 - c * c if line else 1 - c).mean()
    ref.backward()
    rg = torch.cat([w.grad.reshape(-1) for w in W]).numpy()
    # the bounds of the 512-row gradient: BF16 activations and their gradients
    assert loss == pytest.approx(float(ref.detach()), abs=1e-2 if batch < 32 else 1e-3)
    assert np.linalg.norm(g - rg) < 0.03 * np.linalg.norm(rg)


@pytest.mark.parametrize("n", [1, 2, 9, 3000, 30_011])
@pytest.mark.parametrize("screened,bf16,kahan,radii", [(True, False, False, False), (True, True, True, True),
                                                       (False, False, True, False), (False, True, False, False)])
def test_own_points_equal_the_shared_walk(ctx, n, screened, bf16, kahan, radii):
    # the sums at the tree's own points, 8 lanes a point, against the shared walk
    # of as many explicit points as take it: the same terms in the same order
    P, N = shapes.sphere(n, 9)
    P = P.astype(np.float32)
    P[: n // 20] = P[0]  # a leaf of several points
    A = np.full(n, 2e-6, np.float32)
    R = np.linspace(0.0, 0.05, n, dtype=np.float32) if radii else None
    tree = gpu.Octree(ctx, P.astype(np.float64), None, max_depth=10)
    tree.update(N, A, R)
    out = torch.full((n,), float("nan"), device="cuda")
    flags = tree._flags(screened, None, kahan, bf16)
    ctx.check(ctx.L.dwg_gwn_tree_self(ctx.h, tree.h, ctypes.c_float(2.3), ctypes.c_float(SIGMA), flags,
                                      ctypes.c_void_p(out.data_ptr())))
    many = torch.from_numpy(np.tile(P, (200_000 // n + 1, 1)))
    want = tree.eval(many, 2.3, sigma=SIGMA, screened=screened, bf16=bf16, kahan=kahan)[:n]
    np.testing.assert_array_equal(out.cpu().numpy(), want.cpu().numpy())


@pytest.mark.parametrize("n,ntri", [(300, 20_000), (2500, 90_000), (40_000, 41_000)])
def test_diffusion_of_crowded_tiles(ctx, n, ntri):
    # tiles of up to thousands of centroids, split over blocks: every face normal
    # reaches its 15 nearest sources once, in the same fixed-point sums
    rng = np.random.default_rng(n)
    P, N = shapes.sphere(n, 6)
    P = (0.5 * P).astype(np.float32)
    C = (P[rng.integers(0, n, ntri)] + rng.normal(0, 0.01, (ntri, 3))).astype(np.float32)
    T = rng.normal(size=(ntri, 3)).astype(np.float32)
    T /= np.linalg.norm(T, axis=1, keepdims=True)
    nrm = torch.from_numpy(N.astype(np.float32)).cuda()
    gpu.diffuse_normals(ctx, gpu.KnnIndex(ctx, P, 15), C, T, nrm, zero_threshold=n)
    idx = O.knn_brute(P, C, 15) if n * ntri < 1e9 else O.knn_grid(P, C, 15)
    acc = np.zeros((n, 3), np.int64)
    fixed = np.rint(T.astype(np.float64) * 2.0 ** 40).astype(np.int64)
    for k in range(15):
        np.add.at(acc, idx[:, k], fixed)
    a = acc * 2.0 ** -40
    length = np.linalg.norm(a, axis=1, keepdims=True)
    want = np.where(length < 1e-10, N, a / (length + 1e-8))
    # FP64 until the last rounding on both sides
    np.testing.assert_allclose(nrm.cpu().numpy(), want, rtol=2.0 ** -23, atol=1e-12)


@pytest.mark.parametrize("res,crossed", [((2, 2, 2), "all"), ((65, 9, 17), "all"), ((66, 10, 19), "all"),
                                         ((130, 19, 35), "all"), ((9, 1030, 1030), "few")])
def test_marching_cubes_by_runs(ctx, res, crossed):
    """Runs of 64 cubes that end on, before and past the grid's end, by a block
    and by a wave (the last size), with every cube crossed or few, and samples
    that are infinite or not a number (above no level): the ordered mesh is the
    oracle's in brick order, and the any-order pass has its rows bit for bit."""
    rng = np.random.default_rng(sum(res))
    n = res[0] * res[1] * res[2]
    if crossed == "all":
        f = rng.normal(size=n).astype(np.float32)
        if n > 8:
            f[rng.integers(0, n, 20)] = np.repeat(np.float32([np.nan, np.inf, -np.inf, 0.0]), 5)
        f[:2] = 1.0, -1.0  # a triangle at least
    else:
        z, y, x = np.meshgrid(*(np.arange(r, dtype=np.float32) for r in res[::-1]), indexing="ij")
        f = (np.hypot(y - 512, z - 500) - 480 + np.sin(x)).astype(np.float32).ravel()
    origin, h = np.float32([-1.1, -0.9, -1.0]), np.float32(0.05)
    grid = gpu.make_grid(origin, h, np.int32(res))
    ft = torch.from_numpy(f).cuda()
    tris, cent, nrm = gpu.marching_cubes(ctx, ft, grid, 0.0, tris=True)
    with np.errstate(all="ignore"):
        rt, rc, _ = O.marching_cubes(f.astype(np.float64), np.int32(res), origin.astype(float), float(h), 0.0)
    order = to_brick_order(f, res, np.float32(0))
    assert len(rt) == tris.shape[0] > 0
    # a vertex: two rounded corners, their difference, its multiple and the sum,
    # each half a unit of the largest coordinate; a centroid: three more
    ulp = 2.0 ** -23 * (1.1 + float(h) * max(res))
    for got, want, tol in ((tris, rt, 4 * ulp), (cent, rc, 8 * ulp)):
        got, want = got.cpu().numpy(), want[order]
        assert np.array_equal(np.isnan(got), np.isnan(want))
        ok = ~np.isnan(want)
        assert np.abs(got[ok] - want[ok]).max() <= tol
    c1, n1 = gpu.marching_cubes_any_order(ctx, ft, grid, 0.0, capacity=len(rt))
    rows = [np.concatenate([c.cpu().numpy(), m.cpu().numpy()], 1).view(np.uint32) for c, m in ((cent, nrm), (c1, n1))]
    assert np.array_equal(*(r[np.lexsort(r.T[::-1])] for r in rows))


@pytest.mark.parametrize("wanted", [(1, 1, 1), (1, 0, 0), (0, 0, 1), (0, 0, 0), None])
def test_marching_cubes_into_given_buffers(ctx, wanted):
    """The buffers that the allocator gives hold what the two calls with a
    capacity write; an allocator that gives up leaves an error, not a result."""
    rng = np.random.default_rng(8)
    res = (40, 21, 33)
    f = torch.from_numpy(rng.normal(size=res[0] * res[1] * res[2]).astype(np.float32)).cuda()
    grid = gpu.make_grid([0.0, 0.0, 0.0], 0.1, np.int32(res))
    want = gpu.marching_cubes(ctx, f, grid, 0.0, tris=True)
    T, n = want[0].shape[0], ctypes.c_int64()
    ref = [torch.empty_like(w) for w in want]
    args = (ctx.h, ctypes.c_void_p(f.data_ptr()), ctypes.byref(grid), 0.0)
    ctx.check(ctx.L.dwg_marching_cubes(*args, T, *(ctypes.c_void_p(r.data_ptr()) for r in ref), ctypes.byref(n)))
    assert n.value == T > 1000 and all(torch.equal(a, b) for a, b in zip(want, ref))
    got, calls = [torch.zeros_like(w) for w in want], []

    def alloc(_, count, *where):
        calls.append(count)
        if wanted is None:
            return 1
        for b, use, w in zip(got, wanted, where):
            w[0] = b.data_ptr() if use else None
        return 0

    rc = ctx.L.dwg_marching_cubes_alloc(*args, _lib.MC_ALLOC(alloc), None, ctypes.byref(n))
    assert calls == [T] and rc == (0 if wanted else _lib.DWG_ERR_ARG)
    torch.cuda.synchronize()
    for b, use, w in zip(got, wanted or (0, 0, 0), want):
        assert torch.equal(b, w) if use else not b.any()

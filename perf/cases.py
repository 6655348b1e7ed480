"""The calls a DWG user makes, over the sizes they are made at.

Each case is one call (or the few calls of one step) through the package's
public entry points on inputs made on the GPU from a seed.  ``listed`` names
the fixed cases, ``draw`` gives others of the same kinds and ranges,
``prepare`` makes what a program holds before the call, ``run`` is one pass,
``work`` counts the bytes and operations a pass cannot do without, and
``exact`` gives the outputs in 64 bits from plain torch where that is
affordable.
"""
from __future__ import annotations

import math
import os

import numpy as np
import torch

import dwg_amd
from dwg_amd import gpu, pipeline

WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(dwg_amd.__file__)), "weights", "dwg_mlp.bin")
AREA = 2e-6            # the method's constant source area
BETA = 2.3             # its default Barnes-Hut accuracy
EPS_PLAIN, EPS_SCREENED, SCREEN = 1e-8, 1e-7, 0.0015
MAX_DEPTH = 10
F64 = torch.float64

_CTX = None


def _ctx():
    """One context for the program, as a user keeps it."""
    global _CTX
    if _CTX is None:
        _CTX = gpu.Context(0)
    return _CTX


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the field of a tiny cloud on a tiny grid: one call of an interactive
        # preview, where launches count (the package's smoke step is this size)
        dict(name="grid_2k_ragged33", kind="grid", n=2_000, rx=33, ry=29, rz=31, sigma=20.0, screened=True,
             bf16=False, kahan=False),
        # the headline's dominant call: one million sources, a 512^3 grid,
        # mixed precision as the learned iterations run it
        dict(name="grid_1m_512_mixed", kind="grid", n=1_000_000, rx=512, ry=512, rz=512, sigma=10.0, screened=True,
             bf16=True, kahan=True),
        # winding numbers at a cloud's own and at free points, in the caller's
        # order (inside / outside tests, the sums at the sources)
        dict(name="points_400k_300k", kind="points", n=400_000, nq=300_000, sigma=10.0, screened=True, grad=False,
             kahan=False),
        # value and gradient at points: the backward direction of the sums
        dict(name="grad_100k_100k", kind="points", n=100_000, nq=100_000, sigma=10.0, screened=True, grad=True,
             kahan=False),
        # the small-sphere configuration: all pairs of 10,000 sources with a
        # 128^3 grid's points
        dict(name="direct_10k_2m", kind="direct", n=10_000, nq=128 ** 3, sigma=10.0, screened=True, grad=False,
             kahan=False),
        # reference sums at a few thousand probes over a large cloud, with
        # compensated accumulation and the gradient
        dict(name="direct_200k_2k_grad", kind="direct", n=200_000, nq=2_000, sigma=10.0, screened=True, grad=True,
             kahan=True),
        # one diffusion step of the headline: 15 nearest sources of 3 million
        # triangle centroids, scatter, normalisation, refill of the zero ones
        dict(name="diffuse_1m_3m", kind="diffuse", n=1_000_000, ncent=3_000_000, far=0.06),
        # a small neighbour query (the reference's default k of radii and
        # normal transfer)
        dict(name="knn_100k_1500", kind="knn", n=100_000, nq=1_500, k=10),
        # the final mesh: ordered marching cubes of a ragged large grid
        dict(name="mc_480x512x451", kind="mc", rx=480, ry=512, rz=451, tris=True),
        # one training step of the learned start (the trainer's batch)
        dict(name="mlp_train_8192", kind="train", batch=8192, line=True),
        # the learned start of a mid-sized cloud: patches and network
        dict(name="mlp_init_300k", kind="init", n=300_000),
        # a whole default reconstruction of a small cloud, for its normals (as
        # the trainer's data sets are made)
        dict(name="recon_30k_128", kind="recon", n=30_000, reso=128, iters=6),
    ]


def _log(rng, lo, hi):
    """log-uniform integer, odd half of the time or more"""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, v | 1 if rng.random() < 0.5 else v))


def draw(rng):
    kind = rng.choice(["grid", "grid", "points", "points", "direct", "direct", "diffuse", "knn", "mc", "train", "init",
                       "recon"])
    sigma = rng.choice([10.0, 20.0, 7.5])
    if kind == "grid":
        n, s = _log(rng, 500, 1_000_000), _log(rng, 16, 400)
        r = [max(5, int(s * rng.uniform(0.6, 1.0))) for _ in range(3)]
        return dict(kind=kind, n=n, rx=r[0], ry=r[1], rz=r[2], sigma=sigma, screened=rng.random() < 0.75,
                    bf16=rng.random() < 0.4, kahan=rng.random() < 0.4)
    if kind == "points":
        n, nq = _log(rng, 1_000, 600_000), _log(rng, 300, 500_000)
        return dict(kind=kind, n=n, nq=nq, sigma=sigma, screened=rng.random() < 0.75, grad=rng.random() < 0.5,
                    kahan=False)
    if kind == "direct":
        n = _log(rng, 300, 200_000)
        nq = _log(rng, 300, max(301, min(2_000_000, int(2e10 / n) // 2)))
        return dict(kind=kind, n=n, nq=nq, sigma=sigma, screened=rng.random() < 0.5, grad=rng.random() < 0.4,
                    kahan=rng.random() < 0.5)
    if kind == "diffuse":
        n = _log(rng, 5_000, 1_000_000)
        return dict(kind=kind, n=n, ncent=int(n * rng.uniform(1.2, 3.0)), far=round(rng.uniform(0.01, 0.2), 3))
    if kind == "knn":
        return dict(kind=kind, n=_log(rng, 2_000, 400_000), nq=_log(rng, 100, 4_000), k=rng.choice([1, 8, 10, 15, 16]))
    if kind == "mc":
        s = _log(rng, 24, 440)
        r = [max(9, int(s * rng.uniform(0.6, 1.0))) for _ in range(3)]
        return dict(kind=kind, rx=r[0], ry=r[1], rz=r[2], tris=rng.random() < 0.5)
    if kind == "train":
        return dict(kind=kind, batch=_log(rng, 500, 16_384), line=rng.random() < 0.7)
    if kind == "init":
        return dict(kind=kind, n=_log(rng, 2_000, 600_000))
    return dict(kind=kind, n=_log(rng, 3_000, 50_000), reso=_log(rng, 48, 144), iters=rng.choice([2, 4, 6]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _unit(v):
    return v / v.norm(dim=-1, keepdim=True).clamp_min(1e-12)


def _cloud(n, seed, m=32):
    """n points on the boundary of a union of m random balls and ellipsoids in
    the unit cube, noise 0.001, in random order, with outward normals; scaled
    as the reader scales its input (centred, longest side 1)."""
    g = _gen(seed)

    def u(*shape):
        return torch.rand(*shape, generator=g, device="cuda", dtype=F64)

    axes = 0.06 + 0.22 * u(m, 3)
    ball = torch.arange(m, device="cuda") % 2 == 0
    axes[ball] = axes[ball, :1].expand(-1, 3)
    ctr = 0.28 + 0.44 * u(m, 3)
    share = (axes.prod(1) ** (2 / 3))
    pts, nrm, have = [], [], 0
    while have < n:
        c = 2 * (n - have) + 4096
        i = torch.multinomial(share, c, replacement=True, generator=g)
        d = _unit(torch.randn(c, 3, generator=g, device="cuda", dtype=F64))
        x = ctr[i] + axes[i] * d
        keep = torch.ones(c, dtype=torch.bool, device="cuda")
        for j in range(m):
            z = (x - ctr[j]) / axes[j]
            keep &= (z.square().sum(1) > 1 - 1e-9) | (i == j)
        pts.append(x[keep])
        nrm.append(_unit(d / axes[i])[keep])
        have += int(keep.sum())
    p, q = torch.cat(pts)[:n], torch.cat(nrm)[:n]
    p = p + 0.001 * torch.randn(n, 3, generator=g, device="cuda", dtype=F64)
    p = p - (p.amax(0) + p.amin(0)) / 2
    p = p / (2 * p.abs().max())
    return p.float(), q.float().contiguous(), g


def _grid(p, r, pad=0.05):
    lo, hi = p.double().amin(0) - pad, p.double().amax(0) + pad
    h = float(max((float(hi[d] - lo[d])) / (r[d] - 1) for d in range(3)))
    return gpu.make_grid([float((lo[d] + hi[d]) / 2 - (r[d] - 1) / 2 * h) for d in range(3)], h, r)


def _tree(p, nrm):
    tree = gpu.Octree(_ctx(), p.double().cpu().numpy(), None, max_depth=MAX_DEPTH)
    tree.update(nrm, torch.full((p.shape[0],), AREA, device="cuda"))
    return tree


def _queries(p, nq, g):
    """half near the cloud (a point moved by 0.004), half anywhere in its box, mixed"""
    a = nq // 2
    i = torch.randint(0, p.shape[0], (a,), generator=g, device="cuda")
    near = p[i] + 0.004 * torch.randn(a, 3, generator=g, device="cuda")
    free = (torch.rand(nq - a, 3, generator=g, device="cuda") - 0.5) * 1.1
    q = torch.cat([near, free])
    return q[torch.randperm(nq, generator=g, device="cuda")].contiguous()


def _centroids(p, nrm, ncent, far, g, cell=1.1 / 512):
    """triangle centroids and face normals of an iteration: most within a grid
    cell of a source, `far` of them on spurious closed pieces inside, none in
    a few bare patches (whose sources stay without a face), in brick order"""
    nf = int(ncent * far)
    covered = torch.ones(p.shape[0], dtype=torch.bool, device="cuda")
    for b in p[torch.randint(0, p.shape[0], (24,), generator=g, device="cuda")]:
        covered &= (p - b).norm(dim=1) > 0.02
    have = torch.nonzero(covered)[:, 0]
    i = have[torch.randint(0, have.numel(), (ncent - nf,), generator=g, device="cuda")]
    near = p[i] + cell * (torch.rand(ncent - nf, 3, generator=g, device="cuda") - 0.5) * 2
    nn = _unit(nrm[i] + 0.2 * torch.randn(ncent - nf, 3, generator=g, device="cuda"))
    s = torch.randint(0, 12, (nf,), generator=g, device="cuda")
    c, r = p[torch.randint(0, p.shape[0], (12,), generator=g, device="cuda")] * 0.5, 0.02 + 0.1 * torch.rand(
        12, generator=g, device="cuda")
    d = _unit(torch.randn(nf, 3, generator=g, device="cuda"))
    cent, tn = torch.cat([near, c[s] + r[s, None] * d]), torch.cat([nn, d])
    b = ((cent + 0.6) / cell).long().clamp(0, 4095)
    key = (b[:, 2] // 16 * 512 + b[:, 1] // 8) * 512 + b[:, 0] // 8
    o = torch.argsort(key, stable=True)
    return cent[o].contiguous(), tn[o].contiguous()


def _field(case, seed):
    """an iso-surface like a winding field's: a soft union of balls, rippled,
    at a place of the grid that the seed chooses (so that every seed has the
    same number of triangles)"""
    g = _gen(1)
    r = (case["rx"], case["ry"], case["rz"])
    h = 1.0 / (max(r) - 1)
    rng = np.random.default_rng(seed)
    x, y, z = ((torch.arange(k, device="cuda") - int(rng.integers(0, k // 8 + 1))) * h for k in r)
    c = torch.rand(24, 3, generator=g, device="cuda")
    c = (0.2 + 0.45 * c) * (torch.tensor(r, device="cuda") / max(r))
    rad = (0.04 + 0.08 * torch.rand(24, generator=g, device="cuda")) * (min(r) / max(r))
    f = torch.full((r[2], r[1], r[0]), -9.0, device="cuda")
    for j in range(24):
        d2 = ((z - c[j, 2]) ** 2)[:, None, None] + ((y - c[j, 1]) ** 2)[None, :, None] + (x - c[j, 0]) ** 2
        f = torch.maximum(f, (rad[j] - d2.sqrt_()) / 0.05)
    f = 0.5 + 0.5 * torch.tanh(f)
    f += 0.01 * (torch.sin(61 * x)[None, None, :] * torch.sin(53 * y)[None, :, None] * torch.sin(47 * z)[:, None, None])
    return f.contiguous(), gpu.make_grid((0.0, 0.0, 0.0), h, r)


def _train_batch(case, seed):
    """BF16 patches (offsets in the unit ball, distance order) and unit targets"""
    g = _gen(seed)
    b = case["batch"]
    off = torch.randn(b, 16, 3, generator=g, device="cuda")
    off[..., 2] *= 0.15
    t = _unit(torch.randn(b, 3, generator=g, device="cuda"))
    e = _unit(torch.linalg.cross(t, torch.randn(b, 3, generator=g, device="cuda")))
    frame = torch.stack([e, torch.linalg.cross(t, e), t], 1)
    off = (off[..., :, None] * frame[:, None]).sum(2)
    o = off.norm(dim=-1).argsort(1)
    off = off.gather(1, o[..., None].expand(-1, -1, 3))
    off = off / off[:, -1:].norm(dim=-1, keepdim=True)
    return off.reshape(b, 48).bfloat16().view(torch.int16).contiguous(), t.contiguous()


def prepare(case, seed):
    ctx, k = _ctx(), case["kind"]
    s = dict(case=case, ctx=ctx)
    if k == "mc":
        s["field"], s["grid"] = _field(case, seed)
        return s
    if k == "train":
        s["x"], s["t"] = _train_batch(case, seed)
        s["net"] = gpu.Mlp(ctx, seed=int(seed))
        return s
    p, nrm, g = _cloud(case["n"], seed)
    s["p"], s["nrm"] = p, nrm
    if k == "grid":
        s["tree"] = _tree(p, nrm)
        s["grid"] = _grid(p, (case["rx"], case["ry"], case["rz"]))
        s["out"] = torch.empty(case["rx"] * case["ry"] * case["rz"], device="cuda")
    elif k == "points":
        s["tree"], s["q"] = _tree(p, nrm), _queries(p, case["nq"], g)
    elif k == "direct":
        s["area"], s["q"] = torch.full((case["n"],), AREA, device="cuda"), _queries(p, case["nq"], g)
    elif k == "diffuse":
        s["cent"], s["tn"] = _centroids(p, nrm, case["ncent"], case["far"], g)
        s["index"] = gpu.KnnIndex(ctx, p, 15)
    elif k == "knn":
        s["index"], s["q"] = gpu.KnnIndex(ctx, p, case["k"]), _queries(p, case["nq"], g)
    elif k == "init":
        s["net"] = gpu.Mlp(ctx, path=WEIGHTS)
        s["center"] = tuple(float(v) for v in (p.amax(0) + p.amin(0)).cpu() / 2)
    else:
        s["host"] = p.cpu().numpy()
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    c, ctx, k = s["case"], s["ctx"], s["case"]["kind"]
    if k == "grid":
        return s["tree"].eval_grid(s["grid"], BETA, sigma=c["sigma"], screened=c["screened"], kahan=c["kahan"],
                                   bf16=c["bf16"], out=s["out"])
    if k == "points":
        if c["grad"]:
            return s["tree"].eval_grad(s["q"], BETA, sigma=c["sigma"], screened=c["screened"])
        return s["tree"].eval(s["q"], BETA, sigma=c["sigma"], screened=c["screened"], kahan=c["kahan"])
    if k == "direct":
        return ctx.gwn_direct(s["p"], s["nrm"], s["area"], s["q"], sigma=c["sigma"], screened=c["screened"],
                              kahan=c["kahan"], grad=c["grad"])
    if k == "diffuse":
        nz = gpu.diffuse_normals(ctx, s["index"], s["cent"], s["tn"], s["nrm"])
        return s["nrm"], nz
    if k == "knn":
        return s["index"].query(s["q"], c["k"], d2=True)
    if k == "mc":
        t, cen, n = gpu.marching_cubes(ctx, s["field"], s["grid"], 0.5, tris=c["tris"])
        return (t, cen, n) if c["tris"] else (cen, n)
    if k == "train":
        loss = s["net"].loss_grad(s["x"], s["t"], line=c["line"])
        return s["net"].grad(), loss
    if k == "init":
        return s["net"].init_normals(s["p"], s["center"])
    r = pipeline.reconstruct(ctx, s["host"], want_mesh=False, source_mode=1, grid_reso=c["reso"],
                             final_reso=c["reso"], total_iter=c["iters"], input_normal=3)
    return r.normals, r.w_mean


# ---------------------------------------------------------------------------
# the work of a pass
# ---------------------------------------------------------------------------
def _terms(n):
    """Barnes-Hut terms a query takes, about (185 for a million sources)"""
    return 9.3 * math.log2(n)


def work(c):
    k = c["kind"]
    f = 27.0 if c.get("screened", True) else 20.0
    if k == "grid":
        g = c["rx"] * c["ry"] * c["rz"]
        return dict(bytes=4.0 * g + 32.0 * c["n"], flops=f * g * _terms(c["n"]))
    if k == "points":
        return dict(bytes=(28.0 if c["grad"] else 16.0) * c["nq"] + 32.0 * c["n"],
                    flops=(2.0 if c["grad"] else 1.0) * f * c["nq"] * _terms(c["n"]))
    if k == "direct":
        return dict(bytes=(28.0 if c["grad"] else 16.0) * c["nq"] + 28.0 * c["n"],
                    flops=(2.0 if c["grad"] else 1.0) * f * c["nq"] * c["n"])
    if k == "diffuse":  # centroids and face normals read, sources read and their normals written; ~60 candidates
        return dict(bytes=24.0 * c["ncent"] + 24.0 * c["n"], flops=8.0 * 60 * c["ncent"])
    if k == "knn":
        return dict(bytes=12.0 * c["nq"] + 8.0 * c["nq"] * c["k"] + 16.0 * 60 * c["nq"], flops=8.0 * 60 * c["nq"])
    if k == "mc":
        g = c["rx"] * c["ry"] * c["rz"]
        return dict(bytes=4.0 * g + (60.0 if c["tris"] else 24.0) * 4.0 * g ** (2 / 3), flops=8.0 * g)
    mac = 48 * 128 + 128 * 128 + 128 * 3
    if k == "train":
        return dict(bytes=108.0 * c["batch"] + 4.0 * 2 * mac, flops=2.0 * (3 * mac - 48 * 128) * c["batch"])
    if k == "init":
        return dict(bytes=24.0 * c["n"], flops=2.0 * mac * c["n"] + 8.0 * 60 * c["n"])
    g = c["reso"] ** 3
    return dict(bytes=(c["iters"] + 1) * (8.0 * g + 64.0 * c["n"]),
                flops=(c["iters"] + 1) * 27.0 * (g + c["n"]) * _terms(c["n"]))


# ---------------------------------------------------------------------------
# 64-bit values
# ---------------------------------------------------------------------------
def _pair(d, b, s, kind):
    """term and gradient factor of offsets d = p − q with b = A·n, screening
    radius s (None: plain): w, and c with ∇w = c·d − g·b; returns (w, g, c)"""
    sigma = kind
    r2 = d.square().sum(-1)
    r = r2.sqrt()
    dot = (d * b).sum(-1)
    if sigma is None:
        den = 4 * math.pi * r2 * r + EPS_PLAIN
        g = 1 / den
        return dot * g, g, 3 * 4 * math.pi * r * dot * g * g
    rho = r.clamp_min(s)
    e = torch.exp(sigma * rho) * 4 * math.pi
    den = e * rho ** 3 + EPS_SCREENED
    g = (sigma * rho + 1) / den
    gp = (sigma * EPS_SCREENED - e * rho ** 2 * (sigma ** 2 * rho ** 2 + 3 * sigma * rho + 3)) / den ** 2
    ok = r > 1e-10
    cc = torch.where(ok & (r >= s), -dot * gp / r.clamp_min(1e-300), torch.zeros_like(r))
    z = torch.zeros_like(r)
    return torch.where(ok, g * dot, z), torch.where(ok, g, z), cc


def _exact_direct(c, p, nrm, q):
    sigma = c["sigma"] if c["screened"] else None
    P, B, Q = p.double(), nrm.double() * float(np.float32(AREA)), q.double()
    s = float(np.float32(SCREEN))
    w = torch.zeros(Q.shape[0], dtype=F64, device="cuda")
    G = torch.zeros(Q.shape[0], 3, dtype=F64, device="cuda")
    step = max(1, int(2e7) // P.shape[0])
    for a in range(0, Q.shape[0], step):
        d = P[None] - Q[a:a + step, None]
        t, g, cc = _pair(d, B[None], s, sigma)
        w[a:a + step] = t.sum(1)
        if c["grad"]:
            G[a:a + step] = (cc[..., None] * d - g[..., None] * B[None]).sum(1)
    return (w, G) if c["grad"] else w


def _exact_octree(p):
    """octreeDWG's split rule (split while > 1 point and above the depth limit):
    per level, the nodes' first and last point, children and moments"""
    P = p.double()
    lo, hi = P.amin(0), P.amax(0)
    c = ((lo + hi) / 2).expand_as(P).clone()
    w = float((hi - lo).max())
    code = torch.zeros(P.shape[0], dtype=torch.int64, device="cuda")
    for _ in range(MAX_DEPTH):
        o = P >= c
        code = code * 8 + (o * torch.tensor([1, 2, 4], device="cuda")).sum(1)
        c += torch.where(o, w / 4, -w / 4)
        w /= 2
    order = torch.argsort(code, stable=True)
    code = code[order]
    levels, live = [], torch.ones_like(code, dtype=torch.bool)  # live: the point's node of this level exists
    for d in range(MAX_DEPTH + 1):
        pre = code >> (3 * (MAX_DEPTH - d))
        key, inv, cnt = torch.unique_consecutive(pre, return_inverse=True, return_counts=True)
        end = cnt.cumsum(0)
        levels.append(dict(key=key, inv=inv, cnt=cnt, begin=end - cnt, live=live.clone()))
        live = live & (cnt[inv] > 1)
    return order, levels


def _exact_tree(c, p, nrm, q):
    """the Barnes-Hut sums of the same term sets: a breadth-first walk of all
    (query, node) pairs"""
    sigma = c["sigma"] if c["screened"] else None
    order, levels = _exact_octree(p)
    P = p.double()[order]
    B = (nrm.double() * float(np.float32(AREA)))[order]
    for L in levels:
        m = L["key"].numel()
        cm = torch.zeros(m, 3, dtype=F64, device="cuda").index_add_(0, L["inv"], P) / L["cnt"][:, None]
        L["ec"] = torch.zeros(m, 3, dtype=F64, device="cuda").index_add_(0, L["inv"], B)
        r = torch.zeros(m, dtype=F64, device="cuda").scatter_reduce_(0, L["inv"], (P - cm[L["inv"]]).norm(dim=1), "amax")
        L["cm"] = cm
        L["far"] = (float(np.float32(BETA)) * r.float()).square().double()  # (β·R)² as the walk rounds it
    s = float(np.float32(SCREEN))
    Q = q.double()
    w = torch.zeros(Q.shape[0], dtype=F64, device="cuda")
    G = torch.zeros(Q.shape[0], 3, dtype=F64, device="cuda")

    def add(iq, d, b):
        for a in range(0, iq.numel(), 1 << 23):
            t, g, cc = _pair(d[a:a + (1 << 23)], b[a:a + (1 << 23)], s, sigma)
            w.index_add_(0, iq[a:a + (1 << 23)], t)
            if c.get("grad"):
                G.index_add_(0, iq[a:a + (1 << 23)], cc[:, None] * d[a:a + (1 << 23)] - g[:, None] * b[a:a + (1 << 23)])

    for a in range(0, Q.shape[0], 1 << 18):
        qc = Q[a:a + (1 << 18)]
        iq = torch.arange(qc.shape[0], device="cuda")
        nd = torch.zeros_like(iq)
        for lv, L in enumerate(levels):
            if iq.numel() == 0:
                break
            single = L["cnt"][nd] == 1
            d32 = (L["cm"].float()[nd].double() - qc[iq])
            # a leaf of several points is never far
            far = (d32.square().sum(1) > L["far"][nd]) & ~single & (lv < MAX_DEPTH)
            i1 = L["begin"][nd[single]]
            add(a + iq[single], P[i1] - qc[iq[single]], B[i1])
            add(a + iq[far], L["cm"][nd[far]] - qc[iq[far]], L["ec"][nd[far]])
            opn = ~single & ~far
            iq, nd = iq[opn], nd[opn]
            if lv == MAX_DEPTH:  # leaves of several points
                n = L["cnt"][nd]
                rep = torch.repeat_interleave(torch.arange(nd.numel(), device="cuda"), n)
                j = L["begin"][nd][rep] + torch.arange(rep.numel(), device="cuda") - (n.cumsum(0) - n)[rep]
                add(a + iq[rep], P[j] - qc[iq[rep]], B[j])
                break
            nxt = levels[lv + 1]  # the children of each open node: a run of the next level's keys
            kb = torch.searchsorted(nxt["key"], L["key"][nd] * 8)
            ke = torch.searchsorted(nxt["key"], L["key"][nd] * 8 + 8)
            n = ke - kb
            rep = torch.repeat_interleave(torch.arange(nd.numel(), device="cuda"), n)
            nd = kb[rep] + torch.arange(rep.numel(), device="cuda") - (n.cumsum(0) - n)[rep]
            iq = iq[rep]
    return (w, G) if c.get("grad") else w


def _grid_points(grid):
    r = [grid.res[d] for d in range(3)]
    ax = [(torch.arange(r[d], device="cuda", dtype=F64) * grid.h + grid.origin[d]).float() for d in range(3)]
    z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    return torch.stack([x, y, z], -1).reshape(-1, 3)


def _knn64(p, q, k):
    """k nearest points of each query: (indices, squared distances) in 64 bits"""
    P, Q = p.double(), q.double()
    idx, dd = [], []
    step = max(1, int(1.5e8) // P.shape[0])
    for a in range(0, Q.shape[0], step):
        d2 = torch.zeros(min(step, Q.shape[0] - a), P.shape[0], dtype=F64, device="cuda")
        for d in range(3):
            d2 += (Q[a:a + step, d, None] - P[None, :, d]).square_()
        v, i = d2.topk(min(k, P.shape[0]), dim=1, largest=False, sorted=True)
        idx.append(i)
        dd.append(v)
    return torch.cat(idx), torch.cat(dd)


def _exact_diffuse(p, nrm, cent, tn):
    n = p.shape[0]
    acc = torch.zeros(n, 3, dtype=F64, device="cuda")
    i, _ = _knn64(p, cent, 15)
    acc.index_add_(0, i.reshape(-1), tn.double().repeat_interleave(i.shape[1], 0))
    length = acc.norm(dim=1)
    zero = length < 1e-10
    out = torch.where(zero[:, None], nrm.double(), acc / (length[:, None] + 1e-8))
    if int(zero.sum()) > 10:
        have = torch.nonzero(~zero)[:, 0]
        j, _ = _knn64(p[have], p[zero], 10)
        v = out[have][j].sum(1)
        out[zero] = v / (v.norm(dim=1, keepdim=True) + 1e-8)
    return out, None


def _params(net):
    t = torch.from_numpy(net.params()).to("cuda").double()
    out, at = [], 0
    for shape in ((128, 48), (128,), (128, 128), (128,), (3, 128), (3,)):
        m = math.prod(shape)
        out.append(t[at:at + m].reshape(shape).clone().requires_grad_(True))
        at += m
    return out


def _mlp64(w, x):
    gelu = torch.nn.functional.gelu
    h = gelu(x @ w[0].T + w[1], approximate="tanh")
    h = gelu(h @ w[2].T + w[3], approximate="tanh")
    return h @ w[4].T + w[5]


def exact(case, seed):
    k = case["kind"]
    if k in ("mc", "recon"):
        return None
    if k == "train":
        s = prepare(case, seed)
        w = _params(s["net"])
        y = _mlp64(w, s["x"].view(torch.bfloat16).double())
        cos = ((y / (y.norm(dim=1, keepdim=True) + 1e-12)) * s["t"].double()).sum(1)
        loss = (1 - cos * cos if case["line"] else 1 - cos).mean()
        loss.backward()
        return torch.cat([v.grad.reshape(-1) for v in w]).cpu().numpy(), float(loss)
    p, nrm, g = _cloud(case["n"], seed)
    if k == "grid":
        if case["rx"] * case["ry"] * case["rz"] > 4_000_000:
            return None
        return _exact_tree(case, p, nrm, _grid_points(_grid(p, (case["rx"], case["ry"], case["rz"]))))
    if k == "points":
        return _exact_tree(case, p, nrm, _queries(p, case["nq"], g))
    if k == "direct":
        if case["n"] * case["nq"] > 3e10:
            return None
        return _exact_direct(case, p, nrm, _queries(p, case["nq"], g))
    if k == "diffuse":
        if case["n"] * case["ncent"] > 3e9:
            return None
        return _exact_diffuse(p, nrm, *_centroids(p, nrm, case["ncent"], case["far"], g))
    if k == "knn":
        _, d2 = _knn64(p, _queries(p, case["nq"], g), case["k"])
        return None, d2
    if case["n"] > 50_000:  # larger clouds take their patches from a subsample
        return None
    i, d2 = _knn64(p, p, 17)
    off = p.double()[i[:, 1:]] - p.double()[:, None]
    off = off / d2[:, 16:17, None].sqrt()
    net = gpu.Mlp(_ctx(), path=WEIGHTS)
    with torch.no_grad():
        y = _unit(_mlp64(_params(net), off.reshape(-1, 48)))
    ctr = torch.tensor([float(v) for v in (p.amax(0) + p.amin(0)).cpu() / 2], dtype=F64, device="cuda")
    side = (y * (p.double() - ctr)).sum(1, keepdim=True)
    return torch.where(side < 0, -y, y)

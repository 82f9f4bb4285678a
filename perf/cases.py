"""The work a refinement driver has this library do, as a dozen timed cases.

Each case is a dict of plain values; prepare() makes its inputs on the GPU from
the seed, run() is one pass through the entry points of tetwild_amd.ops, as a
driver calls them.  The kinds:

  amips     per-tet energy, gradient, Hessian (amips_eval, amips_eval_mixed)
  quality   calTetQualities over a mesh or a one-ring (tet_qualities)
  flip      isFlip over a mesh (tet_flip)
  faces     isFaceOutEnvelop of query triangles (envelope_faces)
  points    isPointOutEnvelop of query points (envelope_points)
  smooth    one-ring Newton smoothing (SmoothBatch, SmoothPlan)
  collapse  edge-collapse candidates (CollapseBatch, CollapsePlan)
  groups    edge-removal configurations (tet_groups)
  stats     pass-terminating energy reductions (energy_stats)
  tree      the envelope tree of an input surface and its first queries
"""
import functools
import math

import numpy as np
import torch

from tetwild_amd import _capi as C
from tetwild_amd import workloads as W
from tetwild_amd.ops import CollapseBatch, Context, SmoothBatch

DEV = "cuda:0"
PREC = {"fp64": C.TWG_FP64, "mixed": C.TWG_MIXED}


def listed():
    return [
        # a whole 10.1M-tet mesh: energies, gradients and Hessians of a global pass
        {"name": "amips_mesh", "kind": "amips", "tets": "lattice", "size": 119,
         "precision": "fp64", "mode": 2},
        # a mesh's worst tets (aspect ratio to 1e4) in mixed precision, where
        # part of them falls back to FP64
        {"name": "amips_slivers_mixed", "kind": "amips", "tets": "slivers", "size": 600_000,
         "precision": "mixed", "mode": 2},
        # calTetQualities of a 1.3M-tet mesh, once per operator pass
        {"name": "quality_mesh", "kind": "quality", "size": 60, "precision": "fp64"},
        # every surface face of a large mesh against its envelope
        {"name": "faces_large", "kind": "faces", "n": 3_000_000, "freq": 111, "edge": 2.0,
         "precision": "fp64"},
        # the faces of one vertex's one-ring, the test of a single operation: faces
        # as long as the input's facets, a few hundred samples each
        {"name": "faces_one_ring", "kind": "faces", "n": 12, "freq": 16, "edge": 40.0,
         "precision": "fp64"},
        # boundary points near the envelope's limit, about four per facet
        {"name": "points_mixed", "kind": "points", "n": 1_000_001, "freq": 111,
         "precision": "mixed"},
        # one smoothing pass over a mesh's independent vertices, replayed as a graph
        {"name": "smooth_pass", "kind": "smooth", "n": 60_000, "freq": 111, "surface": 0.2,
         "precision": "fp64", "tile": C.TWG_SMOOTH_TILE_SPLIT, "chunk": 4, "plan": True},
        # one dependency level of the index-order pass: about forty vertices a call
        {"name": "smooth_level", "kind": "smooth", "n": 40, "freq": 16, "surface": 0.25,
         "precision": "fp64", "tile": C.TWG_SMOOTH_TILE_SPLIT, "chunk": 1, "plan": False},
        # the collapse candidates of a mesh with an embedded sheet
        {"name": "collapse_pass", "kind": "collapse", "cubes": 40, "n": 200_000,
         "precision": "fp64", "plan": True},
        # every configuration of the removable edges of a pass, groups of 2 to 6 tets
        {"name": "groups_pass", "kind": "groups", "n": 150_000, "size": 30},
        # the reductions that end a pass, over a 3.1M-tet mesh with locks
        {"name": "stats_mesh", "kind": "stats", "size": 80, "locks": True},
        # the tree of a 246k-facet input surface and its first point queries
        {"name": "tree_build", "kind": "tree", "freq": 111, "n": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["amips", "amips", "quality", "flip", "faces", "faces", "faces", "points",
                       "points", "smooth", "smooth", "collapse", "groups", "stats", "tree"])
    prec = rng.choice(["fp64", "mixed"])
    if kind == "amips":
        if rng.random() < 0.5:
            return {"kind": kind, "tets": "lattice", "size": _log(rng, 2, 110), "precision": prec,
                    "mode": rng.randrange(4)}
        return {"kind": kind, "tets": "slivers", "size": _log(rng, 24, 2_000_000),
                "precision": prec, "mode": rng.randrange(4)}
    if kind == "quality":
        return {"kind": kind, "size": _log(rng, 2, 110), "precision": prec}
    if kind == "flip":
        return {"kind": kind, "size": _log(rng, 4, 110)}
    if kind == "faces":
        n = _log(rng, 32, 3_000_000)
        edge = rng.uniform(1.5, 4.0) if n > 50_000 else rng.uniform(2.0, 40.0)
        return {"kind": kind, "n": n, "freq": _log(rng, 8, 160), "edge": round(edge, 3),
                "precision": prec}
    if kind == "points":
        return {"kind": kind, "n": _log(rng, 64, 4_000_000), "freq": _log(rng, 8, 160),
                "precision": prec}
    if kind == "smooth":
        return {"kind": kind, "n": _log(rng, 1, 60_000), "freq": _log(rng, 16, 160),
                "surface": round(rng.uniform(0.0, 0.5), 3), "precision": prec,
                "tile": rng.choice([0, 16, 32, 64, C.TWG_SMOOTH_TILE_SPLIT]),
                "chunk": rng.choice([0, 1, 4]), "plan": rng.random() < 0.5}
    if kind == "collapse":
        cubes = _log(rng, 4, 40)
        return {"kind": kind, "cubes": cubes, "n": min(_log(rng, 8, 200_000), 40 * cubes ** 3),
                "precision": prec, "plan": rng.random() < 0.5}
    if kind == "groups":
        return {"kind": kind, "n": _log(rng, 4, 600_000), "size": _log(rng, 4, 60)}
    if kind == "stats":
        return {"kind": kind, "size": _log(rng, 2, 110), "locks": rng.random() < 0.5}
    return {"kind": kind, "freq": _log(rng, 4, 160), "n": _log(rng, 16, 16384)}


# ------------------------------------------------------------------ inputs --
@functools.lru_cache(maxsize=None)
def _ctx():
    return Context(0)  # a driver keeps one


@functools.lru_cache(maxsize=4)
def _sphere(freq):
    return W.geodesic_sphere(freq)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float64)


def _surface(freq, seed):
    """a geodesic sphere of 20 freq^2 facets with smooth random bumps"""
    V, F = _sphere(freq)
    r = np.random.default_rng(seed)
    k = r.normal(size=(6, 3)) * 3.0
    ph = r.uniform(0, 2 * np.pi, 6)
    bump = 0.02 * np.sin(V @ k.T + ph).sum(1)
    return np.ascontiguousarray(V * (1.0 + bump)[:, None]), F


def _surface_points(V, F, n, g):
    """n points uniform by area on the surface, and the facets' unit normals there"""
    v = torch.from_numpy(V).to(DEV)
    T = v[torch.from_numpy(F.astype(np.int64)).to(DEV)]
    N = torch.linalg.cross(T[:, 1] - T[:, 0], T[:, 2] - T[:, 0])
    area = N.norm(dim=1)
    cdf = torch.cumsum(area, 0)
    f = torch.searchsorted(cdf, _rand(g, n) * cdf[-1]).clamp_(max=len(F) - 1)
    s, t = _rand(g, n).sqrt(), _rand(g, n)
    b = torch.stack([1 - s, s * (1 - t), s * t], 1)
    P = (T[f] * b[:, :, None]).sum(1)
    return P, N[f] / area[f][:, None]


def _triangles(V, F, n, eps, edge, g):
    """near-equilateral triangles of edge length `edge` in the facets' planes,
    offset along the normal by up to 2 eps either way"""
    P, N = _surface_points(V, F, n, g)
    a = torch.zeros_like(N)
    a[:, 0] = (N[:, 0].abs() < 0.9).double()
    a[:, 1] = 1 - a[:, 0]
    t1 = torch.linalg.cross(N, a)
    t1 = t1 / t1.norm(dim=1, keepdim=True)
    t2 = torch.linalg.cross(N, t1)
    ang = _rand(g, n) * (2 * math.pi)
    rad = edge * (1 + (2 * _rand(g, n) - 1) * 0.1) / math.sqrt(3)
    P = P + ((2 * _rand(g, n) - 1) * 2 * eps)[:, None] * N
    out = torch.empty(n, 9, dtype=torch.float64, device=DEV)
    for j in range(3):
        th = ang + j * (2 * math.pi / 3)
        out[:, 3 * j:3 * j + 3] = P + rad[:, None] * (th.cos()[:, None] * t1 + th.sin()[:, None] * t2)
    return out


def _lattice(c, seed):
    """a jittered Kuhn lattice of c^3 cubes, six positive tets each"""
    g = _gen(seed)
    n1 = c + 1
    h = 1.0 / c
    i = torch.arange(n1, device=DEV, dtype=torch.float64) * h
    z, y, x = torch.meshgrid(i, i, i, indexing="ij")
    xyz = [a.reshape(-1) + _randn(g, n1 ** 3) * (0.12 * h) for a in (x, y, z)]
    k = torch.arange(c, device=DEV)
    kk, jj, ii = torch.meshgrid(k, k, k, indexing="ij")
    base = (ii + n1 * (jj + n1 * kk)).reshape(-1)
    step = (1, n1, n1 * n1)
    tets = torch.empty(c ** 3, 6, 4, dtype=torch.int64, device=DEV)
    for t, p in enumerate(((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0))):
        tets[:, t, 0] = base
        tets[:, t, 1] = base + step[p[0]]
        tets[:, t, 2] = base + step[p[0]] + step[p[1]]
        tets[:, t, 3] = base + sum(step)
    tets = tets.reshape(-1, 4)
    return xyz, _oriented(tets, xyz)


def _det(tets, xyz):
    p = torch.stack([torch.stack([a[tets[:, j].long()] for a in xyz], 1) for j in range(4)], 1)
    e = p[:, 1:] - p[:, :1]
    return (e[:, 0] * torch.linalg.cross(e[:, 1], e[:, 2])).sum(1)


def _oriented(tets, xyz):
    bad = _det(tets, xyz) < 0
    swapped = tets[:, [0, 1, 3, 2]]
    return torch.where(bad[:, None], swapped, tets).to(torch.int32).contiguous()


def _slivers(n, seed):
    """separate tets stretched by 10^U[0, 4] along one axis or two"""
    g = _gen(seed)
    a = 10.0 ** (4 * _rand(g, n))
    needle = _rand(g, n) < 0.5
    S = torch.ones(n, 3, dtype=torch.float64, device=DEV)
    S[:, 2] = torch.where(needle, a, 1 / a)
    S[:, 1] = torch.where(needle, a, torch.ones_like(a))
    R = torch.from_numpy(W.REGULAR_TET - W.REGULAR_TET.mean(0)).to(DEV)
    P = R[None] * S[:, None] * 0.01
    q = _randn(g, n, 4)
    q = q / q.norm(dim=1, keepdim=True)
    w, u = q[:, :1, None], q[:, None, 1:].expand(n, 4, 3)
    t = 2 * torch.linalg.cross(u, P)
    P = P + w * t + torch.linalg.cross(u, t) + (2 * _rand(g, n, 1, 3) - 1)
    P = P.reshape(-1, 3)
    xyz = [P[:, k].contiguous() for k in range(3)]
    return xyz, _oriented(torch.arange(4 * n, device=DEV).reshape(n, 4), xyz)


# the envelope of the large surfaces: eps = sampling distance = 1e-3 of the unit sphere
EPS = 1e-3


def prepare(case, seed):
    kind = case["kind"]
    ctx = _ctx()
    s = {"case": case, "ctx": ctx}
    if kind in ("amips", "quality", "flip"):
        make = _slivers if case.get("tets") == "slivers" else _lattice
        s["xyz"], s["tets"] = make(case["size"], seed)
        if kind == "flip":  # a tenth of them inverted by a move
            inv = _rand(_gen(seed + 1), len(s["tets"]), 1) < 0.1
            s["tets"] = torch.where(inv, s["tets"][:, [0, 1, 3, 2]], s["tets"]).contiguous()
        if kind == "amips":  # a driver keeps its output arrays
            n, mode = len(s["tets"]), case["mode"]
            mixed = case["precision"] == "mixed"
            dt = torch.float32 if mixed else torch.float64
            out = [torch.zeros(n, dtype=torch.float64, device=DEV),
                   torch.zeros(n, 3, dtype=dt, device=DEV) if mode >= 1 else None,
                   torch.zeros(n, 6 if mode == C.TWG_AMIPS_EGH_SYM else 9, dtype=dt, device=DEV)
                   if mode >= 2 else None]
            s["out"] = out + [torch.zeros(n, dtype=torch.uint8, device=DEV)] if mixed else out
    elif kind in ("faces", "points", "tree"):
        V, F = _surface(case["freq"], seed)
        g = _gen(seed)
        if kind == "faces":
            s["queries"] = _triangles(V, F, case["n"], EPS, case["edge"] * EPS, g)
        else:  # within a hundredth of eps of the limit, either side of the surface
            P, N = _surface_points(V, F, case["n"], g)
            d = EPS * (1 + 0.01 * (2 * _rand(g, case["n"]) - 1))
            d = torch.where(_rand(g, case["n"]) < 0.5, d, -d)
            s["queries"] = (P + d[:, None] * N).contiguous()
        if kind == "tree":
            s["V"], s["F"] = V, F
        else:
            s["surf"] = ctx.surface(V, F)
    elif kind == "smooth":
        V, F = _surface(case["freq"], seed)
        surf = ctx.surface(V, F)
        # the rings' sizes are the case's, their places and shapes the seed's
        B = W.smoothing_batch(case["n"], seed=1, surface_frac=case["surface"], V=V, F=F)
        r = np.random.default_rng(seed)
        for k in "xyz":
            B[k] = B[k] + 2e-4 * (2 * r.random(len(B[k])) - 1)
        dev = [torch.from_numpy(B[k]).to(DEV) for k in ("ring_tets", "x", "y", "z")]
        q = ctx.tet_qualities(*dev)[0].cpu().numpy()
        s["batch"] = SmoothBatch(ctx, B, sf=surf, bt=surf, eps2=EPS * EPS, sampling_dist=EPS, old_q=q)
        if case["plan"]:
            s["plan"] = s["batch"].plan(PREC[case["precision"]], case["tile"], case["chunk"])
    elif kind == "collapse":
        M = W.sheet_mesh(case["cubes"], seed=seed)
        dev = [torch.from_numpy(M[k]).to(DEV) for k in ("tets", "x", "y", "z")]
        q = ctx.tet_qualities(*dev)[0].cpu().numpy()
        B = W.collapse_batch(M, q, n_cand=case["n"], seed=1)  # the case's edges
        eps = 0.05 / case["cubes"]
        s["batch"] = CollapseBatch(ctx, B, ctx.surface(M["sf_V"], M["sf_F"]),
                                   ctx.surface(M["b_V"], M["b_F"]), eps * eps, eps)
        if case["plan"]:
            s["plan"] = s["batch"].plan(PREC[case["precision"]])
    elif kind == "groups":
        s["xyz"], tets = _lattice(case["size"], seed)
        g = _gen(seed + 1)
        size = torch.randint(2, 7, (case["n"],), generator=_gen(1), device=DEV)
        off = torch.zeros(case["n"] + 1, dtype=torch.int64, device=DEV)
        off[1:] = torch.cumsum(size, 0)
        # a configuration's tets are neighbours: runs of the lattice's order
        first = torch.randint(0, max(1, len(tets) - 6), (case["n"],), generator=g, device=DEV)
        own = torch.repeat_interleave(torch.arange(case["n"], device=DEV), size)
        at = first[own] + torch.arange(len(own), device=DEV) - off[own]
        s["tets"], s["off"] = tets[at].contiguous(), off.to(torch.int32)
    else:  # stats
        xyz, tets = _lattice(case["size"], seed)
        g = _gen(seed + 1)
        s["q"] = ctx.tet_qualities(tets, *xyz)[0]
        s["removed"] = (_rand(g, len(tets)) < 0.05).to(torch.uint8)
        s["tets"] = tets if case["locks"] else None
        s["locked"] = (_rand(g, len(xyz[0])) < 0.01).to(torch.uint8) if case["locks"] else None
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    prec = PREC[case.get("precision", "fp64")]
    if kind == "amips":
        f = ctx.amips_eval_mixed if prec == C.TWG_MIXED else ctx.amips_eval
        return list(f(s["tets"], *s["xyz"], mode=case["mode"], out=s["out"]))
    if kind == "quality":
        return list(ctx.tet_qualities(s["tets"], *s["xyz"], precision=prec)[:2 if prec else 1])
    if kind == "flip":
        return ctx.tet_flip(s["tets"], *s["xyz"])
    if kind == "faces":
        return ctx.envelope_faces(s["surf"], s["queries"], EPS * EPS, EPS, precision=prec)
    if kind == "points":
        return ctx.envelope_points(s["surf"], s["queries"], EPS * EPS, precision=prec)
    if kind in ("smooth", "collapse"):
        if "plan" in s:
            return list(s["plan"].run())
        return list(s["batch"].run(prec, case.get("tile", 0), case.get("chunk", 0)))
    if kind == "groups":
        return list(ctx.tet_groups(s["tets"], s["off"], *s["xyz"]))
    if kind == "stats":
        return list(ctx.energy_stats(s["q"], s["removed"], s["tets"], s["locked"]))
    s["surf"] = ctx.surface(s["V"], s["F"])
    out = ctx.envelope_points(s["surf"], s["queries"], EPS * EPS)
    near = ctx.nearest(s["surf"], s["queries"])
    return [s["surf"].order(), s["surf"].nnode, s["surf"].depth, s["surf"].rmax, out, *near]


def work(case):
    """Bytes: each input and output once.  Flops: 164 per tet's energy, gradient
    and Hessian, 86 per energy, 34 per orientation, 60 per point-triangle
    distance (one per sample of an inside triangle, one per point)."""
    kind = case["kind"]
    if kind in ("amips", "quality", "flip", "stats"):
        c = case["size"]
        sl = case.get("tets") == "slivers"
        n, nv = (c, 4 * c) if sl else (6 * c ** 3, (c + 1) ** 3)
        if kind == "amips":
            w = 4 if case["precision"] == "mixed" else 8
            rows = (0, 3, 12, 9)[case["mode"]]
            b = 16 + 8 + w * rows + (1 if w == 4 else 0)
            return {"bytes": n * b + 24 * nv, "flops": n * (86, 118, 164, 164)[case["mode"]]}
        if kind == "quality":
            return {"bytes": n * 25 + 24 * nv, "flops": n * 120}
        if kind == "flip":
            return {"bytes": n * 17 + 24 * nv, "flops": n * 34}
        return {"bytes": n * (25 if case["locks"] else 9) + (nv if case["locks"] else 0), "flops": n}
    if kind == "groups":
        nv = (case["size"] + 1) ** 3
        return {"bytes": case["n"] * (4 * 24 + 4 + 9) + 24 * min(nv, 16 * case["n"]),
                "flops": case["n"] * 4 * 120}
    if kind in ("faces", "points", "tree"):
        nf = 20 * case["freq"] ** 2
        if kind == "tree":  # facets and vertices in; boxes, triangles and order out
            return {"bytes": nf * (12 + 12 + 128 + 72 + 12 + 4) + case["n"] * 61, "flops": nf * 40}
        near = min(nf, 8 * case["n"])  # facets a query can meet
        if kind == "points":
            return {"bytes": case["n"] * 25 + near * 72, "flops": case["n"] * 60}
        e = case["edge"]
        samples = 3 + 2 * e + e * e / 2  # corners, edges, the lattice inside
        return {"bytes": case["n"] * 73 + near * 72, "flops": case["n"] * 0.5 * samples * 60}
    if kind == "smooth":
        n, ring = case["n"], 29
        return {"bytes": n * (ring * (16 + 8 + 8 + 12) + 24 + 2 + 4),
                "flops": n * ring * 4 * (164 + 86 + 34)}
    n, ring = case["n"], 24  # collapse
    return {"bytes": n * (ring * (16 + 8 + 8) + 10) + 24 * (case["cubes"] + 1) ** 3,
            "flops": n * ring * 120}


def tolerance(case):
    """About four times what the library shows against exact()."""
    kind = case["kind"]
    if kind == "amips":
        # the worst tets' determinants lose digits; mixed holds gradient and
        # Hessian in FP32 and certifies the energy to 2^-16
        if case["precision"] == "mixed":
            return {"rel": 6e-7, "max": 1e-5, "differ": 1e-4}
        return {"rel": 3e-12, "max": 2e-11}
    if kind == "quality":
        if case["precision"] == "mixed":
            return {"rel": 6e-7, "max": 4e-6, "differ": 1e-4}
        return {"rel": 1e-14, "max": 2e-13}
    if kind == "groups":
        return {"rel": 2e-15, "max": 2e-14}
    if kind == "stats":
        return {"rel": 1e-13, "max": 1e-13}
    if kind in ("smooth", "collapse"):
        # a ring sum in another order can turn a line-search step near convergence
        return {"rel": 1e-9, "max": 1e-6, "differ": 1e-4}
    if kind == "tree":
        return {"rel": 1e-13, "max": 1e-12}
    return "exact"  # decisions


# ---------------------------------------------------------- 64-bit results --
def _energies(tets, xyz, mode):
    """E = |M|^2 / |det M|^(2/3) with M the map from the regular tet, and its
    derivatives with respect to vertex 0, from their definition"""
    if len(tets) > 1 << 20:  # in parts: a dozen 3 x 3 intermediates per tet
        parts = [_energies(t, xyz, mode) for t in tets.split(1 << 20)]
        return [torch.cat(v) if v[0] is not None else None for v in zip(*parts)]
    R = W.REGULAR_TET
    Wt = torch.from_numpy(np.linalg.inv((R[1:] - R[:1]).T)).to(xyz[0])
    p = torch.stack([torch.stack([a[tets[:, j].long()] for a in xyz], 1) for j in range(4)], 2)
    M = ((p[:, :, 1:] - p[:, :, :1])[:, :, :, None] * Wt).sum(2)
    S = (M * M).sum((1, 2))
    x, y, z = M[:, :, 0], M[:, :, 1], M[:, :, 2]
    cof = torch.stack([torch.linalg.cross(y, z), torch.linalg.cross(z, x), torch.linalg.cross(x, y)], 2)
    d = (x * cof[:, :, 0]).sum(1)
    k = (d * d) ** (-1.0 / 3.0)
    E = S * k
    if mode == 0:
        return [E, None, None]
    c0 = -Wt.sum(0)
    u = 2 * (M * c0).sum(2)
    n = (cof * c0).sum(2) / d[:, None]
    G = k[:, None] * (u - (2.0 / 3.0) * S[:, None] * n)
    if mode == 1:
        return [E, G, None]
    un = u[:, :, None] * n[:, None, :]
    H = 2 * float(c0 @ c0) * torch.eye(3, dtype=E.dtype, device=E.device) \
        - (2.0 / 3.0) * (un + un.transpose(1, 2)) \
        + (10.0 / 9.0) * S[:, None, None] * (n[:, :, None] * n[:, None, :])
    H = (k[:, None, None] * H).reshape(-1, 9)
    return [E, G, H[:, [0, 1, 2, 4, 5, 8]] if mode == C.TWG_AMIPS_EGH_SYM else H]


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("amips", "quality", "groups", "stats"):
        return None  # decisions, and iterations that end on them
    s = prepare(case, seed)
    if kind == "amips":
        return _energies(s["tets"], s["xyz"], case["mode"]) + [None]
    if kind == "quality":
        return [_energies(s["tets"], s["xyz"], 0)[0], None]
    if kind == "groups":
        q = _energies(s["tets"], s["xyz"], 0)[0]
        off = s["off"].long()
        own = torch.repeat_interleave(torch.arange(case["n"], device=DEV), off[1:] - off[:-1])
        m = torch.zeros(case["n"], dtype=q.dtype, device=DEV).scatter_reduce(0, own, q, "amax")
        return [None, m, q]
    q, keep = s["q"], s["removed"] == 0
    free = keep
    if case["locks"]:
        free = keep & ~(s["locked"].bool()[s["tets"].long()].any(1))
    v = q[free].cpu().numpy()
    return [math.fsum(v), float(v.max()) if len(v) else 0.0, None, None, None]

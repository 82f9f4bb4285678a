"""The query order and the list kernels' edges: batches around a sort tile, the
two- and three-pass sorts, clustered and degenerate boxes, and waves whose
facets overflow their list, each against the per-query tree walk (the
statistics path, whose decisions the other tests pin to the oracle)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65536, 65537, 4096 * 17 - 1, (1 << 18) - 1, 1 << 18, 300001])
@pytest.mark.parametrize("where", ["spread", "cluster", "one_place"])
def test_sorted_batches(n, where):
    import torch

    from tetwild_amd import workloads as W
    from tetwild_amd.ops import Context
    ctx = Context(0)
    V, F = W.bumpy_sphere(freq=24, seed=2)
    surf = ctx.surface(V, F)
    eps = 2e-3
    Q = W.query_triangles(V, F, n, eps=eps, edge=0.004, seed=n % 7)
    if where != "spread":  # about one facet, the last items far away and not finite
        c = V[F[5]].mean(0)
        Q = c + (Q.reshape(n, 3, 3) * (0.02 if where == "cluster" else 0.0)).reshape(n, 3, 3)
        if where == "one_place":
            Q = Q + np.array([[0, 0, 0], [0.004, 0, 0], [0, 0.004, 0.001]])
        Q[-3:-1] += 1e6
        Q = np.ascontiguousarray(Q.reshape(n, 9))
        Q[-1, 4] = np.inf
    tq = torch.from_numpy(Q).to("cuda:0")
    for prec in (0, 1):
        out = ctx.envelope_faces(surf, tq, eps * eps, eps, precision=prec)
        walk, _ = ctx.envelope_faces(surf, tq, eps * eps, eps, precision=prec, stats=True)
        assert torch.equal(out, walk), (prec, int((out != walk).sum()))
        p3 = tq[:, :3].contiguous()
        pout = ctx.envelope_points(surf, p3, eps * eps, precision=prec)
        pwalk, _ = ctx.envelope_points(surf, p3, eps * eps, precision=prec, stats=True)
        assert torch.equal(pout, pwalk), prec
    ctx.close()


@pytest.mark.parametrize("eps,edge", [(1e-3, 0.03), (0.05, 0.02), (1e-9, 1e-7), (0.0, 0.004)])
def test_lists_overflow_and_limits(eps, edge):
    """Dense facets under wide queries (every list overflows), an envelope wider
    than the facets, one far below the coordinates' rounding, and eps = 0"""
    import torch

    from tetwild_amd import workloads as W
    from tetwild_amd.ops import Context
    ctx = Context(0)
    V, F = W.bumpy_sphere(freq=40, seed=3)
    surf = ctx.surface(V, F)
    d = max(eps, 1e-9) if edge < 1e-3 else max(eps, 2e-3)
    Q = W.query_triangles(V, F, 70000, eps=eps, edge=edge, seed=5)
    for nf in (len(F), 700):  # 2.2 and 100 queries a facet
        s = surf if nf == len(F) else ctx.surface(V, F[:nf])
        tq = torch.from_numpy(Q).to("cuda:0")
        for prec in (0, 1):
            out = ctx.envelope_faces(s, tq, eps * eps, d, precision=prec)
            walk, _ = ctx.envelope_faces(s, tq, eps * eps, d, precision=prec, stats=True)
            assert torch.equal(out, walk), (nf, prec, int((out != walk).sum()))
            p3 = tq[:, :3].contiguous()
            assert torch.equal(ctx.envelope_points(s, p3, eps * eps, precision=prec),
                               ctx.envelope_points(s, p3, eps * eps, precision=prec, stats=True)[0])
        small = tq[:200].contiguous()  # a wave per triangle
        o = ctx.envelope_faces(s, small, eps * eps, d)
        assert torch.equal(o, ctx.envelope_faces(s, small, eps * eps, d, stats=True)[0])
    ctx.close()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 32767, 32768, 65535])
@pytest.mark.parametrize("reach", ["near", "far", "wide"])
def test_small_points_and_nearest(n, reach):
    """Lanes-per-point kernels: the decision and the nearest facet of every
    point, where groups decide, where their lists overflow (an envelope wider
    than the list holds) and where they cannot be sure (far points, ties on a
    flat grid), NaN and infinite points among them, against the oracle"""
    import torch

    from oracle import oracle as O
    from tetwild_amd import workloads as W
    from tetwild_amd.ops import Context
    ctx = Context(0)
    V, F = W.bumpy_sphere(freq=12, seed=3)
    if reach == "far":  # a flat grid: ties above its edges and corners
        g = np.arange(20.0)
        V = np.stack(np.meshgrid(g, g, [0.0], indexing="ij"), -1).reshape(-1, 3)
        q = (np.arange(19)[:, None] * 20 + np.arange(19)).reshape(-1)
        F = np.concatenate([np.stack([q, q + 20, q + 1], 1), np.stack([q + 1, q + 20, q + 21], 1)]).astype(np.int32)
    r = np.random.default_rng(n)
    k = min(n, 3000)  # distinct points, repeated over the batch
    P = V[r.integers(0, len(V), k)] + r.normal(size=(k, 3)) * (0.02 if reach != "far" else 0.0)
    if reach == "far":
        P[:, 2] += r.uniform(0, 5, k) * (np.arange(k) % 3)
    eps = 0.4 if reach == "wide" else 0.02
    surf = ctx.surface(V, F)
    S = O.Surface(V, F[surf.order()])
    cp, d2, fid = S.nearest(P)
    at = np.arange(n) % k
    Q = np.ascontiguousarray(P[at])
    tq = torch.from_numpy(Q).to("cuda:0")
    for prec in (0, 1):
        out = ctx.envelope_points(surf, tq, eps * eps, precision=prec).cpu().numpy()
        assert np.array_equal(out, S.point_out(P, eps * eps)[at]), prec
    gcp, gd2, gf = (t.cpu().numpy() for t in ctx.nearest(surf, tq))
    assert np.array_equal(gcp, cp[at]) and np.array_equal(gd2, d2[at]) and np.array_equal(gf, fid[at])
    if n > 16:
        Q[3], Q[7, 1] = np.nan, np.inf
        tq = torch.from_numpy(Q).to("cuda:0")
        out = ctx.envelope_points(surf, tq, eps * eps)
        assert torch.equal(out, ctx.envelope_points(surf, tq, eps * eps, stats=True)[0])
    ctx.close()


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 95, 96, 97, 140])
def test_rows_per_wave(rows):
    """Triangles of about `rows` sample rows, a wave each: the row table's one
    and two rounds, its last rows and the sampler beyond it; needles and short
    triangles among them, against the oracle"""
    import torch

    from oracle import oracle as O
    from tetwild_amd import workloads as W
    from tetwild_amd.ops import Context
    ctx = Context(0)
    V, F = W.bumpy_sphere(freq=6, seed=3)
    V = V * 4.0
    d, eps = 0.01, 0.012
    surf = ctx.surface(V, F)
    S = O.Surface(V, F[surf.order()])
    Q = W.query_triangles(V, F, 40, eps=eps, edge=(rows + 0.5) * d * 0.75 ** 0.5 / 0.75, seed=rows)
    Q = Q.reshape(-1, 3, 3)
    # in the plane of a facet, within the envelope: every sample is tested
    T = V[F[:10]]
    c = T.mean(1, keepdims=True)
    size = np.linalg.norm(T - c, axis=2).min(1)
    flat = c + (T - c) * (rows * d / (1.5 * size))[:, None, None]
    needle = flat.copy()
    needle[:, 2] = needle[:, 0] + 0.5 * (needle[:, 1] - needle[:, 0]) + 0.01 * (needle[:, 2] - needle[:, 0])
    short = c + (T - c) * (0.4 * d / size)[:, None, None]
    Q = np.ascontiguousarray(np.concatenate([Q, flat, needle, short]).reshape(-1, 9))
    ref, _ = S.face_out(Q, eps * eps, d)
    assert 0 < ref.sum() < len(ref)
    for prec in (0, 1):
        out = ctx.envelope_faces(surf, torch.from_numpy(Q).to("cuda:0"), eps * eps, d, precision=prec)
        assert np.array_equal(out.cpu().numpy(), ref), prec
    ctx.close()


@pytest.mark.parametrize("what", ["faces", "sparse_faces", "points", "nearest"])
def test_captured_batch_outlives_larger_calls(what):
    """A captured batch keeps its ordering and queue memory when larger eager
    calls on the context outgrow it: replays between such calls, each against
    the eager result, on inputs that change in place"""
    import torch

    from tetwild_amd import workloads as W
    from tetwild_amd.ops import Context
    ctx = Context(0)
    V, F = W.bumpy_sphere(freq=70 if what == "sparse_faces" else 24, seed=2)
    surf = ctx.surface(V, F)
    eps, n = 2e-3, 70001
    sets = [torch.from_numpy(W.query_triangles(V, F, n, eps=eps, edge=0.004, seed=s)).to("cuda:0") for s in (1, 2, 3)]
    for t in sets:
        t[5, 3:6] = t[5, 0:3]  # degenerate: the queue is used
    more = sets[0].repeat(4, 1)
    q = sets[0].clone()
    p3 = q[:, :3].contiguous()
    big3 = more[:, :3].contiguous()
    if what == "nearest":
        def call(t, p):
            return list(ctx.nearest(surf, p))
    elif what == "points":
        def call(t, p):
            return [ctx.envelope_points(surf, p, eps * eps)]
    else:
        def call(t, p):
            return [ctx.envelope_faces(surf, t, eps * eps, eps)]
    refs = [[r.clone() for r in call(t, t[:, :3].contiguous())] for t in sets]
    assert not all(torch.equal(a, b) for a, b in zip(refs[0], refs[1]))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(q, p3)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        out = call(q, p3)
    for k in range(6):
        q.copy_(sets[k % 3])
        p3.copy_(sets[k % 3][:, :3])
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, refs[k % 3])), (what, k)
        if k == 1:
            ctx.nearest(surf, big3)
        if k == 2:
            ctx.envelope_points(surf, big3, eps * eps)
            ctx.envelope_faces(surf, more, eps * eps, eps)
        if k == 3:
            ctx.envelope_faces(surf, more.repeat(2, 1), eps * eps, eps)
        torch.cuda.synchronize()
    ctx.close()

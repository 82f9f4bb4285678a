"""Surfaces whose facets shrink towards one side, and envelopes wider than the
facets: the query order that such a surface takes (as many bits as keep crowded
cells rare), wave lists that overflow, and the batches that leave the list and
lanes-per-point kernels, against the per-query tree walk (the statistics path)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def graded_sphere(freq, k):
    """a geodesic sphere drawn k-fold together towards its south pole (a
    conformal map, so the facets keep their shapes)"""
    from tetwild_amd import workloads as W
    V, F = W.geodesic_sphere(freq)
    x, y, z = V.T
    X, Y = (a / (1 - z + 1e-9) / k for a in (x, y))
    s = X * X + Y * Y
    return np.ascontiguousarray(np.stack([2 * X / (1 + s), 2 * Y / (1 + s), (s - 1) / (1 + s)], 1)), F


def facet_queries(V, F, n, eps, seed):
    """triangles on facets drawn one by one, their size at most 2.5e-3, offset
    by up to 2 eps"""
    r = np.random.default_rng(seed)
    T = V[F[r.integers(0, len(F), n)]]
    c = T.mean(1, keepdims=True)
    N = np.cross(T[:, 1] - T[:, 0], T[:, 2] - T[:, 0])
    N /= np.linalg.norm(N, axis=1, keepdims=True)
    size = np.linalg.norm(T - np.roll(T, 1, axis=1), axis=2).max(1)
    Q = c + (T - c) * np.minimum(1.0, 2.5e-3 / size)[:, None, None] + (r.uniform(-2, 2, n) * eps)[:, None, None] * N[:, None]
    return np.ascontiguousarray(Q.reshape(n, 9))


@pytest.mark.parametrize("freq,k", [(40, 30), (60, 30), (60, 300)])
def test_order_resolves_the_small_facets(freq, k):
    """Where all queries of the small side fell into a few cells of the order, a
    wave's 64 queries lay apart and most lists overflowed"""
    import torch

    from tetwild_amd.ops import Context
    ctx = Context(0)
    V, F = graded_sphere(freq, k)
    surf = ctx.surface(V, F)
    eps = 0.1 / 60 / k
    tq = torch.from_numpy(facet_queries(V, F, 12 * len(F), eps, k)).to("cuda:0")
    p3 = tq[:, :3].contiguous()
    tq = tq[:6 * len(F)]
    for q, call in ((tq, lambda: ctx.envelope_faces(surf, tq, eps * eps, 1e-3)),
                    (p3, lambda: ctx.envelope_points(surf, p3, eps * eps))):
        ctx.list_stats(True)
        call()
        listed, walked = ctx.list_stats(False)
        print(freq, k, listed, walked)
        assert listed + walked == -(-len(q) // 256) * 4
        assert walked < 0.2 * listed
    ctx.close()


@pytest.mark.parametrize("k", [1, 10, 300])
@pytest.mark.parametrize("n", [32767, 32768, 70001, 300000])
@pytest.mark.parametrize("eps", [1e-5, 1e-3, 0.05])
def test_decisions(k, n, eps):
    """Both sides of every rule, coordinates that are not finite in many waves"""
    import torch

    from tetwild_amd.ops import Context
    ctx = Context(0)
    V, F = graded_sphere(34, k)
    Q = facet_queries(V, F, n, eps, n)
    Q[7::61, 4] = np.nan
    Q[11::173, 1] = np.inf
    Q[13::977] = -np.inf
    tq = torch.from_numpy(Q).to("cuda:0")
    p3 = tq[:, :3].contiguous()
    for nf in (len(F), 500):  # (500: built on the host)
        surf = ctx.surface(V, F[:nf])
        for prec in (0, 1):
            out = ctx.envelope_faces(surf, tq, eps * eps, 1e-3, precision=prec)
            walk, _ = ctx.envelope_faces(surf, tq, eps * eps, 1e-3, precision=prec, stats=True)
            assert torch.equal(out, walk), (nf, prec, int((out != walk).sum()))
            out = ctx.envelope_points(surf, p3, eps * eps, precision=prec)
            walk, _ = ctx.envelope_points(surf, p3, eps * eps, precision=prec, stats=True)
            assert torch.equal(out, walk), (nf, prec, int((out != walk).sum()))
        surf.close()
    ctx.close()

"""Groups around the lanes of one (8) and beyond: every mix of flipped,
out-of-range and undecided (exactly coplanar) tets at every place, against the
oracle's verdict on each tet: the first bad or certainly flipped tet decides,
then a coplanar one; groups with offsets out of range and empty ones among
them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [1, 2, 6, 7, 8, 9, 15, 16, 17, 40])
def test_group_sizes(size):
    import torch

    from oracle import oracle as O
    from tetwild_amd import workloads as W
    from tetwild_amd.ops import Context
    ctx = Context(0)
    x, y, z, tets, _ = W.kuhn_lattice(6, seed=3)
    x, y, z = (np.concatenate([a, b]) for a, b in zip((x, y, z), ([0, 1, 0, 1, 0.5], [0, 0, 1, 1, 0.5], [0.0] * 5)))
    nv = len(x)
    flat = np.array([nv - 5, nv - 4, nv - 3, nv - 2], np.int32)
    r = np.random.default_rng(size)
    n = 700
    T = tets[r.integers(0, len(tets), n * size)].copy()
    for k in range(n * size):
        u = r.random() * size
        if u < 0.3:
            T[k] = T[k][[0, 1, 3, 2]]
        elif u < 0.5:
            T[k, r.integers(0, 4)] = (-1, nv, 2**31 - 1)[r.integers(0, 3)]
        elif u < 0.7:
            T[k] = flat
    off = np.arange(0, n * size + 1, size, dtype=np.int32)
    off[5] = off[4]  # an empty group, and a long one after it
    dev = [torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0") for a in (T, off, x, y, z)]
    fl, mq, q = (t.cpu().numpy() for t in ctx.tet_groups(*dev))
    out = ((T < 0) | (T >= nv)).any(1)
    coplanar = (T == flat).all(1)
    one, _, oq = O.tet_groups(np.where(out[:, None], tets[0], T), np.arange(n * size + 1, dtype=np.int32), x, y, z)
    ofl, omq = np.zeros(n, np.uint8), np.zeros(n)
    for g in range(n):
        for k in range(off[g], off[g + 1]):
            if out[k] or (one[k] and not coplanar[k]):
                ofl[g] = 2 if out[k] else 1
                break
        else:
            ofl[g] = coplanar[off[g]:off[g + 1]].any()
            omq[g] = max(oq[off[g]:off[g + 1]], default=0.0)
    assert np.array_equal(fl, ofl)
    assert np.array_equal(mq[ofl == 0], omq[ofl == 0]) and np.isnan(mq[ofl != 0]).all()
    own = np.repeat(np.arange(n), np.diff(off))
    assert np.array_equal(q[ofl[own] == 0], oq[ofl[own] == 0])
    assert 0 < (ofl == 0).sum() < n or size > 20
    bad = dev[1].clone()
    bad[3], bad[9] = -1, n * size + 1
    fl2 = ctx.tet_groups(dev[0], bad, *dev[2:], want_q=False)[0].cpu().numpy()
    assert (fl2[[2, 3, 8, 9]] == 2).all() and np.array_equal(np.delete(fl2, [2, 3, 8, 9]), np.delete(fl, [2, 3, 8, 9]))
    ctx.close()


@pytest.mark.parametrize("n,lo,hi", [(1, 1, 6), (63, 4, 4), (64, 4, 4), (65, 4, 4), (257, 0, 9), (900, 2, 6),
                                     (64, 40, 40), (70, 36, 44), (40, 60, 70), (300000, 4, 4), (270001, 5, 5),
                                     (300001, 0, 8)])
@pytest.mark.parametrize("extra", [0, 1])
def test_groups_of_a_wave(n, lo, hi, extra):
    """Waves whose groups just fill their LDS, miss it by one tet, straddle the
    batch's end or hold an offset out of range, groups of mixed sizes and empty
    ones, flipped and coplanar tets among them"""
    import torch

    from oracle import oracle as O
    from tetwild_amd import workloads as W
    from tetwild_amd.ops import Context
    ctx = Context(0)
    x, y, z, tets, _ = W.kuhn_lattice(6, seed=3)
    r = np.random.default_rng(n * 100 + hi)
    size = r.integers(lo, hi + 1, n)
    size[n // 2] += extra
    off = np.concatenate([[0], np.cumsum(size)]).astype(np.int32)
    T = tets[r.integers(0, len(tets), off[-1])].copy()
    flip = r.random(len(T)) < 0.3 / max(hi, 1)
    T[flip] = T[flip][:, [0, 1, 3, 2]]
    flat = r.random(len(T)) < min(0.1, 20 / n) / max(hi, 1)
    T[flat, 3] = T[flat, 2]
    dev = [torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0") for a in (T, off, x, y, z)]
    fl, mq, q = (t.cpu().numpy() for t in ctx.tet_groups(*dev))
    ofl, omq, oq = O.tet_groups(T, off, x, y, z)
    fine = ofl == 0
    own = np.repeat(np.arange(n), size)
    assert np.array_equal(fl, ofl) and np.array_equal(mq[fine], omq[fine]) and np.isnan(mq[~fine]).all()
    assert np.array_equal(q[fine[own]], oq[fine[own]])
    for k, v in ((n // 3, -1), (n // 2, 2**31 - 1), (n, off[-1] + 1)):
        bad = dev[1].clone()
        bad[k] = v
        fl2, mq2, _ = (t.cpu().numpy() for t in ctx.tet_groups(dev[0], bad, *dev[2:]))
        hit = np.isin(np.arange(n), (k - 1, k))
        assert (fl2[hit] == 2).all() and np.isnan(mq2[hit]).all()
        assert np.array_equal(fl2[~hit], ofl[~hit]) and np.array_equal(mq2[fine & ~hit], omq[fine & ~hit])
    ctx.close()

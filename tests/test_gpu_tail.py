"""Counts whose last depths are leaves (each generated from and checked against
earlier depths only): the leaves are counted without being placed, against the
digest run, which expands every level, and the oracle."""
import numpy as np
import pytest

import gfsm_amd as G
from helpers import oracle_solve

pytestmark = pytest.mark.gpu


def _graph(kind, mode, seed):
    """sparse: short segments; hubs: segments around and far past the eight
    entries that are read whole; loops: self loops and repeated entries."""
    rng = np.random.default_rng(seed)
    n = 400
    e = [(int(a), int(b)) for a, b in rng.integers(0, n, size=(n * 3 // 2, 2)) if a != b]
    if kind == "hubs":
        for h, deg in enumerate((7, 8, 9, 16, 17, 130)):
            e += [(h, int(b)) for b in rng.choice(np.arange(6, n), size=deg, replace=False)]
    e = sorted({(min(a, b), max(a, b)) for a, b in e})
    e = e + [(b, a) for a, b in e]
    if kind == "loops":
        e += [(int(v), int(v)) for v in rng.choice(n, size=60, replace=False)]
        e += [e[int(i)] for i in rng.integers(0, len(e), size=80)]  # entries given twice
    vl = rng.integers(1, 4, size=n)
    return G.Graph.from_edges(n, [a for a, _ in e], [b for _, b in e], [1] * len(e), vlabel=vl, mode=mode)


def _query(edges, labels, mode):
    src = [a for a, b in edges] + [b for a, b in edges]
    dst = [b for a, b in edges] + [a for a, b in edges]
    return G.Graph.from_edges(len(labels), src, dst, [1] * len(src), vlabel=labels, mode=mode)


def _queries(mode, rng):
    shapes = [
        [(0, 1), (1, 2)], [(0, 1), (1, 2), (2, 3)], [(0, 1), (1, 2), (2, 3), (3, 4)],  # paths: two leaves that meet
        [(0, 1), (0, 2), (0, 3)], [(0, 1), (0, 2), (0, 3), (0, 4)],  # stars: leaves with one set
        [(0, 1), (1, 2), (0, 3), (1, 4)], [(0, 1), (0, 2), (0, 3), (1, 4), (1, 5)],  # comb, double star
        [(0, 1), (1, 2), (2, 0), (2, 3)], [(0, 1), (1, 2), (2, 0), (0, 3), (1, 4)],  # triangle with one, two tails
        [(0, 1), (1, 2), (2, 3), (3, 0)], [(0, 1), (1, 2), (2, 3), (3, 4), (4, 0)],  # cycles: a checked leaf
        [(0, 1), (1, 2), (3, 4), (4, 5), (0, 3), (1, 4), (2, 5)],  # 2 x 3 patch: checked leaves
        [(0, 1), (0, 2), (0, 3), (1, 4), (2, 4), (2, 5), (3, 5)],  # two checked leaves that meet
        [(0, 1), (1, 2), (2, 0), (0, 3), (1, 3), (2, 3)],  # K4: a leaf with two checks
    ]
    return [_query(s, [1] * (max(map(max, s)) + 1) if k % 2 else rng.integers(1, 4, size=max(map(max, s)) + 1), mode)
            for s in shapes for k in (0, 1)]


@pytest.mark.parametrize("mode", [G.MODE_REF, G.MODE_VLABEL])
@pytest.mark.parametrize("kind", ["sparse", "hubs", "loops"])
def test_counts_equal_the_expanded_run(ctx, kind, mode):
    data = _graph(kind, mode, seed=8000)
    rng = np.random.default_rng(8001)
    for i, q in enumerate(_queries(mode, rng)):
        full = ctx.match(data, q, digest=True)
        if kind != "loops":
            assert full.count == oracle_solve(data, q, mode, rows=False).count, i
        for kw in (dict(), dict(tile=256), dict(tile=2048), dict(mem_budget=2 << 20)):
            m = ctx.match(data, q, **kw)
            assert m.count == full.count, (i, kw)
            assert m.stats["level"] == full.stats["level"] and m.stats["cand"] == full.stats["cand"], (i, kw)
        assert ctx.match_batch(data, [q])[0].count == full.count, i
        # caps before, inside and past every depth's candidates, and some that are exactly enough
        last = full.stats["cand"][-1]
        caps = {1, max(1, last // 3), max(1, last - 1), max(1, last), last + 1, 1 << 40}
        for c in full.stats["cand"][1:]:
            caps |= {max(1, c - 1), max(1, c), c + 1}
        for cap in sorted(caps):
            a = ctx.match(data, q, max_depth_cand=cap, allow_partial=True, digest=True)
            for kw in (dict(), dict(tile=256), dict(mem_budget=2 << 20)):
                b = ctx.match(data, q, max_depth_cand=cap, allow_partial=True, **kw)
                assert (b.count, b.status) == (a.count, a.status), (i, cap, kw)
            c, = ctx.match_batch(data, [q], max_depth_cand=cap)
            assert (c.count, c.status) == (a.count, a.status), (i, cap)
        total = sum(full.stats["cand"][1:])
        assert ctx.match(data, q, max_cand=total).count == full.count, i
        if total > 1:
            part = ctx.match(data, q, max_cand=total - 1, allow_partial=True)
            assert part.status == 5 and part.count <= full.count, i


def test_many_tiles_under_a_cap(ctx):
    """Steps of thousands of tiles whose cap falls early, late and between."""
    data = G.Graph.er(30000, 14.0, nvlabels=2, nelabels=1, seed=8100, mode=G.MODE_VLABEL)
    q = G.Graph.walk_query(data, 5, kind=G.WALK_SPARSE, seed=8101)
    full = ctx.match(data, q, digest=True)
    assert ctx.match(data, q).count == full.count
    last = full.stats["cand"][-1]
    for cap in (5000, last // 7, last // 2, last - 1, last, last + 1):
        a = ctx.match(data, q, max_depth_cand=cap, allow_partial=True, digest=True)
        b = ctx.match(data, q, max_depth_cand=cap, allow_partial=True)
        assert (a.count, a.status) == (b.count, b.status), cap


@pytest.mark.parametrize("degree", [10, 14, 18])
def test_checked_leaves_by_mean_length(ctx, degree):
    """Around the mean segment length up to which checked leaves are compared, and
    where only a larger or a smaller number of leaves qualifies."""
    data = G.Graph.er(300, degree, seed=degree)
    ctx.upload(data)
    shapes = [
        [(0, 1), (1, 2), (2, 0)], [(0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3)],  # triangle, clique
        [(0, 1), (1, 2), (2, 0), (0, 3), (1, 4)],  # a pair behind a check
        [(0, 1), (1, 2), (2, 3), (3, 0)], [(0, 1), (1, 2), (3, 4), (4, 5), (0, 3), (1, 4), (2, 5)],
    ]
    for edges in shapes:
        q = _query(edges, [1] * (max(map(max, edges)) + 1), G.MODE_REF)
        full, m = ctx.match(data, q, digest=True), ctx.match(data, q)
        assert m.count == full.count == oracle_solve(data, q, G.MODE_REF, rows=False).count, edges
        assert m.stats["level"] == full.stats["level"] and m.stats["cand"] == full.stats["cand"], edges

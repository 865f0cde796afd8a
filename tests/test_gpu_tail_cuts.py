"""Counted leaves under caps that their rule admits, and in batches of many queries:
steps of thousands of tiles cut in the first, a middle and the last round of the
cut's scan, and steps of many slots side by side.  The launches show that the
leaves were counted; the digest run, which expands every level, gives the counts."""
import numpy as np
import pytest

import gfsm_amd as G
from helpers import oracle_solve
from test_gpu_tail import _graph, _queries, _query

pytestmark = pytest.mark.gpu

PATH3, STAR4, PATH4 = [(0, 1), (1, 2)], [(0, 1), (0, 2), (0, 3)], [(0, 1), (1, 2), (2, 3)]
STAR5 = [(0, 1), (0, 2), (0, 3), (0, 4)]


@pytest.fixture(scope="module")
def er():
    return G.Graph.er(60000, 12.0, nvlabels=1, nelabels=1, seed=8300, mode=G.MODE_REF)


# One leaf: 720,000 candidates in the step before it, 2,813 tiles of 256 (the scan
# takes 1,024 a round) and 352 of 2,048; about 13 leaf candidates each.
@pytest.mark.parametrize("tile", [256, 2048])
def test_cut_in_every_round(ctx, er, tile):
    q = _query(PATH3, [1] * 3, G.MODE_REF)
    full = ctx.match(er, q, digest=True)
    last = full.stats["cand"][-1]
    rounds = -(-full.stats["cand"][1] // (1024 * tile))
    caps = {last - 1, last, last + 1, 1 << 40}
    for r in range(rounds):
        caps |= {int(last * (r + f) / rounds) for f in (0.25, 0.6, 0.999)}
    for cap in sorted(c for c in caps if c >= 8192 * 16):
        a = ctx.match(er, q, max_depth_cand=cap, allow_partial=True, digest=True)
        b = ctx.match(er, q, max_depth_cand=cap, allow_partial=True, tile=tile)
        assert (b.count, b.status) == (a.count, a.status), cap
        c, = ctx.match_batch(er, [q], max_depth_cand=cap)
        assert (c.count, c.status) == (a.count, a.status), cap
        d = ctx.match_noalloc(er, q, max_depth_cand=cap)
        assert d[:2] == (a.status, a.count), cap
    m = ctx.match(er, q, max_depth_cand=1 << 40, tile=tile)
    assert m.stats["launches"] == 2 < full.stats["launches"]


# Two and three leaves: the cap ends at the first or at a later leaf's depth.
@pytest.mark.parametrize("edges,leaves", [(STAR4, 2), (PATH4, 2), (STAR5, 3)])
def test_cut_of_several_leaves(ctx, edges, leaves):
    data = G.Graph.er(4000, 12.0, nvlabels=1, nelabels=1, seed=8301, mode=G.MODE_REF)
    q = _query(edges, [1] * (leaves + 2), G.MODE_REF)
    full = ctx.match(data, q, digest=True)
    for c in full.stats["cand"][-leaves:]:
        for cap in (c // 3, c // 2, c - 1, c, c + 1):
            if cap < 8192 * 16**leaves:
                continue
            a = ctx.match(data, q, max_depth_cand=cap, allow_partial=True, digest=True)
            for kw in (dict(), dict(tile=256)):
                b = ctx.match(data, q, max_depth_cand=cap, allow_partial=True, **kw)
                assert (b.count, b.status) == (a.count, a.status), (cap, kw)
            b, = ctx.match_batch(data, [q], max_depth_cand=cap)
            assert (b.count, b.status) == (a.count, a.status), cap
    m = ctx.match(data, q, max_depth_cand=1 << 40)
    assert m.count == full.count and m.stats["launches"] < full.stats["launches"]


@pytest.mark.parametrize("mode", [G.MODE_REF, G.MODE_VLABEL])
@pytest.mark.parametrize("kind", ["sparse", "hubs", "loops"])
def test_batch_of_counts(ctx, kind, mode):
    data = _graph(kind, mode, seed=8302)
    qs = _queries(mode, np.random.default_rng(8303))
    full = [ctx.match(data, q, digest=True) for q in qs]
    if kind == "sparse":
        assert [m.count for m in full] == [oracle_solve(data, q, mode, rows=False).count for q in qs]
    for b, m in zip(ctx.match_batch(data, qs), full):
        assert (b.count, b.status) == (m.count, 0)
        assert b.stats["level"] == m.stats["level"] and b.stats["cand"] == m.stats["cand"]
    srv = G.Server(ctx, data, max_inflight=8)
    t = [srv.submit(q) for q in qs]
    assert [srv.wait(x).count for x in t] == [m.count for m in full]
    srv.stop()


# Tail steps of many slots at once, each cut elsewhere; batches that begin with large
# tiles, with small ones, and that come down to a few slots.
@pytest.mark.parametrize("slots", [4, 64])
def test_batch_of_cuts(er, slots):
    qs = [_query(e, [1] * (max(map(max, e)) + 1), G.MODE_REF) for e in (PATH3, STAR4, PATH4)]
    cases = []
    for i in range(36):
        lo = 1500 * (i % 12)
        window = (lo, lo + (64 << (i % 7)))
        q = qs[i % 3]
        cap = (1 << 40, 140000, 2300000, 3000000)[i % 4]
        cases.append((q, window, cap))
    with G.Context(0, mem_budget=2 << 30) as ctx:
        ctx.set_tuning(batch_slots=slots)
        want = [ctx.match(er, q, root_lo=w[0], root_hi=w[1], max_depth_cand=c, allow_partial=True, digest=True)
                for q, w, c in cases]
        assert {m.status for m in want} == {0, 5}
        kw = dict(windows=[w for _, w, _ in cases], depth_caps=[c for _, _, c in cases])
        got = ctx.match_batch(er, [q for q, _, _ in cases], **kw)
        assert [(m.count, m.status) for m in got] == [(m.count, m.status) for m in want]
        # a step less than with the digest, which places the leaves
        full = ctx.match_batch(er, [q for q, _, _ in cases], digest=True, **kw)
        assert [(m.count, m.status) for m in full] == [(m.count, m.status) for m in want]
        assert sum(m.stats["launches"] for m in got) < sum(m.stats["launches"] for m in full)

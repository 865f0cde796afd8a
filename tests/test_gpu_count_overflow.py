"""Counts around 2^64: leaves are counted without being placed, so stars on a hub
reach such numbers at once.  The exact count below, an error of its own from there
on, on every path."""
import math

import numpy as np
import pytest

import gfsm_amd as G

pytestmark = pytest.mark.gpu


def _biclique(hubs, n):
    a = np.repeat(np.arange(hubs, dtype=np.uint32), n)
    b = np.tile(np.arange(hubs, hubs + n, dtype=np.uint32), hubs)
    return G.Graph.from_edges(hubs + n, np.concatenate([a, b]), np.concatenate([b, a]), np.ones(2 * hubs * n, np.uint32))


def _star(leaves):
    c, lf = [0] * leaves, list(range(1, leaves + 1))
    return G.Graph.from_edges(leaves + 1, c + lf, lf + c, [1] * (2 * leaves))


def _limit(leaves):
    n = int((2.0**64) ** (1 / leaves))
    while math.perm(n, leaves) >= 2**64:
        n -= 1
    while math.perm(n + 1, leaves) < 2**64:
        n += 1
    return n


@pytest.mark.parametrize("leaves", [4, 5])
def test_star_around_the_limit(ctx, leaves):
    n, q = _limit(leaves), _star(leaves)
    data = _biclique(1, n)
    ctx.upload(data)
    want = math.perm(n, leaves)
    m = ctx.match(data, q)
    assert m.count == want
    # the segment's n entries for each of the choices before; the hub's neighbours as
    # roots find the hub, and it once more
    cand = [n + 1, 2 * n] + [math.perm(n, k) * n + (n if k == 1 else 0) for k in range(1, leaves)]
    assert m.stats["cand"] == [min(c, 2**64 - 1) for c in cand]
    assert ctx.match_noalloc(data, q)[:2] == (0, want)
    b, = ctx.match_batch(data, [q])
    assert (b.status, b.count) == (0, want) and b.stats["cand"] == m.stats["cand"]

    data = _biclique(1, n + 1)
    ctx.upload(data)
    for call in (ctx.match, ctx.match_noalloc):
        with pytest.raises(G.GfsmError) as e:
            call(data, q)
        assert e.value.code == G.ERR_OVERFLOW
    small = _star(3)
    a, b, c = ctx.match_batch(data, [small, q, small])
    assert (b.status, b.count) == (G.ERR_OVERFLOW, 0)
    assert (a.status, a.count) == (c.status, c.count) == (0, math.perm(n + 1, 3))
    srv = G.Server(ctx, data)
    t = [srv.submit(x) for x in (q, small)]
    b, a = [srv.wait(x) for x in t]
    srv.stop()
    assert (b.status, b.count) == (G.ERR_OVERFLOW, 0) and (a.status, a.count) == (0, math.perm(n + 1, 3))


def test_capped_counts_stay_exact(ctx):
    n = _limit(5) + 1
    data, q = _biclique(1, n), _star(5)
    for cap in (1 << 30, 1 << 40, 3 << 50):
        a = ctx.match(data, _star(4), max_depth_cand=cap, allow_partial=True)
        b, = ctx.match_batch(data, [_star(4)], max_depth_cand=cap)
        assert (a.count, a.status) == (b.count, b.status)
    assert ctx.match(data, q, max_depth_cand=1 << 30, allow_partial=True).status == 5


def test_tiles_of_almost_2_to_62():
    """More tiles than workgroups, each near the most that a tile may count: launches
    of few enough for a workgroup's own sum."""
    with G.Context(0) as ctx:
        ctx.set_tuning(wgs_per_cu=1)
        data = _biclique(25, 130000)
        with pytest.raises(G.GfsmError) as e:
            ctx.match(data, _star(4), tile=2048)
        assert e.value.code == G.ERR_OVERFLOW

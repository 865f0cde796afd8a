"""Counting steps whose tiles all have a workgroup of their own, and the first that
have not: every tile is counted once, whatever the number of tiles."""
import numpy as np
import pytest

import gfsm_amd as G

pytestmark = pytest.mark.gpu

N = 1 << 14


@pytest.fixture(scope="module")
def ring():
    a = np.arange(N, dtype=np.uint32)
    b = (a + 1) % N
    return G.Graph.from_edges(N, np.concatenate([a, b]), np.concatenate([b, a]), np.ones(2 * N, np.uint32))


# A ring's path of three: 2 candidates a root in the step before the last, 2 of
# those 4 survive; tiles of 256 candidates.
@pytest.mark.parametrize("tiles", [1, 7, 8, 9, 15, 16, 17, 64, 120, 127, 128])
@pytest.mark.parametrize("wgs", [None, 1])
def test_tiles_of_a_small_step(ring, tiles, wgs):
    q = G.Graph.from_edges(3, [0, 1, 1, 2], [1, 0, 2, 1], [1] * 4)
    with G.Context(0, mem_budget=1 << 28) as ctx:
        if wgs:
            ctx.set_tuning(wgs_per_cu=wgs)
        for roots in (128 * tiles - 1, 128 * tiles):
            for kw in (dict(), dict(digest=True)):  # counted leaves; a last depth
                m = ctx.match(ring, q, root_lo=0, root_hi=roots, tile=256, **kw)
                assert m.count == 2 * roots, (roots, kw)
        full = ctx.match(ring, q, tile=256, digest=True)
        assert full.count == 2 * N and full.digest == ctx.match(ring, q, digest=True).digest

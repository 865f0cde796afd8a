"""Sorted rows against a host sort of the unsorted ones: the device sorts the
table where one chunk holds it, the host where it does not."""
import numpy as np
import pytest

import gfsm_amd as G

pytestmark = pytest.mark.gpu


def _path(labels, num, mode):
    q = len(labels)
    pairs = [(num[i], num[i + 1]) for i in range(q - 1)]
    src = [a for a, _ in pairs] + [b for _, b in pairs]
    dst = [b for _, b in pairs] + [a for a, _ in pairs]
    return G.Graph.from_edges(q, src, dst, [1] * len(src), vlabel=labels, mode=mode)


# vertices around the digit width (one to three digits a column), rows around a
# block of 2,048 and far past it; every numbering of the columns' roles
@pytest.mark.parametrize("n,degree", [(60, 6.0), (128, 9.0), (129, 9.0), (256, 6.0), (300, 12.0), (5000, 5.0), (66000, 4.0)])
@pytest.mark.parametrize("num", [(0, 1, 2), (2, 1, 0), (1, 0, 2), (0, 2, 1), (1, 2, 3, 0), (3, 0, 2, 1)])
def test_sorted_rows(ctx, n, degree, num):
    data = G.Graph.er(n, degree, nvlabels=1, nelabels=1, seed=9000 + n, mode=G.MODE_REF)
    query = _path([1] * len(num), num, G.MODE_REF)
    rows = ctx.match(data, query, rows=True).rows
    want = rows[np.lexsort(rows.T[::-1])]
    assert len(want) > 0
    got = ctx.match(data, query, rows=True, sorted=True)
    assert got.count == len(want) and np.array_equal(got.rows, want)
    small = ctx.match(data, query, rows=True, sorted=True, mem_budget=2 << 20)  # chunks: sorted on the host
    assert np.array_equal(small.rows, want)


def test_sorted_rows_under_caps(ctx):
    data = G.Graph.er(3000, 8.0, nvlabels=1, nelabels=1, seed=9100, mode=G.MODE_REF)
    query = _path([1] * 3, (2, 0, 1), G.MODE_REF)
    a = ctx.match(data, query, rows=True, max_depth_cand=50000, allow_partial=True)
    b = ctx.match(data, query, rows=True, sorted=True, max_depth_cand=50000, allow_partial=True)
    assert a.status == b.status == 5
    assert np.array_equal(b.rows, a.rows[np.lexsort(a.rows.T[::-1])])
    full = ctx.match(data, query, rows=True, sorted=True)
    assert ctx.match(data, query, rows=True, sorted=True, max_rows=full.count).count == full.count
    with pytest.raises(G.GfsmError):
        ctx.match(data, query, rows=True, sorted=True, max_rows=full.count - 1)


@pytest.mark.parametrize("n", [50, 5000, 60000])  # below and above the size from which the table is pinned
def test_rows_outlive_match_and_context(n):
    """The rows are a view of the result's memory: they stay valid, and can be
    written, after the match, the graphs and the context are gone."""
    ctx = G.Context(0)
    data = G.Graph.er(n, 6.0, nvlabels=1, nelabels=1, seed=9200, mode=G.MODE_REF)
    query = _path([1] * 3, (0, 1, 2), G.MODE_REF)
    m = ctx.match(data, query, rows=True)
    rows, copy = m.rows, m.rows.copy()
    again = ctx.match(data, query, rows=True).rows  # another result in between
    del m, data, query
    ctx.close()
    assert np.array_equal(rows, copy) and np.array_equal(again, copy)
    rows[0, 0] += 1
    assert rows[0, 0] == copy[0, 0] + 1 and np.array_equal(again, copy)

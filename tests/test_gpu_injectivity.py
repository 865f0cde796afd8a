"""Injectivity masks: which placed vertices a candidate is compared with
depends on the labels along the matching order and on whether the data graph
has self loops."""
import numpy as np
import pytest

import gfsm_amd as G
from helpers import assert_same, oracle_solve

pytestmark = pytest.mark.gpu


def _data(mode, labels, loops, seed, n=160, degree=9):
    rng = np.random.default_rng(seed)
    pairs = {(int(min(a, b)), int(max(a, b))) for a, b in rng.integers(0, n, size=(n * degree // 2, 2))}
    pairs = {(a, b) for a, b in pairs if a != b}
    if loops:
        pairs |= {(int(v), int(v)) for v in rng.choice(n, size=n // 3, replace=False)}
    e = sorted(pairs | {(b, a) for a, b in pairs})
    vl = rng.integers(1, labels + 1, size=n)
    return G.Graph.from_edges(n, [a for a, _ in e], [b for _, b in e], [1] * len(e), vlabel=vl, mode=mode)


@pytest.mark.parametrize("mode", [G.MODE_REF, G.MODE_VLABEL])
@pytest.mark.parametrize("labels", [1, 2, 4])
@pytest.mark.parametrize("loops", [False, True])
def test_masks_vs_oracle(ctx, tmp_path, mode, labels, loops):
    data = _data(mode, labels, loops, seed=7000 + 10 * labels + loops)
    data.save_bin(tmp_path / "d.bin")
    image = G.Graph.load_bin(tmp_path / "d.bin")  # the masks of a loaded image are the built graph's
    for k, q in enumerate((2, 3, 4, 5)):
        # walks over a loop-free copy: queries without self loops on data with them
        query = G.Graph.walk_query(_data(mode, labels, False, seed=7000 + 10 * labels + loops), q,
                                   kind=k % 2, seed=7100 + k)
        ref = oracle_solve(data, query, mode)
        assert_same(ctx.match(data, query, rows=True, sorted=True, digest=True), ref)
        assert_same(ctx.match(image, query, digest=True), ref, rows=False)
        assert ctx.match(data, query).count == ref.count
        b, = ctx.match_batch(data, [query], digest=True)
        assert (b.count, b.digest) == (ref.count, ref.digest)
        assert ctx.match_batch(data, [query])[0].count == ref.count

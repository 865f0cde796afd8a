"""Embedding tables on the host: whole and right whatever their size against the
copy's pieces, in one chunk or many, in memory or in a file; in ordinary memory."""
import numpy as np
import pytest

import gfsm_amd as G

pytestmark = pytest.mark.gpu

N = 1 << 22
MIB = 1 << 20


@pytest.fixture(scope="module")
def ring():
    a = np.arange(N, dtype=np.uint32)
    b = (a + 1) % N
    return G.Graph.from_edges(N, np.concatenate([a, b]), np.concatenate([b, a]), np.ones(2 * N, np.uint32))


@pytest.fixture(scope="module")
def path3():
    return G.Graph.from_edges(3, [0, 1, 1, 2], [1, 0, 2, 1], [1] * 4)


def _want(roots):
    """Both orders of each root's neighbours, the smaller one first."""
    v = np.arange(roots, dtype=np.int64)
    a, b = np.minimum((v - 1) % N, (v + 1) % N), np.maximum((v - 1) % N, (v + 1) % N)
    return np.stack([np.stack([a, v, b], 1), np.stack([b, v, a], 1)], 1).reshape(-1, 3).astype(np.uint32)


# 24 bytes a root: around one and eight small pieces, the pieces between, eight large ones, past them
@pytest.mark.parametrize("bytes_", [24, MIB // 4, MIB, 2 * MIB, 4 * MIB, 8 * MIB, 16 * MIB, 20 * MIB, 90 * MIB])
def test_rows(ctx, ring, path3, tmp_path, bytes_):
    for roots in sorted({bytes_ // 24, bytes_ // 24 + 1}):
        want = _want(roots)
        assert np.array_equal(ctx.match(ring, path3, rows=True, root_lo=0, root_hi=roots).rows, want)
        for mb in (3, 40):
            m = ctx.match(ring, path3, rows=True, root_lo=0, root_hi=roots, mem_budget=mb * MIB)
            assert np.array_equal(m.rows, want), mb
            ctx.match_to_fs(ring, path3, tmp_path / "o.fs", root_lo=0, root_hi=roots, mem_budget=mb * MIB)
            assert np.array_equal(G.read_fs(tmp_path / "o.fs"), want), mb
        s = ctx.match(ring, path3, sorted=True, root_lo=0, root_hi=roots).rows
        assert np.array_equal(s, want[np.lexsort(want.T[::-1])])


def _device_mapped():
    """Bytes of this process's address space that the device's driver maps: pinned
    memory, not ordinary one."""
    n = 0
    with open("/proc/self/maps") as f:
        for line in f:
            if "/dev/dri/" in line or "/dev/kfd" in line:
                lo, hi = line.split()[0].split("-")
                n += int(hi, 16) - int(lo, 16)
    return n


def test_results_pin_no_memory(ring, path3):
    with G.Context(0, mem_budget=1 << 30) as ctx:
        kw = dict(rows=True, root_lo=0, root_hi=2 * MIB)  # 48 MiB of rows
        ctx.match(ring, path3, **kw)
        before = _device_mapped()
        kept = [ctx.match(ring, path3, **kw) for _ in range(8)]
        assert _device_mapped() - before < 48 * MIB
        assert all(np.array_equal(m.rows, kept[0].rows) for m in kept)

"""Counts on the bit matrix (graphs of few vertices) against the oracle, at the
edges of its 1024-column lines, its passes, its long rows and its largest size."""
from __future__ import annotations

import numpy as np
import pytest

import custingeralg_amd as T
import oracle as O
from tests import graphs as GR

pytestmark = pytest.mark.gpu


def _rand(n, m, seed, loops=False):
    """Directed rows: m drawn entries, vertex 0 pointing to all, sorted and distinct."""
    rng = np.random.default_rng(seed)
    u = np.concatenate([rng.integers(0, n, m), np.zeros(n, np.int64)])
    v = np.concatenate([rng.integers(0, n, m), np.arange(n)])
    key = np.unique(u * n + v)
    if not loops:
        key = key[key // n != key % n]
    off = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))]).astype(np.int64)
    return off, (key % n).astype(np.int32)


def _sym(off, adj):
    src = np.repeat(np.arange(len(off) - 1, dtype=np.int32), np.diff(off))
    return O.canon_csr(len(off) - 1, src, adj)


@pytest.mark.parametrize("n", [1, 2, 31, 33, 1023, 1024, 1025, 2048, 2049, 4097, 16384, 16385])
@pytest.mark.parametrize("loops", [False, True])
def test_sizes(n, loops):
    off, adj = _rand(n, 12 * n, n, loops)
    ref = O.custinger_count(off, adj)
    g = T.cuStinger(off, adj)
    pv, glob, _ = T.static_count(g)
    g.close()
    assert np.array_equal(pv, ref)
    assert glob == int(ref.astype(np.uint64).sum())
    c, tot = T.csr_count_device(off, adj)
    ref = O.csr_count(off, adj)
    assert np.array_equal(c, ref) and tot == int(ref.astype(np.uint64).sum())
    if loops:
        return
    off, adj = _sym(off, adj)
    ref = O.custinger_count(off, adj)
    g = T.cuStinger(off, adj)
    for out in (True, False):
        pv, glob, st = T.static_count(g, None, out)
        assert glob == int(ref.astype(np.uint64).sum())
        assert st["method_used"] == T.METHOD_ORIENTED and st["triangles"] * 6 == glob
        assert not out or np.array_equal(pv, ref)
    g.close()


@pytest.mark.parametrize("n", [127, 128, 129, 130, 257, 600])
def test_complete_rows_around_the_item_length(n):
    off, adj, t = GR.complete_fast(n)
    g = T.cuStinger(off, adj)
    pv, glob, _ = T.static_count(g)
    g.close()
    assert np.array_equal(pv, (2 * t).astype(np.uint32)) and glob == 2 * int(t.sum())


@pytest.mark.parametrize("n", [50, 1500])
def test_declared_symmetric_that_is_not(n):
    off, adj = _sym(*_rand(n, 8 * n, 3))
    k = int(off[n // 2])  # one entry of a middle row removed
    off2 = off.copy()
    off2[n // 2 + 1:] -= 1
    adj2 = np.delete(adj, k)
    ref = O.custinger_count(off2, adj2)
    g = T.cuStinger(off2, adj2, assume_symmetric=True)
    with pytest.raises(T.TCError):
        T.static_count(g, T.default_schedule(method=T.METHOD_ORIENTED))
    pv, glob, st = T.static_count(g)
    g.close()
    assert st["method_used"] == T.METHOD_DIRECT
    assert np.array_equal(pv, ref) and glob == int(ref.astype(np.uint64).sum())


@pytest.mark.parametrize("sizes", [[1, 2, 1024, 1025, 3, 5000], [40] * 300, [16384, 7], [16385, 7]])
@pytest.mark.parametrize("cross", [False, True])
def test_batched(sizes, cross):
    """Per-graph and per-vertex counts of a concatenation; cross: one edge between
    the last two graphs, which the bit matrix cannot hold."""
    voff = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    us, vs = [], []
    for i, n in enumerate(sizes):
        off, adj = _rand(n, 6 * n, i)
        us.append(np.repeat(np.arange(n), np.diff(off)) + voff[i])
        vs.append(adj + voff[i])
    if cross:
        us.append(np.array([voff[-2]]))
        vs.append(np.array([voff[-2] - 1]))
    nv = int(voff[-1])
    off, adj = O.canon_csr(nv, np.concatenate(us).astype(np.int32),
                           np.concatenate(vs).astype(np.int32))
    ref = O.custinger_count(off, adj)
    dv, do, da = (T.DeviceArray.from_host(x) for x in (voff, off, adj))
    bg = T.BatchedGraph(dv, do, da)
    pg, pv = T.DeviceArray(len(sizes), np.uint64), T.DeviceArray(nv, np.uint32)
    for _ in range(2):
        bg.count(pg, pv)
        assert np.array_equal(pv.to_host(), ref)
        want = np.add.reduceat(ref.astype(np.uint64), voff[:-1])
        assert np.array_equal(pg.to_host(), want)
        bg.count(pg)
        assert np.array_equal(pg.to_host(), want)
    bg.close()

"""Counts of graphs whose rows are all short against the oracle: rows around
the longest the kernel takes, means around its lane splits, loops, asymmetric
and declared-symmetric rows, batches, and a store after an update."""
from __future__ import annotations

import numpy as np
import pytest

import custingeralg_amd as T
import oracle as O

pytestmark = pytest.mark.gpu


def _regular(n, d, seed, longest=0, loops=False):
    """Directed rows of about d near entries (many triangles); row 1 has
    longest entries, row 2 one, row 3 none."""
    rng = np.random.default_rng(seed)
    u = np.repeat(np.arange(n), d)
    v = (u + rng.integers(1, 2 * d + 2, len(u))) % n
    keep = (u != 2) & (u != 3)
    if longest:
        keep &= u != 1
    u, v = np.concatenate([u[keep], [2]]), np.concatenate([v[keep], [0]])
    if longest:
        u = np.concatenate([u, np.full(longest, 1)])
        v = np.concatenate([v, 2 + np.arange(longest)])
    if loops:
        x = np.arange(5, n, 7)
        u, v = np.concatenate([u, x]), np.concatenate([v, x])
    key = np.unique(u * n + v)
    if not loops:
        key = key[key // n != key % n]
    off = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))]).astype(np.int64)
    return off, (key % n).astype(np.int32)


def _sym(off, adj):
    return O.canon_csr(len(off) - 1, np.repeat(np.arange(len(off) - 1, dtype=np.int32), np.diff(off)), adj)


@pytest.mark.parametrize("d", [1, 4, 8, 9, 24, 26, 40, 45])
@pytest.mark.parametrize("longest", [0, 63, 64, 65, 127, 128, 129])
def test_rows(d, longest):
    for loops in (False, True):
        off, adj = _regular(3000, d, d, longest, loops)
        ref = O.custinger_count(off, adj)
        g = T.cuStinger(off, adj)
        pv, glob, _ = T.static_count(g)
        g.close()
        assert np.array_equal(pv, ref) and glob == int(ref.astype(np.uint64).sum())
        c, tot = T.csr_count_device(off, adj)
        ref = O.csr_count(off, adj)
        assert np.array_equal(c, ref) and tot == int(ref.astype(np.uint64).sum())
    off, adj = _sym(*_regular(20000, d, d, longest))
    ref = O.custinger_count(off, adj)
    g = T.cuStinger(off, adj)
    pv, glob, st = T.static_count(g)
    assert st["method_used"] == T.METHOD_ORIENTED
    assert np.array_equal(pv, ref) and glob == int(ref.astype(np.uint64).sum())
    # an update: the longest row is no longer known
    u = np.zeros(150, np.int32)
    T.batch_apply(g, u, np.arange(1000, 1150, dtype=np.int32))
    o2, a2 = g.to_csr()
    pv, _, _ = T.static_count(g)
    g.close()
    assert np.array_equal(pv, O.custinger_count(o2, a2))


def test_declared_symmetric_that_is_not():
    off, adj = _sym(*_regular(20000, 6, 1))
    k = int(off[77])
    off2 = off.copy()
    off2[78:] -= 1
    adj2 = np.delete(adj, k)
    ref = O.custinger_count(off2, adj2)
    g = T.cuStinger(off2, adj2, assume_symmetric=True)
    with pytest.raises(T.TCError):
        T.static_count(g, T.default_schedule(method=T.METHOD_ORIENTED))
    pv, glob, st = T.static_count(g)
    g.close()
    assert st["method_used"] == T.METHOD_DIRECT
    assert np.array_equal(pv, ref) and glob == int(ref.astype(np.uint64).sum())


@pytest.mark.parametrize("sym", [True, False])
def test_batched_and_replay(sym):
    sizes = [20000, 1, 700, 4]
    voff = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    us, vs = [], []
    for i, n in enumerate(sizes):
        if n > 100:
            off, adj = _regular(n, 5, i)
            if sym:
                off, adj = _sym(off, adj)
            us.append(np.repeat(np.arange(n), np.diff(off)) + voff[i])
            vs.append(adj + voff[i])
    u, v = np.concatenate(us), np.concatenate(vs)
    nv = int(voff[-1])
    off = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=nv))]).astype(np.int64)
    ref = O.custinger_count(off, v.astype(np.int32))
    dv, do, da = (T.DeviceArray.from_host(x) for x in (voff, off, v.astype(np.int32)))
    bg = T.BatchedGraph(dv, do, da)
    pg, pv = T.DeviceArray(len(sizes), np.uint64), T.DeviceArray(nv, np.uint32)
    sched = T.default_schedule(capture=1)
    for k in range(4):
        st = bg.count(pg, pv, sched)
        assert st["graph_replay"] == (k > 0)
        assert np.array_equal(pv.to_host(), ref)
        assert np.array_equal(pg.to_host(), np.add.reduceat(ref.astype(np.uint64), voff[:-1]))
    bg.close()

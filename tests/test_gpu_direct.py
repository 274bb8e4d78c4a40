"""Direct counts by the larger row against the oracle: directed rows with hubs,
self-loops and vertex 0 in many lists, at the id ranges where the bit rows
change their size and begin to be tiled, and the CSR convention."""
from __future__ import annotations

import numpy as np
import pytest

import custingeralg_amd as T
import oracle as O

pytestmark = pytest.mark.gpu


def _hubs(n, seed, hubs=40, hub_deg=3000, m=30000, loops=True):
    """Directed rows: a few hubs of long rows over all ids (0 among them), many
    rows pointing to hubs, a sparse background, some loops."""
    rng = np.random.default_rng(seed)
    h = np.concatenate([[0, 1, n - 1], rng.choice(n, hubs, replace=False)])
    u = [np.repeat(h, hub_deg), rng.integers(0, n, m), rng.integers(0, n, m), rng.integers(0, n, m // 2)]
    v = [rng.integers(0, n, len(h) * hub_deg), rng.choice(h, m), rng.integers(0, n, m),
         np.zeros(m // 2, np.int64)]
    # dense middle rows among 600 vertices: every row length around the bins' edges
    d = rng.choice(n, 600, replace=False)
    for i, x in enumerate(d):
        u.append(np.full(i, x))
        v.append(d[rng.permutation(600)[:i]])
    u, v = np.concatenate(u), np.concatenate(v)
    if loops:
        u, v = np.concatenate([u, h, d[:50]]), np.concatenate([v, h, d[:50]])
    key = np.unique(u * n + v)
    if not loops:
        key = key[key // n != key % n]
    off = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))]).astype(np.int64)
    return off, (key % n).astype(np.int32)


@pytest.mark.parametrize("n", [16385, 1 << 18, (1 << 18) + 1, 1 << 20, (1 << 20) + 1, 2100000])
@pytest.mark.parametrize("loops", [False, True])
def test_directed(n, loops):
    off, adj = _hubs(n, n, loops=loops)
    ref = O.custinger_count(off, adj)
    g = T.cuStinger(off, adj)
    for method in (T.METHOD_AUTO, T.METHOD_DIRECT):
        pv, glob, st = T.static_count(g, T.default_schedule(method=method))
        assert st["method_used"] == T.METHOD_DIRECT
        assert np.array_equal(pv, ref) and glob == int(ref.astype(np.uint64).sum())
    g.close()
    c, tot = T.csr_count_device(off, adj)
    ref = O.csr_count(off, adj)
    assert np.array_equal(c, ref) and tot == int(ref.astype(np.uint64).sum())


def test_direct_method_on_symmetric_rows_and_replay():
    off, adj = O.rmat_graph(16, 12, 4)
    ref = O.custinger_count(off, adj)
    g = T.cuStinger(off, adj)
    out = T.DeviceArray(g.nv, np.uint32)
    sched = T.default_schedule(method=T.METHOD_DIRECT, capture=1)
    for k in range(4):
        _, glob, st = T.static_count(g, sched, out=out)
        assert np.array_equal(out.to_host(), ref) and glob == int(ref.astype(np.uint64).sum())
        assert st["graph_replay"] == (k > 0)
    out.free()
    g.close()


def test_batched_asymmetric():
    sizes = [20000, 300, 5000]
    voff = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    offs, adjs = [np.zeros(1, np.int64)], []
    for i, n in enumerate(sizes):
        off, adj = _hubs(n, i, hubs=10, hub_deg=min(n // 2, 3000), m=3000) if n > 1000 else \
            O.rmat_graph(8, 4, 1)
        off = np.concatenate([off, np.full(n + 1 - len(off), off[-1])])
        offs.append(off[1:] + offs[-1][-1])
        adjs.append(adj + int(voff[i]))
    off, adj = np.concatenate(offs), np.concatenate(adjs).astype(np.int32)
    ref = O.custinger_count(off, adj)
    pg, pv, st = T.batched_count(voff, off, adj, per_vertex=True)
    assert st["method_used"] == T.METHOD_DIRECT
    assert np.array_equal(pv, ref)
    assert np.array_equal(pg, np.add.reduceat(ref.astype(np.uint64), voff[:-1]))


@pytest.mark.parametrize("entries", [1, 63, 65, 4095, 4096, 4097, 8192, 20481])
@pytest.mark.parametrize("owners", ["one", "all different"])
def test_places_around_the_tiles(entries, owners):
    """Entry counts around the 4096 whose owners a block counts together: tasks
    of one owner only, and of as many as there are entries."""
    n = 70000
    rng = np.random.default_rng(entries)
    if owners == "one":  # rows of two entries, both to vertices with longer rows
        src = np.repeat(np.arange(10, 10 + (entries + 1) // 2), 2)[:entries]
        dst = np.tile([3, 4], (entries + 1) // 2)[:entries]
        hub = np.repeat([3, 4], 5)
        key = np.unique(np.concatenate([src * n + dst, hub * n + np.tile(np.arange(60000, 60005), 2)]))
    else:
        src = rng.choice(n, entries, replace=False)
        dst = (src + rng.integers(1, n, entries)) % n
        key = np.unique(np.concatenate([src * n + dst, src * n + (src + 1) % n]))
    off = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))]).astype(np.int64)
    adj = (key % n).astype(np.int32)
    ref = O.custinger_count(off, adj)
    g = T.cuStinger(off, adj)
    pv, glob, st = T.static_count(g, T.default_schedule(method=T.METHOD_DIRECT))
    g.close()
    assert np.array_equal(pv, ref) and glob == int(ref.astype(np.uint64).sum())

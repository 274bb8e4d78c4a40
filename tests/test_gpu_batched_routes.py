"""Batches on both sides of the rules that choose their route, against the
oracle."""
from __future__ import annotations

import numpy as np
import pytest

import custingeralg_amd as T
import oracle as O

pytestmark = pytest.mark.gpu


def _batch(sizes, mean, hub, seed):
    """Graphs of random pairs, each with a hub row of hub entries."""
    rng = np.random.default_rng(seed)
    voff = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    u, v = [], []
    for a, n in zip(voff, sizes):
        m = int(n * mean / 2)
        x, y = rng.integers(0, n, (2, m))
        h = rng.permutation(n)[:min(hub, n)]
        u += [x + a, np.full(len(h), n // 2) + a]
        v += [y + a, h + a]
    off, adj = O.canon_csr(int(voff[-1]), np.concatenate(u).astype(np.int32), np.concatenate(v).astype(np.int32))
    return voff, off, adj


def _check(voff, off, adj, **sched):
    ref = O.custinger_count(off, adj)
    pg, pv, st = T.batched_count(voff, off, adj, T.default_schedule(**sched), per_vertex=True)
    assert np.array_equal(pv, ref)
    assert np.array_equal(pg, np.add.reduceat(ref.astype(np.uint64), voff[:-1]))
    return sum(st["tasks_bin"])


@pytest.mark.parametrize("graphs,lists", [(1, False), (2, False), (40, True)])
def test_wide_bit_rows(graphs, lists):
    """Graphs of 16384 vertices: their bit rows are 2 KB each."""
    b = _batch([16384] * graphs, 6, 400, graphs)
    assert (_check(*b) > 0) == lists


@pytest.mark.parametrize("mean,core", [(2, False), (12, True)])
def test_cores_of_sparse_batches(mean, core):
    """A batch with a graph above the bit rows' size: its cores take the place of
    task lists only where there are entries enough."""
    b = _batch([17000] + [1500] * 12, mean, 1200, 3)
    fewer = _check(*b) < _check(*b, policy=T.POLICY_HASH)  # (a forced strategy has no cores)
    assert fewer == core


@pytest.mark.parametrize("hub,lists", [(12, False), (110, True)])
def test_short_rows_of_a_large_graph(hub, lists):
    """3M vertices in a million triangles, and one longer row: row by row, or with
    a hub oriented."""
    n = 3000000
    rng = np.random.default_rng(hub)
    a, b, c = rng.integers(0, n, (3, n // 3))
    h = rng.choice(n, hub, replace=False)
    u = np.concatenate([a, b, c, np.full(hub, 77)])
    v = np.concatenate([b, c, a, h])
    off, adj = O.canon_csr(n, u.astype(np.int32), v.astype(np.int32))
    assert np.diff(off).max() <= 128
    ref = O.custinger_count(off, adj)
    g = T.cuStinger(off, adj)
    pv, glob, st = T.static_count(g)
    g.close()
    assert np.array_equal(pv, ref) and glob == int(ref.astype(np.uint64).sum())
    assert (sum(st["tasks_bin"]) > 0) == lists

"""Batched handles whose boundaries the entries do not keep to: rows of N+ are
then as long as the rows themselves, whatever the number of entries."""
from __future__ import annotations

import numpy as np
import pytest

import custingeralg_amd as T
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [100, 300, 600, 5000, 17000])
def test_hub_of_another_graph(k):
    """Vertex 0, of a graph of three, next to k vertices of the other graph;
    vertices 1 and 2 next to it and to some of these."""
    n = k + 1000
    rng = np.random.default_rng(k)
    w = 3 + rng.permutation(n)[:k]
    few = [w[:k // 3], w[k // 4:k // 2]]
    u = [np.zeros(k, np.int64), np.full(len(few[0]), 1), np.full(len(few[1]), 2), np.zeros(2, np.int64),
         np.ones(1, np.int64), 3 + rng.integers(0, n, n // 2)]
    v = [w, few[0], few[1], np.array([1, 2]), np.array([2]), 3 + rng.integers(0, n, n // 2)]
    off, adj = O.canon_csr(n + 3, np.concatenate(u).astype(np.int32), np.concatenate(v).astype(np.int32))
    voff = np.array([0, 3, n + 3], np.int64)
    ref = O.custinger_count(off, adj)
    assert ref[0] > k // 4
    pg, pv, st = T.batched_count(voff, off, adj, per_vertex=True)
    assert st["method_used"] == T.METHOD_ORIENTED
    assert np.array_equal(pv, ref)
    # (a triangle of two graphs is counted whole in either)
    assert int(pg.sum()) == int(ref.astype(np.uint64).sum())


@pytest.mark.parametrize("hub", [0, 300])
def test_boundaries_short_of_the_vertices(hub):
    """Vertices before the first boundary and after the last belong to the first
    and the last graph, whichever route counts (hub: rows above 128 entries)."""
    rng = np.random.default_rng(hub)
    n = 4000
    part = np.array([0, 1500, 2500, n])
    u = np.concatenate([rng.integers(a, b, 6 * (b - a)) for a, b in zip(part, part[1:])] +
                       [np.full(hub, 1600)])
    v = np.concatenate([rng.integers(a, b, 6 * (b - a)) for a, b in zip(part, part[1:])] +
                       [rng.integers(1500, 2500, hub)])
    off, adj = O.canon_csr(n, u.astype(np.int32), v.astype(np.int32))
    ref = O.custinger_count(off, adj)
    want = np.add.reduceat(ref.astype(np.uint64), part[:-1])
    for voff in ([0, 1500, 2500, n], [40, 1500, 2500, n - 70], [0, 1500, 2500, n - 1]):
        pg, pv, _ = T.batched_count(np.array(voff), off, adj, per_vertex=True)
        assert np.array_equal(pv, ref)
        assert np.array_equal(pg, want), voff

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

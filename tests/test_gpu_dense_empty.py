"""Bit-matrix counts of graphs whose first vertices are isolated: their empty
rows stand at the front of the adjacency array."""
from __future__ import annotations

import numpy as np
import pytest

import custingeralg_amd as T
import oracle as O

pytestmark = pytest.mark.gpu


def _graph(n, first, hub, seed):
    """Vertices below first isolated, the next one in a row of hub entries."""
    rng = np.random.default_rng(seed)
    u = np.concatenate([rng.integers(first, n, 6 * n), np.full(hub, first)])
    v = np.concatenate([rng.integers(first, n, 6 * n), first + 1 + rng.permutation(n - first - 1)[:hub]])
    return O.canon_csr(n, u.astype(np.int32), v.astype(np.int32))


@pytest.mark.parametrize("n", [700, 3000, 5000, 9001])
@pytest.mark.parametrize("first", [1, 70])
def test_isolated_first_vertices(n, first):
    off, adj = _graph(n, first, 300, n)
    assert off[first] == 0 and np.diff(off).max() > 128
    ref = O.custinger_count(off, adj)
    g = T.cuStinger(off, adj)
    pv, glob, st = T.static_count(g)
    g.close()
    assert st["method_used"] == T.METHOD_ORIENTED
    assert np.array_equal(pv, ref) and glob == int(ref.astype(np.uint64).sum())


def test_batched_isolated_first_vertices():
    sizes = [3000, 5000, 40]
    voff = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    offs, adjs = [np.zeros(1, np.int64)], []
    for i, n in enumerate(sizes):
        off, adj = _graph(n, 5, min(300, n // 2), i)
        offs.append(off[1:] + offs[-1][-1])
        adjs.append(adj + int(voff[i]))
    off, adj = np.concatenate(offs), np.concatenate(adjs).astype(np.int32)
    ref = O.custinger_count(off, adj)
    pg, pv, _ = T.batched_count(voff, off, adj, per_vertex=True)
    assert np.array_equal(pv, ref)
    assert np.array_equal(pg, np.add.reduceat(ref.astype(np.uint64), voff[:-1]))

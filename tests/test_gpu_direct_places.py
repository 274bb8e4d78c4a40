"""Direct counts by the larger row: entry counts around the 4096 whose owners a
block counts together, with a long row, so that the graph does not go row by
row: tasks of two owners only, and of as many as there are entries."""
from __future__ import annotations

import numpy as np
import pytest

import custingeralg_amd as T
import oracle as O

pytestmark = pytest.mark.gpu

N = 70000


def _csr(rows, entries):
    """Rows {vertex: ids} and a hub's, as long as it takes for so many entries."""
    u = np.concatenate([np.full(len(x), v) for v, x in rows.items()])
    v = np.concatenate(list(rows.values()))
    key = np.unique(u * N + v)
    ids = np.concatenate([np.setdiff1d(np.array(list(rows)), [1]), np.arange(60000, N)])
    hub = entries - len(key)
    assert 129 <= hub <= len(ids)
    key = np.unique(np.concatenate([key, N + ids[:hub]]))
    assert len(key) == entries
    off = np.concatenate([[0], np.cumsum(np.bincount(key // N, minlength=N))]).astype(np.int64)
    return off, (key % N).astype(np.int32)


@pytest.mark.parametrize("entries", [700, 4031, 4095, 4096, 4097, 4159, 8191, 8193, 12288, 20481])
@pytest.mark.parametrize("owners", ["two", "all different"])
def test_places_around_the_tiles(entries, owners):
    rng = np.random.default_rng(entries)
    rest = entries - 400
    if owners == "two":  # rows of two entries, both to vertices with longer rows
        rows = {int(v): np.array([3, 4]) for v in range(10, 10 + rest // 2)}
        for h in (3, 4):
            rows[h] = rng.choice(np.arange(10, 10 + rest // 2), 40, replace=False)
    else:  # rows of two entries, each to a row of three of its own
        few = rest // 8
        a, b = np.arange(10, 10 + few), np.arange(20000, 20000 + 2 * few)
        rows = {int(v): b[2 * i:2 * i + 2] for i, v in enumerate(a)}
        for i, v in enumerate(b):
            w = b[(i // 2 * 2 + 2 + rng.choice(2 * few - 2, 2, replace=False)) % (2 * few)]
            rows[int(v)] = np.concatenate([w, [b[i ^ 1]]])
    off, adj = _csr(rows, entries)
    assert 128 < np.diff(off).max() and np.diff(off).max() * N >= 16 * entries
    ref = O.custinger_count(off, adj)
    g = T.cuStinger(off, adj)
    pv, glob, st = T.static_count(g, T.default_schedule(method=T.METHOD_DIRECT))
    g.close()
    assert st["method_used"] == T.METHOD_DIRECT and sum(st["jobs_bin"]) > 0
    assert np.array_equal(pv, ref) and glob == int(ref.astype(np.uint64).sum()) and ref.any()
    c, tot = T.csr_count_device(off, adj)
    ref = O.csr_count(off, adj)
    assert np.array_equal(c, ref) and tot == int(ref.astype(np.uint64).sum())

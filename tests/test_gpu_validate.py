"""What a graph's validation finds (symmetry, self loops, the largest degree)
against numpy: entry counts around the chunks of 64 and 128, and single entries
moved or taken out of either direction."""
from __future__ import annotations

import numpy as np
import pytest

import custingeralg_amd as T
import oracle as O

pytestmark = pytest.mark.gpu


def _csr(n, keys):
    keys = np.unique(keys)
    off = np.zeros(n + 1, np.int64)
    off[1:] = np.cumsum(np.bincount(keys // n, minlength=n))
    return off, (keys % n).astype(np.int32)


def _keys(off, adj):
    n = len(off) - 1
    return np.repeat(np.arange(n, dtype=np.int64), np.diff(off)) * n + adj


def _check(n, keys):
    off, adj = _csr(n, keys)
    k = np.unique(keys)
    g = T.cuStinger(off, adj)
    info = g.info()
    g.close()
    assert info["symmetric"] == int(np.array_equal(np.sort((k % n) * n + k // n), k))
    assert info["self_loops"] == int((k // n == k % n).sum())
    assert info["max_degree"] == int(np.diff(off).max(initial=0))


@pytest.mark.parametrize("n,pairs", [(2, 1), (70, 32), (70, 64), (40, 65), (300, 511), (5000, 4000), (66000, 300000)])
def test_one_entry_wrong(n, pairs):
    rng = np.random.default_rng(n + pairs)
    u, v = rng.integers(0, n, pairs), np.minimum(rng.integers(0, n, pairs), rng.integers(0, n, pairs))
    u, v = u[u != v], v[u != v]
    if not len(u):
        u, v = np.array([0]), np.array([1])
    keys = np.unique(np.concatenate([u * n + v, v * n + u]))
    _check(n, keys)
    _check(n, np.concatenate([keys, np.arange(0, n, 7, dtype=np.int64) * (n + 1)]))  # self loops
    deg = np.bincount(keys // n, minlength=n)
    a, b = keys // n, keys % n
    lower = deg[b] < deg[a]
    for pick in (np.flatnonzero(lower), np.flatnonzero(~lower), [0], [len(keys) - 1]):
        if len(pick):
            gone = np.delete(keys, pick[len(pick) // 2])
            _check(n, gone)
            if n > 2:  # as many entries as before: another one in its place
                x = int(rng.integers(0, n * n))
                while x in keys or x // n == x % n:
                    x = int(rng.integers(0, n * n))
                _check(n, np.append(gone, x))


@pytest.mark.parametrize("scale", [10, 14])
def test_rmat_and_its_upper_half(scale):
    off, adj = O.rmat_graph(scale, 8, 3)
    keys, n = _keys(off, adj), len(off) - 1
    _check(n, keys)
    _check(n, keys[keys // n < keys % n])
    _check(n, np.empty(0, np.int64))

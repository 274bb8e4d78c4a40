"""Direct counts of graphs whose longest row lies between the small bin's bound
and a little above the middle bin's, against the oracle: all rows above the
small bin's are the largest bin's there."""
from __future__ import annotations

import numpy as np
import pytest

import custingeralg_amd as T
import oracle as O

pytestmark = pytest.mark.gpu


def _rows(n, longest, many, seed):
    """Directed rows: one of the longest length, many of 66 entries up to it, all
    within one set of vertices, and rows of up to three elsewhere."""
    rng = np.random.default_rng(seed)
    top = max(longest + 1, many)
    ids = rng.choice(n, top, replace=False)
    lens = np.concatenate([[longest], rng.integers(min(66, longest), longest + 1, many - 1)])
    if many > 1000:  # as many owners as there can be: 66 entries each
        lens[1:] = 66
    u = np.repeat(ids[:many], lens)
    v = np.concatenate([ids[rng.permutation(top)[:k]] for k in lens])
    bg = rng.integers(0, n, (2, n))
    bg = bg[:, ~np.isin(bg[0], ids[:many])]
    key = np.unique(np.concatenate([u, bg[0]]).astype(np.int64) * n + np.concatenate([v, bg[1]]))
    off = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))]).astype(np.int64)
    return off, (key % n).astype(np.int32)


def _check(off, adj, **sched):
    ref = O.custinger_count(off, adj)
    assert ref.any()
    g = T.cuStinger(off, adj)
    pv, glob, st = T.static_count(g, T.default_schedule(method=T.METHOD_DIRECT, **sched))
    g.close()
    assert np.array_equal(pv, ref) and glob == int(ref.astype(np.uint64).sum())
    return st


@pytest.mark.parametrize("n", [16385, 100000, 1 << 20])
@pytest.mark.parametrize("longest", [129, 300, 512, 513])
def test_longest_row_in_the_middle(n, longest):
    off, adj = _rows(n, longest, 100, longest)
    assert np.diff(off).max() == longest and longest * n >= 16 * len(adj)
    st = _check(off, adj)
    assert st["jobs_bin"][2] > 0
    c, tot = T.csr_count_device(off, adj)
    ref = O.csr_count(off, adj)
    assert np.array_equal(c, ref) and tot == int(ref.astype(np.uint64).sum())


@pytest.mark.parametrize("longest", [65, 100, 400])
def test_learned_policy_on_few_vertices(longest):
    """(the bit matrix takes the default policy only)"""
    off, adj = _rows(5000, longest, 40, longest)
    st = _check(off, adj, policy=T.POLICY_LEARNED)
    assert st["jobs_bin"][2] > 0


def test_more_owners_than_long_rows():
    """14000 rows of 66 entries and one of 600: a job of the largest bin each."""
    off, adj = _rows(200000, 600, 14001, 1)
    st = _check(off, adj)
    assert st["jobs_bin"][2] > 13000

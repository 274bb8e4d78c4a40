"""The delta of long rows (segments of merge positions, hashed bit sets, credits
summed in LDS) against the oracle: list lengths around the group, window and
segment sizes, batches below and above the size that merges shorter rows, and a
vertex credited more often than one slot of the credit table holds."""
from __future__ import annotations

import numpy as np
import pytest

import custingeralg_amd as T
import oracle as O

pytestmark = pytest.mark.gpu


def _insert_and_undo(n, off, adj, bu, bv, slack=0):
    base = O.custinger_count(off, adj)
    ins = np.zeros(len(bu), np.uint8)
    want_off, want_adj = O.apply_batch_csr(n, off, adj, ins_u=bu, ins_v=bv,
                                           del_u=np.zeros(0, np.int32), del_v=np.zeros(0, np.int32))
    now = O.custinger_count(want_off, want_adj)
    change = int(now.astype(np.uint64).sum()) - int(base.astype(np.uint64).sum())
    g = T.cuStinger(off, adj, slack_pct=slack)
    delta = T.DeviceArray(n, np.uint32).zero()
    dg, _ = T.batch_apply(g, bu, bv, ins, delta)
    assert np.array_equal(base + delta.to_host(), now)
    assert dg == change
    dg, _ = T.batch_apply(g, bu, bv, 1 - ins, delta)
    assert dg == -change
    assert not delta.to_host().any()
    got_off, got_adj = g.to_csr()
    assert np.array_equal(got_off, off) and np.array_equal(got_adj, adj)
    g.close()


def _new_pairs(n, off, adj, u, v):
    lo, hi = np.minimum(u, v).astype(np.int64), np.maximum(u, v)
    key = np.unique((lo * n + hi)[lo != hi])
    rows = np.repeat(np.arange(n, dtype=np.int64), np.diff(off))
    key = np.setdiff1d(key, rows * n + adj)
    return (key // n).astype(np.int32), (key % n).astype(np.int32)


@pytest.mark.parametrize("slack", [0, 60])
@pytest.mark.parametrize("lens", [[15, 16, 17, 63, 64, 65, 66], [127, 128, 129, 130, 255, 257, 511],
                                  [126, 128, 4095, 4096, 4097, 8192, 8300], [30, 130, 900, 6000, 12000]])
def test_rows_around_the_limits(lens, slack):
    n, hubs = 20000, 84
    rng = np.random.default_rng(sum(lens) + slack)
    want = np.array([lens[i % len(lens)] for i in range(hubs)])
    ids = rng.permutation(n).astype(np.int32)
    u, v = [], []
    for i in range(hubs):  # neighbours that the hubs have in common more often than not
        pool = ids[hubs:hubs + max(want[i], (3 * want[i]) // 2 if i % 3 else want[i])]
        u.append(np.full(want[i], ids[i], np.int32))
        v.append(rng.choice(pool, want[i], replace=False))
    off, adj = O.canon_csr(n, np.concatenate(u), np.concatenate(v))
    a, b = np.triu_indices(hubs, 1)
    bu, bv = _new_pairs(n, off, adj, ids[a], ids[b])
    assert len(bu) > 1024
    _insert_and_undo(n, off, adj, bu, bv, slack)


@pytest.mark.parametrize("n,deg,pairs", [(3000, 100, 60000), (3000, 90, 150000)])
def test_many_pairs_of_rows_alike(n, deg, pairs):
    rng = np.random.default_rng(pairs)
    off, adj = O.canon_csr(n, rng.integers(0, n, n * deg // 2).astype(np.int32),
                           rng.integers(0, n, n * deg // 2).astype(np.int32))
    bu, bv = _new_pairs(n, off, adj, rng.integers(0, n, pairs), rng.integers(0, n, pairs))
    _insert_and_undo(n, off, adj, bu, bv)


def test_one_vertex_in_every_list():
    """A million new edges whose ends all have vertex 7: its credits fill and
    drain its slot of every block's table."""
    n = 2500
    rng = np.random.default_rng(4)
    off, adj = O.canon_csr(n, np.concatenate([np.full(n, 7), rng.integers(0, n, 90 * n)]).astype(np.int32),
                           np.concatenate([np.arange(n), rng.integers(0, n, 90 * n)]).astype(np.int32))
    a, b = np.triu_indices(n, 1)
    keep = rng.random(len(a)) < 0.45
    bu, bv = _new_pairs(n, off, adj, a[keep], b[keep])
    assert len(bu) > 1_000_000
    _insert_and_undo(n, off, adj, bu, bv)


@pytest.mark.parametrize("pairs", [1, 2, 31, 63, 64, 65, 127, 128, 129, 256, 257, 511, 513, 1023, 1024])
@pytest.mark.parametrize("capture", [0, 1])
def test_small_batches_of_every_sort_size(pairs, capture):
    """Batches whose pairs, and whose directed entries, fill the one-block sort
    up to and past each power of two."""
    n = 3000
    rng = np.random.default_rng(pairs)
    off, adj = O.canon_csr(n, rng.integers(0, n, 9 * n).astype(np.int32), rng.integers(0, n, 9 * n).astype(np.int32))
    bu, bv = _new_pairs(n, off, adj, rng.integers(0, n, 4 * pairs + 8), rng.integers(0, n, 4 * pairs + 8))
    pick = rng.permutation(len(bu))[:pairs]
    bu, bv = np.ascontiguousarray(bu[pick]), np.ascontiguousarray(bv[pick])
    base = O.custinger_count(off, adj)
    want_off, want_adj = O.apply_batch_csr(n, off, adj, ins_u=bu, ins_v=bv,
                                           del_u=np.zeros(0, np.int32), del_v=np.zeros(0, np.int32))
    now = O.custinger_count(want_off, want_adj)
    g = T.cuStinger(off, adj, slack_pct=100)
    sched = T.default_schedule(capture=capture)
    ins = np.zeros(pairs, np.uint8)
    delta = T.DeviceArray(n, np.uint32).zero()
    for _ in range(3 if capture else 1):
        T.batch_apply(g, bu, bv, ins, delta, sched)
        assert np.array_equal(base + delta.to_host(), now)
        got_off, got_adj = g.to_csr()
        assert np.array_equal(got_off, want_off) and np.array_equal(got_adj, want_adj)
        T.batch_apply(g, bu, bv, 1 - ins, delta, sched)
        assert not delta.to_host().any()
        got_off, got_adj = g.to_csr()
        assert np.array_equal(got_off, off) and np.array_equal(got_adj, adj)
    g.close()


@pytest.mark.parametrize("slack", [0, 100])
def test_small_batches_into_rows_of_several_chunks(slack):
    """Rows around the length that several blocks merge and around their chunks,
    with new entries first, last and at chunk borders, in place and moved, more of
    them than the copies have room for."""
    n = 80000
    rng = np.random.default_rng(slack)
    lens = [8191, 8192, 8193, 12287, 12288, 12289, 40000, 66000] + [8193] * 40
    hubs = np.arange(100, 100 + len(lens))
    u, v = [], []
    for h, k in zip(hubs, lens):
        cand = rng.permutation(np.arange(200, n - 200))[:k]
        u.append(np.full(k, h))
        v.append(cand)
    off, adj = O.canon_csr(n, np.concatenate(u).astype(np.int32), np.concatenate(v).astype(np.int32))
    pu, pv = [], []
    for h in hubs:
        row = adj[off[h]:off[h + 1]]
        near = [0, 1, n - 1, n - 2] + [int(row[q]) + 1 for q in (4094, 4095, 4096, 8190) if q < len(row)]
        near += list(rng.integers(0, n, 6))
        pu += [h] * len(near)
        pv += near
    bu, bv = _new_pairs(n, off, adj, np.array(pu), np.array(pv))
    bu, bv = bu[:1024], bv[:1024]
    _insert_and_undo(n, off, adj, bu, bv, slack)

"""The oriented count's core (the highest ranks on a bit matrix) against the
oracle: sizes at its smallest graph, core rows of every length around the
group and wave limits, and rows declared symmetric that are not."""
from __future__ import annotations

import numpy as np
import pytest

import custingeralg_amd as T
import oracle as O

pytestmark = pytest.mark.gpu


def _planted(n, hubs, seed, dense=0.05):
    """hubs vertices of a random graph among themselves, every other vertex
    joined to 0, 1, 2, ... 40 of them in turn, and a sparse background."""
    rng = np.random.default_rng(seed)
    ids = rng.permutation(n).astype(np.int32)
    m = int(dense * hubs * hubs / 2)
    hu, hv = rng.integers(0, hubs, m), rng.integers(0, hubs, m)
    k = np.arange(n - hubs) % 41
    lu = np.repeat(np.arange(hubs, n), k)
    lv = (rng.pareto(0.6, len(lu)) * hubs / 40).astype(np.int64) % hubs
    bu, bv = rng.integers(0, n, n), rng.integers(0, n, n)
    u, v = np.concatenate([hu, lu, bu]), np.concatenate([hv, lv, bv])
    return O.canon_csr(n, ids[u], ids[v])


def _check(off, adj, **kw):
    ref = O.custinger_count(off, adj)
    g = T.cuStinger(off, adj)
    for method in (T.METHOD_AUTO, T.METHOD_ORIENTED):
        pv, glob, st = T.static_count(g, T.default_schedule(method=method, **kw))
        assert st["method_used"] == T.METHOD_ORIENTED
        assert np.array_equal(pv, ref)
        assert glob == int(ref.astype(np.uint64).sum())
    g.close()


@pytest.mark.parametrize("n", [16385, 16999, 40003])
@pytest.mark.parametrize("hubs", [300, 5000])
def test_planted(n, hubs):
    _check(*_planted(n, hubs, n))


@pytest.mark.parametrize("scale,ef", [(15, 3), (17, 24)])
def test_rmat(scale, ef):
    _check(*O.rmat_graph(scale, ef, 11))
    _check(*O.rmat_graph(scale, ef, 12), policy=T.POLICY_LEARNED)


@pytest.mark.parametrize("kw", [dict(job_items=64), dict(job_items=1 << 20), dict(small_max=16, mid_max=64),
                                dict(policy=T.POLICY_MERGE), dict(policy=T.POLICY_HASH)])
def test_owners_in_one_and_several_jobs(kw):
    """Third-vertex counts of core vertices, stored by an owner's only job and
    added by several."""
    _check(*_planted(20000, 600, 3), **kw)
    _check(*O.rmat_graph(15, 16, 13), **kw)


def test_recorded_counts():
    off, adj = _planted(20000, 600, 5)
    ref = O.custinger_count(off, adj)
    g = T.cuStinger(off, adj)
    out = T.DeviceArray(g.nv, np.uint32)
    sched = T.default_schedule(capture=1)
    for k in range(4):
        _, glob, st = T.static_count(g, sched, out=out)
        assert np.array_equal(out.to_host(), ref) and glob == int(ref.astype(np.uint64).sum())
        assert st["graph_replay"] == (k > 0)
    out.free()
    g.close()


def test_declared_symmetric_with_balanced_faults():
    """One entry into a core vertex moved to another core vertex: every total
    still fits, the per-vertex counts of entries do not."""
    off, adj = _planted(20000, 600, 7)
    deg = np.diff(off)
    h1, h2 = (int(x) for x in np.argsort(deg)[-2:])
    for a in range(len(deg)):  # a leaf that points to h1 and not to h2
        row = adj[off[a]:off[a + 1]]
        if 2 < len(row) < 40 and h1 in row and h2 not in row:
            break
    new = np.sort(np.where(row == h1, h2, row))
    adj2 = adj.copy()
    adj2[off[a]:off[a + 1]] = new
    ref = O.custinger_count(off, adj2)
    g = T.cuStinger(off, adj2, assume_symmetric=True)
    with pytest.raises(T.TCError):
        T.static_count(g, T.default_schedule(method=T.METHOD_ORIENTED))
    pv, glob, st = T.static_count(g)
    g.close()
    assert st["method_used"] == T.METHOD_DIRECT
    assert np.array_equal(pv, ref) and glob == int(ref.astype(np.uint64).sum())


@pytest.mark.parametrize("sizes", [[20000, 1, 3, 5000], [4096, 17000, 2, 4097, 2048, 2049] * 3])
def test_batched_cores(sizes):
    """Graphs with their cores behind all other ranks, some all core."""
    voff = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    us, vs = [], []
    for i, n in enumerate(sizes):
        if n < 16:
            continue
        off, adj = _planted(n, n // 8, i, 0.1)
        us.append(np.repeat(np.arange(n), np.diff(off)) + voff[i])
        vs.append(adj + voff[i])
    nv = int(voff[-1])
    off, adj = O.canon_csr(nv, np.concatenate(us).astype(np.int32),
                           np.concatenate(vs).astype(np.int32))
    ref = O.custinger_count(off, adj)
    want = np.add.reduceat(ref.astype(np.uint64), voff[:-1])
    dv, do, da = (T.DeviceArray.from_host(x) for x in (voff, off, adj))
    bg = T.BatchedGraph(dv, do, da)
    pg, pv = T.DeviceArray(len(sizes), np.uint64), T.DeviceArray(nv, np.uint32)
    for sched in (None, T.default_schedule(policy=T.POLICY_HASH), T.default_schedule(capture=1),
                  T.default_schedule(capture=1), T.default_schedule(capture=1)):
        bg.count(pg, pv, sched)
        assert np.array_equal(pv.to_host(), ref)
        assert np.array_equal(pg.to_host(), want)
    bg.close()


def test_rows_of_129_to_512_in_the_largest_bin():
    """A graph large enough that rows of the middle bin's lengths near the top of
    the rank order go to the largest one: schedules that bin them otherwise
    agree."""
    off, adj = O.rmat_graph(21, 16, 5)
    assert len(adj) >= 3 << 24
    g = T.cuStinger(off, adj, assume_symmetric=True)
    a, ga, sa = T.static_count(g, T.default_schedule())
    b, gb, sb = T.static_count(g, T.default_schedule(mid_max=128))
    h, gh, _ = T.static_count(g, T.default_schedule(policy=T.POLICY_HASH))
    m, gm, _ = T.static_count(g, T.default_schedule(mpath_min=1 << 20))  # (kept in the middle bin)
    g.close()
    for x, gx in ((b, gb), (h, gh), (m, gm)):
        assert np.array_equal(a, x) and ga == gx
    assert int(a.astype(np.uint64).sum()) == ga
    assert sum(sa["tasks_bin"]) == sum(sb["tasks_bin"]) and 0 < sa["tasks_bin"][2] <= sb["tasks_bin"][2]
    total, _ = O.forward_count(off, adj)
    assert ga == 6 * total


def test_core_of_the_largest_graphs():
    """From 200M entries on the core has 8192 ranks; a forced policy has none."""
    g = T.rmat_graph_device(22, 28, 7)
    assert g.info()["nnz"] >= 3 << 26
    a, ga, _ = T.static_count(g, T.default_schedule())
    h, gh, _ = T.static_count(g, T.default_schedule(policy=T.POLICY_HASH))
    g.close()
    assert np.array_equal(a, h) and ga == gh
    assert ga % 6 == 0

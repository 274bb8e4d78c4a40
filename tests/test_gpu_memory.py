"""Counts whose bit matrix, core or direct task lists find no memory take the
routes that need none of them, with the same results."""
from __future__ import annotations

import contextlib

import numpy as np
import pytest

import custingeralg_amd as T
import oracle as O

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def _limit(nbytes):
    """No device block above nbytes for this thread."""
    import ctypes as C
    T.lib().tc_test_block_limit(C.c_uint64(nbytes))
    try:
        yield
    finally:
        T.lib().tc_test_block_limit(C.c_uint64(0))


def _graph(n, m, hub, seed, sym=True):
    rng = np.random.default_rng(seed)
    u = np.concatenate([rng.integers(0, n, m), np.repeat(rng.choice(n, 8), hub)])
    v = np.concatenate([rng.integers(0, n, m), rng.integers(0, n, 8 * hub)])
    if sym:
        return O.canon_csr(n, u.astype(np.int32), v.astype(np.int32))
    key = np.unique(u * n + v)
    off = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))]).astype(np.int64)
    return off, (key % n).astype(np.int32)


def _both(off, adj, limit, **sched):
    """The same handle's counts without and under the limit, three times each."""
    ref = O.custinger_count(off, adj)
    g = T.cuStinger(off, adj)
    got = []
    for lim in (0, limit):
        with _limit(lim):
            for _ in range(3):
                pv, glob, st = T.static_count(g, T.default_schedule(**sched))
                assert np.array_equal(pv, ref) and glob == int(ref.astype(np.uint64).sum())
        got.append(st)
        g.close()
        g = T.cuStinger(off, adj)
    g.close()
    return got


@pytest.mark.parametrize("capture", [0, 1])
def test_bit_matrix(capture):
    wide, lean = _both(*_graph(9000, 40000, 400, 1), 4 << 20, capture=capture)  # 10 MB of bit rows
    assert sum(wide["tasks_bin"]) == 0 and sum(lean["tasks_bin"]) > 0


@pytest.mark.parametrize("capture", [0, 1])
def test_core(capture):
    wide, lean = _both(*_graph(17500, 40000, 1500, 2), 3 << 19, capture=capture)  # 2 MB of bit rows
    assert 0 < sum(wide["tasks_bin"]) < sum(lean["tasks_bin"])


def test_direct_task_lists():
    wide, lean = _both(*_graph(20000, 480000, 800, 3, sym=False), 3 << 20, method=T.METHOD_DIRECT)
    assert wide["method_used"] == lean["method_used"] == T.METHOD_DIRECT


@pytest.mark.parametrize("sizes,limit", [([9000, 300], 4 << 20), ([17000, 300, 4000], 1 << 20)])
def test_batched(sizes, limit):
    voff = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    offs, adjs = [np.zeros(1, np.int64)], []
    for i, n in enumerate(sizes):
        off, adj = _graph(n, 3 * n, n // 20, i)
        offs.append(off[1:] + offs[-1][-1])
        adjs.append(adj + int(voff[i]))
    off, adj = np.concatenate(offs), np.concatenate(adjs).astype(np.int32)
    ref = O.custinger_count(off, adj)
    want = np.add.reduceat(ref.astype(np.uint64), voff[:-1])
    d = [T.DeviceArray.from_host(x) for x in (voff, off, adj)]
    pg, pv = T.DeviceArray(len(sizes), np.uint64), T.DeviceArray(int(voff[-1]), np.uint32)
    tasks = []
    for lim in (0, limit):
        bg = T.BatchedGraph(*d)
        with _limit(lim):
            for _ in range(2):
                st = bg.count(pg, pv)
                assert np.array_equal(pv.to_host(), ref) and np.array_equal(pg.to_host(), want)
        tasks.append(sum(st["tasks_bin"]))
        bg.close()
    assert tasks[0] < tasks[1]

"""Rules that kernels and host share, on the host: the capacities of the job
arrays against the jobs that the planner's rule gives, with row lengths around
every bin's bounds, in each mode; the entries that a bit-row count loads."""
from __future__ import annotations

import ctypes as C
import os

import numpy as np
import pytest

import custingeralg_amd as T
import oracle as O

_LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "libplan_test.so")
DIRECT, ORIENTED, BY_TASKS = 0, 1, 2


def _plan(mode, off, adj, skip_lower=0, **sched):
    lib = C.CDLL(_LIB)
    s = T.default_schedule(**sched)
    jobs, caps = (C.c_int64 * 3)(), (C.c_int64 * 3)()
    off, adj = np.ascontiguousarray(off, np.int64), np.ascontiguousarray(adj, np.int32)
    lib.plan_probe(C.c_int32(mode), C.byref(s), C.c_int32(len(off) - 1), C.c_void_p(off.ctypes.data),
                   C.c_void_p(adj.ctypes.data), C.c_int32(skip_lower), jobs, caps)
    return list(jobs), list(caps)


def _rows(n, lens, seed, sym=False):
    """Rows of the given lengths at the first vertices, their entries drawn from the
    first 2 len(lens) vertices or more, and short rows elsewhere."""
    rng = np.random.default_rng(seed)
    top = max(max(lens) + 1, 2 * len(lens))
    rows = [rng.permutation(min(top, n))[:k] for k in lens]
    u = np.concatenate([np.full(len(r), i) for i, r in enumerate(rows)] + [np.arange(len(lens), n)] * 2)
    v = np.concatenate(rows + [rng.integers(0, n, n - len(lens)) for _ in range(2)])
    if sym:
        return O.canon_csr(n, u.astype(np.int32), v.astype(np.int32))
    key = np.unique(u * n + v)
    off = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))]).astype(np.int64)
    return off, (key % n).astype(np.int32)


@pytest.mark.parametrize("mode", [DIRECT, ORIENTED, BY_TASKS])
@pytest.mark.parametrize("longest", [63, 64, 65, 66, 127, 129, 300, 511, 512, 513, 600, 4095, 4097, 9000])
@pytest.mark.parametrize("many", [66, 129])
def test_every_job_has_room(mode, longest, many):
    """One row of the longest length, many of a bin's least, as the planner meets
    them: a job for every owner at least."""
    n = 9000
    lens = [longest] + [min(many, longest)] * 1200
    off, adj = _rows(n, lens, longest, mode == ORIENTED)
    for skip in (0, 1):
        for kw in ({}, {"policy": T.POLICY_LEARNED}, {"small_max": 1, "mid_max": 1}, {"small_max": 8, "mid_max": 40},
                   {"job_items": 1, "flush_items": 1}, {"mid_max": 128}):
            jobs, caps = _plan(mode, off, adj, skip, **kw)
            assert all(j <= c for j, c in zip(jobs, caps)), (kw, jobs, caps)
            assert sum(jobs) > 0


@pytest.mark.parametrize("n", [16385, 200000, (1 << 20) + 1])
def test_many_middle_rows_and_one_longer(n):
    """Directed rows, most of 66 entries: their owners all get jobs of the largest
    bin where there is no middle one."""
    lens = [600] + [66] * min(5000, n // 4)
    off, adj = _rows(n, lens, 7)
    jobs, caps = _plan(BY_TASKS, off, adj)
    assert all(j <= c for j, c in zip(jobs, caps)), (jobs, caps)
    assert max(jobs[1], jobs[2]) > len(lens) // 2


@pytest.mark.parametrize("check_sym", [0, 1])
@pytest.mark.parametrize("unroll", [1, 2, 4])
def test_bit_rows_load_their_own_entries(check_sym, unroll):
    """No place outside the row, and every row of two entries or more is loaded."""
    lib = C.CDLL(_LIB)
    for d in range(200):
        lo, hi = C.c_int32(), C.c_int32()
        lib.dense_probe(C.c_int32(d), C.c_int32(check_sym), C.c_int32(unroll), C.byref(lo), C.byref(hi))
        assert lo.value == 0 and hi.value < d, d
        assert d < 2 or hi.value == d - 1


@pytest.mark.parametrize("graphs,n,nnz,pays", [
    # batches that were measured on both routes, the bit rows' time over the lists'
    (65, 1000, 425986, True),       # 0.3
    (524, 1000, 18218546, True),    # 0.6
    (128, 4000, 3588152, True),     # 0.6
    (2, 16384, 1553072, True),      # 0.4
    (31, 16384, 3719342, False),    # 2.3
    (31, 16384, 24092252, False),   # 3.6
    (128, 8000, 3830094, False),    # 1.9
    (512, 4000, 48571398, False),   # 1.7
    (8192, 1000, 28818864, False),  # 1.4
])
def test_batches_on_bit_rows(graphs, n, nnz, pays):
    """Bytes of bit rows written and read, and the entries, decide together."""
    row = (n + 1023) // 1024 * 128
    lib = C.CDLL(_LIB)
    assert bool(lib.dense_batch_probe(C.c_int64(graphs * n * row), C.c_int64(nnz * row), C.c_int64(graphs * n),
                                      C.c_int64(nnz))) == pays


@pytest.mark.parametrize("nv,nnz,longest,pays", [
    # graphs that were measured on both routes, row by row over oriented
    (65536, 1048000, 40, True),       # 0.1
    (1000000, 1850000, 113, True),    # 0.7
    (3000000, 11900000, 93, False),   # 0.96
    (2000000, 7900000, 94, True),     # 0.9
    (8000000, 14800000, 118, False),  # 1.6
    (8000000, 31600000, 101, False),  # 1.2
    (4000000, 26500000, 48, True),    # 0.7
    (65536, 1048000, 129, False),
    (65536, 2700000, 60, False),
])
def test_rows_one_by_one(nv, nnz, longest, pays):
    lib = C.CDLL(_LIB)
    assert bool(lib.rows_probe(C.c_int32(nv), C.c_int64(nnz), C.c_int32(longest))) == pays

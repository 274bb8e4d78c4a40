"""Recorded counts of graphs above the bit matrix's size, whose sequence is
planned: with other counts between the replays, which may move the handle's
buffers."""
from __future__ import annotations

import numpy as np
import pytest

import custingeralg_amd as T
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture
def graph():
    rng = np.random.default_rng(5)
    n = 20011
    u = np.concatenate([rng.integers(0, n, 8 * n), np.repeat(rng.choice(n, 30), 2000)])
    v = np.concatenate([rng.integers(0, n, 8 * n), rng.integers(0, n, 60000)])
    off, adj = O.canon_csr(n, u.astype(np.int32), v.astype(np.int32))
    ref = O.custinger_count(off, adj)
    g = T.cuStinger(off, adj)
    out = T.DeviceArray(n, np.uint32)

    def count(**sched):
        T.check(T.lib().tc_memset(out.ptr, 0xFF, out.nbytes))
        _, glob, st = T.static_count(g, T.default_schedule(**sched), out=out)
        assert np.array_equal(out.to_host(), ref) and glob == int(ref.astype(np.uint64).sum())
        return st

    yield count
    out.free()
    g.close()


def test_replay_after_a_count_that_moved_buffers(graph):
    """The direct method's task lists are twice the oriented ones: a recording
    made before them is not replayed."""
    rec = dict(method=T.METHOD_AUTO, capture=1)
    assert [graph(**rec)["graph_replay"] for _ in range(3)] == [0, 1, 1]
    assert graph(method=T.METHOD_DIRECT)["method_used"] == T.METHOD_DIRECT
    st = graph(**rec)
    assert st["graph_replay"] == 0 and st["method_used"] == T.METHOD_ORIENTED
    assert [graph(**rec)["graph_replay"] for _ in range(2)] == [1, 1]
    # now everything is large enough: the recording stands, and its method
    graph(method=T.METHOD_DIRECT)
    st = graph(**rec)
    assert st["graph_replay"] == 1 and st["method_used"] == T.METHOD_ORIENTED


@pytest.mark.parametrize("method", [T.METHOD_AUTO, T.METHOD_DIRECT])
def test_planned_sequence_replays(graph, method):
    for items in (8192, 2048):
        st = [graph(method=method, capture=1, job_items=items) for _ in range(4)]
        assert [x["graph_replay"] for x in st] == [0, 1, 1, 1]
        assert sum(st[0]["jobs_bin"]) > 0 and all(x["jobs_bin"] == st[0]["jobs_bin"] for x in st)

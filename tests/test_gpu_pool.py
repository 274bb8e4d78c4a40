"""Handles made and released over and over take their blocks from the pool:
counts stay exact from several threads at once, with updates in between."""
from __future__ import annotations

import ctypes as C
import threading

import numpy as np
import pytest

import custingeralg_amd as T
import oracle as O

pytestmark = pytest.mark.gpu


def test_handles_from_several_threads():
    graphs = [O.rmat_graph(s, ef, s) for s, ef in ((8, 4), (11, 9), (14, 8), (15, 5))]
    refs = [O.custinger_count(*g) for g in graphs]
    faults = []

    def work(k):
        try:
            for i in range(6):
                j = (k + i) % len(graphs)
                off, adj = graphs[j]
                g = T.cuStinger(off, adj, assume_symmetric=i % 2 == 0)
                pv, _, _ = T.static_count(g)
                u, v = np.array([3, 5], np.int32), np.array([201, 202], np.int32)
                T.batch_apply(g, u, v)
                o2, a2 = g.to_csr()
                pv2, _, _ = T.static_count(g)
                g.close()
                if not np.array_equal(pv, refs[j]) or not np.array_equal(pv2, O.custinger_count(o2, a2)):
                    faults.append((k, i))
        except Exception as e:  # noqa: BLE001
            faults.append((k, repr(e)))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not faults


def test_trim_gives_the_blocks_back():
    """A closed handle's blocks stay with the library until they are asked for."""

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert T.lib().hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    T.device_trim()
    free0 = free()
    off, adj = O.rmat_graph(17, 24, 3)
    g = T.cuStinger(off, adj)
    pv, _, _ = T.static_count(g)
    held = free0 - free()
    assert held > 100 << 20
    g.close()
    assert free0 - free() > held // 2
    T.device_trim()
    # (what the runtime keeps for itself: code objects, small blocks)
    assert free0 - free() < held // 4
    g = T.cuStinger(off, adj)
    again, _, _ = T.static_count(g)
    g.close()
    assert np.array_equal(pv, again)

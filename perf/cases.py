"""Timed workloads of the triangle-counting engine.

Each case is one call (or one pair of calls) a user's program makes: a static
count of a graph in the store, a count of a graph that has just arrived, a
count of a directed graph, a count of a raw CSR, an update batch with its
delta, and a count of many small graphs at once.  Graphs are R-MAT
(0.57, 0.19, 0.19, 0.05) or uniform pairs, symmetrised, deduplicated and
loop-free, the two families of this repository's benchmark and tests; all of
them come from the seed alone.  Per-vertex counts are uint32 on the device and
are returned as int32 tensors of the same bits.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import custingeralg_amd as T

_RMAT = (0.57, 0.19, 0.19)
_CHUNK = 1 << 26
_EXACT_WEDGES = 200_000_000  # exact() enumerates at most this many (v, u, w)


class _Buf:
    """A torch tensor in the shape the package's calls take device arrays."""

    def __init__(self, t):
        self.t = t
        self.ptr = t.data_ptr() if t.numel() else None
        self.n = t.numel()


def listed():
    return [
        # the smallest call: a graph of a thousand vertices, all latency
        {"name": "static_1k", "op": "static", "kind": "rmat", "n": 1000, "ef": 8, "pv": True},
        # the uniform graph of the benchmark's smallest configuration: short rows, no hubs
        {"name": "static_er_64k", "op": "static", "kind": "er", "n": 65536, "ef": 8, "pv": True},
        # an ordinary power-law graph, the benchmark's middle configuration
        {"name": "static_rmat20", "op": "static", "kind": "rmat", "n": 1 << 20, "ef": 16, "pv": True},
        # an odd vertex count, between the powers of two
        {"name": "static_odd_3m", "op": "static", "kind": "rmat", "n": 2999999, "ef": 24, "pv": True},
        # the largest: the benchmark's headline graph, a billion entries
        {"name": "static_rmat24", "op": "static", "kind": "rmat", "n": 1 << 24, "ef": 32, "pv": True},
        # a graph that has just arrived: store built and validated, counted once, released
        {"name": "new_graph_250k", "op": "new", "kind": "rmat", "n": 250007, "ef": 16, "pv": True},
        # a directed graph, which only the per-entry formula counts
        {"name": "directed_256k", "op": "directed", "kind": "rmat", "n": 1 << 18, "ef": 16, "pv": True},
        # the raw-CSR call (each entry to a higher id), no store kept
        {"name": "csr_100k", "op": "csr", "kind": "rmat", "n": 100003, "ef": 12, "pv": True},
        # a thousand-pair update of a large graph, recorded as the benchmark does, and its undoing
        {"name": "stream_1k", "op": "stream", "kind": "rmat", "n": 1 << 22, "ef": 16, "pairs": 1000,
         "capture": True},
        # a million-pair update of the same graph, and its undoing
        {"name": "stream_1m", "op": "stream", "kind": "rmat", "n": 1 << 22, "ef": 16,
         "pairs": 1000000, "capture": False},
        # a few dozen small graphs in one call: a serving batch
        {"name": "batched_48", "op": "batched", "graphs": 48, "nmin": 500, "nmax": 6000, "efmin": 4,
         "efmax": 16, "pv": True},
        # a thousand graphs of 1k to 64k vertices, the distribution of the benchmark's batch
        {"name": "batched_1024", "op": "batched", "graphs": 1024, "nmin": 1024, "nmax": 65536,
         "efmin": 4, "efmax": 32, "pv": True},
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["static", "static", "static", "new", "directed", "csr", "stream", "stream",
                     "batched"])
    kind = rng.choice(["rmat", "rmat", "rmat", "er"])
    ef = _logu(rng, 4, 32)
    if op == "batched":
        nmin = _logu(rng, 200, 4000)
        return {"op": op, "graphs": _logu(rng, 8, 512), "nmin": nmin,
                "nmax": nmin * rng.randint(1, 12) + rng.randint(0, 999), "efmin": 4,
                "efmax": max(ef, 4), "pv": rng.random() < 0.5}
    if op == "stream":
        n = _logu(rng, 1 << 14, 1 << 22)
        return {"op": op, "kind": kind, "n": n, "ef": min(ef, 16),
                "pairs": _logu(rng, 20, max(40, min(1000000, n // 4))), "capture": rng.random() < 0.5}
    top = {"static": 1 << 22, "new": 1 << 20, "directed": 1 << 19, "csr": 1 << 18}[op]
    return {"op": op, "kind": kind, "n": _logu(rng, 300, top), "ef": ef,
            "pv": op != "static" or rng.random() < 0.75}


# ------------------------------------------------------------------ inputs
def _rmat(gen, scale, m):
    """m R-MAT pairs of 2^scale vertices as two int32 device tensors."""
    a, ab, abc = _RMAT[0], _RMAT[0] + _RMAT[1], sum(_RMAT)
    u = torch.empty(m, dtype=torch.int32, device="cuda")
    v = torch.empty(m, dtype=torch.int32, device="cuda")
    for s in range(0, m, _CHUNK):
        k = min(_CHUNK, m - s)
        x = torch.zeros(k, dtype=torch.int32, device="cuda")
        y = torch.zeros(k, dtype=torch.int32, device="cuda")
        for _ in range(scale):
            r = torch.rand(k, generator=gen, device="cuda")
            x.mul_(2).add_(r >= ab)
            y.mul_(2).add_(((r >= a) & (r < ab)) | (r >= abc))
        u[s:s + k], v[s:s + k] = x, y
    return u, v


def _pairs(gen, kind, n, m):
    """m pairs over n vertices; an R-MAT pair with an endpoint >= n is dropped later."""
    if kind == "er":
        return tuple(torch.randint(0, n, (m,), generator=gen, device="cuda", dtype=torch.int32)
                     for _ in range(2))
    return _rmat(gen, max(1, (n - 1).bit_length()), m)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1_000_003 * (int(seed) + 1))
    return g


def _directed_csr(n, u, v):
    """Sorted, deduplicated rows of the pairs as given, loops dropped (int64 off, int32 adj)."""
    ok = (u != v) & (u < n) & (v < n)
    key = torch.unique(u[ok].long() * n + v[ok].long())
    off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    off[1:] = torch.cumsum(torch.bincount(key // n, minlength=n), 0)
    return off, (key % n).int()


def _graph_csr(n, u, v):
    """The same pairs symmetrised by the package: (off, adj) DeviceArrays."""
    return T.canon_csr_device(n, _Buf(u), _Buf(v))


def _batch_sizes(case):
    r = np.random.default_rng([case["graphs"], case["nmin"], case["nmax"], case["efmax"]])
    lo, hi = math.log(case["nmin"]), math.log(case["nmax"] + 1)
    n = np.minimum(np.exp(r.uniform(lo, hi, case["graphs"])).astype(np.int64), case["nmax"])
    return n, r.integers(case["efmin"], case["efmax"] + 1, case["graphs"])


def _batched_pairs(case, seed):
    """Pairs of all graphs, ids made global: (voff int64 tensor, u, v).  The top k
    levels of an R-MAT draw are an R-MAT draw of 2^k vertices."""
    n, ef = _batch_sizes(case)
    voff = torch.from_numpy(np.concatenate([[0], np.cumsum(n)])).cuda()
    scale = max(1, int(case["nmax"] - 1).bit_length())
    m = int((n * ef).sum())
    u, v = _rmat(_gen(seed), scale, m)
    cut = torch.from_numpy(np.array([scale - max(1, int(x - 1).bit_length()) for x in n], np.int32)).cuda()
    nn = torch.from_numpy(n.astype(np.int32)).cuda()
    first = torch.from_numpy(np.cumsum(n * ef)).cuda()  # end of each graph's pairs
    for s in range(0, m, _CHUNK):
        e = min(m, s + _CHUNK)
        g = torch.searchsorted(first, torch.arange(s, e, device="cuda"), right=True)
        x, y = u[s:e] >> cut[g], v[s:e] >> cut[g]
        ok = (x < nn[g]) & (y < nn[g])
        base = voff[g].int()
        u[s:e], v[s:e] = torch.where(ok, x, 0) + base, torch.where(ok, y, 0) + base
    return voff, u, v


def _update(case, gen, off, adj):
    """An update batch: 80% insertions of absent pairs (half uniform, half R-MAT),
    20% deletions of present ones; canonical, distinct (int32 u, v, uint8 is_delete)."""
    n, b = case["n"], case["pairs"]
    nins = max(1, int(0.8 * b))
    ndel = max(1, b - nins)

    def keys(x, y):
        ok = (x != y) & (x < n) & (y < n)
        x, y = x[ok].long(), y[ok].long()
        return torch.minimum(x, y) * n + torch.maximum(x, y)

    uu, uv = _pairs(gen, "er", n, nins // 2 + 1)
    ru, rv = _pairs(gen, case["kind"], n, nins - nins // 2)
    ins = torch.unique(torch.cat([keys(uu, uv), keys(ru, rv)]))
    e = torch.randint(0, adj.numel(), (ndel,), generator=gen, device="cuda")
    src = torch.searchsorted(off, e, right=True) - 1
    dele = torch.unique(keys(src.int(), adj[e]))
    # drop the insertions already present: the row of u, searched for v
    iu, iv = ins // n, ins % n
    lo, hi = off[iu].clone(), off[iu + 1].clone()
    end = hi.clone()
    for _ in range(32):
        mid = (lo + hi) // 2
        less = (lo < hi) & (adj[mid.clamp(max=adj.numel() - 1)] < iv)
        lo, hi = torch.where(less, mid + 1, lo), torch.where(less, hi, torch.minimum(hi, mid))
    present = (lo < end) & (adj[lo.clamp(max=adj.numel() - 1)] == iv)
    ins = ins[~present]
    k = torch.cat([ins, dele])
    d = torch.zeros(k.numel(), dtype=torch.uint8, device="cuda")
    d[ins.numel():] = 1
    return (k // n).int().contiguous(), (k % n).int().contiguous(), d


def prepare(case, seed):
    op = case["op"]
    if op == "batched":
        voff, u, v = _batched_pairs(case, seed)
        n = int(voff[-1])
        off, adj = _graph_csr(n, u, v)
        vb = _Buf(voff)
        st = {"op": op, "voff": vb, "g": T.BatchedGraph(vb, off, adj),
              "per_graph": torch.zeros(case["graphs"], dtype=torch.int64, device="cuda"),
              "out": torch.zeros(n, dtype=torch.int32, device="cuda") if case["pv"] else None}
        return st
    n = case["n"]
    gen = _gen(seed)
    u, v = _pairs(gen, case["kind"], n, n * case["ef"])
    st = {"op": op, "n": n, "out": torch.zeros(n, dtype=torch.int32, device="cuda")}
    if op in ("static", "stream"):
        off, adj = _graph_csr(n, u, v)
        del u, v
        st["g"] = T.cuStinger(off, adj, assume_symmetric=True, location=T.TC_DEVICE)
        st["pv"] = case.get("pv", True)
        if op == "stream":
            toff = torch.empty(off.n, dtype=torch.int64, device="cuda")
            tadj = torch.empty(adj.n, dtype=torch.int32, device="cuda")
            T.check(T.lib().tc_graph_to_csr(st["g"].h, toff.data_ptr(), tadj.data_ptr(), T.TC_DEVICE))
            bu, bv, bd = _update(case, gen, toff, tadj)
            st.update(u=bu, v=bv, ins=bd, undo=(1 - bd).contiguous(),
                      back=torch.zeros(n, dtype=torch.int32, device="cuda"),
                      sched=T.default_schedule(capture=1 if case["capture"] else 0))
        off.free()
        adj.free()
    elif op == "directed":
        off, adj = _directed_csr(n, u, v)
        st["g"] = T.cuStinger(_Buf(off), _Buf(adj), location=T.TC_DEVICE)
    else:  # new, csr: the CSR as it arrives
        off, adj = _graph_csr(n, u, v)
        st["off"], st["adj"] = off, adj
    torch.cuda.synchronize()
    return st


# --------------------------------------------------------------------- run
def _apply(st, is_delete, delta):
    delta.zero_()  # the call accumulates
    dg = C.c_int64(0)
    T.check(T.lib().tc_batch_apply(st["g"].h, st["u"].data_ptr(), st["v"].data_ptr(),
                                   is_delete.data_ptr(), st["u"].numel(), delta.data_ptr(),
                                   C.byref(dg), C.byref(st["sched"]), None))
    return dg.value


def run(st):
    op = st["op"]
    if op == "stream":
        a = _apply(st, st["ins"], st["out"])
        b = _apply(st, st["undo"], st["back"])
        return {"delta": st["out"], "delta_total": a, "undo": st["back"], "undo_total": b}
    if op == "batched":
        st["g"].count(_Buf(st["per_graph"]), _Buf(st["out"]) if st["out"] is not None else None)
        got = {"per_graph": st["per_graph"]}
        if st["out"] is not None:
            got["counts"] = st["out"]
        return got
    if op == "csr":
        glob = C.c_uint64(0)
        T.check(T.lib().tc_csr_count_device(st["n"], st["adj"].n, st["off"].ptr, st["adj"].ptr,
                                            st["out"].data_ptr(), C.byref(glob), None))
        return {"counts": st["out"], "total": int(glob.value)}
    if op == "new":
        g = T.cuStinger(st["off"], st["adj"], location=T.TC_DEVICE)
        _, total, _ = T.static_count(g, None, True, _Buf(st["out"]))
        g.close()
        return {"counts": st["out"], "total": total}
    if op == "static" and not st["pv"]:
        _, total, _ = T.static_count(st["g"], None, False)
        return {"total": total}
    _, total, _ = T.static_count(st["g"], None, True, _Buf(st["out"]))
    return {"counts": st["out"], "total": total}


# -------------------------------------------------------------------- work
def work(case):
    """Bytes of one pass: the rows read once (offsets and ids) and the results
    written once; for an update, the batch, the rows of its endpoints read and
    written, and the per-vertex deltas, in each direction.  The entries are those
    of the drawn pairs before deduplication.  Nothing here is floating point."""
    if case["op"] == "batched":
        lo, hi = case["nmin"], case["nmax"]
        n = case["graphs"] * ((hi - lo) / math.log(hi / lo) if hi > lo else lo)
        entries = 2 * n * (case["efmin"] + case["efmax"]) / 2
        return {"bytes": 4 * entries + 8 * n + (4 * n if case["pv"] else 0) + 16 * case["graphs"],
                "flops": 0}
    n, ef = case["n"], case["ef"]
    if case["op"] == "stream":
        rows = 2 * case["pairs"]
        return {"bytes": 2 * (9 * case["pairs"] + rows * (2 * 4 * 2 * ef + 16) + 4 * n), "flops": 0}
    entries = n * ef * (1 if case["op"] == "directed" else 2)
    return {"bytes": 4 * entries + 8 * (n + 1) + (4 * n if case.get("pv", True) else 0) + 8, "flops": 0}


# ------------------------------------------------------------------- exact
def _count64(off, adj, upper):
    """sum over entries (v, u) of |N(u) and N(v)|, both rows of two or more entries
    (upper: only u > v), by enumerating (v, u, w); int64 per vertex, or None."""
    n = off.numel() - 1
    deg = off[1:] - off[:-1]
    src = torch.repeat_interleave(torch.arange(n, device="cuda"), deg)
    a = adj.long()
    ok = (deg[src] >= 2) & (deg[a] >= 2) & ((a > src) if upper else (a != src))
    es, eu = src[ok], a[ok]
    if es.numel() and int(deg[eu].sum()) > _EXACT_WEDGES:
        return None
    key = src * n + a
    out = torch.zeros(n, dtype=torch.int64, device="cuda")
    step = max(1, (1 << 24) // max(1, int(deg.max())))
    for s in range(0, es.numel(), step):
        v, u = es[s:s + step], eu[s:s + step]
        d = deg[u]
        at = torch.repeat_interleave(torch.arange(v.numel(), device="cuda"), d)
        k = torch.arange(at.numel(), device="cuda") - (torch.cumsum(d, 0) - d)[at]
        want = v[at] * n + a[off[u[at]] + k]
        pos = torch.searchsorted(key, want).clamp(max=key.numel() - 1)
        out.index_add_(0, v[at], (key[pos] == want).long())
    return out


def exact(case, seed):
    op = case["op"]
    if op == "stream":
        return None
    voff = None
    if op == "batched":
        voff, u, v = _batched_pairs(case, seed)
        n = int(voff[-1])
    else:
        n = case["n"]
        u, v = _pairs(_gen(seed), case["kind"], n, n * case["ef"])
    if u.numel() > 50_000_000:
        return None
    off, adj = _directed_csr(n, u, v) if op == "directed" else \
        _directed_csr(n, torch.cat([u, v]), torch.cat([v, u]))
    c = _count64(off, adj, op == "csr")
    if c is None:
        return None
    wrapped = c.int()  # the low 32 bits, as the per-vertex counts keep them
    if op == "batched":
        s = torch.cat([torch.zeros(1, dtype=torch.int64, device="cuda"), torch.cumsum(c, 0)])
        got = {"per_graph": s[voff[1:]] - s[voff[:-1]]}
        if case["pv"]:
            got["counts"] = wrapped
        return got
    got = {"counts": wrapped} if case.get("pv", True) else {}
    got["total"] = int(c.sum())
    return got

// tc_graph.hip -- the dynamic adjacency store: creation from CSR, validation,
// snapshots.  Stands in for the cuStinger container the reference builds with
// initializeCuStinger(eInitStateCSR) (tests/cct.cpp:261-277) and reads through
// dVD->getUsed()/getAdj() (src/static_triangle_counting/cct.cu:235-261).
#include "tc_internal.hpp"

#include <algorithm>
#include <map>
#include <mutex>
#include <vector>

namespace tc {

thread_local Error g_last = {TC_OK, ""};

void set_last_error(int code, const std::string &msg)
{
    g_last.code = code;
    g_last.msg = msg;
}

// ------------------------------------------------------- block pool --
// A graph's handle owns some sixty device blocks, and a program that counts
// graphs as they arrive paid for them on every handle: hipMalloc and hipFree
// were 3 to 26 of the 5 to 28 ms that a new graph of 250k vertices took (the
// cost of mapping differs from run to run).  Released blocks are kept here, by
// size and device, and handed to the next handle.
//   Bounded: kHoldBytes in all, no block above kHoldBlock; what exceeds it is
//   freed, the largest first, and everything held is freed when an allocation
//   of this library fails, or by the caller (tc_device_trim).
//   Safe across streams and threads: a block is given back only when its
//   device is idle (DevBuf::release synchronises, as hipFree does), so no
//   kernel of its last owner can still touch it; the lists are under a lock.
namespace {

constexpr size_t kHoldBytes = size_t(4) << 30;
constexpr size_t kHoldBlock = size_t(1) << 30;

struct HostKit {  // pinned words and events of a handle, by device
    int dev;
    unsigned long long *words;
    hipEvent_t ev[16];
};
constexpr size_t kHoldKits = 32;

struct BlockPool {
    std::mutex mu;
    std::multimap<std::pair<int, size_t>, void *> blocks;  // (device, bytes)
    size_t held = 0;
    std::vector<HostKit> kits;
};

// Never destroyed: at exit the runtime may be gone before a destructor runs.
BlockPool &block_pool()
{
    static BlockPool *p = [] {
        BlockPool *q = new BlockPool;
        q->kits.reserve(kHoldKits);
        return q;
    }();
    return *p;
}

// Sizes requests share: powers of two up to 1 MB, then eighths of one; blocks
// that the pool would not keep stay exact, to whole 256 bytes (kernels read the
// 16 bytes that a row's last entries lie in).
size_t block_size(size_t need)
{
    if (need > kHoldBlock) return (need + 255) / 256 * 256;
    size_t p2 = 4096;
    while (p2 < need) p2 <<= 1;
    if (p2 <= (size_t(1) << 20)) return p2;
    const size_t step = p2 / 16;
    return (need + step - 1) / step * step;
}

void *pool_take(int dev, size_t bytes, size_t &got)
{
    BlockPool &P = block_pool();
    std::lock_guard<std::mutex> lock(P.mu);
    auto it = P.blocks.lower_bound({dev, bytes});
    if (it == P.blocks.end() || it->first.first != dev || it->first.second > bytes + bytes / 4) return nullptr;
    void *p = it->second;
    got = it->first.second;
    P.held -= got;
    P.blocks.erase(it);
    return p;
}

// Takes a block over: it is kept, or freed where host memory is short or the
// pool would hold too much.  (Nothing here throws: handles are closed from
// destructors and from C.)
void pool_give(int dev, void *p, size_t bytes) noexcept
{
    BlockPool &P = block_pool();
    bool kept = false;
    if (bytes <= kHoldBlock) {
        std::lock_guard<std::mutex> lock(P.mu);
        try {
            P.blocks.insert({{dev, bytes}, p});
            P.held += bytes;
            kept = true;
        } catch (...) {
        }
    }
    if (!kept) (void)hipFree(p);
    for (;;) {
        void *out = nullptr;
        {
            std::lock_guard<std::mutex> lock(P.mu);
            if (P.held <= kHoldBytes) return;
            auto big = P.blocks.begin();
            for (auto it = P.blocks.begin(); it != P.blocks.end(); ++it)
                if (it->first.second > big->first.second) big = it;
            P.held -= big->first.second;
            out = big->second;
            P.blocks.erase(big);
        }
        (void)hipFree(out);
    }
}

}  // namespace

void pool_flush() noexcept
{
    BlockPool &P = block_pool();
    decltype(P.blocks) out;
    {
        std::lock_guard<std::mutex> lock(P.mu);
        out.swap(P.blocks);
        P.held = 0;
    }
    for (auto &b : out) (void)hipFree(b.second);
}

thread_local size_t block_limit = 0;

hipError_t device_malloc(void **p, size_t bytes)
{
    if (block_limit && bytes > block_limit) {
        *p = nullptr;
        return hipErrorOutOfMemory;
    }
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        pool_flush();
        e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
    }
    return e;
}

int DevBuf::ensure(size_t need)
{
    if (need == 0) need = 16;
    if (bytes >= need) return TC_OK;
    // a buffer that has to grow again gets 25% headroom: batch-sized scratch
    // varies from call to call, and every regrowth stalls the device
    if (p) {
        release();
        need += need / 4;
    }
    (void)hipGetDevice(&dev);
    const size_t want = block_size(need);
    size_t got = want;
    p = block_limit && want > block_limit ? nullptr : pool_take(dev, want, got);
    if (!p) {
        if (device_malloc(&p, want) != hipSuccess) {
            set_last_error(TC_ERR_OOM, "hipMalloc of " + std::to_string(need) + " bytes failed");
            return TC_ERR_OOM;
        }
    }
    bytes = got;
    return TC_OK;
}

void DevBuf::release(bool idle)
{
    if (p) {
        int now = dev;
        (void)hipGetDevice(&now);
        if (now != dev) {  // another device's block: freed, as this thread cannot wait for it
            (void)hipFree(p);
        } else {
            // (a capturing thread cannot synchronise: the block is not reused)
            if (idle || hipDeviceSynchronize() == hipSuccess) {
                pool_give(dev, p, bytes);
            } else {
                (void)hipGetLastError();
                (void)hipFree(p);
            }
        }
    }
    p = nullptr;
    bytes = 0;
}

int Graph::ensure_events()
{
    if (events_ready) return TC_OK;
    int now = 0;
    TC_HIP(hipGetDevice(&now));
    if (!hcounts) {
        BlockPool &P = block_pool();
        std::lock_guard<std::mutex> lock(P.mu);
        for (size_t k = 0; k < P.kits.size(); ++k)
            if (P.kits[k].dev == now) {
                hcounts = P.kits[k].words;
                std::copy(P.kits[k].ev, P.kits[k].ev + 16, ev);
                P.kits.erase(P.kits.begin() + (long)k);
                kit_dev = now;
                events_ready = true;
                return TC_OK;
            }
    }
    if (!hcounts)
        TC_HIP(hipHostMalloc(reinterpret_cast<void **>(&hcounts), 32 * sizeof(unsigned long long),
                             hipHostMallocDefault));
    for (auto &e : ev) TC_HIP(hipEventCreate(&e));
    kit_dev = now;
    events_ready = true;
    return TC_OK;
}

void Graph::drop_events()
{
    if (events_ready) {
        BlockPool &P = block_pool();
        std::lock_guard<std::mutex> lock(P.mu);
        if (P.kits.size() < kHoldKits) {
            HostKit k = {kit_dev, hcounts, {}};
            std::copy(ev, ev + 16, k.ev);
            P.kits.push_back(k);
            hcounts = nullptr;
            events_ready = false;
            return;
        }
    }
    if (events_ready)
        for (auto &e : ev) (void)hipEventDestroy(e);
    if (hcounts) (void)hipHostFree(hcounts);
    hcounts = nullptr;
    events_ready = false;
}

void Graph::drop_capture()
{
    if (cexec) (void)hipGraphExecDestroy(cexec);
    if (cgraph) (void)hipGraphDestroy(cgraph);
    cexec = nullptr;
    cgraph = nullptr;
    cexec_key = 0;
}

namespace {

__global__ void k_len_from_off(const int64_t *__restrict__ off, int32_t nv, int32_t *__restrict__ len,
                               int64_t *__restrict__ boff, int32_t *__restrict__ cap,
                               int32_t slack_pct)
{
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv;
         v += (int64_t)gridDim.x * blockDim.x) {
        int64_t l = off[v + 1] - off[v];
        len[v] = (int32_t)l;
        if (slack_pct <= 0) {
            cap[v] = (int32_t)l;
            boff[v] = off[v];
        } else {
            int64_t want = l + (l * slack_pct + 99) / 100;
            int64_t c = 1;
            while (c < want) c <<= 1;
            cap[v] = (int32_t)c;
        }
    }
}

// int32 offsets (the reference's length_t) widened to int64.
__global__ void k_widen_off(const int32_t *__restrict__ in, int64_t n, int64_t *__restrict__ out)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        out[i] = in[i];
}

// Copy row v of a CSR into its block (blocks laid out by an exclusive scan of cap).
__global__ void k_copy_rows(const int64_t *__restrict__ off, const int32_t *__restrict__ adj,
                            const int64_t *__restrict__ boff, int32_t nv, int32_t *__restrict__ pool)
{
    // one wave per row, rows grid-strided
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t wstride = (int64_t)gridDim.x * (blockDim.x / kWave);
    for (int64_t v = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; v < nv;
         v += wstride) {
        int64_t a = off[v], l = off[v + 1] - a, d = boff[v];
        for (int64_t i = lane; i < l; i += kWave) pool[d + i] = adj[a + i];
    }
}

// Rows that hold the compact entries e[0..N) (the same in every lane): 64 rows
// probed at a time, the N searches in lockstep.
template <int N>
__device__ inline void wave_row_search(const int64_t *__restrict__ coff, int32_t nv, const int64_t (&e)[N],
                                       int32_t (&row)[N])
{
    const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
    for (int q = 0; q < N; ++q) row[q] = 0;
    for (int32_t n = nv; n > 1;) {
        const int32_t step = (n + kWave - 1) / kWave;
        int64_t v[N];
#pragma unroll
        for (int q = 0; q < N; ++q) {
            const int64_t r = (int64_t)row[q] + (int64_t)lane * step;
            v[q] = (int64_t)lane * step < n && r < nv ? coff[r] : INT64_MAX;
        }
#pragma unroll
        for (int q = 0; q < N; ++q) {
            const uint64_t m = __ballot(v[q] <= e[q]);
            row[q] += m ? (63 - __clzll((long long)m)) * step : 0;
        }
        n = step;
    }
}

// Validation over compact entries: [0] unsorted/dup, [1] out of range,
// [2] self loops, [3] missing reverse entries, [4] max degree, [5] entries
// that leave their graph (gid: the graph of every vertex, or null).
//
// Symmetry: an entry (a, b) is looked for in the other row where that is the
// shorter one (ties: the lower id), and [6] counts those entries.  If none
// misses its reverse, the rows are symmetric exactly when the other entries are
// as many.  Half the searches, and none in a hub's row for its leaves' entries.
// Bound by the cache lines of the rows searched, one or two per search (250K
// R-MAT vertices at edge factor 16: 429 -> 250 us; 1.2M entries, each to a higher
// id: 53 -> 22).  A wave takes two chunks of 64 entries in lockstep;
// one or four took 8% longer.
constexpr int kValThreads = 512;

__global__ __launch_bounds__(kValThreads) void k_validate(
    const int64_t *__restrict__ coff, const int64_t *__restrict__ boff, const int32_t *__restrict__ len,
    const int32_t *__restrict__ pool, int32_t nv, int64_t nnz, int check_sym, const int32_t *__restrict__ gid,
    unsigned long long *__restrict__ res)
{
    constexpr int U = 2;
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t npairs = ceil_div(nnz, U * kWave);
    const int64_t wstride = (int64_t)gridDim.x * (blockDim.x / kWave);
    uint32_t bad = 0, oor = 0, loops = 0, miss = 0, cross = 0, down = 0;
    int32_t most = 0;
    for (int64_t c = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; c < npairs;
         c += wstride) {
        const int64_t e0 = c * U * kWave;
        int64_t edge[U + 1];
        int32_t row[U + 1];
#pragma unroll
        for (int u = 0; u <= U; ++u) edge[u] = min(e0 + u * kWave, nnz - 1);
        wave_row_search<U + 1>(coff, nv, edge, row);
        int64_t e[U];
        int32_t a[U], top[U];
        bool go = false;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            e[u] = min(e0 + u * kWave + lane, nnz - 1);
            a[u] = row[u];
            top[u] = max(row[u], row[u + 1]);
            go = go || a[u] < top[u];
        }
        while (go) {
            go = false;
            int64_t v[U];
            int32_t mid[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                mid[u] = a[u] + ((top[u] - a[u] + 1) >> 1);
                v[u] = coff[mid[u]];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (a[u] < top[u]) {
                    if (v[u] <= e[u]) a[u] = mid[u]; else top[u] = mid[u] - 1;
                }
                go = go || a[u] < top[u];
            }
        }
        int32_t b[U], la[U], lb[U], lo[U], hi[U];
        int64_t at[U];
        bool in[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t k = e[u] - coff[a[u]], addr = boff[a[u]] + k;
            la[u] = len[a[u]];
            b[u] = pool[addr];
            const int32_t before = k > 0 ? pool[addr - 1] : -1;
            in[u] = e0 + u * kWave + lane < nnz;
            if (in[u]) {
                if (b[u] < 0 || b[u] >= nv) {
                    ++oor;
                    in[u] = false;
                } else {
                    bad += k > 0 && before >= b[u];
                    loops += b[u] == a[u];
                }
            }
        }
        if (gid) {
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (in[u] && gid[a[u]] != gid[b[u]]) ++cross;
        }
        if (!check_sym) continue;
        go = false;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            lb[u] = in[u] ? len[b[u]] : 0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            in[u] = in[u] && b[u] != a[u] && (lb[u] < la[u] || (lb[u] == la[u] && b[u] < a[u]));
            at[u] = in[u] ? boff[b[u]] : 0;
            lo[u] = 0;
            hi[u] = in[u] ? lb[u] : 0;
            go = go || hi[u] > 0;
        }
        while (go) {
            go = false;
            int32_t x[U], mid[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                mid[u] = (lo[u] + hi[u]) >> 1;
                x[u] = lo[u] < hi[u] ? pool[at[u] + mid[u]] : 0;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (lo[u] < hi[u]) {
                    if (x[u] < a[u])
                        lo[u] = mid[u] + 1;
                    else
                        hi[u] = x[u] == a[u] ? -1 : mid[u];  // (-1: found)
                }
                go = go || lo[u] < hi[u];
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            down += in[u];
            miss += in[u] && hi[u] != -1;
        }
    }
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv; v += (int64_t)gridDim.x * blockDim.x)
        most = max(most, len[v]);
    __shared__ unsigned long long part[kValThreads / kWave][7];
    const uint32_t mine[7] = {bad, oor, loops, miss, (uint32_t)most, cross, down};
#pragma unroll
    for (int q = 0; q < 7; ++q) {
        unsigned long long x = mine[q];
        if (q == 4)
            for (int d = 32; d > 0; d >>= 1) x = max(x, __shfl_xor(x, d));
        else
            x = wave_sum<unsigned long long>(x);
        if (lane == 0) part[threadIdx.x / kWave][q] = x;
    }
    __syncthreads();
    if (threadIdx.x < 7) {
        unsigned long long x = 0;
        const bool top = threadIdx.x == 4;
        for (int w = 0; w < kValThreads / kWave; ++w) {
            const unsigned long long p = part[w][threadIdx.x];
            x = top ? max(x, p) : x + p;
        }
        if (top && x) atomicMax(&res[4], x);
        if (!top && x) atomicAdd(&res[threadIdx.x], x);
    }
}

__global__ void k_zero_u64(unsigned long long *p, int n)
{
    if ((int)threadIdx.x < n) p[threadIdx.x] = 0;
}

__global__ void k_gather_rows(const int64_t *__restrict__ coff, const int64_t *__restrict__ boff,
                              const int32_t *__restrict__ pool, int32_t nv, int32_t *__restrict__ adj)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t wstride = (int64_t)gridDim.x * (blockDim.x / kWave);
    for (int64_t v = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; v < nv;
         v += wstride) {
        int64_t a = coff[v], l = coff[v + 1] - a, s = boff[v];
        for (int64_t i = lane; i < l; i += kWave) adj[a + i] = pool[s + i];
    }
}

}  // namespace

int validate_graph(Graph &g, bool check_symmetry, int64_t *bad_rows)
{
    const int32_t nv = g.st.nv;
    const int64_t nnz = g.st.nnz;
    hipStream_t s = g.stream;
    TC_TRY(g.accum.ensure(32 * sizeof(unsigned long long)));
    unsigned long long *res = g.accum.as<unsigned long long>();
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, s, res, 16);
    TC_HIP(hipGetLastError());
    if (nv > 0) {
        TC_TRY(g.coff.ensure((size_t)(nv + 1) * sizeof(int64_t)));
        int64_t *coff = g.coff.as<int64_t>();
        TC_TRY(scan_counts_i32(g.st.len.as<int32_t>(), coff, nv, g.tmp, s));
        hipLaunchKernelGGL(k_validate, dim3(grid_for(std::max<int64_t>(nnz, nv), 2 * kValThreads, 1024)),
                           dim3(kValThreads), 0, s, coff, g.st.boff.as<int64_t>(), g.st.len.as<int32_t>(),
                           g.st.pool.as<int32_t>(), nv, nnz, check_symmetry ? 1 : 0,
                           g.batch_voff ? g.dgid.as<int32_t>() : nullptr, res);
        TC_HIP(hipGetLastError());
    }
    unsigned long long h[16];
    TC_HIP(hipMemcpyAsync(h, res, sizeof(h), hipMemcpyDeviceToHost, s));
    TC_HIP(hipStreamSynchronize(s));
    if (bad_rows) *bad_rows = (int64_t)(h[0] + h[1]);
    if (h[0] || h[1]) {
        set_last_error(TC_ERR_INVALID,
                       "graph rows must be sorted strictly ascending with ids in [0,nv): " +
                           std::to_string(h[0]) + " unsorted/duplicate, " + std::to_string(h[1]) +
                           " out-of-range entries");
        return TC_ERR_INVALID;
    }
    g.validated = true;
    g.self_loops = (int64_t)h[2];
    if (check_symmetry) g.symmetric = h[3] == 0 && 2 * h[6] + h[2] == (unsigned long long)nnz ? 1 : 0;
    g.max_degree = (int32_t)h[4];
    g.degree_stale = false;
    // bit matrices hold a graph's own columns only
    g.batch_cross = h[5] != 0;
    if (g.batch_cross) {
        g.dense_words = 0;
        g.core_total = 0;
    }
    return TC_OK;
}

int graph_create_csr(int32_t nv, int64_t nnz, const int64_t *off, const int32_t *adj, int location,
                     uint32_t flags, int32_t slack_pct, Graph **out)
{
    if (!out || nv < 0 || nnz < 0 || (nv > 0 && !off) || (nnz > 0 && !adj) ||
        (location != TC_HOST && location != TC_DEVICE)) {
        set_last_error(TC_ERR_INVALID, "tc_graph_create_csr: bad arguments");
        return TC_ERR_INVALID;
    }
    const bool off32 = (flags & TC_GRAPH_OFFSETS_I32) != 0;
    std::vector<int64_t> host_wide;
    if (off32 && location == TC_HOST && nv > 0) {
        const int32_t *o32 = reinterpret_cast<const int32_t *>(off);
        host_wide.assign(o32, o32 + (size_t)nv + 1);
        off = host_wide.data();
    }
    if (location == TC_HOST && nv > 0) {
        if (off[0] != 0 || off[nv] != nnz) {
            set_last_error(TC_ERR_INVALID, "tc_graph_create_csr: off[0] must be 0 and off[nv] == nnz");
            return TC_ERR_INVALID;
        }
        for (int32_t v = 0; v < nv; ++v)
            if (off[v + 1] < off[v] || off[v + 1] - off[v] > INT32_MAX) {
                set_last_error(TC_ERR_INVALID, "tc_graph_create_csr: offsets must be monotone");
                return TC_ERR_INVALID;
            }
    }
    Graph *g = new Graph();
    g->st.nv = nv;
    g->st.nnz = nnz;
    auto fail = [&](int code) {
        graph_destroy(g);
        return code;
    };
    int st;
    size_t nvb = (size_t)std::max<int32_t>(nv, 1);
    if ((st = g->st.boff.ensure(nvb * sizeof(int64_t))) != TC_OK) return fail(st);
    if ((st = g->st.len.ensure(nvb * sizeof(int32_t))) != TC_OK) return fail(st);
    if ((st = g->st.cap.ensure(nvb * sizeof(int32_t))) != TC_OK) return fail(st);
    // device copy of the offsets (temporarily in coff)
    if ((st = g->coff.ensure((nvb + 1) * sizeof(int64_t))) != TC_OK) return fail(st);
    int64_t *doff = g->coff.as<int64_t>();
    hipStream_t s = nullptr;
    if (nv > 0) {
        if (off32 && location == TC_DEVICE) {
            hipLaunchKernelGGL(k_widen_off, dim3(grid_for((int64_t)nv + 1, 256, 65536)), dim3(256), 0, s,
                               reinterpret_cast<const int32_t *>(off), (int64_t)nv + 1, doff);
            if (hipGetLastError() != hipSuccess) {
                set_last_error(TC_ERR_HIP, "widening of the offsets failed");
                return fail(TC_ERR_HIP);
            }
        } else if (hipMemcpy(doff, off, (size_t)(nv + 1) * sizeof(int64_t),
                             location == TC_HOST ? hipMemcpyHostToDevice : hipMemcpyDeviceToDevice) !=
                   hipSuccess) {
            set_last_error(TC_ERR_HIP, "copy of offsets failed");
            return fail(TC_ERR_HIP);
        }
        if (location == TC_DEVICE) {
            int64_t ends[2];
            if (hipMemcpy(&ends[0], doff, sizeof(int64_t), hipMemcpyDeviceToHost) != hipSuccess ||
                hipMemcpy(&ends[1], doff + nv, sizeof(int64_t), hipMemcpyDeviceToHost) != hipSuccess) {
                set_last_error(TC_ERR_HIP, "read-back of the offsets failed");
                return fail(TC_ERR_HIP);
            }
            if (ends[0] != 0 || ends[1] != nnz) {
                set_last_error(TC_ERR_INVALID, "tc_graph_create_csr: off[0] must be 0 and off[nv] == nnz");
                return fail(TC_ERR_INVALID);
            }
        }
        hipLaunchKernelGGL(k_len_from_off, dim3(grid_for(nv, 256, 65536)), dim3(256), 0, s, doff, nv,
                           g->st.len.as<int32_t>(), g->st.boff.as<int64_t>(),
                           g->st.cap.as<int32_t>(), slack_pct);
    }
    int64_t pool_n = nnz;
    if (slack_pct > 0 && nv > 0) {
        // block offsets = exclusive scan of capacities
        DevBuf tmp;
        DevBuf scan;
        if ((st = scan.ensure((nvb + 1) * sizeof(int64_t))) != TC_OK) return fail(st);
        if ((st = scan_counts_i32(g->st.cap.as<int32_t>(), scan.as<int64_t>(), nv, tmp, s)) != TC_OK)
            return fail(st);
        if (hipMemcpy(&pool_n, scan.as<int64_t>() + nv, sizeof(int64_t), hipMemcpyDeviceToHost) !=
                hipSuccess ||
            hipMemcpy(g->st.boff.p, scan.p, (size_t)nv * sizeof(int64_t), hipMemcpyDeviceToDevice) !=
                hipSuccess) {
            set_last_error(TC_ERR_HIP, "copy of the block offsets failed");
            return fail(TC_ERR_HIP);
        }
        tmp.release();
        scan.release();
    }
    // pool gets 25% headroom for block moves before a compaction is needed
    int64_t pool_cap = pool_n + pool_n / 4 + 1024;
    if ((st = g->st.pool.ensure((size_t)pool_cap * sizeof(int32_t))) != TC_OK) return fail(st);
    g->st.pool_used = pool_n;
    if (nnz > 0) {
        if (slack_pct <= 0) {
            if (hipMemcpy(g->st.pool.p, adj, (size_t)nnz * sizeof(int32_t),
                          location == TC_HOST ? hipMemcpyHostToDevice : hipMemcpyDeviceToDevice) !=
                hipSuccess) {
                set_last_error(TC_ERR_HIP, "copy of adjacency failed");
                return fail(TC_ERR_HIP);
            }
        } else {
            const int32_t *dadj = adj;
            DevBuf stage;
            if (location == TC_HOST) {
                if ((st = stage.ensure((size_t)nnz * sizeof(int32_t))) != TC_OK) return fail(st);
                if (hipMemcpy(stage.p, adj, (size_t)nnz * sizeof(int32_t), hipMemcpyHostToDevice) !=
                    hipSuccess) {
                    set_last_error(TC_ERR_HIP, "copy of adjacency failed");
                    return fail(TC_ERR_HIP);
                }
                dadj = stage.as<int32_t>();
            }
            hipLaunchKernelGGL(k_copy_rows, dim3(grid_for(nv, 4, 65536)), dim3(256), 0, s, doff, dadj,
                               g->st.boff.as<int64_t>(), nv, g->st.pool.as<int32_t>());
            if (hipDeviceSynchronize() != hipSuccess) {
                set_last_error(TC_ERR_HIP, "row copy failed");
                return fail(TC_ERR_HIP);
            }
            stage.release();
        }
    }
    if (hipDeviceSynchronize() != hipSuccess) {
        set_last_error(TC_ERR_HIP, "graph creation kernels failed");
        return fail(TC_ERR_HIP);
    }
    if (!(flags & TC_GRAPH_NO_VALIDATE)) {
        int64_t bad = 0;
        st = validate_graph(*g, !(flags & TC_GRAPH_ASSUME_SYMMETRIC), &bad);
        if (st != TC_OK) return fail(st);
        if (flags & TC_GRAPH_ASSUME_SYMMETRIC) g->symmetric = 1;
    } else if (flags & TC_GRAPH_ASSUME_SYMMETRIC) {
        g->symmetric = 1;
    }
    *out = g;
    return TC_OK;
}

int graph_to_csr(Graph &g, int64_t *off, int32_t *adj, int location)
{
    const int32_t nv = g.st.nv;
    TC_TRY(g.coff.ensure((size_t)(nv + 1) * sizeof(int64_t)));
    int64_t *coff = g.coff.as<int64_t>();
    TC_TRY(scan_counts_i32(g.st.len.as<int32_t>(), coff, nv, g.tmp, g.stream));
    int64_t *doff = coff;
    int32_t *dadj = adj;
    DevBuf stage;
    if (location == TC_HOST) {
        TC_TRY(stage.ensure((size_t)std::max<int64_t>(g.st.nnz, 1) * sizeof(int32_t)));
        dadj = stage.as<int32_t>();
    }
    if (g.st.nnz > 0)
        hipLaunchKernelGGL(k_gather_rows, dim3(grid_for(nv, 4, 65536)), dim3(256), 0, g.stream, coff,
                           g.st.boff.as<int64_t>(), g.st.pool.as<int32_t>(), nv, dadj);
    TC_HIP(hipGetLastError());
    TC_HIP(hipStreamSynchronize(g.stream));
    hipMemcpyKind k = location == TC_HOST ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice;
    TC_HIP(hipMemcpy(off, doff, (size_t)(nv + 1) * sizeof(int64_t), k));
    if (location == TC_HOST && g.st.nnz > 0)
        TC_HIP(hipMemcpy(adj, dadj, (size_t)g.st.nnz * sizeof(int32_t), hipMemcpyDeviceToHost));
    stage.release();
    return TC_OK;
}

// A read-only view of a caller's device CSR: per-vertex offsets and lengths
// are built, the adjacency array itself is used in place and never freed.
int graph_borrow_csr(int32_t nv, int64_t nnz, const int64_t *d_off, const int32_t *d_adj,
                     hipStream_t s, Graph **out)
{
    Graph *g = new Graph();
    g->st.nv = nv;
    g->st.nnz = nnz;
    g->stream = s;
    g->borrowed = true;
    const size_t nvb = (size_t)std::max<int32_t>(nv, 1);
    int st;
    if ((st = g->st.boff.ensure(nvb * sizeof(int64_t))) != TC_OK ||
        (st = g->st.len.ensure(nvb * sizeof(int32_t))) != TC_OK ||
        (st = g->st.cap.ensure(nvb * sizeof(int32_t))) != TC_OK) {
        graph_destroy(g);
        return st;
    }
    if (nv > 0)
        hipLaunchKernelGGL(k_len_from_off, dim3(grid_for(nv, 256, 65536)), dim3(256), 0, s, d_off, nv,
                           g->st.len.as<int32_t>(), g->st.boff.as<int64_t>(), g->st.cap.as<int32_t>(),
                           0);
    g->st.pool.p = const_cast<int32_t *>(d_adj);
    g->st.pool.bytes = (size_t)nnz * sizeof(int32_t);
    g->st.pool_used = nnz;
    if (hipStreamSynchronize(s) != hipSuccess || hipGetLastError() != hipSuccess) {
        set_last_error(TC_ERR_HIP, "borrowed graph setup failed");
        graph_destroy(g);
        return TC_ERR_HIP;
    }
    *out = g;
    return TC_OK;
}

namespace {

// compareCUS / comparecus (src/streaming_triangle_counting/cct_upd.cu:442-484):
// one wave per vertex compares the used lengths and then the entries of the
// two stores' rows.  res[0] += rows whose lengths differ, res[1] += rows of
// equal length whose entries differ, res[2] = max(nv - v) over differing
// vertices v (0: none), i.e. the first differing vertex.
__global__ void k_compare_rows(int32_t nv, const int64_t *__restrict__ boff_a,
                               const int32_t *__restrict__ len_a, const int32_t *__restrict__ pool_a,
                               const int64_t *__restrict__ boff_b,
                               const int32_t *__restrict__ len_b, const int32_t *__restrict__ pool_b,
                               unsigned long long *__restrict__ res)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t wstride = (int64_t)gridDim.x * (blockDim.x / kWave);
    unsigned long long nsize = 0, nent = 0;
    for (int64_t v = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; v < nv;
         v += wstride) {
        const int32_t la = len_a[v], lb = len_b[v];
        bool diff = la != lb;
        if (diff) {
            nsize += lane == 0;
        } else {
            const int64_t ba = boff_a[v], bb = boff_b[v];
            bool d = false;
            for (int32_t i = lane; i < la; i += kWave) d |= pool_a[ba + i] != pool_b[bb + i];
            diff = __ballot(d) != 0;
            nent += (diff && lane == 0);
        }
        if (diff && lane == 0) atomicMax(&res[2], (unsigned long long)(nv - v));
    }
    const unsigned long long part[2] = {nsize, nent};
    block_add_u64<2>(part, res);
}

}  // namespace

int graph_compare(Graph &a, Graph &b, int64_t *size_mismatch, int64_t *entry_mismatch,
                  int32_t *first_vertex)
{
    if (a.st.nv != b.st.nv) {
        set_last_error(TC_ERR_INVALID, "tc_graph_compare: the stores have different vertex counts");
        return TC_ERR_INVALID;
    }
    hipStream_t s = a.stream;
    TC_HIP(hipStreamSynchronize(b.stream));
    TC_TRY(a.accum.ensure(32 * sizeof(unsigned long long)));
    unsigned long long *res = a.accum.as<unsigned long long>();
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, s, res, 3);
    if (a.st.nv > 0)
        hipLaunchKernelGGL(k_compare_rows, dim3(grid_for(a.st.nv, 4, 65536)), dim3(256), 0, s,
                           a.st.nv, a.st.boff.as<int64_t>(), a.st.len.as<int32_t>(),
                           a.st.pool.as<int32_t>(), b.st.boff.as<int64_t>(), b.st.len.as<int32_t>(),
                           b.st.pool.as<int32_t>(), res);
    TC_HIP(hipGetLastError());
    unsigned long long h[3];
    TC_HIP(hipMemcpyAsync(h, res, sizeof(h), hipMemcpyDeviceToHost, s));
    TC_HIP(hipStreamSynchronize(s));
    *size_mismatch = (int64_t)h[0];
    *entry_mismatch = (int64_t)h[1];
    *first_vertex = h[2] == 0 ? -1 : (int32_t)((int64_t)a.st.nv - (int64_t)h[2]);
    return TC_OK;
}

void graph_destroy(Graph *g)
{
    if (!g) return;
    const bool idle = hipDeviceSynchronize() == hipSuccess;
    if (g->borrowed) {
        g->st.pool.p = nullptr;
        g->st.pool.bytes = 0;
    }
    g->each_buffer([&](DevBuf &b) { b.release(idle); });
    g->drop_events();
    g->drop_capture();
    if (g->bexec) (void)hipGraphExecDestroy(g->bexec);
    if (g->bgraph) (void)hipGraphDestroy(g->bgraph);
    if (g->cap_stream) (void)hipStreamDestroy(g->cap_stream);
    delete g;
}

}  // namespace tc

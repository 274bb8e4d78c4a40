// tc_dense.hip -- counts of graphs of few vertices on a bit matrix.
//
// A graph of n <= kDenseMax vertices has rows of at most kDenseMax bits, so
// the per-entry formula of devicecuStingerAllTriangles
// (src/static_triangle_counting/cct.cu:233-268),
//     out[v] = sum over u in N(v), u != v, of |N(v) cap N(u)|,
// is an AND and a population count of two bit rows per entry.  It holds for
// any rows (loops, asymmetric ones, the CSR convention), needs no rank order,
// no task lists and no plan whose sizes the host must read, and runs as two
// kernels where the oriented count takes more than fifty launches.
#include "tc_plan.hpp"

#include <algorithm>

namespace tc {

namespace {

constexpr int kChunkWords = 32;                 // one 128-byte line of a row: 1024 columns
constexpr int kChunkCols = kChunkWords * 32;
constexpr int kDenseMax = 16 * kChunkCols;      // vertices of one graph
constexpr int64_t kDenseBytes = int64_t(1) << 30;  // all matrices of a batch
// Rows of more than max(kDenseLong, twice the mean degree) entries are cut
// into items of that many, dealt to all waves: a hub's row is otherwise one
// wave's serial chain.  (Twice the mean: with most rows cut, reserving their
// items costs more than it saves, 317 -> 436 us on 16384 rows of 64.)  The
// items are listed in kParts lists, each with a counter on a line of its own,
// by the XCD of the row's wave.
constexpr int kDenseLong = 64;
constexpr int kParts = 8;
constexpr int kCtrStride = 16;  // counters' words

// The bit rows of one graph: vertex v0 + i owns the words
// [off + i * 32 nch, off + (i + 1) * 32 nch) of the matrix.
struct DenseGraph {
    int32_t v0, n, nch, pad;
    int64_t off;
};

struct DenseArgs {
    const int64_t *boff;
    const int32_t *len;
    const int32_t *pool;
    int32_t nv;
    uint32_t *mat;
    DenseGraph one;            // a single graph
    const DenseGraph *graphs;  // batched graphs (else null), by gid of the vertex
    const int32_t *gid;
    uint32_t *out;
    unsigned long long *global;
    int32_t long_len;
    unsigned long long *nitems;  // [kParts], kCtrStride apart, zero on entry
    int2 *items;                 // [kParts][icap] (row, first entry)
    int64_t icap;
    int32_t *bad;                // set where an entry has no reverse
    int32_t skip_lower;
    int32_t check_sym;
};

__host__ __device__ inline int32_t dense_chunks(int32_t n)
{
    return n <= kChunkCols ? 1 : (n + kChunkCols - 1) / kChunkCols;
}

__device__ inline DenseGraph graph_of_row(const DenseArgs &A, int32_t v)
{
    return A.graphs ? A.graphs[A.gid[v]] : A.one;
}

// The rows of a wave: round-robin over a single graph (a hub's neighbours in id
// order are often hubs); of batched graphs every XCD (blocks go to them in
// turn) deals one run of rows, so that its L2 meets few graphs.
struct RowDeal {
    int64_t r, end, step;
};
__device__ inline RowDeal deal_rows(const DenseArgs &A, int wpb, int wid)
{
    const int nb = (int)gridDim.x, b = (int)blockIdx.x;
    if (!A.graphs) return RowDeal{(int64_t)b * wpb + wid, A.nv, (int64_t)nb * wpb};
    const int nx = min(kParts, nb), x = b % nx;
    const int64_t per = (A.nv + nx - 1) / nx;
    return RowDeal{per * x + (int64_t)(b / nx) * wpb + wid, min(per * (x + 1), (int64_t)A.nv),
                   (int64_t)((nb - x + nx - 1) / nx) * wpb};
}

// Zeroes the counters of the count (32) and of the item lists.
__global__ void k_dense_init(unsigned long long *acc, unsigned long long *nitems)
{
    if (threadIdx.x < 32) acc[threadIdx.x] = 0ull;
    if (threadIdx.x < kParts) nitems[threadIdx.x * kCtrStride] = 0ull;
}

// Bit rows: one wave per row, its bits gathered in LDS and written as whole
// lines (a block per row left most of its lanes idle on rows of a dozen
// entries: 94 -> 40 us for 105k rows).  Rows above kDenseLong list their items
// and zero their output.
constexpr int kRowWaves = 4;
__global__ __launch_bounds__(kRowWaves * kWave) void k_dense_rows(DenseArgs A)
{
    __shared__ alignas(16) uint32_t lds[kRowWaves][kDenseMax / 32];
    const int lane = threadIdx.x & (kWave - 1);
    uint32_t *bits = lds[threadIdx.x / kWave];
    const RowDeal W = deal_rows(A, kRowWaves, __builtin_amdgcn_readfirstlane(threadIdx.x / kWave));
    const int part = blockIdx.x % kParts;
    for (int64_t r = W.r; r < W.end; r += W.step) {
        const int32_t v = (int32_t)r;
        const DenseGraph D = graph_of_row(A, v);
        const int32_t words = D.nch * kChunkWords, d = A.len[v];
        const int32_t *row = A.pool + A.boff[v];
        for (int i = lane; i < words; i += kWave) bits[i] = 0u;
        wave_sync();
        for (int32_t k0 = lane; k0 < d; k0 += 4 * kWave) {
            int32_t c[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) c[q] = row[min(k0 + q * kWave, d - 1)] - D.v0;
#pragma unroll
            for (int q = 0; q < 4; ++q)  // (a repeat of the last entry sets its bit again)
                atomicOr(&bits[c[q] >> 5], 1u << (c[q] & 31));
        }
        if (d > A.long_len) {
            unsigned long long base = 0;
            if (lane == 0) {
                base = atomicAdd(&A.nitems[part * kCtrStride],
                                 (unsigned long long)((d + A.long_len - 1) / A.long_len));
                A.out[v] = 0u;
            }
            base = __shfl(base, 0, kWave);
            for (int64_t q = lane; q * A.long_len < d; q += kWave)
                A.items[part * A.icap + base + q] = make_int2(v, (int32_t)(q * A.long_len));
        }
        wave_sync();
        uint4 *dst = reinterpret_cast<uint4 *>(A.mat + D.off + (int64_t)(v - D.v0) * words);
        for (int i = lane; i < words / 4; i += kWave)
            dst[i] = reinterpret_cast<const uint4 *>(bits)[i];
        wave_sync();
    }
}

// One wave, entries [e0, e1) of row v (at least one): the hits of this lane.  Eight lanes
// share an entry u: each reads 16 bytes of every 128-byte line of u's bit row
// (whole lines, no reduction per entry) against the same words of v's row,
// kept in registers for CH of the lines [c0, c1) at a time; U entries per
// group are in flight.  An entry that does not count reads v's own row, masked.
template <int CH, int U>
__device__ inline uint32_t dense_row(const DenseArgs &A, const DenseGraph &D, int32_t v,
                                     const int32_t *__restrict__ row, int32_t e0, int32_t e1,
                                     uint32_t c0, uint32_t c1, bool &miss)
{
    const int lane = threadIdx.x & (kWave - 1), i = lane & 7, grp = lane >> 3;
    // a graph's matrix is at most 32 MB: 32-bit byte offsets from a base the
    // whole wave shares
    const uint32_t rb = (uint32_t)D.nch * (kChunkWords * 4);
    const char *m = reinterpret_cast<const char *>(A.mat + D.off);
    const int32_t *lens = A.len + D.v0;
    const uint32_t lv = (uint32_t)(v - D.v0);
    uint32_t acc = 0;
#pragma unroll 1
    for (uint32_t cb = c0 * 128 + i * 16; cb < c1 * 128; cb += CH * 128) {
        uint4 S[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c)
            S[c] = *reinterpret_cast<const uint4 *>(m + (lv * rb + cb + c * 128));
        int32_t nu[U];  // the next entries, loaded while these rows are
#pragma unroll
        for (int q = 0; q < U; ++q) nu[q] = row[dense_entry(e0 + grp + q * 8, e1)];
#pragma unroll 1
        for (int32_t eb = e0 + grp; eb - grp < e1; eb += 8 * U) {
            uint32_t u[U];
            bool in[U];
            uint4 R[U][CH];
#pragma unroll
            for (int q = 0; q < U; ++q) {
                u[q] = (uint32_t)(nu[q] - D.v0);
                nu[q] = row[dense_entry(eb + (U + q) * 8, e1)];
            }
#pragma unroll
            for (int q = 0; q < U; ++q) {
                in[q] = eb + q * 8 < e1 && u[q] != lv;
                u[q] = in[q] ? u[q] : lv;
#pragma unroll
                for (int c = 0; c < CH; ++c)
                    R[q][c] = *reinterpret_cast<const uint4 *>(m + (u[q] * rb + cb + c * 128));
            }
#pragma unroll
            for (int q = 0; q < U; ++q) {
                const bool ok = in[q] && lens[u[q]] >= 2 && (!A.skip_lower || u[q] > lv);
                if (A.check_sym && cb == 0 && in[q]) {  // (lane 0 of the group, first pass)
                    const uint32_t w = *reinterpret_cast<const uint32_t *>(m + (u[q] * rb + (lv >> 5) * 4));
                    miss |= !((w >> (lv & 31)) & 1u);
                }
                uint32_t p = 0;
#pragma unroll
                for (int c = 0; c < CH; ++c)
                    p += __popc(R[q][c].x & S[c].x) + __popc(R[q][c].y & S[c].y) +
                         __popc(R[q][c].z & S[c].z) + __popc(R[q][c].w & S[c].w);
                acc += ok ? p : 0u;
            }
        }
    }
    return acc;
}

__device__ inline uint32_t dense_part(const DenseArgs &A, const DenseGraph &D, int32_t v, int32_t e0,
                                      int32_t e1, bool &miss)
{
    const int32_t *row = A.pool + A.boff[v];
    const uint32_t n = D.nch, n4 = n & ~3u;
    uint32_t h = 0;
    if (n4) h = dense_row<4, 1>(A, D, v, row, e0, e1, 0, n4, miss);
    switch (n & 3u) {
    case 1: h += dense_row<1, 4>(A, D, v, row, e0, e1, n4, n, miss); break;
    case 2: h += dense_row<2, 2>(A, D, v, row, e0, e1, n4, n, miss); break;
    case 3: h += dense_row<3, 1>(A, D, v, row, e0, e1, n4, n, miss); break;
    default: break;
    }
    return wave_sum<uint32_t>(h);
}

// out[v] and the total, one wave per row or item of a long row; items first,
// every list by all waves (the XCDs' lists differ: R-MAT hubs are ids with few
// set bits).  Bound by the latency of the entry -> row
// chain on small graphs, by reads of bit rows from L2 above (16384 vertices of
// degree 64: 2.1 GB in 250 us).  Per-graph sums are taken from out afterwards:
// one atomic per row on the few lines of per_graph serialised (48 graphs of
// 105k rows: this kernel 309 -> 120 us with that and with runs of rows).
__global__ __launch_bounds__(256, 8) void k_dense_count(DenseArgs A)
{
    const int lane = threadIdx.x & (kWave - 1);
    // (the same in all lanes: rows, their graphs and lengths stay scalar)
    const int wpb = blockDim.x / kWave, wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    unsigned long long total = 0;
    bool miss = false;
    const int64_t nwaves = (int64_t)gridDim.x * wpb, wave = (int64_t)blockIdx.x * wpb + wid;
    const int32_t ni = lane < kParts ? (int32_t)A.nitems[lane * kCtrStride] : 0;
    int64_t first = wave;  // the lists run on: a wave's share of each starts where the last one's ended
#pragma unroll 1
    for (int p = 0; p < kParts; ++p) {
        const int64_t n = __builtin_amdgcn_readlane(ni, p);
        int64_t k = first;
#pragma unroll 1
        for (; k < n; k += nwaves) {
            const int2 it = A.items[p * A.icap + k];
            const int32_t v = __builtin_amdgcn_readfirstlane(it.x);
            const int32_t e0 = __builtin_amdgcn_readfirstlane(it.y);
            const DenseGraph D = graph_of_row(A, v);
            const uint32_t h = dense_part(A, D, v, e0, min(e0 + A.long_len, A.len[v]), miss);
            if (lane == 0 && h) {
                total += h;
                atomicAdd(&A.out[v], h);
            }
        }
        first = k - n;
    }
    const RowDeal W = deal_rows(A, wpb, wid);
    for (int64_t r = W.r; r < W.end; r += W.step) {
        const int32_t v = (int32_t)r, d = A.len[v];
        if (d > A.long_len) continue;
        const DenseGraph D = graph_of_row(A, v);
        const uint32_t h = dense_walked(d, A.check_sym) ? dense_part(A, D, v, 0, d, miss) : 0u;
        if (lane == 0) {
            A.out[v] = d >= 2 ? h : 0u;
            total += d >= 2 ? h : 0u;
        }
    }
    if (__ballot(miss) && lane == 0) atomicOr(A.bad, 1);
    const unsigned long long part[1] = {total};
    block_add_u64<1>(part, A.global);
}

// per_graph[g] = the sum of its vertices' counts (below 2^28 each, so the
// 32-bit counts have not wrapped); one block per graph.
__global__ __launch_bounds__(256) void k_dense_graph_sums(const DenseGraph *__restrict__ graphs, int32_t nv,
                                                          const uint32_t *__restrict__ out,
                                                          unsigned long long *__restrict__ per_graph)
{
    const DenseGraph D = graphs[blockIdx.x];
    unsigned long long s = 0;
    for (int64_t i = threadIdx.x; i < D.n && D.v0 + i < nv; i += blockDim.x) s += out[D.v0 + i];
    const unsigned long long part[1] = {s};
    block_add_u64<1>(part, &per_graph[blockIdx.x]);
}

// One block: matrix offsets of batched graphs; res[0] = the largest graph's
// vertices, res[1] = words of all matrices, res[2] = words of the rows of all
// entries.
__global__ __launch_bounds__(256) void k_dense_plan(const int64_t *__restrict__ voff, int32_t G,
                                                    const int64_t *__restrict__ boff,
                                                    const int32_t *__restrict__ len, int32_t nv,
                                                    DenseGraph *__restrict__ graphs,
                                                    unsigned long long *__restrict__ res)
{
    __shared__ long long part[256], pmax[256], pread[256];
    const int t = threadIdx.x;
    const int64_t per = (G + 255) / 256, g0 = min(t * per, (int64_t)G), g1 = min(g0 + per, (int64_t)G);
    long long words = 0, most = 0, read = 0;
    for (int64_t g = g0; g < g1; ++g) {
        const int64_t a = voff[g], b = voff[g + 1], n = b - a;
        most = max(most, (long long)n);
        if (n > 0 && n <= kDenseMax) {
            const int64_t row = (int64_t)dense_chunks((int32_t)n) * kChunkWords;
            words += n * row;
            if (a >= 0 && b <= nv) read += (boff[b - 1] + len[b - 1] - boff[a]) * row;
        }
    }
    pread[t] = read;
    part[t] = words;
    pmax[t] = most;
    __syncthreads();
    long long before = 0, all = 0, mx = 0, rd = 0;
    for (int k = 0; k < 256; ++k) {
        rd += pread[k];
        if (k < t) before += part[k];
        all += part[k];
        mx = max(mx, pmax[k]);
    }
    for (int64_t g = g0; g < g1; ++g) {
        const int64_t n = voff[g + 1] - voff[g];
        DenseGraph D = {(int32_t)voff[g], (int32_t)n, 1, 0, (int64_t)before};
        if (n > 0 && n <= kDenseMax) {
            D.nch = dense_chunks((int32_t)n);
            before += n * D.nch * kChunkWords;
        }
        graphs[g] = D;
    }
    if (t == 0) {
        res[0] = (unsigned long long)mx;
        res[1] = (unsigned long long)all;
        res[2] = (unsigned long long)rd;
    }
}

__global__ void k_dense_gid(const DenseGraph *__restrict__ graphs, int32_t G, int32_t nv,
                            int32_t *__restrict__ gid)
{
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv;
         v += (int64_t)gridDim.x * blockDim.x) {
        int32_t lo = 0, hi = G - 1;
        while (lo < hi) {
            const int32_t mid = (lo + hi + 1) >> 1;
            if (graphs[mid].v0 <= v) lo = mid; else hi = mid - 1;
        }
        gid[v] = lo;
    }
}

}  // namespace

int dense_plan_batched(Graph &g)
{
    g.dense_words = 0;
    const int32_t G = g.batch_ngraphs;
    if (G <= 0 || g.st.nv == 0) return TC_OK;
    hipStream_t s = g.stream;
    TC_TRY(g.dgraphs.ensure((size_t)G * sizeof(DenseGraph)));
    TC_TRY(g.accum.ensure(32 * sizeof(unsigned long long)));
    DenseGraph *graphs = g.dgraphs.as<DenseGraph>();
    unsigned long long *res = g.accum.as<unsigned long long>();
    hipLaunchKernelGGL(k_dense_plan, dim3(1), dim3(256), 0, s, g.batch_voff, G, g.st.boff.as<int64_t>(),
                       g.st.len.as<int32_t>(), g.st.nv, graphs, res);
    TC_HIP(hipGetLastError());
    unsigned long long h[3];
    TC_HIP(hipMemcpyAsync(h, res, sizeof(h), hipMemcpyDeviceToHost, s));
    TC_HIP(hipStreamSynchronize(s));
    TC_TRY(g.dgid.ensure((size_t)g.st.nv * sizeof(int32_t)));
    hipLaunchKernelGGL(k_dense_gid, dim3(grid_for(g.st.nv, 256, 4096)), dim3(256), 0, s, graphs, G,
                       g.st.nv, g.dgid.as<int32_t>());
    TC_HIP(hipGetLastError());
    if (h[0] <= (unsigned long long)kDenseMax && h[1] * 4 <= (unsigned long long)kDenseBytes &&
        dense_batch_pays((int64_t)h[1] * 4, (int64_t)h[2] * 4, g.st.nv, g.st.nnz))
        g.dense_words = (int64_t)h[1];
    return TC_OK;
}

bool dense_eligible(const Graph &g, const tc_schedule &sched)
{
    // the default rules only: a forced strategy, merge paths or another build
    // of the oriented layout ask for the kernels they name
    if (sched.policy != TC_POLICY_FIXED || sched.ratio_x16 > 0 || sched.mpath_min > 0 ||
        sched.hub_degree > 0 || sched.build != 0)
        return false;
    if (!g.validated) return false;
    if (g.batch_voff) return g.dense_words > 0;
    return g.st.nv <= kDenseMax;
}

int dense_count(Graph &g, uint32_t *out, unsigned long long *acc, int32_t *bad, bool oriented,
                bool skip_lower, hipEvent_t built)
{
    hipStream_t s = g.stream;
    const int32_t nv = g.st.nv;
    DenseArgs A = {};
    A.boff = g.st.boff.as<int64_t>();
    A.len = g.st.len.as<int32_t>();
    A.pool = g.st.pool.as<int32_t>();
    A.nv = nv;
    A.one = DenseGraph{0, nv, dense_chunks(nv), 0, 0};
    const int64_t words = g.batch_voff ? g.dense_words : (int64_t)nv * A.one.nch * kChunkWords;
    if (g.batch_voff) {
        A.graphs = g.dgraphs.as<DenseGraph>();
        A.gid = g.dgid.as<int32_t>();
    }
    TC_TRY(g.dmat.ensure((size_t)words * sizeof(uint32_t)));
    // a row of d > long_len entries has at most 2 d / long_len items
    A.long_len = (int32_t)std::max<int64_t>(kDenseLong, 2 * g.st.nnz / nv);
    A.icap = 2 * (g.st.nnz / A.long_len) + 1;
    constexpr size_t head = (size_t)kParts * kCtrStride * sizeof(unsigned long long);
    TC_TRY(g.ditems.ensure(head + (size_t)(kParts * A.icap) * sizeof(int2)));
    A.mat = g.dmat.as<uint32_t>();
    A.nitems = g.ditems.as<unsigned long long>();
    A.items = reinterpret_cast<int2 *>(g.ditems.as<char>() + head);
    A.out = out;
    A.global = acc;
    A.bad = bad;
    A.skip_lower = skip_lower ? 1 : 0;
    A.check_sym = oriented ? 1 : 0;
    hipLaunchKernelGGL(k_dense_init, dim3(1), dim3(64), 0, s, acc, A.nitems);
    hipLaunchKernelGGL(k_dense_rows, dim3(grid_for(nv, kRowWaves, 1 << 16)), dim3(kRowWaves * kWave), 0, s, A);
    TC_HIP(hipGetLastError());
    if (built) TC_HIP(hipEventRecord(built, s));
    hipLaunchKernelGGL(k_dense_count, dim3(grid_for(std::max<int64_t>(nv, A.icap), 4, 2048)), dim3(256), 0,
                       s, A);
    if (g.batch_per_graph)
        hipLaunchKernelGGL(k_dense_graph_sums, dim3((unsigned)g.batch_ngraphs), dim3(256), 0, s, A.graphs,
                           nv, out, g.batch_per_graph);
    TC_HIP(hipGetLastError());
    return TC_OK;
}

}  // namespace tc

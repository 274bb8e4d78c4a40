// tc_core.hip -- the top of the rank order on a bit matrix (oriented count).
//
// A triangle a < b < w (rank order) whose b is among the K highest ranks has
// its b and w there.  For every vertex a, S(a) = N+(a) within that core; with
// the core's adjacency as bit rows R(b) (both directions),
//     h(a, b) = |S(a) cap R(b)|,  b in S(a),
// meets the triangle twice: at (a, b) and at (a, w).  So out[a] += sum of
// h(a, .), out[b] += 2 h(a, b) over its a, and the total is 3 times the sum:
// no third-vertex counters and no task lists for the core's owners, only an
// AND and a population count of K bits per plus entry that points into the
// core.  The other owners keep the task lists of tc_static.hip.
#include "tc_internal.hpp"

#include <algorithm>

namespace tc {

namespace {

constexpr int kGroup = 8;                    // lanes per bit row: 128 bytes a load
constexpr int kGroups = kWave / kGroup;
constexpr int kCoreCols = kGroup * 4 * 32;   // columns per such load
// Columns: 4096 for one graph (2 MB of bit rows, an XCD's L2 holds them), 8192 (8
// MB) from 200M entries on, where the lists that they take the place of are the
// longer part: R-MAT 24 (edge factor 16) 131.5 -> 125.8 ms, 4M vertices with edge
// factor 32 22.6 -> 21.4, with 16 (130M entries) 10.9 -> 11.0, 1M 2.85 -> 2.90.
// 2048 for each of batched graphs (1024 graphs of 1k to 64k vertices: 24.2 ms
// a count, against 26.2 with 1024, 25.5 with 3072 and 26.3 with 4096, whose
// matrices cost more to build)
constexpr int kCoreOne = 4, kCoreBatch = 2;  // loads per lane and bit row
constexpr int kCoreLarge = 8;
constexpr int64_t kCoreLargeNnz = int64_t(3) << 26;
constexpr int kCoreThreads = 512;
constexpr int kCoreWaves = kCoreThreads / kWave;
constexpr int kGroupRow = 16;                // rows of S(a) up to this long go four to a wave
constexpr int kPartRows = 4096;              // batched: rows of a graph per block
constexpr int64_t kCoreBytes = int64_t(16) << 30;  // all matrices of a batch
// Entries of a batch per core vertex below which its cores cost more to build (256
// bytes a vertex) than they save: 4000 R-MAT graphs of 2000 vertices took 4.6, 5.0,
// 5.5 and 6.0 ms with 1.9, 3.6, 5.2 and 6.8 entries a vertex, without cores 2.9, 3.8,
// 4.7 and 5.5; 500 of 4000 1.5 with 10.5, 1.6 without.
constexpr int64_t kCoreEntries = 8;

// The core of one graph: its ranks below the core are [nb, nb + n - k), its
// core ranks core_lo + [kpre, kpre + k); its bit rows are the matrix's rows
// from kpre.
struct CoreGraph {
    int32_t nb, n, k, kpre;
};
struct CoreBlock {
    int32_t graph, part, parts, pad;
};

// Sum over the 8 lanes of a group (DPP: within quads, then half rows).
__device__ inline uint32_t group_sum(uint32_t x)
{
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xF, 0xF, true);   // quad_perm 1,0,3,2
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xF, 0xF, true);   // quad_perm 2,3,0,1
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x141, 0xF, 0xF, true);  // row_half_mirror
    return x;
}

// Upper half of the cores' bit rows: row b gets N+(b), whole rows written.
// gid: the graph of every rank (batched) or null.
template <int Q>
__global__ __launch_bounds__(256) void k_core_rows(const VInfo *__restrict__ vi,
                                                   const int32_t *__restrict__ padj, int32_t core_lo,
                                                   int32_t k, CoreGraph one,
                                                   const CoreGraph *__restrict__ graphs,
                                                   const int32_t *__restrict__ gid, uint32_t *__restrict__ mat,
                                                   uint32_t *__restrict__ pcount,
                                                   const unsigned long long *__restrict__ fault)
{
    if (*fault) return;  // (rows not symmetric: the plus array was not written)
    constexpr int words = Q * (kCoreCols / 32);
    __shared__ alignas(16) uint32_t lds[256 / kWave][words];
    const int lane = threadIdx.x & (kWave - 1);
    uint32_t *bits = lds[threadIdx.x / kWave];
    const int64_t nwaves = (int64_t)gridDim.x * (blockDim.x / kWave);
    for (int64_t q = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; q < k; q += nwaves) {
        const int32_t b = (int32_t)q;
        if (lane == 0) pcount[b] = 0u;
        const CoreGraph D = graphs ? graphs[gid[core_lo + b]] : one;
        const int32_t clo = core_lo + D.kpre;
        const VInfo x = vi[core_lo + b];
        const int32_t dp = x.len - x.dm;
        const int32_t *row = padj + x.rb;
        for (int i = lane; i < words; i += kWave) bits[i] = 0u;
        wave_sync();
        for (int32_t i = lane; i < dp; i += kWave) {
            const uint32_t c = (uint32_t)(row[i] - clo);
            if (c < (uint32_t)D.k) atomicOr(&bits[c >> 5], 1u << (c & 31));
        }
        wave_sync();
        uint4 *dst = reinterpret_cast<uint4 *>(mat + (int64_t)b * words);
        for (int i = lane; i < words / 4; i += kWave) dst[i] = reinterpret_cast<const uint4 *>(bits)[i];
        wave_sync();
    }
}

// A 64 x 64 block of bits, a row per lane, transposed.
__device__ inline uint64_t transpose_64(uint64_t x)
{
    const int lane = threadIdx.x & (kWave - 1);
    auto step = [&](int s, uint64_t m0) {
        const uint64_t y = shfl_xor_u64(x, s);
        x = (lane & s) == 0 ? (x & m0) | ((y & m0) << s) : (x & ~m0) | ((y & ~m0) >> s);
    };
    step(32, 0x00000000FFFFFFFFull);
    step(16, 0x0000FFFF0000FFFFull);
    step(8, 0x00FF00FF00FF00FFull);
    step(4, 0x0F0F0F0F0F0F0F0Full);
    step(2, 0x3333333333333333ull);
    step(1, 0x5555555555555555ull);
    return x;
}

// The lower half: every 64 x 64 block on or above the diagonal is transposed
// in registers (lane = row) and stored below it.  One graph: its few blocks are
// dealt to all waves (7 us with 4096 ranks, 36 as below).
template <int Q>
__global__ __launch_bounds__(256) void k_core_transpose(CoreGraph D, uint32_t *__restrict__ mat)
{
    const int lane = threadIdx.x & (kWave - 1);
    constexpr int32_t stride = Q * (kCoreCols / 64);
    uint64_t *m = reinterpret_cast<uint64_t *>(mat) + (int64_t)D.kpre * stride;
    const int32_t k = D.k, nb = (k + 63) / 64;
    const int32_t wpb = blockDim.x / kWave, nw = (int32_t)gridDim.x * wpb;
    for (int32_t q = (int32_t)blockIdx.x * wpb + threadIdx.x / kWave; q < nb * nb; q += nw) {
        const int32_t i = q / nb, j = q % nb;
        if (j < i) continue;
        const int32_t ri = 64 * i + lane, rj = 64 * j + lane;
        const uint64_t x0 = ri < k ? m[(int64_t)ri * stride + j] : 0ull;
        const uint64_t x = transpose_64(x0);
        if (rj < k) m[(int64_t)rj * stride + i] = i == j ? x | x0 : x;
    }
}

// Batched graphs: a 1024 x 1024 block of bits per thread block, wave i the 64 x 64
// blocks of its 64 rows, and the results go through LDS, so that rows are read and
// written as whole 128-byte lines (1024 cores: 8 bytes of a line at a time 0.88
// ms, this 0.39).
template <int Q>
__global__ __launch_bounds__(1024) void k_core_transpose_batch(const CoreGraph *__restrict__ graphs,
                                                               uint32_t *__restrict__ mat)
{
    constexpr int W = kCoreCols / 64;              // words of such a block's row
    constexpr int kPairs = Q * (Q + 1) / 2;        // blocks on or above the diagonal
    static_assert(W == 16, "a wave per 64 rows");
    __shared__ uint64_t tile[kCoreCols][W + 1];
    const int t = threadIdx.x, lane = t & (kWave - 1), wid = t / kWave;
    const CoreGraph D = graphs[blockIdx.x / kPairs];
    int I = 0, J = (int)(blockIdx.x % kPairs);
    while (J >= Q - I) J -= Q - I++;
    J += I;
    constexpr int32_t stride = Q * W;
    uint64_t *m = reinterpret_cast<uint64_t *>(mat) + (int64_t)D.kpre * stride;
    const int32_t k = D.k;
    if (J * kCoreCols >= k) return;  // (the whole block: no such rows or columns)
    const int32_t r = I * kCoreCols + 64 * wid + lane;
    uint64_t x[W];
    const ulonglong2 *src = reinterpret_cast<const ulonglong2 *>(m + (int64_t)(r < k ? r : 0) * stride + J * W);
#pragma unroll
    for (int j = 0; j < W; j += 2) {
        const ulonglong2 v = r < k ? src[j / 2] : make_ulonglong2(0ull, 0ull);
        x[j] = v.x;
        x[j + 1] = v.y;
    }
#pragma unroll
    for (int j = 0; j < W; ++j) {
        if (I == J && j < wid) continue;  // (below the diagonal: the whole wave)
        const uint64_t y = transpose_64(x[j]);
        tile[64 * j + lane][wid] = I == J && j == wid ? y | x[j] : y;
    }
    __syncthreads();
    for (int q = t; q < kCoreCols * W / 2; q += 1024) {
        const int row = q / (W / 2), c = 2 * (q % (W / 2)), last = I == J ? row / 64 : W - 1;
        if (J * kCoreCols + row >= k || c > last) continue;
        uint64_t *dst = m + (int64_t)(J * kCoreCols + row) * stride + I * W + c;
        if (c < last)
            *reinterpret_cast<ulonglong2 *>(dst) = make_ulonglong2(tile[row][c], tile[row][c + 1]);
        else
            *dst = tile[row][c];
    }
}

struct CoreArgs {
    const VInfo *vi;
    const int32_t *padj;
    const uint32_t *mat;
    int32_t core_lo;
    CoreGraph one;
    const CoreGraph *graphs;  // batched (else null): graphs and the blocks' shares of them
    const CoreBlock *blocks;
    int32_t nblocks;
    uint32_t *outr;
    uint32_t *pcount;  // plus entries that point to each core vertex, zero on entry
    unsigned long long *global;
    unsigned long long *per_graph;  // may be null
    const unsigned long long *fault;
};

template <int Q>
struct CoreShared {
    uint32_t cnt[Q * kCoreCols];
    uint32_t pairs[Q * kCoreCols / 2];  // two 16-bit counts a word
    alignas(16) uint32_t bits[kCoreWaves][4][Q * (kCoreCols / 32)];
};

// The group's entries lst[first], lst[first + step], ... below n against the
// bits of S(a), two of them in flight: h of each is credited, their sum
// returned (the same in the group's lanes).
template <int Q>
__device__ inline uint32_t core_run(CoreShared<Q> &S, const char *__restrict__ mat, int32_t clo,
                                    const int32_t *__restrict__ lst, int32_t n, int32_t first, int32_t step,
                                    int32_t iters, const uint32_t *bits)
{
    constexpr int U = 2;
    const int i = threadIdx.x & (kGroup - 1);
    uint4 A[Q];
#pragma unroll
    for (int c = 0; c < Q; ++c) A[c] = reinterpret_cast<const uint4 *>(bits)[c * kGroup + i];
    uint32_t sum = 0;
    int32_t nw[U];  // the next entries, loaded while these rows are
#pragma unroll
    for (int u = 0; u < U; ++u) nw[u] = lst[first + u * step < n ? first + u * step : 0];
#pragma unroll 1
    for (int32_t it = 0; it < iters; ++it) {
        uint32_t col[U];
        bool in[U];
        uint4 R[U][Q];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int32_t e = first + (it * U + u) * step, e2 = e + U * step;
            in[u] = e < n;
            col[u] = in[u] ? (uint32_t)(nw[u] - clo) : 0u;
            nw[u] = lst[e2 < n ? e2 : 0];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int c = 0; c < Q; ++c)
                R[u][c] = *reinterpret_cast<const uint4 *>(mat + (col[u] * (Q * 128) + c * 128 + i * 16));
#pragma unroll
        for (int u = 0; u < U; ++u) {
            uint32_t p = 0;
#pragma unroll
            for (int c = 0; c < Q; ++c)
                p += __popc(R[u][c].x & A[c].x) + __popc(R[u][c].y & A[c].y) +
                     __popc(R[u][c].z & A[c].z) + __popc(R[u][c].w & A[c].w);
            const uint32_t h = in[u] ? group_sum(p) : 0u;
            sum += h;
            if (in[u] && i < 2)
                atomicAdd(i == 0 ? &S.cnt[col[u]] : &S.pairs[col[u] >> 1],
                          i == 0 ? h : 1u << (16 * (col[u] & 1)));
        }
    }
    return sum;
}

// The rows of one block's share of a graph (part of parts).  One wave takes 64
// rows a at a time: a lane finds where the core part of its N+ begins (a
// binary search), then S(a) is built as bits in LDS, read into registers by
// every 8-lane group, and ANDed with R(b), one b per group: eight b of one a,
// or, where S(a) has at most 16 entries, two b of four a.  (8 lanes a group:
// what is not AND and count is paid once for 8 b; on 1024 batched graphs 3.6
// ms, 4.5 with 16 lanes.)
template <int Q>
__device__ inline unsigned long long core_rows(CoreShared<Q> &S, const CoreArgs &A, const CoreGraph &D,
                                               int32_t part, int32_t parts)
{
    constexpr int kWords = Q * (kCoreCols / 32);
    const int lane = threadIdx.x & (kWave - 1), i = lane & (kGroup - 1), grp = lane / kGroup;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const char *mat = reinterpret_cast<const char *>(A.mat + (int64_t)D.kpre * kWords);
    const int32_t clo = A.core_lo + D.kpre, nlow = D.n - D.k;
    // row q of the graph as a rank: its lower ranks, then its core
    auto rank_of = [&](int64_t q) { return q < nlow ? D.nb + q : clo + (q - nlow); };
    unsigned long long total = 0;
    // Rows are dealt to all waves of the graph four at a time (64 bytes of
    // vertex records): neighbouring ranks have similar rows, and the top 512 in
    // one block made the others wait for it (3.35 -> 0.32 ms at R-MAT 20)
    const int64_t nwaves = (int64_t)parts * kCoreWaves;
    const int64_t wave = (int64_t)part * kCoreWaves + wid;
    for (int64_t q0 = wave; q0 * 4 < D.n; q0 += nwaves * (kWave / 4)) {
        const int64_t q = (q0 + nwaves * (lane >> 2)) * 4 + (lane & 3);
        const int32_t r = q < D.n ? (int32_t)rank_of(q) : 0;
        int32_t n = 0;
        int64_t lb = 0;
        if (q < D.n) {
            const VInfo x = A.vi[r];
            const int32_t dp = x.len - x.dm;
            int32_t lo = 0, hi = q >= nlow ? 0 : dp;
            while (lo < hi) {
                const int32_t mid = (lo + hi) >> 1;
                if (A.padj[x.rb + mid] < clo) lo = mid + 1; else hi = mid;
            }
            n = dp - lo;
            lb = x.rb + lo;
        }
        if (n == 1) {  // no pair, but an entry to count
            const uint32_t c = (uint32_t)(A.padj[lb] - clo);
            atomicAdd(&S.pairs[c >> 1], 1u << (16 * (c & 1)));
        }
        // rows of a few entries, four at a time, 16 lanes each
        for (uint64_t m = __ballot(n >= 2 && n <= kGroupRow); m;) {
            int j = -1;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                if (lane / 16 == g && m) j = __ffsll((unsigned long long)m) - 1;
                m &= m - 1;
            }
            const int src = max(j, 0), i16 = lane & 15;
            // (shuffles by every lane: src may sit in an idle group)
            const int32_t sn = __shfl(n, src, kWave), sr = __shfl(r, src, kWave);
            const int32_t gn = j < 0 ? 0 : sn;
            const int64_t glb = ((int64_t)__shfl((int32_t)(lb >> 32), src, kWave) << 32) |
                                (uint32_t)__shfl((int32_t)lb, src, kWave);
            uint32_t *bits = S.bits[wid][lane / 16];
            for (int w = i16; w < kWords / 4; w += 16) reinterpret_cast<uint4 *>(bits)[w] = make_uint4(0, 0, 0, 0);
            wave_sync();
            const int32_t *lst = A.padj + (gn > 0 ? glb : 0);
            if (i16 < gn) {
                const uint32_t c = (uint32_t)(lst[i16] - clo);
                atomicOr(&bits[c >> 5], 1u << (c & 31));
            }
            wave_sync();
            int32_t most = gn;  // over the rows
            most = max(most, __shfl_xor(most, 16, kWave));
            most = max(most, __shfl_xor(most, 32, kWave));
            const uint32_t h = core_run<Q>(S, mat, clo, lst, gn, grp & 1, 2,
                                           (__builtin_amdgcn_readfirstlane(most) + 3) / 4, bits);
            if (i == 0 && h) {
                atomicAdd(&A.outr[sr], h);
                total += h;
            }
            wave_sync();
        }
        // longer rows, one at a time
        for (uint64_t m = __ballot(n > kGroupRow); m; m &= m - 1) {
            const int j = __ffsll((unsigned long long)m) - 1;
            const int32_t rn = __builtin_amdgcn_readlane(n, j);
            const int64_t rlb = ((int64_t)__builtin_amdgcn_readlane((int32_t)(lb >> 32), j) << 32) |
                                (uint32_t)__builtin_amdgcn_readlane((int32_t)lb, j);
            const int32_t *lst = A.padj + rlb;
            uint32_t *bits = S.bits[wid][0];
            for (int w = lane; w < kWords; w += kWave) bits[w] = 0u;
            wave_sync();
            for (int32_t e = lane; e < rn; e += kWave) {
                const uint32_t c = (uint32_t)(lst[e] - clo);
                atomicOr(&bits[c >> 5], 1u << (c & 31));
            }
            wave_sync();
            uint32_t h = core_run<Q>(S, mat, clo, lst, rn, grp, kGroups,
                                     (rn + 2 * kGroups - 1) / (2 * kGroups), bits);
            h += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)h, 0x140, 0xF, 0xF, true);  // row_mirror
            const uint32_t sum = (uint32_t)__builtin_amdgcn_readlane((int)h, 0) +
                                 (uint32_t)__builtin_amdgcn_readlane((int)h, 16) +
                                 (uint32_t)__builtin_amdgcn_readlane((int)h, 32) +
                                 (uint32_t)__builtin_amdgcn_readlane((int)h, 48);
            if (lane == j && sum) {
                atomicAdd(&A.outr[r], sum);
                total += sum;
            }
            wave_sync();
        }
    }
    return total;
}

// Lane 0 of a group adds h to b's counter in LDS, lane 1 counts the entry (the
// symmetry check: b must be met |N-(b)| times); both are flushed once per
// block.  Bound by L2 reads of bit rows: the 2 MB of 4096 columns fit each XCD's L2
// (R-MAT 24 with 4096: 18.7 TB/s), the 8 MB of 8192 do not, and a third of the 191
// GB that R-MAT 24 reads comes from beyond (17.8 TB/s, 10.7 ms).
template <int Q>
__global__ __launch_bounds__(kCoreThreads, Q <= 2 ? 7 : Q <= 4 ? 6 : 2) void k_core_count(CoreArgs A)
{
    __shared__ CoreShared<Q> S;
    if (*A.fault) return;  // (set before this kernel: the same for all)
    const int t = threadIdx.x;
    CoreGraph D = A.one;
    int32_t part = blockIdx.x, parts = gridDim.x, graph = 0;
    if (A.blocks) {
        // blocks go to the XCDs in turn: each takes one run of the table, so
        // that a graph's bit rows are read through one L2
        const int32_t per = (A.nblocks + 7) / 8;
        const int32_t e = (int32_t)(blockIdx.x & 7) * per + (int32_t)(blockIdx.x >> 3);
        if (e >= A.nblocks || (int32_t)(blockIdx.x >> 3) >= per) return;
        const CoreBlock B = A.blocks[e];
        graph = B.graph;
        part = B.part;
        parts = B.parts;
        D = A.graphs[graph];
    }
    for (int q = t; q < D.k; q += kCoreThreads) S.cnt[q] = 0u;
    for (int q = t; q < (D.k + 1) / 2; q += kCoreThreads) S.pairs[q] = 0u;
    __syncthreads();
    const unsigned long long total = core_rows<Q>(S, A, D, part, parts);
    __syncthreads();
    const int32_t clo = A.core_lo + D.kpre;
    for (int32_t q = t; q < D.k; q += kCoreThreads) {
        const uint32_t c = S.cnt[q], p = (S.pairs[q >> 1] >> (16 * (q & 1))) & 0xFFFFu;
        if (c) atomicAdd(&A.outr[clo + q], 2u * c);
        if (p) atomicAdd(&A.pcount[D.kpre + q], p);
    }
    const unsigned long long part3[1] = {3ull * total};
    block_add_u64<1>(part3, A.global);
    if (A.per_graph) {
        __syncthreads();
        block_add_u64<1>(part3, &A.per_graph[graph]);
    }
}

// Every core vertex was met by |N-(b)| plus entries.
__global__ void k_core_check(const VInfo *__restrict__ vi, int32_t core_lo, int32_t k,
                             const uint32_t *__restrict__ pcount, int32_t *__restrict__ bad)
{
    const int32_t q = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);
    if (q < k && pcount[q] != (uint32_t)vi[core_lo + q].dm) atomicOr(bad, 1);
}

// One block: the cores of batched graphs and the blocks that count them; res =
// {core vertices, blocks} of all, and whether the boundaries are
// not an ascending cover of the nv vertices.
__global__ __launch_bounds__(256) void k_core_plan(const int64_t *__restrict__ voff, int32_t G, int32_t nv,
                                                   CoreGraph *__restrict__ graphs,
                                                   CoreBlock *__restrict__ blocks,
                                                   unsigned long long *__restrict__ res)
{
    __shared__ long long part[2][256];
    const int t = threadIdx.x;
    const int64_t per = (G + 255) / 256, g0 = min(t * per, (int64_t)G), g1 = min(g0 + per, (int64_t)G);
    auto core_of = [](int64_t n) { return (int32_t)min(n, (int64_t)kCoreBatch * kCoreCols); };
    auto parts_of = [](int64_t n) { return (int32_t)((n + kPartRows - 1) / kPartRows); };
    long long before[2] = {0, 0}, all[2] = {0, 0};
    bool odd = t == 0 && (voff[0] != 0 || voff[G] != nv);
    for (int64_t g = g0; g < g1; ++g) {
        const int64_t n = voff[g + 1] - voff[g];
        odd = odd || n < 0;
        before[0] += core_of(n);
        before[1] += parts_of(n);
    }
    for (int q = 0; q < 2; ++q) part[q][t] = before[q];
    if (__syncthreads_or(odd)) {  // (no tables: sums over such boundaries mean nothing)
        if (t == 0) res[2] = 1ull;
        return;
    }
    for (int q = 0; q < 2; ++q) {
        before[q] = 0;
        for (int i = 0; i < 256; ++i) {
            if (i < t) before[q] += part[q][i];
            all[q] += part[q][i];
        }
    }
    for (int64_t g = g0; g < g1; ++g) {
        const int64_t n = voff[g + 1] - voff[g];
        const CoreGraph D = {(int32_t)(voff[g] - before[0]), (int32_t)n, core_of(n), (int32_t)before[0]};
        graphs[g] = D;
        const int32_t parts = parts_of(n);
        for (int32_t i = 0; i < parts; ++i) blocks[before[1] + i] = CoreBlock{(int32_t)g, i, parts, 0};
        before[0] += D.k;
        before[1] += parts;
    }
    if (t == 0) {
        res[0] = (unsigned long long)all[0];
        res[1] = (unsigned long long)all[1];
        res[2] = 0ull;
    }
}

// Batched graphs, ranks by (graph, degree, id) in order: every graph's core is
// moved behind all other ranks, (core, graph, degree, id) -- still ascending by
// degree within a graph, where all edges are.  order2 and rnk receive it.
__global__ void k_core_order(const int32_t *__restrict__ order, const int32_t *__restrict__ vgid,
                             const CoreGraph *__restrict__ graphs, int32_t nv, int32_t core_lo,
                             int32_t *__restrict__ order2, int32_t *__restrict__ rnk)
{
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < nv;
         p += (int64_t)gridDim.x * blockDim.x) {
        const int32_t v = order[p];
        const CoreGraph D = graphs[vgid[v]];
        const int64_t i = p - ((int64_t)D.nb + D.kpre);  // rank within the graph
        const int64_t r = i < D.n - D.k ? D.nb + i : (int64_t)core_lo + D.kpre + (i - (D.n - D.k));
        order2[r] = v;
        rnk[v] = (int32_t)r;
    }
}

}  // namespace

int core_plan_batched(Graph &g)
{
    g.core_total = 0;
    const int32_t G = g.batch_ngraphs;
    if (G <= 0 || g.st.nv == 0) return TC_OK;
    hipStream_t s = g.stream;
    TC_TRY(g.cgraphs.ensure((size_t)G * sizeof(CoreGraph)));
    TC_TRY(g.accum.ensure(32 * sizeof(unsigned long long)));
    unsigned long long *res = g.accum.as<unsigned long long>();
    const int64_t most = G + g.st.nv / kPartRows + 1;  // blocks, at most
    TC_TRY(g.cblocks.ensure((size_t)most * sizeof(CoreBlock)));
    hipLaunchKernelGGL(k_core_plan, dim3(1), dim3(256), 0, s, g.batch_voff, G, g.st.nv,
                       g.cgraphs.as<CoreGraph>(), g.cblocks.as<CoreBlock>(), res);
    TC_HIP(hipGetLastError());
    unsigned long long h[3];
    TC_HIP(hipMemcpyAsync(h, res, sizeof(h), hipMemcpyDeviceToHost, s));
    TC_HIP(hipStreamSynchronize(s));
    if (h[2] || h[0] * (kCoreBatch * kCoreCols / 8) > (unsigned long long)kCoreBytes) return TC_OK;
    g.core_total = (int32_t)h[0];
    g.core_blocks = (int32_t)h[1];
    return TC_OK;
}

int core_order_batched(Graph &g, const int32_t *order, const int32_t *vgid, int32_t *order2, int32_t *rnk)
{
    const int32_t nv = g.st.nv;
    hipLaunchKernelGGL(k_core_order, dim3(grid_for(nv, 256, 65536)), dim3(256), 0, g.stream, order, vgid,
                       g.cgraphs.as<CoreGraph>(), nv, nv - g.core_total, order2, rnk);
    TC_HIP(hipGetLastError());
    return TC_OK;
}

int32_t core_size(const Graph &g, const tc_schedule &sched)
{
    if ((sched.policy != TC_POLICY_FIXED && sched.policy != TC_POLICY_LEARNED) || sched.ratio_x16 > 0 ||
        sched.mpath_min > 0 || sched.hub_degree > 0 || sched.build != 0)
        return 0;
    if (g.batch_voff) return g.st.nnz >= kCoreEntries * g.core_total ? g.core_total : 0;
    const int32_t k = (g.st.nnz >= kCoreLargeNnz ? kCoreLarge : kCoreOne) * kCoreCols;
    return g.st.nv > 4 * k ? k : 0;
}

namespace {

template <int Q>
int core_launch(Graph &g, CoreArgs A, int32_t *bad, const int32_t *gid, int64_t grid)
{
    hipStream_t s = g.stream;
    const int32_t k = g.core_k;
    const size_t words = (size_t)k * Q * (kCoreCols / 32);
    TC_TRY(g.cmat.ensure((words + (size_t)k) * sizeof(uint32_t)));
    uint32_t *mat = g.cmat.as<uint32_t>();
    A.mat = mat;
    A.pcount = mat + words;
    hipLaunchKernelGGL(k_core_rows<Q>, dim3(grid_for(k, 4)), dim3(256), 0, s, A.vi, A.padj, A.core_lo, k, A.one,
                       A.graphs, gid, mat, A.pcount, A.fault);
    if constexpr (Q == kCoreBatch)
        hipLaunchKernelGGL(k_core_transpose_batch<Q>, dim3((unsigned)((int64_t)g.batch_ngraphs * (Q * (Q + 1) / 2))),
                           dim3(1024), 0, s, A.graphs, mat);
    else
        hipLaunchKernelGGL(k_core_transpose<Q>, dim3(512), dim3(256), 0, s, A.one, mat);
    hipLaunchKernelGGL(k_core_count<Q>, dim3((unsigned)grid), dim3(kCoreThreads), 0, s, A);
    hipLaunchKernelGGL(k_core_check, dim3(grid_for(k, 256)), dim3(256), 0, s, A.vi, A.core_lo, k, A.pcount, bad);
    TC_HIP(hipGetLastError());
    return TC_OK;
}

}  // namespace

int core_count(Graph &g, unsigned long long *acc, int32_t *bad, const int32_t *gid)
{
    const int32_t nv = g.st.nv, k = g.core_k;
    CoreArgs A = {};
    A.one = CoreGraph{0, nv, k, 0};
    A.vi = g.vinfo.as<VInfo>();
    A.padj = g.padj.as<int32_t>();
    A.core_lo = nv - k;
    A.outr = g.outr.as<uint32_t>();
    A.global = acc;
    A.fault = acc + 27;
    if (g.batch_voff) {
        A.graphs = g.cgraphs.as<CoreGraph>();
        A.blocks = g.cblocks.as<CoreBlock>();
        A.nblocks = g.core_blocks;
        A.per_graph = g.batch_per_graph;
        return core_launch<kCoreBatch>(g, A, bad, gid, 8 * ceil_div(A.nblocks, 8));
    }
    // a block counts the entries of each core vertex in 16 bits: at most 2^15
    // rows a block (and three blocks a CU otherwise)
    int dev = 0, cus = 0;
    TC_HIP(hipGetDevice(&dev));
    TC_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int64_t grid = std::min<int64_t>(ceil_div(nv, kCoreThreads),
                                           std::max<int64_t>(3 * cus, ceil_div(nv, 1 << 15)));
    return k > kCoreOne * kCoreCols ? core_launch<kCoreLarge>(g, A, bad, nullptr, grid)
                                    : core_launch<kCoreOne>(g, A, bad, nullptr, grid);
}

}  // namespace tc

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

constexpr int kGroup = 16;                   // lanes per bit row: 256 bytes a load
constexpr int kCoreCols = kGroup * 4 * 32;   // columns per such load
constexpr int kCoreMax = kCoreCols * 2;      // widest core
constexpr int kCoreThreads = 512;
constexpr int kCoreWaves = kCoreThreads / kWave;
constexpr int kGroups = kWave / kGroup;
constexpr int kGroupRow = 16;            // rows of S(a) up to this long go four to a wave

__device__ inline void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sum over the 16 lanes of a row (DPP: within quads, halves, rows).
__device__ inline uint32_t row16_sum(uint32_t x)
{
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xF, 0xF, true);   // quad_perm 1,0,3,2
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xF, 0xF, true);   // quad_perm 2,3,0,1
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x141, 0xF, 0xF, true);  // row_half_mirror
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x140, 0xF, 0xF, true);  // row_mirror
    return x;
}

// Upper half of the core's bit rows: row b gets N+(b), whole rows written.
__global__ __launch_bounds__(256) void k_core_rows(const VInfo *__restrict__ vi,
                                                   const int32_t *__restrict__ padj, int32_t core_lo,
                                                   int32_t k, int32_t words, uint32_t *__restrict__ mat)
{
    __shared__ alignas(16) uint32_t lds[256 / kWave][kCoreMax / 32];
    const int lane = threadIdx.x & (kWave - 1);
    uint32_t *bits = lds[threadIdx.x / kWave];
    const int32_t b = (int32_t)(blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave);
    if (b >= k) return;  // (no block barrier below)
    const VInfo x = vi[core_lo + b];
    const int32_t dp = x.len - x.dm;
    const int32_t *row = padj + x.rb;
    for (int i = lane; i < words; i += kWave) bits[i] = 0u;
    wave_lds_sync();
    for (int32_t i = lane; i < dp; i += kWave) {
        const uint32_t c = (uint32_t)(row[i] - core_lo);
        if (c < (uint32_t)k) atomicOr(&bits[c >> 5], 1u << (c & 31));
    }
    wave_lds_sync();
    for (int i = lane; i < words / 4; i += kWave)
        reinterpret_cast<uint4 *>(mat + (int64_t)b * words)[i] = reinterpret_cast<const uint4 *>(bits)[i];
}

// The lower half: every 64 x 64 block on or above the diagonal is transposed
// in registers (lane = row) and stored below it.
__global__ __launch_bounds__(256) void k_core_transpose(int32_t k, int32_t words, uint64_t *__restrict__ mat)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int32_t nb = (k + 63) / 64;
    const int32_t q = (int32_t)(blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave);
    const int32_t i = q / nb, j = q % nb;
    if (i >= nb || j < i) return;
    const int32_t stride = words / 2;
    const int32_t ri = 64 * i + lane, rj = 64 * j + lane;
    const uint64_t x0 = ri < k ? mat[(int64_t)ri * stride + j] : 0ull;
    uint64_t x = x0;
    for (int s = 32; s > 0; s >>= 1) {
        const uint64_t m0 = s == 32 ? 0x00000000FFFFFFFFull : s == 16 ? 0x0000FFFF0000FFFFull
                          : s == 8 ? 0x00FF00FF00FF00FFull : s == 4 ? 0x0F0F0F0F0F0F0F0Full
                          : s == 2 ? 0x3333333333333333ull : 0x5555555555555555ull;
        const uint64_t y = shfl_xor_u64(x, s);
        x = (lane & s) == 0 ? (x & m0) | ((y & m0) << s) : (x & ~m0) | ((y & ~m0) >> s);
    }
    if (rj < k) mat[(int64_t)rj * stride + i] = i == j ? x | x0 : x;
}

struct CoreArgs {
    const VInfo *vi;
    const int32_t *padj;
    const uint4 *mat;
    int32_t nv, core_lo, k;
    uint32_t *outr;
    uint32_t *pcount;  // [k] plus entries that point to each core vertex, zero on entry
    unsigned long long *global;
};

// One wave takes 64 rows a at a time: a lane finds where the core part of its
// N+ begins (a binary search), then S(a) is built as bits in LDS, read into
// registers by every 16-lane group, and ANDed with R(b), one b per group: four
// b of one a, or, where S(a) has at most 16 entries, one b of four a.  Lane 0
// of a group adds h to b's counter, lane 1 counts the entry (the symmetry
// check: b must be met |N-(b)| times).  Bound by L2 reads of bit rows (2 MB for
// 4096 columns: an XCD's L2 holds all of it).
template <int CH>
__global__ __launch_bounds__(kCoreThreads, 6) void k_core_count(CoreArgs A)
{
    constexpr int kWords = CH * kGroup * 4;  // per row
    __shared__ uint32_t cnt[CH * kCoreCols];
    __shared__ uint32_t pairs[CH * kCoreCols / 2];  // two 16-bit counts a word
    __shared__ alignas(16) uint32_t lds[kCoreWaves][kGroups][kWords];
    const int t = threadIdx.x, lane = t & (kWave - 1), i = lane & (kGroup - 1), grp = lane / kGroup;
    const int wid = __builtin_amdgcn_readfirstlane(t / kWave);
    const char *mat = reinterpret_cast<const char *>(A.mat);
    for (int q = t; q < CH * kCoreCols; q += kCoreThreads) cnt[q] = 0u;
    for (int q = t; q < CH * kCoreCols / 2; q += kCoreThreads) pairs[q] = 0u;
    __syncthreads();
    unsigned long long total = 0;
    // the group's entries lst[first], lst[first + step], ... below n against
    // S, U of them in flight; returns the hits (the same in the group's lanes)
    auto run = [&](const int32_t *lst, int32_t n, int32_t first, int32_t step, int32_t iters,
                   const uint32_t *bits) -> uint32_t {
        constexpr int U = 2;
        uint4 S[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) S[c] = reinterpret_cast<const uint4 *>(bits)[c * kGroup + i];
        uint32_t sum = 0;
        int32_t nw[U];  // the next entries, loaded while these rows are
#pragma unroll
        for (int u = 0; u < U; ++u) nw[u] = lst[first + u * step < n ? first + u * step : 0];
#pragma unroll 1
        for (int32_t it = 0; it < iters; ++it) {
            uint32_t col[U];
            bool in[U];
            uint4 R[U][CH];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int32_t e = first + (it * U + u) * step, e2 = e + U * step;
                in[u] = e < n;
                col[u] = in[u] ? (uint32_t)(nw[u] - A.core_lo) : 0u;
                nw[u] = lst[e2 < n ? e2 : 0];
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int c = 0; c < CH; ++c)
                    R[u][c] = *reinterpret_cast<const uint4 *>(mat + (col[u] * (kWords * 4) + c * 256 + i * 16));
#pragma unroll
            for (int u = 0; u < U; ++u) {
                uint32_t p = 0;
#pragma unroll
                for (int c = 0; c < CH; ++c)
                    p += __popc(R[u][c].x & S[c].x) + __popc(R[u][c].y & S[c].y) +
                         __popc(R[u][c].z & S[c].z) + __popc(R[u][c].w & S[c].w);
                const uint32_t h = in[u] ? row16_sum(p) : 0u;
                sum += h;
                if (in[u] && i < 2)
                    atomicAdd(i == 0 ? &cnt[col[u]] : &pairs[col[u] >> 1],
                              i == 0 ? h : 1u << (16 * (col[u] & 1)));
            }
        }
        return sum;
    };
    // Rows are dealt to all waves four at a time (64 bytes of vertex records):
    // neighbouring ranks have similar rows, and the top 512 in one block made
    // the others wait for it
    const int64_t nwaves = (int64_t)gridDim.x * kCoreWaves;
    const int64_t wave = (int64_t)blockIdx.x * kCoreWaves + wid;
    for (int64_t q0 = wave; q0 * 4 < A.nv; q0 += nwaves * (kWave / 4)) {
        const int64_t r = (q0 + nwaves * (lane >> 2)) * 4 + (lane & 3);
        int32_t n = 0;
        int64_t lb = 0;
        if (r < A.nv) {
            const VInfo x = A.vi[r];
            const int32_t dp = x.len - x.dm;
            int32_t lo = 0, hi = r >= A.core_lo ? 0 : dp;
            while (lo < hi) {
                const int32_t mid = (lo + hi) >> 1;
                if (A.padj[x.rb + mid] < A.core_lo) lo = mid + 1; else hi = mid;
            }
            n = dp - lo;
            lb = x.rb + lo;
        }
        if (n == 1) {  // no pair, but an entry to count
            const uint32_t c = (uint32_t)(A.padj[lb] - A.core_lo);
            atomicAdd(&pairs[c >> 1], 1u << (16 * (c & 1)));
        }
        // rows of a few entries, four at a time
        for (uint64_t m = __ballot(n >= 2 && n <= kGroupRow); m;) {
            int j = -1;
            uint64_t mm = m;
#pragma unroll
            for (int g = 0; g < kGroups; ++g) {
                if (grp == g && mm) j = __ffsll((unsigned long long)mm) - 1;
                mm &= mm - 1;
                if (!mm) mm = 0;
            }
            m = mm;
            const int src = max(j, 0);
            const int32_t sn = __shfl(n, src, kWave);  // (by every lane: src may sit in an idle group)
            const int32_t gn = j < 0 ? 0 : sn;
            const int64_t glb = ((int64_t)__shfl((int32_t)(lb >> 32), src, kWave) << 32) |
                                (uint32_t)__shfl((int32_t)lb, src, kWave);
            uint32_t *bits = lds[wid][grp];
#pragma unroll
            for (int c = 0; c < CH; ++c) reinterpret_cast<uint4 *>(bits)[c * kGroup + i] = make_uint4(0, 0, 0, 0);
            wave_lds_sync();
            const int32_t *lst = A.padj + glb;
            if (i < gn) {
                const uint32_t c = (uint32_t)(lst[i] - A.core_lo);
                atomicOr(&bits[c >> 5], 1u << (c & 31));
            }
            wave_lds_sync();
            int32_t most = gn;  // over the groups
            most = max(most, __shfl_xor(most, 16, kWave));
            most = max(most, __shfl_xor(most, 32, kWave));
            const uint32_t h = run(gn > 0 ? lst : A.padj, gn, 0, 1, (__builtin_amdgcn_readfirstlane(most) + 1) / 2, bits);
            if (i == 0 && h) {
                atomicAdd(&A.outr[(q0 + nwaves * (src >> 2)) * 4 + (src & 3)], h);
                total += h;
            }
            wave_lds_sync();
        }
        // longer rows, one at a time
        for (uint64_t m = __ballot(n > kGroupRow); m; m &= m - 1) {
            const int j = __ffsll((unsigned long long)m) - 1;
            const int32_t rn = __builtin_amdgcn_readlane(n, j);
            const int64_t rlb = ((int64_t)__builtin_amdgcn_readlane((int32_t)(lb >> 32), j) << 32) |
                                (uint32_t)__builtin_amdgcn_readlane((int32_t)lb, j);
            const int32_t *lst = A.padj + rlb;
            uint32_t *bits = lds[wid][0];
            for (int q = lane; q < kWords; q += kWave) bits[q] = 0u;
            wave_lds_sync();
            for (int32_t e = lane; e < rn; e += kWave) {
                const uint32_t c = (uint32_t)(lst[e] - A.core_lo);
                atomicOr(&bits[c >> 5], 1u << (c & 31));
            }
            wave_lds_sync();
            const uint32_t h = run(lst, rn, grp, kGroups, (rn + 2 * kGroups - 1) / (2 * kGroups), bits);
            const uint32_t sum = (uint32_t)__builtin_amdgcn_readlane((int)h, 0) +
                                 (uint32_t)__builtin_amdgcn_readlane((int)h, 16) +
                                 (uint32_t)__builtin_amdgcn_readlane((int)h, 32) +
                                 (uint32_t)__builtin_amdgcn_readlane((int)h, 48);
            if (lane == 0 && sum) {
                atomicAdd(&A.outr[(q0 + nwaves * (j >> 2)) * 4 + (j & 3)], sum);
                total += sum;
            }
            wave_lds_sync();
        }
    }
    __syncthreads();
    for (int32_t q = t; q < A.k; q += kCoreThreads) {
        const uint32_t c = cnt[q], p = (pairs[q >> 1] >> (16 * (q & 1))) & 0xFFFFu;
        if (c) atomicAdd(&A.outr[A.core_lo + q], 2u * c);
        if (p) atomicAdd(&A.pcount[q], p);
    }
    const unsigned long long part[1] = {3ull * total};
    block_add_u64<1>(part, A.global);
}

// Every core vertex was met by |N-(b)| plus entries.
__global__ void k_core_check(const VInfo *__restrict__ vi, int32_t core_lo, int32_t k,
                             const uint32_t *__restrict__ pcount, int32_t *__restrict__ bad)
{
    const int32_t q = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);
    if (q < k && pcount[q] != (uint32_t)vi[core_lo + q].dm) atomicOr(bad, 1);
}

__global__ void k_zero_u32s(uint32_t *p, int32_t n)
{
    const int32_t q = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);
    if (q < n) p[q] = 0u;
}

}  // namespace

int32_t core_size(const Graph &g, const tc_schedule &sched)
{
    if ((sched.policy != TC_POLICY_FIXED && sched.policy != TC_POLICY_LEARNED) || sched.ratio_x16 > 0 ||
        sched.mpath_min > 0 || sched.hub_degree > 0 || sched.build != 0 || g.batch_voff)
        return 0;
    return g.st.nv > 4 * kCoreMax ? kCoreMax : 0;
}

int core_count(Graph &g, unsigned long long *acc, int32_t *bad)
{
    hipStream_t s = g.stream;
    const int32_t nv = g.st.nv, k = g.core_k, lo = nv - k;
    constexpr int CH = kCoreMax / kCoreCols;
    constexpr int32_t words = kCoreMax / 32;
    TC_TRY(g.cmat.ensure((size_t)k * words * sizeof(uint32_t) + (size_t)k * sizeof(uint32_t)));
    uint32_t *mat = g.cmat.as<uint32_t>();
    uint32_t *pcount = mat + (size_t)k * words;
    const VInfo *vi = g.vinfo.as<VInfo>();
    const int32_t *padj = g.padj.as<int32_t>();
    hipLaunchKernelGGL(k_core_rows, dim3(grid_for(k, 4)), dim3(256), 0, s, vi, padj, lo, k, words, mat);
    const int64_t nb = ceil_div(k, 64);
    hipLaunchKernelGGL(k_core_transpose, dim3(grid_for(nb * nb, 4)), dim3(256), 0, s, k, words,
                       reinterpret_cast<uint64_t *>(mat));
    hipLaunchKernelGGL(k_zero_u32s, dim3(grid_for(k, 256)), dim3(256), 0, s, pcount, k);
    TC_HIP(hipGetLastError());
    CoreArgs A = {};
    A.vi = vi;
    A.padj = padj;
    A.mat = reinterpret_cast<const uint4 *>(mat);
    A.nv = nv;
    A.core_lo = lo;
    A.k = k;
    A.outr = g.outr.as<uint32_t>();
    A.pcount = pcount;
    A.global = acc;
    // a block counts the entries of each core vertex in 16 bits: at most
    // 2^15 rows a block (and three blocks a CU otherwise)
    int dev = 0, cus = 0;
    TC_HIP(hipGetDevice(&dev));
    TC_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int64_t grid = std::min<int64_t>(ceil_div(nv, kCoreThreads),
                                           std::max<int64_t>(3 * cus, ceil_div(nv, 1 << 15)));
    hipLaunchKernelGGL(k_core_count<CH>, dim3((unsigned)grid), dim3(kCoreThreads), 0, s, A);
    hipLaunchKernelGGL(k_core_check, dim3(grid_for(k, 256)), dim3(256), 0, s, vi, lo, k, pcount, bad);
    TC_HIP(hipGetLastError());
    return TC_OK;
}

}  // namespace tc

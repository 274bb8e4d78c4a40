// tc_rows.hip -- counts of graphs whose rows are all short.
//
// Without hubs (meshes, road networks, uniform random graphs) a rank order
// saves little: building it -- sorts, the oriented rows, the task lists, the
// plan -- took most of such a count.  Here every row is counted by one wave as
// the reference does (src/static_triangle_counting/cct.cu:233-268): the row in
// a small LDS table, its neighbours' rows streamed past it, out[v] written
// once.  One kernel, no atomics but the total's, and no sizes to read back.
#include "tc_plan.hpp"

#include <algorithm>

namespace tc {

namespace {

constexpr int kRowSlots = 512;  // of a wave's table: at most a quarter is used
constexpr int kWavesPerBlock = 4;

struct RowArgs {
    const int64_t *boff;
    const int32_t *len;
    const int32_t *pool;
    int32_t nv;
    uint32_t *out;
    unsigned long long *global;
    int32_t *bad;  // set where an entry has no reverse (check_sym)
    int32_t skip_lower;
    int32_t check_sym;
};

__device__ inline uint32_t row_slot(int32_t w) { return ((uint32_t)w * 0x9E3779B1u) >> 23; }  // of 512

// G lanes stream one neighbour's row, 64 / G rows at a time, two rounds of
// them in flight.  Bound by the latency of row -> neighbour -> its row, which
// 8 waves a SIMD hide.
template <int G>
__global__ __launch_bounds__(kWavesPerBlock * kWave, 8) void k_count_rows(RowArgs A)
{
    constexpr int GN = kWave / G;
    __shared__ int32_t table[kWavesPerBlock][kRowSlots];
    const int lane = threadIdx.x & (kWave - 1), i = lane % G, grp = lane / G;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    int32_t *T = table[wid];
    for (int q = lane; q < kRowSlots; q += kWave) T[q] = -1;
    wave_sync();
    unsigned long long total = 0;
    bool miss = false;
    const int64_t nwaves = (int64_t)gridDim.x * kWavesPerBlock;
    for (int64_t r = (int64_t)blockIdx.x * kWavesPerBlock + wid; r < A.nv; r += nwaves) {
        const int32_t v = (int32_t)r, d = A.len[v];
        const int32_t *row = A.pool + A.boff[v];
        if (d < 2 && !A.check_sym) {
            if (lane == 0) A.out[v] = 0u;
            continue;
        }
        int32_t mine[2] = {-1, -1};
        uint32_t at[2] = {0, 0};
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (h * kWave + lane < d) mine[h] = row[h * kWave + lane];
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (mine[h] >= 0)
                for (at[h] = row_slot(mine[h]); atomicCAS(&T[at[h]], -1, mine[h]) != -1;)
                    at[h] = (at[h] + 1) & (kRowSlots - 1);
        wave_sync();
        uint32_t hits = 0;
        for (int h = 0; h * kWave < d; ++h) {
            // this lane's neighbour: its row, empty where there is nothing to do
            const int32_t u = h ? mine[1] : mine[0];
            const bool in = u >= 0 && u != v;
            const int32_t lu0 = in ? A.len[u] : 0;
            const bool counts = d >= 2 && lu0 >= 2 && (!A.skip_lower || u > v);
            const int32_t lu = counts || A.check_sym ? lu0 : 0;
            const int64_t bu = in ? A.boff[u] : 0;
            const uint64_t cm = __ballot(counts), im = __ballot(in);
            const int cnt = min(kWave, d - h * kWave);
            for (int j0 = 0; j0 < cnt; j0 += 2 * GN) {
                const int32_t *lst[2];
                int32_t n[2];
                bool cj[2], ij[2], found[2] = {false, false};
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const int j = j0 + q * GN + grp, jj = j & (kWave - 1);
                    const int32_t sl = __shfl(lu, jj, kWave);
                    const int64_t sb = ((int64_t)__shfl((int32_t)(bu >> 32), jj, kWave) << 32) |
                                       (uint32_t)__shfl((int32_t)bu, jj, kWave);
                    n[q] = j < cnt ? sl : 0;
                    lst[q] = A.pool + sb;
                    cj[q] = (cm >> jj) & 1;
                    ij[q] = j < cnt && ((im >> jj) & 1);
                }
                for (int32_t k = i; __ballot(k < n[0] || k < n[1]); k += G) {
                    int32_t w[2], x[2];
                    uint32_t s[2];
#pragma unroll
                    for (int q = 0; q < 2; ++q) w[q] = k < n[q] ? lst[q][k] : -2;
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        s[q] = row_slot(w[q]);
                        x[q] = T[s[q]];
                    }
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        while (x[q] != -1 && x[q] != w[q]) {
                            s[q] = (s[q] + 1) & (kRowSlots - 1);
                            x[q] = T[s[q]];
                        }
                        hits += (x[q] == w[q] && cj[q]) ? 1u : 0u;
                        found[q] |= w[q] == v;
                    }
                }
                if (A.check_sym)
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const uint64_t f = (__ballot(found[q]) >> (grp * G)) & (G == 64 ? ~0ull : (1ull << G) - 1);
                        miss |= ij[q] && f == 0;
                    }
            }
        }
        wave_sync();
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (mine[h] >= 0) T[at[h]] = -1;
        wave_sync();
        hits = wave_sum<uint32_t>(hits);
        if (lane == 0) {
            A.out[v] = hits;
            total += hits;
        }
    }
    if (__ballot(miss) && lane == 0) atomicOr(A.bad, 1);
    const unsigned long long part[1] = {total};
    block_add_u64<1>(part, A.global);
}

// per_graph[g] = the sum of its vertices' counts (at most kRowMax^2 each); one
// block per graph.  Vertices outside all boundaries are the first and the last
// graph's, as everywhere.
__global__ __launch_bounds__(256) void k_row_graph_sums(const int64_t *__restrict__ voff, int32_t nv,
                                                        const uint32_t *__restrict__ out,
                                                        unsigned long long *__restrict__ per_graph)
{
    const int64_t v0 = blockIdx.x == 0 ? 0 : max(voff[blockIdx.x], (int64_t)0);
    const int64_t v1 = blockIdx.x + 1 == gridDim.x ? nv : min(voff[blockIdx.x + 1], (int64_t)nv);
    unsigned long long s = 0;
    for (int64_t v = v0 + threadIdx.x; v < v1; v += blockDim.x) s += out[v];
    const unsigned long long part[1] = {s};
    block_add_u64<1>(part, &per_graph[blockIdx.x]);
}

__global__ void k_zero_counters(unsigned long long *acc)
{
    if (threadIdx.x < 32) acc[threadIdx.x] = 0ull;
}

}  // namespace

bool rows_eligible(const Graph &g, const tc_schedule &sched)
{
    // the default rules only: a forced strategy, merge paths or another build
    // of the oriented layout ask for the kernels they name
    if (sched.policy != TC_POLICY_FIXED || sched.ratio_x16 > 0 || sched.mpath_min > 0 ||
        sched.hub_degree > 0 || sched.build != 0)
        return false;
    // (a triangle of two graphs is counted whole in its job's graph)
    if (g.batch_voff && g.batch_cross) return false;
    return g.validated && !g.degree_stale && rows_pay(g.st.nv, g.st.nnz, g.max_degree);
}

int rows_count(Graph &g, uint32_t *out, unsigned long long *acc, int32_t *bad, bool oriented, bool skip_lower,
               hipEvent_t built)
{
    hipStream_t s = g.stream;
    RowArgs A = {};
    A.boff = g.st.boff.as<int64_t>();
    A.len = g.st.len.as<int32_t>();
    A.pool = g.st.pool.as<int32_t>();
    A.nv = g.st.nv;
    A.out = out;
    A.global = acc;
    A.bad = bad;
    A.skip_lower = skip_lower ? 1 : 0;
    A.check_sym = oriented ? 1 : 0;
    hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, s, acc);
    if (built) TC_HIP(hipEventRecord(built, s));
    const dim3 grid(grid_for(g.st.nv, kWavesPerBlock, 2048)), block(kWavesPerBlock * kWave);
    const int64_t mean = g.st.nnz / std::max(g.st.nv, 1);
    if (mean <= 8)
        hipLaunchKernelGGL(k_count_rows<8>, grid, block, 0, s, A);
    else if (mean <= 24)
        hipLaunchKernelGGL(k_count_rows<16>, grid, block, 0, s, A);
    else
        hipLaunchKernelGGL(k_count_rows<32>, grid, block, 0, s, A);
    if (g.batch_per_graph)
        hipLaunchKernelGGL(k_row_graph_sums, dim3((unsigned)g.batch_ngraphs), dim3(256), 0, s, g.batch_voff,
                           g.st.nv, out, g.batch_per_graph);
    TC_HIP(hipGetLastError());
    return TC_OK;
}

}  // namespace tc

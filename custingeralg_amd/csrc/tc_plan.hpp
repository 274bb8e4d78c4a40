// tc_plan.hpp -- rules that kernels and host share, and that are checked
// without a device (tests/cpp/plan_test.hip): how an owner's work is cut into
// jobs beside the host's bounds on them, which the job arrays are sized by, and
// the entries that a bit-row count loads.
#pragma once

#include "tc_internal.hpp"

#include <algorithm>
#include <cmath>

namespace tc {

enum { kDirect = 0, kOriented = 1, kByTasks = 2 };

constexpr int kL0 = 64, kL1 = 512, kL2 = 4096;
#ifndef TC_MID_NW
#define TC_MID_NW 2
#endif
constexpr int kNW0 = 1, kNW1 = TC_MID_NW, kNW2 = 8;
// (the ranks that k_count_long's bitmap holds, its guard word left)
constexpr int32_t kWideMin = 128, kWideTasks = 64, kWideSpan = (kL2 - 1) * 32;
constexpr int64_t kWideNnz = int64_t(3) << 24;
// ids of a bit row in LDS (k_direct_bits): 32 KB, four blocks of 8 waves a CU,
// and 128 KB, one block of 16
constexpr int kBitsIds0 = 1 << 18, kBitsIds1 = 1 << 20;

struct PlanParams {
    int32_t lmax[3];     // owner-list capacity of each bin's kernel
    int32_t nw[3];       // wavefronts per block of each bin's kernel
    int32_t bin_max[2];  // |owner| <= bin_max[0] -> bin 0, <= bin_max[1] -> bin 1, else 2
    // owners from wide_lo up with wide_tasks: above wide_max -> bin 2 as well
    int32_t wide_lo, wide_max, wide_tasks;
    int32_t job_items;   // target estimated items per job (per wavefront)
    int32_t flush_items; // minimum items per owner slot in a job
    int32_t owner_end;   // owners from here up get no jobs (the core's)
    int32_t id_tiles;    // > 0: owners of bin 2 are tiled by id range, into this many
};

__host__ __device__ inline int32_t owner_tiles(int32_t L, int bin, const PlanParams &P)
{
    return bin == 2 && P.id_tiles > 0 ? P.id_tiles : (int32_t)ceil_div(L, P.lmax[bin]);
}

// The cheaper of streaming a task's list (pl) and searching the owner's in it
// (L log pl).
__host__ __device__ inline int32_t est_items(int32_t L, int32_t pl)
{
    const int32_t bits = pl > 0 ? 32 - __builtin_clz((uint32_t)pl) : 0;  // smallest lg with 2^lg > pl
    const int64_t bs = (int64_t)L * (bits > 1 ? bits : 1);
    return (int32_t)(pl < bs ? pl : bs) + 4;
}

__host__ __device__ inline int owner_bin(int32_t v, int32_t L, int32_t tasks, const PlanParams &P)
{
    const bool wide = v >= P.wide_lo && L > P.wide_max && tasks >= P.wide_tasks;
    return L <= P.bin_max[0] ? 0 : (L <= P.bin_max[1] && !wide ? 1 : 2);
}

// Parts that the task list of an owner (L entries, tasks > 0 tasks of work w) is
// cut into, for each tile of its bin.  wmin: the least work of a part.
__host__ __device__ inline int32_t owner_split(int32_t L, int32_t tasks, unsigned long long w, int bin,
                                               int64_t wmin, const PlanParams &P)
{
    const int64_t per_tile = (int64_t)(w / (unsigned long long)owner_tiles(L, bin, P)) + 1;
    // a job amortises building its LDS table and, at its end, the flush of up to
    // one global atomic per owner slot: at least flush_items items per slot
    const int64_t items = (int64_t)P.job_items * P.nw[bin];
    const int64_t flush = (int64_t)P.flush_items * (L < P.lmax[bin] ? L : P.lmax[bin]);
    int64_t grain = items > flush ? items : flush;
    grain = grain > wmin ? grain : wmin;
    int64_t sp = ceil_div(per_tile, grain);
    if (sp > tasks) sp = tasks;
    if (sp < 1) sp = 1;
    return (int32_t)sp;
}

// The least work of a part for a count of total work w: at most 2^20 parts (and
// a few) beyond one per owner and tile.
__host__ __device__ inline int64_t plan_wmin(unsigned long long w) { return (int64_t)(w >> 20); }

// The parameters of a count (mode: kDirect and so on); core_k: the ranks that the
// core counts; batched: of batched graphs.
inline PlanParams plan_params(const tc_schedule &sched, int mode, bool batched, int32_t nv, int64_t nnz,
                              int32_t core_k)
{
    PlanParams P;
    P.lmax[0] = kL0;
    P.lmax[1] = kL1;
    P.lmax[2] = kL2;
    P.nw[0] = kNW0;
    P.nw[1] = kNW1;
    P.nw[2] = kNW2;
    P.bin_max[0] = std::min(std::max(sched.small_max, 1), kL0);
    P.bin_max[1] = std::min(std::max(sched.mid_max, P.bin_max[0]), kL1);
    P.job_items = std::max(sched.job_items, 256);
    P.flush_items = sched.flush_items > 0 ? sched.flush_items : 1024;
    P.owner_end = nv - (mode == kOriented ? core_k : 0);
    // by tasks: bit rows hold any list whole, and a job of theirs ends without a
    // flush.  Beyond kBitsIds1 ids a row is tiled by id range, which pays for
    // the largest bin only (the mid bin's lists go through LDS tables).
    P.id_tiles = 0;
    if (mode == kByTasks) {
        P.id_tiles = (int32_t)ceil_div(nv, kBitsIds1);
        P.lmax[2] = INT32_MAX;
        P.nw[2] = 8;
        P.flush_items = 16;
        if (nv <= kBitsIds1) P.bin_max[1] = P.bin_max[0];  // (no mid bin)
    }
    // Owners whose rows fit k_count_long's bitmap by their rank (a row of N+ spans
    // at most the ranks above its owner) go to the largest bin from kWideMin
    // entries on: it streams 1300 G entries a second against the mid bin's 440,
    // whose bitmap holds an eighth of the ranks, and hash tables beyond (3M ragged
    // vertices 12.2 -> 10.3 ms; 96, 192, 256, 384 entries: 10.3, 10.3, 10.6, 10.7).
    // Its jobs of eight waves need a large graph to fill the chip: R-MAT graphs of
    // 8M to 48M entries took 1.01 to 1.12 times as long, of 63M and more 0.84 to
    // 0.96.  Without enough tasks the bitmap is not repaid; the largest bin's hash
    // tables are no gain either (R-MAT 24 with all rows from 256 on 131 -> 149 ms),
    // nor are batched graphs, whose cores lie behind all other ranks.
    // (after the last change of bin_max: plan_caps takes rows above wide_max for
    // bin 2's)
    P.wide_lo = INT32_MAX;
    P.wide_max = P.bin_max[1];
    P.wide_tasks = kWideTasks;
    if (mode == kOriented && !batched && nnz >= kWideNnz && P.bin_max[1] > kWideMin &&
        (sched.policy == TC_POLICY_HASH || sched.policy == TC_POLICY_LEARNED ||
         (sched.policy == TC_POLICY_FIXED && sched.ratio_x16 <= 0 && sched.mpath_min <= 0))) {
        P.wide_lo = std::max(nv - kWideSpan, 0);
        P.wide_max = kWideMin;
    }
    return P;
}

// A bound on the longest owner list of a count (max_degree: the longest row, or a
// bound on it).  In the order by degree an entry of N+ points to a row no shorter
// than its own, so that |N+| <= sqrt(nnz); in that by graph and degree too, unless
// entries leave their graph.
inline int64_t longest_list(bool by_degree, int32_t nv, int64_t nnz, int64_t max_degree)
{
    const int64_t most = std::min<int64_t>(nv, max_degree);
    return by_degree ? std::min<int64_t>(most, (int64_t)std::sqrt((double)nnz) + 1) : most;
}

inline int64_t longest_list(const Graph &g, bool oriented)
{
    const int32_t nv = g.st.nv;
    return longest_list(oriented && !g.batch_cross, nv, g.st.nnz,
                        g.validated && !g.degree_stale ? g.max_degree : nv);
}

// The most jobs that the owners of each bin can have: one per owner and tile, and
// what the work gives beyond that, at most 2^21 (owner_split, plan_wmin).  lists:
// entries of all owners' lists, and a bound on their tasks; lmost: a bound on the
// longest list.
inline void plan_caps(const PlanParams &P, int32_t nv, int64_t lists, int64_t lmost, int64_t cap[3])
{
    const int64_t least[3] = {0, P.bin_max[0], std::min(P.bin_max[1], P.wide_max)};  // a bin's lists are longer
    for (int b = 0; b < 3; ++b) {
        const int64_t owners = std::min<int64_t>(nv, lists / (least[b] + 1));
        const bool any = b == 0 || lmost > least[b];
        const double more = (double)lists * (double)(lmost + 4) / ((double)P.job_items * P.nw[b]);
        cap[b] = any ? owners + 64 + (int64_t)std::min(more, 2097152.0) : 0;
        if (b == 2 && any) cap[b] += P.id_tiles > 0 ? owners * P.id_tiles : 2 * (lists / P.lmax[2]);
    }
}

// Whether a graph's rows are counted one by one (tc_rows.hip): none longer than
// kRowMax, and a mean of kRowMean at most, above which the oriented count wins.  Nor
// where hubs (a longest row of 16 times the mean, as for the core) have many rows to
// be streamed past: the oriented count streams each pair's shorter list and starts
// to win near a longest row times the vertices of 2^28.  8M vertices in R-MAT
// communities of 1000 and edge factor 1 4.2 ms row by row, 2.7 oriented; 2M 1.05 and
// 1.03, 1M 0.54 and 0.79; of 300 and edge factor 3 at 8M 4.9 and 4.2, at 3M 1.80 and
// 1.87; 4M of 60 and edge factor 6 (no such hubs) 2.3 and 3.3.
constexpr int32_t kRowMax = 128, kRowMean = 40;
inline bool rows_pay(int32_t nv, int64_t nnz, int32_t longest)
{
    if (longest > kRowMax || nnz > (int64_t)kRowMean * nv) return false;
    const double reach = (double)longest * nv;
    return reach < 16.0 * (double)nnz || reach <= 268435456.0;
}

// Whether a batch of graphs is counted on bit rows: mat bytes of them are written
// and, a row per entry, read bytes read.  1.4 us per MiB written, 60 per GB read and
// 300 per million vertices against the task lists' 700 and 40 per million entries:
// fitted to 845 batches (300 to 16384 vertices a graph, edge factors 1 to 32, up to
// 1 GB of bit rows and 8M vertices); none of them takes 1.3 times the other route's
// time.  By size alone 31 R-MAT graphs of 16384 vertices and edge factor 32 took 8.0
// ms on bit rows, 2.2 on lists; with edge factor 4 2.0 and 0.86 (two graphs: 0.17
// and 0.53); 8192 graphs of 1000 vertices and edge factor 2 5.5 and 4.0.
inline bool dense_batch_pays(int64_t mat, int64_t read, int64_t nv, int64_t nnz)
{
    return 1.4 * (double)mat / 1048576 + 60e-9 * (double)read + 300e-6 * (double)nv <= 700 + 40e-6 * (double)nnz;
}

// Bit rows (tc_dense.hip): whether a row of d entries is walked.  A row of one
// entry counts nothing (the reference skips it) but is looked at for its
// reverse; an empty one has no entry to load.
__host__ __device__ inline bool dense_walked(int32_t d, int32_t check_sym)
{
    return d >= 2 || (check_sym && d == 1);
}

// The place that entry e of the part that ends at e1 is loaded from: past the end
// the last entry again.
__host__ __device__ inline int32_t dense_entry(int32_t e, int32_t e1) { return e < e1 ? e : e1 - 1; }

}  // namespace tc

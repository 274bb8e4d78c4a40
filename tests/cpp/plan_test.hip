// Rules that kernels and host share, on the host.  Loaded by tests/test_plan.py;
// nothing here touches a device.
#include "../../custingeralg_amd/csrc/tc_plan.hpp"

#include <numeric>
#include <vector>

using namespace tc;

// The planner's rule applied to a CSR, owner by owner as the kernels apply it,
// beside the capacities that the job arrays get.
// mode: kDirect, kOriented or kByTasks.  Rows sorted, distinct; oriented ones
// symmetric and loop-free.  jobs[b], caps[b]: jobs of bin b, and room for them.
extern "C" int plan_probe(int32_t mode, const tc_schedule *sched, int32_t nv, const int64_t *off,
                          const int32_t *adj, int32_t skip_lower, int64_t jobs[3], int64_t caps[3])
{
    const int64_t nnz = off[nv];
    std::vector<int32_t> len(nv), L(nv), rank(nv), order(nv);
    int32_t longest = 0;
    for (int32_t v = 0; v < nv; ++v) {
        len[v] = (int32_t)(off[v + 1] - off[v]);
        longest = std::max(longest, len[v]);
    }
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) { return len[a] < len[b]; });
    for (int32_t r = 0; r < nv; ++r) rank[order[r]] = r;
    // the owners' tasks: the list lengths that the planner estimates
    std::vector<std::vector<int32_t>> tasks(nv);
    for (int32_t v = 0; v < nv; ++v) {
        L[v] = len[v];
        if (mode == kOriented) {
            std::vector<int32_t> plus;
            for (int64_t e = off[v]; e < off[v + 1]; ++e)
                if (rank[adj[e]] > rank[v]) plus.push_back(adj[e]);
            std::sort(plus.begin(), plus.end(), [&](int32_t a, int32_t b) { return rank[a] < rank[b]; });
            L[v] = (int32_t)plus.size();
            for (size_t i = 0; i < plus.size(); ++i) tasks[plus[i]].push_back((int32_t)(plus.size() - 1 - i));
            continue;
        }
        for (int64_t e = off[v]; e < off[v + 1]; ++e) {
            const int32_t u = adj[e];
            const bool ok = u != v && len[v] >= 2 && len[u] >= 2;
            if (mode == kDirect)
                tasks[v].push_back(ok ? len[u] : -1);  // (-1: a task without work)
            else if (ok && (!skip_lower || u > v))
                tasks[len[u] <= len[v] ? v : u].push_back(len[u] <= len[v] ? len[u] : len[v]);
        }
    }
    const PlanParams P = plan_params(*sched, mode, false, nv, nnz, 0);
    const int64_t lists = mode == kOriented ? nnz / 2 : nnz;
    plan_caps(P, nv, lists, longest_list(mode == kOriented, nv, nnz, longest), caps);
    std::vector<unsigned long long> work(nv, 0);
    unsigned long long total = 0;
    for (int32_t v = 0; v < nv; ++v)
        for (int32_t pl : tasks[v])
            if (L[v] > 0 && pl >= 0 && (mode != kOriented || pl > 0)) {
                const uint32_t w = (uint32_t)est_items(std::min(L[v], P.lmax[2]), pl);
                work[v] += w;
                total += w;
            }
    for (int b = 0; b < 3; ++b) jobs[b] = 0;
    for (int32_t r = 0; r < nv; ++r) {
        const int32_t v = mode == kOriented ? order[r] : r, T = (int32_t)tasks[v].size();
        if (L[v] <= 0 || T <= 0 || work[v] == 0 || (mode == kDirect && len[v] < 2)) continue;
        const int b = owner_bin(r, L[v], T, P);
        jobs[b] += (int64_t)owner_split(L[v], T, work[v], b, plan_wmin(total), P) * owner_tiles(L[v], b, P);
    }
    return TC_OK;
}

// The least and the largest place that a bit-row count loads of a row of d entries
// (none: 0, -1), in the order of dense_row: 8 groups, U entries each in flight.
extern "C" void dense_probe(int32_t d, int32_t check_sym, int32_t U, int32_t *lo, int32_t *hi)
{
    *lo = 0;
    *hi = -1;
    if (!dense_walked(d, check_sym)) return;
    auto load = [&](int32_t e) {
        const int32_t k = dense_entry(e, d);
        *lo = std::min(*lo, k);
        *hi = std::max(*hi, k);
    };
    for (int32_t grp = 0; grp < 8; ++grp) {
        for (int32_t q = 0; q < U; ++q) load(grp + q * 8);
        for (int32_t eb = grp; eb - grp < d; eb += 8 * U)
            for (int32_t q = 0; q < U; ++q) load(eb + (U + q) * 8);
    }
}

extern "C" int dense_batch_probe(int64_t mat, int64_t read, int64_t nv, int64_t nnz)
{
    return dense_batch_pays(mat, read, nv, nnz);
}

extern "C" int rows_probe(int32_t nv, int64_t nnz, int32_t longest) { return rows_pay(nv, nnz, longest); }

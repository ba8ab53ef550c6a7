// pict_schedule.hpp -- schedules of batched solves (pict_solve.hip): list scheduling of the systems' jobs, and the time
// estimates of k_cg_block_jobs, which the choice of its rows per thread and the lists that run have to share.
#pragma once

#include <algorithm>
#include <vector>

namespace pict {

// List scheduling of the systems' jobs onto `grid` workgroups (cost: estimated time of each solve); returns the
// makespan.
inline double list_schedule(int count, const std::vector<int> &nwg, unsigned grid, const std::vector<double> &cost,
                std::vector<unsigned> &job_off, std::vector<unsigned> &jobs) {
    std::vector<int> order(count);
    for (int s = 0; s < count; ++s) order[s] = s;
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return cost[x] > cost[y]; });
    std::vector<double> avail(grid, 0.0);
    std::vector<std::vector<unsigned>> lists(grid);
    std::vector<unsigned> idx(grid);
    double makespan = 0.0;
    for (int s : order) {
        const unsigned k = (unsigned)nwg[s];
        for (unsigned g = 0; g < grid; ++g) idx[g] = g;
        auto earlier = [&](unsigned x, unsigned y) { return avail[x] < avail[y] || (avail[x] == avail[y] && x < y); };
        std::nth_element(idx.begin(), idx.begin() + (k - 1), idx.end(), earlier);
        std::sort(idx.begin(), idx.begin() + k);
        double start = 0.0;
        for (unsigned j = 0; j < k; ++j) start = std::max(start, avail[idx[j]]);
        const double fin = start + cost[s];
        for (unsigned j = 0; j < k; ++j) {
            lists[idx[j]].push_back(((unsigned)s << 16) | j);
            avail[idx[j]] = fin;
        }
        makespan = std::max(makespan, fin);
    }
    job_off.assign(grid + 1, 0);
    jobs.clear();
    for (unsigned g = 0; g < grid; ++g) {
        job_off[g] = (unsigned)jobs.size();
        jobs.insert(jobs.end(), lists[g].begin(), lists[g].end());
    }
    job_off[grid] = (unsigned)jobs.size();
    return makespan;
}
// us per iteration of a system in k_cg_block_jobs (256 x 256 on 32 workgroups and more; one workgroup (rpt 0): by rows)
inline double block_job_us(int n, int rpt) {
    return rpt == 0 ? 0.6 + 0.7 * n / 2048 : rpt <= 2 ? 1.8 : rpt == 4 ? 2.1 : 2.9;
}
// estimated times of solves from their iterations.  (Lists by iterations alone take a 0.6 and a 2.9 us iteration for the
// same: not the schedule that the rows per thread were chosen for.)
inline std::vector<double> block_job_costs(const std::vector<int> &n, const std::vector<int> &rpt,
                                           const std::vector<double> &iterations) {
    std::vector<double> us(iterations);
    for (size_t s = 0; s < us.size(); ++s) us[s] *= block_job_us(n[s], rpt[s]);
    return us;
}

}  // namespace pict

// cns_runs.h -- z runs of the z-marching kernels (internal; host code without HIP).
#pragma once

#include <cstdint>

namespace cns {

// Calls f(kz) for the lengths that n planes have when cut into 1, 2, .. n even runs, at most
// `most` planes long, longest first and each once: about 2 sqrt(n) of them.  (Trying every number of
// runs cost a launch 8 ns a plane: for 400000 planes 3.1 ms, where hypterm's kernel takes 2.05.)
template <typename F>
inline void each_run_length(int n, int most, F f)
{
    for (int kz = most < n ? most : n, nz = (n + kz - 1) / kz;; nz = (n + kz - 2) / (kz - 1)) {
        kz = (n + nz - 1) / nz;
        f(kz);
        if (kz == 1) return;
    }
}

// The run length whose rounds of workgroups end first: a launch takes ceil(workgroups / slots)
// rounds of kz + fill plane times.
inline int stage_run(int n, int64_t tiles, int slots, double fill)
{
    int best = n;
    double cost = 1e300;
    each_run_length(n, n, [&](int kz) {
        const int64_t rounds = (tiles * ((n + kz - 1) / kz) + slots - 1) / slots;
        const double c = (double)rounds * (kz + fill);
        if (c < cost) {
            cost = c;
            best = kz;
        }
    });
    return best;
}

// The same, at most `most` planes, and of runs within 1 % of the best before them the shortest.
inline int pipe_run(int n, int most, int64_t tiles, int slots, int fill)
{
    int best = most;
    int64_t cost = INT64_MAX / 2;
    each_run_length(n, most, [&](int kz) {
        const int64_t c = (tiles * ((n + kz - 1) / kz) + slots - 1) / slots * (kz + fill);
        if (c > cost + cost / 100) return;
        best = kz;
        if (c < cost) cost = c;
    });
    return best;
}

}  // namespace cns

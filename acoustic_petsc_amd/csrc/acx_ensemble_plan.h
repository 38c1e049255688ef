// acx_ensemble_plan.h -- work items of an ensemble and their schedule over the
// workgroups of a persistent kernel (plain C++, no device).
//
// Work items are (problem, column tile, z-chunk) triples.  Each XCD gets a
// contiguous run of the items with an eighth of the work, so that neighbouring
// tiles meet in its L2, and each workgroup of the XCD a list of them, the
// longest items handed out first and each to the workgroup with the least so
// far.
#pragma once
#include <stddef.h>
#include <algorithm>
#include <functional>
#include <queue>
#include <utility>
#include <vector>
#include "acx_plan.h"

namespace acx {

struct EnsProblem {
    size_t off;          // first cell
    int n[3];
    int ntx, nty, ntz;
    int zc;              // planes per work item
};

struct EnsItem {
    int prob;            // index into the problem table
    int tile;            // column tile and z-chunk, x fastest, then y, then z
};

constexpr int ENS_BX = 64;   // columns of a tile along x

struct EnsConfig { int by, zc; };   // rows of a tile, most planes per work item

// The problems of a configuration (dims: n of each problem, off: its first
// cell): each one's planes divided evenly into chunks of at most c.zc.
inline std::vector<EnsProblem> ens_problems(const std::vector<int> &dims, const std::vector<size_t> &off,
                                            const EnsConfig &c)
{
    std::vector<EnsProblem> probs(off.size());
    for (size_t p = 0; p < off.size(); ++p) {
        EnsProblem &q = probs[p];
        for (int d = 0; d < 3; ++d) q.n[d] = dims[3 * p + d];
        q.off = off[p];
        q.ntx = (q.n[0] + ENS_BX - 1) / ENS_BX;
        q.nty = (q.n[1] + c.by - 1) / c.by;
        q.ntz = (q.n[2] + c.zc - 1) / c.zc;
        q.zc = (q.n[2] + q.ntz - 1) / q.ntz;
    }
    return probs;
}

// Whether a problem's planes are beyond the 32-bit offsets of the all-periodic
// march (16 bytes a cell); the whole ensemble then takes the general one.
inline bool ens_wide(const std::vector<int> &dims)
{
    for (size_t p = 0; p + 2 < dims.size(); p += 3)
        if (plane_beyond_32_bits(dims[p], dims[p + 1], 16)) return true;
    return false;
}

// Lists of the items per workgroup: workgroup b runs items[first[b]] ..
// items[first[b + 1] - 1], so the launch has blocks() workgroups, neither fewer
// (items would not run) nor more (there is no list for them).
struct EnsSchedule {
    std::vector<EnsItem> items;
    std::vector<int> first;
    double most = 0.0;   // work of the busiest workgroup, zc + 10 planes per item
    int blocks() const { return (int)first.size() - 1; }
};

// Workgroups b, b + 8, ... run on XCD b % 8.
inline EnsSchedule ens_schedule(const std::vector<EnsProblem> &probs, int blocks)
{
    EnsSchedule r;
    std::vector<EnsItem> all;
    double work = 0.0;
    for (int p = 0; p < (int)probs.size(); ++p) {
        const int n = probs[p].ntx * probs[p].nty * probs[p].ntz;
        for (int t = 0; t < n; ++t) all.push_back({p, t});
        work += (double)n * (probs[p].zc + 10);
    }
    const int xcds = std::min(kNumXcd, blocks);   // those with a workgroup
    std::vector<std::vector<EnsItem>> list(blocks);
    size_t k = 0;
    double done = 0.0;
    for (int x = 0; x < xcds; ++x) {
        // this XCD's share of the items, longest first
        std::vector<EnsItem> part;
        const double upto = work * (x + 1) / xcds;
        for (; k < all.size() && (x == xcds - 1 || done + 0.5 * (probs[all[k].prob].zc + 10) < upto); ++k) {
            part.push_back(all[k]);
            done += probs[all[k].prob].zc + 10;
        }
        std::stable_sort(part.begin(), part.end(),
                         [&](const EnsItem &a, const EnsItem &b) { return probs[a.prob].zc > probs[b.prob].zc; });
        using Load = std::pair<double, int>;   // (work so far, workgroup)
        std::priority_queue<Load, std::vector<Load>, std::greater<Load>> least;
        for (int b = x; b < blocks; b += kNumXcd) least.push({0.0, b});
        for (const EnsItem &i : part) {
            Load l = least.top();
            least.pop();
            list[l.second].push_back(i);
            l.first += probs[i.prob].zc + 10;
            r.most = std::max(r.most, l.first);
            least.push(l);
        }
    }
    r.first.assign(1, 0);
    for (const auto &l : list) {
        r.items.insert(r.items.end(), l.begin(), l.end());
        r.first.push_back((int)r.items.size());
    }
    return r;
}

// A configuration's problems and its two schedules: stages 1-3 and the last
// stage.  fit: workgroups of the kernels of either (the middle stages' and the
// last one's) that fit the device at once.  The first stage's kernel, which
// needs less, runs the middle ones' schedule on their grid.
struct EnsPlan {
    std::vector<EnsProblem> probs;
    EnsSchedule schedule[2];
};

constexpr int ens_schedule_of(int stage) { return stage == F32_LAST ? 1 : 0; }

inline EnsPlan ens_plan(std::vector<EnsProblem> probs, const int (&fit)[2])
{
    EnsPlan r;
    for (int k = 0; k < 2; ++k) r.schedule[k] = ens_schedule(probs, fit[k]);
    r.probs = std::move(probs);
    return r;
}

} // namespace acx

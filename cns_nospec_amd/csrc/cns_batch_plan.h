// cns_batch_plan.h -- the work list of the batched engine's one-kernel stage (internal; host code
// without HIP).
//
// A CU holds one workgroup of the stage kernel, which takes about planes + 1.5 plane times, and XCD x
// runs the x-th eighth of the list in order on its 32 CUs.  So the list is made of eight equally
// long parts (dummy tiles fill them up): the z runs of all boxes, longest first, each go whole
// (its tiles share halos) to the part with the least work.  Long runs fill their windows less
// often, short ones end together: the boxes are split in one of a few ways, the one whose
// slowest part is predicted to end first.
//   Predicted / measured with 16-row tiles alone, 64 boxes of edges 16..96 (the work alone: 125
// plane times of every CU): runs of 16 planes 140 / 2.86 ms a step (FP64), of 32 151 / 3.17, this
// list 134 / 2.80; 40 boxes of 24..128 (233): runs of 16 in the boxes' order 5.12 ms (FP32 flux), of
// 32 longest first 260 / 4.86, this list 248 / 4.64.
#pragma once

#include <algorithm>
#include <climits>
#include <cstddef>
#include <cstdint>
#include <initializer_list>
#include <utility>
#include <vector>

namespace cns {

struct TileDev {
    int box;
    short x0, y0, z0, nz;  // tile origin (cells) and z run
    short ltx;             // log2 of the tile width (4, 5 or 6)
    short rows;            // of a tile of the fused kernel
};

constexpr int kShortRows = 16, kTallRows = 24;  // tiles of the fused kernel (tall: FP32 flux only)
constexpr int kXcds = 8, kCusPerXcd = 32;
constexpr int kTallCost = 4, kShortCost = 3;  // of a plane
// Tiles, counted at runs of 12 planes, up to which the splits are compared; a longer list takes the first of
// them: its tail is short however it is split, and the comparison would cost the host more than that.
constexpr size_t kMostSimulated = 1 << 14;
// Tiles of a list at most: a launch has fewer than 2^32 threads, 768 a tile.
constexpr size_t kMostListed = 1 << 22;

struct Split {
    int run, last, eighths;  // runs of `run` planes, and of `last` for so many eighths:
    bool boxes;              // of the work, the smallest boxes (or the last planes of every box)
};
constexpr Split kSplits[] = {{24, 0, 0, false}, {16, 0, 0, false}, {32, 0, 0, false}, {48, 0, 0, false},
                             {64, 0, 0, false}, {48, 16, 3, true}, {32, 16, 2, true}, {24, 16, 2, true},
                             {40, 8, 2, true},  {64, 12, 1, false}, {48, 8, 1, false}, {24, 8, 4, false},
                             {8, 0, 0, false},  {4, 0, 0, false},  {2, 0, 0, false}};
// The last three are for boxes that leave most CUs idle (1 / 4 / 8 boxes of 48^3, FP32 flux, 89 / 138 / 213
// us a step, in runs of 16 planes 357 / 362 / 365).  The shorter the runs, the more of the prediction rests on the
// window fill, which for tall tiles is nearer 2.5 planes: they have to be an eighth better than the rest.
constexpr int kShortRun = 16;

// Small boxes.  A 32 x 16 tile of the one-kernel stage takes its time however few of its cells a box
// has; the separate kernels' 16 x 16 tiles of four waves share a CU instead, but are nine launches a
// step.  So boxes of at most small_edge() cells take 16-wide tiles where they are many: more than one a CU,
// or two beside other boxes, whose stage goes on without them.  us a step with one kernel a stage / 16-wide
// tiles, FP32 flux: 256 boxes of 8^3 190 / 170, 320 308 / 190, 1024 675 / 298; of 16^3 256 346 / 338, 320 499 /
// 387, 1024 1308 / 931; beside 30 of 64^3 320 of 16^3 1597 / 1716, 512 1781 / 1783, 1024 2357 / 2159. FP64: 320 boxes
// of 8^3 330 / 263, of 14^3 505 / 483, 1024 740 / 479 and 1309 / 1135; of 16^3 1459 / 1409, 320 562 / 611.
constexpr int small_edge(bool fp32) { return fp32 ? 16 : 14; }
constexpr bool small_apart(size_t small, size_t others)
{
    return small > (others ? 2 : 1) * (size_t)(kXcds * kCusPerXcd);
}

struct FusedBox {
    int id, e, kz;      // kz: longest run allowed
    int nx, tall, low;  // tiles of a plane: nx times so many of kTallRows and of kShortRows rows
    int cost() const { return nx * (kTallCost * tall + kShortCost * low); }
    int tiles() const { return nx * (tall + low); }
};

// A box's rows in the fewest plane times: of FP32 flux a tall tile's plane takes 1.35 times a
// short one's (cns_batch_stage.hip; edges 96 and 64 measured), e.g. 16 rows one short tile, 24 one
// tall, 32 two short, 40 one of each.
inline void tile_rows(FusedBox &b, bool fp32)
{
    int best = INT_MAX;
    for (int tall = 0; tall <= (fp32 ? (b.e + kTallRows - 1) / kTallRows : 0); tall++) {
        const int low = std::max(0, (b.e - tall * kTallRows + kShortRows - 1) / kShortRows);
        const int cost = kTallCost * tall + kShortCost * low;
        if (cost < best) {
            best = cost;
            b.tall = tall;
            b.low = low;
        }
    }
}

// Boxes of one edge and cap, which have the same runs: boxes first .. first + n - 1, largest edge first.
struct BoxGroup {
    int first, n;
};

// The runs of a group's boxes, in z order.
struct GroupRuns {
    BoxGroup boxes;
    std::vector<std::pair<short, short>> runs;  // z0, planes
    bool operator==(const GroupRuns &o) const { return boxes.first == o.boxes.first && boxes.n == o.boxes.n && runs == o.runs; }
};

struct Unit {
    int box, z0, nz;  // index of the FusedBox
};

// The CUs of one XCD as a heap of the times at which they end, earliest on top.
struct CuHeap {
    int64_t end[kCusPerXcd] = {};
    // a tile of time t on the CU that is free first; returns its end
    int64_t add(int64_t t)
    {
        const int64_t e = end[0] + t;
        int i = 0;
        for (int c = 1; c < kCusPerXcd; c = 2 * i + 1) {
            if (c + 1 < kCusPerXcd && end[c + 1] < end[c]) c++;
            if (end[c] >= e) break;
            end[i] = end[c];
            i = c;
        }
        end[i] = e;
        return e;
    }
};

struct FusedPlan {
    std::vector<Unit> part[kXcds];
    int64_t end = INT64_MAX;  // of the slowest part, in sixths of a short tile's plane time
    size_t tiles = 0;
};

// The runs of all boxes under a split: planes z0 .. z1-1 of a box in even runs of about `run`, at
// most the box's kz.
inline std::vector<GroupRuns> split_runs(const std::vector<FusedBox> &boxes, const std::vector<BoxGroup> &groups,
                                         int64_t all, const Split &sp)
{
    std::vector<GroupRuns> out;
    auto add = [&](int first, int n, std::initializer_list<std::pair<int, int>> parts) {  // (end, run) of each part
        if (n <= 0) return;
        GroupRuns g{{first, n}, {}};
        int z0 = 0;
        for (const auto &[z1, run] : parts) {
            const int len = z1 - z0;
            if (len <= 0) continue;
            const int k = std::max({1, (len + run / 2) / run, (len + boxes[first].kz - 1) / boxes[first].kz});
            const int nz = (len + k - 1) / k;
            for (; z0 < z1; z0 += nz) g.runs.push_back({(short)z0, (short)std::min(nz, z1 - z0)});
            z0 = z1;
        }
        out.push_back(std::move(g));
    };
    int64_t done = 0;
    for (const BoxGroup &g : groups) {
        const int e = boxes[g.first].e;
        const int64_t work = (int64_t)boxes[g.first].cost() * e;
        if (sp.boxes) {
            // the boxes that begin before the last `eighths` of the work
            const int64_t left = (8 - sp.eighths) * all - 8 * done;
            const int n = left <= 0 ? 0 : (int)std::min<int64_t>(g.n, (left + 8 * work - 1) / (8 * work));
            add(g.first, n, {{e, sp.run}});
            add(g.first + n, g.n - n, {{e, sp.last}});
            done += g.n * work;
        } else {
            add(g.first, g.n, {{e - e * sp.eighths / 8, sp.run}, {e, sp.last}});
        }
    }
    return out;
}

// Lays the runs out in the eight parts; returns false, with the plan unfinished, as soon as it cannot end
// before `before`.
inline bool plan_runs(const std::vector<FusedBox> &boxes, const std::vector<GroupRuns> &runs, int64_t before,
                      bool simulate, FusedPlan &p)
{
    int64_t work = 0;
    std::vector<std::pair<int, int>> order;  // (planes, group)
    for (int g = 0; g < (int)runs.size(); g++) {
        const FusedBox &b = boxes[runs[g].boxes.first];
        for (const auto &r : runs[g].runs) {
            work += (int64_t)runs[g].boxes.n * b.cost() * (2 * r.second + 3);
            if (order.empty() || order.back() != std::make_pair((int)r.second, g)) order.push_back({r.second, g});
        }
    }
    if (simulate && work / (kXcds * kCusPerXcd) >= before) return false;
    // longest first, then in the boxes' order and up a box
    std::sort(order.begin(), order.end(), [](const auto &a, const auto &b) {
        return a.first != b.first ? a.first > b.first : a.second < b.second;
    });
    order.erase(std::unique(order.begin(), order.end()), order.end());
    int64_t load[kXcds] = {};
    for (const auto &[nz, g] : order)
        for (int b = runs[g].boxes.first, end = b + runs[g].boxes.n; b < end; b++)
            for (const auto &r : runs[g].runs)
                if (r.second == nz) {
                    const int x = (int)(std::min_element(load, load + kXcds) - load);
                    load[x] += (int64_t)boxes[b].cost() * (2 * nz + 3);
                    p.part[x].push_back({b, r.first, nz});
                    p.tiles += (size_t)boxes[b].tiles();
                }
    p.end = 0;
    for (int x = 0; simulate && x < kXcds; x++) {
        CuHeap cu;
        for (const Unit &u : p.part[x]) {
            const FusedBox &b = boxes[u.box];
            int64_t end = 0;
            for (int t = 0; t < b.nx * b.tall; t++) end = std::max(end, cu.add(kTallCost * (2 * u.nz + 3)));
            for (int t = 0; t < b.nx * b.low; t++) end = std::max(end, cu.add(kShortCost * (2 * u.nz + 3)));
            p.end = std::max(p.end, end);
            if (p.end >= before) return false;
        }
    }
    return true;
}

// Appends the list; returns the number of its real tiles.  Boxes of one edge are split alike and a
// split that cannot end first is dropped as early as that shows, since the list is made anew whenever a
// box comes or goes.
inline size_t fused_list(std::vector<FusedBox> &boxes, std::vector<TileDev> &out)
{
    std::stable_sort(boxes.begin(), boxes.end(), [](const FusedBox &a, const FusedBox &b) { return a.e > b.e; });
    size_t capped = 0;  // tiles that the caps of the runs alone ask for
    for (const FusedBox &b : boxes) capped += (size_t)b.tiles() * ((b.e + b.kz - 1) / b.kz);
    if (capped > kMostListed)
        for (FusedBox &b : boxes) b.kz = b.e;
    std::vector<BoxGroup> groups;
    size_t most = 0;
    int64_t all = 0;
    for (int i = 0; i < (int)boxes.size(); i++) {
        const FusedBox &b = boxes[i];
        most += (size_t)b.tiles() * ((b.e + 11) / 12);
        all += (int64_t)b.cost() * b.e;
        if (i && boxes[i - 1].e == b.e && boxes[i - 1].kz == b.kz)
            groups.back().n++;
        else
            groups.push_back({i, 1});
    }
    const bool simulate = most <= kMostSimulated;
    FusedPlan best;
    std::vector<std::vector<GroupRuns>> tried;
    for (const Split &sp : kSplits) {
        std::vector<GroupRuns> runs = split_runs(boxes, groups, all, sp);
        if (std::find(tried.begin(), tried.end(), runs) != tried.end()) continue;
        FusedPlan p;
        if (plan_runs(boxes, runs, sp.run < kShortRun ? best.end - best.end / 8 : best.end, simulate, p)) best = std::move(p);
        if (!simulate) break;
        tried.push_back(std::move(runs));
    }
    std::vector<TileDev> part[kXcds];
    most = 0;
    for (int x = 0; x < kXcds; x++) {
        for (const Unit &u : best.part[x]) {
            const FusedBox &b = boxes[u.box];
            for (int y0 = 0, r = 0; r < b.tall + b.low; r++) {
                const short rows = r < b.tall ? kTallRows : kShortRows;
                for (int x0 = 0; x0 < b.e; x0 += 32)
                    part[x].push_back({b.id, (short)x0, (short)y0, (short)u.z0, (short)u.nz, 5, rows});
                y0 += rows;
            }
        }
        most = std::max(most, part[x].size());
    }
    for (int x = 0; x < kXcds; x++) {
        part[x].resize(most, {boxes[0].id, 0, 0, 0, 0, 5, 0});  // no planes: ends at once
        out.insert(out.end(), part[x].begin(), part[x].end());
    }
    return best.tiles;
}

}  // namespace cns

"""The choices that the library makes on the host before a launch (cns_runs.h), compiled here
with the host compiler and compared with the plain search that they stand for."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "cns_nospec_amd", "csrc")


def compiled(tmp_path_factory, name, source, compiler=("g++", "-Wall", "-Werror")):
    folder = tmp_path_factory.mktemp(name)
    src, exe = folder / f"{name}.cpp", folder / name
    src.write_text(source)
    subprocess.run([*compiler, "-std=c++17", "-O2", f"-I{CSRC}", "-o", str(exe), str(src)], check=True)

    def run(*args):
        return subprocess.run([str(exe), *map(str, args)], check=True, capture_output=True, text=True).stdout

    return run


RUNS = r"""
#include <cmath>
#include <cstdio>
#include <initializer_list>
#include "cns_runs.h"
using namespace cns;

// every number of runs, from 1 (stage) or the fewest that the cap allows (pipe) to one a plane
static int plain_stage(int n, int64_t tiles, int slots, double fill)
{
    int best = n;
    double cost = 1e300;
    for (int nz = 1; nz <= n; nz++) {
        const int kz = (n + nz - 1) / nz, runs = (n + kz - 1) / kz;
        const double c = (double)((tiles * runs + slots - 1) / slots) * (kz + fill);
        if (c < cost) {
            cost = c;
            best = kz;
        }
    }
    return best;
}
static int plain_pipe(int n, int most, int64_t tiles, int slots, int fill)
{
    int best = most;
    int64_t cost = INT64_MAX / 2;
    for (int nz = (n + most - 1) / most; nz <= n; nz++) {
        const int kz = (n + nz - 1) / nz, runs = (n + kz - 1) / kz;
        const int64_t c = (tiles * runs + slots - 1) / slots * (kz + fill);
        if (c > cost + cost / 100) continue;
        best = kz;
        if (c < cost) cost = c;
    }
    return best;
}

int main()
{
    long bad = 0;
    for (int n = 1; n <= 700; n++) {
        for (int64_t tiles : {1, 2, 7, 35, 256, 1024, 16384}) {
            bad += stage_run(n, tiles, 256, 1.6) != plain_stage(n, tiles, 256, 1.6);
            for (int most : {4, 61, n})
                if (most <= n)
                    for (int fill : {1, 3}) bad += pipe_run(n, most, tiles, 512, fill) != plain_pipe(n, most, tiles, 512, fill);
        }
    }
    // tall boxes: a choice looks at about 2 sqrt(n) lengths, not at n of them
    for (int n : {1, 2, 1023, 400000, 33554432}) {
        long seen = 0;
        int last = n + 1;
        each_run_length(n, n, [&](int kz) {
            bad += kz >= last;
            last = kz;
            seen++;
        });
        bad += last != 1 || seen > 2 * std::sqrt((double)n) + 2;
    }
    printf("%ld\n", bad);
}
"""


@pytest.fixture(scope="module")
def runs(tmp_path_factory):
    return compiled(tmp_path_factory, "runs", RUNS)


def test_run_lengths_are_those_of_the_plain_search(runs):
    assert int(runs()) == 0


# The work list of the batched engine's one-kernel stage (cns_batch_plan.h): "check" compares it with
# the plain search (every split laid out in full and simulated tile by tile) on random sets of boxes, and
# covers every cell of every box with its tiles; "time" compares the two searches' times.
LIST = r"""
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <queue>
#include <random>
#include "cns_batch_plan.h"
using namespace cns;

struct Plain {
    std::vector<Unit> part[kXcds];
    int64_t end = 0;
};

static Plain plain_plan(const std::vector<FusedBox> &boxes, const Split &sp)
{
    Plain p;
    std::vector<Unit> units;
    int64_t all = 0, done = 0, load[kXcds] = {};
    for (const FusedBox &b : boxes) all += (int64_t)b.cost() * b.e;
    auto runs = [&](int b, int z0, int z1, int run) {
        const int len = z1 - z0;
        if (len <= 0) return;
        const int n = std::max({1, (len + run / 2) / run, (len + boxes[b].kz - 1) / boxes[b].kz});
        const int nz = (len + n - 1) / n;
        for (int z = z0; z < z1; z += nz) units.push_back({b, z, std::min(nz, z1 - z)});
    };
    for (int b = 0; b < (int)boxes.size(); b++) {
        const int e = boxes[b].e, first = e - e * sp.eighths / 8;
        if (sp.boxes) {
            runs(b, 0, e, 8 * done < (8 - sp.eighths) * all ? sp.run : sp.last);
            done += (int64_t)boxes[b].cost() * e;
        } else {
            runs(b, 0, first, sp.run);
            runs(b, first, e, sp.last);
        }
    }
    std::stable_sort(units.begin(), units.end(), [](const Unit &a, const Unit &b) { return a.nz > b.nz; });
    for (const Unit &u : units) {
        const int x = (int)(std::min_element(load, load + kXcds) - load);
        load[x] += (int64_t)boxes[u.box].cost() * (2 * u.nz + 3);
        p.part[x].push_back(u);
    }
    for (int x = 0; x < kXcds; x++) {
        std::priority_queue<int64_t, std::vector<int64_t>, std::greater<int64_t>> cu;
        for (int i = 0; i < kCusPerXcd; i++) cu.push(0);
        for (const Unit &u : p.part[x])
            for (int t = 0; t < boxes[u.box].tiles(); t++) {
                const int c = t < boxes[u.box].nx * boxes[u.box].tall ? kTallCost : kShortCost;
                const int64_t end = cu.top() + c * (2 * u.nz + 3);
                cu.pop();
                cu.push(end);
                p.end = std::max(p.end, end);
            }
    }
    return p;
}

static std::vector<TileDev> plain_list(std::vector<FusedBox> boxes)
{
    std::stable_sort(boxes.begin(), boxes.end(), [](const FusedBox &a, const FusedBox &b) { return a.e > b.e; });
    size_t most = 0;
    for (const FusedBox &b : boxes) most += (size_t)b.tiles() * ((b.e + 11) / 12);
    Plain best;
    for (const Split &sp : kSplits) {
        Plain p = plain_plan(boxes, sp);
        if (&sp == kSplits || p.end < (sp.run < kShortRun ? best.end - best.end / 8 : best.end)) best = p;
        if (most > kMostSimulated) break;
    }
    std::vector<TileDev> part[kXcds], out;
    most = 0;
    for (int x = 0; x < kXcds; x++) {
        for (const Unit &u : best.part[x]) {
            const FusedBox &b = boxes[u.box];
            for (int y0 = 0, r = 0; r < b.tall + b.low; r++) {
                const short rows = r < b.tall ? kTallRows : kShortRows;
                for (int x0 = 0; x0 < b.e; x0 += 32) part[x].push_back({b.id, (short)x0, (short)y0, (short)u.z0, (short)u.nz, 5, rows});
                y0 += rows;
            }
        }
        most = std::max(most, part[x].size());
    }
    for (int x = 0; x < kXcds; x++) {
        part[x].resize(most, {boxes[0].id, 0, 0, 0, 0, 5, 0});
        out.insert(out.end(), part[x].begin(), part[x].end());
    }
    return out;
}

static FusedBox box(int id, int e, int kz, bool fp32)
{
    FusedBox b{id, e, std::min(kz, e), (e + 31) / 32, 0, 0};
    tile_rows(b, fp32);
    return b;
}

// whether the list covers every cell of every box once, in runs of at most its kz
static bool covers(const std::vector<FusedBox> &boxes, const std::vector<TileDev> &list, size_t real, bool fp32)
{
    std::vector<std::vector<int>> n(boxes.size());
    for (size_t i = 0; i < boxes.size(); i++) n[i].assign((size_t)boxes[i].nx * boxes[i].e * boxes[i].e, 0);  // (x tile, y, z)
    for (const TileDev &t : list) {
        if (!t.nz) continue;
        real--;
        const FusedBox &b = boxes[t.box];
        if (t.ltx != 5 || t.x0 % 32 || t.x0 >= b.e || t.nz > b.kz || t.z0 + t.nz > b.e ||
            (t.rows != kShortRows && !(fp32 && t.rows == kTallRows)))
            return false;
        for (int z = t.z0; z < t.z0 + t.nz; z++)
            for (int y = t.y0; y < std::min(b.e, t.y0 + t.rows); y++) n[t.box][((size_t)z * b.e + y) * b.nx + t.x0 / 32]++;
    }
    for (const auto &v : n)
        for (int c : v)
            if (c != 1) return false;
    return real == 0 && list.size() % kXcds == 0;
}

static double seconds(const std::function<void()> &f)
{
    double best = 1e9;
    for (int i = 0; i < 5; i++) {
        const auto t = std::chrono::steady_clock::now();
        f();
        best = std::min(best, std::chrono::duration<double>(std::chrono::steady_clock::now() - t).count());
    }
    return best;
}

int main(int, char **argv)
{
    std::mt19937 rng(7);
    auto in = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
    if (!strcmp(argv[1], "time")) {
        std::vector<FusedBox> boxes;
        for (int i = 0; i < 4000; i++) boxes.push_back(box(i, 24, 512, false));
        const double fast = seconds([&] { auto b = boxes; std::vector<TileDev> out; fused_list(b, out); });
        const double plain = seconds([&] { plain_list(boxes); });
        printf("%g\n", fast / plain);
        return 0;
    }
    if (!strcmp(argv[1], "few")) {
        // tiles of n boxes of edge e
        std::vector<FusedBox> boxes;
        for (int i = 0; i < atoi(argv[2]); i++) boxes.push_back(box(i, atoi(argv[3]), 512, argv[4][0] == '1'));
        std::vector<TileDev> out;
        printf("%zu\n", fused_list(boxes, out));
        return 0;
    }
    if (!strcmp(argv[1], "long")) {
        // tiles of n boxes of edge e in runs of one plane
        std::vector<FusedBox> boxes;
        for (int i = 0; i < atoi(argv[2]); i++) boxes.push_back(box(i, atoi(argv[3]), 1, true));
        std::vector<TileDev> out;
        fused_list(boxes, out);
        printf("%zu\n", out.size());
        return 0;
    }
    if (!strcmp(argv[1], "small")) {
        printf("%d %d %d\n", small_edge(false), small_edge(true), small_apart(atoi(argv[2]), atoi(argv[3])));
        return 0;
    }
    int bad = 0;
    for (int t = 0; t < 400; t++) {
        const bool fp32 = t & 1, alike = t & 2, capped = t & 4;
        const int n = t < 8 ? 1 : (t % 40 ? in(1, 60) : in(500, 900)), hi = t % 40 ? in(9, 140) : 24;
        std::vector<FusedBox> boxes;
        for (int i = 0; i < n; i++)
            boxes.push_back(box(i, alike ? 8 * in(1, hi / 8) : in(8, hi), capped ? in(1, 40) : 512, fp32));
        const std::vector<TileDev> want = plain_list(boxes);
        std::vector<FusedBox> b = boxes;
        std::vector<TileDev> got;
        const size_t real = fused_list(b, got);
        bad += got.size() != want.size() || memcmp(got.data(), want.data(), got.size() * sizeof(TileDev));
        bad += !covers(boxes, got, real, fp32);
    }
    // past the limit of the simulation, and the largest box
    for (const auto &[n, e] : {std::pair{2500, 64}, std::pair{9, 512}, std::pair{1, 512}}) {
        std::vector<FusedBox> boxes;
        for (int i = 0; i < n; i++) boxes.push_back(box(i, e, 512, true));
        std::vector<FusedBox> b = boxes;
        std::vector<TileDev> got;
        const size_t real = fused_list(b, got);
        bad += !covers(boxes, got, real, true);
    }
    printf("%d\n", bad);
}
"""


@pytest.fixture(scope="module")
def work_list(tmp_path_factory):
    return compiled(tmp_path_factory, "work_list", LIST)


def test_work_list_is_that_of_the_plain_search_and_covers_every_cell(work_list):
    assert int(work_list("check")) == 0


def test_work_list_is_made_in_a_fraction_of_the_plain_search(work_list):
    """The list is made anew whenever a box comes or goes: of 4000 boxes of one edge in about a tenth of
    the time of the plain search (the limit leaves a factor of five for a busy machine)."""
    assert float(work_list("time")) < 0.5


@pytest.mark.parametrize("n,e,fp32", [(1, 48, 1), (1, 32, 0), (4, 48, 1), (1, 64, 1), (2, 64, 0)])
def test_few_boxes_are_split_until_they_use_the_gpu(work_list, n, e, fp32):
    """Few boxes are cut into runs short enough to give many CUs one (runs of 16 planes gave one box
    of 48^3 twelve workgroups and one of 32^3 four)."""
    assert int(work_list("few", n, e, fp32)) >= 32


@pytest.mark.parametrize("n,e,fp32", [(64, 96, 1), (64, 96, 0), (1000, 24, 1), (600, 17, 0), (16, 64, 0)])
def test_boxes_that_fill_the_gpu_keep_long_runs(work_list, n, e, fp32):
    """Runs of fewer than 16 planes (or a whole box) cost more window fills than they save here."""
    rows = -(-e // 24) if fp32 else -(-e // 16)
    assert int(work_list("few", n, e, fp32)) <= n * -(-e // 32) * (rows + 1) * max(1, -(-e // 12))


@pytest.mark.parametrize("small,others,apart", [(0, 0, 0), (256, 0, 0), (257, 0, 1), (257, 1, 0), (512, 9, 0), (513, 9, 1)])
def test_small_boxes_take_narrow_tiles_where_they_are_many(work_list, small, others, apart):
    """More than one small box a CU, or two beside other boxes."""
    assert work_list("small", small, others).split() == ["14", "16", str(apart)]


def test_a_list_of_short_runs_fits_one_launch(work_list):
    """Boxes that fill the GPU's memory with runs capped at one plane: a launch has fewer than 2^32 threads,
    768 of them a tile, so the caps give way; fewer boxes keep them."""
    assert int(work_list("long", 45000, 33)) * 768 < 1 << 32
    assert int(work_list("long", 1000, 33)) >= 1000 * 4 * 33


# The enumeration of the ghost cells (cns_fill.h) in 32 and in 64 bits: every ghost cell of a box once,
# in the same order; and the last cells of a box with more than 2^32 of them.
SHELL = r"""
#include <cstdio>
#include <vector>
#include "cns_fill.h"
using namespace cns;

int main()
{
    long bad = 0;
    const int sizes[][3] = {{4, 4, 4}, {5, 4, 7}, {16, 16, 16}, {33, 9, 5}, {4, 61, 4}, {70, 4, 21}};
    for (const auto &n : sizes) {
        const Geom g = make_geom(n[0], n[1], n[2]);
        const Shell h = make_shell(g, kOneBox);
        const ShellOf<uint64_t> w = make_shell<uint64_t>(g, kOneBox);
        std::vector<int> seen((size_t)g.g0 * g.g1 * g.g2);
        bad += h.total != w.total || (int64_t)h.total != shell_cells(g);
        for (unsigned e = 0; e < h.total; e++) {
            int i, j, k, a, b, c;
            shell_cell(g, h, e, i, j, k);
            shell_cell(g, w, (uint64_t)e, a, b, c);
            bad += i != a || j != b || k != c || i < 0 || j < 0 || k < 0 || i >= g.g0 || j >= g.g1 || k >= g.g2;
            seen[((size_t)k * g.g1 + j) * g.g0 + i]++;
        }
        for (int k = 0; k < g.g2; k++)
            for (int j = 0; j < g.g1; j++)
                for (int i = 0; i < g.g0; i++) {
                    const bool in = i >= NG && i < g.n0 + NG && j >= NG && j < g.n1 + NG && k >= NG && k < g.n2 + NG;
                    bad += seen[((size_t)k * g.g1 + j) * g.g0 + i] != !in;
                }
    }
    const Geom g = make_geom(1 << 25, 4, 4);
    const ShellOf<uint64_t> w = make_shell<uint64_t>(g, kOneBox);
    int i, j, k;
    shell_cell(g, w, w.elems_a - 1, i, j, k);  // the last full row: the upper y ghosts of the last interior plane
    bad += w.total != (1ull << 32) + 1152 || i != g.g0 - 1 || j != g.g1 - 1 || k != g.n2 + NG - 1;
    shell_cell(g, w, w.total - 1, i, j, k);  // the upper x ghosts of the last interior row
    bad += i != g.g0 - 1 || j != g.n1 + NG - 1 || k != g.n2 + NG - 1;
    printf("%ld\n", bad);
}
"""


def test_ghost_cells_are_enumerated_once_in_32_and_64_bits(tmp_path_factory):
    from cns_nospec_amd import build
    shell = compiled(tmp_path_factory, "shell", SHELL, (build.hipcc(), "-x", "hip", f"--offload-arch={build.ARCH}"))
    assert int(shell()) == 0


@pytest.mark.parametrize("gain", [1.0, 1.02])
def test_autotuner_does_not_time_a_replaced_choice_again(monkeypatch, gain):
    """A bucket takes one trial of every other run length, also when one of them is the faster (gain: of
    every trial of a bucket over the last)."""
    from cns_nospec_amd import batch, serve

    class Engine:
        def __init__(self, *args, **kwargs):
            self.table = {}

        def add(self, u, e):
            self.table[e] = None

        def set_tile(self, e, w, kz):
            self.table[e] = (w, kz)

        def close(self):
            pass

    class Request:
        def __init__(self, edge):
            self.edge = edge

    class State:
        def reshape(self, n):
            return self

    seen = []

    def rate(eng, cells, steps, reps):
        seen.append(tuple(sorted(eng.table.items())))
        return gain ** max(0, len(seen) - 4)

    monkeypatch.setattr(batch, "BatchEngine", Engine)
    monkeypatch.setattr(batch, "_rate", rate)
    monkeypatch.setattr(serve, "request_state", lambda r: State())
    table, log = batch.autotune([Request(16), Request(24)], True, widths=(16, 32), kzs=(8, 16), buckets=((8, 20), (21, 40)))
    assert len(seen) == 2 * 2 + 2 * 1 and len(log) == len(seen) + 1
    assert set(table.values()) == {(16, 16 if gain == 1.0 else 8)}

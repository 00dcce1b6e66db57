"""The choices that the library makes on the host before a launch (cns_runs.h), compiled here
with the host compiler and compared with the plain search that they stand for."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "cns_nospec_amd", "csrc")


def compiled(tmp_path_factory, name, source):
    folder = tmp_path_factory.mktemp(name)
    src, exe = folder / f"{name}.cpp", folder / name
    src.write_text(source)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", f"-I{CSRC}", "-o", str(exe), str(src)], check=True)

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

"""The prefill's (block, run) lookup against the count it replaces, block by
block, over the sizes and cuts the plan can make, and the cuts the plan takes
where they were measured; CPU only."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HARNESS = r"""
#include <cstdio>
#include <initializer_list>
#include "prefill_runs.hpp"
using namespace tq;
int main() {
    long seen = 0, wrong = 0, mixed = 0;
    for (int qb : {16, 32, 64, 128})
        for (int pos0 : {0, 1, 31, 32, 97, 1000, 4095, 8000, 65000})
            for (int n : {1, 15, 16, 17, 32, 33, 100, 127, 128, 129, 333, 2048, 4097, 8176})
                for (int k = 1; k <= 8; k++) {
                    const int qblocks = (n + qb - 1) / qb;
                    const int most = block_tiles(pos0, n, qb, qblocks - 1);
                    const int chunk = k == 1 ? 0 : (((most + k - 1) / k) + 1) & ~1;
                    long item = 0;
                    for (int b = qblocks - 1; b >= 0; b--) {
                        const int runs = block_runs(block_tiles(pos0, n, qb, b), chunk);
                        for (int s = 0; s < runs; s++, item++, seen++) {
                            const BlockRun r = block_of_run(pos0, n, qb, qblocks, chunk, (int)item);
                            wrong += r.blk != b || r.run != s || r.runs != runs;
                        }
                    }
                    wrong += total_runs(pos0, n, qb, qblocks, chunk) != item;
                }
    // the plans themselves: every run once, whole blocks first, all counted
    for (int nkv : {1, 2, 4, 8, 16, 32, 64, 100, 300})
        for (int qb : {16, 32, 64, 128})
            for (int pos0 : {0, 500, 2000, 4000, 8000, 30000})
                for (int n = 1; n < 4300; n += n < 200 ? 13 : 101) {
                    const int qblocks = (n + qb - 1) / qb;
                    const RunPlan p = plan_runs(128, qb, nkv, pos0, n, qblocks, -1);
                    mixed += p.whole > 0;
                    int item = 0, most = 1;
                    for (int b = qblocks - 1; b >= 0; b--) {
                        const int cut = qblocks - 1 - b < p.whole ? 0 : p.chunk;
                        const int runs = block_runs(block_tiles(pos0, n, qb, b), cut);
                        most = runs > most ? runs : most;
                        for (int s = 0; s < runs; s++, item++) {
                            const BlockRun r = plan_item(pos0, n, qb, qblocks, p.whole, p.chunk, item);
                            wrong += r.blk != b || r.run != s || r.runs != runs;
                        }
                    }
                    wrong += item != p.items || most != p.runs || p.runs > kMaxRuns;
                }
    std::printf("%ld %ld %ld\n", seen, wrong, mixed);
}
"""


PLAN = r"""
#include <cstdio>
#include <cstdlib>
#include "prefill_runs.hpp"
int main(int, char **v) {
    const int nq = atoi(v[1]), nkv = atoi(v[2]), hd = atoi(v[3]), n = atoi(v[4]), pos0 = atoi(v[5]), qb = 128 / (nq / nkv);
    const tq::RunPlan p = tq::plan_runs(hd, qb, nkv, pos0, n, (n + qb - 1) / qb, -1);
    std::printf("%d %d\n", p.whole, p.runs);
}
"""

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


def build(tmp, text):
    src, exe = tmp / "runs.cpp", tmp / "runs"
    src.write_text(text)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-D__host__=", "-D__device__=",
                    "-I", os.path.join(ROOT, "tailorquantkernel_amd", "csrc"), "-o", str(exe), str(src)], check=True)
    return lambda *args: subprocess.run([str(exe), *map(str, args)], check=True, capture_output=True, text=True).stdout.split()


def test_block_of_run_equals_the_count(tmp_path):
    seen, wrong, mixed = map(int, build(tmp_path, HARNESS)())
    assert seen > 100_000 and mixed > 100 and wrong == 0, (seen, wrong, mixed)


def test_plan_takes_the_measured_cuts(tmp_path):
    """Whole blocks in more than one round of the CUs where those were the
    fastest of 1 to 8 runs (the times beside each), runs where runs were."""
    plan = build(tmp_path, PLAN)
    for shape, runs in (((32, 8, 128, 2000, 2000), 1),     # us whole 227, two runs 277
                        ((32, 8, 128, 2000, 8000), 1),     # 597, 627
                        ((16, 4, 128, 4000, 0), 1),        # 155, 195
                        ((16, 2, 128, 4000, 0), 1),        # 151, 192
                        ((64, 8, 128, 1000, 16000), 1),    # 1059, 1111
                        ((8, 1, 128, 8000, 0), 1),         # 275, 336
                        ((8, 2, 64, 4000, 4000), 2),       # two runs 141, whole 174
                        ((16, 4, 128, 2048, 0), 3),        # three 73, whole 77
                        ((32, 8, 128, 333, 1000), 2),
                        ((32, 8, 128, 100, 8000), 8),
                        ((8, 2, 64, 2048, 0), 3)):
        assert plan(*shape) == ["0", str(runs)], shape
    # a little over one round: 32 of 35 blocks whole, the others in runs
    assert plan(32, 8, 128, 1100, 2000) == ["32", "3"]
    assert plan(64, 8, 128, 600, 4000) == ["32", "4"]

"""The prefill's (block, run) lookup against the count it replaces, block by
block, over the sizes and cuts the plan can make; CPU only."""
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
    long seen = 0, wrong = 0;
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
    std::printf("%ld %ld\n", seen, wrong);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_block_of_run_equals_the_count(tmp_path):
    src, exe = tmp_path / "runs.cpp", tmp_path / "runs"
    src.write_text(HARNESS)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-D__host__=", "-D__device__=",
                    "-I", os.path.join(ROOT, "tailorquantkernel_amd", "csrc"), "-o", str(exe), str(src)], check=True)
    seen, wrong = map(int, subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split())
    assert seen > 100_000 and wrong == 0, (seen, wrong)

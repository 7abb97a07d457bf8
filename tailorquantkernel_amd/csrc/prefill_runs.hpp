// The prefill's work items: query blocks, longest first, each cut into runs of
// its key tiles.  Host (the plan) and device (a work-group finding its run)
// use the same functions.
#pragma once

namespace tq {

constexpr int kKT = 32;   // keys per tile

// Key tiles query block b of qb tokens reads: keys [0, pos0 + its last query + 1).
__host__ __device__ inline int block_tiles(int pos0, int n, int qb, int b) {
    const int last = (b + 1) * qb < n ? (b + 1) * qb : n;
    return (pos0 + last + kKT - 1) / kKT;
}

// Runs a block of nt tiles is cut into (chunk 0: every block is one run).
__host__ __device__ inline int block_runs(int nt, int chunk) { return chunk == 0 ? 1 : (nt + chunk - 1) / chunk; }

struct BlockRun {
    int blk, run, runs;   // query block, which of its runs, how many it has
};

// Run `item` in order of falling blocks.  Block b < the last ends at key
// e = pos0 + (b + 1) qb and has ceil(e / (kKT chunk)) runs, so the blocks of r
// runs are one interval: a step per run count (at most the longest block's, 8),
// not one per block, of which 1 or 2 kv heads have hundreds (8 / 1 heads of
// 128, 8,000 tokens after none: 464 us with a work-group counting block by
// block, 348 so; 4,000 tokens 132 and 107).
__host__ __device__ inline BlockRun block_of_run(int pos0, int n, int qb, int qblocks, int chunk, int item) {
    if (chunk == 0) return BlockRun{qblocks - 1 - item, 0, 1};
    const int last = block_runs(block_tiles(pos0, n, qb, qblocks - 1), chunk);
    if (item < last || qblocks == 1) return BlockRun{qblocks - 1, item < last ? item : last - 1, last};
    item -= last;
    const int keys = kKT * chunk;
    int hi = qblocks - 2;   // the blocks still to pass are 0..hi
    for (int r = (pos0 + (hi + 1) * qb + keys - 1) / keys;; r--) {
        const int below = (r - 1) * keys - pos0;   // blocks of r runs end past this token
        const int lo = below < 0 ? 0 : below / qb;
        const int runs = (hi - lo + 1) * r;
        if (item < runs) return BlockRun{hi - item / r, item % r, r};
        if (lo == 0) return BlockRun{0, r - 1, r};
        item -= runs;
        hi = lo - 1;
    }
}

// Runs of all blocks.
__host__ __device__ inline long total_runs(int pos0, int n, int qb, int qblocks, int chunk) {
    if (chunk == 0) return qblocks;
    long sum = block_runs(block_tiles(pos0, n, qb, qblocks - 1), chunk);
    const int keys = kKT * chunk;
    for (int hi = qblocks - 2; hi >= 0;) {
        const int r = (pos0 + (hi + 1) * qb + keys - 1) / keys;
        const int below = (r - 1) * keys - pos0;
        const int lo = below < 0 ? 0 : below / qb;
        sum += (long)(hi - lo + 1) * r;
        hi = lo - 1;
    }
    return sum;
}

}  // namespace tq

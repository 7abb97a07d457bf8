// The prefill's work items: query blocks, longest first, each cut into runs of
// its key tiles.  Host (the plan) and device (a work-group finding its run)
// use the same functions.
#pragma once

#include <algorithm>
#include <cmath>

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

// How the blocks are cut: the `whole` longest are one run each, the others have
// runs of at most `chunk` key tiles (0: one run); `runs` is the most of a block,
// `items` all of them.
struct RunPlan {
    int whole, chunk, runs, items;
};

// Item `item` of a plan.
__host__ __device__ inline BlockRun plan_item(int pos0, int n, int qb, int qblocks, int whole, int chunk, int item) {
    if (item < whole) return BlockRun{qblocks - 1 - item, 0, 1};
    const int cut = qblocks - whole;
    return block_of_run(pos0, whole > 0 ? cut * qb : n, qb, cut, chunk, item - whole);
}

constexpr int kCUs = 256;       // compute units of an MI355X
constexpr int kMaxRuns = 8;     // runs of one query block
// The plan's costs, in steps (a pair of key tiles, about 1.7 us at head_dim
// 128): a work-group's prologue and store, its partial, and each run the last
// one merges.
constexpr double kItemCost = 3.5, kRunCost = 1.5, kMergeCost = 1.0;

// With at least two query blocks per CU, every (query block, kv head) is one
// work-group: dealt longest first, the blocks pair up on the CUs by
// themselves.  With fewer, blocks may be cut into runs of `chunk` key tiles,
// the length that minimises the modelled time.  While the launch is one round
// of the CUs that is one work-group's (steps, fixed cost).  Whole blocks of
// head_dim 128 in more than one round are exactly predictable: a CU holds one
// work-group, so the shortest of the first round frees the first CU, and block
// 257 of the order pairs with 256, 258 with 255, ...  Otherwise it is the CUs'
// share of all work, rounds taken halfway to whole ones, and a third of a
// work-group's at the end.  The merge of all runs by the last comes on top.
//
// A little over one round of equal blocks (keys before the prompt) suits no
// such cut: whole, the second round is nearly empty, and in runs of all blocks
// every one pays for the cut.  There the longest blocks that fill the CUs once stay
// whole and only the others are cut, to run on the CUs left and then beside
// them: share of all work and half a run at the end.  32 / 8 heads of 128, us so,
// whole and in three runs: 1,100 after 2,000 129, 161, 166; after 8,000 346, 511,
// 400; 64 / 8, 600 after 4,000 201, 274, 236.
//
// Over 100 measured shapes, each with its blocks in 1 to 8 runs, the choice among
// those eight takes 1.0 % longer than the best in the mean, 15 % at most.  Choices, us of the choice and the next best: 32 / 8
// heads of 128, 2,000 after 2,000: whole 227, two runs 277; 333 after 1,000: two
// 46, whole 56; 100 after 8,000: eight 74, four 95; 16 / 4, 4,000 after none: whole
// 155, two 195; 8 / 2 of 64, 4,000 after 4,000: two 141, whole 174; 2,048 after
// none: three 32, two 35.
//
// forced: 1 keeps every block one run, 0 cuts every block into as many runs as
// may be, -1 lets the costs decide.
inline RunPlan plan_runs(int hd, int qb, int n_kv_heads, int pos0, int n, int qblocks, int forced) {
    RunPlan p{0, 0, 1, qblocks};
    if (forced == 1 || (forced < 0 && (long)qblocks * n_kv_heads >= 2L * kCUs)) return p;
    const int most = block_tiles(pos0, n, qb, qblocks - 1);   // of the last, longest block
    // time of the i-th longest (block, kv head) as one work-group
    auto whole = [&](int i) { return 0.5 * block_tiles(pos0, n, qb, qblocks - 1 - i / n_kv_heads) + kItemCost; };
    long tiles = 0;
    for (int b = 0; b < qblocks; b++) tiles += block_tiles(pos0, n, qb, b);
    double best = 0.0;
    for (int k = 1; k <= kMaxRuns && (k == 1 || (most + 1) / 2 >= k); k++) {
        const int chunk = (((most + k - 1) / k) + 1) & ~1;
        const long items = total_runs(pos0, n, qb, qblocks, chunk), wgs = items * n_kv_heads;
        const int runs = block_runs(most, chunk);
        const double item = kItemCost + (runs > 1 ? kRunCost : 0.0), one = 0.5 * (k == 1 ? most : chunk) + item;
        double cost;
        if (wgs <= kCUs) {
            cost = one;
        } else if (k == 1 && hd == 128 && wgs < 2 * kCUs) {
            cost = std::max({one, whole(kCUs - 1) + whole(kCUs), whole(2 * kCUs - 1 - (int)wgs) + whole((int)wgs - 1)});
        } else {
            const double rounds = (double)wgs / kCUs, share = n_kv_heads * (0.5 * tiles + items * item) / kCUs;
            cost = std::max(one, share * 0.5 * (1.0 + std::ceil(rounds) / rounds) + 0.3 * one);
        }
        if (runs > 1) cost += kMergeCost * runs;
        if (forced == 0 || k == 1 || cost < best) {
            best = cost;
            p = RunPlan{0, k == 1 ? 0 : chunk, runs, (int)items};
        }
    }
    const int full = kCUs / n_kv_heads, cut = qblocks - full;   // blocks of one round, and those beyond it
    if (forced == 0 || hd != 128 || full < 1 || cut < 1 || qblocks * n_kv_heads <= kCUs) return p;
    const int longest = block_tiles(pos0, n, qb, cut - 1);
    for (int k = 2; k <= kMaxRuns && (longest + 1) / 2 >= k; k++) {
        const int chunk = (((longest + k - 1) / k) + 1) & ~1;
        const long items = total_runs(pos0, cut * qb, qb, cut, chunk);
        const double run = kItemCost + kRunCost, share = n_kv_heads * (0.5 * tiles + full * kItemCost + items * run) / kCUs;
        const int runs = block_runs(longest, chunk);
        const double cost = std::max(0.5 * most + kItemCost, share + 0.5 * (0.5 * chunk + run)) + kMergeCost * runs;
        if (cost < best) {
            best = cost;
            p = RunPlan{full, chunk, runs, full + (int)items};
        }
    }
    return p;
}

}  // namespace tq

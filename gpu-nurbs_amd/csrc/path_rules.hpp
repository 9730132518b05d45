// path_rules.hpp -- which kernels an inversion takes: pure functions of sizes and options (no HIP).
#pragma once
#include <cstddef>

namespace gn {

// Iteration limits of a call.
struct PathOpts {
    bool mixed;
    bool newton64;
    int max_iter, fp32_iters, fp64_tail;
};

// The longest chain a lane can hold its wave up for, in FP32 iterations (an FP64 one costs about three).
inline size_t chain_limit(const PathOpts &o) {
    return o.mixed ? (size_t)o.fp32_iters + 3 * (size_t)o.fp64_tail : (size_t)o.max_iter;
}

// Batched calls: whether a class group's `points` go to the persistent kernels (batch_refill.hip), whose
// lanes take another point when theirs has stopped, and not to k_batch_tile, whose waves end with their
// slowest lane.  k_batch_tile needs one launch and keeps the lanes' patches at hand, and wins wherever
// its waves all run at once; with every further round the lanes that wait cost more, the longer a chain
// may get.  In rounds of the lanes resident at once: mixed 8, 4 and 4 waves per CU for the three groups, FP64
// 4, 3 and 2 (registers and LDS).  Times refill / tile on 16 surfaces, points offset by 1e-2 of the
// model's size, without / with 2% of them anywhere:
//   group 0, FP64 Gauss-Newton of at most 20 steps: 1.42 / 1.27 at 1,048,576 points (2% of points
//     anywhere among others on the surface: 0.72): tile.
//     Group 1 (4,4): 1.11 / 0.96 at 131,072 points, 1.05 / 0.88 at twice as many.
//   other FP64: Newton, 20 steps, (3,3) 0.98 / 0.93 at one round, 0.80 / 0.63 at 16; (5,5) Gauss-Newton 1.19 /
//     1.07 at one round, 0.67 / 0.62 at two.  50 Newton steps (3,3) 1.03 / 1.00 at half a round, 0.79 / 0.73
//     at one.
//   mixed, 6 FP32 and 3 FP64 steps (chain limit 15): group 0 1.19 / 1.08 at 1,048,576, 1.13 / 1.00 at 4
//     times that: tile; (5,5) 1.16 / 1.01 at 4 rounds, 1.02 / 0.85 at 16.  20 and 3 (29): group 0 1.08 / 0.84 at
//     1,048,576; (5,5) 1.13 / 0.89 at two rounds, 0.90 / 0.58 at 16.  6 and 12 (42): (3,3) 1.16 / 1.01 at two,
//     0.96 / 0.77 at 8.  30 and 40 (150): (3,3) 1.01 / 0.93 at half a round, 0.68 / 0.45 at 8.
inline bool batch_takes_refill(int grp, size_t points, const PathOpts &o, size_t cus) {
    const size_t limit = chain_limit(o);
    const size_t waves = o.mixed ? (grp == 0 ? 8 : 4) : (size_t)(4 - grp), round = 64 * waves * cus;
    if (!o.mixed) {
        if (grp == 0 && !o.newton64 && limit <= 20) return false;
        return points > (limit > 20 ? round / 2 : grp == 1 && !o.newton64 ? 3 * round : round);
    }
    if (grp == 0 && limit <= 32) return false;
    return points * limit > round * (grp == 0 ? 84 : 64);
}

}  // namespace gn

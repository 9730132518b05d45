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

// Single-surface calls of exact degrees (2..5) with their knots in LDS: whether `n` points go from seed to
// result in one kernel (k_gn_tile), or to seeds and the persistent kernels, which refill lanes whose
// points have stopped where that kernel starts a new wave and waits for its slowest lane.  knots: of both
// directions.  All ratios are persistent / tile, without / with 2% of the points anywhere.
// Mixed: points times patch entries times chain limit up to 120 M on 256 CUs.  6 FP32 and 3 FP64 steps
// (15): (3,3) 1.26 / 1.15 at 262,144 points, 1.10 / 0.96 at 500,000, 0.91 / 0.77 at 1,000,000; (5,5) 1.25 / 1.09 at
// 131,072, 1.08 / 0.84 at 262,144.  20 and 3 (29): (3,3) 1.21 / 0.97 at 262,144, 1.03 / 0.73 at 500,000; (5,5) 1.55 /
// 1.28 at 65,536, 1.37 / 0.86 at 131,072.  6 and 12 (42): (3,3) 1.07 / 1.17 at 131,072, 1.03 / 0.86 at 262,144.  30
// and 40 (150): (3,3) 1.08 / 0.96 at 65,536, 0.84 / 0.96 at 131,072; (5,5) 1.24 / 1.25 at 32,768, 1.04 / 0.86 at
// 65,536: whatever the limit, 98,304 bicubic points win or lose little.  A patch of 9 entries counts as 5:
// (2,2) 1.26 / 0.98 at 500,000 points for 29; for 15 it wins nearly always, 1.28 / 1.12 at 1,000,000, 1.04 / 0.92 at
// 4,000,000, 1.16 / 1.11 at 16,000,000.  Without Newton steps in FP64 the persistent closing pass is the
// slower one, and the limit counts half: 20 and 3, (3,3) 1.47 / 1.38 at 262,144, 1.05 / 0.93 at 500,000.
// FP64: by rounds, as many points as the chip's LDS holds patches for (65,536 bicubic, 114,688 biquadratic,
// 32,768 of degree (5,5)); 20 Gauss-Newton steps: one round always wins, (3,3) 1.19 / 1.17 at 65,536, 0.91 / 0.86
// at 131,072; (2,2) 1.29 / 1.27 at 262,144; (5,5) 1.13 / 1.05 at 32,768, 0.61 / 0.57 at 65,536.  Newton steps end
// most points early, half as many: (3,3) 1.07 / 1.11 at 32,768, 0.92 / 0.90 at 65,536; (2,2) 1.08 / 1.11 at 131,072,
// 0.92 / 0.86 at 262,144.  More than 20 steps, a third: 50 Newton steps (3,3) 0.95 / 1.02 at 32,768, 0.81 / 0.79 at
// 65,536; 100 Gauss-Newton steps (2,2) 1.09 / 1.13 at 131,072, 0.78 / 0.74 at 262,144.
inline bool call_takes_tile(int p, int q, size_t knots, size_t n, const PathOpts &o, size_t cus) {
    if (knots > 1024 || p < 2 || p > 5 || q < 2 || q > 5) return false;
    const size_t entries = (size_t)((p + 1) * (q + 1)), limit = chain_limit(o);
    if (o.mixed)
        return n * entries <= 6144 * cus ||
               (n < ((size_t)1 << 31) &&
                ((entries <= 9 && limit <= 16) ||
                 n * (entries <= 9 ? 5 : entries) * limit <= 468750 * cus * (o.newton64 ? 1 : 2)));
    // a wave's LDS: the lanes' patches; knots and reciprocal span lengths, two of them short of the knots
    const size_t lds = ((entries * 2) | 1) * 16 * 64 + sizeof(double) * 2 * (knots - p - q - 1);
    const size_t w = 160 * 1024 / lds, most = cus * 32 * w * (w >= 6 ? 6 : w >= 4 ? 3 : 2);
    return n <= (limit > 20 ? most / 3 : o.newton64 ? most / 2 : most);
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
// Beside other groups a persistent launch, which fills the chip, costs more: uneven surfaces of all three
// groups, the second group by refill and by tile, us: 236,000 points (3.6 rounds) 340 / 287 for a limit of 42, 339 /
// 287 for 29; 448,000 (6.8 rounds) 473 / 492 for 29, 398 / 365 for 15; 1,068,000 798 / 791 for 15.
inline bool batch_takes_refill(int grp, size_t points, bool several, const PathOpts &o, size_t cus) {
    const size_t limit = chain_limit(o);
    const size_t waves = o.mixed ? (grp == 0 ? 8 : 4) : (size_t)(4 - grp), round = 64 * waves * cus;
    if (!o.mixed) {
        if (grp == 0 && !o.newton64 && limit <= 20) return false;
        return points > (limit > 20 ? round / 2 : grp == 1 && !o.newton64 ? 3 * round : round);
    }
    if (grp == 0 && limit <= 32) return false;
    return points * limit > round * (grp == 0 ? 84 : several ? 160 : 64);
}

}  // namespace gn

// invert_tile.hpp -- a point's whole inversion on one lane: the seed, the FP32 bulk and the FP64
// iterations, for the single-surface and the batched small-call kernels.
#pragma once
#include "gn_search.hpp"
#include "invert_common.hpp"

namespace gn {

// Levels of the seed quadtree whose boxes a wave stages (with the root 341 boxes, 8 KB).
constexpr int kTileSeedLevels = 4;
constexpr int kTileBoxBytes = (((1 << (2 * (kTileSeedLevels + 1))) - 1) / 3) * 24;

// 16-byte vectors of a wave's LDS: the lanes' patches, at first the staged boxes.  Mixed precision
// keeps the FP32 patches here and reads the FP64 ones (one iteration for 95% of the points) from
// memory: half the LDS, twice the waves per CU (100,000 points (4,4) 66 -> 51 us, 250,001 bicubic
// 76 -> 59).
template <int K1, int K2, bool MIXED>
constexpr int tile_patch_vecs() {
    const int v = 64 * (MIXED ? lane_patch_stride<K1, K2, float>() : lane_patch_stride<K1, K2, double>());
    return v > kTileBoxBytes / 16 + 1 ? v : kTileBoxBytes / 16 + 1;
}


// Stages the boxes of levels 0..kTileSeedLevels for the greedy seeds (1, 2) into `boxes`, where the
// patches go afterwards; returns the levels staged.
__device__ __forceinline__ int tile_stage_boxes(const GnSearchDev &sd, int seed, float4 *boxes) {
    if (seed != 1 && seed != 2) return 0;
    const int ll = sd.depth < kTileSeedLevels ? sd.depth : kTileSeedLevels;
    const float2 *src = reinterpret_cast<const float2 *>(sd.box32);
    float2 *dst = reinterpret_cast<float2 *>(boxes);
    const int nf2 = (int)qoff(ll + 1) * 3;
#pragma unroll 8
    for (int e = threadIdx.x; e < nf2; e += 64) dst[e] = src[e];
    return ll;
}

// seed: 1 the greedy descent's leaf, 2 with its step; 3 the seed grid's leaf with its step.
__device__ __forceinline__ void tile_seed(const GnSearchDev &sd, int seed, const float4 *boxes, int ll,
                                          const double P[3], double &cu, double &cv) {
    if (seed == 3) {
        const uint32_t c = sd.grid_wide ? grid_leaf<true>(sd, P) : grid_leaf<false>(sd, P);
        step_seed(sd, c, sd.rec[(size_t)c * kRecVec], P, cu, cv);
        return;
    }
    float4 cq;
    const uint32_t c = greedy_leaf(sd, P, reinterpret_cast<const float *>(boxes) + 6, ll, &cq,
                                   seed == 1);
    if (seed == 2) {
        step_seed(sd, c, cq, P, cu, cv);
    } else {
        cu = sd.seed_uv[c * 2 + 0];
        cv = sd.seed_uv[c * 2 + 1];
    }
}

// All iterations of the workgroup's (one wave's) points; returns the status, it32 and it64 the
// iteration counts.  patches: tile_patch_vecs (EXACT).  Called by the whole wave; a lane without a
// point passes valid == false.
template <int K1, int K2, bool EXACT, bool MIXED, bool NEWTON32, bool NEWTON64>
__device__ __forceinline__ int tile_iterate(const GnSurfDev &d, const double *ku, const double *kv,
                                            const Domain &dom, const gn_invert_opts &o,
                                            const double P[3], bool valid, float4 *patches,
                                            double &cu, double &cv, int &it32, int &it64) {
    constexpr int P32 = EXACT ? kPatchLane : kPatchGlobal, P64 = MIXED ? kPatchGlobal : P32;
    int lim = o.max_iter;
    it32 = 0;
    if constexpr (MIXED) {
        const double su = cu, sv = cv;
        SpanCache sc;
        int st = valid && o.fp32_iters > 0 ? kStepContinue : GN_PT_MAXITER;
        while (st == kStepContinue) {
            st = gn_step<K1, K2, EXACT, float, NEWTON32, P32, false, true>(
                d, ku, kv, (float)P[0], (float)P[1], (float)P[2], cu, cv, 0.0, o.tol_step32, 0.0,
                o.clamp, dom, sc, nullptr,
                patches + threadIdx.x * lane_patch_stride<K1, K2, float>());
            if (st == kStepContinue || st == GN_PT_CONVERGED) it32++;
            if (st == kStepContinue && it32 >= o.fp32_iters) st = GN_PT_MAXITER;
        }
        if (st == GN_PT_SINGULAR || st == GN_PT_NONFINITE) {  // a breakdown restarts from the seed
            cu = su;
            cv = sv;
        } else {
            lim = o.fp64_tail;
        }
    }
    const double tq = NEWTON64 ? o.tol_quad : 0.0;
    SpanCache sc;
    int st = valid && lim > 0 ? kStepContinue : GN_PT_MAXITER;
    it64 = 0;
    while (st == kStepContinue) {
        st = gn_step<K1, K2, EXACT, double, NEWTON64, P64, false, true>(
            d, ku, kv, P[0], P[1], P[2], cu, cv, o.tol_dist, o.tol_step, tq, o.clamp, dom, sc, nullptr,
            patches + threadIdx.x * lane_patch_stride<K1, K2, double>());
        if (st == kStepContinue || st == GN_PT_CONVERGED) it64++;
        if (st == kStepContinue && it64 >= lim) st = GN_PT_MAXITER;
    }
    return st;
}

}  // namespace gn

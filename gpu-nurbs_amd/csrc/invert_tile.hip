// invert_tile.hip -- inversion of calls of up to a few points per lane of the chip: the seed, the FP32
// bulk and the FP64 iterations of a point in one kernel.
#include "gn_search.hpp"
#include "invert_common.hpp"

namespace gn {

// Levels of the seed quadtree whose boxes a wave stages (with the root 341 boxes, 8 KB): what the
// smallest patches' LDS holds.
constexpr int kTileSeedLevels = 4;

// Every lane keeps one point from its seed to its result; a wave is a workgroup, so a call of n
// points is n / 64 waves on as many CUs as there are.  What bounds a small call is the latency of
// one point's chain: an FP64 iteration of the persistent kernels takes 3 us, most of it row loads
// that wait for each other and for the counters' atomics.  Here an iteration touches memory only
// where a point enters another span: the lane's patch lies in its own LDS (in registers it needs an
// accumulator copy per operand: 54 against 49 us), the loads of a new one are issued together, and
// the seed and the FP32 bulk cost no launch and no pass over the parameters.  The arithmetic is the
// persistent kernels', so the results are the same bits.
// 4,096 points in one kernel, before (two launches plain, four mixed) and now: plain FP64 8 x 8
// bicubic 26.5 -> 14.3 us, 32 x 32 72.6 -> 46.2, degree (4,4) 94 -> 60; mixed 31 -> 11, 47.5 -> 20.8
// and 57 -> 28.  Of the 46 us, 22 iterations of the slowest lane are 1.6 us each.

// seed: 0 the parameters in a.u, a.v; 1 the greedy descent's leaf, 2 with its step; 3 the seed grid's
// leaf with its step.
template <int K1, int K2, bool MIXED, bool NEWTON32, bool NEWTON64>
__global__ __launch_bounds__(64, 1) void k_gn_tile(GnSurfDev d_in, GnSearchDev sd, InvArgs a,
                                                   int seed) {
    constexpr int kStride = lane_patch_stride<K1, K2, double>();
    __shared__ float4 patches[64 * kStride];
    extern __shared__ double sk[];
    const size_t i = (size_t)blockIdx.x * 64 + threadIdx.x;
    const bool valid = i < a.n;
    double P[3] = {0, 0, 0}, cu = 0, cv = 0;
    if (valid) {
        P[0] = a.x[i];
        P[1] = a.y[i];
        P[2] = a.z[i];
        if (seed == 0) {
            cu = a.u[i];
            cv = a.v[i];
        }
    }
    int ll = 0;
    if (seed == 1 || seed == 2) {  // the boxes of levels 0..ll, where the patches go afterwards
        static_assert((((1 << (2 * (kTileSeedLevels + 1))) - 1) / 3) * 24 <= sizeof(patches), "");
        ll = sd.depth < kTileSeedLevels ? sd.depth : kTileSeedLevels;
        const float2 *src = reinterpret_cast<const float2 *>(sd.box32);
        float2 *dst = reinterpret_cast<float2 *>(patches);
        const int nf2 = (int)qoff(ll + 1) * 3;
#pragma unroll 8
        for (int e = threadIdx.x; e < nf2; e += 64) dst[e] = src[e];
    }
    const GnSurfDev d = stage_knots_lds(d_in, sk);
    if (seed != 0 && valid) {
        if (seed == 3) {
            const uint32_t c = sd.grid_wide ? grid_leaf<true>(sd, P) : grid_leaf<false>(sd, P);
            step_seed(sd, c, sd.rec[(size_t)c * kRecVec], P, cu, cv);
        } else {
            float4 cq;
            const uint32_t c = greedy_leaf(sd, P, reinterpret_cast<const float *>(patches) + 6, ll,
                                           &cq, seed == 1);
            if (seed == 2) {
                step_seed(sd, c, cq, P, cu, cv);
            } else {
                cu = sd.seed_uv[c * 2 + 0];
                cv = sd.seed_uv[c * 2 + 1];
            }
        }
    }
    __syncthreads();  // every lane has left the boxes
    const double *ku = sk, *kv = sk + d.nu + d.p + 1;
    const Domain dom = domain_of(d);
    int lim = a.o.max_iter;
    if constexpr (MIXED) {
        const double su = cu, sv = cv;
        SpanCache sc;
        int it = 0, st = valid && a.o.fp32_iters > 0 ? kStepContinue : GN_PT_MAXITER;
        while (st == kStepContinue) {
            st = gn_step<K1, K2, true, float, NEWTON32, kPatchLane, false, true>(
                d, ku, kv, (float)P[0], (float)P[1], (float)P[2], cu, cv, 0.0, a.o.tol_step32, 0.0,
                a.o.clamp, dom, sc, nullptr,
                patches + threadIdx.x * lane_patch_stride<K1, K2, float>());
            if (st == kStepContinue || st == GN_PT_CONVERGED) it++;
            if (st == kStepContinue && it >= a.o.fp32_iters) st = GN_PT_MAXITER;
        }
        if (valid && a.it32) a.it32[i] = sat8(it);
        if (st == GN_PT_SINGULAR || st == GN_PT_NONFINITE) {
            cu = su;
            cv = sv;
        } else {
            lim = a.o.fp64_tail;
        }
        __syncthreads();
    } else {
        if (valid && a.it32) a.it32[i] = 0;
    }
    const double tq = NEWTON64 ? a.o.tol_quad : 0.0;
    SpanCache sc;
    int it = 0, st = valid && lim > 0 ? kStepContinue : GN_PT_MAXITER;
    while (st == kStepContinue) {
        st = gn_step<K1, K2, true, double, NEWTON64, kPatchLane, false, true>(
            d, ku, kv, P[0], P[1], P[2], cu, cv, a.o.tol_dist, a.o.tol_step, tq, a.o.clamp, dom, sc,
            nullptr, patches + threadIdx.x * kStride);
        if (st == kStepContinue || st == GN_PT_CONVERGED) it++;
        if (st == kStepContinue && it >= lim) st = GN_PT_MAXITER;
    }
    if (!valid) return;
    a.u[i] = cu;
    a.v[i] = cv;
    a.status[i] = (uint8_t)st;
    if (a.it64) a.it64[i] = sat8(it);
}

struct TileLaunch {
    const GnSurfDev &d;
    const GnSearchDev &sd;
    const InvArgs &a;
    int seed;
    hipStream_t st;
    template <int K1, int K2, bool EXACT>
    int operator()() {
        if constexpr (EXACT) {
            const bool n64 = a.o.newton & GN_NEWTON_FP64, n32 = a.o.newton & GN_NEWTON_FP32;
            auto k = a.o.precision != GN_MIXED
                         ? (n64 ? k_gn_tile<K1, K2, false, false, true>
                                : k_gn_tile<K1, K2, false, false, false>)
                     : n32 ? (n64 ? k_gn_tile<K1, K2, true, true, true>
                                  : k_gn_tile<K1, K2, true, true, false>)
                           : (n64 ? k_gn_tile<K1, K2, true, false, true>
                                  : k_gn_tile<K1, K2, true, false, false>);
            const size_t lds = sizeof(double) * (2 * (d.nu + d.nv) + 2);
            k<<<(unsigned)((a.n + 63) / 64), 64, lds, st>>>(d, sd, a, seed);
            GN_HIP(hipGetLastError());
        }
        return GN_OK;
    }
};

// Waves of this kernel that a CU's 160 KB of LDS hold (registers would allow four to eight).
static int tile_waves_per_cu(const GnSurfDev &d) {
    const size_t vec = (size_t)((d.p + 1) * (d.q + 1) * 2) | 1;
    return (int)((160 * 1024) / (vec * 16 * 64 + sizeof(double) * (2 * (d.nu + d.nv) + 2)));
}

// Whether the call runs faster here than as seeds plus persistent kernels.  A round is as many
// points as the chip's LDS holds patches for: 65,536 for bicubic FP64, 114,688 biquadratic, 32,768
// of degree (5,5).  Within one round this kernel always wins (FP64: (3,3) 46 against 72 us at 4,096
// points, 63 against 77 at 65,536; (5,5) 102 against 171 at 16,000; mixed: (3,3) 21 against 47 and
// 26 against 50).  Past it the persistent kernels refill lanes whose points have stopped, this one
// starts over: FP64 (3,3) 87 against 105 us at 80,000 but 114 against 105 at 131,072, (2,2) 112
// against 150 at 320,000, (5,5) 201 against 146 at 65,000; mixed (3,3) 44 against 57 at 131,072 and
// 76 against 72 at 250,001, (2,2) 50 against 70 at 320,000, (5,5) 78 against 73 at 65,000.
bool gn_tile_takes(const GnSurfDev &d, const InvArgs &a) {
    if (!knots_fit_lds(d) || d.p < 2 || d.p > 5 || d.q < 2 || d.q > 5) return false;
    const int w = tile_waves_per_cu(d);
    const int halves = w >= 6 ? 6 : a.o.precision != GN_MIXED ? (w >= 4 ? 3 : 2) : w >= 3 ? 4 : 3;
    return a.n <= (size_t)cu_count() * 32 * w * halves;
}

int launch_gn_tile(const GnSurfDev &d, const GnSearchDev &sd, const InvArgs &a, int seed,
                   hipStream_t st) {
    return dispatch_degrees(d.p, d.q, TileLaunch{d, sd, a, seed, st});
}

}  // namespace gn

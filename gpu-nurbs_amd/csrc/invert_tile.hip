// invert_tile.hip -- inversion of calls of up to a few points per lane of the chip: the seed, the FP32
// bulk and the FP64 iterations of a point in one kernel.
#include "invert_tile.hpp"
#include "path_rules.hpp"

namespace gn {

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

// seed: 0 the parameters in a.u, a.v, else as tile_seed.
template <int K1, int K2, bool MIXED, bool NEWTON32, bool NEWTON64>
__global__ __launch_bounds__(64, 1) void k_gn_tile(GnSurfDev d_in, GnSearchDev sd, InvArgs a,
                                                   int seed) {
    __shared__ float4 patches[tile_patch_vecs<K1, K2, MIXED>()];
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
    const int ll = tile_stage_boxes(sd, seed, patches);
    const GnSurfDev d = stage_knots_lds(d_in, sk);
    if (seed != 0 && valid) tile_seed(sd, seed, patches, ll, P, cu, cv);
    __syncthreads();  // every lane has left the boxes
    int it32, it64;
    const int st = tile_iterate<K1, K2, true, MIXED, NEWTON32, NEWTON64>(
        d, sk, sk + d.nu + d.p + 1, domain_of(d), a.o, P, valid, patches, cu, cv, it32, it64);
    if (!valid) return;
    a.u[i] = cu;
    a.v[i] = cv;
    a.status[i] = (uint8_t)st;
    if (a.it32) a.it32[i] = sat8(it32);
    if (a.it64) a.it64[i] = sat8(it64);
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

bool gn_tile_takes(const GnSurfDev &d, const InvArgs &a) {
    const PathOpts o{a.o.precision == GN_MIXED, (a.o.newton & GN_NEWTON_FP64) != 0, a.o.max_iter,
                     a.o.fp32_iters, a.o.fp64_tail};
    return call_takes_tile(d.p, d.q, (size_t)(d.nu + d.p + 1 + d.nv + d.q + 1), a.n, o, (size_t)cu_count());
}

int launch_gn_tile(const GnSurfDev &d, const GnSearchDev &sd, const InvArgs &a, int seed,
                   hipStream_t st) {
    return dispatch_degrees(d.p, d.q, TileLaunch{d, sd, a, seed, st});
}

}  // namespace gn

// batch.hip -- inversion of many surfaces of uneven degree and net size (the batched form of
// NewInverse + GaussNewton, src/kernel/kernel.cu:151-249, 433-469).
//
// A batch packs the span tables, knots and seed trees of its surfaces into one allocation and
// describes each surface by a GnBatchObj (pointers into the pack, degree class).  Work is a list
// of tiles (object, contiguous point range, request) sorted by degree class.  The 17 degree
// classes (exact unrolled contraction for degrees 2..5 in each direction, padded generic form
// otherwise) fall into three groups by patch size (K1*K2 <= 16, <= 25, larger or generic); each
// group present gets its own launch, on its own side stream, of a kernel instantiated for that
// group alone, so a launch has the registers and LDS of its group -- one kernel holding every class
// would be sized by the largest.  A workgroup is one wave: 64 points of one tile, seeded and
// iterated to the end on their lanes (invert_tile.hpp), so the class dispatch is workgroup-uniform.
// Where many rounds of such waves would wait for their slowest lanes, the group takes the persistent
// kernels of batch_refill.hip (batch_takes_refill).
// Point arrays are addressed through a request table (GnReq): a tile names its request, so one
// launch serves the points of many independent requests (the serving loop) or of one call (a
// one-entry table).
#include <algorithm>
#include <mutex>

#include "invert_tile.hpp"
#include "path_rules.hpp"

namespace gn {

struct BatchTileArgs {
    const GnBatchObj *objs;
    const GnTile *tiles;
    const GnReq *reqs;
    int per_tile;
    int seed;
    gn_invert_opts o;
};

// LDS of a group's wave: the patches of its largest class.
template <int GRP, bool MIXED>
constexpr int group_patch_vecs() {
    return GRP == 0 ? tile_patch_vecs<4, 4, MIXED>()
         : GRP == 1 ? tile_patch_vecs<5, 5, MIXED>() : tile_patch_vecs<6, 6, MIXED>();
}

// Workgroup b takes points (b % per_tile) * 64 .. + 63 of tile b / per_tile.  The tiles are of many
// small nets, so nothing is shared between waves; the bound is one point's chain of iterations, and
// past a few rounds of waves their VALU and patch loads.  Before, a seed launch, persistent FP32 and
// FP64 launches that claimed tiles and refilled stopped lanes: one launch instead of three per
// group, and no drain where a wave's next tile is of another class.  Uneven batches, every group on the
// persistent kernels and on this one, mixed with 6 and 3 steps: 16 surfaces 79,297 points 107 and 69 us, 64
// surfaces 221,393 points 159 and 121, 256 surfaces 1,090,341 points 428 and 365, 1,024 surfaces 4.9 M
// points 1,640 and 1,600; FP64, 20 Gauss-Newton steps, 256 surfaces 1,404 and 1,274.  (The knots in LDS:
// no gain at 55,347 points, 10% slower at 1,090,341, fewer waves.)
template <int GRP, bool MIXED, bool NEWTON32, bool NEWTON64>
__global__ __launch_bounds__(64, 1) void k_batch_tile(BatchTileArgs a) {
    __shared__ float4 patches[group_patch_vecs<GRP, MIXED>()];
    const GnTile tl = a.tiles[blockIdx.x / a.per_tile];
    const int first = (int)(blockIdx.x % a.per_tile) * 64;
    if (first >= tl.count) return;  // workgroup-uniform
    const int cls = a.objs[tl.obj].cls;
    const GnSurfDev d = global_view(a.objs[tl.obj].s);
    const GnReq R = global_view(a.reqs[tl.req]);
    const bool valid = first + (int)threadIdx.x < tl.count;
    const int64_t i = tl.start + first + threadIdx.x;
    double P[3] = {0, 0, 0}, cu = 0, cv = 0;
    if (valid) {
        P[0] = R.x[i];
        P[1] = R.y[i];
        P[2] = R.z[i];
        if (a.seed == 0) {
            cu = R.u[i];
            cv = R.v[i];
        }
    }
    if (a.seed != 0) {
        const GnSearchDev sd = global_view(a.objs[tl.obj].sd);
        const int ll = tile_stage_boxes(sd, a.seed, patches);
        __syncthreads();
        if (valid) tile_seed(sd, a.seed, patches, ll, P, cu, cv);
        __syncthreads();  // every lane has left the boxes
    }
    const Domain dom = domain_of(d);
    int it32 = 0, it64 = 0, st = GN_PT_NONFINITE;
    switch (cls) {  // workgroup-uniform
#define GN_CLS(P_, Q_)                                                                          \
    case (P_ - 2) * 4 + (Q_ - 2):                                                               \
        if constexpr (class_group((P_ - 2) * 4 + (Q_ - 2)) == GRP)                              \
            st = tile_iterate<P_ + 1, Q_ + 1, true, MIXED, NEWTON32, NEWTON64>(                 \
                d, d.ku, d.kv, dom, a.o, P, valid, patches, cu, cv, it32, it64);                \
        break;
        GN_CLS(2, 2) GN_CLS(2, 3) GN_CLS(2, 4) GN_CLS(2, 5)
        GN_CLS(3, 2) GN_CLS(3, 3) GN_CLS(3, 4) GN_CLS(3, 5)
        GN_CLS(4, 2) GN_CLS(4, 3) GN_CLS(4, 4) GN_CLS(4, 5)
        GN_CLS(5, 2) GN_CLS(5, 3) GN_CLS(5, 4) GN_CLS(5, 5)
#undef GN_CLS
        default:
            if constexpr (GRP == 2)
                st = tile_iterate<GN_MAXK, GN_MAXK, false, MIXED, NEWTON32, NEWTON64>(
                    d, d.ku, d.kv, dom, a.o, P, valid, patches, cu, cv, it32, it64);
            break;
    }
    if (!valid) return;
    R.u[i] = cu;
    R.v[i] = cv;
    R.status[i] = (uint8_t)st;
    if (R.it32) R.it32[i] = sat8(it32);
    if (R.it64) R.it64[i] = sat8(it64);
}

template <int GRP, bool MIXED, bool NEWTON32, bool NEWTON64>
static int launch_tiles(BatchTileArgs a, int ntiles, int bpc_cap, hipStream_t st) {
    // blocks_per_cu caps the resident waves (256-lane workgroups, four waves each) by claiming LDS
    const size_t have = 16 * (size_t)group_patch_vecs<GRP, MIXED>(), lds = 160 * 1024;
    const size_t share = bpc_cap > 0 ? lds / (4 * (size_t)bpc_cap) : 0;
    const size_t pad = share > have ? share - have : 0;
    // a grid holds below 2^32 lanes
    const int most = (int)(((size_t)1 << 25) / a.per_tile);
    for (; ntiles > 0; ntiles -= most, a.tiles += most) {
        const unsigned grid = (unsigned)(ntiles < most ? ntiles : most) * (unsigned)a.per_tile;
        k_batch_tile<GRP, MIXED, NEWTON32, NEWTON64><<<grid, 64, pad, st>>>(a);
        GN_HIP(hipGetLastError());
    }
    return GN_OK;
}

template <int GRP>
static int launch_group(const BatchTileArgs &a, int ntiles, int bpc_cap, hipStream_t st) {
    const bool n64 = a.o.newton & GN_NEWTON_FP64, n32 = a.o.newton & GN_NEWTON_FP32;
    auto k = a.o.precision != GN_MIXED ? (n64 ? launch_tiles<GRP, false, false, true>
                                              : launch_tiles<GRP, false, false, false>)
           : n32 ? (n64 ? launch_tiles<GRP, true, true, true> : launch_tiles<GRP, true, true, false>)
                 : (n64 ? launch_tiles<GRP, true, false, true>
                        : launch_tiles<GRP, true, false, false>);
    return k(a, ntiles, bpc_cap, st);
}

int batch_waves(int bpc_cap) {
    auto k = k_batch_tile<0, true, true, true>;
    int w = blocks_per_cu((const void *)k, 64);
    if (bpc_cap > 0 && 4 * bpc_cap < w) w = 4 * bpc_cap;
    return cu_count() * w;
}

int class_tile(size_t points, int waves, int cap) {
    size_t t = points / (2 * (size_t)(waves > 0 ? waves : 1)) / 64 * 64;
    if (t > (size_t)cap) t = (size_t)cap;
    if (t < 64) t = 64;
    return (int)t;
}

std::vector<GroupRange> group_ranges(const GnTile *tiles, size_t ntiles, const std::vector<int> &cls) {
    std::vector<GroupRange> r;
    for (size_t t = 0; t < ntiles; t++) {
        const int g = class_group(cls[tiles[t].obj]);
        if (r.empty() || r.back().grp != g) r.push_back(GroupRange{g, (int)t, (int)t, 0, 0});
        r.back().t1 = (int)t + 1;
        r.back().points += (size_t)tiles[t].count;
        if (tiles[t].count > r.back().max_count) r.back().max_count = tiles[t].count;
    }
    return r;
}

int side_streams_create(SideStreams *ss) {
    for (int k = 0; k < kSideStreams; k++) {
        GN_HIP(hipStreamCreateWithFlags(&ss->s[k], hipStreamNonBlocking));
        GN_HIP(hipEventCreateWithFlags(&ss->join[k], hipEventDisableTiming));
    }
    GN_HIP(hipEventCreateWithFlags(&ss->fork, hipEventDisableTiming));
    return GN_OK;
}

void side_streams_destroy(SideStreams *ss) {
    for (int k = 0; k < kSideStreams; k++) {
        if (ss->s[k]) (void)hipStreamDestroy(ss->s[k]);
        if (ss->join[k]) (void)hipEventDestroy(ss->join[k]);
    }
    if (ss->fork) (void)hipEventDestroy(ss->fork);
    *ss = SideStreams();
}

namespace {
std::mutex g_side_mu;
SideStreams g_side[64];  // per device, created on first use
}  // namespace

static int run_range(const GnBatchObj *objs, const GnTile *tiles, const GroupRange &gr,
                     const GnReq *reqs, const gn_invert_opts &o, int bpc_cap, hipStream_t st,
                     bool several, bool captured = false) {
    const PathOpts limits{o.precision == GN_MIXED, (o.newton & GN_NEWTON_FP64) != 0, o.max_iter,
                          o.fp32_iters, o.fp64_tail};
    const bool refill = !captured && batch_takes_refill(gr.grp, gr.points, several, limits, (size_t)cu_count());
    if (o.seed_mode != GN_SEED_GIVEN && (refill || o.seed_mode == GN_SEED_NEAREST_LEAF)) {
        const int rc = launch_batch_seed(objs, tiles, gr, reqs, o.seed_mode, st);
        if (rc) return rc;
    }
    if (refill) return launch_batch_refill(objs, tiles, gr, reqs, o, bpc_cap, st);
    const int seed = o.seed_mode == GN_SEED_GREEDY_LEAF ? 1 : o.seed_mode == GN_SEED_GREEDY_STEP ? 2
                   : o.seed_mode == GN_SEED_GRID_STEP ? 3 : 0;
    const int ntiles = gr.t1 - gr.t0;
    const BatchTileArgs a{objs, tiles + gr.t0, reqs, (std::max(gr.max_count, 1) + 63) / 64, seed, o};
    return gr.grp == 0 ? launch_group<0>(a, ntiles, bpc_cap, st)
         : gr.grp == 1 ? launch_group<1>(a, ntiles, bpc_cap, st)
                       : launch_group<2>(a, ntiles, bpc_cap, st);
}

static int launch_ranges(const GnBatchObj *objs, const GnTile *tiles,
                         const std::vector<GroupRange> &ranges, const GnReq *reqs,
                         const gn_invert_opts &o, int bpc_cap, hipStream_t st,
                         const SideStreams &ss, const std::function<int(hipStream_t)> &beside,
                         std::vector<std::pair<int, hipEvent_t>> *group_done) {
    if (ranges.size() == 1 && !beside)  // one group, nothing beside it: no fork
        return run_range(objs, tiles, ranges[0], reqs, o, bpc_cap, st, false);
    if (ranges.size() > (size_t)kSideStreams)
        return fail(GN_EDEVICE, "more group ranges than side streams (tiles not sorted by class)");
    GN_HIP(hipEventRecord(ss.fork, st));
    // st joins every side stream that was forked, also when a later launch fails: the caller
    // may then synchronise st alone (or free buffers in its order) before it reuses what the
    // kernels already enqueued still read or write
    int k = 0, rc = GN_OK;
    // the group of the largest patches, whose points take longest, first: on st itself, without the
    // wait for the fork, where nothing else has to run there
    const bool own = !beside && !group_done;
    for (auto it = ranges.rbegin(); it != ranges.rend(); ++it) {
        const GroupRange &gr = *it;
        if (gr.points == 0) continue;
        if (own && it == ranges.rbegin()) {
            rc = run_range(objs, tiles, gr, reqs, o, bpc_cap, st, ranges.size() > 1);
            if (rc) break;
            continue;
        }
        const hipError_t e = hipStreamWaitEvent(ss.s[k], ss.fork, 0);
        if (e != hipSuccess) {
            rc = hip_fail(e, "hipStreamWaitEvent(fork)");
            break;
        }
        rc = run_range(objs, tiles, gr, reqs, o, bpc_cap, ss.s[k], ranges.size() > 1);
        const hipError_t ej = hipEventRecord(ss.join[k], ss.s[k]);
        if (ej != hipSuccess) {
            if (!rc) rc = hip_fail(ej, "hipEventRecord(join)");
            (void)hipStreamSynchronize(ss.s[k]);  // no join event: wait for it here
            break;
        }
        k++;
        if (rc) break;
        if (group_done) group_done->emplace_back(gr.grp, ss.join[k - 1]);
    }
    if (!rc && beside) rc = beside(st);
    for (int j = 0; j < k; j++) {
        const hipError_t e = hipStreamWaitEvent(st, ss.join[j], 0);
        if (e != hipSuccess) {
            (void)hipStreamSynchronize(ss.s[j]);
            if (!rc) rc = hip_fail(e, "hipStreamWaitEvent(join)");
        }
    }
    return rc;
}

int launch_batch_captured(const GnBatchObj *objs, const GnTile *tiles,
                          const std::vector<GroupRange> &ranges, const GnReq *reqs,
                          const gn_invert_opts &o, int bpc_cap, hipStream_t st) {
    for (auto it = ranges.rbegin(); it != ranges.rend(); ++it) {
        if (it->points == 0) continue;
        const int rc = run_range(objs, tiles, *it, reqs, o, bpc_cap, st, false, true);
        if (rc) return rc;
    }
    return GN_OK;
}

static int shared_side_locked(int dev) {
    if (g_side[dev].fork) return GN_OK;
    const int rc = side_streams_create(&g_side[dev]);
    if (rc) side_streams_destroy(&g_side[dev]);
    return rc;
}

int launch_batch_invert(const GnBatchObj *objs, const GnTile *tiles,
                        const std::vector<GroupRange> &ranges, const GnReq *reqs,
                        const gn_invert_opts &o, int bpc_cap, hipStream_t st,
                        const SideStreams *side, const std::function<int(hipStream_t)> &beside,
                        std::vector<std::pair<int, hipEvent_t>> *group_done) {
    if (ranges.empty()) return beside ? beside(st) : GN_OK;
    if (side)
        return launch_ranges(objs, tiles, ranges, reqs, o, bpc_cap, st, *side, beside, group_done);
    int dev = 0;
    GN_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) return fail(GN_EDEVICE, "device index out of range");
    std::lock_guard<std::mutex> lk(g_side_mu);  // one user of the shared set at a time
    const int rc = shared_side_locked(dev);
    if (rc) return rc;
    return launch_ranges(objs, tiles, ranges, reqs, o, bpc_cap, st, g_side[dev], beside, group_done);
}

}  // namespace gn

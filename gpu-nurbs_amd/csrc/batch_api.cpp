// batch_api.cpp -- C ABI of the batched inversion: packing many surfaces into one device
// allocation, the tile list, the tile-shape autotuner and hipGraph capture of a batch launch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <mutex>
#include <sstream>
#include <string>
#include <vector>

#include "gn_internal.hpp"

using gn::fail;

namespace {

// Staging of one batched call: a pinned, coherent host buffer the tile list is written into and the
// device buffer a small kernel copies it to.  In use from the host's write until `ev`, recorded in the
// call's stream after its last kernel.
struct CallBuf {
    char *h = nullptr, *d = nullptr;
    void *h_dev = nullptr;  // h's device-side address
    size_t cap = 0;
    hipEvent_t ev = nullptr;
    hipStream_t st = nullptr;  // the stream of the call in flight
    bool taken = false, pending = false;
    unsigned long long seq = 0;  // order of use
};

// At most kMax staging buffers per batch, kept for its lifetime and handed to one call at a time.
class CallPool {
  public:
    static constexpr size_t kMax = 8;
    // A buffer of at least `bytes` for a call on st.  With all buffers in flight it waits for the oldest
    // call of the same stream; null if there is none (another stream's work may take any time, or wait
    // for this host thread), or if no buffer could be allocated.
    CallBuf *take(size_t bytes, hipStream_t st) {
        CallBuf *best = nullptr;
        {
            std::lock_guard<std::mutex> lk(mu_);
            for (CallBuf *b : all_) {
                if (b->taken) continue;
                if (b->pending) {
                    if (hipEventQuery(b->ev) != hipSuccess) {
                        (void)hipGetLastError();  // not ready is no error to report
                        continue;
                    }
                    b->pending = false;
                }
                if (!best || (b->cap >= bytes && best->cap < bytes)) best = b;
            }
            if ((!best || best->cap < bytes) && all_.size() < kMax) {
                best = new CallBuf();
                if (hipEventCreateWithFlags(&best->ev, hipEventDisableTiming) != hipSuccess) {
                    (void)hipGetLastError();
                    delete best;
                    return nullptr;
                }
                all_.push_back(best);
            }
            if (!best)
                for (CallBuf *b : all_)
                    if (!b->taken && b->st == st && (!best || b->seq < best->seq)) best = b;
            if (!best) return nullptr;
            best->taken = true;
            best->st = st;
            best->seq = ++seq_;
        }
        if (best->pending && hipEventSynchronize(best->ev) != hipSuccess) (void)hipGetLastError();
        best->pending = false;
        if (best->cap < bytes && !grow(best, bytes)) {
            std::lock_guard<std::mutex> lk(mu_);
            best->taken = false;
            return nullptr;
        }
        return best;
    }
    // A first buffer, made with the batch rather than in its first call; calls do without if it fails.
    void reserve(size_t bytes) {
        CallBuf *b = take(bytes, nullptr);
        if (b) b->taken = false;
    }
    // After the call's work has been enqueued on st.
    void give(CallBuf *b, hipStream_t st) {
        const bool rec = hipEventRecord(b->ev, st) == hipSuccess;
        if (!rec) {
            (void)hipGetLastError();
            (void)hipStreamSynchronize(st);
        }
        std::lock_guard<std::mutex> lk(mu_);
        b->pending = rec;
        b->taken = false;
    }
    // Device memory held.
    size_t device_bytes() const {
        std::lock_guard<std::mutex> lk(mu_);
        return bytes_;
    }
    // The device must be idle.
    void clear() {
        for (CallBuf *b : all_) {
            release(b->h, b->d);
            (void)hipEventDestroy(b->ev);
            delete b;
        }
        for (const Outgrown &o : outgrown_) release(o.h, o.d);
        all_.clear();
        outgrown_.clear();
        bytes_ = 0;
    }

  private:
    struct Outgrown {
        char *h, *d;
    };
    static void release(char *h, char *d) {
        if (h) (void)hipHostFree(h);
        if (d) (void)hipFree(d);
    }
    // A free waits for the whole device: what a buffer outgrew stays until the batch is destroyed.  (Sizes
    // double, so that is less than the buffer's own size.)
    bool grow(CallBuf *b, size_t bytes) {
        size_t cap = 1 << 16;
        while (cap < bytes) cap <<= 1;
        CallBuf n;
        if (hipHostMalloc((void **)&n.h, cap, hipHostMallocCoherent) != hipSuccess ||
            hipHostGetDevicePointer(&n.h_dev, n.h, 0) != hipSuccess ||
            hipMalloc((void **)&n.d, cap) != hipSuccess) {
            (void)hipGetLastError();
            release(n.h, n.d);
            return false;
        }
        std::lock_guard<std::mutex> lk(mu_);
        if (b->h) outgrown_.push_back(Outgrown{b->h, b->d});
        bytes_ += cap;
        b->h = n.h;
        b->h_dev = n.h_dev;
        b->d = n.d;
        b->cap = cap;
        return true;
    }
    mutable std::mutex mu_;
    std::vector<CallBuf *> all_;
    std::vector<Outgrown> outgrown_;
    size_t bytes_ = 0;
    unsigned long long seq_ = 0;
};

}  // namespace

struct gn_batch {
    CallPool calls;
    int count = 0;
    std::vector<int> cls;
    GnBatchObj *d_objs = nullptr;
    char *d_pack = nullptr;
    size_t bytes = 0;
    int tile = 1024;  // points per tile
    int bpc = 0;      // workgroups per CU cap (0: occupancy limit)
    bool grids = false;  // every surface brought its seed grid (GN_SEED_GRID_STEP allowed)
};

struct gn_graph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    char *d_buf = nullptr;  // tile list + request table of the captured call
    // the claim-counter slots of persistent launches baked into the graph: its own, so no eager launch is
    // ever given them (each replay leaves them zeroed for the next)
    unsigned long long *d_ctr = nullptr;
};

namespace {

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

int degree_class(int p, int q) {
    if (p >= 2 && p <= 5 && q >= 2 && q <= 5) return (p - 2) * 4 + (q - 2);
    return 16;
}

int check_segments(const gn_batch *b, const gn_segment *segs, int nseg, size_t n) {
    if (nseg < 0 || (nseg > 0 && !segs)) return fail(GN_EINVAL, "bad segment list");
    for (int i = 0; i < nseg; i++) {
        const gn_segment &s = segs[i];
        if (s.obj < 0 || s.obj >= b->count) return fail(GN_EINVAL, "segment object out of range");
        if (s.count < 0 || s.start < 0 || (size_t)s.start + (size_t)s.count > n)
            return fail(GN_EINVAL, "segment outside the point arrays");
    }
    return GN_OK;
}

// Device image of one batched call: the tile list, then (256-byte aligned) a one-entry request table
// holding the call's point arrays.  Tiles are in class order (group, then class, then segment order);
// each group gets its own tile size (at most `tile`), sized for the group's own launch.
constexpr int kKeys = 3 * 32;  // class_order keys
struct CallPlan {
    int64_t tsz[3];
    size_t pos[kKeys];  // first tile of each class
    size_t ntiles = 0, req_off = 0, bytes = 0;
    std::vector<gn::GroupRange> ranges;
};

CallPlan call_plan(const gn_batch *b, const gn_segment *segs, int nseg, int tile, bool captured = false) {
    CallPlan c;
    size_t per[3] = {0, 0, 0}, cnt[kKeys] = {};
    int64_t most[3] = {0, 0, 0};
    for (int i = 0; i < nseg; i++) per[gn::class_group(b->cls[segs[i].obj])] += (size_t)segs[i].count;
    // (a captured call's list goes into kernel arguments: whole tiles keep it short)
    const int waves = captured ? 1 : gn::batch_waves(b->bpc);
    for (int g = 0; g < 3; g++) c.tsz[g] = captured ? std::max(tile, 64) : gn::class_tile(per[g], waves, tile);
    for (int i = 0; i < nseg; i++) {
        const int cls = b->cls[segs[i].obj], g = gn::class_group(cls);
        cnt[gn::class_order(cls)] += (size_t)((segs[i].count + c.tsz[g] - 1) / c.tsz[g]);
        most[g] = std::max(most[g], std::min<int64_t>(segs[i].count, c.tsz[g]));
    }
    for (int k = 0; k < kKeys; k++) {
        c.pos[k] = c.ntiles;
        c.ntiles += cnt[k];
    }
    for (int g = 0; g < 3; g++) {
        const size_t t0 = c.pos[32 * g], t1 = g < 2 ? c.pos[32 * (g + 1)] : c.ntiles;
        if (t1 > t0) c.ranges.push_back(gn::GroupRange{g, (int)t0, (int)t1, per[g], (int)most[g]});
    }
    c.req_off = align256(sizeof(GnTile) * c.ntiles);
    c.bytes = c.req_off + sizeof(GnReq);
    return c;
}

void write_image(const gn_batch *b, const gn_segment *segs, int nseg, const CallPlan &c, const GnReq &r,
                 char *dst) {
    GnTile *t = reinterpret_cast<GnTile *>(dst);
    size_t pos[kKeys];
    std::copy(c.pos, c.pos + kKeys, pos);
    for (int i = 0; i < nseg; i++) {
        const int cls = b->cls[segs[i].obj];
        const int64_t T = c.tsz[gn::class_group(cls)];
        size_t &p = pos[gn::class_order(cls)];
        for (int64_t off = 0; off < segs[i].count; off += T)
            t[p++] = GnTile{segs[i].obj, (int32_t)std::min<int64_t>(T, segs[i].count - off),
                            segs[i].start + off, 0, 0};
    }
    std::memcpy(dst + c.req_off, &r, sizeof(GnReq));
}

void free_image_host(void *p) { delete static_cast<std::vector<char> *>(p); }

// Under stream capture the image travels in the arguments of kernel nodes, which the graph keeps, to a
// buffer that the graph allocates and frees: a replay reads nothing of the host's and nothing that another
// launch may be given (the kernels take no counter slots, and the shared side streams stay out of the
// capture).  A copy node from the call's host image would read freed memory from the second replay on.
int run_captured(gn_batch *b, const gn_segment *segs, int nseg, const GnReq &req, const gn_invert_opts &o,
                 int tile, int bpc, hipStream_t st) {
    const CallPlan c = call_plan(b, segs, nseg, tile, true);
    if (c.ntiles == 0) return GN_OK;
    std::vector<char> img((c.bytes + 15) & ~(size_t)15);
    write_image(b, segs, nseg, c, req, img.data());
    char *d = nullptr;
    GN_HIP(hipMallocAsync((void **)&d, img.size(), st));
    int rc = gn::launch_stage_args(img.data(), d, img.size(), st);
    if (!rc)
        rc = gn::launch_batch_captured(b->d_objs, (const GnTile *)d, c.ranges,
                                       (const GnReq *)(d + c.req_off), o, bpc, st);
    const hipError_t e = hipFreeAsync(d, st);
    if (!rc && e != hipSuccess) rc = gn::hip_fail(e, "hipFreeAsync(tiles)");
    return rc;
}

// The call image is written into pinned staging of the batch's pool and a small kernel carries it to
// the device, so a call neither allocates nor waits.  (A stream-ordered allocation, a copy from
// pageable memory and a host callback that freed it put 0.4 ms of host time and a bubble before the
// first kernel: 256 surfaces and 1.09M points, 897 us for a call on an idle device.)  A call without a
// staging buffer takes that stream-ordered form.
int run_batch(gn_batch *b, const gn_segment *segs, int nseg, const double *x, const double *y,
              const double *z, size_t n, const gn_invert_opts &o, double *u, double *v,
              uint8_t *status, uint8_t *it32, uint8_t *it64, int tile, int bpc, hipStream_t st) {
    (void)n;
    const GnReq req{x, y, z, u, v, status, it32, it64};
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) != hipSuccess) (void)hipGetLastError();  // (the null stream, beside a capture)
    if (cs != hipStreamCaptureStatusNone) return run_captured(b, segs, nseg, req, o, tile, bpc, st);
    const CallPlan c = call_plan(b, segs, nseg, tile);
    if (c.ntiles == 0) return GN_OK;
    CallBuf *buf = b->calls.take(c.bytes + 16, st);
    if (buf) {
        write_image(b, segs, nseg, c, req, buf->h);
        int rc = gn::launch_stage_copy(buf->h_dev, buf->d, c.bytes, st);
        if (!rc)
            rc = gn::launch_batch_invert(b->d_objs, (const GnTile *)buf->d, c.ranges,
                                         (const GnReq *)(buf->d + c.req_off), o, bpc, st);
        b->calls.give(buf, st);
        return rc;
    }
    // the host copy is released by a host callback in stream order, after the upload has consumed it
    auto *img = new std::vector<char>(c.bytes);
    write_image(b, segs, nseg, c, req, img->data());
    char *d = nullptr;
    hipError_t e = hipMallocAsync((void **)&d, c.bytes, st);
    if (e != hipSuccess) {
        delete img;
        return gn::hip_fail(e, "hipMallocAsync(tiles)");
    }
    e = hipMemcpyAsync(d, img->data(), c.bytes, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hipLaunchHostFunc(st, free_image_host, img);
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(st);
        delete img;
        (void)hipFreeAsync(d, st);
        return gn::hip_fail(e, "tile upload");
    }
    int rc = gn::launch_batch_invert(b->d_objs, (const GnTile *)d, c.ranges,
                                     (const GnReq *)(d + c.req_off), o, bpc, st);
    GN_HIP(hipFreeAsync(d, st));
    return rc;
}

int check_opts(const gn_batch *b, const gn_invert_opts &o) {
    if (o.precision != GN_FP64 && o.precision != GN_MIXED)
        return fail(GN_EINVAL, "precision must be GN_FP64 or GN_MIXED");
    if (o.seed_mode == GN_SEED_REF_FIRST_HIT)
        return fail(GN_EINVAL, "first-hit seeding is a single-surface reference mode");
    if (o.seed_mode == GN_SEED_GLOBAL)
        return fail(GN_EINVAL, "the global projection is a single-surface mode");
    if (o.seed_mode == GN_SEED_GRID_STEP && !b->grids)
        return fail(GN_ESTATE, "grid seeds need every surface's seed grid (gn_build_seed_grid) "
                               "built before gn_batch_create");
    if (o.seed_mode < GN_SEED_NEAREST_LEAF || o.seed_mode > GN_SEED_GRID_STEP)
        return fail(GN_EINVAL, "bad seed_mode");
    if (o.max_iter < 0 || o.fp32_iters < 0 || o.fp64_tail < 0 || o.max_iter > 10000 ||
        o.fp32_iters > 10000 || o.fp64_tail > 10000)
        return fail(GN_EINVAL, "iteration counts must be 0..10000");
    return GN_OK;
}

std::string signature(const gn_batch *b, const gn_segment *segs, int nseg, size_t n) {
    std::vector<double> per(17, 0.0);
    for (int i = 0; i < nseg; i++) per[b->cls[segs[i].obj]] += (double)segs[i].count;
    std::ostringstream os;
    os << "objs=" << b->count << ",n2=" << (n ? (int)std::log2((double)n) : 0);
    for (int c = 0; c < 17; c++) os << "," << (per[c] > 0 ? (int)std::log2(per[c]) : -1);
    return os.str();
}

}  // namespace

namespace gn {
// Read-only view of a batch for the inversion server.
int batch_view(const gn_batch *b, const GnBatchObj **objs, int *count, std::vector<int> *cls,
               int *tile, int *bpc, size_t *bytes, bool *grids) {
    if (!b) return fail(GN_EINVAL, "null batch");
    *grids = b->grids;
    *objs = b->d_objs;
    *count = b->count;
    *cls = b->cls;
    *tile = b->tile;
    *bpc = b->bpc;
    *bytes = b->bytes + b->calls.device_bytes();
    return GN_OK;
}
}  // namespace gn

extern "C" {

int gn_batch_create(gn_surface *const *surfaces, int count, gn_stream stream, gn_batch **out) {
    if (!out) return fail(GN_EINVAL, "out is null");
    *out = nullptr;
    if (count <= 0 || !surfaces) return fail(GN_EINVAL, "empty surface list");
    hipStream_t st = (hipStream_t)stream;
    // layout of the pack
    struct Part {
        const void *src;
        size_t bytes;
        size_t off;
    };
    std::vector<std::vector<Part>> parts(count);
    size_t total = 0;
    for (int i = 0; i < count; i++) {
        const gn_surface *s = surfaces[i];
        if (!s) return fail(GN_EINVAL, "null surface in the list");
        if (!s->tree_levels) return fail(GN_ESTATE, "every surface needs its tree (gn_build_tree)");
        const int D = 3 * (s->tree_levels - 1);
        const size_t qnodes = (((size_t)1 << (2 * (D + 1))) - 1) / 3, leaves = (size_t)1 << (2 * D);
        const Part ps[] = {
            {s->d_ku, sizeof(double) * s->ku.size(), 0},
            {s->d_kv, sizeof(double) * s->kv.size(), 0},
            {s->d_ihu, sizeof(double) * (s->nu - s->p), 0},
            {s->d_ihv, sizeof(double) * (s->nv - s->q), 0},
            {s->d_tab64, sizeof(double) * s->tab_entries, 0},
            {s->d_tab32, sizeof(float) * s->tab_entries, 0},
            {s->d_sbox32, sizeof(float) * qnodes * 6, 0},
            {s->d_scentre, sizeof(double) * leaves * 3, 0},
            {s->d_sseed, sizeof(double) * leaves * 2, 0},
            {s->d_sref, sizeof(int32_t) * leaves, 0},
            {s->d_sleaf32, sizeof(float4) * leaves, 0},
            {s->d_srec, sizeof(float4) * leaves * kRecVec, 0},
            {s->d_grid, s->grid_bytes, 0},  // none (0 bytes) without a seed grid
        };
        for (Part p : ps) {
            p.off = total;
            total += align256(p.bytes);
            parts[i].push_back(p);
        }
    }
    gn_batch *b = new gn_batch();
    b->count = count;
    b->cls.resize(count);
    b->grids = true;
    for (int i = 0; i < count; i++) b->grids = b->grids && surfaces[i]->d_grid != nullptr;
    hipError_t e = hipMalloc((void **)&b->d_pack, total);
    if (e != hipSuccess) {
        delete b;
        return gn::hip_fail(e, "hipMalloc(batch pack)");
    }
    e = hipMalloc((void **)&b->d_objs, sizeof(GnBatchObj) * count);
    if (e != hipSuccess) {
        (void)hipFree(b->d_pack);
        delete b;
        return gn::hip_fail(e, "hipMalloc(batch objects)");
    }
    b->bytes = total + sizeof(GnBatchObj) * count;
    std::vector<GnBatchObj> objs(count);
    for (int i = 0; i < count && e == hipSuccess; i++) {
        const gn_surface *s = surfaces[i];
        for (const Part &p : parts[i])
            if (e == hipSuccess && p.bytes)
                e = hipMemcpyAsync(b->d_pack + p.off, p.src, p.bytes, hipMemcpyDeviceToDevice, st);
        char *base = b->d_pack;
        GnBatchObj &ob = objs[i];
        ob.s = s->dev();
        ob.s.ku = (const double *)(base + parts[i][0].off);
        ob.s.kv = (const double *)(base + parts[i][1].off);
        ob.s.ihu = (const double *)(base + parts[i][2].off);
        ob.s.ihv = (const double *)(base + parts[i][3].off);
        ob.s.tab64 = (const double *)(base + parts[i][4].off);
        ob.s.tab32 = (const float *)(base + parts[i][5].off);
        ob.sd = s->search();
        ob.sd.box = nullptr;
        ob.sd.box32 = (const float *)(base + parts[i][6].off);
        ob.sd.centre = (const double *)(base + parts[i][7].off);
        ob.sd.seed_uv = (const double *)(base + parts[i][8].off);
        ob.sd.ref_index = (const int32_t *)(base + parts[i][9].off);
        ob.sd.leaf32 = (const float4 *)(base + parts[i][10].off);
        ob.sd.rec = (const float4 *)(base + parts[i][11].off);
        ob.sd.cone32 = nullptr;  // normal cones serve the global projection only
        ob.sd.grid = s->d_grid ? (const void *)(base + parts[i][12].off) : nullptr;
        ob.cls = degree_class(s->p, s->q);
        ob.pad_ = 0;
        b->cls[i] = ob.cls;
    }
    if (e == hipSuccess)
        e = hipMemcpyAsync(b->d_objs, objs.data(), sizeof(GnBatchObj) * count,
                           hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) {
        (void)hipFree(b->d_pack);
        (void)hipFree(b->d_objs);
        delete b;
        return gn::hip_fail(e, "batch packing copies");
    }
    b->calls.reserve((size_t)1 << 18);  // about 10,000 tiles
    *out = b;
    return GN_OK;
}

int gn_batch_destroy(gn_batch *b) {
    if (!b) return GN_OK;
    (void)hipDeviceSynchronize();
    b->calls.clear();
    (void)hipFree(b->d_pack);
    (void)hipFree(b->d_objs);
    delete b;
    return GN_OK;
}

size_t gn_batch_device_bytes(const gn_batch *b) {
    return b ? b->bytes + b->calls.device_bytes() : 0;
}

int gn_batch_set_shape(gn_batch *b, int tile_points, int blocks_per_cu) {
    if (!b) return fail(GN_EINVAL, "null batch");
    if (tile_points < 1 || tile_points > (1 << 24) || blocks_per_cu < 0 || blocks_per_cu > 64)
        return fail(GN_EINVAL, "tile_points 1..2^24, blocks_per_cu 0..64");
    b->tile = tile_points;
    b->bpc = blocks_per_cu;
    return GN_OK;
}

int gn_batch_get_shape(const gn_batch *b, int *tile_points, int *blocks_per_cu) {
    if (!b) return fail(GN_EINVAL, "null batch");
    if (tile_points) *tile_points = b->tile;
    if (blocks_per_cu) *blocks_per_cu = b->bpc;
    return GN_OK;
}

int gn_batch_invert(gn_batch *b, const gn_segment *segs, int nseg, const double *x,
                    const double *y, const double *z, size_t n, const gn_invert_opts *opts,
                    double *u, double *v, uint8_t *status, gn_stream stream) {
    if (!b) return fail(GN_EINVAL, "null batch");
    gn_invert_opts o;
    if (opts) o = *opts;
    else gn_invert_opts_default(&o);
    int rc = check_opts(b, o);
    if (rc) return rc;
    if ((rc = check_segments(b, segs, nseg, n))) return rc;
    if (n && (!x || !y || !z || !u || !v || !status)) return fail(GN_EINVAL, "null buffer");
    return run_batch(b, segs, nseg, x, y, z, n, o, u, v, status, nullptr, nullptr, b->tile, b->bpc,
                     (hipStream_t)stream);
}

int gn_batch_tune(gn_batch *b, const gn_segment *segs, int nseg, const double *x, const double *y,
                  const double *z, size_t n, const gn_invert_opts *opts, double *u, double *v,
                  uint8_t *status, const char *cache_path, gn_stream stream) {
    if (!b) return fail(GN_EINVAL, "null batch");
    gn_invert_opts o;
    if (opts) o = *opts;
    else gn_invert_opts_default(&o);
    int rc = check_opts(b, o);
    if (rc) return rc;
    if ((rc = check_segments(b, segs, nseg, n))) return rc;
    if (n && (!x || !y || !z || !u || !v || !status)) return fail(GN_EINVAL, "null buffer");
    const std::string sig = signature(b, segs, nseg, n);
    if (cache_path) {  // cached shape for this signature?
        std::ifstream in(cache_path);
        std::string line;
        while (std::getline(in, line)) {
            std::istringstream ls(line);
            std::string s;
            int t, c;
            if (ls >> s >> t >> c && s == sig && t > 0 && c >= 0) {
                b->tile = t;
                b->bpc = c;
                return GN_OK;
            }
        }
    }
    hipStream_t st = (hipStream_t)stream;
    // given seeds live in u and v, which every run overwrites: keep a copy and put it back
    // before each run (outside the timed region)
    double *seeds = nullptr;
    const bool given = o.seed_mode == GN_SEED_GIVEN && n > 0;
    if (given) {
        GN_HIP(hipMallocAsync((void **)&seeds, sizeof(double) * 2 * n, st));
        GN_HIP(hipMemcpyAsync(seeds, u, sizeof(double) * n, hipMemcpyDeviceToDevice, st));
        GN_HIP(hipMemcpyAsync(seeds + n, v, sizeof(double) * n, hipMemcpyDeviceToDevice, st));
    }
    hipEvent_t e0, e1;
    GN_HIP(hipEventCreate(&e0));
    GN_HIP(hipEventCreate(&e1));
    const int tiles[] = {128, 256, 512, 1024, 4096};
    const int caps[] = {0, 1};
    float best = 1e30f;
    int bt = b->tile, bc = b->bpc;
    for (int t : tiles) {
        for (int c : caps) {
            float sum = 0;
            for (int r = 0; r < 3 && !rc; r++) {  // first run warms up, not counted
                if (given) {
                    GN_HIP(hipMemcpyAsync(u, seeds, sizeof(double) * n, hipMemcpyDeviceToDevice, st));
                    GN_HIP(hipMemcpyAsync(v, seeds + n, sizeof(double) * n, hipMemcpyDeviceToDevice, st));
                }
                GN_HIP(hipEventRecord(e0, st));
                rc = run_batch(b, segs, nseg, x, y, z, n, o, u, v, status, nullptr, nullptr, t, c, st);
                GN_HIP(hipEventRecord(e1, st));
                GN_HIP(hipEventSynchronize(e1));
                float ms = 0;
                GN_HIP(hipEventElapsedTime(&ms, e0, e1));
                if (r) sum += ms;
            }
            if (rc) break;
            if (sum > 0 && sum < best) {
                best = sum;
                bt = t;
                bc = c;
            }
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (given) GN_HIP(hipFreeAsync(seeds, st));
    if (rc) return rc;
    b->tile = bt;
    b->bpc = bc;
    if (cache_path) {
        std::ofstream outf(cache_path, std::ios::app);
        outf << sig << " " << bt << " " << bc << "\n";
    }
    return GN_OK;
}

int gn_batch_graph_create(gn_batch *b, const gn_segment *segs, int nseg, const double *x,
                          const double *y, const double *z, size_t n, const gn_invert_opts *opts,
                          double *u, double *v, uint8_t *status, gn_stream stream,
                          gn_graph **out) {
    if (!b || !out) return fail(GN_EINVAL, "null argument");
    *out = nullptr;
    if (!stream) return fail(GN_EINVAL, "graph capture needs a created (non-null) stream");
    gn_invert_opts o;
    if (opts) o = *opts;
    else gn_invert_opts_default(&o);
    int rc = check_opts(b, o);
    if (rc) return rc;
    if ((rc = check_segments(b, segs, nseg, n))) return rc;
    if (n && (!x || !y || !z || !u || !v || !status)) return fail(GN_EINVAL, "null buffer");
    if ((rc = gn::ensure_runtime())) return rc;
    const GnReq req{x, y, z, u, v, status, nullptr, nullptr};
    const CallPlan plan = call_plan(b, segs, nseg, b->tile);
    std::vector<char> img(plan.bytes);
    write_image(b, segs, nseg, plan, req, img.data());
    gn_graph *g = new gn_graph();
    hipStream_t st = (hipStream_t)stream;
    // a slot per persistent launch: at most one per class group and precision phase
    gn::SlotPool pool;
    pool.nslots = (int)plan.ranges.size() * (o.precision == GN_MIXED ? 2 : 1);
    const size_t ctr_bytes = sizeof(unsigned long long) * gn::slot_words() * (pool.nslots ? pool.nslots : 1);
    hipError_t e = hipMalloc((void **)&g->d_buf, img.size());
    if (e == hipSuccess)
        e = hipMemcpy(g->d_buf, img.data(), img.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMalloc((void **)&g->d_ctr, ctr_bytes);
    if (e == hipSuccess) e = hipMemset(g->d_ctr, 0, ctr_bytes);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e != hipSuccess) {
        (void)hipFree(g->d_buf);
        (void)hipFree(g->d_ctr);
        delete g;
        return gn::hip_fail(e, "graph tile list / counter slots");
    }
    pool.ctr = g->d_ctr;
    // side streams of its own: they stay in the capture until it ends, and a call of another thread that
    // was given the shared ones meanwhile would fail
    gn::SideStreams side;
    if ((rc = gn::side_streams_create(&side))) {
        gn::side_streams_destroy(&side);
        (void)hipFree(g->d_buf);
        (void)hipFree(g->d_ctr);
        delete g;
        return rc;
    }
    e = hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) {
        gn::side_streams_destroy(&side);
        (void)hipFree(g->d_buf);
        (void)hipFree(g->d_ctr);
        delete g;
        return gn::hip_fail(e, "hipStreamBeginCapture");
    }
    {
        gn::PoolScope scope(&pool);
        rc = gn::launch_batch_invert(b->d_objs, (const GnTile *)g->d_buf, plan.ranges,
                                     (const GnReq *)(g->d_buf + plan.req_off), o, b->bpc, st, &side);
    }
    e = hipStreamEndCapture(st, &g->graph);
    gn::side_streams_destroy(&side);
    if (!rc && e == hipSuccess) e = hipGraphInstantiate(&g->exec, g->graph, nullptr, nullptr, 0);
    if (rc || e != hipSuccess) {
        if (g->graph) (void)hipGraphDestroy(g->graph);
        (void)hipFree(g->d_buf);
        (void)hipFree(g->d_ctr);
        delete g;
        return rc ? rc : gn::hip_fail(e, "graph capture / instantiate");
    }
    *out = g;
    return GN_OK;
}

int gn_graph_launch(gn_graph *g, gn_stream stream) {
    if (!g) return fail(GN_EINVAL, "null graph");
    GN_HIP(hipGraphLaunch(g->exec, (hipStream_t)stream));
    return GN_OK;
}

int gn_graph_destroy(gn_graph *g) {
    if (!g) return GN_OK;
    (void)hipDeviceSynchronize();
    if (g->exec) (void)hipGraphExecDestroy(g->exec);
    if (g->graph) (void)hipGraphDestroy(g->graph);
    (void)hipFree(g->d_buf);
    (void)hipFree(g->d_ctr);
    delete g;
    return GN_OK;
}

}  // extern "C"

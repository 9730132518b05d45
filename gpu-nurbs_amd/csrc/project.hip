// project.hip -- global projection (GN_SEED_GLOBAL): the nearest point of the surface to each
// query, not just the local minimum that Newton reaches from one seed.  The reference's version
// (normal-cone culling, src/kernel/kernel.cu:471-513, 623-704) is unfinished: its test tries the
// box corners only, for one sign of the normal.  This one is a branch and bound over the seed
// quadtree whose leaf boxes contain their pieces of surface:
//   1. bound: the greedy seed leaf (descent + 3 x 3), then projected Newton over the whole domain
//      (any start gives a valid bound; the exact nearest leaf centre cost a second tree walk);
//   2. every leaf whose FP32 box (a conservative lower bound) is not farther than the best foot
//      point so far, and whose normal cone allows a foot point inside it (cone_may_hold; leaves
//      on the domain boundary, where the nearest point need not be a foot point, always pass),
//      gets a projected Newton solve clamped to its uv cell, from the leaf's stepped seed; a nearer
//      result tightens the bound, which prunes the rest of the depth-first walk;
//   3. the nearest foot point is polished by projected Newton over the whole domain (kept unless it
//      is farther by more than rounding, 1e-9 relative in squared distance).
// The minimum is found whenever the solve inside the leaf that holds it reaches it: leaves of the
// depth-3 tree (64 x 64 cells) are nearly flat, so the distance restricted to one is close to
// convex.  Projected Newton (gn_step with ACTIVE) holds a coordinate on its bound while the
// descent points outward, so minima on cell edges and on the surface boundary are reached too.
// FP64, exact-Hessian steps.  Also the fallback of gn_invert (opts.fallback):
// the queries an inversion left unconverged are listed and solved again this way.
#include "gn_search.hpp"
#include "invert_common.hpp"

namespace gn {

constexpr int kLeafIter = 8;  // projected Newton steps inside one leaf cell

// Whether a leaf can hold an interior foot point of P: a point X of its box b with P - X parallel
// to a normal n of its cone (unit axis a, half-angle theta < 90 degrees), i.e. whether the box meets
// the double cone {X : ((X - P) . a)^2 >= cos^2(theta) |X - P|^2} with apex P.  The angle between
// X - P and the line of a has, over a box that the line misses, its minimum on an edge (inside the
// box or a face it could only have one where the line meets it), so the test is: P in the box, or
// the line P + t a meets the box, or some edge has a point with q(s) >= 0, q being that quadratic
// along the edge.  Exact up to rounding; FP64 on the FP32 box's bounds, with the half-angle widened
// by another 2e-6 rad.
// c2: cos^2 of the widened half-angle, stored with the leaf's record at build time.
__device__ __forceinline__ bool cone_may_hold(const float4 cn, double c2, const float (&b)[6],
                                              const double P[3]) {
    if (!(cn.w < 1.5f)) return true;  // no bounded cone
    const double a[3] = {cn.x, cn.y, cn.z};
    const double lo[3] = {b[0], b[1], b[2]}, hi[3] = {b[3], b[4], b[5]};
    if (!(P[0] == P[0] && P[1] == P[1] && P[2] == P[2])) return true;
    // the line P + t a against the slabs
    double t0 = -INFINITY, t1 = INFINITY;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        if (a[k] != 0.0) {
            const double r = 1.0 / a[k];
            const double ta = (lo[k] - P[k]) * r, tb = (hi[k] - P[k]) * r;
            t0 = fmax(t0, fmin(ta, tb));
            t1 = fmin(t1, fmax(ta, tb));
        } else if (P[k] < lo[k] || P[k] > hi[k]) {
            t0 = INFINITY;  // parallel to this slab and outside it
        }
    }
    if (t0 <= t1) return true;  // also P inside the box (t = 0)
    // the 12 edges: along axis k, the other two coordinates at their bounds
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int k1 = k == 0 ? 1 : 0, k2 = k == 2 ? 1 : 2;
        const double d[3] = {k == 0 ? hi[0] - lo[0] : 0.0, k == 1 ? hi[1] - lo[1] : 0.0,
                             k == 2 ? hi[2] - lo[2] : 0.0};
        const double be = d[k] * a[k], ee = d[k] * d[k];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            double w[3];
            w[k] = lo[k] - P[k];
            w[k1] = ((e & 1) ? hi[k1] : lo[k1]) - P[k1];
            w[k2] = ((e & 2) ? hi[k2] : lo[k2]) - P[k2];
            const double al = w[0] * a[0] + w[1] * a[1] + w[2] * a[2];
            const double ga = w[0] * w[0] + w[1] * w[1] + w[2] * w[2];
            const double de = w[k] * d[k];
            // q(s) = A s^2 + 2 B s + C on s in [0, 1]
            const double A = be * be - c2 * ee, B = al * be - c2 * de, C = al * al - c2 * ga;
            if (C >= 0.0 || A + 2.0 * B + C >= 0.0) return true;
            if (A < 0.0 && B > 0.0 && B < -A && C - B * B / A >= 0.0) return true;  // vertex -B/A
        }
    }
    return false;
}

// Projected Newton with backtracking, one evaluation per call: a step after which the squared
// distance grew by more than 1e-6 relative is halved, up to kHalvings times in a row, before a new
// step is taken.  (Near a minimum the squared distance carries rounding of the surface point
// relative to the residual, ~1e-12 of it at a 1e-3 offset; smaller growth is not a failed step.)  Once
// the steps are over (`left` used up, or a final status) one more evaluation gives the distance of the
// last iterate, and the nearer of it and the last accepted point is the solve's result.
constexpr int kHalvings = 8;
struct Solve {
    double cu, cv;        // the iterate
    double pu, pv, prr;   // the last accepted point and its squared distance
    int left, back, st;   // steps left; halvings in a row; status (kStepContinue while stepping)
    __device__ __forceinline__ void start(double u, double v, int iters) {
        cu = pu = u;
        cv = pv = v;
        prr = INFINITY;
        left = iters;
        back = 0;
        st = kStepContinue;
    }
    // o: the surface at (cu, cv).  True when the solve is over: (cu, cv), d2 and st are its result.
    __device__ __forceinline__ bool advance(const GnSurfDev &d, const Cart<double> &o, const double *P,
                                            const Domain &dom, double tol_step, const SpanCache &sc,
                                            double &d2) {
        if (left > 0 && st == kStepContinue) {
            left--;
            const double su = cu, sv = cv;
            double rr = INFINITY;
            const int s = gn_update<double, true, true>(d, o, P[0], P[1], P[2], cu, cv, 0.0, tol_step,
                                                        0.0, 1, dom, sc, &rr);
            if (!(rr <= prr * (1.0 + 1e-6)) && back < kHalvings) {  // grew, beyond rounding
                cu = pu + 0.5 * (su - pu);
                cv = pv + 0.5 * (sv - pv);
                back++;
            } else {
                back = 0;
                pu = su;
                pv = sv;
                prr = rr;
                st = s;
            }
            return false;
        }
        const double dx = o.S[0] - P[0], dy = o.S[1] - P[1], dz = o.S[2] - P[2];
        d2 = fma(dz, dz, fma(dy, dy, dx * dx));
        if (!(d2 <= prr)) {  // the final step did not help: keep the last accepted point
            cu = pu;
            cv = pv;
            d2 = prr;
        }
        if (st == kStepContinue) st = GN_PT_MAXITER;
        return true;
    }
};

// Two waves per SIMD are forced where the spills that costs stay small: patches of up to 20
// entries and the generic kernel.  Larger exact patches run one wave with AGPRs as spill room.
template <int K1, int K2, bool EXACT>
constexpr int project_waves() { return (!EXACT || K1 * K2 <= 20) ? 2 : 1; }

// Levels of the seed quadtree whose FP32 boxes a workgroup stages in LDS: levels 1..4 are 340
// boxes, 8 KB.
constexpr int kProjLdsLevels = 4;

// The largest float not above x: a float is <= x exactly when it is <= floor32(x).
__device__ __forceinline__ float floor32(double x) { return __double2float_rd(x); }

// N consecutive boxes (6 floats each): the mask of those not farther than best32.
template <int N, typename PTR>
__device__ __forceinline__ uint32_t box_mask(PTR boxes, const float p[3], float best32) {
    uint32_t m = 0;
#pragma unroll
    for (int k = 0; k < N; k++) {
        float b[6];
        __builtin_memcpy(b, boxes + 6 * k, sizeof(b));
        if (box_d2(b, p) <= best32) m |= 1u << k;
    }
    return m;
}

// The branch and bound over a wave's chunk of up to kProjQ consecutive queries (grid-stride), its state
// in LDS.  The wave alternates between two kinds of phases:
//   - lane per query: the queries' starts; walks of the tree (Morton order, so the same leaves in the
//     same order as a walk that solved each leaf on arrival) that collect the next leaves to solve into
//     a pool of kProjItems; the choice among solved leaves; the results;
//   - lane per solve: the bound solves, the pool's leaf solves, the polishes.  Lanes take the next
//     solve of the phase as they finish, and a query's leaves are solved by several lanes at once.
// A collected leaf counts only if its box is not farther than the best point so far when its turn
// comes in the query's order; a leaf whose box is farther cannot hold a nearer point, so solving it
// ahead of its turn changes no result.
// What bounds the kernel is FP64 evaluation (one step of up to 64 solves: 2.9 us per wave at two waves
// per SIMD; over the whole kernel 26 of 64 lanes are active per VALU instruction) and then the walks, about a
// fifth; for small calls the longest
// chain of solves.  One query per lane, its solves gathered into rounds with the other lanes', kept 19%
// of the lanes active: 262,144 queries on a bicubic 32 x 32 net took 1194 us and now take 501, 1,000
// queries 463 and 133 us.  One wave per SIMD without spills (273 registers): 696 us.
// LIST: the fallback over list[0 .. *count): the (u, v) already in place is kept when it is nearer, and
// the counts are left alone.  Otherwise it32 receives the number of leaves solved.  chunk: queries per
// wave; for a list, whose length the host doesn't know, project_chunk of that length.
constexpr int kProjQ = 128, kProjItems = 224, kProjPer = 6;
struct ProjWave {
    double P[3][kProjQ];
    double best[kProjQ], bu[kProjQ], bv[kProjQ];
    // per tree level, 4 bits: passing children not yet visited; at level depth - 2, 16 bits: leaves
    unsigned long long stack[kProjQ];
    uint32_t c0[kProjQ], path[kProjQ];
    uint16_t solved[kProjQ];
    uint8_t level[kProjQ], bst[kProjQ];
    uint8_t first[kProjQ], taken[kProjQ];  // the query's places in the pool
    // the pool: query, leaf, box distance; start, then result
    union {
        struct {
            double iu[kProjItems], iv[kProjItems], id2[kProjItems];
        };
        struct {  // while the pool is filled: the leaves the walks found, and which may hold a foot point
            uint32_t found[kProjQ][kProjPer];
            uint16_t cand[kProjQ * kProjPer];
            uint32_t holds[kProjQ];
        };
    };
    uint32_t ileaf[kProjItems];
    float ilb[kProjItems];
    uint8_t iq[kProjItems], ist[kProjItems];
};
static_assert(kProjItems <= 256 && kProjPer <= 8, "pool places and leaf counts are bytes");
enum { kProjBound = 0, kProjLeaves = 1, kProjPolish = 2 };

__device__ __forceinline__ void wave_lds_order() {  // LDS accesses before stay before, across lanes
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Queries per wave chunk: a full pool's worth (kProjQ) once that still gives every resident wave (two
// per SIMD) a chunk, fewer for smaller calls, whose time is the longest chain of solves in a wave.
__host__ __device__ inline int project_chunk(size_t n, unsigned cus) {
    const size_t c = (n / (8 * (size_t)cus) + 15) / 16 * 16;
    return (int)(c < 16 ? 16 : c > (size_t)kProjQ ? (size_t)kProjQ : c);
}

template <int K1, int K2, bool EXACT, bool LIST>
__global__ __launch_bounds__(256, (project_waves<K1, K2, EXACT>())) void k_project(
    GnSurfDev d_in, GnSearchDev sd, InvArgs a, const uint32_t *__restrict__ order,
    const uint32_t *__restrict__ count, int chunk, unsigned cus) {
    const size_t n = LIST ? (size_t)*count : a.n;
    if constexpr (LIST) {
        chunk = project_chunk(n, cus);
        if ((size_t)blockIdx.x * 4 * (size_t)chunk >= n) return;  // before anything is staged
    }
    extern __shared__ double sk[];  // EXACT: knots and reciprocal span lengths
    __shared__ __align__(16) float lbox[(((1 << (2 * (kProjLdsLevels + 1))) - 1) / 3 - 1) * 6];
    __shared__ ProjWave waves[4];
    const int D = sd.depth, ll = D < kProjLdsLevels ? D : kProjLdsLevels;
    {
        const int nf2 = (int)(qoff(ll + 1) - 1) * 3;
        const float2 *src = reinterpret_cast<const float2 *>(sd.box32 + 6);
        float2 *dst = reinterpret_cast<float2 *>(lbox);
        for (int i = threadIdx.x; i < nf2; i += blockDim.x) dst[i] = src[i];
    }
    GnSurfDev d = d_in;
    const double *ku = d_in.ku, *kv = d_in.kv;
    if constexpr (EXACT) {  // (also waits for the boxes)
        d = stage_knots_lds(d_in, sk);
        ku = sk;
        kv = sk + d.nu + d.p + 1;
    } else {
        __syncthreads();
    }
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    ProjWave &w = waves[wv];
    const unsigned long long lt = (1ull << lane) - 1ull;
    const Domain full{ku[d.p], ku[d.nu], kv[d.q], kv[d.nv]};
    const uint32_t side = 1u << D;
    // leaf cells: the unit square's 2^D x 2^D cells mapped onto the knot domain, exactly as the
    // tree lays out its nodes' uv rectangles
    const double cell = 1.0 / (double)side;
    const double wu = full.u1 - full.u0, wvv = full.v1 - full.v0;
    auto leaf_cell = [&](uint32_t c) __attribute__((always_inline)) {
        const uint32_t ix = compact2(c >> 1), iy = compact2(c);
        return Domain{full.u0 + wu * (ix * cell), full.u0 + wu * ((ix + 1) * cell),
                      full.v0 + wvv * (iy * cell), full.v0 + wvv * ((iy + 1) * cell)};
    };
    const int max_iter = a.o.max_iter;
    const double tol_step = a.o.tol_step;
    for (size_t q0 = ((size_t)blockIdx.x * 4 + wv) * (size_t)chunk; q0 < n;
         q0 += (size_t)gridDim.x * 4 * (size_t)chunk) {  // wave-uniform
        const int nq = (int)(n - q0 < (size_t)chunk ? n - q0 : (size_t)chunk);
        // starts: the greedy leaf's stepped seed (step_seed: one Gauss-Newton step and two on the
        // leaf's quadratic model), a few Newton iterations nearer than its centre
        for (int q = lane; q < nq; q += 64) {
            const size_t i = LIST || order ? (size_t)order[q0 + q] : q0 + q;
            const double P[3] = {a.x[i], a.y[i], a.z[i]};
            float4 cq;
            const uint32_t c0 = greedy_leaf(sd, P, lbox, ll, &cq);
            double bu, bv;
            step_seed(sd, c0, cq, P, bu, bv);
            w.P[0][q] = P[0];
            w.P[1][q] = P[1];
            w.P[2][q] = P[2];
            w.bu[q] = bu;
            w.bv[q] = bv;
            w.c0[q] = c0;
            w.solved[q] = 1;
        }
        int phase = kProjBound, items = nq;  // wave-uniform
        while (true) {
            // ---- a lane per solve
            wave_lds_order();
            {
                int next = 0, it = 0;
                bool act = false;
                Solve sv;
                sv.start(full.u0, full.v0, 0);
                SpanCache sc;
                Domain dom = full;
                double P[3] = {0, 0, 0};
                while (true) {
                    const unsigned long long idle = __ballot(!act);
                    if (idle && next < items) {
                        const int rank = __popcll(idle & lt);
                        if (!act && rank < items - next) {
                            it = next + rank;
                            int q = it;
                            double su, s_v;
                            if (phase == kProjLeaves) {
                                q = w.iq[it];
                                su = w.iu[it];
                                s_v = w.iv[it];
                                dom = leaf_cell(w.ileaf[it]);
                            } else {
                                su = w.bu[it];
                                s_v = w.bv[it];
                                dom = full;
                            }
                            P[0] = w.P[0][q];
                            P[1] = w.P[1][q];
                            P[2] = w.P[2][q];
                            sv.start(su, s_v, phase == kProjLeaves ? kLeafIter : max_iter);
                            act = true;
                        }
                        const int took = __popcll(idle);
                        next += took < items - next ? took : items - next;
                    }
                    if (!__any(act)) break;
                    if (act) {
                        Cart<double> o;
                        eval_point_cached<K1, K2, 2, EXACT, double, kPatchGlobal, true>(
                            d, ku, kv, sv.cu, sv.cv, sc, o);
                        double d2;
                        if (sv.advance(d, o, P, dom, tol_step, sc, d2)) {
                            act = false;
                            if (phase == kProjLeaves) {
                                w.iu[it] = sv.cu;
                                w.iv[it] = sv.cv;
                                w.id2[it] = d2;
                                w.ist[it] = (uint8_t)sv.st;
                            } else if (phase == kProjBound || d2 <= w.best[it] * (1.0 + 1e-9)) {
                                // the bound; or the polished point, if not farther beyond rounding
                                w.best[it] = d2;
                                w.bu[it] = sv.cu;
                                w.bv[it] = sv.cv;
                                w.bst[it] = (uint8_t)sv.st;
                            }
                        }
                    }
                }
            }
            wave_lds_order();
            if (phase == kProjPolish) break;
            // ---- a lane per query: the best of the leaves solved, in the query's order
            for (int q = lane; q < nq; q += 64) {
                const float p[3] = {(float)w.P[0][q], (float)w.P[1][q], (float)w.P[2][q]};
                if (phase == kProjBound) {
                    // the root's children (a tree of one leaf has nothing to walk)
                    unsigned long long stk = 0;
                    if (D > 0) stk = box_mask<4>(lbox, p, floor32(w.best[q]));
                    w.stack[q] = stk;
                    w.path[q] = 0;
                    w.level[q] = 0;
                    // The bound solve stands for leaf c0's own solve only if it ended inside c0's
                    // cell; a solve that wandered off may have passed a nearer minimum in the
                    // cell, so c0 then stays a candidate (no leaf is left out).
                    const uint32_t c0 = w.c0[q];
                    const Domain cr = leaf_cell(c0);
                    const double bu = w.bu[q], bv = w.bv[q];
                    if (!(bu >= cr.u0 && bu <= cr.u1 && bv >= cr.v0 && bv <= cr.v1)) w.c0[q] = 0xffffffffu;
                } else {
                    double best = w.best[q];
                    const int i0 = w.first[q], i1 = i0 + w.taken[q];
                    for (int i = i0; i < i1; i++) {
                        if (!((double)w.ilb[i] <= best)) continue;
                        w.solved[q] += w.solved[q] < 0xffffu;
                        if (w.id2[i] < best) {
                            best = w.id2[i];
                            w.bu[q] = w.iu[i];
                            w.bv[q] = w.iv[i];
                            w.bst[q] = w.ist[i];
                        }
                    }
                    w.best[q] = best;
                }
            }
            wave_lds_order();
            // ---- the queries' walks: up to kProjPer leaves each, from where the last walk stopped
            unsigned long long stk[kProjQ / 64];
            uint32_t path[kProjQ / 64];
            int level[kProjQ / 64], nf[kProjQ / 64];
            int cands = 0;  // wave-uniform
#pragma unroll
            for (int g = 0; g < kProjQ / 64; g++) {
                const int q = 64 * g + lane, qs = q < nq ? q : 0;
                stk[g] = q < nq ? w.stack[qs] : 0ull;
                path[g] = w.path[qs];
                level[g] = w.level[qs];
                nf[g] = 0;
                if (__any(stk[g] != 0)) {
                    const float p[3] = {(float)w.P[0][qs], (float)w.P[1][qs], (float)w.P[2][qs]};
                    const float best32 = floor32(w.best[qs]);
                    const uint32_t c0 = w.c0[qs];
                    unsigned long long sk_ = stk[g];
                    uint32_t c = path[g];
                    int l = level[g], k = 0;
                    bool look = sk_ != 0;
                    while (look) {
                        const bool low = l == D - 2;  // a node whose 16 leaves are left
                        const uint32_t m = (uint32_t)(sk_ >> (4 * l)) & (low ? 0xffffu : 15u);
                        if (!m) {
                            if (l == 0) break;
                            c >>= 2;
                            l--;
                            continue;
                        }
                        const int j = __ffs(m) - 1;
                        sk_ &= ~(1ull << (4 * l + j));
                        if (low) {
                            if (16 * c + j == c0) continue;
                            w.found[q][k++] = 16 * c + j;
                            look = k < kProjPer;
                            continue;
                        }
                        c = 4 * c + j;
                        l++;
                        uint32_t cm;
                        if (l == D - 2) cm = box_mask<16>(sd.box32 + (qoff(D) + 16 * c) * 6, p, best32);
                        else if (l < ll) cm = box_mask<4>(lbox + (qoff(l + 1) - 1 + 4 * c) * 6, p, best32);
                        else cm = box_mask<4>(sd.box32 + (qoff(l + 1) + 4 * c) * 6, p, best32);
                        sk_ |= (unsigned long long)cm << (4 * l);
                    }
                    stk[g] = sk_;
                    path[g] = c;
                    level[g] = l;
                    nf[g] = k;
                }
                // the candidates of all queries, one list
                if (q < nq) w.holds[q] = 0u;
                for (int k = 0; __any(nf[g] > k); k++) {
                    const unsigned long long m = __ballot(nf[g] > k);
                    if (nf[g] > k) w.cand[cands + __popcll(m & lt)] = (uint16_t)(q * 8 + k);
                    cands += __popcll(m);
                }
            }
            wave_lds_order();
            // a lane per candidate: may the leaf hold a nearer foot point?  (The bound may have fallen
            // since its box was tested; the two index tests pass the leaves on the domain boundary, ix
            // or iy 0 or side - 1, by unsigned wrap-around.)
            for (int e = lane; e < cands; e += 64) {
                const int q = w.cand[e] >> 3, k = w.cand[e] & 7;
                const uint32_t leaf = w.found[q][k];
                const double P[3] = {w.P[0][q], w.P[1][q], w.P[2][q]};
                const float p[3] = {(float)P[0], (float)P[1], (float)P[2]};
                float b[6];
                __builtin_memcpy(b, sd.box32 + (qoff(D) + leaf) * 6, sizeof(b));
                if (box_d2(b, p) <= floor32(w.best[q]) &&
                    (!sd.cone32 || compact2(leaf >> 1) - 1u >= side - 2u ||
                     compact2(leaf) - 1u >= side - 2u ||
                     cone_may_hold(sd.cone32[leaf],
                                   *reinterpret_cast<const double *>(sd.rec + (size_t)leaf * kRecVec + 7),
                                   b, P)))
                    __hip_atomic_fetch_or(&w.holds[q], 1u << k, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_WAVEFRONT);
            }
            wave_lds_order();
            // into the pool, queries in order while there is room for all of a query's leaves (the
            // others walk again next time)
            items = 0;
#pragma unroll
            for (int g = 0; g < kProjQ / 64; g++) {
                const int q = 64 * g + lane;
                const uint32_t h = q < nq ? w.holds[q] : 0u;
                const int cnt = __popc(h);
                int end = cnt;  // inclusive prefix sum over the wave
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const int x = __shfl_up(end, o, 64);
                    if (lane >= o) end += x;
                }
                const bool fits = items + end <= kProjItems;
                int at = items + end - cnt;
                if (q < nq) {
                    w.first[q] = (uint8_t)at;
                    w.taken[q] = (uint8_t)(fits ? cnt : 0);
                    if (fits) {
                        w.stack[q] = stk[g];
                        w.path[q] = path[g];
                        w.level[q] = (uint8_t)level[g];
                        for (uint32_t m = h; m; m &= m - 1) {
                            w.ileaf[at] = w.found[q][__ffs(m) - 1];
                            w.iq[at++] = (uint8_t)q;
                        }
                    }
                }
                const unsigned long long fm = __ballot(fits);
                // prefix sums do not fall, so the fitting lanes are a leading run
                const int last = __popcll(fm) - 1;
                items += last >= 0 ? __shfl(end, last < 0 ? 0 : last, 64) : 0;
                if (fm != ~0ull) {  // later groups wait too
#pragma unroll
                    for (int g2 = g + 1; g2 < kProjQ / 64; g2++) {
                        const int q2 = 64 * g2 + lane;
                        if (q2 < nq) w.taken[q2] = 0;
                    }
                    break;
                }
            }
            wave_lds_order();
            // a lane per leaf: its start, the leaf's stepped seed for P clamped into its cell (fewer
            // Newton steps than from the cell centre)
            for (int i = lane; i < items; i += 64) {
                const int q = w.iq[i];
                const uint32_t leaf = w.ileaf[i];
                const double P[3] = {w.P[0][q], w.P[1][q], w.P[2][q]};
                const float p[3] = {(float)P[0], (float)P[1], (float)P[2]};
                float b[6];
                __builtin_memcpy(b, sd.box32 + (qoff(D) + leaf) * 6, sizeof(b));
                const Domain cr = leaf_cell(leaf);
                double cu, cv;
                step_seed(sd, leaf, sd.rec[(size_t)leaf * kRecVec], P, cu, cv);
                w.ilb[i] = box_d2(b, p);
                w.iu[i] = fmin(fmax(cu, cr.u0), cr.u1);
                w.iv[i] = fmin(fmax(cv, cr.v0), cr.v1);
            }
            // nothing in the pool, and every walk at its end: the polish
            phase = kProjLeaves;
            if (!items) {
                bool left = false;
                for (int q = lane; q < nq; q += 64) left |= w.stack[q] != 0;
                if (!__any(left)) {
                    phase = kProjPolish;
                    items = nq;
                }
            }
        }
        // ---- results
        for (int q = lane; q < nq; q += 64) {
            const size_t i = LIST || order ? (size_t)order[q0 + q] : q0 + q;
            if constexpr (LIST) {  // the earlier result stays if it is nearer
                Cart<double> e;
                eval_point<K1, K2, 0, EXACT, double>(d, ku, kv, a.u[i], a.v[i], e);
                const double dx = e.S[0] - w.P[0][q], dy = e.S[1] - w.P[1][q], dz = e.S[2] - w.P[2][q];
                if (fma(dz, dz, fma(dy, dy, dx * dx)) < w.best[q]) continue;
            }
            a.u[i] = w.bu[q];
            a.v[i] = w.bv[q];
            a.status[i] = w.bst[q];
            if constexpr (!LIST) {
                if (a.it32) a.it32[i] = sat8(w.solved[q]);
                if (a.it64) a.it64[i] = 0;
            }
        }
        wave_lds_order();
    }
}

// Spatial order of the queries: the key is the 16 x 16 x 16 cell of P within the tree's root box
// (Morton order, 12 bits; points outside the box take its border cells, NaN coordinates cell 0).
// One workgroup per block of kOrdBlock consecutive queries counts its keys in LDS, scans them and
// writes each query's index to its key's next slot within the block's own range of `order`.  Keys stay
// in registers between the two passes and the block's loads are issued together: with blocks of 65,536
// read twice in sequence, four workgroups took 103 us for 262,144 queries.  The
// order within one key is unspecified; each query's result is its own and does not depend
// on it.
constexpr int kOrdThreads = 1024;
constexpr int kOrdPer = 16;  // queries per thread
constexpr size_t kOrdBlock = (size_t)kOrdPer * kOrdThreads;
constexpr int kOrdKeys = 4096;

__device__ __forceinline__ uint32_t proj_key(const float *__restrict__ root, const double P[3]) {
    uint32_t q[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const float lo = root[k], w = root[3 + k] - root[k];
        const float t = w > 0.f ? ((float)P[k] - lo) * (16.f / w) : 0.f;
        q[k] = (uint32_t)fminf(fmaxf(t, 0.f), 15.f);
    }
    uint32_t m = 0;
#pragma unroll
    for (int b = 0; b < 4; b++)
        m |= ((q[0] >> b & 1u) << (3 * b + 2)) | ((q[1] >> b & 1u) << (3 * b + 1)) |
             ((q[2] >> b & 1u) << (3 * b));
    return m;
}

__global__ __launch_bounds__(kOrdThreads) void k_proj_order(const float *__restrict__ root,
                                                            const double *__restrict__ x,
                                                            const double *__restrict__ y,
                                                            const double *__restrict__ z, size_t n,
                                                            uint32_t *__restrict__ order) {
    __shared__ uint32_t cnt[kOrdKeys];
    __shared__ uint32_t part[kOrdThreads];
    for (int k = threadIdx.x; k < kOrdKeys; k += kOrdThreads) cnt[k] = 0u;
    __syncthreads();
    const size_t i0 = (size_t)blockIdx.x * kOrdBlock;
    const size_t i1 = i0 + kOrdBlock < n ? i0 + kOrdBlock : n;
    uint32_t key[kOrdPer];
#pragma unroll
    for (int k = 0; k < kOrdPer; k++) {
        const size_t i = i0 + (size_t)k * kOrdThreads + threadIdx.x;
        const size_t j = i < i1 ? i : i1 - 1;
        const double P[3] = {x[j], y[j], z[j]};
        key[k] = proj_key(root, P);
    }
#pragma unroll
    for (int k = 0; k < kOrdPer; k++)
        if (i0 + (size_t)k * kOrdThreads + threadIdx.x < i1) atomicAdd(&cnt[key[k]], 1u);
    __syncthreads();
    // exclusive scan: each thread a run of kOrdKeys / kOrdThreads keys, then the runs' sums
    constexpr int per = kOrdKeys / kOrdThreads;
    const int k0 = threadIdx.x * per;
    uint32_t sum = 0;
#pragma unroll
    for (int k = 0; k < per; k++) sum += cnt[k0 + k];
    part[threadIdx.x] = sum;
    __syncthreads();
    for (int o = 1; o < kOrdThreads; o <<= 1) {  // inclusive Hillis-Steele scan of the sums
        const uint32_t v = threadIdx.x >= (unsigned)o ? part[threadIdx.x - o] : 0u;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    uint32_t run = (uint32_t)i0 + (threadIdx.x ? part[threadIdx.x - 1] : 0u);
#pragma unroll
    for (int k = 0; k < per; k++) {
        const uint32_t c = cnt[k0 + k];
        cnt[k0 + k] = run;
        run += c;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kOrdPer; k++) {
        const size_t i = i0 + (size_t)k * kOrdThreads + threadIdx.x;
        if (i < i1) order[atomicAdd(&cnt[key[k]], 1u)] = (uint32_t)i;
    }
}

__global__ void k_fb_zero(uint32_t *count) { *count = 0u; }

// indices of the queries whose status is not converged
__global__ void k_fb_compact(const uint8_t *__restrict__ status, size_t n, uint32_t *__restrict__ list,
                             uint32_t *__restrict__ count) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x)
        if (status[i] != GN_PT_CONVERGED && status[i] != GN_PT_CONVERGED_DIST)
            list[atomicAdd(count, 1u)] = (uint32_t)i;
}

struct ProjectLaunch {
    const GnSurfDev &d;
    const GnSearchDev &sd;
    const InvArgs &a;
    const uint32_t *order, *count;  // count: the fallback's list length
    hipStream_t st;
    template <int K1, int K2, bool EXACT>
    int operator()() {
        const unsigned cus = (unsigned)cu_count();
        const int chunk = project_chunk(a.n, cus);
        const size_t lds = EXACT ? sizeof(double) * (2 * d.nu + 2 * d.nv + 2) : 0;
        if (count) {
            // eight workgroups per CU at most, four rounds: the list is seldom as long as the call, and a
            // workgroup past its end costs its start (inversion and fallback of 16,000,000 queries, none of
            // them listed: 2,442 us with a workgroup per 64 queries of the call, 1,975 with this grid; 5% of
            // 1,000,000 listed: 1,399 and 1,221)
            const unsigned grid = grid_for(a.n, 4 * 16, 8 * cus);
            k_project<K1, K2, EXACT, true><<<grid, 256, lds, st>>>(d, sd, a, order, count, 0, cus);
        } else {
            const unsigned grid = grid_for(a.n, 4 * chunk, 1u << 23);
            k_project<K1, K2, EXACT, false><<<grid, 256, lds, st>>>(d, sd, a, order, nullptr, chunk, cus);
        }
        GN_HIP(hipGetLastError());
        return GN_OK;
    }
};

// Calls of at least kOrdMin queries (fewer than 2^32) take them in spatial order: a stream-ordered
// scratch index array of n words, filled by k_proj_order.  Calls that must not allocate (the
// no-allocation entry point) take them in input order.
constexpr size_t kOrdMin = 16384;

int launch_project_global(const GnSurfDev &d, const GnSearchDev &sd, const InvArgs &a,
                          hipStream_t st) {
    if (a.n == 0) return GN_OK;
    uint32_t *order = nullptr;
    if (a.n >= kOrdMin && a.n < 0xffffffffull && sd.depth > 0 && !slot_pool_active()) {
        GN_HIP(hipMallocAsync((void **)&order, sizeof(uint32_t) * a.n, st));
        k_proj_order<<<(unsigned)((a.n + kOrdBlock - 1) / kOrdBlock), kOrdThreads, 0, st>>>(
            sd.box32, a.x, a.y, a.z, a.n, order);
        if (hipGetLastError() != hipSuccess) {
            (void)hipFreeAsync(order, st);
            return fail(GN_EDEVICE, "query ordering launch");
        }
    }
    const int rc = dispatch_inv(d, ProjectLaunch{d, sd, a, order, nullptr, st});
    if (order) GN_HIP(hipFreeAsync(order, st));
    return rc;
}

// After an inversion on st: the unconverged queries are listed on the device (stream-ordered
// scratch of n + 1 words) and solved again by the global projection.
int launch_project_fallback(const GnSurfDev &d, const GnSearchDev &sd, const InvArgs &a,
                            hipStream_t st) {
    if (a.n == 0) return GN_OK;
    if (a.n > 0xffffffffull) return fail(GN_EINVAL, "the fallback lists at most 2^32 - 1 queries");
    uint32_t *buf = nullptr;
    GN_HIP(hipMallocAsync((void **)&buf, sizeof(uint32_t) * (a.n + 1), st));
    uint32_t *count = buf, *list = buf + 1;
    k_fb_zero<<<1, 1, 0, st>>>(count);
    k_fb_compact<<<grid_for(a.n, 256, 256 * 16), 256, 0, st>>>(a.status, a.n, list, count);
    int rc = hipGetLastError() == hipSuccess ? GN_OK : fail(GN_EDEVICE, "fallback compaction launch");
    if (!rc) rc = dispatch_inv(d, ProjectLaunch{d, sd, a, list, count, st});
    GN_HIP(hipFreeAsync(buf, st));
    return rc;
}

}  // namespace gn

// eval.hip -- batch evaluation of a surface and its derivatives up to third order (EvaluateRandom,
// src/NURBS/Evaluate.cu:1023-1038, extended to the derivatives of 288-502 and 535-1020).
//
// One lane per query point, grid-stride over the batch.  Parameters stream in and results stream
// out as SoA arrays, so every global load and store of the batch is a fully coalesced 256-byte
// (FP32) or 512-byte (FP64) wave access.  Span patches come from the L2-resident span table:
// for exact degrees they are staged through LDS one row at a time by cooperative contiguous
// loads, with knots and reciprocal span lengths also in LDS (k_eval_rows); otherwise each lane
// gathers its own patch and reads knots through L1 (k_eval).  The target roof is HBM traffic
// (8 or 16 bytes in, 12..240 bytes out per point).
#include "invert_common.hpp"

namespace gn {

constexpr int kEvalBlock = 256;

// Streams one point's fields into the SoA output: S, then Su Sv, Suu Suv Svv, Suuu Suuv Suvv Svvv
// up to ORDER, each field three blocks (x, y, z) of n values.
template <int ORDER, typename T>
__device__ __forceinline__ void store_fields(const Cart<T> &o, T *__restrict__ out, size_t n,
                                             size_t i) {
#pragma unroll
    for (int c = 0; c < 3; c++) __builtin_nontemporal_store(o.S[c], out + c * n + i);
    if (ORDER >= 1) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            __builtin_nontemporal_store(o.Su[c], out + (3 + c) * n + i);
            __builtin_nontemporal_store(o.Sv[c], out + (6 + c) * n + i);
        }
    }
    if (ORDER >= 2) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            __builtin_nontemporal_store(o.Suu[c], out + (9 + c) * n + i);
            __builtin_nontemporal_store(o.Suv[c], out + (12 + c) * n + i);
            __builtin_nontemporal_store(o.Svv[c], out + (15 + c) * n + i);
        }
    }
    if (ORDER >= 3) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            __builtin_nontemporal_store(o.Suuu[c], out + (18 + c) * n + i);
            __builtin_nontemporal_store(o.Suuv[c], out + (21 + c) * n + i);
            __builtin_nontemporal_store(o.Suvv[c], out + (24 + c) * n + i);
            __builtin_nontemporal_store(o.Svvv[c], out + (27 + c) * n + i);
        }
    }
}

template <int K1, int K2, bool EXACT, int ORDER, typename T, typename TP>
__global__ __launch_bounds__(kEvalBlock) void k_eval(GnSurfDev d, const TP *__restrict__ u,
                                                     const TP *__restrict__ v, size_t n,
                                                     T *__restrict__ out) {
    const double *ku = d.ku, *kv = d.kv;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x) {
        Cart<T> o;
        eval_point<K1, K2, ORDER, EXACT, T>(d, ku, kv, (double)u[i], (double)v[i], o);
        store_fields<ORDER>(o, out, n, i);
    }
}

constexpr int kLdsKnotsSmall = 512;

// Row-staged form for exact degrees with knots in LDS: a wave takes 64 points at a time and
// stages their patches one row at a time through a small LDS buffer (WaveRowsPipe: contiguous
// 16-byte loads covering whole rows of several lanes, the next row prefetched while the current
// one is contracted).  The buffer is one row per lane (9 KB per wave for FP64 bicubic), so
// occupancy is set by registers rather than LDS.  A block takes `tiles` * 256 consecutive points and
// the blocks start in order, so the rows are written in a narrow moving window: with a fixed grid of
// blocks striding over the batch the waves drift apart, and 16.8M bicubic FP64 points of second order
// took 906 us against 791, 9,999,991 FP32 points 372 against 277, 1,000,003 points of degree (5,4) and
// third order 133 against 98.  What is left is the writes' (the same rows streamed without any
// evaluation take 515 us).
constexpr int kRowBlock = 256;
constexpr int kRowWaves = kRowBlock / 64;

template <int K1, int K2, int ORDER, typename T, typename TP>
__global__ __launch_bounds__(kRowBlock) void k_eval_rows(GnSurfDev d, const TP *__restrict__ u,
                                                         const TP *__restrict__ v, size_t n,
                                                         T *__restrict__ out, size_t tiles) {
    using Rows = WaveRowsPipe<K1, K2, T>;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const size_t chunk = tiles * kRowBlock, first = blockIdx.x * chunk;
    const size_t end = first + chunk < n ? first + chunk : n;
    size_t base = first + (size_t)wv * 64;
    // parameters of the next tile are loaded one tile ahead
    TP pu = 0, pv = 0;
    if (base + lane < end) { pu = u[base + lane]; pv = v[base + lane]; }
    // knots and reciprocal span lengths: nku + nkv + (nu - p) + (nv - q) <= 2 * kLdsKnotsSmall
    __shared__ double sk[2 * kLdsKnotsSmall];
    __shared__ float4 stage[kRowWaves * 64 * Rows::STRIDE];
    const int nku = d.nu + d.p + 1, nkv = d.nv + d.q + 1, nsu = d.nu - d.p, nsv = d.nv - d.q;
    // four loads in flight, then the four stores (one after the other they are four round trips)
    for (int i = threadIdx.x; i < nku || i < nkv; i += kRowBlock) {
        const double a = i < nku ? d.ku[i] : 0, b = i < nkv ? d.kv[i] : 0;
        const double e = i < nsu ? d.ihu[i] : 0, f = i < nsv ? d.ihv[i] : 0;
        if (i < nku) sk[i] = a;
        if (i < nkv) sk[nku + i] = b;
        if (i < nsu) sk[nku + nkv + i] = e;
        if (i < nsv) sk[nku + nkv + nsu + i] = f;
    }
    __syncthreads();
    const double *ku = sk, *kv = sk + nku, *ihus = sk + nku + nkv, *ihvs = ihus + nsu;
    const double inv_u = (double)(d.nu - d.p) / (ku[d.nu] - ku[d.p]);
    const double inv_v = (double)(d.nv - d.q) / (kv[d.nv] - kv[d.q]);
    float4 *my = stage + (size_t)wv * 64 * Rows::STRIDE;
    const T *tab = sizeof(T) == 8 ? reinterpret_cast<const T *>(d.tab64)
                                  : reinterpret_cast<const T *>(d.tab32);
    for (; base < end; base += kRowBlock) {
        const size_t i = base + lane;
        const bool live = i < end;
        const double uu = live ? (double)pu : 0.0, vv = live ? (double)pv : 0.0;
        const size_t inext = base + kRowBlock + lane;
        if (inext < end) { pu = u[inext]; pv = v[inext]; }
        const int m = find_span_guess(ku, d.p, d.nu, uu, inv_u);
        const int nn = find_span_guess(kv, d.q, d.nv, vv, inv_v);
        const int im = m - d.p, in = nn - d.q;
        const T *patch = tab + (size_t)(im * d.sv + in) * (K1 * K2 * 4);
        Rows rows(patch, my);
        const double ihu = ihus[im], ihv = ihvs[in];
        const T t = T((uu - ku[m]) * ihu), s = T((vv - kv[nn]) * ihv);
        HomDer<T> h;
        contract_rows<K1, K2, ORDER, true, T>(rows, K1, K2, t, s, h);
        Cart<T> o;
        quotient<ORDER, T>(h, T(ihu), T(ihv), o);
        if (live) store_fields<ORDER>(o, out, n, i);
    }
}

template <typename T, typename TP>
struct EvalLaunch {
    const GnSurfDev &d;
    const TP *u, *v;
    size_t n;
    int order;
    T *out;
    hipStream_t st;
    // Tiles of 64 points per wave.  A block costs a start (its knots into LDS, the first parameters from
    // HBM), so a wave should take several; but the more of them are under way, the further apart the
    // lines written at one time, and where rows don't start on a line a line's two halves must meet in
    // L2.  What decides is the bytes written per unit of work, per patch entry: few, and the writes wait
    // for the waves whatever they do.  us for 1 / 2 / 4 / 8 tiles, inputs and outputs not in cache, on rows
    // of whole lines:
    //   FP64 under 7 (orders 0 and 1; (4,4) order 2): 16 M points, order 1 737 / 626 / 594 / 596, (4,4) order 2
    //     1682 / 1399 / 1232 / 1162: eight; also where patches hold more than 16 entries.  (3,3) order 2 831 /
    //     789 / 768 / 815, order 3 1118 / 1115 / 1104 / 1146: four.  (2,2) order 2 726 / 653 / 778 / 804: two; order 3
    //     at 4,194,304 points 171 / 191 / 217 / 238: one.
    //   FP32 (3,3) order 2, 12 M points 322 / 313 / 312 / 321, order 1, 16 M 360 / 333 / 329 / 341, (5,5) order 2 863 /
    //     697 / 662 / 666: four.  (2,2) order 2 441 / 446 / 465 / 482: two; order 3 at 8,388,608 204 / 212 / 211 / 243:
    //     one.
    // and on others:
    //   FP64 (3,3) order 2, 5,000,003 points 249 / 229 / 246 / 256: two; order 3, 4,194,305 295 / 418 / 404 / 426, (2,2)
    //     order 2 168 / 235 / 245 / 248: one.  Patches of more than 20 entries, a block per CU: (5,4) order 3, 1,000,003
    //     120 / 107 / 98 / 94: eight; (4,4) order 3, 4,194,305 426 / 380 / 393 / 462, 8,388,613 998 / 802 / 786 / 745: four.
    //   FP32 (3,3) order 1, 5,000,003 108 / 98 / 93 / 94: four; (4,4) order 2, 2,000,005 78 / 74 / 77 / 85: two; (3,3)
    //     order 2, 4,194,305 107 / 138 / 183 / 227: one.  (2,5) order 2 lies between, 2,000,005 points 61 / 66 / 70 / 77,
    //     4,194,305 128 / 130, 8,388,613 248 / 226: two from 6 M points.
    // Rows a multiple of 64 MiB apart start on the same channels: four tiles lose to two, FP64 (3,3) order 2
    // 16,777,216 points 837 / 800, FP32 482 / 462.
    // All that holds over many rounds.  Where one round of the resident blocks takes all the points, it has no
    // last round that is part empty, and over (2,2) to (5,5) and orders 0 to 3, 131,072 to 1,500,001 points, it wins
    // up to eight tiles, us for that against the number above: FP64 (3,3) order 2, 800,000 points 41.9 / 45.4, order 3
    // 51.1 / 56.3, FP32 (2,5) order 2 27.4 / 31.8.  On rows of partial lines up to seven, and only where the rule
    // above has four for FP32 ((5,5) order 1, 800,003 points 0.80 of the time; where it has two or one, 1.0 to 1.3)
    // and two for FP64 ((4,4) order 3, 300,003 34 / 48; eight tiles 1.03 to 1.08); where it has one, two rounds only:
    // FP64 (2,2) order 2, 200,003 14.5 / 16.8, three 1.15.  FP32 waves of two tiles leave the last round half empty
    // where the rounds are odd: with one, (5,5) order 3, 300,003 24.8 / 27.4, (4,4) order 2, 400,001 23.6 /
    // 24.7; at order 1 two stay ahead, (2,2) 800,003 0.95.
    static bool one_round(size_t tiles, size_t most, size_t n) {
        if (n % (128 / sizeof(T)) == 0) return most > 1 && tiles <= 8;
        if (sizeof(T) == 4) return most == 4 && tiles <= 7;
        return most > 1 ? tiles <= 7 : tiles == 2;
    }
    static size_t most_tiles(int entries, int order, size_t n) {
        const size_t fields = order == 0 ? 3 : order == 1 ? 9 : order == 2 ? 18 : 30;
        const double per = (double)(fields * sizeof(T)) / entries;  // bytes written per patch entry
        if (n % (128 / sizeof(T)) != 0) {
            if (sizeof(T) == 4) return per < 2.5 ? 4 : per < (order >= 2 && n < 6000000 ? 3.7 : 4.4) ? 2 : 1;
            if (entries > 20) return per < 9 ? 8 : 4;
            return per < 7 ? 8 : per < 14 ? 2 : 1;
        }
        if (sizeof(T) == 8 && (per < 7 || entries > 16)) return 8;
        const bool four = per < (sizeof(T) == 8 ? 15.5 : 7.8), two = per < (sizeof(T) == 8 ? 20 : 10);
        return four && !(order >= 2 && n * sizeof(T) % ((size_t)1 << 26) == 0) ? 4 : two ? 2 : 1;
    }
    static bool odd_rounds(size_t tiles, size_t most, size_t n) {
        return sizeof(T) == 4 && n % 32 != 0 && most == 2 && tiles % 2 == 1 && tiles <= 7;
    }
    template <int K1, int K2, int ORDER>
    int rows() {
        auto k = k_eval_rows<K1, K2, ORDER, T, TP>;
        const size_t blocks = (n + kRowBlock - 1) / kRowBlock;
        const size_t cus = (size_t)cu_count();
        const size_t resident = blocks > cus ? cus * blocks_per_cu((const void *)k, kRowBlock) : cus;
        const size_t most = most_tiles(K1 * K2, ORDER, n);
        size_t tiles = (blocks + resident - 1) / resident;
        if (ORDER >= 2 && odd_rounds(tiles, most, n)) tiles = 1;
        // the rounds that `most` tiles would take, evenly filled: FP64 (4,4) order 0, 600,001 points are 10 tiles for
        // each resident wave, two rounds of 5 45 us, 8 and a rest 65; order 0 (3,3) 1,500,000, 12, 52 and 55
        if (tiles > most && !one_round(tiles, most, n)) {
            const size_t rounds = (tiles + most - 1) / most;
            tiles = (tiles + rounds - 1) / rounds;
        }
        if (tiles < n >> 31) tiles = n >> 31;  // a grid holds below 2^32 lanes
        if (tiles < 1) tiles = 1;
        const unsigned grid = (unsigned)((blocks + tiles - 1) / tiles);
        k<<<grid, kRowBlock, 0, st>>>(d, u, v, n, out, tiles);
        GN_HIP(hipGetLastError());
        return GN_OK;
    }
    template <int K1, int K2, bool EXACT>
    int operator()() {
        const unsigned grid = grid_for(n, kEvalBlock, 256 * 16);
        const bool knots_fit = d.nu + d.p + 1 + d.nv + d.q + 1 <= kLdsKnotsSmall;
        if constexpr (EXACT) if (knots_fit) {
            switch (order) {
                case 0: return rows<K1, K2, 0>();
                case 1: return rows<K1, K2, 1>();
                case 2: return rows<K1, K2, 2>();
                default: return rows<K1, K2, 3>();
            }
        }
        switch (order) {
            case 0: k_eval<K1, K2, EXACT, 0, T, TP><<<grid, kEvalBlock, 0, st>>>(d, u, v, n, out); break;
            case 1: k_eval<K1, K2, EXACT, 1, T, TP><<<grid, kEvalBlock, 0, st>>>(d, u, v, n, out); break;
            case 2: k_eval<K1, K2, EXACT, 2, T, TP><<<grid, kEvalBlock, 0, st>>>(d, u, v, n, out); break;
            default: k_eval<K1, K2, EXACT, 3, T, TP><<<grid, kEvalBlock, 0, st>>>(d, u, v, n, out); break;
        }
        GN_HIP(hipGetLastError());
        return GN_OK;
    }
};

int launch_eval64(const GnSurfDev &d, const double *u, const double *v, size_t n, int order,
                  double *out, hipStream_t st) {
    if (n == 0) return GN_OK;
    return dispatch_degrees(d.p, d.q, EvalLaunch<double, double>{d, u, v, n, order, out, st});
}

int launch_eval32(const GnSurfDev &d, const float *u, const float *v, size_t n, int order,
                  float *out, hipStream_t st) {
    if (n == 0) return GN_OK;
    return dispatch_degrees(d.p, d.q, EvalLaunch<float, float>{d, u, v, n, order, out, st});
}

}  // namespace gn

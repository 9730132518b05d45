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
// took 910 us against 770, 9,999,991 FP32 points 374 against 296, 1,000,003 points of degree (5,4) and
// third order 128 against 94.  What is left is the writes' (the same rows streamed without any
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
    // L2.  Up to eight rounds of the resident blocks, one round.  Beyond, us for 1 / 2 / 4 / 8 tiles
    // (bicubic, second order unless said): FP64 16.8M points 889 / 770 / 855 / 901, 4.2M 197 / 175 /
    // 165 / 166, 3,999,999 193 / 170 / 196 / 217; order 0, 4M 140 / 116 / 106 / 102; FP32 9,999,872
    // points 231 / 209 / 191 / 191, 9,999,991 296 / 307 / 322 / 341, order 1 16M 343 / 319 / 334 / 346.
    // FP64 patches of more than 16 entries run a block per CU: degree (5,4), third order, 1,000,003
    // points 120 / 107 / 98 / 94.
    template <int K1, int K2, int ORDER>
    int rows() {
        auto k = k_eval_rows<K1, K2, ORDER, T, TP>;
        const size_t blocks = (n + kRowBlock - 1) / kRowBlock;
        const size_t cus = (size_t)cu_count();
        const size_t resident = blocks > cus ? cus * blocks_per_cu((const void *)k, kRowBlock) : cus;
        const bool lines = n % (128 / sizeof(T)) == 0, many = ORDER >= 2;
        const size_t bytes = n * (ORDER == 0 ? 3 : ORDER == 1 ? 9 : ORDER == 2 ? 18 : 30) * sizeof(T);
        size_t most = 4;
        if (sizeof(T) == 8) most = K1 * K2 > 16 ? 8 : many && (!lines || bytes > 800000000) ? 2 : 4;
        else if (many && !lines) most = 1;
        size_t tiles = (blocks + resident - 1) / resident;
        if (tiles > 8 || !lines) tiles = tiles < most ? tiles : most;
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

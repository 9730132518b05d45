// grid.hip -- FP32 evaluation of a tensor-product parameter grid (the form of the FP16 cuBLAS
// span-GEMM experiment of src/main.cu:533-663 and src/kernel/kernel.cu:1558-1604 for parameters on a
// grid).
//
// The grid's rows are u-samples, its columns v-samples, and a row's points are contiguous in the output.
// A lane owns one column and a wave 64 consecutive ones.  Per span of u the lane contracts its column's
// patch along v once,
//     Y^(b)_c[r] = sum_s M_c(m, n)[r][s] V^(b)_s            (b = 0 .. max_order),
// and keeps Y in registers; every row of that span then costs the u side alone,
//     R^(a,b)_c = sum_r U^(a)_r Y^(b)_c[r],
// whose U is the same for the whole wave (scalar operands), and the rational quotient.  No point loads
// anything, so the kernel never waits for memory between span changes, and each store of a field is
// 256 contiguous bytes per wave.  Grids of few columns take k_grid_strip.
//
// Bound: HBM writes (72 bytes per point at order 2; about 160 VALU instructions per 64 points, under a
// third of the time the writes take).  The 16 x 16 blocks on v_mfma_f32_16x16x4f32 that this replaces
// needed half the VALU work but wrote 64-byte pieces and searched spans anew per block: 4096 x 4096
// points at order 2 took 376 us (3.2 TB/s) there and 246 us (4.9 TB/s) here.  Sparse grids take the
// same kernel: a row in a new span costs the v side again, which is what a point on its own costs.
// Stores are ordinary ones: a row pitch that is no multiple of 128 bytes leaves partial lines at both
// ends of every store, which L2 joins and non-temporal stores send out as they are (2500 x 2500
// points at order 2: 136 against 196 us; 2501 x 2499 at order 1: 43 against 102 us).
#include "gn_device.hpp"

namespace gn {

constexpr int kGridBlock = 256;
constexpr int kGridRows = 32;  // most rows per workgroup, and per lane of a strip
constexpr int kStripCols = 32;

// Powers of a column's local parameter and their derivatives.
template <int K2, int ORDER>
__device__ __forceinline__ void column_powers(float s, float (&V)[ORDER + 1][K2]) {
    V[0][0] = 1.f;
#pragma unroll
    for (int c = 1; c < K2; c++) V[0][c] = V[0][c - 1] * s;
#pragma unroll
    for (int c = 0; c < K2; c++) {
        if (ORDER >= 1) V[1][c] = c >= 1 ? float(c) * V[0][c - 1] : 0.f;
        if (ORDER >= 2) V[2][c] = c >= 2 ? float(c * (c - 1)) * V[0][c - 2] : 0.f;
    }
}

// The column's patch contracted along v.
template <int K1, int K2, bool EXACT, int ORDER>
__device__ __forceinline__ void column_side(const float *patch, int k1, int k2,
                                            const float (&V)[ORDER + 1][K2],
                                            Hom<float> (&Y)[K1][ORDER + 1]) {
#pragma unroll
    for (int r = 0; r < K1; r++) {
        if (!EXACT && r >= k1) break;
#pragma unroll
        for (int e = 0; e <= ORDER; e++) hzero(Y[r][e]);
#pragma unroll
        for (int c = 0; c < K2; c++) {
            if (!EXACT && c >= k2) break;
            const Hom<float> h = load_hom<float>(patch + (r * k2 + c) * 4);
#pragma unroll
            for (int e = 0; e <= ORDER; e++)
                if (c >= e) hfma(Y[r][e], V[e][c], h);
        }
    }
}

// One point from its column side and its row's local parameter t.
template <int K1, bool EXACT, int ORDER>
__device__ __forceinline__ void row_side(const Hom<float> (&Y)[K1][ORDER + 1], int k1, float t, float ihu,
                                         float ihv, Cart<float> &o) {
    HomDer<float> h;
    hzero(h.R);
    if (ORDER >= 1) { hzero(h.Ru); hzero(h.Rv); }
    if (ORDER >= 2) { hzero(h.Ruu); hzero(h.Ruv); hzero(h.Rvv); }
    float p0 = 1.f, p1 = 0.f, p2 = 0.f;  // t^r, t^(r-1), t^(r-2)
#pragma unroll
    for (int r = 0; r < K1; r++) {
        if (!EXACT && r >= k1) break;
        hfma(h.R, p0, Y[r][0]);
        if constexpr (ORDER >= 1) {
            hfma(h.Rv, p0, Y[r][1]);
            if (r >= 1) hfma(h.Ru, float(r) * p1, Y[r][0]);
        }
        if constexpr (ORDER >= 2) {
            hfma(h.Rvv, p0, Y[r][2]);
            if (r >= 1) hfma(h.Ruv, float(r) * p1, Y[r][1]);
            if (r >= 2) hfma(h.Ruu, float(r * (r - 1)) * p2, Y[r][0]);
        }
        p2 = p1;
        p1 = p0;
        p0 *= t;
    }
    quotient<ORDER, float>(h, ihu, ihv, o);
}

template <int ORDER>
__device__ __forceinline__ void store_point(const Cart<float> &o, float *dst, size_t npts) {
#pragma unroll
    for (int c = 0; c < 3; c++) *(dst + c * npts) = o.S[c];
    if (ORDER >= 1) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            *(dst + (3 + c) * npts) = o.Su[c];
            *(dst + (6 + c) * npts) = o.Sv[c];
        }
    }
    if (ORDER >= 2) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            *(dst + (9 + c) * npts) = o.Suu[c];
            *(dst + (12 + c) * npts) = o.Suv[c];
            *(dst + (15 + c) * npts) = o.Svv[c];
        }
    }
}

template <int K1, int K2, bool EXACT, int ORDER>
__global__ __launch_bounds__(kGridBlock) void k_grid(GnSurfDev d, const float *__restrict__ us, int nua,
                                                     const float *__restrict__ vs, int nvb, int rows,
                                                     unsigned col_blocks, float *__restrict__ out) {
    __shared__ float row_t[kGridRows], row_ih[kGridRows];
    __shared__ int row_m[kGridRows];
    const int k1 = EXACT ? K1 : d.p + 1, k2 = EXACT ? K2 : d.q + 1;
    const unsigned cb = blockIdx.x % col_blocks, rb = blockIdx.x / col_blocks;
    const int a0 = (int)(rb * (unsigned)rows);
    int na = min(rows, nua - a0);
    if ((int)threadIdx.x < na) {
        const double uu = (double)us[a0 + threadIdx.x];
        const int m = find_span_near(d.ku, d.p, d.nu, uu) - d.p;
        const double ih = d.ihu[m];
        row_t[threadIdx.x] = (float)((uu - d.ku[m + d.p]) * ih);
        row_ih[threadIdx.x] = (float)ih;
        row_m[threadIdx.x] = m;
    }
    const int b = (int)(cb * kGridBlock + threadIdx.x);
    const bool live = b < nvb;
    const double vv = (double)vs[live ? b : nvb - 1];
    const int nv = find_span_near(d.kv, d.q, d.nv, vv) - d.q;
    const float ihv = (float)d.ihv[nv];
    const float s = (float)((vv - d.kv[nv + d.q]) * d.ihv[nv]);
    float V[ORDER + 1][K2];  // s^c and its derivatives
    column_powers<K2, ORDER>(s, V);
    __syncthreads();
    if (!__any(live)) {  // a wave past the last column
        if constexpr (ORDER == 0) return;
        na = 0;
    }
    const size_t npts = (size_t)nua * nvb, kk = (size_t)k1 * k2 * 4;
    float *dst = out + (size_t)a0 * nvb + b;
    Hom<float> Y[K1][ORDER + 1];
    int cur = -1;
    for (int a = 0; a < na; a++, dst += nvb) {  // workgroup-uniform
        const int m = __builtin_amdgcn_readfirstlane(row_m[a]);
        const float t = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(row_t[a])));
        const float ihu = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(row_ih[a])));
        if (m != cur) {
            cur = m;
            column_side<K1, K2, EXACT, ORDER>(d.tab32 + ((size_t)m * d.sv + nv) * kk, k1, k2, V, Y);
        }
        Cart<float> o;
        row_side<K1, EXACT, ORDER>(Y, k1, t, ihu, ihv, o);
        if (live) store_point<ORDER>(o, dst, npts);
    }
    // With derivatives a wave without columns waits for the others: in its place more workgroups would
    // write at a time, and the ends of their rows' lines leave L2 before they meet (200,000 x 40 points,
    // order 2: 132 us, 158 where it leaves at once; order 0 33 and 26).
    if constexpr (ORDER > 0) __syncthreads();
}

// Grids of at most kStripCols columns.  A workgroup's lanes are spread over G = 256 / columns rows at a
// time (lane l: row l / columns, column l % columns), so consecutive lanes still write consecutive points.
// A lane keeps its column's v side as above; its rows, G apart, are its own, so their parameters are vector
// operands that it finds itself.  k_grid leaves the lanes past the last column idle: bicubic, order 2, there
// and here, 1,048,576 x 1 points 313 and 17 us, x 4 314 and 91, x 16 359 and 230, 500,000 x 32 226 and 224;
// order 0 x 16 88 and 38, x 32 49 and 37, 333,333 x 48 37 and 42.  Wider grids of partial lines differ either
// way (order 2, 160,000 x 100 463 and 355, 80,000 x 200 333 and 356).
template <int K1, int K2, bool EXACT, int ORDER>
__global__ __launch_bounds__(kGridBlock) void k_grid_strip(GnSurfDev d, const float *__restrict__ us,
                                                           int nua, const float *__restrict__ vs, int nvb,
                                                           int rows, float *__restrict__ out) {
    const int k1 = EXACT ? K1 : d.p + 1, k2 = EXACT ? K2 : d.q + 1;
    const int G = kGridBlock / nvb, g = (int)threadIdx.x / nvb, b = (int)threadIdx.x - g * nvb;
    const int a0 = (int)blockIdx.x * rows, a1 = min(a0 + rows, nua);
    int a = a0 + g;
    if (g >= G || a >= a1) return;
    float un = us[a];
    const double vv = (double)vs[b];
    const int nv = find_span_near(d.kv, d.q, d.nv, vv) - d.q;
    const float ihv = (float)d.ihv[nv];
    const float s = (float)((vv - d.kv[nv + d.q]) * d.ihv[nv]);
    float V[ORDER + 1][K2];
    column_powers<K2, ORDER>(s, V);
    const size_t npts = (size_t)nua * nvb, kk = (size_t)k1 * k2 * 4;
    float *dst = out + (size_t)a * nvb + b;
    Hom<float> Y[K1][ORDER + 1];
    int cur = -1;
    double lo = 0, hi = 0, ih = 0;  // the span the lane's rows are in
    while (true) {
        const double uu = (double)un;
        const int next = a + G;
        if (next < a1) un = us[next];
        if (!(uu > lo && uu < hi)) {
            const int m = find_span_near(d.ku, d.p, d.nu, uu) - d.p;
            lo = d.ku[m + d.p];
            hi = d.ku[m + d.p + 1];
            ih = d.ihu[m];
            if (m != cur) {
                cur = m;
                column_side<K1, K2, EXACT, ORDER>(d.tab32 + ((size_t)m * d.sv + nv) * kk, k1, k2, V, Y);
            }
        }
        Cart<float> o;
        row_side<K1, EXACT, ORDER>(Y, k1, (float)((uu - lo) * ih), (float)ih, ihv, o);
        store_point<ORDER>(o, dst, npts);
        if (next >= a1) break;
        a = next;
        dst += (size_t)G * nvb;
    }
}

struct GridLaunch {
    const GnSurfDev &d;
    const float *us;
    int nua;
    const float *vs;
    int nvb, order;
    float *out;
    hipStream_t st;
    template <int K1, int K2, bool EXACT>
    int strip() {
        // rows per lane: as many as leave two workgroups per CU (a lane's searches and its column's v side
        // are paid once; 100,000 x 4 points, order 0: 15 us at eight, 10 at two)
        const size_t G = kGridBlock / nvb, groups = ((size_t)nua + G - 1) / G;
        size_t per = groups / 512;
        per = per < 1 ? 1 : per > kGridRows ? kGridRows : per;
        const unsigned grid = (unsigned)((groups + per - 1) / per);
        const int r = (int)(G * per);
        if (order == 0) k_grid_strip<K1, K2, EXACT, 0><<<grid, kGridBlock, 0, st>>>(d, us, nua, vs, nvb, r, out);
        else if (order == 1) k_grid_strip<K1, K2, EXACT, 1><<<grid, kGridBlock, 0, st>>>(d, us, nua, vs, nvb, r, out);
        else k_grid_strip<K1, K2, EXACT, 2><<<grid, kGridBlock, 0, st>>>(d, us, nua, vs, nvb, r, out);
        GN_HIP(hipGetLastError());
        return GN_OK;
    }
    template <int K1, int K2, bool EXACT>
    int operator()() {
        if (nvb <= kStripCols) return strip<K1, K2, EXACT>();
        const size_t cols = ((size_t)nvb + kGridBlock - 1) / kGridBlock;
        // rows per workgroup: as many as leave about eight workgroups per CU, so that a small grid
        // still spreads over the chip and a large one amortises its span searches
        size_t rows = (size_t)nua * cols / 2048;
        rows = rows < 4 ? 4 : rows > kGridRows ? kGridRows : rows;
        const unsigned grid = (unsigned)(cols * (((size_t)nua + rows - 1) / rows));  // <= 2^30
        const int r = (int)rows;
        const unsigned cb = (unsigned)cols;
        if (order == 0) k_grid<K1, K2, EXACT, 0><<<grid, kGridBlock, 0, st>>>(d, us, nua, vs, nvb, r, cb, out);
        else if (order == 1) k_grid<K1, K2, EXACT, 1><<<grid, kGridBlock, 0, st>>>(d, us, nua, vs, nvb, r, cb, out);
        else k_grid<K1, K2, EXACT, 2><<<grid, kGridBlock, 0, st>>>(d, us, nua, vs, nvb, r, cb, out);
        GN_HIP(hipGetLastError());
        return GN_OK;
    }
};

int launch_eval_grid32(const GnSurfDev &d, const float *us, int nu_pts, const float *vs,
                       int nv_pts, int order, float *out, hipStream_t st) {
    if ((size_t)nu_pts * nv_pts == 0) return GN_OK;
    return dispatch_degrees(d.p, d.q, GridLaunch{d, us, nu_pts, vs, nv_pts, order, out, st});
}

}  // namespace gn

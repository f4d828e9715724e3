// LNCC similarity (reg_lncc) on gfx950.
//
// The measure needs Gaussian-weighted local statistics of both images over the combined mask
// (reference mask minus the NaN voxels of either image): five masked convolutions per value
// (ref, ref^2, warped, warped^2, ref*warped) and three more per gradient.  All of them share one
// density (the combined mask), so one set of separable passes carries the numerators and the
// density together: planar [K + 1][N] arrays, one launch per axis, ping-ponging between two
// buffers.  Each output sample is the reference's line sum in the reference's order (float
// products added in double, reg-lib/cpu/_reg_tools.cpp:1047-1053), so the results equal the
// reference's scalar build bit for bit.  That is the per-operation measure (op_lncc_value,
// op_lncc_voxel_gradient).  The evaluations take the passes at the end of the kernels below, which
// form the same sums in fewer trips to memory.

#include "f3d_handle.hpp"
#include "device.hpp"
#include <cmath>
#include <type_traits>

namespace nrh {

namespace {

constexpr int kB = 256;
constexpr int kRedBlocks = 1024;

unsigned blocks_of(size_t n) { return (unsigned)((n + kB - 1) / kB); }

// Combined mask and the numerators of the first convolution set, with the density last.
__global__ void __launch_bounds__(kB)
k_lncc_prepare(const float *__restrict__ ref, const float *__restrict__ war, const int *__restrict__ mask, size_t N,
               uint8_t *__restrict__ comb, float *__restrict__ A) {
#pragma clang fp contract(off)
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const float r = ref[i], w = war[i];
    const bool ok = (!mask || mask[i] > -1) && r == r && w == w;
    comb[i] = ok ? 1 : 0;
    A[i] = ok ? r : 0.f;
    A[N + i] = ok ? r * r : 0.f;
    A[2 * N + i] = ok ? w : 0.f;
    A[3 * N + i] = ok ? w * w : 0.f;
    A[4 * N + i] = ok ? r * w : 0.f;
    A[5 * N + i] = ok ? 1.f : 0.f;
}

// One separable pass of reg_tools_kernelConvolution along `axis` for K <= 6 planar arrays.  The K
// sums of a voxel advance together tap by tap (K independent FP64 chains in flight, each in the
// reference's tap order).
constexpr int kConvArrays = 6;

__global__ void __launch_bounds__(kB)
k_conv_axis(const float *__restrict__ in, float *__restrict__ out, int K, size_t N, int nx, int ny, int nz, int axis,
            const float *__restrict__ kern, int radius) {
#pragma clang fp contract(off)
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    int x, y, z;
    index_xyz(i, nx, ny, x, y, z);
    int l, L;
    size_t stride;
    if (axis == 0) { l = x; L = nx; stride = 1; }
    else if (axis == 1) { l = y; L = ny; stride = (size_t)nx; }
    else { l = z; L = nz; stride = (size_t)nx * ny; }
    int pre = l - radius, k0 = 0;
    const int pst = min(l + radius + 1, L);
    if (pre < 0) { k0 = -pre; pre = 0; }
    const size_t base = i - (size_t)l * stride;
    double acc[kConvArrays] = { 0.0, 0.0, 0.0, 0.0, 0.0, 0.0 };
    for (int k = pre, kk = k0; k < pst; ++k, ++kk) {
        const float kv = kern[kk];
        const float *src = in + base + (size_t)k * stride;
#pragma unroll
        for (int a = 0; a < kConvArrays; ++a)
            if (a < K) acc[a] += (double)(kv * src[(size_t)a * N]);
    }
#pragma unroll
    for (int a = 0; a < kConvArrays; ++a)
        if (a < K) out[(size_t)a * N + i] = (float)acc[a];
}

// Line-tiled passes.  A workgroup stages a stretch of lines (outputs plus `radius` samples on each
// side, zero outside the image) of one array at a time in LDS, so each input sample is fetched
// from memory about once per pass instead of once per tap.  Every output is still summed tap by
// tap in ascending order in double; the zero samples outside the line add +0 to a sum that starts
// at +0 and cannot become -0, so each sum equals the reference's over the in-range taps only.
constexpr int kLineOut = 64;      // outputs per workgroup along y or z (four waves of 16)
constexpr int kRowsX = 32;        // rows per workgroup for the x pass (four waves of 8)
constexpr int kMaxTileRadius = 96;

size_t lds_yz(int radius) { return (size_t)(kLineOut + 2 * radius) * 64 * sizeof(float); }
size_t lds_x(int radius) { return (size_t)kRowsX * (64 + 2 * radius) * sizeof(float); }

// y or z pass: 64 neighbouring x columns of one plane (blockIdx.y) and kLineOut positions of the
// line (blockIdx.z); LDS tile [kLineOut + 2 radius][64], lanes on x, conflict-free reads.
__global__ void __launch_bounds__(kB)
k_conv_lines_yz(const float *__restrict__ in, float *__restrict__ out, int K, size_t N, int nx, int L,
                size_t outerStride, size_t lineStride, const float *__restrict__ kern, int radius) {
#pragma clang fp contract(off)
    extern __shared__ float tile[];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int x = blockIdx.x * 64 + lane;
    const bool col = x < nx;
    const size_t base = (size_t)blockIdx.y * outerStride + (size_t)blockIdx.x * 64 + lane;
    const int t0 = blockIdx.z * kLineOut;
    const int rows = kLineOut + 2 * radius, taps = 2 * radius + 1;
    for (int a = 0; a < K; ++a) {
        const float *src = in + (size_t)a * N + base;
        for (int p = w; p < rows; p += kB / 64) {
            const int pos = t0 - radius + p;
            tile[p * 64 + lane] = col && pos >= 0 && pos < L ? src[(size_t)pos * lineStride] : 0.f;
        }
        __syncthreads();
        float *dst = out + (size_t)a * N + base;
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const int o0 = w * 16 + g * 8;
            const float *c = tile + o0 * 64 + lane;
            double acc[8] = { 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0 };
            for (int kk = 0; kk < taps; ++kk) {
                const float kv = kern[kk];
#pragma unroll
                for (int o = 0; o < 8; ++o) acc[o] += (double)(kv * c[(o + kk) * 64]);
            }
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                const int pos = t0 + o0 + o;
                if (col && pos < L) dst[(size_t)pos * lineStride] = (float)acc[o];
            }
        }
        __syncthreads();
    }
}

// x pass: kRowsX rows (row = y + ny z, blockIdx.x) and 64 outputs of each (blockIdx.y); LDS tile
// [kRowsX][64 + 2 radius], lanes on x.
__global__ void __launch_bounds__(kB)
k_conv_lines_x(const float *__restrict__ in, float *__restrict__ out, int K, size_t N, int nx, int nrows,
               const float *__restrict__ kern, int radius) {
#pragma clang fp contract(off)
    extern __shared__ float tile[];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int W = 64 + 2 * radius, taps = 2 * radius + 1;
    const int x0 = blockIdx.y * 64, row0 = blockIdx.x * kRowsX;
    for (int a = 0; a < K; ++a) {
        const float *src = in + (size_t)a * N;
        for (int idx = threadIdx.x; idx < kRowsX * W; idx += kB) {
            const int r = idx / W, p = idx - r * W;
            const int xx = x0 - radius + p, row = row0 + r;
            tile[idx] = xx >= 0 && xx < nx && row < nrows ? src[(size_t)row * nx + xx] : 0.f;
        }
        __syncthreads();
        const int r0 = w * (kRowsX / 4);
        const float *c = tile + r0 * W + lane;
        double acc[kRowsX / 4] = { 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0 };
        for (int kk = 0; kk < taps; ++kk) {
            const float kv = kern[kk];
#pragma unroll
            for (int r = 0; r < kRowsX / 4; ++r) acc[r] += (double)(kv * c[r * W + kk]);
        }
        float *dst = out + (size_t)a * N;
        const int x = x0 + lane;
#pragma unroll
        for (int r = 0; r < kRowsX / 4; ++r)
            if (x < nx && row0 + r0 + r < nrows) dst[(size_t)(row0 + r0 + r) * nx + x] = (float)acc[r];
        __syncthreads();
    }
}

// The local means and deviations of UpdateLocalStatImages (reg-lib/cpu/_reg_lncc.cpp:236-244) from a
// voxel's six convolved sums (ref, ref^2, warped, warped^2, ref * warped, density).
struct LocalStats {
    float mean, wmean, corr, sdev, wsdev;
};

__device__ __forceinline__ LocalStats local_stats(float r, float rr, float w, float ww, float rw, float d) {
#pragma clang fp contract(off)
    LocalStats s;
    s.mean = r / d;
    s.wmean = w / d;
    s.corr = rw / d;
    const float sq = rr / d, wsq = ww / d;
    s.sdev = sqrtf(sq - s.mean * s.mean);
    s.wsdev = sqrtf(wsq - s.wmean * s.wmean);
    if (s.sdev < 1.e-06) s.sdev = 0.f;
    if (s.wsdev < 1.e-06) s.wsdev = 0.f;
    return s;
}

// |local correlation| of reg_getLnccValue (:282-297); false where it is no number.
__device__ __forceinline__ bool lncc_value_term(const LocalStats& s, double& v) {
#pragma clang fp contract(off)
    const double l = (double)((s.corr - (s.mean * s.wmean)) / (s.sdev * s.wsdev));
    v = fabs(l);
    return l == l && !isinf(l);
}

// The three derivative terms of reg_getVoxelBasedLnccGradient (:441-470); false (and zero) where one
// is no number.
__device__ __forceinline__ bool lncc_gradient_terms(const LocalStats& s, float t[3]) {
#pragma clang fp contract(off)
    const double rm = s.mean, wm = s.wmean, rs = s.sdev, ws = s.wsdev;
    const double c = (double)s.corr - (rm * wm);
    double t1 = 1.0 / (rs * ws);
    double t2 = c / (rs * ws * ws * ws);
    double t3 = (c * wm) / (rs * ws * ws * ws) - rm / (rs * ws);
    t[0] = t[1] = t[2] = 0.f;
    if (!(t1 == t1 && !isinf(t1) && t2 == t2 && !isinf(t2) && t3 == t3 && !isinf(t3))) return false;
    if (c < 0) {
        t1 = -t1;
        t2 = -t2;
        t3 = -t3;
    }
    t[0] = (float)t1;
    t[1] = (float)t2;
    t[2] = (float)t3;
    return true;
}

// The value's terms (term(i, l): whether voxel i counts, and its l), reduced per block in a fixed order.
template<class Term>
__device__ __forceinline__ void value_partials(size_t N, Term term, double *__restrict__ partSum,
                                               unsigned long long *__restrict__ partCnt) {
    __shared__ double sS[kB / 64];
    __shared__ unsigned long long sC[kB / 64];
    double sum = 0.0;
    unsigned long long cnt = 0;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (size_t)gridDim.x * blockDim.x) {
        double l;
        if (term(i, l)) {
            sum += l;
            ++cnt;
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        sum += __shfl_down(sum, off, 64);
        cnt += __shfl_down(cnt, off, 64);
    }
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) {
        sS[wv] = sum;
        sC[wv] = cnt;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        unsigned long long c = 0;
        for (int w = 0; w < kB / 64; ++w) {
            s += sS[w];
            c += sC[w];
        }
        partSum[blockIdx.x] = s;
        partCnt[blockIdx.x] = c;
    }
}

__global__ void __launch_bounds__(kB)
k_lncc_value(const float *__restrict__ C, const uint8_t *__restrict__ comb, size_t N, double *__restrict__ partSum,
             unsigned long long *__restrict__ partCnt) {
    value_partials(
        N,
        [&](size_t i, double& l) {
            return comb[i] &&
                   lncc_value_term(local_stats(C[i], C[N + i], C[2 * N + i], C[3 * N + i], C[4 * N + i], C[5 * N + i]), l);
        },
        partSum, partCnt);
}

// Sum of the block partials in block order; out[0] = sum / count, out[1] = count.
__global__ void k_lncc_finish(const double *__restrict__ partSum, const unsigned long long *__restrict__ partCnt,
                              int nb, double *__restrict__ out) {
    // one wave: lane l sums its run of partials in order, then a fixed tree over the lanes
    const int l = threadIdx.x, per = (nb + 63) / 64;
    double s = 0.0;
    unsigned long long c = 0;
    for (int k = 0; k < per; ++k) {
        const int b = l * per + k;
        if (b < nb) {
            s += partSum[b];
            c += partCnt[b];
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        s += __shfl_down(s, off, 64);
        c += __shfl_down(c, off, 64);
    }
    if (l == 0) {
        out[0] = s / (double)c;
        out[1] = (double)c;
    }
}

// The three per-voxel derivative terms, written as
// the numerators of the second convolution set (density last), and the active-voxel count.
__global__ void __launch_bounds__(kB)
k_lncc_terms(const float *__restrict__ C, const uint8_t *__restrict__ comb, size_t N, float *__restrict__ T,
             unsigned long long *__restrict__ partCnt) {
#pragma clang fp contract(off)
    __shared__ unsigned long long sC[kB / 64];
    unsigned long long cnt = 0;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (size_t)gridDim.x * blockDim.x) {
        float t[3] = { 0.f, 0.f, 0.f };
        if (comb[i] &&
            lncc_gradient_terms(local_stats(C[i], C[N + i], C[2 * N + i], C[3 * N + i], C[4 * N + i], C[5 * N + i]), t))
            ++cnt;
        T[i] = t[0];
        T[N + i] = t[1];
        T[2 * N + i] = t[2];
        T[3 * N + i] = comb[i] ? 1.f : 0.f;
    }
    for (int off = 32; off > 0; off >>= 1) cnt += __shfl_down(cnt, off, 64);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) sC[wv] = cnt;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long c = 0;
        for (int w = 0; w < kB / 64; ++w) c += sC[w];
        partCnt[blockIdx.x] = c;
    }
}

__global__ void k_lncc_weight(const unsigned long long *__restrict__ partCnt, int nb, double weight,
                              double *__restrict__ out) {
    unsigned long long c = 0;
    for (int b = threadIdx.x; b < nb; b += 64) c += partCnt[b];
    for (int off = 32; off > 0; off >>= 1) c += __shfl_down(c, off, 64);
    if (threadIdx.x == 0) out[0] = weight / (double)c;
}

// grad -= warped gradient * (T1 ref - T2 war + T3) * adjusted weight (:486-500), then non-finite
// entries of every component set to 0 (:502-511).
__global__ void __launch_bounds__(kB)
k_lncc_apply(const float *__restrict__ T, const uint8_t *__restrict__ comb, const float *__restrict__ ref,
             const float *__restrict__ war, const float *__restrict__ wgrad, const double *__restrict__ adjusted,
             size_t N, float *__restrict__ grad) {
#pragma clang fp contract(off)
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const double aw = adjusted[0];
    if (comb[i]) {
        const float d = T[3 * N + i];
        const float t1 = T[i] / d, t2 = T[N + i] / d, t3 = T[2 * N + i] / d;
        const double common = (double)(t1 * ref[i] - t2 * war[i] + t3) * aw;
        for (int c = 0; c < 3; ++c) grad[c * N + i] -= (float)((double)wgrad[c * N + i] * common);
    }
    for (int c = 0; c < 3; ++c) {
        const float v = grad[c * N + i];
        if (v != v || isinf(v)) grad[c * N + i] = 0.f;
    }
}

// ------------------------------------------------------------------ evaluation passes
// The evaluations' convolutions: the sums of the per-operation passes, product by product, in fewer
// trips to memory.  The x pass forms the six numerators from the two images as it stages them, with a
// sliding window of samples in registers for eight neighbouring outputs, and the z pass ends in the value's
// or the derivative's terms, so that the six arrays cross memory four times instead of ten.  The value's
// terms, one array, are added in the per-operation order by a pass of their own (20 us).
// At 256 x 256 x 160, sigma 5 voxels (31 taps): the x, y and z passes of the six sums take 225, 219 and
// 278 us (with the derivative's terms 305), about 300 each by the per-operation passes, with a preparing
// and a reducing pass of 52 and 70 us; the derivative's three arrays 109, 110 and 152 us.  A tap is a
// float product, its widening and an addition in double: bound by these.  Two shifts of the product's bits
// in place of the widening, 2^-896 scaled, took longer (281, about 305 and 314 us).  Fused multiply-adds
// in double took 137, 175 and 205 us, but an unrounded product moves the node gradient by 1e-4.
// Radii above take the per-operation passes.  The x pass stages two samples of a row a lane, 64 outputs and
// the radius on each side; 30 is a sigma of 10 voxels, whose tiles take 25 KB (x) and 23.5 KB of LDS.
constexpr int kEvalRadius = 30;
static_assert(64 + 2 * kEvalRadius <= 128, "a row's samples are two a lane");
constexpr int kColOut = 32;      // outputs along y / z per workgroup: four waves of 8
constexpr int kEvalRows = 32;    // rows per workgroup of the x pass

size_t eval_lds_cols(int radius) { return (size_t)(kColOut + 2 * radius) * 64 * sizeof(float); }
// x rows: chunk k of a row starts at 9 k (the ninth unused), rows at a stride of 1 modulo 64: the
// 8 segments of 8 neighbouring rows then read distinct banks but for seven.  8 outputs over `taps`
// taps touch taps / 8 + 2 chunks
__host__ __device__ constexpr int eval_row_stride(int taps) { return (9 * (9 + taps / 8) + 62) / 64 * 64 + 1; }
size_t eval_lds_rows(int radius) { return (size_t)kEvalRows * eval_row_stride(2 * radius + 1) * sizeof(float); }

// out[o] = sum_k (double)(kern[k] s[o + k]), o < 8, in ascending k.  Column: sample p at base[64 p],
// which the lanes read without conflicts, so a tap reads its eight samples.
__device__ __forceinline__ void conv8_column(const float *base, const float *__restrict__ kern, int taps,
                                             float (&out)[8]) {
#pragma clang fp contract(off)
    double acc[8] = { 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0 };
    for (int k = 0; k < taps; ++k) {
        const float kv = kern[k];
#pragma unroll
        for (int o = 0; o < 8; ++o) acc[o] += (double)(kv * base[(o + k) * 64]);
    }
#pragma unroll
    for (int o = 0; o < 8; ++o) out[o] = (float)acc[o];
}

// The same along a row in chunks of 8 samples, sample 8 c + e at base[9 c + e], from a window of 16 in
// registers.  Samples past o + k = 7 + taps - 1 are loaded, not used.
__device__ __forceinline__ void conv8_row(const float *base, const float *__restrict__ kern, int taps, float (&out)[8]) {
#pragma clang fp contract(off)
    float w[16];
    double acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        w[e] = base[e];
        acc[e] = 0.0;
    }
    int c = 0;
    for (; 8 * c + 8 <= taps; ++c) {
#pragma unroll
        for (int e = 0; e < 8; ++e) w[8 + e] = base[(c + 1) * 9 + e];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float kv = kern[8 * c + k];
#pragma unroll
            for (int o = 0; o < 8; ++o) acc[o] += (double)(kv * w[o + k]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = w[8 + e];
    }
    const int rest = taps - 8 * c;
    if (rest > 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) w[8 + e] = base[(c + 1) * 9 + e];
#pragma unroll
        for (int k = 0; k < 7; ++k)
            if (k < rest) {  // uniform
                const float kv = kern[8 * c + k];
#pragma unroll
                for (int o = 0; o < 8; ++o) acc[o] += (double)(kv * w[o + k]);
            }
    }
#pragma unroll
    for (int o = 0; o < 8; ++o) out[o] = (float)acc[o];
}

// x pass.  A lane takes 8 neighbouring outputs of one row (8 segments by 32 rows a workgroup).
// FIRST: the six numerators of k_lncc_prepare, formed from the images, and the combined mask; else
// array blockIdx.z of `in`.
template<bool FIRST>
__global__ void __launch_bounds__(kB)
k_eval_x(const float *__restrict__ ref, const float *__restrict__ war, const int *__restrict__ mask,
         const float *__restrict__ in, float *__restrict__ out, uint8_t *__restrict__ comb, size_t N, int nx, int nrows,
         const float *__restrict__ kern, int radius) {
#pragma clang fp contract(off)
    extern __shared__ float rowsF[];
    const int taps = 2 * radius + 1, W = 64 + 2 * radius, S = eval_row_stride(taps);
    const int x0 = blockIdx.y * 64, row0 = blockIdx.x * kEvalRows;
    // a wave stages every fourth row, a lane its samples `lane` and 64 + lane: every load in flight
    // before one is used, addresses clamped to the image
    constexpr int kEl = kEvalRows / (kB / 64);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float a[kEl][2], b[kEl][2];
    bool ok[kEl][2];
#pragma unroll
    for (int e = 0; e < kEl; ++e)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int p = lane + 64 * h, x = x0 - radius + p, row = row0 + w + e * (kB / 64);
            ok[e][h] = p < W && x >= 0 && x < nx && row < nrows;
            const size_t i = (size_t)min(row, nrows - 1) * nx + min(max(x, 0), nx - 1);
            if (FIRST) {
                a[e][h] = ref[i];
                b[e][h] = war[i];
                if (mask) ok[e][h] = ok[e][h] && mask[i] > -1;
            } else {
                a[e][h] = in[blockIdx.z * N + i];
            }
        }
    if (FIRST) {
#pragma unroll
        for (int e = 0; e < kEl; ++e)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int p = lane + 64 * h, x = x0 - radius + p, row = row0 + w + e * (kB / 64);
                ok[e][h] = ok[e][h] && a[e][h] == a[e][h] && b[e][h] == b[e][h];
                if (p >= radius && p < radius + 64 && x < nx && row < nrows)
                    comb[(size_t)row * nx + x] = ok[e][h] ? 1 : 0;
            }
    }
    const int seg = threadIdx.x & 7, r = threadIdx.x >> 3, row = row0 + r, x = x0 + 8 * seg;
    const int at0 = (lane >> 3) * 9 + (lane & 7);
    for (int q = 0; q < (FIRST ? 6 : 1); ++q) {
#pragma unroll
        for (int e = 0; e < kEl; ++e)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float u = a[e][h], t = b[e][h];
                const float v = !FIRST ? u : q == 0 ? u : q == 1 ? u * u : q == 2 ? t : q == 3 ? t * t : q == 4 ? u * t : 1.f;
                if (lane + 64 * h < W) rowsF[(w + e * (kB / 64)) * S + at0 + 72 * h] = ok[e][h] ? v : 0.f;
            }
        __syncthreads();
        float acc[8];
        conv8_row(rowsF + r * S + 9 * seg, kern, taps, acc);
        float *dst = out + (size_t)(FIRST ? q : blockIdx.z) * N + (size_t)row * nx + x;
        if (row < nrows && x + 8 <= nx) {
            // two 16-byte stores (4-byte aligned)
            typedef float Float4 __attribute__((ext_vector_type(4), aligned(4)));
            *reinterpret_cast<Float4 *>(dst) = Float4{ acc[0], acc[1], acc[2], acc[3] };
            *reinterpret_cast<Float4 *>(dst + 4) = Float4{ acc[4], acc[5], acc[6], acc[7] };
        } else {
#pragma unroll
            for (int o = 0; o < 8; ++o)
                if (row < nrows && x + o < nx) dst[o] = acc[o];
        }
        __syncthreads();
    }
}

// Columns of a y or z pass: column c of the flattened (x, outer) pairs starts at
// c % nx + (c / nx) * outerStride, so a workgroup's 64 lanes are full whatever nx is.
struct Columns {
    size_t count, outerStride, lineStride;
    int nx, L;
};

__device__ __forceinline__ size_t column_base(const Columns& c, size_t col) {
    // (the column number fits 32 bits: an image of 2^32 columns has no room for its six arrays)
    const uint32_t outer = (uint32_t)col / (uint32_t)c.nx;
    return ((uint32_t)col - outer * (uint32_t)c.nx) + (size_t)outer * c.outerStride;
}

// One array's tile of 64 columns, positions t0 - radius ..: loaded (every load in flight before one is
// used, addresses clamped to the line), then stored into LDS with zeros outside the line.  A pass
// over several arrays loads the next while it sums the last.
constexpr int kStage = (kColOut + 2 * kEvalRadius + kB / 64 - 1) / (kB / 64);

__device__ __forceinline__ void load_columns(const float *__restrict__ src, const Columns& c, int t0, int radius,
                                             float (&v)[kStage]) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), rows = kColOut + 2 * radius;
#pragma unroll
    for (int u = 0; u < kStage; ++u) {
        const int p = w + u * (kB / 64);
        if (p < rows) v[u] = src[(size_t)min(max(t0 - radius + p, 0), c.L - 1) * c.lineStride];
    }
}

__device__ __forceinline__ void store_columns(const float (&v)[kStage], const Columns& c, bool col, int t0, int radius,
                                              float *tile) {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rows = kColOut + 2 * radius;
#pragma unroll
    for (int u = 0; u < kStage; ++u) {
        const int p = w + u * (kB / 64), pos = t0 - radius + p;
        if (p < rows) tile[p * 64 + lane] = col && pos >= 0 && pos < c.L ? v[u] : 0.f;
    }
}

// y pass of array blockIdx.z.
__global__ void __launch_bounds__(kB)
k_eval_cols(const float *__restrict__ in, float *__restrict__ out, size_t N, Columns c, const float *__restrict__ kern,
            int radius) {
    extern __shared__ float tileF[];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const size_t colIdx = (size_t)blockIdx.x * 64 + lane;
    const bool col = colIdx < c.count;
    const size_t base = blockIdx.z * N + column_base(c, col ? colIdx : 0);
    const int t0 = blockIdx.y * kColOut;
    float v[kStage];
    load_columns(in + base, c, t0, radius, v);
    store_columns(v, c, col, t0, radius, tileF);
    __syncthreads();
    float acc[8];
    conv8_column(tileF + w * 8 * 64 + lane, kern, 2 * radius + 1, acc);
#pragma unroll
    for (int o = 0; o < 8; ++o) {
        const int pos = t0 + w * 8 + o;
        if (col && pos < c.L) out[base + (size_t)pos * c.lineStride] = acc[o];
    }
}

// z pass of the six sums, ending in the value's terms (GRAD = false: in T, NaN where there is none) or the
// derivative's (GRAD = true: three arrays and the convolved density into T, and their number per block).
template<bool GRAD>
__global__ void __launch_bounds__(kB)
k_eval_stats(const float *__restrict__ in, const uint8_t *__restrict__ comb, size_t N, Columns c,
             const float *__restrict__ kern, int radius, float *__restrict__ T,
             unsigned long long *__restrict__ partCnt) {
    extern __shared__ float tileF[];
    __shared__ unsigned long long sC[kB / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const size_t colIdx = (size_t)blockIdx.x * 64 + lane;
    const bool col = colIdx < c.count;
    const size_t base = column_base(c, col ? colIdx : 0);
    const int t0 = blockIdx.y * kColOut;
    float sum[6][8], v[kStage];
    load_columns(in + base, c, t0, radius, v);
    // one call an array: unrolled, so that the sums stay in registers
    auto array = [&](auto q) __attribute__((always_inline)) {
        store_columns(v, c, col, t0, radius, tileF);
        __syncthreads();
        if (q < 5) load_columns(in + (q + 1) * N + base, c, t0, radius, v);
        conv8_column(tileF + w * 8 * 64 + lane, kern, 2 * radius + 1, sum[q]);
        __syncthreads();
    };
    array(std::integral_constant<int, 0>{});
    array(std::integral_constant<int, 1>{});
    array(std::integral_constant<int, 2>{});
    array(std::integral_constant<int, 3>{});
    array(std::integral_constant<int, 4>{});
    array(std::integral_constant<int, 5>{});
    unsigned long long cnt = 0;
#pragma unroll
    for (int o = 0; o < 8; ++o) {
        const int pos = t0 + w * 8 + o;
        if (!(col && pos < c.L)) continue;
        const size_t i = base + (size_t)pos * c.lineStride;
        const bool used = comb[i] != 0;
        const LocalStats st = local_stats(sum[0][o], sum[1][o], sum[2][o], sum[3][o], sum[4][o], sum[5][o]);
        if (GRAD) {
            float t[3] = { 0.f, 0.f, 0.f };
            if (used && lncc_gradient_terms(st, t)) ++cnt;
            T[i] = t[0];
            T[N + i] = t[1];
            T[2 * N + i] = t[2];
            T[3 * N + i] = sum[5][o];
        } else {
            double l;
            T[i] = used && lncc_value_term(st, l) ? (float)l : __builtin_nanf("");  // l is a float's value
        }
    }
    if (!GRAD) return;
    for (int off = 32; off > 0; off >>= 1) cnt += __shfl_down(cnt, off, 64);
    if (lane == 0) sC[w] = cnt;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < kB / 64; ++k) cnt += sC[k];
        partCnt[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = cnt;
    }
}

// The value's partials from the z pass's terms, in k_lncc_value's order.
__global__ void __launch_bounds__(kB)
k_eval_value(const float *__restrict__ T, size_t N, double *__restrict__ partSum, unsigned long long *__restrict__ partCnt) {
    value_partials(
        N,
        [&](size_t i, double& l) {
            l = (double)T[i];
            return l == l;
        },
        partSum, partCnt);
}

// z pass of the three derivative arrays, ending in k_lncc_apply's voxel gradient, which is written
// (not added to); the density is the one of the six sums, convolved already.
__global__ void __launch_bounds__(kB)
k_eval_apply(const float *__restrict__ in, const uint8_t *__restrict__ comb, const float *__restrict__ dens, size_t N,
             Columns c, const float *__restrict__ kern, int radius, const float *__restrict__ ref,
             const float *__restrict__ war, const float *__restrict__ wgrad, const double *__restrict__ adjusted,
             float *__restrict__ grad) {
#pragma clang fp contract(off)
    extern __shared__ float tileF[];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const size_t colIdx = (size_t)blockIdx.x * 64 + lane;
    const bool col = colIdx < c.count;
    const size_t base = column_base(c, col ? colIdx : 0);
    const int t0 = blockIdx.y * kColOut;
    float sum[3][8], v[kStage];
    load_columns(in + base, c, t0, radius, v);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        store_columns(v, c, col, t0, radius, tileF);
        __syncthreads();
        if (q < 2) load_columns(in + (q + 1) * N + base, c, t0, radius, v);
        conv8_column(tileF + w * 8 * 64 + lane, kern, 2 * radius + 1, sum[q]);
        __syncthreads();
    }
    const double aw = adjusted[0];
#pragma unroll
    for (int o = 0; o < 8; ++o) {
        const int pos = t0 + w * 8 + o;
        if (!(col && pos < c.L)) continue;
        const size_t i = base + (size_t)pos * c.lineStride;
        float g[3] = { 0.f, 0.f, 0.f };
        if (comb[i]) {
            const float d = dens[i];
            const float t1 = sum[0][o] / d, t2 = sum[1][o] / d, t3 = sum[2][o] / d;
            const double common = (double)(t1 * ref[i] - t2 * war[i] + t3) * aw;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const float v = 0.f - (float)((double)wgrad[k * N + i] * common);
                g[k] = v != v || isinf(v) ? 0.f : v;
            }
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) grad[k * N + i] = g[k];
    }
}

// The gradient's weight over the number of terms, one workgroup of 1024.
__global__ void __launch_bounds__(1024)
k_eval_weight(const unsigned long long *__restrict__ partCnt, int nb, double weight, double *__restrict__ out) {
    __shared__ double red[16];
    double n = 0.0;  // counts below 2^53 add exactly
    for (int b = threadIdx.x; b < nb; b += 1024) n += (double)partCnt[b];
    n = block_sum_double(n, red);
    if (threadIdx.x == 0) out[0] = weight / n;
}

// Gaussian kernel of reg_tools_kernelConvolution (:866-901); returns the radius.
int gaussian_kernel(float sigma, float pixdim, std::vector<float>& k) {
    const double temp = sigma > 0 ? (double)(sigma / pixdim) : std::fabs((double)sigma);
    const int radius = (int)(temp * 3.0f);
    k.assign(2 * std::max(radius, 0) + 1, 0.f);
    for (int i = -radius; i <= radius; ++i)
        k[i + radius] = (float)(std::exp(-(double)(i * i) / (2.0 * (temp * temp))) / (temp * 2.506628274631));
    return radius;
}

// columns and lines of the evaluation's z pass
Columns z_columns(const nrh_f3d *h) {
    const size_t plane = (size_t)h->ref.nx * h->ref.ny;
    return { plane, (size_t)h->ref.nx, plane, h->ref.nx, h->ref.nz };
}
dim3 column_grid(const Columns& c, unsigned arrays) {
    return dim3((unsigned)((c.count + 63) / 64), (unsigned)((c.L + kColOut - 1) / kColOut), arrays);
}
size_t eval_blocks(const nrh_f3d *h) {
    const dim3 g = column_grid(z_columns(h), 1);
    return (size_t)g.x * g.y;
}

void ensure_lncc(nrh_f3d *h) {
    const size_t N = h->N;
    h->lnccA.alloc(6 * N);
    h->lnccB.alloc(6 * N);
    h->lnccComb.alloc(N);
    // partial sums and counts: the per-operation measure's blocks, or the evaluation's z-pass blocks
    h->lnccPart.alloc(2 * std::max<size_t>(kRedBlocks, eval_blocks(h)));
    h->lnccScalars.alloc(4);
    if (h->lnccKern.empty() || h->lnccSigma != h->params.lncc_sigma) {
        std::vector<float> all;
        const float pix[3] = { h->ref.dx, h->ref.dy, h->ref.dz };
        for (int a = 0; a < 3; ++a) {
            std::vector<float> k;
            h->lnccRadius[a] = gaussian_kernel(h->params.lncc_sigma, pix[a], k);
            h->lnccKernOff[a] = (int)all.size();
            all.insert(all.end(), k.begin(), k.end());
        }
        all.push_back(1.f);  // the evaluations' kernel of an axis that is not smoothed
        h->lnccKern.alloc(all.size());
        NRH_HIP(hipMemcpyAsync(h->lnccKern.p, all.data(), all.size() * sizeof(float), hipMemcpyHostToDevice,
                               h->stream));
        NRH_HIP(hipStreamSynchronize(h->stream));
        h->lnccSigma = h->params.lncc_sigma;
    }
}

// Three axis passes over K + 1 planar arrays starting in `a`; returns the buffer holding the result.
float *convolve_set(nrh_f3d *h, float *a, float *b, int K1) {
    NRH_REQUIRE(K1 >= 1 && K1 <= kConvArrays, NRH_ERR_ARG, "at most six arrays per convolution pass");
    const int dims[3] = { h->ref.nx, h->ref.ny, h->ref.nz };
    float *src = a, *dst = b;
    for (int axis = 0; axis < 3; ++axis) {
        const int r = h->lnccRadius[axis];
        if (dims[axis] <= 1 || r <= 0) continue;
        const float *kern = h->lnccKern.p + h->lnccKernOff[axis];
        if (r > kMaxTileRadius) {
            hipLaunchKernelGGL(k_conv_axis, dim3(blocks_of(h->N)), dim3(kB), 0, h->stream, src, dst, K1, h->N,
                               dims[0], dims[1], dims[2], axis, kern, r);
        } else if (axis == 0) {
            const int nrows = dims[1] * dims[2];
            hipLaunchKernelGGL(k_conv_lines_x, dim3((nrows + kRowsX - 1) / kRowsX, (dims[0] + 63) / 64),
                               dim3(kB), lds_x(r), h->stream, src, dst, K1, h->N, dims[0], nrows, kern, r);
        } else {
            const size_t plane = (size_t)dims[0] * dims[1];
            const int L = dims[axis], outer = axis == 1 ? dims[2] : dims[1];
            const size_t outerStride = axis == 1 ? plane : (size_t)dims[0];
            const size_t lineStride = axis == 1 ? (size_t)dims[0] : plane;
            hipLaunchKernelGGL(k_conv_lines_yz, dim3((dims[0] + 63) / 64, outer, (L + kLineOut - 1) / kLineOut),
                               dim3(kB), lds_yz(r), h->stream, src, dst, K1, h->N, dims[0], L, outerStride,
                               lineStride, kern, r);
        }
        NRH_HIP(hipGetLastError());
        std::swap(src, dst);
    }
    return src;
}

float *lncc_statistics(nrh_f3d *h) {
    NRH_REQUIRE(!h->warped.empty(), NRH_ERR_STATE, "LNCC needs the warped image");
    ensure_lncc(h);
    h->evalVersion = 0;  // the evaluation's sums are overwritten
    hipLaunchKernelGGL(k_lncc_prepare, dim3(blocks_of(h->N)), dim3(kB), 0, h->stream, ref_ptr(h), h->warped.p,
                       h->mask.p, h->N, h->lnccComb.p, h->lnccA.p);
    NRH_HIP(hipGetLastError());
    return convolve_set(h, h->lnccA.p, h->lnccB.p, 6);
}

// Radius and kernel of one axis of the evaluation's passes: an axis that is not smoothed has the
// single tap 1.
int eval_axis(const nrh_f3d *h, int axis, const float **kern) {
    const int dims[3] = { h->ref.nx, h->ref.ny, h->ref.nz };
    const int r = h->lnccRadius[axis];
    if (dims[axis] <= 1 || r <= 0) {
        *kern = h->lnccKern.p + (h->lnccKern.n - 1);
        return 0;
    }
    *kern = h->lnccKern.p + h->lnccKernOff[axis];
    return r;
}

// The tiled passes hold lines with up to kEvalRadius voxels on each side.
bool eval_tiled(const nrh_f3d *h) {
    return h->lnccRadius[0] <= kEvalRadius && h->lnccRadius[1] <= kEvalRadius && h->lnccRadius[2] <= kEvalRadius;
}

// x then y pass of `arrays` planar arrays: in (null: the six numerators of the images) -> mid -> out.
void eval_xy(nrh_f3d *h, const float *in, float *mid, float *out, int arrays) {
    const int nx = h->ref.nx, ny = h->ref.ny, nz = h->ref.nz, nrows = ny * nz;
    const float *kern;
    int r = eval_axis(h, 0, &kern);
    const dim3 rows((nrows + kEvalRows - 1) / kEvalRows, (nx + 63) / 64, in ? arrays : 1);
    if (in)
        hipLaunchKernelGGL(k_eval_x<false>, rows, dim3(kB), eval_lds_rows(r), h->stream, nullptr, nullptr, nullptr, in, mid,
                           nullptr, h->N, nx, nrows, kern, r);
    else
        hipLaunchKernelGGL(k_eval_x<true>, rows, dim3(kB), eval_lds_rows(r), h->stream, ref_ptr(h), h->warped.p, h->mask.p,
                           nullptr, mid, h->lnccComb.p, h->N, nx, nrows, kern, r);
    NRH_HIP(hipGetLastError());
    r = eval_axis(h, 1, &kern);
    const Columns c{ (size_t)nx * nz, (size_t)nx * ny, (size_t)nx, nx, ny };
    hipLaunchKernelGGL(k_eval_cols, column_grid(c, arrays), dim3(kB), eval_lds_cols(r), h->stream, mid, out, h->N, c, kern,
                       r);
    NRH_HIP(hipGetLastError());
}

}  // namespace

void op_lncc_eval(nrh_f3d *h) {
    NRH_REQUIRE(!h->warped.empty(), NRH_ERR_STATE, "LNCC needs the warped image");
    ensure_lncc(h);
    if (eval_tiled(h)) eval_xy(h, nullptr, h->lnccA.p, h->lnccB.p, 6);  // in lnccB for the z pass
}

void op_lncc_eval_value(nrh_f3d *h, double *out_device) {
    if (!eval_tiled(h)) {
        const uint64_t keep = h->evalVersion;  // the warped image stays
        op_lncc_value(h, out_device);
        h->evalVersion = keep;
        return;
    }
    const float *kern;
    const int r = eval_axis(h, 2, &kern);
    const Columns c = z_columns(h);
    const dim3 grid = column_grid(c, 1);
    hipLaunchKernelGGL(k_eval_stats<false>, grid, dim3(kB), eval_lds_cols(r), h->stream, h->lnccB.p, h->lnccComb.p, h->N, c,
                       kern, r, h->lnccA.p, nullptr);
    NRH_HIP(hipGetLastError());
    const unsigned nb = std::min<unsigned>(blocks_of(h->N), kRedBlocks);
    double *ps = h->lnccPart.p;
    auto *pc = reinterpret_cast<unsigned long long *>(h->lnccPart.p + kRedBlocks);
    hipLaunchKernelGGL(k_eval_value, dim3(nb), dim3(kB), 0, h->stream, h->lnccA.p, h->N, ps, pc);
    NRH_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_lncc_finish, dim3(1), dim3(64), 0, h->stream, ps, pc, (int)nb, out_device);
    NRH_HIP(hipGetLastError());
}

void op_lncc_eval_voxel_gradient(nrh_f3d *h, double weight) {
    h->evalVersion = 0;  // the sums are used up
    if (!eval_tiled(h)) {
        zero_voxel_gradient(h);
        op_lncc_voxel_gradient(h, weight);
        return;
    }
    ensure_voxel_grad(h);
    h->voxelGradPending = false;
    NRH_REQUIRE(!h->warpedGrad.empty(), NRH_ERR_STATE, "LNCC gradient needs the warped image gradient");
    const float *kern;
    const int r = eval_axis(h, 2, &kern);
    const Columns c = z_columns(h);
    const dim3 grid = column_grid(c, 1);
    const int nb = (int)eval_blocks(h);
    auto *pc = reinterpret_cast<unsigned long long *>(h->lnccPart.p);
    float *T = h->lnccA.p, *dens = h->lnccA.p + 3 * h->N;
    hipLaunchKernelGGL(k_eval_stats<true>, grid, dim3(kB), eval_lds_cols(r), h->stream, h->lnccB.p, h->lnccComb.p, h->N, c,
                       kern, r, T, pc);
    NRH_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_eval_weight, dim3(1), dim3(1024), 0, h->stream, pc, nb, weight, h->lnccScalars.p);
    NRH_HIP(hipGetLastError());
    // the six sums are done with: their buffer takes the terms' x and y passes
    eval_xy(h, T, h->lnccB.p, h->lnccB.p + 3 * h->N, 3);
    hipLaunchKernelGGL(k_eval_apply, grid, dim3(kB), eval_lds_cols(r), h->stream, h->lnccB.p + 3 * h->N, h->lnccComb.p,
                       dens, h->N, c, kern, r, ref_ptr(h), h->warped.p, h->warpedGrad.p, h->lnccScalars.p,
                       h->voxelGrad.p);
    NRH_HIP(hipGetLastError());
}

void op_lncc_value(nrh_f3d *h, double *out_device) {
    const float *C = lncc_statistics(h);
    const unsigned nb = std::min<unsigned>(blocks_of(h->N), kRedBlocks);
    double *ps = h->lnccPart.p;
    auto *pc = reinterpret_cast<unsigned long long *>(h->lnccPart.p + kRedBlocks);
    hipLaunchKernelGGL(k_lncc_value, dim3(nb), dim3(kB), 0, h->stream, C, h->lnccComb.p, h->N, ps, pc);
    NRH_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_lncc_finish, dim3(1), dim3(64), 0, h->stream, ps, pc, (int)nb, out_device);
    NRH_HIP(hipGetLastError());
}

void op_lncc_voxel_gradient(nrh_f3d *h, double weight) {
    ensure_voxel_grad(h);
    NRH_REQUIRE(!h->warpedGrad.empty(), NRH_ERR_STATE, "LNCC gradient needs the warped image gradient");
    const float *C = lncc_statistics(h);
    float *T = (C == h->lnccA.p) ? h->lnccB.p : h->lnccA.p;
    const unsigned nb = std::min<unsigned>(blocks_of(h->N), kRedBlocks);
    auto *pc = reinterpret_cast<unsigned long long *>(h->lnccPart.p + kRedBlocks);
    hipLaunchKernelGGL(k_lncc_terms, dim3(nb), dim3(kB), 0, h->stream, C, h->lnccComb.p, h->N, T, pc);
    NRH_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_lncc_weight, dim3(1), dim3(64), 0, h->stream, pc, (int)nb, weight, h->lnccScalars.p);
    NRH_HIP(hipGetLastError());
    // the statistics buffer is free now: it becomes the ping-pong partner of the terms
    const float *S = convolve_set(h, T, const_cast<float *>(C), 4);
    hipLaunchKernelGGL(k_lncc_apply, dim3(blocks_of(h->N)), dim3(kB), 0, h->stream, S, h->lnccComb.p, ref_ptr(h),
                       h->warped.p, h->warpedGrad.p, h->lnccScalars.p, h->N, h->voxelGrad.p);
    NRH_HIP(hipGetLastError());
}

}  // namespace nrh

using namespace nrh;

extern "C" {

int nrh_f3d_lncc_value(nrh_f3d *h, double *value) {
    return guard([&] {
        NRH_REQUIRE(h && value, NRH_ERR_ARG, "null argument");
        ensure_lncc(h);
        op_lncc_value(h, h->lnccScalars.p + 2);
        *value = read_scalar(h, h->lnccScalars.p + 2);
    });
}

int nrh_f3d_lncc_voxel_gradient(nrh_f3d *h, double weight) {
    return guard([&] {
        NRH_REQUIRE(h, NRH_ERR_ARG, "null handle");
        settle_voxel_gradient(h);
        op_lncc_voxel_gradient(h, weight);
    });
}

}  // extern "C"

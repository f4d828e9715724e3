// Aladin (block-matching affine registration) on gfx950.
//
// One handle holds one pyramid level of reg_aladin (the HIP counterpart of AladinContent,
// reg-lib/AladinContent.cpp:6-29).  The per-iteration loop of reg_aladin::ResolveMatrix
// (reg-lib/_reg_aladin.cpp:302-313) is three launches on the handle's stream with the current
// matrix kept in device memory:
//   k_affine_warp   field = (A * ref.sto_xyz) * voxel in FP64, trilinear warp of the floating image
//   k_block_match   five active 4x4x4 blocks a workgroup, a lane per (y, z) of their capture offsets
//                   (few blocks: one, a lane per offset)
//   k_lts           one workgroup: compaction, FP64 moment fits, radix-select trimming
// Block variances for the active-block choice are computed on the device; their heap-sort
// ranking runs on the host because its tie order is part of the reference's result.

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <memory>
#include <vector>

#include "common.hpp"
#include <array>
#include <chrono>
#include <thread>
#include <map>
#include <mutex>
#include "device.hpp"
#include "recip_x87.hpp"
#include "m44.hpp"
#include "host.hpp"

struct nrh_aladin {
    nrh_geom ref{}, flo{};
    nrh_aladin_params params{};
    hipStream_t stream = nullptr;
    bool ownsStream = true;           // false when the stream is another handle's (symmetric pair)
    int device = 0;
    size_t N = 0, Nf = 0;
    nrh::DevBuf<float> refImg, floImg, warped;
    nrh::DevBuf<int> mask;  // empty: every voxel active
    int nb[3] = { 0, 0, 0 };
    int totalBlocks = 0, activeBlocks = 0;
    std::vector<int> totalBlock;      // _reg_blockMatchingParam::totalBlock
    nrh::DevBuf<int2> activeList;     // (block index, rank), in block order
    nrh::DevBuf<float> refPos, warpPos;
    nrh::DevBuf<float> matrix;        // current affine, 16 floats row-major
    nrh::DevBuf<int> counters;        // [0] defined blocks of the last matching, [1] LTS status,
                                      // [2] symmetric-update status
    nrh::DevBuf<float> ltsP, ltsQ;    // compacted correspondences
    nrh::DevBuf<uint32_t> ltsRes;     // residual bit patterns
    int *pinned = nullptr;            // 4 ints of host-visible status
};

namespace nrh {
namespace {

constexpr int kBlock = 256;
constexpr int kLtsThreads = 512;
constexpr int kLtsUnroll = 8;  // points per thread whose loads the LTS passes issue together

struct Mat4 {
    float m[16];
};

// The reference's products and sums in double; a product of two floats is exact there, so the fused
// multiply-adds round as its separate operations do.
template<class T>
__device__ __forceinline__ float3 mat44_mul_f(const T *m, float x, float y, float z) {
#pragma clang fp contract(off)
    const double X = (double)x, Y = (double)y, Z = (double)z;
    float3 r;
    r.x = (float)(fma((double)m[2], Z, fma((double)m[1], Y, (double)m[0] * X)) + (double)m[3]);
    r.y = (float)(fma((double)m[6], Z, fma((double)m[5], Y, (double)m[4] * X)) + (double)m[7]);
    r.z = (float)(fma((double)m[10], Z, fma((double)m[9], Y, (double)m[8] * X)) + (double)m[11]);
    return r;
}

// ------------------------------------------------------------------ active blocks
// Variance of each 4x4x4 block (reg-lib/cpu/_reg_blockMatching.cpp:70-128): the mean over finite
// voxels with mask > -1, the variance over every finite voxel, float sums in z, y, x order.
__global__ void __launch_bounds__(kBlock)
k_block_variance(const float *__restrict__ img, const int *__restrict__ mask, int nx, int ny, int nz, int nbx,
                 int nby, int nbz, float *__restrict__ var) {
#pragma clang fp contract(off)
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nbx * nby * nbz) return;
    const int bi = b % nbx, bj = (b / nbx) % nby, bk = b / (nbx * nby);
    const int x1 = min(4 * bi + 4, nx), y1 = min(4 * bj + 4, ny), z1 = min(4 * bk + 4, nz);
    float mean = 0.f, count = 0.f;
    for (int z = 4 * bk; z < z1; ++z)
        for (int y = 4 * bj; y < y1; ++y)
            for (int x = 4 * bi; x < x1; ++x) {
                const size_t i = ((size_t)z * ny + y) * nx + x;
                const float v = img[i];
                if (v == v && (!mask || mask[i] > -1)) {
                    mean += v;
                    count += 1.f;
                }
            }
    mean /= count;
    float variance = 0.f;
    for (int z = 4 * bk; z < z1; ++z)
        for (int y = 4 * bj; y < y1; ++y)
            for (int x = 4 * bi; x < x1; ++x) {
                const float v = img[((size_t)z * ny + y) * nx + x];
                if (v == v) variance += (mean - v) * (mean - v);
            }
    variance /= count;
    var[b] = (count > 32.f && variance > 0.f) ? variance : -1.f;
}

// Heap sort of values with a companion index, ascending: the Numerical-Recipes sift-down
// sequence of HeapSort(float*, int*, int) (reg-lib/cpu/Maths.cpp:114-153), whose order of equal
// values decides which of several equal-variance blocks are kept.
void heap_sort_indexed(std::vector<float>& v, std::vector<int>& ix) {
    const int n = (int)v.size();
    if (n < 2) return;
    float *a = v.data() - 1;
    int *id = ix.data() - 1;
    int l = (n >> 1) + 1, ir = n;
    for (;;) {
        float val;
        int iv;
        if (l > 1) {
            --l;
            val = a[l];
            iv = id[l];
        } else {
            val = a[ir];
            iv = id[ir];
            a[ir] = a[1];
            id[ir] = id[1];
            if (--ir == 1) {
                a[1] = val;
                id[1] = iv;
                return;
            }
        }
        int i = l, j = l + l;
        while (j <= ir) {
            if (j < ir && a[j] < a[j + 1]) ++j;
            if (!(val < a[j])) break;
            a[i] = a[j];
            id[i] = id[j];
            i = j;
            j <<= 1;
        }
        a[i] = val;
        id[i] = iv;
    }
}

// ------------------------------------------------------------------ affine warp
// reg_affine_deformationField3D (reg-lib/cpu/_reg_globalTrans.cpp:74-127): T = A * ref.sto_xyz
// (mat44 product with double sums, float entries), position = T * voxel in double, stored as
// float; then the trilinear resampling of that position (reg-lib/cpu/_reg_resampling.cpp:316-464).
__global__ void __launch_bounds__(kBlock)
k_affine_warp(const float *__restrict__ flo, int fnx, int fny, int fnz, Affine floIjk,
              const float *__restrict__ A, Mat4 refXyz, int nx, int ny, int nz, const int *__restrict__ mask,
              float pad, float *__restrict__ warped) {
#pragma clang fp contract(off)
    __shared__ double T[12];
    if (threadIdx.x < 12) {
        const int r = threadIdx.x >> 2, c = threadIdx.x & 3;
        const float t = (float)((double)A[r * 4 + 0] * (double)refXyz.m[c] +
                                (double)A[r * 4 + 1] * (double)refXyz.m[4 + c] +
                                (double)A[r * 4 + 2] * (double)refXyz.m[8 + c] +
                                (double)A[r * 4 + 3] * (double)refXyz.m[12 + c]);
        T[threadIdx.x] = (double)t;
    }
    __syncthreads();
    const size_t N = (size_t)nx * ny * nz;
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= N) return;
    if (mask && mask[idx] < 0) return;
    const double x = (double)(idx % nx), y = (double)((idx / nx) % ny), z = (double)(idx / ((size_t)nx * ny));
    const float fx = (float)(T[0] * x + T[1] * y + T[2] * z + T[3]);
    const float fy = (float)(T[4] * x + T[5] * y + T[6] * z + T[7]);
    const float fz = (float)(T[8] * x + T[9] * y + T[10] * z + T[11]);
    const float3 p = affine_apply_d(floIjk, fx, fy, fz);
    warped[idx] = sample_linear(flo, fnx, fny, fnz, p, pad);
}

// ------------------------------------------------------------------ block matching
// block_matching_method3D<float> (reg-lib/cpu/_reg_blockMatching.cpp:455-690).  A workgroup takes NB
// active blocks (neighbours: the list is in block order, as undefined values come in clusters); a lane
// takes one (m, n) of a block's 7 x 7 capture offsets along y and z and NX of the 7 along x: all 7, so
// that the 10 warped values of a row are read from LDS once for the 28 products that they enter, or one.
// Each offset runs the reference's two float passes (means, then variances and covariance) in voxel
// order; a wave per block then replays the sequential "cc > best -> best = cc + 1e-7" rule with ballots,
// which gives the same winner as the reference's scan over offsets (l, m, n) = (o % 7, o / 7 % 7, o / 49) - 3.
//
// Bound by vector instructions: 343 offsets x 64 voxels x 6 for a block whose values are all defined
// (its mean and variance are the same for every offset and come from one lane), 16 with a check of
// each value otherwise; a wave takes the short way when every block it works on allows.  One offset
// a lane, both checks always and an atomic per block on the count of defined blocks: 254 us for the
// 16384 blocks of 128^3; with NB = 5 (245 of 256 lanes) and NX = 7, 93 us (in rank order, which scatters
// the blocks with undefined values, and with the coordinates of each staged value found by division, 179
// us).  That many blocks keep the chip busy; few of them wait for one lane's seven offsets, 28 us however
// few, and go a block a workgroup of 384, an offset a lane (NB = NX = 1).  us by active blocks, 5 / 7 and
// 1 / 1: 256: 28, 10; 500: 28, 14; 1008: 28, 21; 1372: 28, 26; 2048: 30, 34; 4000: 39, 56.
constexpr int kMatchFew = 1536;

template<int NB, int NX>
struct MatchShape {
    static constexpr int kLanes = 49 * (7 / NX);  // of a block
    static constexpr int kThreads = (NB * kLanes + 63) / 64 * 64;
    static constexpr int kStage = NX == 7 ? 1 : 4;  // fifties of threads that stage a block
    static_assert(7 % NX == 0 && 50 * kStage * NB <= kThreads, "threads of a block");
};

template<int NB>
struct MatchShared {
    float W[NB][1000];    // warped values, 3 voxels around the block
    float R[NB][68];      // reference values (NaN: undefined or masked)
    float rt[NB][64];     // reference values less their mean (blocks without NaN)
    float rv[NB];         // and the sum of their squares
    float cc[NB][343];
    int rank[NB];
    int org[NB][3];       // first voxel
    int bad[NB];          // an undefined value among R or W
    int defined;
};

// The NX + 3 warped values of a row that NX offsets of 4 voxels take; all seven offsets' rows start on
// even indices: pairs are aligned.
template<int NX>
__device__ __forceinline__ void match_row(const float *p, float (&w)[NX + 3]) {
    if constexpr (NX == 7) {
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            const float2 v = *reinterpret_cast<const float2 *>(p + 2 * k);
            w[2 * k] = v.x;
            w[2 * k + 1] = v.y;
        }
    } else {
#pragma unroll
        for (int k = 0; k < NX + 3; ++k) w[k] = p[k];
    }
}

// cc of NX offsets along x from w0 (the first offset's first voxel), every value of the block and its
// surroundings defined.
template<int NX>
__device__ __forceinline__ void match_defined(const float *w0, const float *rts, float rv, float (&cc)[NX]) {
#pragma clang fp contract(off)
    float wm[NX] = {};
    for (int z = 0; z < 4; ++z)
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            float w[NX + 3];
            match_row<NX>(w0 + z * 100 + y * 10, w);
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int l = 0; l < NX; ++l) wm[l] += w[l + x];
        }
    float wv[NX] = {}, c[NX] = {};
#pragma unroll
    for (int l = 0; l < NX; ++l) wm[l] /= 64.f;
    for (int z = 0; z < 4; ++z)
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            float w[NX + 3];
            match_row<NX>(w0 + z * 100 + y * 10, w);
            const float4 r4 = *reinterpret_cast<const float4 *>(rts + z * 16 + y * 4);
            const float rt[4] = { r4.x, r4.y, r4.z, r4.w };
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int l = 0; l < NX; ++l) {
                    const float wt = w[l + x] - wm[l];
                    wv[l] += wt * wt;
                    c[l] += rt[x] * wt;
                }
        }
#pragma unroll
    for (int l = 0; l < NX; ++l) cc[l] = (rv * wv[l]) > 0.f ? fabsf(c[l] / sqrtf(rv * wv[l])) : 0.f;
}

// The same over the pairs whose two values are defined (an undefined one adds 0), more than 32 of them.
template<int NX>
__device__ __forceinline__ void match_checked(const float *w0, const float *R, float (&cc)[NX]) {
#pragma clang fp contract(off)
    // a row's values and which of them are defined: one comparison each, for all that they enter
    float w[NX + 3], r[4];
    bool wok[NX + 3], rok[4];
    auto row = [&](int q) {
        match_row<NX>(w0 + (q >> 2) * 100 + (q & 3) * 10, w);
        const float4 v = *reinterpret_cast<const float4 *>(R + q * 4);
        r[0] = v.x;
        r[1] = v.y;
        r[2] = v.z;
        r[3] = v.w;
#pragma unroll
        for (int k = 0; k < NX + 3; ++k) wok[k] = w[k] == w[k];
#pragma unroll
        for (int x = 0; x < 4; ++x) rok[x] = r[x] == r[x];
    };
    float rm[NX] = {}, wm[NX] = {}, cnt[NX] = {};
    for (int q = 0; q < 16; ++q) {
        row(q);
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int l = 0; l < NX; ++l) {
                const bool ok = rok[x] && wok[l + x];
                rm[l] += ok ? r[x] : 0.f;
                wm[l] += ok ? w[l + x] : 0.f;
                cnt[l] += ok ? 1.f : 0.f;
            }
    }
    float rv[NX] = {}, wv[NX] = {}, c[NX] = {};
#pragma unroll
    for (int l = 0; l < NX; ++l) {
        rm[l] /= cnt[l];
        wm[l] /= cnt[l];
    }
    for (int q = 0; q < 16; ++q) {
        row(q);
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int l = 0; l < NX; ++l) {
                const bool ok = rok[x] && wok[l + x];
                const float rt = ok ? r[x] - rm[l] : 0.f, wt = ok ? w[l + x] - wm[l] : 0.f;
                rv[l] += rt * rt;
                wv[l] += wt * wt;
                c[l] += rt * wt;
            }
    }
#pragma unroll
    for (int l = 0; l < NX; ++l) {
        const float v = (rv[l] * wv[l]) > 0.f ? fabsf(c[l] / sqrtf(rv[l] * wv[l])) : 0.f;
        cc[l] = cnt[l] > 32.f ? v : -1.f;
    }
}

template<int NB, int NX>
__global__ void __launch_bounds__((MatchShape<NB, NX>::kThreads))
k_block_match(const float *__restrict__ ref, const float *__restrict__ warped, const int *__restrict__ mask,
              int nx, int ny, int nz, int nbx, int nby, const int2 *__restrict__ activeList, int nActive, Affine xyz,
              float *__restrict__ refPos, float *__restrict__ warpPos, int *__restrict__ definedCount) {
#pragma clang fp contract(off)
    using Shape = MatchShape<NB, NX>;
    constexpr int kThreads = Shape::kThreads, kLanes = Shape::kLanes, kStage = Shape::kStage;
    __shared__ __align__(16) MatchShared<NB> S;
    const int t = threadIdx.x, first = blockIdx.x * NB, nb = min(NB, nActive - first);
    const float qnan = __builtin_nanf("");
    if (t < NB) {
        const int2 a = activeList[first + min(t, nb - 1)];  // blocks past the last repeat it, unused
        S.rank[t] = a.y;
        S.org[t][0] = 4 * (a.x % nbx);
        S.org[t][1] = 4 * ((a.x / nbx) % nby);
        S.org[t][2] = 4 * (a.x / (nbx * nby));
        S.bad[t] = 0;
    }
    if (t == 0) S.defined = 0;
    __syncthreads();
    {
        // the warped values first, all loads in flight before the first is stored: fifty r of a block's
        // threads takes the halves j kStage + r of its slices, columns (x, y) or (x, y + 5)
        const int wb = min(t / (50 * kStage), NB - 1), p = t % 50, r = t / 50 % kStage;
        const int x = S.org[wb][0] - 3 + p % 10, y = S.org[wb][1] - 3 + p / 10, z0 = S.org[wb][2] - 3;
        const bool in0 = x > -1 && x < nx && y > -1 && y < ny, in1 = x > -1 && x < nx && y + 5 > -1 && y + 5 < ny;
        const float *c0 = warped + (in0 ? (size_t)y * nx + x : 0), *c1 = warped + (in1 ? (size_t)(y + 5) * nx + x : 0);
        const size_t slice = (size_t)nx * ny;
        constexpr int kLoads = 20 / kStage;
        float v[kLoads];
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int h = j * kStage + r, zj = z0 + (h >> 1);
            const int z = min(max(zj, 0), nz - 1);
            v[j] = (h & 1 ? c1 : c0)[z * slice];
            if (!(h & 1 ? in1 : in0) || z != zj) v[j] = qnan;
        }
        for (int i = t; i < NB * 64; i += kThreads) {
            const int blk = i >> 6, a = i & 63;
            const int rx = S.org[blk][0] + (a & 3), ry = S.org[blk][1] + ((a >> 2) & 3), rz = S.org[blk][2] + (a >> 4);
            float r = qnan;
            if (rx < nx && ry < ny && rz < nz) {
                const size_t k = ((size_t)rz * ny + ry) * nx + rx;
                if (!mask || mask[k] > -1) r = ref[k];
            }
            S.R[blk][a] = r;
            if (!(r == r)) S.bad[blk] = 1;
        }
        if (t < 50 * kStage * NB) {
            bool bad = false;
#pragma unroll
            for (int j = 0; j < kLoads; ++j) {
                S.W[wb][(j * kStage + r) * 50 + p] = v[j];
                bad = bad || !(v[j] == v[j]);
            }
            if (bad) S.bad[wb] = 1;
        }
    }
    __syncthreads();
    if (t < NB && !S.bad[t]) {
        const float *R = S.R[t];
        float rm = 0.f, rv = 0.f;
#pragma unroll 16
        for (int a = 0; a < 64; ++a) rm += R[a];
        rm /= 64.f;
#pragma unroll 16
        for (int a = 0; a < 64; ++a) {
            const float rt = R[a] - rm;
            S.rt[t][a] = rt;
            rv += rt * rt;
        }
        S.rv[t] = rv;
    }
    __syncthreads();
    {
        constexpr int kX = 7 / NX;  // lanes along x
        const int blk = min(t / kLanes, NB - 1), o = t - t / kLanes * kLanes;
        const int l0 = o % kX * NX, m = o / kX % 7, n = o / (7 * kX);
        const float *w0 = S.W[blk] + n * 100 + m * 10 + l0;
        float cc[NX];
        if (__any(S.bad[blk])) match_checked<NX>(w0, S.R[blk], cc);
        else match_defined<NX>(w0, S.rt[blk], S.rv[blk], cc);
        if (t < NB * kLanes)
            for (int l = 0; l < NX; ++l) S.cc[blk][n * 49 + m * 7 + l0 + l] = cc[l];
    }
    __syncthreads();
    for (int blk = t >> 6; blk < nb; blk += kThreads / 64) {
        const int lane = t & 63;
        float best = 0.f;
        int win = -1;
        for (int c = 0; c < (343 + 63) / 64; ++c) {
            const int o = c * 64 + lane;
            const float v = o < 343 ? S.cc[blk][o] : -1.f;
            unsigned long long mk = __ballot(v > best);
            while (mk) {
                const int f = __ffsll((long long)mk) - 1;
                best = __shfl(v, f, 64) + 1.0e-7f;
                win = c * 64 + f;
                mk = __ballot(v > best && lane > f);
            }
        }
        if (lane != 0) continue;
        const int rank = S.rank[blk];
        const float cx = (float)S.org[blk][0], cy = (float)S.org[blk][1], cz = (float)S.org[blk][2];
        float dx = qnan, dy = 0.f, dz = 0.f;
        if (win >= 0) {
            dx = (float)(win % 7 - 3);
            dy = (float)((win / 7) % 7 - 3);
            dz = (float)(win / 49 - 3);
            atomicAdd(&S.defined, 1);
        }
        dx += cx;
        dy += cy;
        dz += cz;
        const float3 rp = affine_apply_d(xyz, cx, cy, cz);
        const float3 wp = affine_apply_d(xyz, dx, dy, dz);
        refPos[3 * rank + 0] = rp.x;
        refPos[3 * rank + 1] = rp.y;
        refPos[3 * rank + 2] = rp.z;
        warpPos[3 * rank + 0] = wp.x;
        warpPos[3 * rank + 1] = wp.y;
        warpPos[3 * rank + 2] = wp.z;
    }
    __syncthreads();
    if (t == 0 && S.defined > 0) atomicAdd(definedCount, S.defined);
}

// ------------------------------------------------------------------ LTS
// Four words of padding after every 32: the lanes of the wave that selects each read 32 of the
// histogram's, which without it lie in the same banks for all.
__device__ __forceinline__ uint32_t lts_bin(uint32_t b) { return b + ((b >> 5) << 2); }

template<int NT>
struct alignas(16) LtsShared {
    double red[NT / 64][24];
    double out[24];
    double kept[24];  // the kept points' sums: p, q, count, p_a p_b (00 01 02 11 12 22), p_a q_b
    double fit[21];   // the fit's centred moments and means
    uint32_t hist[2048 + 256];                  // bin b at lts_bin(b)
    uint32_t list[NT / 64][128];                // per wave: points that enter or leave the kept set
    int wave[kLtsUnroll][NT / 64];
    float M[16], last[16];
    int scal[4];
};

template<int CTRL>
__device__ __forceinline__ double dpp_double(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

__device__ __forceinline__ double uniform_double(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b), hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

// a + b over the pairs of lanes that differ in bit 5 (ROWS: bit 4): the lanes with the bit clear get
// a's sum, the others b's.
template<bool ROWS>
__device__ __forceinline__ double swap_add(double a, double b) {
    const unsigned long long ua = (unsigned long long)__double_as_longlong(a);
    const unsigned long long ub = (unsigned long long)__double_as_longlong(b);
    auto swap = [](uint32_t x, uint32_t y) {
        if constexpr (ROWS) return __builtin_amdgcn_permlane16_swap(x, y, false, false);
        else return __builtin_amdgcn_permlane32_swap(x, y, false, false);
    };
    const auto lo = swap((uint32_t)ua, (uint32_t)ub), hi = swap((uint32_t)(ua >> 32), (uint32_t)(ub >> 32));
    return __longlong_as_double((long long)((unsigned long long)hi[0] << 32 | lo[0])) +
           __longlong_as_double((long long)((unsigned long long)hi[1] << 32 | lo[1]));
}

// Sum of K doubles over the workgroup in a fixed order; the result lands in s.out[0..K).
// Inside a wave the values are halved at each exchange: the lanes whose exchange bit is clear keep
// the lower half of the (zero-padded, power-of-two) set and send the upper half, the others the
// reverse, so the wave makes W/2 + W/4 + ... + 1 exchanges instead of K per lane bit; after log2 W
// of them lane l holds value (l >> (6 - log2 W)) summed over its group, and the remaining lane bits
// are summed by plain exchanges.  The exchanges are lane swaps and data-parallel moves (lane l with
// l ^ 32, l ^ 16, l ^ 8, 7 - l of its eight, l ^ 2, l ^ 1): through LDS, 16 waves took 4800 cycles
// for 23 values.
template<int K, int NT>
__device__ void wg_sum(double (&v)[K], LtsShared<NT>& s) {
    static_assert(K <= 32, "at most 32 values");
    constexpr int W = K <= 8 ? 8 : K <= 16 ? 16 : 32;
    constexpr int LW = W == 8 ? 3 : W == 16 ? 4 : 5;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    double a[W];
#pragma unroll
    for (int k = 0; k < W; ++k) a[k] = k < K ? v[k] : 0.0;
#pragma unroll
    for (int j = 0; j < W / 2; ++j) a[j] = swap_add<false>(a[j], a[j + W / 2]);
#pragma unroll
    for (int j = 0; j < W / 4; ++j) a[j] = swap_add<true>(a[j], a[j + W / 4]);
    auto halve = [&](auto move, int half, bool upper) {
#pragma unroll
        for (int j = 0; j < W / 8; ++j) {
            if (j >= half) break;
            const double send = upper ? a[j] : a[j + half];
            const double keep = upper ? a[j + half] : a[j];
            a[j] = keep + move(send);
        }
    };
    auto ror8 = [](double x) { return dpp_double<0x128>(x); };
    auto mirror8 = [](double x) { return dpp_double<0x141>(x); };
    auto xor2 = [](double x) { return dpp_double<0x4e>(x); };
    auto xor1 = [](double x) { return dpp_double<0xb1>(x); };
    halve(ror8, W / 8, (lane & 8) != 0);
    if constexpr (LW > 3) halve(mirror8, W / 16, (lane & 4) != 0);
    else a[0] += mirror8(a[0]);
    if constexpr (LW > 4) halve(xor2, W / 32, (lane & 2) != 0);
    else a[0] += xor2(a[0]);
    a[0] += xor1(a[0]);
    const int idx = lane >> (6 - LW);
    if ((lane & ((1 << (6 - LW)) - 1)) == 0 && idx < K) s.red[wv][idx] = a[0];
    __syncthreads();
    if (threadIdx.x < K) {
        double r = 0;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) r += s.red[w][threadIdx.x];
        s.out[threadIdx.x] = r;
    }
    __syncthreads();
}

// Requires every value of a batch of loads in registers at this point, so that the batch's loads
// are all issued before the first is used (the compiler otherwise sinks each load into the
// conditional code that uses it, and the loads wait one after another).
template<int U>
__device__ __forceinline__ void batch_loaded(const float (&v)[U][6]) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < 6; ++c) asm volatile("" : : "v"(v[u][c]));
}

// Exclusive prefix sum over the 64 lanes of a wave (all lanes active), by data-parallel
// primitives (DPP): shifts right by 1, 2, 4 and 8 lanes inside each row of 16 (lanes with no source
// add 0), then lane 15 of each row added to the next row and lane 31 to the upper half.
__device__ __forceinline__ uint32_t wave_excl_scan(uint32_t v) {
    int incl = (int)v;
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x111, 0xf, 0xf, false);  // row_shr:1
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x112, 0xf, 0xf, false);  // row_shr:2
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x114, 0xf, 0xf, false);  // row_shr:4
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x118, 0xf, 0xf, false);  // row_shr:8
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x142, 0xa, 0xf, false);  // row_bcast:15
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return (uint32_t)incl - v;
}

// Positions of U chunks' flags over the workgroup (chunk after chunk, lane order = index order) into
// pos; returns their number (uniform).
template<int U, int NT>
__device__ __forceinline__ int wg_scan(const bool (&flag)[U], int (&pos)[U], LtsShared<NT>& s) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const unsigned long long bal = __ballot(flag[u]);
        pos[u] = __popcll(bal & ((1ull << lane) - 1ull));
        if (lane == 0) s.wave[u][wv] = __popcll(bal);
    }
    __syncthreads();
    int all = 0;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) {
            if (w == wv) pos[u] += all;
            all += s.wave[u][w];
        }
    __syncthreads();
    return all;
}

// H = U S V^T of a 3x3 matrix by one-sided Jacobi rotations; singular values descending.
__device__ void svd3(const double H[3][3], double U[3][3], double V[3][3]) {
    double A[3][3];
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) {
            A[i][j] = H[i][j];
            V[i][j] = i == j ? 1.0 : 0.0;
        }
    for (int sweep = 0; sweep < 60; ++sweep) {
        bool rotated = false;
        // unrolled: every index is a compile-time constant, so A and V stay in registers
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int q = p + 1; q < 3; ++q) {
                const double a = A[0][p] * A[0][p] + A[1][p] * A[1][p] + A[2][p] * A[2][p];
                const double b = A[0][q] * A[0][q] + A[1][q] * A[1][q] + A[2][q] * A[2][q];
                const double c = A[0][p] * A[0][q] + A[1][p] * A[1][q] + A[2][p] * A[2][q];
                if (fabs(c) <= 1e-300 || fabs(c) <= 1e-15 * sqrt(a * b)) continue;
                rotated = true;
                // tan of the rotation, the smaller root of t^2 + t (b - a) / c - 1 = 0
                const double d = b - a, h = sqrt(d * d + 4 * c * c);
                const double tn = 2 * c / (d >= 0 ? d + h : d - h);
                const double cs = 1 / sqrt(1 + tn * tn), sn = cs * tn;
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const double x = A[i][p], y = A[i][q];
                    A[i][p] = cs * x - sn * y;
                    A[i][q] = sn * x + cs * y;
                    const double vx = V[i][p], vy = V[i][q];
                    V[i][p] = cs * vx - sn * vy;
                    V[i][q] = sn * vx + cs * vy;
                }
            }
        if (!rotated) break;
    }
    double sv[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) sv[j] = sqrt(A[0][j] * A[0][j] + A[1][j] * A[1][j] + A[2][j] * A[2][j]);
    // columns by descending singular value: exchanges of columns known at compile time
#pragma unroll
    for (int e = 0; e < 3; ++e) {
        const int p = e == 1 ? 1 : 0, q = p + 1;
        const bool swap = sv[q] > sv[p];
        auto exchange = [&](double& x, double& y) {
            const double t = swap ? y : x;
            y = swap ? x : y;
            x = t;
        };
        exchange(sv[p], sv[q]);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            exchange(A[i][p], A[i][q]);
            exchange(V[i][p], V[i][q]);
        }
    }
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 3; ++i) U[i][j] = sv[j] > 0 ? A[i][j] / sv[j] : 0.0;
}

// Thread 0's half of the fit: the 3x3 solve from s.fit (the centred moments Spp 00 01 02 11 12 22,
// Spq row-major, then the means of p and q) into M.  Out of line, so that its
// registers do not add to those of the passes over the points.
__device__ __noinline__ void lts_solve(const double *fit, float *M, int *solved, bool affine) {
    const double *o = fit, *mp = fit + 15, *mq = fit + 18;
    // Spq[a][b] = sum (p_a - mp_a)(q_b - mq_b)
    const double Spq[3][3] = { { o[6], o[7], o[8] }, { o[9], o[10], o[11] }, { o[12], o[13], o[14] } };
    double L[3][3];
    int ok = 1;
    if (affine) {
        // Spp X = Spq by Gaussian elimination with partial pivoting; L = X^T.
        double a[3][6] = { { o[0], o[1], o[2], Spq[0][0], Spq[0][1], Spq[0][2] },
                           { o[1], o[3], o[4], Spq[1][0], Spq[1][1], Spq[1][2] },
                           { o[2], o[4], o[5], Spq[2][0], Spq[2][1], Spq[2][2] } };
        const double scale = fmax(fabs(o[0]), fmax(fabs(o[3]), fabs(o[5])));
        // fully unrolled, the pivot row swapped in by selects: a stays in registers
#pragma unroll
        for (int col = 0; col < 3; ++col) {
            int piv = col;
            double best = fabs(a[col][col]);
#pragma unroll
            for (int r = col + 1; r < 3; ++r)
                if (fabs(a[r][col]) > best) {
                    best = fabs(a[r][col]);
                    piv = r;
                }
            if (!(best > 1e-12 * scale)) ok = 0;
#pragma unroll
            for (int r = col + 1; r < 3; ++r)
                if (piv == r)
#pragma unroll
                    for (int k = 0; k < 6; ++k) {
                        const double tmp = a[col][k];
                        a[col][k] = a[r][k];
                        a[r][k] = tmp;
                    }
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                if (r == col) continue;
                const double f = a[r][col] / a[col][col];
#pragma unroll
                for (int k = col; k < 6; ++k) a[r][k] -= f * a[col][k];
            }
        }
        if (ok)
            for (int r = 0; r < 3; ++r)
                for (int k = 0; k < 3; ++k) L[k][r] = a[r][3 + k] / a[r][r];
    } else {
        double U[3][3], V[3][3];
        svd3(Spq, U, V);
        auto vut = [&] {
            for (int a = 0; a < 3; ++a)
                for (int b = 0; b < 3; ++b) L[a][b] = V[a][0] * U[b][0] + V[a][1] * U[b][1] + V[a][2] * U[b][2];
        };
        vut();
        const double det = L[0][0] * (L[1][1] * L[2][2] - L[1][2] * L[2][1]) -
                           L[0][1] * (L[1][0] * L[2][2] - L[1][2] * L[2][0]) +
                           L[0][2] * (L[1][0] * L[2][1] - L[1][1] * L[2][0]);
        if (det < 0) {
            for (int i = 0; i < 3; ++i) V[i][2] = -V[i][2];
            vut();
        }
    }
    if (ok) {
        for (int r = 0; r < 3; ++r) {
            for (int k = 0; k < 3; ++k) M[r * 4 + k] = (float)L[r][k];
            M[r * 4 + 3] = (float)(mq[r] - (L[r][0] * mp[0] + L[r][1] * mp[1] + L[r][2] * mp[2]));
        }
        M[12] = M[13] = M[14] = 0.f;
        M[15] = 1.f;
    }
    *solved = ok;
}

// Least-squares fit into s.M of the points whose centred moments and means lts_moments or
// lts_kept_moments left in s.fit.  Affine: the FP64 solution of [p 1] P = q through centred normal
// equations (the same minimiser as EstimateAffineLeastSquares' QR, reg-lib/cpu/Maths.cpp:325-349).
// Rigid: Kabsch on the centred cross-covariance with the reflection guard
// (reg-lib/cpu/Maths.cpp:351-390).  Returns false (uniformly) when the normal matrix is singular.
template<int NT>
__device__ __forceinline__ bool lts_fit(bool affine, LtsShared<NT>& s) {
    if (threadIdx.x == 0) lts_solve(s.fit, s.M, &s.scal[0], affine);
    __syncthreads();
    return s.scal[0] != 0;
}

// Loads kLtsUnroll points of P and Q (planes of stride floats), NT apart from i0, clamped to n - 1: all
// loads issued together, each from a uniform base.
template<int NT>
__device__ __forceinline__ void lts_load(const float *__restrict__ P, const float *__restrict__ Q, int stride, int i0,
                                         int n, float (&pq)[kLtsUnroll][6]) {
#pragma unroll
    for (int u = 0; u < kLtsUnroll; ++u) {
        const uint32_t i = (uint32_t)min(i0 + u * NT, n - 1);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float *p = P + (size_t)c * stride, *q = Q + (size_t)c * stride;
            pq[u][c] = p[i];
            pq[u][3 + c] = q[i];
        }
    }
    batch_loaded(pq);
}

// The centred moments of all n points, from their sums m (this thread's): a pass over the points
// about the means.
template<int NT>
__device__ __forceinline__ void lts_moments(const float *__restrict__ P, const float *__restrict__ Q, int stride, int n,
                                            double (&m)[7], LtsShared<NT>& s) {
    wg_sum(m, s);
    double mean[6];
    for (int k = 0; k < 6; ++k) mean[k] = s.out[k] / s.out[6];
    __syncthreads();
    double c[15] = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
    for (int i0 = threadIdx.x; i0 < n; i0 += kLtsUnroll * NT) {
        float pq[kLtsUnroll][6];
        lts_load<NT>(P, Q, stride, i0, n, pq);
#pragma unroll
        for (int u = 0; u < kLtsUnroll; ++u) {
            if (i0 + u * NT >= n) break;
            double p[3], q[3];
            for (int k = 0; k < 3; ++k) {
                p[k] = (double)pq[u][k] - mean[k];
                q[k] = (double)pq[u][3 + k] - mean[3 + k];
            }
            c[0] += p[0] * p[0]; c[1] += p[0] * p[1]; c[2] += p[0] * p[2];
            c[3] += p[1] * p[1]; c[4] += p[1] * p[2]; c[5] += p[2] * p[2];
            for (int a = 0; a < 3; ++a)
                for (int b = 0; b < 3; ++b) c[6 + a * 3 + b] += p[a] * q[b];
        }
    }
    wg_sum(c, s);
    if (threadIdx.x == 0) {
        for (int k = 0; k < 15; ++k) s.fit[k] = s.out[k];
        for (int k = 0; k < 6; ++k) s.fit[15 + k] = mean[k];
    }
}

// The same of the kept points, from their sums in s.kept: S = sum - count m m^T in FP64.
template<int NT>
__device__ __forceinline__ void lts_kept_moments(LtsShared<NT>& s) {
    if (threadIdx.x != 0) return;
    const double *sums = s.kept;
    double *oc = s.fit, *mp = s.fit + 15, *mq = s.fit + 18;
    const double cnt = sums[6];
    for (int k = 0; k < 3; ++k) {
        mp[k] = sums[k] / cnt;
        mq[k] = sums[3 + k] / cnt;
    }
    const int pa[6] = { 0, 0, 0, 1, 1, 2 }, pb[6] = { 0, 1, 2, 1, 2, 2 };
    for (int k = 0; k < 6; ++k) oc[k] = sums[7 + k] - cnt * mp[pa[k]] * mp[pb[k]];
    for (int a = 0; a < 3; ++a)
        for (int b = 0; b < 3; ++b) oc[6 + a * 3 + b] = sums[13 + a * 3 + b] - cnt * mp[a] * mq[b];
}

// dv += (or -=) the sums of the first c points of the wave's list: p, q, count and the products, each
// exact in FP64 before it is added (a product of two floats has 48 bits).
__device__ __forceinline__ void lts_add_listed(const float *__restrict__ P, const float *__restrict__ Q, int stride,
                                               const volatile uint32_t *list, int c, double *dv) {
    if ((int)(threadIdx.x & 63) >= c) return;
    const uint32_t e = list[threadIdx.x & 63], i = e & 0x7fffffffu;
    const double sign = e >> 31 ? -1.0 : 1.0;
    double p[3], q[3], sp[3];
    for (int k = 0; k < 3; ++k) {
        const float *pk = P + (size_t)k * stride, *qk = Q + (size_t)k * stride;
        p[k] = (double)pk[i];
        q[k] = (double)qk[i];
    }
    for (int k = 0; k < 3; ++k) sp[k] = sign * p[k];
    for (int k = 0; k < 3; ++k) {
        dv[k] += sp[k];
        dv[3 + k] = fma(sign, q[k], dv[3 + k]);
    }
    dv[6] += sign;
    dv[7] = fma(sp[0], p[0], dv[7]);
    dv[8] = fma(sp[0], p[1], dv[8]);
    dv[9] = fma(sp[0], p[2], dv[9]);
    dv[10] = fma(sp[1], p[1], dv[10]);
    dv[11] = fma(sp[1], p[2], dv[11]);
    dv[12] = fma(sp[2], p[2], dv[12]);
    for (int a = 0; a < 3; ++a)
        for (int b = 0; b < 3; ++b) dv[13 + a * 3 + b] = fma(sp[a], q[b], dv[13 + a * 3 + b]);
}

// optimize + optimize_3D (reg-lib/cpu/_reg_blockMatching.cpp:722-821,
// reg-lib/cpu/_reg_globalTrans.cpp:328-394).  status: 0 ok, 1 too few correspondences,
// 2 singular fit (the matrix is then left unchanged).  The trimmed subset is the keep smallest
// residuals (float bit patterns, found by a three-digit radix select); ties at the threshold
// keep the lowest indices.  P and Q: the defined correspondences, planar with nActive floats a plane
// (the 12-byte rows of the inputs cost every load three times the cache lines).  LDS: res is in LDS and
// holds at most 32 points a thread, whose kept flags are then a word's bits; otherwise the flags are
// bytes after the residuals.
//
// One workgroup, as the 20 or so iterations are a serial chain of a residual pass, three digits and a
// fit each, so its cost is the instructions and barriers of one compute unit.  The kept points' sums
// are carried from one iteration to the next: only points that enter or leave the set are added or
// subtracted, gathered in a list per wave so that 64 at a time fill the lanes (all kept points summed
// anew took as long as the residuals).  What that loses in FP64 is far below the matrix's floats; but a
// point with an infinite coordinate that is in the set once leaves its sums NaN to the end of the fit,
// where sums formed anew would be numbers again after it left.  19 iterations over 16384 points 470 -> 426 us, of which the
// residuals are 40 % (their conversions to and from double run at a quarter of the rate) and the digits
// 25 %; the 1000 points of a coarse level, 4 iterations, 57 -> 42 us.
template<int NT, bool LDS>
__device__ __forceinline__ void
lts_body(const float *__restrict__ refPos, const float *__restrict__ warpPos, int nActive, float *__restrict__ matrix,
         float *__restrict__ P, float *__restrict__ Q, uint32_t *__restrict__ res, int percent, int affine,
         int *__restrict__ status, LtsShared<NT>& s) {
#pragma clang fp contract(off)
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, stride = nActive;
    if (tid < 16) s.M[tid] = matrix[tid];
    __syncthreads();
    double M0[12];
    for (int k = 0; k < 12; ++k) M0[k] = uniform_double((double)s.M[k]);
    // defined correspondences in rank order, warped side mapped through the current matrix
    int n = 0;
    double m[7] = { 0, 0, 0, 0, 0, 0, 0 };
    for (int base = 0; base < nActive; base += kLtsUnroll * NT) {
        float rw[kLtsUnroll][6];
        bool flag[kLtsUnroll];
        int pos[kLtsUnroll];
#pragma unroll
        for (int u = 0; u < kLtsUnroll; ++u) {
            const uint32_t i = 3u * (uint32_t)min(base + u * NT + tid, nActive - 1);
            for (int c = 0; c < 3; ++c) {
                rw[u][c] = refPos[i + c];
                rw[u][3 + c] = warpPos[i + c];
            }
        }
        batch_loaded(rw);
#pragma unroll
        for (int u = 0; u < kLtsUnroll; ++u)
            flag[u] = base + u * NT + tid < nActive && rw[u][3] == rw[u][3];
        const int total = wg_scan(flag, pos, s);
#pragma unroll
        for (int u = 0; u < kLtsUnroll; ++u)
            if (flag[u]) {
                const float3 q = mat44_mul_f(M0, rw[u][3], rw[u][4], rw[u][5]);
                const float v[6] = { rw[u][0], rw[u][1], rw[u][2], q.x, q.y, q.z };
                for (int c = 0; c < 3; ++c) {
                    float *p = P + (size_t)c * stride, *q = Q + (size_t)c * stride;
                    p[(uint32_t)(n + pos[u])] = v[c];
                    q[(uint32_t)(n + pos[u])] = v[3 + c];
                }
                for (int c = 0; c < 6; ++c) m[c] += (double)v[c];
                m[6] += 1.0;
            }
        n += total;
    }
    const unsigned keep = (unsigned)((float)n * ((float)percent / 100.0f));
    if (n < (affine ? 8 : 4) || keep < 4) {
        if (tid == 0) *status = 1;
        return;
    }
    __threadfence_block();
    __syncthreads();
    lts_moments(P, Q, stride, n, m, s);
    if (!lts_fit(affine != 0, s)) {
        if (tid == 0) *status = 2;
        return;
    }
    uint8_t *keepFlag = LDS ? nullptr : reinterpret_cast<uint8_t *>(res + n);
    uint32_t keptBits = 0;
    double lastDistance = DBL_MAX;
    if (tid < 16) s.last[tid] = 0.f;
    if (tid < 24) s.kept[tid] = 0.0;
    __syncthreads();
    for (int it = 0; it < 30; ++it) {
        // residuals, counted into the first digit's histogram as they are formed
        for (int b = tid; b < 2048 + 256; b += NT) s.hist[b] = 0;
        __syncthreads();
        double M[12];  // uniform: scalar registers
        for (int k = 0; k < 12; ++k) M[k] = uniform_double((double)s.M[k]);
        for (int i0 = tid; i0 < n; i0 += kLtsUnroll * NT) {
            float pq[kLtsUnroll][6];
            lts_load<NT>(P, Q, stride, i0, n, pq);
#pragma unroll
            for (int u = 0; u < kLtsUnroll; ++u) {
                const int i = i0 + u * NT;
                if (i >= n) break;
                const float3 t = mat44_mul_f(M, pq[u][0], pq[u][1], pq[u][2]);
                const float dx = t.x - pq[u][3], dy = t.y - pq[u][4], dz = t.z - pq[u][5];
                const uint32_t key = __float_as_uint(sqrtf(dx * dx + dy * dy + dz * dz));
                res[i] = key;
                atomicAdd(&s.hist[lts_bin(key >> 21)], 1u);
            }
        }
        __syncthreads();
        // radix select of the keep-th smallest residual: digits of 11, 11 and 10 bits
        uint32_t prefix = 0, prefMask = 0, eqCount = 0;
        int k = (int)keep;
        const int shifts[3] = { 21, 10, 0 }, widths[3] = { 11, 11, 10 };
        for (int d = 0; d < 3; ++d) {
            const int sh = shifts[d];
            const uint32_t dm = (1u << widths[d]) - 1u;
            if (d > 0) {
                for (int b = tid; b < 2048 + 256; b += NT) s.hist[b] = 0;
                __syncthreads();
                for (int i0 = tid; i0 < n; i0 += kLtsUnroll * NT) {
                    uint32_t key[kLtsUnroll];
#pragma unroll
                    for (int u = 0; u < kLtsUnroll; ++u) key[u] = res[(uint32_t)min(i0 + u * NT, n - 1)];
#pragma unroll
                    for (int u = 0; u < kLtsUnroll; ++u)
                        if (i0 + u * NT < n && (key[u] & prefMask) == prefix)
                            atomicAdd(&s.hist[lts_bin((key[u] >> sh) & dm)], 1u);
                }
                __syncthreads();
            }
            if (tid < 64) {
                // the group of 32 bins holding the k-th key (prefix sums over the 64 groups),
                // then the bin inside it (prefix sums over the group's 32 bins), both found
                // by a ballot: the first bin whose inclusive count reaches k
                const uint4 *grp = reinterpret_cast<const uint4 *>(&s.hist[lts_bin(tid * 32)]);
                uint32_t local = 0;
#pragma unroll
                for (int b = 0; b < 8; ++b) {
                    const uint4 v = grp[b];
                    local += v.x + v.y + v.z + v.w;
                }
                const uint32_t excl = wave_excl_scan(local);
                const unsigned long long inGroup = __ballot(excl < (uint32_t)k && (uint32_t)k <= excl + local);
                const int g = inGroup ? __ffsll((long long)inGroup) - 1 : 0;
                const uint32_t base = __shfl(excl, g, 64);
                const uint32_t h = tid < 32 ? s.hist[lts_bin(g * 32 + tid)] : 0u;
                const uint32_t before = base + wave_excl_scan(h);
                const unsigned long long inBin = __ballot(tid < 32 && before + h >= (uint32_t)k);
                if (tid == (inBin ? __ffsll((long long)inBin) - 1 : 0)) {
                    s.scal[1] = g * 32 + tid;
                    s.scal[2] = k - (int)before;
                    s.scal[3] = (int)h;
                }
            }
            __syncthreads();
            eqCount = (uint32_t)s.scal[3];  // after the last digit: keys equal to the whole threshold
            prefix |= (uint32_t)s.scal[1] << sh;
            prefMask |= dm << sh;
            k = s.scal[2];
            __syncthreads();
        }
        // keep: residual below the threshold, or equal to it within the first k in index order (when
        // every key equal to the threshold is kept, the order plays no part); the distance is summed
        // anew, the sums for the next fit (dv[0..22)) over the points that enter or leave the set
        double dv[23];
        for (int c = 0; c < 23; ++c) dv[c] = 0.0;
        volatile uint32_t *list = s.list[wv];
        int listed = 0, seenEqual = 0;
        const bool allEqual = (uint32_t)k == eqCount;
        for (int base = 0; base < n; base += kLtsUnroll * NT) {
            uint32_t key[kLtsUnroll];
            bool kept[kLtsUnroll], was[kLtsUnroll];
#pragma unroll
            for (int u = 0; u < kLtsUnroll; ++u) {
                const int i = base + u * NT + tid;
                key[u] = res[(uint32_t)min(i, n - 1)];
                was[u] = !LDS && it > 0 && keepFlag[(uint32_t)min(i, n - 1)] != 0;
                kept[u] = i < n && key[u] <= prefix;
                if (i >= n) was[u] = false;
            }
            if (!allEqual) {
                bool equal[kLtsUnroll];
                int eqPos[kLtsUnroll];
#pragma unroll
                for (int u = 0; u < kLtsUnroll; ++u) equal[u] = kept[u] && key[u] == prefix;
                const int total = wg_scan(equal, eqPos, s);
#pragma unroll
                for (int u = 0; u < kLtsUnroll; ++u)
                    kept[u] = kept[u] && (key[u] < prefix || seenEqual + eqPos[u] < k);
                seenEqual += total;
            }
#pragma unroll
            for (int u = 0; u < kLtsUnroll; ++u) {
                const int i = base + u * NT + tid;
                if (kept[u]) dv[22] += (double)__uint_as_float(key[u]);
                if (LDS) {
                    was[u] = keptBits & 1u;
                    keptBits = keptBits >> 1 | (kept[u] ? 0x80000000u : 0u);
                } else if (i < n && (it == 0 || kept[u] != was[u])) {
                    keepFlag[i] = kept[u] ? 1 : 0;
                }
                const bool flip = kept[u] != was[u];
                const unsigned long long flips = __ballot(flip);
                if (flips) {  // uniform over the wave; its lanes' accesses to the list are in program order
                    if (flip)
                        list[listed + __popcll(flips & ((1ull << lane) - 1ull))] =
                            (uint32_t)i | (kept[u] ? 0u : 0x80000000u);
                    listed += __popcll(flips);
                    if (listed >= 64) {
                        lts_add_listed(P, Q, stride, list, 64, dv);
                        listed -= 64;
                        if (lane < listed) list[lane] = list[64 + lane];
                    }
                }
            }
        }
        if (LDS) keptBits >>= (32 - kLtsUnroll * ((n + kLtsUnroll * NT - 1) / (kLtsUnroll * NT))) & 31;
        lts_add_listed(P, Q, stride, list, listed, dv);
        wg_sum(dv, s);
        const double distance = s.out[22];
        if (distance > lastDistance || (lastDistance - distance) < 1e-3) {
            if (tid < 16) s.M[tid] = s.last[tid];
            __syncthreads();
            break;
        }
        lastDistance = distance;
        if (tid < 16) s.last[tid] = s.M[tid];
        if (tid < 22) s.kept[tid] += s.out[tid];
        __syncthreads();
        lts_kept_moments(s);
        if (!lts_fit(affine != 0, s)) {
            if (tid == 0) *status = 2;
            return;
        }
    }
    if (tid < 16) matrix[tid] = s.M[tid];
}

// Past the LDS: the residuals and the kept flags in memory.
__global__ void __launch_bounds__(kLtsThreads)
k_lts(const float *__restrict__ refPos, const float *__restrict__ warpPos, int nActive, float *__restrict__ matrix,
      float *__restrict__ P, float *__restrict__ Q, uint32_t *__restrict__ res, int percent, int affine,
      int *__restrict__ status) {
    __shared__ LtsShared<kLtsThreads> s;
    lts_body<kLtsThreads, false>(refPos, warpPos, nActive, matrix, P, Q, res, percent, affine, status, s);
}

// The same fit with the residuals of up to N correspondences in LDS.  Few of them go to 256 threads:
// what an iteration over 1000 points takes is its barriers and the sums over the workgroup's waves.
template<int NT, int N>
__global__ void __launch_bounds__(NT)
k_lts_lds(const float *__restrict__ refPos, const float *__restrict__ warpPos, int nActive, float *__restrict__ matrix,
          float *__restrict__ P, float *__restrict__ Q, int percent, int affine, int *__restrict__ status) {
    static_assert(N <= 32 * NT, "a thread's kept flags are a word");
    __shared__ LtsShared<NT> s;
    __shared__ uint32_t sRes[N];
    lts_body<NT, true>(refPos, warpPos, nActive, matrix, P, Q, sRes, percent, affine, status, s);
}

constexpr int kLtsSmallThreads = 256, kLtsSmallN = 4096, kLtsLdsN = 16384;

// One LTS fit of nActive correspondences on `stream`: in LDS when they fit, else with the
// residual scratch `res` (nActive + nActive / 4 words) in memory.
void launch_lts(hipStream_t stream, const float *refPos, const float *warpPos, int nActive, float *matrix, float *P,
                float *Q, uint32_t *res, int percent, int affine, int *status) {
    if (nActive <= kLtsSmallN)
        hipLaunchKernelGGL((k_lts_lds<kLtsSmallThreads, kLtsSmallN>), dim3(1), dim3(kLtsSmallThreads), 0, stream, refPos,
                           warpPos, nActive, matrix, P, Q, percent, affine, status);
    else if (nActive <= kLtsLdsN)
        hipLaunchKernelGGL((k_lts_lds<kLtsThreads, kLtsLdsN>), dim3(1), dim3(kLtsThreads), 0, stream, refPos, warpPos,
                           nActive, matrix, P, Q, percent, affine, status);
    else
        hipLaunchKernelGGL(k_lts, dim3(1), dim3(kLtsThreads), 0, stream, refPos, warpPos, nActive, matrix, P, Q, res,
                           percent, affine, status);
}

// The LTS fits of a batch of pairs in one launch: one workgroup per pair.
struct LtsArgs {
    const float *refPos, *warpPos;
    int nActive;
    float *matrix, *P, *Q;
    uint32_t *res;
    int percent;
    int *status;
};

__global__ void __launch_bounds__(kLtsThreads) k_lts_batch(const LtsArgs *__restrict__ A, int affine) {
    __shared__ LtsShared<kLtsThreads> s;
    const LtsArgs& a = A[blockIdx.x];
    lts_body<kLtsThreads, false>(a.refPos, a.warpPos, a.nActive, a.matrix, a.P, a.Q, a.res, a.percent, affine, a.status, s);
}

// Empties the defined-block count before a block matching (a kernel, so that an iteration can be
// captured in a graph).
__global__ void k_zero_int(int *p) {
    if (threadIdx.x == 0) *p = 0;
}

// ------------------------------------------------------------------ symmetric update
// reg_aladin_sym::UpdateTransformationMatrix (reg-lib/_reg_aladin_sym.cpp:128-157) after the two
// LTS fits: forward <- avg(forward, inv(backward)), backward <- avg(inv(forward), backward), where
// avg = NiftyReg::Mat44Avg2 (reg-lib/cpu/Maths.cpp:479-491) = expm((logm A + logm B) / 2).  The
// reference evaluates logm / expm with Eigen in double; here they are computed in double by
// inverse scaling and squaring (Denman-Beavers square roots, then the [8/8] Pade approximant of
// log(I + X) in Gauss-Legendre form) and by Taylor scaling and squaring, with the reference's
// float roundings between the steps.
//
// One wave: 16 lanes hold one 4x4 matrix, an element each, so the four logarithms of an update run
// beside one another, and every product and elimination step is one instruction per lane where a
// single thread makes 16 to 32 and keeps the pivoted rows in scratch memory.  The arithmetic of each
// element and the order of every sum are those of m44.hpp's functions (d4_inverse, d4_logm, d4_expm),
// which the host and the oracle use, so the results are equal.  Latency-bound, a chain of FP64
// divisions and lane exchanges: 75 us an update, 395 with one thread (181 x 217 x 181 pair).
struct WaveMat {
    int i, j, base;  // row, column, first lane of the group
    __device__ WaveMat(): i((threadIdx.x >> 2) & 3), j(threadIdx.x & 3), base(threadIdx.x & 48) {}
    __device__ double get(double v, int r, int c) const { return __shfl(v, base + 4 * r + c, 64); }
    __device__ double eye() const { return i == j ? 1.0 : 0.0; }
    __device__ double mul(double a, double b) const {
        double acc = 0.0;
#pragma unroll
        for (int k = 0; k < 4; ++k) acc = fma(get(a, i, k), get(b, k, j), acc);
        return acc;
    }
    // the largest column sum of absolute values, the same in every lane of the group
    __device__ double norm1(double a) const {
        const double m = fabs(a);
        const double c = get(m, 0, j) + get(m, 1, j) + get(m, 2, j) + get(m, 3, j);
        double best = 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const double v = get(c, 0, q);
            best = v > best ? v : best;
        }
        return best;
    }
    // the sum over the 16 elements, row by row
    __device__ double sum(double a) const {
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < 16; ++q) s += __shfl(a, base + q, 64);
        return s;
    }
    // Gauss-Jordan with partial pivoting; *singular is set for the group on a zero pivot
    __device__ double inverse(double a, bool *singular) const {
        double m0 = a, m1 = eye();
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            double v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = get(m0, r, c);
            int p = c;
            double vp = v[c];
#pragma unroll
            for (int r = c + 1; r < 4; ++r)
                if (fabs(v[r]) > fabs(vp)) {
                    p = r;
                    vp = v[r];
                }
            if (vp == 0.0) *singular = true;
            // row c of the exchanged matrix is the pivot row, scaled; the lane's own row and its
            // factor follow the exchange
            const double inv = 1.0 / vp;
            const double p0 = get(m0, p, j) * inv, p1 = get(m1, p, j) * inv;
            const int src = i == p ? c : i;
            const double o0 = get(m0, src, j), o1 = get(m1, src, j);
            const double f = src == 0 ? v[0] : src == 1 ? v[1] : src == 2 ? v[2] : v[3];
            m0 = i == c ? p0 : fma(-f, p0, o0);
            m1 = i == c ? p1 : fma(-f, p1, o1);
        }
        return m1;
    }
};

// Every lane of the wave calls these; loops end when no group of 16 lanes needs another turn.
// *failed is set for the group where d4_logm returns false.
__device__ double wave_logm(const WaveMat& w, double a, const GaussLegendre8& gl, bool *failed) {
    double y = a, x = 0.0;
    int k = 0;
    bool settled = false;  // the group's matrix is near enough to the identity, or has failed
    for (;;) {
        if (!settled) x = y - w.eye();
        if (w.norm1(x) <= 0.25) settled = true;
        if (!settled && k >= 60) *failed = settled = true;
        if (__all(settled)) break;
        double z = w.eye();
        bool done = settled;
        for (int it = 0; it < 100; ++it) {
            bool singular = false;
            const double yi = w.inverse(y, &singular), zi = w.inverse(z, &singular);
            if (singular && !done) *failed = settled = done = true;
            const double yn = 0.5 * (y + zi);
            const double diff = w.sum(fabs(yn - y)), zn = 0.5 * (z + yi);
            const double norm = w.norm1(done ? y : yn);
            if (!done) {
                z = zn;
                y = yn;
                if (diff <= 1e-15 * norm) done = true;
            }
            if (__all(done)) break;
        }
        if (!settled) ++k;
    }
    double s = 0.0;
    for (int q = 0; q < 8; ++q) {
        bool singular = false;
        const double ti = w.inverse(fma(gl.x[q], x, w.eye()), &singular);
        if (singular) *failed = true;
        s = fma(gl.w[q], w.mul(x, ti), s);
    }
    return ldexp(1.0, k) * s;
}

__device__ double wave_expm(const WaveMat& w, double a) {
    const double n = w.norm1(a);
    int s = 0;
    if (n > 0.5) s = (int)ceil(log2(n / 0.5));
    const double b = a * ldexp(1.0, -s);
    double term = w.eye(), sum = term;
    for (int k = 1; k <= 20; ++k) {
        term = w.mul(term, b);
        term /= k;
        sum += term;
    }
    for (int q = 0; !__all(q >= s); ++q) {
        const double sq = w.mul(sum, sum);
        if (q < s) sum = sq;
    }
    return sum;
}

__global__ void __launch_bounds__(64)
k_symmetric_update(float *__restrict__ fw, float *__restrict__ bw, GaussLegendre8 gl, int *__restrict__ status) {
    // the groups' matrices: forward, inverse of backward, inverse of forward, backward; each pair
    // is averaged (Mat44Avg2: the logarithms rounded to float with zero bottom rows, summed in
    // double and rounded to float, halved, exponentiated in double, rounded to float)
    __shared__ float M[4][16];
    if (threadIdx.x < 2) {
        float a[16], inv[16];
        const float *src = threadIdx.x == 0 ? fw : bw;
        for (int q = 0; q < 16; ++q) a[q] = src[q];
        nifti_inverse(a, inv);
        for (int q = 0; q < 16; ++q) {
            M[threadIdx.x == 0 ? 0 : 3][q] = a[q];
            M[threadIdx.x == 0 ? 2 : 1][q] = inv[q];
        }
    }
    __syncthreads();
    const int group = threadIdx.x >> 4, e = threadIdx.x & 15;
    const WaveMat w;
    bool failed = false;
    const double l = wave_logm(w, (double)M[group][e], gl, &failed);
    if (__any(failed)) {
        if (threadIdx.x == 0) *status = 3;  // matrices left unchanged
        return;
    }
    const float own = e >= 12 ? 0.f : (float)l;
    const float other = __shfl_xor(own, 16, 64);
    const float sum = (float)((double)own + (double)other);
    float r = (float)wave_expm(w, (double)(sum * 0.5f));
    if (e >= 12) r = e == 15 ? 1.f : 0.f;
    if (group == 0) fw[e] = r;
    if (group == 2) bw[e] = r;
}

// ------------------------------------------------------------------ host side
unsigned blocks_for(size_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

void check_aladin_params(const nrh_aladin_params *p) {
    NRH_REQUIRE(p, NRH_ERR_ARG, "null Aladin parameters");
    NRH_REQUIRE(p->block_percent > 0 && p->block_percent <= 100, NRH_ERR_ARG, "block percentage must be in (0, 100]");
    NRH_REQUIRE(p->inlier_lts > 0 && p->inlier_lts <= 100, NRH_ERR_ARG, "LTS inlier percentage must be in (0, 100]");
}

// initialise_block_matching_method (reg-lib/cpu/_reg_blockMatching.cpp:213-273) and
// _reg_set_active_blocks<float> (:49-206).
void select_blocks(nrh_aladin *h) {
    h->nb[0] = (h->ref.nx + 3) / 4;
    h->nb[1] = (h->ref.ny + 3) / 4;
    h->nb[2] = (h->ref.nz + 3) / 4;
    const int total = h->nb[0] * h->nb[1] * h->nb[2];
    h->totalBlocks = total;
    DevBuf<float> var;
    var.alloc(total);
    hipLaunchKernelGGL(k_block_variance, dim3(blocks_for(total)), dim3(kBlock), 0, h->stream, h->refImg.p,
                       h->mask.p, h->ref.nx, h->ref.ny, h->ref.nz, h->nb[0], h->nb[1], h->nb[2], var.p);
    NRH_HIP(hipGetLastError());
    std::vector<float> v(total);
    NRH_HIP(hipMemcpyAsync(v.data(), var.p, total * sizeof(float), hipMemcpyDeviceToHost, h->stream));
    NRH_HIP(hipStreamSynchronize(h->stream));
    int unusable = 0;
    for (float x : v) unusable += x < 0.f;
    int active = (int)((double)total * ((double)h->params.block_percent / 100.0));
    active = std::min(active, total - unusable);
    std::vector<int> ix(total);
    for (int b = 0; b < total; ++b) ix[b] = b;
    heap_sort_indexed(v, ix);
    h->totalBlock.assign(total, -1);
    for (int r = 0; r < active; ++r) h->totalBlock[ix[total - 1 - r]] = r;
    std::vector<int2> list;  // (block, rank) in block order
    list.reserve(std::max(active, 0));
    for (int b = 0; b < total; ++b)
        if (h->totalBlock[b] >= 0) list.push_back(make_int2(b, h->totalBlock[b]));
    NRH_REQUIRE(active >= 2, NRH_ERR_NUMERIC, "There are less than 2 active blocks");
    h->activeBlocks = active;
    h->activeList.alloc(active);
    NRH_HIP(hipMemcpyAsync(h->activeList.p, list.data(), active * sizeof(int2), hipMemcpyHostToDevice, h->stream));
    h->refPos.alloc(3 * (size_t)active);
    h->warpPos.alloc(3 * (size_t)active);
    h->ltsP.alloc(3 * (size_t)active);
    h->ltsQ.alloc(3 * (size_t)active);
    h->ltsRes.alloc((size_t)active + (active + 3) / 4);  // residual bits, then one keep byte per point
    NRH_HIP(hipStreamSynchronize(h->stream));
}

Mat4 mat4_of(const float *m) {
    Mat4 r;
    for (int i = 0; i < 16; ++i) r.m[i] = m[i];
    return r;
}

void launch_warp(nrh_aladin *h) {
    hipLaunchKernelGGL(k_affine_warp, dim3(blocks_for(h->N)), dim3(kBlock), 0, h->stream, h->floImg.p, h->flo.nx,
                       h->flo.ny, h->flo.nz, to_affine(h->flo.ijk), h->matrix.p, mat4_of(h->ref.xyz), h->ref.nx,
                       h->ref.ny, h->ref.nz, h->mask.p, h->params.padding, h->warped.p);
    NRH_HIP(hipGetLastError());
}

template<int NB, int NX>
void launch_match(nrh_aladin *h) {
    hipLaunchKernelGGL((k_block_match<NB, NX>), dim3((h->activeBlocks + NB - 1) / NB), dim3(MatchShape<NB, NX>::kThreads), 0,
                       h->stream, h->refImg.p, h->warped.p, h->mask.p, h->ref.nx, h->ref.ny, h->ref.nz, h->nb[0], h->nb[1],
                       h->activeList.p, h->activeBlocks, to_affine(h->ref.xyz), h->refPos.p, h->warpPos.p, h->counters.p);
    NRH_HIP(hipGetLastError());
}

void launch_block_matching(nrh_aladin *h) {
    hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(64), 0, h->stream, h->counters.p);
    if (h->activeBlocks <= kMatchFew) launch_match<1, 1>(h);
    else launch_match<5, 7>(h);
}

void launch_lts(nrh_aladin *h, bool affine) {
    launch_lts(h->stream, h->refPos.p, h->warpPos.p, h->activeBlocks, h->matrix.p, h->ltsP.p, h->ltsQ.p,
               h->ltsRes.p, h->params.inlier_lts, affine ? 1 : 0, h->counters.p + 1);
    NRH_HIP(hipGetLastError());
}

void read_counters(nrh_aladin *h) {
    NRH_HIP(hipMemcpyAsync(h->pinned, h->counters.p, 3 * sizeof(int), hipMemcpyDeviceToHost, h->stream));
    NRH_HIP(hipStreamSynchronize(h->stream));
}

void raise_lts_status(int status) {
    NRH_REQUIRE(status != 1, NRH_ERR_NUMERIC,
                "Not enough correspondences were found - it is impossible to estimate the transformation");
    NRH_REQUIRE(status != 2, NRH_ERR_NUMERIC, "singular least-squares system in the LTS fit");
}

void raise_symmetric_status(int status) {
    NRH_REQUIRE(status == 0, NRH_ERR_NUMERIC,
                "the matrix logarithm of the symmetric update failed (a matrix with a non-positive determinant)");
}

// Both matrices live on the device; the kernel runs on the forward handle's stream after the
// backward handle's queued work.
void launch_symmetric_update(nrh_aladin *fw, nrh_aladin *bw) {
    static const GaussLegendre8 gl = gauss_legendre8();
    if (fw->stream != bw->stream) {
        hipEvent_t ev;
        NRH_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
        NRH_HIP(hipEventRecord(ev, bw->stream));
        NRH_HIP(hipStreamWaitEvent(fw->stream, ev, 0));
        NRH_HIP(hipEventDestroy(ev));
    }
    hipLaunchKernelGGL(k_symmetric_update, dim3(1), dim3(64), 0, fw->stream, fw->matrix.p, bw->matrix.p, gl,
                       fw->counters.p + 2);
    NRH_HIP(hipGetLastError());
}

void destroy(nrh_aladin *h);

// A handle over the two images, which it takes over (device) or, where a buffer is empty, uploads
// from ref_data / flo_data (host).
nrh_aladin *create(const nrh_geom *ref, DevBuf<float>&& refImg, const float *ref_data, const nrh_geom *flo,
                   DevBuf<float>&& floImg, const float *flo_data, const int *mask, const nrh_aladin_params *params,
                   hipStream_t sharedStream = nullptr) {
    check_geom(ref, "reference");
    check_geom(flo, "floating");
    check_aladin_params(params);
    NRH_REQUIRE((ref_data || !refImg.empty()) && (flo_data || !floImg.empty()), NRH_ERR_ARG, "null image data");
    NRH_REQUIRE(ref->nz > 1, NRH_ERR_UNSUPPORTED, "2-D images are not supported");
    std::unique_ptr<nrh_aladin> h(new nrh_aladin);
    h->ref = *ref;
    h->flo = *flo;
    h->params = *params;
    h->N = voxels(*ref);
    h->Nf = voxels(*flo);
    NRH_HIP(hipGetDevice(&h->device));
    if (sharedStream) {
        h->stream = sharedStream;
        h->ownsStream = false;
    } else {
        NRH_HIP(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
    }
    NRH_HIP(hipHostMalloc((void **)&h->pinned, 4 * sizeof(int), hipHostMallocDefault));
    auto image = [&](DevBuf<float>& img, DevBuf<float>&& from, const float *data, size_t n) {
        NRH_REQUIRE(from.empty() || from.n == n, NRH_ERR_ARG, "image sizes differ from the geometries");
        img = std::move(from);
        if (!img.empty()) return;
        img.alloc(n);
        NRH_HIP(hipMemcpyAsync(img.p, data, n * sizeof(float), hipMemcpyHostToDevice, h->stream));
    };
    image(h->refImg, std::move(refImg), ref_data, h->N);
    image(h->floImg, std::move(floImg), flo_data, h->Nf);
    h->warped.alloc(h->N);
    NRH_HIP(hipMemsetAsync(h->warped.p, 0, h->warped.bytes(), h->stream));
    if (mask) {
        bool any = false;
        for (size_t i = 0; i < h->N && !any; ++i) any = mask[i] < 0;
        if (any) {
            h->mask.alloc(h->N);
            NRH_HIP(hipMemcpyAsync(h->mask.p, mask, h->N * sizeof(int), hipMemcpyHostToDevice, h->stream));
        }
    }
    h->matrix.alloc(16);
    const float eye[16] = { 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1 };
    NRH_HIP(hipMemcpyAsync(h->matrix.p, eye, sizeof(eye), hipMemcpyHostToDevice, h->stream));
    h->counters.alloc(4);
    NRH_HIP(hipMemsetAsync(h->counters.p, 0, h->counters.bytes(), h->stream));
    h->pinned[0] = -1;
    h->pinned[1] = 0;
    h->pinned[2] = 0;
    try {
        select_blocks(h.get());
    } catch (...) {
        destroy(h.release());
        throw;
    }
    return h.release();
}

void destroy(nrh_aladin *h) {
    if (!h) return;
    if (h->stream) (void)hipStreamSynchronize(h->stream);
    if (h->pinned) (void)hipHostFree(h->pinned);
    hipStream_t s = h->ownsStream ? h->stream : nullptr;
    delete h;
    if (s) (void)hipStreamDestroy(s);
}

void set_matrix(nrh_aladin *h, const float *m) {
    NRH_HIP(hipMemcpyAsync(h->matrix.p, m, 16 * sizeof(float), hipMemcpyHostToDevice, h->stream));
    NRH_HIP(hipStreamSynchronize(h->stream));
}

void get_matrix(nrh_aladin *h, float *m) {
    NRH_HIP(hipMemcpyAsync(m, h->matrix.p, 16 * sizeof(float), hipMemcpyDeviceToHost, h->stream));
    NRH_HIP(hipStreamSynchronize(h->stream));
}

struct AladinHandle {
    nrh_aladin *h = nullptr;
    ~AladinHandle() { destroy(h); }
};

// reg_aladin<float>::Run (reg-lib/_reg_aladin.cpp:315-364) with InitialiseRegistration's
// centre alignment (:160-183); with cfg.symmetric, reg_aladin_sym<float> (reg-lib/_reg_aladin_sym.cpp):
// a backward handle (floating -> reference, every voxel active) shares the forward handle's
// stream, its matrix starts as the inverse of the forward one, and each iteration warps both
// ways, fits both ways and averages the two matrices on the device.
void aladin_register(const nrh_geom& refG, const float *refData, const nrh_geom& floG, const float *floData,
                     const nrh_aladin_config& cfg, float *out) {
    NRH_REQUIRE(cfg.levels >= 1 && cfg.max_iterations >= 0, NRH_ERR_ARG, "invalid Aladin configuration");
    NRH_REQUIRE(cfg.rigid || cfg.affine, NRH_ERR_ARG, "neither a rigid nor an affine stage requested");
    const int toPerform = cfg.levels_to_perform > 0 ? std::min(cfg.levels_to_perform, cfg.levels) : cfg.levels;
    float M[16] = { 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1 };
    if (cfg.align_centre) {
        auto centre = [](const nrh_geom& g, float c[3]) {
            const float v[3] = { (float)g.nx / 2.0f, (float)g.ny / 2.0f, (float)g.nz / 2.0f };
            for (int r = 0; r < 3; ++r)
                c[r] = (float)((double)g.xyz[r * 4] * v[0] + (double)g.xyz[r * 4 + 1] * v[1] +
                               (double)g.xyz[r * 4 + 2] * v[2] + (double)g.xyz[r * 4 + 3]);
        };
        float fc[3], rc[3];
        centre(floG, fc);
        centre(refG, rc);
        M[3] = fc[0] - rc[0];
        M[7] = fc[1] - rc[1];
        M[11] = fc[2] - rc[2];
    }
    float Mb[16];
    mat44_inverse(M, Mb);
    std::vector<DevLevel> rp, fp;
    {
        ScopedStream st;
        rp = device_pyramid(refG, refData, cfg.levels, toPerform, st.s);
        fp = device_pyramid(floG, floData, cfg.levels, toPerform, st.s);
    }
    const nrh_aladin_params params{ cfg.block_percent, cfg.inlier_lts, std::numeric_limits<float>::quiet_NaN() };
    for (int level = 0; level < toPerform; ++level) {
        AladinHandle ah, bh;  // bh (sharing ah's stream) is destroyed first
        ah.h = create(&rp[level].geom, std::move(rp[level].img), nullptr, &fp[level].geom, std::move(fp[level].img),
                      nullptr, nullptr, &params);
        nrh_aladin *h = ah.h, *b = nullptr;
        set_matrix(h, M);
        if (cfg.symmetric) {
            DevBuf<float> ri, fi;
            ri.alloc(h->N);
            fi.alloc(h->Nf);
            NRH_HIP(hipMemcpyAsync(ri.p, h->refImg.p, ri.bytes(), hipMemcpyDeviceToDevice, h->stream));
            NRH_HIP(hipMemcpyAsync(fi.p, h->floImg.p, fi.bytes(), hipMemcpyDeviceToDevice, h->stream));
            bh.h = create(&fp[level].geom, std::move(fi), nullptr, &rp[level].geom, std::move(ri), nullptr, nullptr,
                          &params, h->stream);
            b = bh.h;
            set_matrix(b, Mb);
        }
        const int maxIt = level == 0 ? 2 * cfg.max_iterations : cfg.max_iterations;
        auto resolve = [&](int iterations, bool affine) {
            for (int it = 0; it < iterations; ++it) {
                launch_warp(h);
                if (b) launch_warp(b);
                launch_block_matching(h);
                launch_lts(h, affine);
                if (b) {
                    launch_block_matching(b);
                    launch_lts(b, affine);
                    launch_symmetric_update(h, b);
                }
            }
        };
        if ((cfg.rigid && !cfg.affine) || (cfg.affine && cfg.rigid && level == 0))
            resolve(maxIt * ((cfg.affine && cfg.rigid && level == 0) ? 4 : 1), false);
        if (cfg.affine) resolve(maxIt, true);
        read_counters(h);
        raise_lts_status(h->pinned[1]);
        raise_symmetric_status(h->pinned[2]);
        if (b) {
            read_counters(b);
            raise_lts_status(b->pinned[1]);
            get_matrix(b, Mb);
        }
        get_matrix(h, M);
    }
    std::memcpy(out, M, sizeof(M));
}

// reg_aladin<float>::Run for many pairs at once (non-symmetric): every pair runs aladin_register's
// levels, stages and iterations, with the pairs' warps and block matchings launched in turn on one
// stream and all pairs' LTS fits in one launch (a workgroup each); an iteration of all pairs is
// captured once per stage as a HIP graph and replayed.  A pair whose block selection or fit fails
// (a flat image: fewer than 2 active blocks, or too few correspondences) stops with its error in
// status[q]; the other pairs go on.
void aladin_register_batch(int n, const nrh_geom *refs, const float *const *refData, const nrh_geom *flos,
                           const float *const *floData, const nrh_aladin_config& cfg, float *out, int *status,
                           nrh_batch_stats *stats) {
    NRH_REQUIRE(cfg.levels >= 1 && cfg.max_iterations >= 0, NRH_ERR_ARG, "invalid Aladin configuration");
    NRH_REQUIRE(cfg.rigid || cfg.affine, NRH_ERR_ARG, "neither a rigid nor an affine stage requested");
    NRH_REQUIRE(!cfg.symmetric, NRH_ERR_UNSUPPORTED, "batched Aladin runs the non-symmetric registration");
    const auto t0 = std::chrono::steady_clock::now();
    const int toPerform = cfg.levels_to_perform > 0 ? std::min(cfg.levels_to_perform, cfg.levels) : cfg.levels;
    std::vector<std::array<float, 16>> M(n);
    std::vector<std::vector<DevLevel>> rp(n), fp(n);
    std::vector<std::string> errs(n);
    std::vector<int> codes(n, NRH_ERR_ARG);
    {
        int device = 0;
        NRH_HIP(hipGetDevice(&device));
        std::vector<std::thread> pool;
        const int T = std::max(1, std::min(n, (int)std::thread::hardware_concurrency()));
        for (int t = 0; t < T; ++t)
            pool.emplace_back([&, t] {
                for (int q = t; q < n; q += T) {
                    try {
                        NRH_HIP(hipSetDevice(device));
                        ScopedStream st;
                        rp[q] = device_pyramid(refs[q], refData[q], cfg.levels, toPerform, st.s);
                        fp[q] = device_pyramid(flos[q], floData[q], cfg.levels, toPerform, st.s);
                    } catch (const Error& e) {
                        errs[q] = e.what();
                        codes[q] = e.code;
                    } catch (const std::exception& e) {
                        errs[q] = e.what();
                    }
                }
            });
        for (auto& th : pool) th.join();
    }
    for (int q = 0; q < n; ++q) {
        NRH_REQUIRE(errs[q].empty(), codes[q], "pair " + std::to_string(q) + ": " + errs[q]);
        float m[16] = { 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1 };
        if (cfg.align_centre) {
            auto centre = [](const nrh_geom& g, float c[3]) {
                const float v[3] = { (float)g.nx / 2.0f, (float)g.ny / 2.0f, (float)g.nz / 2.0f };
                for (int r = 0; r < 3; ++r)
                    c[r] = (float)((double)g.xyz[r * 4] * v[0] + (double)g.xyz[r * 4 + 1] * v[1] +
                                   (double)g.xyz[r * 4 + 2] * v[2] + (double)g.xyz[r * 4 + 3]);
            };
            float fc[3], rc[3];
            centre(flos[q], fc);
            centre(refs[q], rc);
            m[3] = fc[0] - rc[0];
            m[7] = fc[1] - rc[1];
            m[11] = fc[2] - rc[2];
        }
        std::copy(m, m + 16, M[q].begin());
        status[q] = NRH_OK;
    }
    hipStream_t stream;
    NRH_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    struct StreamOwner {
        hipStream_t s;
        ~StreamOwner() { (void)hipStreamSynchronize(s); (void)hipStreamDestroy(s); }
    } so{ stream };
    const nrh_aladin_params params{ cfg.block_percent, cfg.inlier_lts, std::numeric_limits<float>::quiet_NaN() };
    double deviceSeconds = 0.0;
    int replays = 0;
    for (int level = 0; level < toPerform; ++level) {
        std::vector<AladinHandle> hs(n);
        std::vector<nrh_aladin *> live;
        std::vector<int> liveIdx;
        for (int q = 0; q < n; ++q) {
            if (status[q] != NRH_OK) continue;
            try {
                hs[q].h = create(&rp[q][level].geom, std::move(rp[q][level].img), nullptr, &fp[q][level].geom,
                                 std::move(fp[q][level].img), nullptr, nullptr, &params, stream);
                set_matrix(hs[q].h, M[q].data());
                live.push_back(hs[q].h);
                liveIdx.push_back(q);
            } catch (const Error& e) {
                if (e.code != NRH_ERR_NUMERIC) throw;
                status[q] = e.code;  // this pair stops; the others go on
            }
        }
        if (live.empty()) break;
        const int L = (int)live.size();
        std::vector<LtsArgs> la(L);
        for (int k = 0; k < L; ++k) {
            nrh_aladin *h = live[k];
            la[k] = LtsArgs{ h->refPos.p, h->warpPos.p, h->activeBlocks, h->matrix.p, h->ltsP.p, h->ltsQ.p, h->ltsRes.p,
                             h->params.inlier_lts, h->counters.p + 1 };
        }
        DevBuf<LtsArgs> dla;
        dla.alloc(L);
        NRH_HIP(hipMemcpyAsync(dla.p, la.data(), L * sizeof(LtsArgs), hipMemcpyHostToDevice, stream));
        NRH_HIP(hipStreamSynchronize(stream));
        const int maxIt = level == 0 ? 2 * cfg.max_iterations : cfg.max_iterations;
        auto resolve = [&](int iterations, bool affine) {
            if (iterations <= 0) return;
            hipGraph_t graph = nullptr;
            hipGraphExec_t exec = nullptr;
            NRH_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
            for (nrh_aladin *h : live) {
                launch_warp(h);
                launch_block_matching(h);
            }
            hipLaunchKernelGGL(k_lts_batch, dim3(L), dim3(kLtsThreads), 0, stream, dla.p, affine ? 1 : 0);
            NRH_HIP(hipStreamEndCapture(stream, &graph));
            const hipError_t ie = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
            (void)hipGraphDestroy(graph);
            NRH_HIP(ie);
            const auto d0 = std::chrono::steady_clock::now();
            hipError_t ge = hipSuccess;
            for (int it = 0; it < iterations && ge == hipSuccess; ++it, ++replays) ge = hipGraphLaunch(exec, stream);
            if (ge == hipSuccess) ge = hipStreamSynchronize(stream);
            (void)hipGraphExecDestroy(exec);
            NRH_HIP(ge);
            deviceSeconds += std::chrono::duration<double>(std::chrono::steady_clock::now() - d0).count();
        };
        if ((cfg.rigid && !cfg.affine) || (cfg.affine && cfg.rigid && level == 0))
            resolve(maxIt * ((cfg.affine && cfg.rigid && level == 0) ? 4 : 1), false);
        if (cfg.affine) resolve(maxIt, true);
        for (int k = 0; k < L; ++k) {
            nrh_aladin *h = live[k];
            read_counters(h);
            const int q = liveIdx[k];
            if (h->pinned[1] != 0) {
                status[q] = NRH_ERR_NUMERIC;  // too few correspondences or a singular fit
                continue;
            }
            get_matrix(h, M[q].data());
        }
    }
    for (int q = 0; q < n; ++q) std::copy(M[q].begin(), M[q].end(), out + 16 * q);
    if (stats) {
        stats->seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
        stats->device_seconds = deviceSeconds;
        stats->graph_replays = replays;
    }
}

// ------------------------------------------------------------------ allocation-free LTS
// Scratch of nrh_lts_static: the compacted correspondences (3 n floats each) and the residual
// bits plus keep bytes (n + n / 4 words) of one fit of at most kLtsStaticMax correspondences
// (7.6 MB on every GPU the library runs on, held until the process ends).  Host code never uses
// the array's name as an address: each device's address comes from hipGetSymbolAddress.
constexpr int kLtsStaticMax = 262144;
constexpr size_t kLtsScratchWords = 6 * (size_t)kLtsStaticMax + kLtsStaticMax + (kLtsStaticMax + 3) / 4;
static __device__ __align__(256) uint32_t scratch[kLtsScratchWords];

}  // namespace

// The address of `scratch` on the current device, looked up once per device (nrh_init does it for
// the device it selects; nrh_lts_static for any other current device on its first call there).
uint32_t *lts_static_scratch() {
    static std::mutex mu;
    static std::map<int, uint32_t *> ptrs;
    int dev = 0;
    NRH_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(mu);
    auto it = ptrs.find(dev);
    if (it != ptrs.end()) return it->second;
    uint32_t *ptr = nullptr;
    NRH_HIP(hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch)));
    NRH_REQUIRE(ptr != nullptr, NRH_ERR_HIP, "no device address for the LTS scratch");
    ptrs[dev] = ptr;
    return ptr;
}

}  // namespace nrh

using namespace nrh;

extern "C" {

int nrh_aladin_create(const nrh_geom *ref, const float *ref_data, const nrh_geom *flo, const float *flo_data,
                      const int *mask, const nrh_aladin_params *params, nrh_aladin **out) {
    return guard([&] {
        NRH_REQUIRE(out, NRH_ERR_ARG, "null output handle");
        *out = nullptr;
        *out = create(ref, DevBuf<float>(), ref_data, flo, DevBuf<float>(), flo_data, mask, params);
    });
}

int nrh_aladin_register_batch(int n, const nrh_geom *refs, const float *const *ref_data, const nrh_geom *flos,
                              const float *const *flo_data, const nrh_aladin_config *cfg, float *matrices,
                              int *status, nrh_batch_stats *stats) {
    return guard([&] {
        NRH_REQUIRE(n >= 1 && refs && ref_data && flos && flo_data && cfg && matrices && status, NRH_ERR_ARG,
                    "null argument");
        for (int q = 0; q < n; ++q) {
            check_geom(&refs[q], "reference");
            check_geom(&flos[q], "floating");
            NRH_REQUIRE(ref_data[q] && flo_data[q], NRH_ERR_ARG, "null image");
            NRH_REQUIRE(refs[q].nz > 1, NRH_ERR_UNSUPPORTED, "2-D images are not supported");
        }
        if (stats) *stats = nrh_batch_stats{};
        aladin_register_batch(n, refs, ref_data, flos, flo_data, *cfg, matrices, status, stats);
    });
}

int nrh_aladin_destroy(nrh_aladin *h) {
    return guard([&] { destroy(h); });
}

int nrh_aladin_blocks(nrh_aladin *h, int counts[3], int *total_block) {
    return guard([&] {
        NRH_REQUIRE(h && counts, NRH_ERR_ARG, "null argument");
        read_counters(h);
        counts[0] = h->totalBlocks;
        counts[1] = h->activeBlocks;
        counts[2] = h->pinned[0];
        if (total_block) std::memcpy(total_block, h->totalBlock.data(), h->totalBlocks * sizeof(int));
    });
}

int nrh_aladin_set_matrix(nrh_aladin *h, const float m[16]) {
    return guard([&] {
        NRH_REQUIRE(h && m, NRH_ERR_ARG, "null argument");
        set_matrix(h, m);
    });
}

int nrh_aladin_get_matrix(nrh_aladin *h, float m[16]) {
    return guard([&] {
        NRH_REQUIRE(h && m, NRH_ERR_ARG, "null argument");
        get_matrix(h, m);
    });
}

int nrh_aladin_warp(nrh_aladin *h) {
    return guard([&] {
        NRH_REQUIRE(h, NRH_ERR_ARG, "null handle");
        launch_warp(h);
    });
}

int nrh_aladin_upload_warped(nrh_aladin *h, const float *warped) {
    return guard([&] {
        NRH_REQUIRE(h && warped, NRH_ERR_ARG, "null argument");
        NRH_HIP(hipMemcpyAsync(h->warped.p, warped, h->N * sizeof(float), hipMemcpyHostToDevice, h->stream));
        NRH_HIP(hipStreamSynchronize(h->stream));
    });
}

int nrh_aladin_download_warped(nrh_aladin *h, float *warped) {
    return guard([&] {
        NRH_REQUIRE(h && warped, NRH_ERR_ARG, "null argument");
        NRH_HIP(hipMemcpyAsync(warped, h->warped.p, h->N * sizeof(float), hipMemcpyDeviceToHost, h->stream));
        NRH_HIP(hipStreamSynchronize(h->stream));
    });
}

int nrh_aladin_block_matching(nrh_aladin *h) {
    return guard([&] {
        NRH_REQUIRE(h, NRH_ERR_ARG, "null handle");
        launch_block_matching(h);
    });
}

int nrh_aladin_download_positions(nrh_aladin *h, float *ref_pos, float *warp_pos, int *defined) {
    return guard([&] {
        NRH_REQUIRE(h, NRH_ERR_ARG, "null handle");
        const size_t bytes = 3 * (size_t)h->activeBlocks * sizeof(float);
        if (ref_pos) NRH_HIP(hipMemcpyAsync(ref_pos, h->refPos.p, bytes, hipMemcpyDeviceToHost, h->stream));
        if (warp_pos) NRH_HIP(hipMemcpyAsync(warp_pos, h->warpPos.p, bytes, hipMemcpyDeviceToHost, h->stream));
        read_counters(h);
        if (defined) *defined = h->pinned[0];
    });
}

int nrh_aladin_lts(nrh_aladin *h, int affine) {
    return guard([&] {
        NRH_REQUIRE(h, NRH_ERR_ARG, "null handle");
        NRH_HIP(hipMemsetAsync(h->counters.p + 1, 0, sizeof(int), h->stream));
        launch_lts(h, affine != 0);
        read_counters(h);
        raise_lts_status(h->pinned[1]);
    });
}

int nrh_lts_static(const float *ref_pos, const float *warp_pos, int n, int inlier_lts, int affine, float *matrix,
                   int *status, void *stream) {
    return guard([&] {
        NRH_REQUIRE(ref_pos && warp_pos && matrix && status, NRH_ERR_ARG, "null argument");
        NRH_REQUIRE(n > 0, NRH_ERR_ARG, "no correspondences");
        NRH_REQUIRE(n <= kLtsStaticMax, NRH_ERR_ARG,
                    "nrh_lts_static takes at most 262144 correspondences (its static scratch); use nrh_lts");
        NRH_REQUIRE(inlier_lts > 0 && inlier_lts <= 100, NRH_ERR_ARG, "LTS inlier percentage must be in (0, 100]");
        uint32_t *base = lts_static_scratch();
        float *P = (float *)base, *Q = P + 3 * (size_t)n;
        uint32_t *res = (uint32_t *)(Q + 3 * (size_t)n);
        hipStream_t st = (hipStream_t)stream;
        hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(64), 0, st, status);
        launch_lts(st, ref_pos, warp_pos, n, matrix, P, Q, res, inlier_lts, affine ? 1 : 0, status);
        NRH_HIP(hipGetLastError());
    });
}

int nrh_lts(const float *ref_pos, const float *warp_pos, int n, int inlier_lts, int affine, float m[16]) {
    return guard([&] {
        NRH_REQUIRE(ref_pos && warp_pos && m, NRH_ERR_ARG, "null argument");
        NRH_REQUIRE(n > 0, NRH_ERR_ARG, "no correspondences");
        NRH_REQUIRE(inlier_lts > 0 && inlier_lts <= 100, NRH_ERR_ARG, "LTS inlier percentage must be in (0, 100]");
        hipStream_t stream;
        NRH_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
        struct StreamGuard {
            hipStream_t s;
            ~StreamGuard() { (void)hipStreamSynchronize(s); (void)hipStreamDestroy(s); }
        } sg{ stream };
        DevBuf<float> rp, wp, mat, P, Q;
        DevBuf<uint32_t> res;
        DevBuf<int> status;
        const size_t bytes = 3 * (size_t)n * sizeof(float);
        rp.alloc(3 * (size_t)n);
        wp.alloc(3 * (size_t)n);
        P.alloc(3 * (size_t)n);
        Q.alloc(3 * (size_t)n);
        res.alloc((size_t)n + (n + 3) / 4);
        mat.alloc(16);
        status.alloc(1);
        NRH_HIP(hipMemcpyAsync(rp.p, ref_pos, bytes, hipMemcpyHostToDevice, stream));
        NRH_HIP(hipMemcpyAsync(wp.p, warp_pos, bytes, hipMemcpyHostToDevice, stream));
        NRH_HIP(hipMemcpyAsync(mat.p, m, 16 * sizeof(float), hipMemcpyHostToDevice, stream));
        NRH_HIP(hipMemsetAsync(status.p, 0, sizeof(int), stream));
        launch_lts(stream, rp.p, wp.p, n, mat.p, P.p, Q.p, res.p, inlier_lts, affine ? 1 : 0, status.p);
        NRH_HIP(hipGetLastError());
        int st = 0;
        float out[16];
        NRH_HIP(hipMemcpyAsync(&st, status.p, sizeof(int), hipMemcpyDeviceToHost, stream));
        NRH_HIP(hipMemcpyAsync(out, mat.p, sizeof(out), hipMemcpyDeviceToHost, stream));
        NRH_HIP(hipStreamSynchronize(stream));
        raise_lts_status(st);
        std::memcpy(m, out, sizeof(out));
    });
}

int nrh_aladin_symmetric_update(nrh_aladin *forward, nrh_aladin *backward) {
    return guard([&] {
        NRH_REQUIRE(forward && backward && forward != backward, NRH_ERR_ARG, "two distinct handles are required");
        NRH_HIP(hipMemsetAsync(forward->counters.p + 2, 0, sizeof(int), forward->stream));
        launch_symmetric_update(forward, backward);
        read_counters(forward);
        if (backward->stream != forward->stream) NRH_HIP(hipStreamSynchronize(backward->stream));
        raise_symmetric_status(forward->pinned[2]);
    });
}

int nrh_aladin_register(const nrh_geom *ref, const float *ref_data, const nrh_geom *flo, const float *flo_data,
                        const nrh_aladin_config *cfg, float matrix[16]) {
    return guard([&] {
        check_geom(ref, "reference");
        check_geom(flo, "floating");
        NRH_REQUIRE(ref_data && flo_data && cfg && matrix, NRH_ERR_ARG, "null argument");
        aladin_register(*ref, ref_data, *flo, flo_data, *cfg, matrix);
    });
}

}  // extern "C"

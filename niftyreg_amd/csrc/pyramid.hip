// The image pyramid of a registration, built on the device: reg_createImagePyramid<float>
// (reg-lib/cpu/_reg_tools.cpp:1705-1733), whose levels are reg_downsampleImage<float> (:1343-1467):
// Gaussian smoothing (sigma 0.7355 voxel) and nearest-neighbour decimation by 2.

#include "device.hpp"
#include "host.hpp"
#include <cmath>

namespace nrh {
namespace {

// The smoothing's kernel, reg_tools_kernelConvolution's Gaussian of 0.7355 voxel
// (reg-lib/cpu/_reg_tools.cpp:868-904): radius (int)(3 sigma) = 2.
constexpr int kRadius = 2, kTaps = 2 * kRadius + 1;
struct SmoothKernel {
    float k[kTaps];
};

// One line sum of reg_tools_kernelConvolution in the order of the reference's default x86 build
// (USE_SSE with SSE3, reg-lib/cpu/_reg_tools.cpp:1017-1047) at position c of a line of L values, v
// the values under the kernel's taps (those outside the line are not used): four float lanes over a
// whole group of four taps, reduced pairwise, the other taps added in double.  Five taps hold at
// most one group, the first four inside the line.  Every index is a constant: v stays in registers.
__device__ __forceinline__ float line_sum(const SmoothKernel& K, const int c, const int L, const float (&v)[kTaps]) {
#pragma clang fp contract(off)
    static_assert(kTaps == 5, "the groups below are written for five taps");
    const int first = max(kRadius - c, 0), last = min(c + kRadius + 1, L) - c + kRadius;  // taps [first, last)
    float p[kTaps];
#pragma unroll
    for (int j = 0; j < kTaps; ++j) p[j] = K.k[j] * v[j];
    double s = 0.0;
    if (last - first >= 4) {
        const bool from0 = first == 0;
        const float a0 = (from0 ? p[0] : p[1]) + 0.f, a1 = (from0 ? p[1] : p[2]) + 0.f;
        const float a2 = (from0 ? p[2] : p[3]) + 0.f, a3 = (from0 ? p[3] : p[4]) + 0.f;
        s = (double)((a3 + a2) + (a1 + a0));
        if (last - first == 5) s += (double)p[4];
    } else {
#pragma unroll
        for (int j = 0; j < kTaps; ++j)
            if (j >= first && j < last) s += (double)p[j];
    }
    return (float)s;
}

// One voxel of the next level per thread: the input voxel it takes (the reference's float mapping
// through both matrices, whatever they are), and the three axis sums of image and density there.
// The separable passes round to float between the axes, and a sum at one voxel needs the earlier
// axis's sums only in its own 5 x 5 neighbourhood, so a thread forms those itself: 125 loads (L1 and
// L2 serve all but the first) and no smoothed copy in memory, so a pyramid needs no more memory
// than its levels.  Bound by those cached loads.  It replaces loops on the host, which were most of
// a registration's time: one symmetric affine registration at 181 x 217 x 181 went from 298 to
// 74 ms, 16 affine ones at 128^3 from 735 to 123 ms, one F3D registration at 128 x 144 x 112 (70
// iterations) from 113 to 13 ms.
__global__ void __launch_bounds__(256)
k_downsample(const float *__restrict__ in, int nx, int ny, int nz, Affine inIjk, float *__restrict__ out, int mx,
             int my, int mz, Affine outXyz, SmoothKernel K) {
#pragma clang fp contract(off)
    const size_t n = (size_t)mx * my * mz, idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n) return;
    int x, y, z;
    index_xyz(idx, mx, my, x, y, z);
    float real[3];
    int pos[3];
    for (int r = 0; r < 3; ++r) real[r] = node_pos(outXyz, r, x, y, z);
    for (int r = 0; r < 3; ++r) {
        const float *m = inIjk.m + 4 * r;
        const float p = real[0] * m[0] + real[1] * m[1] + real[2] * m[2] + m[3];
        // (int) of a value outside the int range is undefined: such a voxel lies outside anyway
        pos[r] = fabsf(p) < 1e9f ? (int)(p + (p >= 0 ? 0.5f : -0.5f)) : -1;
    }
    if (nz == 1) pos[2] = 0;
    const float nan = __builtin_nanf("");
    if (pos[0] < 0 || pos[0] >= nx || pos[1] < 0 || pos[1] >= ny || pos[2] < 0 || pos[2] >= nz) {
        out[idx] = nan;
        return;
    }
    const float *centre = in + ((size_t)pos[2] * ny + pos[1]) * nx + pos[0];
    if (!(*centre == *centre)) {
        out[idx] = nan;
        return;
    }
    float iz[kTaps], dz[kTaps];
#pragma unroll
    for (int c = 0; c < kTaps; ++c) {
        const int Z = pos[2] + c - kRadius;
        iz[c] = dz[c] = 0.f;
        if (Z < 0 || Z >= nz) continue;
        float iy[kTaps], dy[kTaps];
#pragma unroll
        for (int b = 0; b < kTaps; ++b) {
            const int Y = pos[1] + b - kRadius;
            iy[b] = dy[b] = 0.f;
            if (Y < 0 || Y >= ny) continue;
            const float *row = in + ((size_t)Z * ny + Y) * nx;
            float v[kTaps], d[kTaps];
#pragma unroll
            for (int a = 0; a < kTaps; ++a) v[a] = row[min(max(pos[0] + a - kRadius, 0), nx - 1)];
#pragma unroll
            for (int a = 0; a < kTaps; ++a) {
                d[a] = v[a] == v[a] ? 1.f : 0.f;
                v[a] = v[a] == v[a] ? v[a] : 0.f;
            }
            // an axis of one voxel is not smoothed
            iy[b] = nx > 1 ? line_sum(K, pos[0], nx, v) : v[kRadius];
            dy[b] = nx > 1 ? line_sum(K, pos[0], nx, d) : d[kRadius];
        }
        iz[c] = ny > 1 ? line_sum(K, pos[1], ny, iy) : iy[kRadius];
        dz[c] = ny > 1 ? line_sum(K, pos[1], ny, dy) : dy[kRadius];
    }
    const float i = nz > 1 ? line_sum(K, pos[2], nz, iz) : iz[kRadius];
    const float d = nz > 1 ? line_sum(K, pos[2], nz, dz) : dz[kRadius];
    out[idx] = i / d;
}

void downsample_device(const DevLevel& in, DevLevel& out, hipStream_t stream) {
    const bool axes[3] = { in.geom.nx / 2 >= 32, in.geom.ny / 2 >= 32, in.geom.nz / 2 >= 32 };
    downsampled_geometry(in.geom, axes, out.geom);
    const size_t n = voxels(out.geom);
    out.img.alloc(n);
    SmoothKernel K;
    const double sigma = std::fabs((double)-0.7355f);
    for (int i = -kRadius; i <= kRadius; ++i)
        K.k[i + kRadius] = (float)(std::exp(-(double)(i * i) / (2.0 * (sigma * sigma))) / (sigma * 2.506628274631));
    hipLaunchKernelGGL(k_downsample, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, in.img.p, in.geom.nx,
                       in.geom.ny, in.geom.nz, to_affine(in.geom.ijk), out.img.p, out.geom.nx, out.geom.ny,
                       out.geom.nz, to_affine(out.geom.xyz), K);
    NRH_HIP(hipGetLastError());
}

}  // namespace

std::vector<DevLevel> device_pyramid(const nrh_geom& g, const float *data, int levels, int toPerform,
                                     hipStream_t stream) {
    std::vector<DevLevel> p(toPerform);
    DevLevel cur;
    cur.geom = g;
    cur.img.alloc(voxels(g));
    NRH_HIP(hipMemcpyAsync(cur.img.p, data, voxels(g) * sizeof(float), hipMemcpyHostToDevice, stream));
    std::vector<DevLevel> dropped;  // levels above the first one performed, read by queued kernels
    for (int l = toPerform; l < levels; ++l) {
        DevLevel nxt;
        downsample_device(cur, nxt, stream);
        dropped.push_back(std::move(cur));
        cur = std::move(nxt);
    }
    p[toPerform - 1] = std::move(cur);
    for (int l = toPerform - 2; l >= 0; --l) downsample_device(p[l + 1], p[l], stream);
    NRH_HIP(hipStreamSynchronize(stream));
    return p;
}

}  // namespace nrh

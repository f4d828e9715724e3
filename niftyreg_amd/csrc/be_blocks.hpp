// Bending-energy building blocks shared by the per-operation kernels (f3d_ops.hip) and the
// fused exact-pass launch (f3d_fused.hip): the 27-point basis table, the node bricks and the
// value block body.
#pragma once

#include "device.hpp"

namespace nrh {

// Tensor products of the cubic B-spline at a node and its neighbours (value {1/6, 2/3, 1/6}, first
// derivative {-1/2, 0, 1/2}, second derivative {1, -2, 1}), rounded to the 6-decimal literals the
// reference tabulates (reg-lib/cpu/_reg_splineBasis.cpp:292-457).  A constant: in the unrolled
// stencils every value is an instruction's literal, where a table in LDS cost a read per neighbour.
struct BeBasis {
    float b[6][27];  // xx, yy, zz, xy, yz, xz
};

constexpr float round6(double v) {
    const double a = (v < 0 ? -v : v) * 1e6 + 0.5;
    const double r = (double)(long long)a / 1e6;
    return (float)(v < 0 ? -r : r);
}

constexpr BeBasis make_be_basis() {
    const double v[3] = { 1.0 / 6.0, 2.0 / 3.0, 1.0 / 6.0 }, d1[3] = { -0.5, 0.0, 0.5 }, d2[3] = { 1.0, -2.0, 1.0 };
    BeBasis B{};
    int i = 0;
    for (int c = 0; c < 3; ++c)
        for (int b = 0; b < 3; ++b)
            for (int a = 0; a < 3; ++a, ++i) {
                B.b[0][i] = round6(d2[a] * v[b] * v[c]);
                B.b[1][i] = round6(v[a] * d2[b] * v[c]);
                B.b[2][i] = round6(v[a] * v[b] * d2[c]);
                B.b[3][i] = round6(d1[a] * d1[b] * v[c]);
                B.b[4][i] = round6(v[a] * d1[b] * d1[c]);
                B.b[5][i] = round6(d1[a] * v[b] * d1[c]);
            }
    return B;
}

// Bending energy on bricks of 8 x 8 x 4 nodes: a workgroup takes one component of a brick, one node
// per thread, and stages the component's control points of the brick and its halo in LDS once, so
// every 27-neighbour stencil reads LDS instead of global memory.  The three components of a brick
// are independent until its energy is summed; a workgroup each fills the chip three times better
// (16 bricks at 64^3, 441 at 256 x 256 x 160, for 256 compute units) at a third of the LDS.
constexpr int BBX = 8, BBY = 8, BBZ = 4;

struct BrickGrid {
    int bx, by, bz;  // bricks per axis
};

__device__ __forceinline__ void brick_origin(const BrickGrid& g, int b, int& x0, int& y0, int& z0) {
    x0 = (b % g.bx) * BBX;
    y0 = ((b / g.bx) % g.by) * BBY;
    z0 = (b / (g.bx * g.by)) * BBZ;
}

// Stages component c of the control points of a brick at (x0, y0, z0) with a halo of H nodes into
// sC; DISP: as displacements from the nodes.  Points outside the grid are 0, so a stencil over them
// adds nothing and needs no bounds checks.
template<int H, bool DISP>
__device__ __forceinline__ void stage_brick(const float *__restrict__ cpp, int gnx, int gny, int gnz, const Affine& xyz,
                                            int c, int x0, int y0, int z0, float *sC) {
#pragma clang fp contract(off)
    constexpr int HX = BBX + 2 * H, HY = BBY + 2 * H, HZ = BBZ + 2 * H, HN = HX * HY * HZ;
    constexpr int kIter = (HN + 255) / 256;
    const float *p = cpp + (size_t)c * gnx * gny * gnz;
    float v[kIter];
#pragma unroll
    for (int u = 0; u < kIter; ++u) {
        // clamped, unconditional loads: all in flight before the first is used
        const int r = min((int)threadIdx.x + u * 256, HN - 1);
        const int X = x0 - H + r % HX, Y = y0 - H + (r / HX) % HY, Z = z0 - H + r / (HX * HY);
        const int cx = min(max(X, 0), gnx - 1), cy = min(max(Y, 0), gny - 1), cz = min(max(Z, 0), gnz - 1);
        v[u] = p[((size_t)cz * gny + cy) * gnx + cx];
        if (DISP) v[u] -= node_pos(xyz, c, cx, cy, cz);
        if (cx != X || cy != Y || cz != Z) v[u] = 0.f;
    }
#pragma unroll
    for (int u = 0; u < kIter; ++u)
        if ((int)threadIdx.x + u * 256 < HN) sC[threadIdx.x + u * 256] = v[u];
}

// reg_spline_approxBendingEnergyValue3D (reg-lib/cpu/_reg_localTrans_regul.cpp:73-153): component c
// over the interior nodes of brick bid, an FP64 partial into partials[3 bid + c].  The partials are
// summed by sum_partials_256 in the kernel that needs the energy: a ticket here, with its fence and
// an atomic on one address per workgroup, took longer than the bricks.
__device__ __forceinline__ void
be_value_block(const float *__restrict__ cpp, int gnx, int gny, int gnz, BrickGrid bg, double *__restrict__ partials,
               int bid, int c) {
#pragma clang fp contract(off)
    constexpr BeBasis B = make_be_basis();
    constexpr int HX = BBX + 2, HY = BBY + 2, HN = HX * HY * (BBZ + 2);
    __shared__ float sC[HN];
    __shared__ double red[16];
    int x0, y0, z0;
    brick_origin(bg, bid, x0, y0, z0);
    stage_brick<1, false>(cpp, gnx, gny, gnz, Affine{}, c, x0, y0, z0, sC);
    __syncthreads();
    const int tx = threadIdx.x % BBX, ty = (threadIdx.x / BBX) % BBY, tz = threadIdx.x / (BBX * BBY);
    const int x = x0 + tx, y = y0 + ty, z = z0 + tz;
    double s = 0;
    if (x > 0 && y > 0 && z > 0 && x < gnx - 1 && y < gny - 1 && z < gnz - 1) {
        float d[6] = {};
#pragma unroll
        for (int i = 0; i < 27; ++i) {
            const float cv = sC[((tz + i / 9) * HY + ty + (i / 3) % 3) * HX + tx + i % 3];
#pragma unroll
            for (int t = 0; t < 6; ++t) d[t] += B.b[t][i] * cv;
        }
        if (c == 0) {
            s = (double)(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]) +
                2.0 * (double)(d[3] * d[3] + d[4] * d[4] + d[5] * d[5]);
        } else {
            s += (double)(d[0] * d[0]);
            s += (double)(d[1] * d[1]);
            s += (double)(d[2] * d[2]);
            s += 2.0 * (double)(d[3] * d[3] + d[4] * d[4] + d[5] * d[5]);
        }
    }
    s = block_sum_double(s, red);
    if (threadIdx.x == 0) partials[3 * bid + c] = s;
}

// reg_spline_approxBendingEnergyGradient3D (regul.cpp:287-451) for component c of brick bid: the
// displacement (cpp - node) of the brick with a two-node halo in LDS, the 6 second derivatives of
// every node of the brick with a one-node halo (regul.cpp:317-379, the cross terms doubled in
// double), then the adjoint 27-point gather (regul.cpp:381-448) into out (planar [3][G]) for a later
// grad += weight / G * value.  The derivatives of nodes outside the grid are 0.
__device__ __forceinline__ void
be_gradient_block(const float *__restrict__ cpp, int gnx, int gny, int gnz, BrickGrid bg, const Affine& xyz,
                  float *__restrict__ out, int bid, int c) {
#pragma clang fp contract(off)
    constexpr BeBasis B = make_be_basis();
    constexpr int CX = BBX + 4, CY = BBY + 4, CN = CX * CY * (BBZ + 4);  // points: two-node halo
    constexpr int DX = BBX + 2, DY = BBY + 2, DN = DX * DY * (BBZ + 2);  // derivatives: one-node halo
    __shared__ float sC[CN];
    __shared__ float sD[6][DN];
    int x0, y0, z0;
    brick_origin(bg, bid, x0, y0, z0);
    stage_brick<2, true>(cpp, gnx, gny, gnz, xyz, c, x0, y0, z0, sC);
    __syncthreads();
    for (int r = threadIdx.x; r < DN; r += 256) {
        const int hx = r % DX, hy = (r / DX) % DY, hz = r / (DX * DY);
        const int x = x0 - 1 + hx, y = y0 - 1 + hy, z = z0 - 1 + hz;
        const bool in = x >= 0 && y >= 0 && z >= 0 && x < gnx && y < gny && z < gnz;
        float d[6] = {};
#pragma unroll
        for (int i = 0; i < 27; ++i) {
            const float cv = sC[((hz + i / 9) * CY + hy + (i / 3) % 3) * CX + hx + i % 3];
#pragma unroll
            for (int t = 0; t < 6; ++t) d[t] += B.b[t][i] * cv;
        }
#pragma unroll
        for (int t = 0; t < 6; ++t) sD[t][r] = !in ? 0.f : t < 3 ? d[t] : (float)(2.0 * (double)d[t]);
    }
    __syncthreads();
    const int tx = threadIdx.x % BBX, ty = (threadIdx.x / BBX) % BBY, tz = threadIdx.x / (BBX * BBY);
    const int x = x0 + tx, y = y0 + ty, z = z0 + tz;
    if (x >= gnx || y >= gny || z >= gnz) return;
    float g = 0.f;
#pragma unroll
    for (int i = 0; i < 27; ++i) {
        const int r = ((tz + i / 9) * DY + ty + (i / 3) % 3) * DX + tx + i % 3;
#pragma unroll
        for (int t = 0; t < 6; ++t) g += sD[t][r] * B.b[t][i];
    }
    out[(((size_t)c * gnz + z) * gny + y) * gnx + x] = g;
}

// The sum of n partials in the order of one workgroup of 256 (thread t sums partials t, t + 256, ...,
// then block_sum_double), for any workgroup of at least 256 threads; valid on thread 0.
__device__ __forceinline__ double sum_partials_256(const double *__restrict__ partials, int n, double *red) {
    double t = 0;
    if (threadIdx.x < 256)
        for (int i = threadIdx.x; i < n; i += 256) t += partials[i];
    return block_sum_double(t, red);
}

// max(*maxBits, the block's largest bits): one atomic per block, and none once a larger value is
// there (lengths >= 0 order like their bit patterns).  Every thread of the workgroup calls it.  An
// atomic per wave on the one address held a kernel of 1664 waves up for 12 us.
__device__ __forceinline__ void block_track_max(uint32_t *maxBits, uint32_t bits) {
    __shared__ uint32_t sMax[16];
    for (int off = 32; off > 0; off >>= 1) {
        const uint32_t o = __shfl_down(bits, off, 64);
        bits = o > bits ? o : bits;
    }
    if ((threadIdx.x & 63) == 0) sMax[threadIdx.x >> 6] = bits;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (unsigned w = 1; w < (blockDim.x + 63) / 64; ++w) bits = sMax[w] > bits ? sMax[w] : bits;
        if (bits > __hip_atomic_load(maxBits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(maxBits, bits);
    }
}

// The brick grid of a control-point grid.
inline BrickGrid be_brick_grid(int gnx, int gny, int gnz) {
    BrickGrid g;
    g.bx = (gnx + BBX - 1) / BBX;
    g.by = (gny + BBY - 1) / BBY;
    g.bz = (gnz + BBZ - 1) / BBZ;
    return g;
}

}  // namespace nrh

// The reference-order convolution of the voxel gradient and its sampling at the nodes, evaluated
// only where the nodes read it.
//
// Compute::ConvolveVoxelBasedMeasureGradient (reg-lib/Compute.cpp:230-281) convolves the voxel
// gradient along x, y and z over the whole image and interpolates the result at the nodes.  On a
// grid whose spacing is s voxels a node reads two voxels per axis, so of the x pass only about 2 / s
// of the columns are ever used, of the y pass (2 / s)^2 and of the z pass (2 / s)^3.  Each pass here
// writes a compact array of the positions that are read further on.  Every sum is the one that
// op_convolve_voxel_gradient forms at that voxel (same taps, same order, same density, same division
// after each axis) and the interpolation is k_voxel_to_node's, so the node gradient is equal bit for
// bit.

#include "f3d_handle.hpp"
#include "device.hpp"
#include <algorithm>
#include <cmath>

namespace nrh {

namespace {

constexpr int kB = 256;

struct PassArgs {
    const float *in;   // [3][iz][iy][ix]
    float *out;        // the same with the pass's axis replaced by its listed positions
    int ox, oy, oz;    // output size
    int L;             // input size along the axis
    size_t inPlane, outPlane, stride, rowStride, sliceStride;  // strides of the input
    int axis;
    const int *list;   // position of each listed output along the axis
    const float *dens; // density at each listed position where every tap is a number
    const float *kern;
    int radius, order;
};

// One output per thread, the three components in blockIdx.y.  The density of a line without NaN
// depends on the position alone (dens); a NaN among the taps sends the lane through the loop that
// sums the density as well.  Bound by its cached tap loads and FP64 sums: at 181 x 150 x 120 with a
// 5 mm grid over 1.1 x 0.95 x 1.2 mm voxels the three passes take 118 us, where the
// whole-image convolution took 650 (the evaluation 1144 -> 601 us).
__global__ void __launch_bounds__(kB) k_conv_listed(PassArgs p) {
#pragma clang fp contract(off)
    const size_t t = (size_t)blockIdx.x * kB + threadIdx.x;
    if (t >= p.outPlane) return;
    int x, y, z;
    index_xyz(t, p.ox, p.oy, x, y, z);
    const int u = p.axis == 0 ? x : p.axis == 1 ? y : z;
    const int l = p.list[u];
    const float *line = p.in + blockIdx.y * p.inPlane;
    line += p.axis == 0 ? (size_t)y * p.rowStride + (size_t)z * p.sliceStride
          : p.axis == 1 ? (size_t)x + (size_t)z * p.sliceStride
                        : (size_t)x + (size_t)y * p.rowStride;
    const float centre = line[(size_t)l * p.stride];
    float *out = p.out + blockIdx.y * p.outPlane + t;
    if (!(centre == centre)) {
        *out = __builtin_nanf("");
        return;
    }
    if (p.radius <= 0 || p.L <= 1) {
        *out = centre;
        return;
    }
    const int pre = max(l - p.radius, 0), pst = min(l + p.radius + 1, p.L), k0 = max(p.radius - l, 0);
    double is = 0;
    bool bad = false;
    int k = pre, kk = k0;
    if (p.order == NRH_FIELD_ORDER_SSE) {
        float li[4] = { 0.f, 0.f, 0.f, 0.f };
        for (; k < pst - 3; k += 4, kk += 4)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float v = line[(size_t)(k + 3 - j) * p.stride];
                bad |= !(v == v);
                li[j] = p.kern[kk + 3 - j] * v + li[j];
            }
        is = (double)((li[0] + li[1]) + (li[2] + li[3]));
    }
    for (; k < pst; ++k, ++kk) {
        const float v = line[(size_t)k * p.stride];
        bad |= !(v == v);
        is += (double)(p.kern[kk] * v);
    }
    float ds = p.dens[u];
    if (bad) {
        double s = 0;
        is = 0;
        k = pre;
        kk = k0;
        if (p.order == NRH_FIELD_ORDER_SSE) {
            float li[4] = { 0.f, 0.f, 0.f, 0.f }, ld[4] = { 0.f, 0.f, 0.f, 0.f };
            for (; k < pst - 3; k += 4, kk += 4)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float v = line[(size_t)(k + 3 - j) * p.stride], kv = p.kern[kk + 3 - j];
                    li[j] = kv * (v == v ? v : 0.f) + li[j];
                    ld[j] = kv * (v == v ? 1.f : 0.f) + ld[j];
                }
            is = (double)((li[0] + li[1]) + (li[2] + li[3]));
            s = (double)((ld[0] + ld[1]) + (ld[2] + ld[3]));
        }
        for (; k < pst; ++k, ++kk) {
            const float v = line[(size_t)k * p.stride], kv = p.kern[kk];
            is += (double)(kv * (v == v ? v : 0.f));
            s += (double)(kv * (v == v ? 1.f : 0.f));
        }
        ds = (float)s;
    }
    *out = (float)is / ds;
}

// k_voxel_to_node on the compact result: mapX / mapY / mapZ give a voxel's place in the lists.
__global__ void __launch_bounds__(kB)
k_listed_to_node(const float *__restrict__ c, int ux, int uy, int uz, const int *__restrict__ mapX,
                 const int *__restrict__ mapY, const int *__restrict__ mapZ, int nx, int ny, int nz, int gnx, int gny,
                 int gnz, Affine T, Affine reorient, float weight, float *__restrict__ ng) {
#pragma clang fp contract(off)
    const size_t G = (size_t)gnx * gny * gnz, plane = (size_t)ux * uy * uz;
    const size_t n = (size_t)blockIdx.x * kB + threadIdx.x;
    if (n >= G) return;
    int x, y, z;
    index_xyz(n, gnx, gny, x, y, z);
    const float3 vc = affine_apply_d(T, (float)x, (float)y, (float)z);
    const int pre[3] = { floor_int(vc.x), floor_int(vc.y), floor_int(vc.z) };
    float bx[2], by[2], bz[2];
    bx[1] = vc.x - (float)pre[0]; bx[0] = 1.f - bx[1];
    by[1] = vc.y - (float)pre[1]; by[0] = 1.f - by[1];
    bz[1] = vc.z - (float)pre[2]; bz[0] = 1.f - bz[1];
    float iv0 = 0.f, iv1 = 0.f, iv2 = 0.f;
    for (int k = 0; k < 2; ++k) {
        const int Z = pre[2] + k;
        if (Z < 0 || Z >= nz) continue;
        for (int b = 0; b < 2; ++b) {
            const int Y = pre[1] + b;
            if (Y < 0 || Y >= ny) continue;
            for (int a = 0; a < 2; ++a) {
                const int X = pre[0] + a;
                if (X < 0 || X >= nx) continue;
                const size_t idx = ((size_t)mapZ[Z] * uy + mapY[Y]) * ux + mapX[X];
                float w = bx[a] * by[b];
                w *= bz[k];
                iv0 += w * c[idx];
                iv1 += w * c[idx + plane];
                iv2 += w * c[idx + 2 * plane];
            }
        }
    }
    const float *R = reorient.m;
    const float r0 = R[0] * iv0 + R[4] * iv1 + R[8] * iv2;
    const float r1 = R[1] * iv0 + R[5] * iv1 + R[9] * iv2;
    const float r2 = R[2] * iv0 + R[6] * iv1 + R[10] * iv2;
    ng[n] = r0 * weight;
    ng[n + G] = r1 * weight;
    ng[n + 2 * G] = r2 * weight;
}

// The density at position l of a line of L voxels without NaN, in the order of k_conv_axis.
float line_density(const std::vector<float>& kern, int radius, int l, int L, int order) {
#pragma clang fp contract(off)
    const int pre = std::max(l - radius, 0), pst = std::min(l + radius + 1, L);
    int k = pre, kk = std::max(radius - l, 0);
    double s = 0;
    if (order == NRH_FIELD_ORDER_SSE) {
        float ld[4] = { 0.f, 0.f, 0.f, 0.f };
        for (; k < pst - 3; k += 4, kk += 4)
            for (int j = 0; j < 4; ++j) ld[j] = kern[kk + 3 - j] + ld[j];
        s = (double)((ld[0] + ld[1]) + (ld[2] + ld[3]));
    }
    for (; k < pst; ++k, ++kk) s += (double)kern[kk];
    return (float)s;
}

// The positions that the nodes of the grid read, per axis, as T (grid voxel -> image voxel) places
// them; the off-diagonal entries of T are rounding on a grid laid along the image, and are covered
// by taking each column's range over the grid with a margin above the float rounding of T's result.
void build(nrh_f3d *h, const Affine& T) {
    NodeConv& c = h->nodeConv;
    c.T = T;
    c.order = h->params.field_order;
    c.built = true;
    c.ok = false;
    const int dims[3] = { h->ref.nx, h->ref.ny, h->ref.nz }, gd[3] = { h->cpp.nx, h->cpp.ny, h->cpp.nz };
    const float pix[3] = { h->ref.dx, h->ref.dy, h->ref.dz }, sp[3] = { h->cpp.dx, h->cpp.dy, h->cpp.dz };
    std::vector<int> list[3], map[3];
    double share[3];
    for (int a = 0; a < 3; ++a) {
        std::vector<char> used(dims[a], 0);
        for (int q = 0; q < gd[a]; ++q) {
            double lo = T.m[a * 4 + 3], hi = lo, size = std::fabs(lo);
            for (int b = 0; b < 3; ++b) {
                const double m = T.m[a * 4 + b], far = m * (b == a ? q : gd[b] - 1), near = b == a ? far : 0.0;
                lo += std::min(near, far);
                hi += std::max(near, far);
                size += std::fabs(far);
            }
            const double margin = 1e-6 * (size + 1.0);
            if (!(std::fabs(lo) < 1e8 && std::fabs(hi) < 1e8)) return;
            const int first = std::max((int)std::floor(lo - margin), 0);
            const int last = std::min((int)std::floor(hi + margin) + 1, dims[a] - 1);
            for (int v = first; v <= last; ++v) used[v] = 1;
        }
        map[a].assign(dims[a], -1);
        for (int v = 0; v < dims[a]; ++v)
            if (used[v]) {
                map[a][v] = (int)list[a].size();
                list[a].push_back(v);
            }
        if (list[a].empty()) return;
        share[a] = (double)list[a].size() / dims[a];
    }
    // Worth it, and no more scratch than the full convolution's 13 bytes a voxel, while the first two
    // compact arrays (12 bytes an entry; the third reuses the first) stay below that: grids of about
    // 3.1 voxels and more.  Finer ones take the full convolution.
    if (12.0 * (share[0] + share[0] * share[1]) > 13.0) return;
    for (int a = 0; a < 3; ++a) {
        c.n[a] = (int)list[a].size();
        // the cubic B-spline kernel as op_convolve_voxel_gradient forms it
        std::vector<float> kern;
        c.radius[a] = convolution_kernel(sp[a], pix[a], kern);
        std::vector<float> dens(list[a].size());
        for (size_t u = 0; u < dens.size(); ++u) dens[u] = line_density(kern, c.radius[a], list[a][u], dims[a], c.order);
        c.list[a].alloc(list[a].size());
        c.map[a].alloc(map[a].size());
        c.kern[a].alloc(kern.size());
        c.dens[a].alloc(dens.size());
        NRH_HIP(hipMemcpyAsync(c.list[a].p, list[a].data(), c.list[a].bytes(), hipMemcpyHostToDevice, h->stream));
        NRH_HIP(hipMemcpyAsync(c.map[a].p, map[a].data(), c.map[a].bytes(), hipMemcpyHostToDevice, h->stream));
        NRH_HIP(hipMemcpyAsync(c.kern[a].p, kern.data(), c.kern[a].bytes(), hipMemcpyHostToDevice, h->stream));
        NRH_HIP(hipMemcpyAsync(c.dens[a].p, dens.data(), c.dens[a].bytes(), hipMemcpyHostToDevice, h->stream));
        NRH_HIP(hipStreamSynchronize(h->stream));  // the host vectors end here
    }
    c.a.alloc(3 * std::max((size_t)c.n[0] * dims[1] * dims[2], (size_t)c.n[0] * c.n[1] * c.n[2]));
    c.b.alloc(3 * (size_t)c.n[0] * c.n[1] * dims[2]);
    c.ok = true;
}

}  // namespace

void op_voxel_gradient_to_nodes(nrh_f3d *h, float weight) {
    NRH_REQUIRE(!h->voxelGrad.empty(), NRH_ERR_STATE, "no voxel-based gradient to convolve");
    Affine T, R;
    node_transforms(h, T, R);
    NodeConv& c = h->nodeConv;
    if (!c.built || c.order != h->params.field_order || std::memcmp(&c.T, &T, sizeof T) != 0) {
        c.built = false;
        build(h, T);
    }
    if (!c.ok) {
        op_convolve_voxel_gradient(h);
        op_voxel_to_node(h, weight);
        return;
    }
    int n[3] = { h->ref.nx, h->ref.ny, h->ref.nz };
    const float *in = h->voxelGrad.p;
    for (int axis = 0; axis < 3; ++axis) {
        PassArgs p;
        p.in = in;
        p.out = axis == 1 ? c.b.p : c.a.p;
        p.L = n[axis];
        p.inPlane = (size_t)n[0] * n[1] * n[2];
        p.rowStride = (size_t)n[0];
        p.sliceStride = (size_t)n[0] * n[1];
        p.stride = axis == 0 ? 1 : axis == 1 ? p.rowStride : p.sliceStride;
        n[axis] = c.n[axis];
        p.ox = n[0];
        p.oy = n[1];
        p.oz = n[2];
        p.outPlane = (size_t)n[0] * n[1] * n[2];
        p.axis = axis;
        p.list = c.list[axis].p;
        p.dens = c.dens[axis].p;
        p.kern = c.kern[axis].p;
        p.radius = c.radius[axis];
        p.order = c.order;
        hipLaunchKernelGGL(k_conv_listed, dim3((unsigned)((p.outPlane + kB - 1) / kB), 3), dim3(kB), 0, h->stream, p);
        in = p.out;
    }
    hipLaunchKernelGGL(k_listed_to_node, dim3((unsigned)((h->G + kB - 1) / kB)), dim3(kB), 0, h->stream, in, n[0], n[1],
                       n[2], c.map[0].p, c.map[1].p, c.map[2].p, h->ref.nx, h->ref.ny, h->ref.nz, h->cpp.nx, h->cpp.ny,
                       h->cpp.nz, T, R, node_weight_ratio(h, weight), h->nodeGrad.p);
    NRH_HIP(hipGetLastError());
    h->voxelGradPending = true;
}

void settle_voxel_gradient(nrh_f3d *h) {
    if (!h->voxelGradPending) return;
    h->voxelGradPending = false;
    op_convolve_voxel_gradient(h);
}

}  // namespace nrh

// Per-operation F3D kernels: one launch per reference Compute / reg_nmi virtual.
//
// These kernels keep the reference's rounding (float/double split, summation order, no fused
// multiply-adds) so that each stage can be compared element by element with the CPU path.
// The hot loop of a registration uses the fused kernels of f3d_fused.hip instead.

#include "device.hpp"
#include "be_blocks.hpp"
#include "m33.hpp"
#include "m44.hpp"
#include "host.hpp"
#include "f3d_handle.hpp"
#include "f3d_batch.hpp"
#include <cmath>

namespace nrh {

namespace {

constexpr int kBlock = 256;

inline unsigned blocks_for(size_t n, int block = kBlock) {
    size_t b = (n + block - 1) / block;
    return (unsigned)(b > 0 ? b : 1);
}

// ------------------------------------------------------------------ deformation field
// reg_cubic_spline_getDeformationField3D, non-composition (reg-lib/cpu/_reg_localTrans.cpp:1080-1453)
__global__ void __launch_bounds__(kBlock)
k_spline_field(int nx, int ny, int nz, int gnx, int gny, size_t G, const float *__restrict__ cpp,
               const int *__restrict__ mask, float gx, float gy, float gz, int lut, int order,
               float *__restrict__ field, size_t N) {
#pragma clang fp contract(off)
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= N) return;
    const int x = (int)(idx % nx);
    const int y = (int)((idx / nx) % ny);
    const int z = (int)(idx / ((size_t)nx * ny));
    if (mask && mask[idx] < 0) {
        if (!lut) { field[idx] = 0.f; field[idx + N] = 0.f; field[idx + 2 * N] = 0.f; }
        return;
    }
    int px, py, pz;
    float tx, ty, tz, xb[4], yb[4], zb[4];
    cell_of(x, gx, lut, px, tx);
    cell_of(y, gy, lut, py, ty);
    cell_of(z, gz, lut, pz, tz);
    bspline_basis(tx, xb);
    bspline_basis(ty, yb);
    bspline_basis(tz, zb);
    const float3 r = ref_spline_point(cpp, G, gnx, gny, px, py, pz, xb, yb, zb, order, lut != 0);
    field[idx] = r.x;
    field[idx + N] = r.y;
    field[idx + 2 * N] = r.z;
}

// ------------------------------------------------------------------ resampling
// ResampleImage3D, linear kernel (reg-lib/cpu/_reg_resampling.cpp:316-464)
__global__ void __launch_bounds__(kBlock)
k_resample_linear(const float *__restrict__ field, size_t N, const int *__restrict__ mask,
                  const float *__restrict__ flo, int fnx, int fny, int fnz, Affine ijk, float pad,
                  float *__restrict__ warped) {
#pragma clang fp contract(off)
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= N) return;
    if (mask && mask[idx] < 0) return;
    const float3 p = affine_apply_d(ijk, field[idx], field[idx + N], field[idx + 2 * N]);
    warped[idx] = sample_linear(flo, fnx, fny, fnz, p, pad);
}

// TrilinearImageGradient (reg-lib/cpu/_reg_resampling.cpp:1797-1915)
__global__ void __launch_bounds__(kBlock)
k_image_gradient_linear(const float *__restrict__ field, size_t N, const int *__restrict__ mask,
                        const float *__restrict__ flo, int fnx, int fny, int fnz, Affine ijk, float pad,
                        float *__restrict__ grad) {
#pragma clang fp contract(off)
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= N) return;
    float3 g = make_float3(0.f, 0.f, 0.f);
    if (!mask || mask[idx] > -1)
        g = image_gradient_at(flo, fnx, fny, fnz, affine_apply_d(ijk, field[idx], field[idx + N], field[idx + 2 * N]),
                              pad);
    const float g0 = g.x, g1 = g.y, g2 = g.z;
    grad[idx] = g0;
    grad[idx + N] = g1;
    grad[idx + 2 * N] = g2;
}

// ------------------------------------------------------------------ joint histogram
// Approximate-Parzen count fill of reg_getNmiValue (reg-lib/cpu/_reg_nmi.cpp:211-248):
// integer counts, privatised per workgroup in LDS, merged with integer atomics (exact in
// any order).
__global__ void __launch_bounds__(kBlock)
k_joint_histogram(const float *__restrict__ ref, const float *__restrict__ war, const int *__restrict__ mask,
                  size_t N, int rb, int fb, uint32_t *__restrict__ counts) {
    extern __shared__ uint32_t lh[];
    const int nb = rb * fb;
    for (int i = threadIdx.x; i < nb; i += blockDim.x) lh[i] = 0;
    __syncthreads();
    for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < N; idx += (size_t)gridDim.x * blockDim.x) {
        if (mask && mask[idx] < 0) continue;
        const float r = ref[idx], w = war[idx];
        if (r == r && w == w && 0.f <= r && r < (float)rb && 0.f <= w && w < (float)fb)
            atomicAdd(&lh[(int)r + (int)w * rb], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nb; i += blockDim.x)
        if (lh[i]) atomicAdd(&counts[i], lh[i]);
}

// Smoothing, normalisation, marginals and entropies of reg_getNmiValue (reg-lib/cpu/_reg_nmi.cpp:249-344)
// in FP64, one workgroup.  ent: H_r, H_f, H_rf, total, nmi.
__global__ void __launch_bounds__(1024)
k_nmi_finalize(uint32_t *__restrict__ counts, int rb, int fb, double *__restrict__ pro,
               double *__restrict__ logh, float *__restrict__ logf, double *__restrict__ ent) {
    __shared__ double red[16];
    const int nb = rb * fb, total = nb + rb + fb;
    const double k0 = 1.0 / 6.0, k1 = (double)(2.f / 3.f);  // GetBasisSplineValue(-1), (0)
    // the counts are consumed: zeroed as they are read, ready for the next histogram
    for (int i = threadIdx.x; i < total; i += blockDim.x) {
        pro[i] = i < nb ? (double)counts[i] : 0.0;
        if (i < nb) counts[i] = 0u;
    }
    __syncthreads();
    // along the reference axis into logh
    for (int i = threadIdx.x; i < nb; i += blockDim.x) {
        const int r = i % rb, f = i / rb;
        double v = 0;
        if (r - 1 > -1) v += pro[i - 1] * k0;
        v += pro[i] * k1;
        if (r + 1 < rb) v += pro[i + 1] * k0;
        logh[r + rb * f] = v;
    }
    __syncthreads();
    // along the floating axis back into pro
    for (int i = threadIdx.x; i < nb; i += blockDim.x) {
        const int f = i / rb;
        double v = 0;
        if (f - 1 > -1) v += logh[i - rb] * k0;
        v += logh[i] * k1;
        if (f + 1 < fb) v += logh[i + rb] * k0;
        pro[i] = v;
    }
    __syncthreads();
    double s = 0;
    for (int i = threadIdx.x; i < total; i += blockDim.x) s += pro[i];
    s = block_sum_double(s, red);
    __shared__ double totalS;
    if (threadIdx.x == 0) totalS = s;
    __syncthreads();
    const double act = totalS;
    for (int i = threadIdx.x; i < total; i += blockDim.x) pro[i] /= act;
    __syncthreads();
    for (int i = threadIdx.x; i < rb + fb; i += blockDim.x) {
        double m = 0;
        if (i < rb) {
            for (int f = 0; f < fb; ++f) m += pro[i + rb * f];
        } else {
            const int f = i - rb;
            for (int r = 0; r < rb; ++r) m += pro[rb * f + r];
        }
        pro[nb + i] = m;
    }
    __syncthreads();
    double hr = 0, hf = 0, hj = 0;
    for (int i = threadIdx.x; i < total; i += blockDim.x) {
        const double p = pro[i];
        double l = 0;
        if (p > 0) {
            l = log(p);
            if (i < nb) hj -= p * l;
            else if (i < nb + rb) hr -= p * l;
            else hf -= p * l;
        }
        logh[i] = l;
        logf[i] = (float)l;
    }
    hr = block_sum_double(hr, red);
    __syncthreads();
    hf = block_sum_double(hf, red);
    __syncthreads();
    hj = block_sum_double(hj, red);
    if (threadIdx.x == 0) {
        ent[0] = hr;
        ent[1] = hf;
        ent[2] = hj;
        ent[3] = act;
        ent[4] = (hr + hf) / hj;
    }
}

// K[i] = log p_r + log p_w - NMI log p_rw for joint bin i = r + w rb, rounded once to float.
__device__ __forceinline__ float nmi_table_value(double lr, double lw, double nmi, double l) {
#pragma clang fp contract(off)
    return (float)((lr + lw) - nmi * l);
}

// The same finalisation with the working array in LDS (histograms of up to kFinLds entries):
// identical arithmetic and thread partition, no global-memory round trips between phases.
constexpr int kFinLds = 7936;
constexpr int kFinPer = (kFinLds + 1023) / 1024;

// Phase 1: v[q] = the smoothed joint histogram, normalised by its total, at entries
// tid + 1024 q (also in P, LDS), r[q] and f[q] their bins; then its marginals in P.  The counts are
// zeroed as they are read, ready for the next histogram.
__device__ __forceinline__ void fin_probabilities(uint32_t *__restrict__ counts, int rb, int fb, double *P, double *red,
                                                  double& totalS, double (&v)[kFinPer], int (&r)[kFinPer],
                                                  int (&f)[kFinPer]) {
    const int nb = rb * fb, tid = threadIdx.x;
    const double k0 = 1.0 / 6.0, k1 = (double)(2.f / 3.f);
    {
        // one division per thread: the bins of the next entry are 1024 entries further
        const int dr = 1024 % rb, df = 1024 / rb;
        r[0] = tid % rb;
        f[0] = tid / rb;
#pragma unroll
        for (int q = 1; q < kFinPer; ++q) {
            const bool wrap = r[q - 1] + dr >= rb;
            r[q] = r[q - 1] + dr - (wrap ? rb : 0);
            f[q] = f[q - 1] + df + (wrap ? 1 : 0);
        }
    }
#pragma unroll
    for (int q = 0; q < kFinPer; ++q) {
        const int i = tid + q * 1024;
        if (i < nb) {
            P[i] = (double)counts[i];
            counts[i] = 0u;
        }
    }
    __syncthreads();
    // along the reference axis
#pragma unroll
    for (int q = 0; q < kFinPer; ++q) {
        const int i = tid + q * 1024;
        v[q] = 0;
        if (i < nb) {
            double t = 0;
            if (r[q] - 1 > -1) t += P[i - 1] * k0;
            t += P[i] * k1;
            if (r[q] + 1 < rb) t += P[i + 1] * k0;
            v[q] = t;
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kFinPer; ++q) {
        const int i = tid + q * 1024;
        if (i < nb) P[i] = v[q];
    }
    __syncthreads();
    // along the floating axis, and the total
    double s = 0;
#pragma unroll
    for (int q = 0; q < kFinPer; ++q) {
        const int i = tid + q * 1024;
        v[q] = 0;
        if (i < nb) {
            double t = 0;
            if (f[q] - 1 > -1) t += P[i - rb] * k0;
            t += P[i] * k1;
            if (f[q] + 1 < fb) t += P[i + rb] * k0;
            v[q] = t;
            s += t;
        }
    }
    s = block_sum_double(s, red);  // its barriers also end the reads of P
    if (tid == 0) totalS = s;
    __syncthreads();
    const double act = totalS;
#pragma unroll
    for (int q = 0; q < kFinPer; ++q) {
        const int i = tid + q * 1024;
        if (i < nb) {
            v[q] /= act;
            P[i] = v[q];
        }
    }
    __syncthreads();
    for (int i = tid; i < rb + fb; i += 1024) {
        double m = 0;
        const double *p = i < rb ? P + i : P + rb * (i - rb);
        const int n = i < rb ? fb : rb, stride = i < rb ? rb : 1;
        int k = 0;
        for (; k + 8 <= n; k += 8) {
            double w[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) w[u] = p[(k + u) * stride];
#pragma unroll
            for (int u = 0; u < 8; ++u) m += w[u];
        }
        for (; k < n; ++k) m += p[k * stride];
        P[nb + i] = m;
    }
}

// Phase 2: the logarithms (written with the probabilities), the entropies (each thread's strided
// terms, then block sums: H_r, H_f, H_rf), ent[] and the table K.
__device__ __forceinline__ void fin_entropies(int rb, int fb, double *P, double *red /* 48 */, double& totalS,
                                              const double (&v)[kFinPer], const int (&r)[kFinPer],
                                              const int (&f)[kFinPer], double *__restrict__ pro,
                                              double *__restrict__ logh, float *__restrict__ logf,
                                              double *__restrict__ ent, float *__restrict__ kTab) {
    const int nb = rb * fb, total = nb + rb + fb, tid = threadIdx.x;
    const double act = totalS;
    double hr = 0, hf = 0, hj = 0, l[kFinPer];
    // the joint entries need no marginal: no barrier keeps them waiting for the threads that sum those
#pragma unroll
    for (int q = 0; q < kFinPer; ++q) {
        const int i = tid + q * 1024;
        l[q] = 0;
        if (i < nb) {
            if (v[q] > 0) {
                l[q] = log(v[q]);
                hj -= v[q] * l[q];
            }
            pro[i] = v[q];
            logh[i] = l[q];
            logf[i] = (float)l[q];
        }
    }
    __syncthreads();
    for (int i = nb + (tid - nb % 1024 + 1024) % 1024; i < total; i += 1024) {
        const double p = P[i];
        double lm = 0;
        if (p > 0) {
            lm = log(p);
            if (i < nb + rb) hr -= p * lm;
            else hf -= p * lm;
        }
        pro[i] = p;
        logh[i] = lm;
        logf[i] = (float)lm;
        P[i] = lm;  // for the table K
    }
    block_sum_double3(hr, hf, hj, red);
    if (tid == 0) {
        ent[0] = hr;
        ent[1] = hf;
        ent[2] = hj;
        ent[3] = act;
        ent[4] = (hr + hf) / hj;
        totalS = (hr + hf) / hj;  // the NMI, for K
    }
    if (kTab) {
        // the fused gradient sweep's table K[r + w rb] = log p_r + log p_w - NMI log p_rw (as
        // k_nmi_table computes it, from the same FP64 logs)
        __syncthreads();
        const double nmi = totalS;
#pragma unroll
        for (int q = 0; q < kFinPer; ++q) {
            const int i = tid + q * 1024;
            if (i < nb) kTab[i] = nmi_table_value(P[nb + r[q]], P[nb + rb + f[q]], nmi, l[q]);
        }
    }
}

// The whole finalisation in one workgroup of 1024 threads.  One workgroup does it all because every
// step needs the one before it whole; what it takes is the instructions of its 16 waves, so each
// entry is loaded, smoothed and logged by one thread that keeps it in registers.  64 x 64 bins:
// 20 us with every entry's bins found by division in each of five passes over LDS, 15 us so.
__device__ __forceinline__ void
nmi_finalize_lds_block(uint32_t *__restrict__ counts, int rb, int fb, double *__restrict__ pro,
                   double *__restrict__ logh, float *__restrict__ logf, double *__restrict__ ent,
                   float *__restrict__ kTab = nullptr) {
    __shared__ double P[kFinLds];
    __shared__ double red[48];
    __shared__ double totalS;
    double v[kFinPer];
    int r[kFinPer], f[kFinPer];
    fin_probabilities(counts, rb, fb, P, red, totalS, v, r, f);
    fin_entropies(rb, fb, P, red, totalS, v, r, f, pro, logh, logf, ent, kTab);
}

// reg_getVoxelBasedNmiGradient3d<float> (reg-lib/cpu/_reg_nmi.cpp:501-593); grad +=
__global__ void __launch_bounds__(kBlock)
k_nmi_voxel_gradient(const float *__restrict__ ref, const float *__restrict__ war, const float *__restrict__ wg,
                     const int *__restrict__ mask, size_t N, int rb, int fb, const double *__restrict__ logh,
                     const double *__restrict__ ent, double weight, float *__restrict__ grad) {
#pragma clang fp contract(off)
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    if (mask && mask[i] < 0) return;
    const float rv = ref[i], wv = war[i];
    if (!(rv == rv && wv == wv)) return;
    const float g[3] = { wg[i], wg[i + N], wg[i + 2 * N] };
    float d[3];
    nmi_voxel_term(rv, wv, g, logh, ent, rb, fb, weight, d);
    for (int k = 0; k < 3; ++k) grad[i + k * N] += d[k];
}

// The same voxel term with the log histogram staged in LDS once per workgroup (its 16 joint and 8
// marginal look-ups per voxel then hit LDS): a persistent grid over the voxels, identical
// arithmetic.  logLds: rb * fb + rb + fb doubles of dynamic LDS.
__global__ void __launch_bounds__(kBlock)
k_nmi_voxel_gradient_lds(const float *__restrict__ ref, const float *__restrict__ war, const float *__restrict__ wg,
                         const int *__restrict__ mask, size_t N, int rb, int fb, const double *__restrict__ logh,
                         const double *__restrict__ ent, double weight, float *__restrict__ grad) {
#pragma clang fp contract(off)
    extern __shared__ double logLds[];
    const int total = rb * fb + rb + fb;
    for (int i = threadIdx.x; i < total; i += blockDim.x) logLds[i] = logh[i];
    __syncthreads();
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (size_t)gridDim.x * blockDim.x) {
        if (mask && mask[i] < 0) continue;
        const float rv = ref[i], wv = war[i];
        if (!(rv == rv && wv == wv)) continue;
        const float g[3] = { wg[i], wg[i + N], wg[i + 2 * N] };
        float d[3];
        nmi_voxel_term(rv, wv, g, logLds, ent, rb, fb, weight, d);
        for (int k = 0; k < 3; ++k) grad[i + k * N] += d[k];
    }
}

// The voxel gradient of an evaluation, written rather than added to zeros.  The sums over the 4 x 4
// bins factor: sum_r sum_w B_r B'_w g (log p_r + log p_w - NMI log p_rw) = g sum_w B'_w sum_r B_r K[r, w],
// with K in FP64 from the FP64 logs, in LDS; where the operation of its own keeps the reference's
// three sums of 16 terms per component (350 FP64 operations a voxel, and the Parzen windows by their
// general form), this takes 60.  Voxels whose bins are not four inside the histogram take the
// operation's form.  256 x 256 x 160, both directions' launches overlapping: 240 us a launch and a
// zero fill of 20 before, 83 so; 336 MB at 5.2 TB/s are 64.
__global__ void __launch_bounds__(kBlock)
k_nmi_voxel_gradient_eval(const float *__restrict__ ref, const float *__restrict__ war, const float *__restrict__ wg,
                          const int *__restrict__ mask, size_t N, int rb, int fb, const double *__restrict__ logh,
                          const double *__restrict__ ent, float *__restrict__ grad) {
    extern __shared__ double sK[];
    const int nb = rb * fb;
    const double nmi = (ent[0] + ent[1]) / ent[2], coef = 1.0 / (ent[2] * ent[3]);
    for (int i = threadIdx.x; i < nb; i += kBlock) {
        const int w = i / rb, r = i - w * rb;
        sK[i] = (logh[nb + r] + logh[nb + rb + w]) - nmi * logh[i];
    }
    __syncthreads();
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < N; i += (size_t)gridDim.x * kBlock) {
        const float rv = ref[i], wv = war[i], g[3] = { wg[i], wg[i + N], wg[i + 2 * N] };
        float d[3] = { 0.f, 0.f, 0.f };
        if (rv == rv && wv == wv && !(mask && mask[i] < 0)) {
            const int r0 = (int)(rv - 1.f), w0 = (int)(wv - 1.f);
            if (rv >= 1.f && wv >= 1.f && (int)(rv + 3.f) == r0 + 4 && (int)(wv + 3.f) == w0 + 4 && r0 + 3 < rb &&
                w0 + 3 < fb) {
                const double t = (double)(rv - (float)(r0 + 1)), u = 1.0 - t, h = (double)(wv - (float)(w0 + 1)), v = 1.0 - h;
                // GetBasisSplineValue at 1 + t, t, 1 - t and 2 - t, whose pieces use 2 / 3 rounded to float
                const double c = (double)(2.f / 3.f), sixth = 1.0 / 6.0;
                const double B[4] = { u * u * u * sixth, c + (0.5 * t - 1.0) * t * t,
                                      t == 0.0 ? sixth : c + (0.5 * u - 1.0) * u * u, t * t * t * sixth };
                // GetBasisSplineDerivativeValue at 1 + h, h, h - 1 and h - 2
                const double D[4] = { -0.5 * v * v, (1.5 * h - 2.0) * h, -(1.5 * v - 2.0) * v, 0.5 * h * h };
                const double *K = sK + r0 + w0 * rb;
                double S = 0.0;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    S += D[k] * (B[0] * K[k * rb] + B[1] * K[k * rb + 1] + B[2] * K[k * rb + 2] + B[3] * K[k * rb + 3]);
                S *= coef;
#pragma unroll
                for (int k = 0; k < 3; ++k) d[k] = g[k] == g[k] ? (float)(S * (double)g[k]) : 0.f;
            } else {
                nmi_voxel_term(rv, wv, g, logh, ent, rb, fb, 1.0, d);
            }
        }
        grad[i] = d[0];
        grad[i + N] = d[1];
        grad[i + 2 * N] = d[2];
    }
}

// ------------------------------------------------------------------ convolution
// Density preparation of reg_tools_kernelConvolution (reg-lib/cpu/_reg_tools.cpp:860-866).
__global__ void __launch_bounds__(kBlock)
k_conv_prepare(float *__restrict__ data, const int *__restrict__ mask, size_t N, float *__restrict__ dens,
               uint8_t *__restrict__ isnan_) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const float v = data[i];
    const float d = ((!mask || mask[i] >= 0) && v == v) ? 1.f : 0.f;
    dens[i] = d;
    isnan_[i] = d == 0.f;
    if (d == 0.f) data[i] = 0.f;
}

// One axis of the density-normalised line convolution (reg-lib/cpu/_reg_tools.cpp:977-1093,
// scalar path: kernel-weighted sums in double over the in-range taps).
__global__ void __launch_bounds__(kBlock)
k_conv_axis(const float *__restrict__ data, const float *__restrict__ dens, int nx, int ny, int nz, int axis,
            const float *__restrict__ kernel, int radius, float *__restrict__ outData, float *__restrict__ outDens,
            int order) {
#pragma clang fp contract(off)
    const size_t N = (size_t)nx * ny * nz;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    int x, y, z;
    index_xyz(i, nx, ny, x, y, z);
    const int L = axis == 0 ? nx : axis == 1 ? ny : nz;
    const int l = axis == 0 ? x : axis == 1 ? y : z;
    const size_t stride = axis == 0 ? 1 : axis == 1 ? (size_t)nx : (size_t)nx * ny;
    const size_t base = i - (size_t)l * stride;
    int pre = l - radius, pst = l + radius + 1;
    int k0 = 0;
    if (pre < 0) { k0 = -pre; pre = 0; }
    if (pst > L) pst = L;
    double is = 0, ds = 0;
    int k = pre, kk = k0;
    if (order == NRH_FIELD_ORDER_SSE) {
        // the SSE build (reg-lib/cpu/_reg_tools.cpp:1018-1049): blocks of four taps summed in four
        // float lanes (lane j takes the block's tap 3 - j), the lanes reduced as SSE3's two
        // horizontal adds do, (l0 + l1) + (l2 + l3); the last < 4 taps added in double
        float li[4] = { 0.f, 0.f, 0.f, 0.f }, ld[4] = { 0.f, 0.f, 0.f, 0.f };
        for (; k < pst - 3; k += 4, kk += 4)
            for (int j = 0; j < 4; ++j) {
                const float kv = kernel[kk + 3 - j];
                const size_t o = base + (size_t)(k + 3 - j) * stride;
                li[j] = kv * data[o] + li[j];
                ld[j] = kv * dens[o] + ld[j];
            }
        is = (double)((li[0] + li[1]) + (li[2] + li[3]));
        ds = (double)((ld[0] + ld[1]) + (ld[2] + ld[3]));
    }
    for (; k < pst; ++k, ++kk) {
        const float kv = kernel[kk];
        is += (double)(kv * data[base + (size_t)k * stride]);
        ds += (double)(kv * dens[base + (size_t)k * stride]);
    }
    outData[i] = (float)is;
    outDens[i] = (float)ds;
}

__global__ void __launch_bounds__(kBlock)
k_conv_normalise(float *__restrict__ data, const float *__restrict__ dens, const uint8_t *__restrict__ isnan_, size_t N) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    data[i] = isnan_[i] ? __builtin_nanf("") : data[i] / dens[i];
}

// ------------------------------------------------------------------ voxel -> node
// reg_voxelCentricToNodeCentric, update = false (reg-lib/cpu/_reg_localTrans.cpp:1540-1684)
__global__ void __launch_bounds__(kBlock)
k_voxel_to_node(const float *__restrict__ vg, int nx, int ny, int nz, int gnx, int gny, int gnz, Affine T,
                Affine reorient, float weight, float *__restrict__ ng) {
#pragma clang fp contract(off)
    const size_t G = (size_t)gnx * gny * gnz, N = (size_t)nx * ny * nz;
    const size_t n = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
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
    for (int c = 0; c < 2; ++c) {
        const int Z = pre[2] + c;
        if (Z < 0 || Z >= nz) continue;
        for (int b = 0; b < 2; ++b) {
            const int Y = pre[1] + b;
            if (Y < 0 || Y >= ny) continue;
            for (int a = 0; a < 2; ++a) {
                const int X = pre[0] + a;
                if (X < 0 || X >= nx) continue;
                const size_t idx = ((size_t)Z * ny + Y) * nx + X;
                float w = bx[a] * by[b];
                w *= bz[c];
                iv0 += w * vg[idx];
                iv1 += w * vg[idx + N];
                iv2 += w * vg[idx + 2 * N];
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

// ------------------------------------------------------------------ bending energy
// (the basis, the brick grid and the bodies over bricks are in be_blocks.hpp)

// The end of the bending-energy gradient at node n: grad += ratio * (the gathered sums), and the
// in-place reg_getDisplacementFromDeformation / reg_getDeformationFromDisplacement pair the
// reference wraps around it (regul.cpp:312, 450): p <- (p - node) + node.  Returns the float bits
// of the final gradient's length (0 past the grid).
__device__ __forceinline__ uint32_t
be_apply_at(float *__restrict__ cpp, int gnx, int gny, int gnz, const Affine& xyz, const float *__restrict__ beGrad,
            float ratio, float *__restrict__ grad, size_t n) {
#pragma clang fp contract(off)
    const size_t G = (size_t)gnx * gny * gnz;
    if (n >= G) return 0u;
    int x, y, z;
    index_xyz(n, gnx, gny, x, y, z);
    float g[3];
    for (int k = 0; k < 3; ++k) {
        g[k] = grad[n + k * G] + ratio * beGrad[n + k * G];
        grad[n + k * G] = g[k];
        const float node = node_pos(xyz, k, x, y, z);
        cpp[n + k * G] = (cpp[n + k * G] - node) + node;
    }
    return __float_as_uint(sqrtf(g[0] * g[0] + g[1] * g[1] + g[2] * g[2]));
}

// ------------------------------------------------------------------ linear energy
struct LeBasis {
    float b[3][27];  // first-order tensor products along x, y, z
};

// Rotation-free displacement Jacobian at an interior node (reg-lib/cpu/_reg_localTrans_regul.cpp:596-634).
// B: the first-order basis in LDS (broadcast reads; as a kernel argument its 81 values would not
// fit the scalar registers).
__device__ M33 le_matrix(const float *__restrict__ cpp, size_t G, int gnx, int gny, int x, int y, int z,
                         const float (*B)[27], const M33& reo) {
#pragma clang fp contract(off)
    M33 M = {};
    int i = 0;
#pragma unroll
    for (int c = -1; c < 2; ++c)
#pragma unroll
        for (int b = -1; b < 2; ++b)
#pragma unroll
            for (int a = -1; a < 2; ++a, ++i) {
                const size_t idx = ((size_t)(z + c) * gny + y + b) * gnx + x + a;
                const float cv[3] = { cpp[idx], cpp[idx + G], cpp[idx + 2 * G] };
                const float b0 = B[0][i], b1 = B[1][i], b2 = B[2][i];
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    M.m[0][k] += b0 * cv[k];
                    M.m[1][k] += b1 * cv[k];
                    M.m[2][k] += b2 * cv[k];
                }
            }
    M = m33_mul(reo, M);
    const M33 R = m33_inverse(m33_polar(M));
    M = m33_mul(R, M);
    M.m[0][0] -= 1.f;
    M.m[1][1] -= 1.f;
    M.m[2][2] -= 1.f;
    return M;
}

// Per-node terms of reg_spline_approxLinearEnergyValue3D (:559-647) and the diagonal the gradient
// uses; the last block to finish sums the block partials in block order into *out (/ 3G).
__global__ void __launch_bounds__(kBlock)
k_le_terms(const float *__restrict__ cpp, int gnx, int gny, int gnz, LeBasis B, M33 reo, float *__restrict__ diag,
           double *__restrict__ partials, uint32_t *__restrict__ ticket, double scale, double *__restrict__ out) {
#pragma clang fp contract(off)
    __shared__ double red[16];
    __shared__ bool last;
    __shared__ float sB[3][27];
    if (threadIdx.x < 81) sB[threadIdx.x / 27][threadIdx.x % 27] = B.b[threadIdx.x / 27][threadIdx.x % 27];
    __syncthreads();
    const size_t G = (size_t)gnx * gny * gnz;
    const size_t n = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    double s = 0;
    if (n < G) {
        int x, y, z;
    index_xyz(n, gnx, gny, x, y, z);
        float d0 = 0.f, d1 = 0.f, d2 = 0.f;
        if (x > 0 && y > 0 && z > 0 && x < gnx - 1 && y < gny - 1 && z < gnz - 1) {
            const M33 M = le_matrix(cpp, G, gnx, gny, x, y, z, sB, reo);
            for (int b = 0; b < 3; ++b)
                for (int a = 0; a < 3; ++a) {
                    const double v = 0.5 * (double)(M.m[a][b] + M.m[b][a]);
                    s += v * v;
                }
            d0 = M.m[0][0];
            d1 = M.m[1][1];
            d2 = M.m[2][2];
        }
        diag[n] = d0;
        diag[n + G] = d1;
        diag[n + 2 * G] = d2;
    }
    s = block_sum_double(s, red);
    if (threadIdx.x == 0) {
        partials[blockIdx.x] = s;
        __threadfence();
        last = atomicAdd(ticket, 1u) == gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    __threadfence();
    double t = 0;
    for (int i = threadIdx.x; i < (int)gridDim.x; i += blockDim.x) t += partials[i];
    t = block_sum_double(t, red);
    if (threadIdx.x == 0) {
        *out = t * scale;
        *ticket = 0u;
    }
}

// reg_spline_approxLinearEnergyGradient3D (:739-824) as a gather: each node adds the
// contributions of the interior nodes around it in the reference's source order, so every sum
// runs in the same order as the reference's scatter.  Optionally tracks the final max length.
__global__ void __launch_bounds__(kBlock)
k_le_grad(const float *__restrict__ diag, int gnx, int gny, int gnz, LeBasis B, M33 inv, float ratio,
          float *__restrict__ grad, uint32_t *__restrict__ maxBits) {
#pragma clang fp contract(off)
    __shared__ float sB[3][27];
    if (threadIdx.x < 81) sB[threadIdx.x / 27][threadIdx.x % 27] = B.b[threadIdx.x / 27][threadIdx.x % 27];
    __syncthreads();
    const size_t G = (size_t)gnx * gny * gnz;
    const size_t n = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = n < G;
    const size_t m = valid ? n : 0;
    int x, y, z;
    index_xyz(m, gnx, gny, x, y, z);
    float g0 = grad[m], g1 = grad[m + G], g2 = grad[m + 2 * G];
    for (int c = 1; c > -2; --c)
        for (int b = 1; b > -2; --b)
            for (int a = 1; a > -2; --a) {
                const int X = x - a, Y = y - b, Z = z - c;  // the source node
                if (X < 1 || Y < 1 || Z < 1 || X > gnx - 2 || Y > gny - 2 || Z > gnz - 2) continue;
                const size_t s = ((size_t)Z * gny + Y) * gnx + X;
                const int i = 26 - ((c + 1) * 9 + (b + 1) * 3 + (a + 1));
                const float v0 = -2.f * diag[s] * sB[0][i];
                const float v1 = -2.f * diag[s + G] * sB[1][i];
                const float v2 = -2.f * diag[s + 2 * G] * sB[2][i];
                g0 += ratio * (inv.m[0][0] * v0 + inv.m[0][1] * v1 + inv.m[0][2] * v2);
                g1 += ratio * (inv.m[1][0] * v0 + inv.m[1][1] * v1 + inv.m[1][2] * v2);
                g2 += ratio * (inv.m[2][0] * v0 + inv.m[2][1] * v1 + inv.m[2][2] * v2);
            }
    if (valid) {
        grad[n] = g0;
        grad[n + G] = g1;
        grad[n + 2 * G] = g2;
    }
    if (maxBits) block_track_max(maxBits, valid ? __float_as_uint(sqrtf(g0 * g0 + g1 * g1 + g2 * g2)) : 0u);
}

// ------------------------------------------------------------------ optimiser helpers
// reg_getMaximalLength<float> (reg-lib/cpu/_reg_tools.cpp:335-353): lengths are >= 0, so their
// IEEE bit patterns order like unsigned integers.
__global__ void __launch_bounds__(kBlock)
k_max_length(const float *__restrict__ g, size_t G, uint32_t *__restrict__ out) {
#pragma clang fp contract(off)
    uint32_t best = 0;
    for (size_t n = (size_t)blockIdx.x * blockDim.x + threadIdx.x; n < G; n += (size_t)gridDim.x * blockDim.x) {
        const float x = g[n], y = g[n + G], z = g[2 * G + n];
        const float l = sqrtf(x * x + y * y + z * z);
        const uint32_t b = __float_as_uint(l);
        best = b > best ? b : best;
    }
    block_track_max(out, best);
}

__global__ void k_max_to_scalar(const uint32_t *__restrict__ bits, double *__restrict__ out) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *out = (double)__uint_as_float(*bits);
}

// Compute::NormaliseGradient (reg-lib/Compute.cpp:152-183)
__global__ void __launch_bounds__(kBlock)
k_normalise(float *__restrict__ g, size_t n, double inv) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) g[i] = (float)((double)g[i] * inv);
}

// Normalisation by the max length held as float bits; block 0 also publishes it as a double.
__device__ __forceinline__ void
normalise_bits_block(float *__restrict__ g, size_t n, const uint32_t *__restrict__ bits, double *__restrict__ maxLen, int bid) {
    const size_t i = (size_t)bid * blockDim.x + threadIdx.x;
    const double m = (double)__uint_as_float(*bits);
    if (i == 0) *maxLen = m;
    if (i < n && m != 0.0) g[i] = (float)((double)g[i] * (1.0 / m));
}

// Normalisation by a device-resident max length (fused gradient path): skips when it is 0.
__global__ void __launch_bounds__(kBlock)
k_normalise_dev(float *__restrict__ g, size_t n, const double *__restrict__ maxLen) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const double m = *maxLen;
    if (i < n && m != 0.0) g[i] = (float)((double)g[i] * (1.0 / m));
}

// ConjugateGradient<float>::UpdateGradientValues (reg-lib/Optimiser.cpp:231-317)
__device__ __forceinline__ void
cg_init_block(float *__restrict__ grad, float *__restrict__ G_, float *__restrict__ H, size_t n, int bid) {
    const size_t i = (size_t)bid * blockDim.x + threadIdx.x;
    if (i < n) H[i] = G_[i] = -grad[i];
}

__device__ __forceinline__ void
cg_dots_block(const float *__restrict__ grad, const float *__restrict__ G_, const float *__restrict__ H, size_t n,
          double *__restrict__ partials, int bid, int nbk) {
#pragma clang fp contract(off)
    __shared__ double red[16];
    double gg = 0, dgg = 0;
    for (size_t i = (size_t)bid * blockDim.x + threadIdx.x; i < n; i += (size_t)nbk * blockDim.x) {
        gg += (double)(H[i] * G_[i]);
        dgg += (double)((grad[i] + G_[i]) * grad[i]);
    }
    gg = block_sum_double(gg, red);
    __syncthreads();
    dgg = block_sum_double(dgg, red);
    if (threadIdx.x == 0) {
        partials[2 * bid] = gg;
        partials[2 * bid + 1] = dgg;
    }
}

__device__ __forceinline__ void
cg_gamma_block(const double *__restrict__ partials, int nb, double *__restrict__ gam) {
    __shared__ double red[16];
    double gg = 0, dgg = 0;
    for (int i = threadIdx.x; i < nb; i += blockDim.x) {
        gg += partials[2 * i];
        dgg += partials[2 * i + 1];
    }
    gg = block_sum_double(gg, red);
    __syncthreads();
    dgg = block_sum_double(dgg, red);
    if (threadIdx.x == 0) *gam = dgg / gg;
}

__device__ __forceinline__ void
cg_apply_block(float *__restrict__ grad, float *__restrict__ G_, float *__restrict__ H, size_t n, const double *__restrict__ gam, int bid) {
#pragma clang fp contract(off)
    const size_t i = (size_t)bid * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double gm = *gam;
    G_[i] = -grad[i];
    H[i] = (float)((double)G_[i] + gm * (double)H[i]);
    grad[i] = -H[i];
}

// Compute::UpdateControlPointPosition (reg-lib/Compute.cpp:91-127)
__device__ __forceinline__ void
update_dof_block(float *__restrict__ cur, const float *__restrict__ best, const float *__restrict__ grad, float scale, size_t n, int bid) {
#pragma clang fp contract(off)
    const size_t i = (size_t)bid * blockDim.x + threadIdx.x;
    if (i < n) cur[i] = best[i] + scale * grad[i];
}

// ------------------------------------------------------------------ intensity rescale
// reg_intensityRescale_core<float> (reg-lib/cpu/_reg_tools.cpp:93-183): min/max over finite values.
__global__ void __launch_bounds__(kBlock)
k_minmax(const float *__restrict__ d, size_t n, uint32_t *__restrict__ mm) {
    float lo = INFINITY, hi = -INFINITY;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float v = d[i];
        if (v == v) { lo = fminf(lo, v); hi = fmaxf(hi, v); }
    }
    for (int off = 32; off > 0; off >>= 1) {
        lo = fminf(lo, __shfl_down(lo, off, 64));
        hi = fmaxf(hi, __shfl_down(hi, off, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        // order-preserving integer keys of the floats
        auto key = [](float f) {
            uint32_t u = __float_as_uint(f);
            return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
        };
        atomicMin(&mm[0], key(lo));
        atomicMax(&mm[1], key(hi));
    }
}

__device__ __forceinline__ float unkey(uint32_t k) {
    const uint32_t u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
    return __uint_as_float(u);
}

__global__ void __launch_bounds__(kBlock)
k_rescale(float *__restrict__ d, size_t n, const uint32_t *__restrict__ mm, float newMin, float newMax) {
#pragma clang fp contract(off)
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float lo = unkey(mm[0]), hi = unkey(mm[1]);
    const double diff = (double)(hi - lo), newDiff = (double)(newMax - newMin);
    double v = (double)d[i];
    if (v == v) {
        v = (v - (double)lo) / diff;
        v = v * newDiff + (double)newMin;
    }
    d[i] = (float)v;
}

__global__ void k_fill_u32(uint32_t *p, size_t n, uint32_t v) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

__global__ void k_fill_f32(float *p, size_t n, float v) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

// ------------------------------------------------------------------ single-pair kernels
// Each wraps the block body above with the launch's own block index and count.
// The single-pair finalisation (one workgroup).  pub (may be null): it then publishes ent[0..4]
// and s1[0..n1) to coherent host memory followed by the sequence number seq (k_publish's
// layout), so the objective needs no publishing kernel of its own.
// be (may be null): the bending-energy partials of the launch before, summed into *beOut as k_be_sum
// does.  beOut may lie in s1, whose value is then the one published: neither is __restrict__.
__global__ void __launch_bounds__(1024)
k_nmi_finalize_lds(uint32_t *__restrict__ counts, int rb, int fb, double *__restrict__ pro,
                   double *__restrict__ logh, float *__restrict__ logf, double *__restrict__ ent,
                   float *__restrict__ kTab, const double *__restrict__ be, int nBe, double beScale,
                   double *beOut, double *__restrict__ pub, const double *s1, int n1, uint64_t seq) {
    __shared__ double redBe[16];
    if (be) {
        const double t = sum_partials_256(be, nBe, redBe);
        if (threadIdx.x == 0) *beOut = t * beScale;
    }
    nmi_finalize_lds_block(counts, rb, fb, pro, logh, logf, ent, kTab);
    if (pub) {
        __syncthreads();
        const int i = threadIdx.x;
        if (i < 64) {  // the first wave alone publishes
            if (i < 5) pub[i] = ent[i];
            else if (i < 5 + n1) pub[i] = s1[i - 5];
            __threadfence_system();
            if (i == 0)
                __hip_atomic_store((uint64_t *)(pub + 15), seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// Bending energy: a workgroup per brick (x) and component (y).
__global__ void __launch_bounds__(256)
k_be_value(const float *__restrict__ cpp, int gnx, int gny, int gnz, BrickGrid bg, double *__restrict__ partials) {
    be_value_block(cpp, gnx, gny, gnz, bg, partials, blockIdx.x, blockIdx.y);
}

__global__ void __launch_bounds__(256)
k_be_sum(const double *__restrict__ partials, int n, double scale, double *__restrict__ out) {
    __shared__ double red[16];
    const double t = sum_partials_256(partials, n, red);
    if (threadIdx.x == 0) *out = t * scale;
}

__global__ void __launch_bounds__(256)
k_be_gradient(const float *__restrict__ cpp, int gnx, int gny, int gnz, BrickGrid bg, Affine xyz,
              float *__restrict__ out) {
    be_gradient_block(cpp, gnx, gny, gnz, bg, xyz, out, blockIdx.x, blockIdx.y);
}

__global__ void __launch_bounds__(256)
k_be_apply(float *__restrict__ cpp, int gnx, int gny, int gnz, Affine xyz, const float *__restrict__ beGrad, float ratio,
           float *__restrict__ grad, uint32_t *__restrict__ maxBits) {
    const uint32_t bits = be_apply_at(cpp, gnx, gny, gnz, xyz, beGrad, ratio, grad,
                                      (size_t)blockIdx.x * blockDim.x + threadIdx.x);
    if (maxBits) block_track_max(maxBits, bits);
}

__global__ void __launch_bounds__(kBlock)
k_normalise_bits(float *__restrict__ g, size_t n, const uint32_t *__restrict__ bits, double *__restrict__ maxLen) {
    normalise_bits_block(g, n, bits, maxLen, blockIdx.x);
}

__global__ void __launch_bounds__(kBlock) k_cg_init(float *__restrict__ grad, float *__restrict__ G_, float *__restrict__ H,
                                                  size_t n) {
    cg_init_block(grad, G_, H, n, blockIdx.x);
}

__global__ void __launch_bounds__(kBlock)
k_cg_dots(const float *__restrict__ grad, const float *__restrict__ G_, const float *__restrict__ H, size_t n,
          double *__restrict__ partials) {
    cg_dots_block(grad, G_, H, n, partials, blockIdx.x, gridDim.x);
}

__global__ void __launch_bounds__(1024) k_cg_gamma(const double *__restrict__ partials, int nb, double *__restrict__ gam) {
    cg_gamma_block(partials, nb, gam);
}

__global__ void __launch_bounds__(kBlock)
k_cg_apply(float *__restrict__ grad, float *__restrict__ G_, float *__restrict__ H, size_t n, const double *__restrict__ gam) {
    cg_apply_block(grad, G_, H, n, gam, blockIdx.x);
}

__global__ void __launch_bounds__(kBlock)
k_update_dof(float *__restrict__ cur, const float *__restrict__ best, const float *__restrict__ grad, float scale, size_t n) {
    update_dof_block(cur, best, grad, scale, n, blockIdx.x);
}

// ------------------------------------------------------------------ batched kernels
// A batch of pairs runs every small kernel of an evaluation in one launch: the blocks of all
// pairs are listed in an item table (pair, block of that pair), and each block runs the same body
// as the single-pair kernel with that pair's arguments, its own block index and count, so every
// pair's arithmetic and reduction order are those of the pair alone.  Pairs whose flag in
// `active` is 0 are skipped.
struct PairOps {
    float *cpp, *best, *grad, *cgG, *cgH;
    int gnx, gny, gnz;
    size_t G;
    Affine xyz;
    BrickGrid bg;
    int beBlocks, cgBlocks;
    double beScale;        // 1 / (3 G)
    double *partials;      // bending-energy value and CG dot partials
    float *beGrad;
    double *beOut;         // bending energy (scalars[0])
    uint32_t *maxBits;     // max gradient length as float bits
    double *maxLen;        // scalars[1]
    double *gam;           // scalars[2]
    uint32_t *counts;
    double *pro, *logh;
    float *logf;
    double *ent;
    int rb, fb;
};

__device__ __forceinline__ bool skip_pair(const int *active, int pair) { return active && !active[pair]; }

__global__ void __launch_bounds__(1024) k_nmi_finalize_batch(const PairOps *__restrict__ P, const int *active) {
    if (skip_pair(active, blockIdx.x)) return;
    const PairOps& q = P[blockIdx.x];
    nmi_finalize_lds_block(q.counts, q.rb, q.fb, q.pro, q.logh, q.logf, q.ent);
}

__global__ void __launch_bounds__(256)
k_be_value_batch(const PairOps *__restrict__ P, const int2 *__restrict__ items, const int *active) {
    const int2 it = items[blockIdx.x];
    if (skip_pair(active, it.x)) return;
    const PairOps& q = P[it.x];
    be_value_block(q.cpp, q.gnx, q.gny, q.gnz, q.bg, q.partials, it.y, blockIdx.y);
}

__global__ void __launch_bounds__(256)
k_be_gradient_batch(const PairOps *__restrict__ P, const int2 *__restrict__ items, const int *active) {
    const int2 it = items[blockIdx.x];
    if (skip_pair(active, it.x)) return;
    const PairOps& q = P[it.x];
    be_gradient_block(q.cpp, q.gnx, q.gny, q.gnz, q.bg, q.xyz, q.beGrad, it.y, blockIdx.y);
}

// items over 3 G: element-wise kernels of the control-point arrays
__global__ void __launch_bounds__(kBlock)
k_normalise_batch(const PairOps *__restrict__ P, const int2 *__restrict__ items, const int *active) {
    const int2 it = items[blockIdx.x];
    if (skip_pair(active, it.x)) return;
    const PairOps& q = P[it.x];
    normalise_bits_block(q.grad, 3 * q.G, q.maxBits, q.maxLen, it.y);
}

// first[pair]: 1 = steepest descent (reset G, H), 0 = conjugate update
__global__ void __launch_bounds__(kBlock)
k_cg_init_batch(const PairOps *__restrict__ P, const int2 *__restrict__ items, const int *active,
                const int *__restrict__ first) {
    const int2 it = items[blockIdx.x];
    if (skip_pair(active, it.x) || !first[it.x]) return;
    const PairOps& q = P[it.x];
    cg_init_block(q.grad, q.cgG, q.cgH, 3 * q.G, it.y);
}

__global__ void __launch_bounds__(kBlock)
k_cg_dots_batch(const PairOps *__restrict__ P, const int2 *__restrict__ items, const int *active,
                const int *__restrict__ first) {
    const int2 it = items[blockIdx.x];
    if (skip_pair(active, it.x) || first[it.x]) return;
    const PairOps& q = P[it.x];
    cg_dots_block(q.grad, q.cgG, q.cgH, 3 * q.G, q.partials, it.y, q.cgBlocks);
}

__global__ void __launch_bounds__(1024)
k_cg_gamma_batch(const PairOps *__restrict__ P, const int *active, const int *__restrict__ first) {
    if (skip_pair(active, blockIdx.x) || first[blockIdx.x]) return;
    const PairOps& q = P[blockIdx.x];
    cg_gamma_block(q.partials, q.cgBlocks, q.gam);
}

__global__ void __launch_bounds__(kBlock)
k_cg_apply_batch(const PairOps *__restrict__ P, const int2 *__restrict__ items, const int *active,
                 const int *__restrict__ first) {
    const int2 it = items[blockIdx.x];
    if (skip_pair(active, it.x) || first[it.x]) return;
    const PairOps& q = P[it.x];
    cg_apply_block(q.grad, q.cgG, q.cgH, 3 * q.G, q.gam, it.y);
}

__global__ void __launch_bounds__(kBlock)
k_update_dof_batch(const PairOps *__restrict__ P, const int2 *__restrict__ items, const int *active,
                   const float *__restrict__ scales) {
    const int2 it = items[blockIdx.x];
    if (skip_pair(active, it.x)) return;
    const PairOps& q = P[it.x];
    update_dof_block(q.cpp, q.best, q.grad, scales[it.x], 3 * q.G, it.y);
}

// toBest: best <- cpp (Optimiser::StoreCurrentDof), else cpp <- best (RestoreBestDof)
__global__ void __launch_bounds__(kBlock)
k_copy_dof_batch(const PairOps *__restrict__ P, const int2 *__restrict__ items, const int *active, int toBest) {
    const int2 it = items[blockIdx.x];
    if (skip_pair(active, it.x)) return;
    const PairOps& q = P[it.x];
    const size_t i = (size_t)it.y * blockDim.x + threadIdx.x;
    if (i >= 3 * q.G) return;
    if (toBest) q.best[i] = q.cpp[i];
    else q.cpp[i] = q.best[i];
}

__global__ void k_zero_max_bits_batch(const PairOps *__restrict__ P, int n, const int *active) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && !skip_pair(active, i)) *P[i].maxBits = 0u;
}

}  // namespace

// ------------------------------------------------------------------ launches
void op_fill_u32(uint32_t *p, size_t n, uint32_t v, hipStream_t s) {
    const unsigned b = std::min(blocks_for(n), 4096u);
    hipLaunchKernelGGL(k_fill_u32, dim3(b), dim3(kBlock), 0, s, p, n, v);
}

void op_fill_f32(float *p, size_t n, float v, hipStream_t s) {
    const unsigned b = std::min(blocks_for(n), 4096u);
    hipLaunchKernelGGL(k_fill_f32, dim3(b), dim3(kBlock), 0, s, p, n, v);
}

static bool lut_rule(const nrh_f3d *h, float g[3]) {
    g[0] = h->cpp.dx / h->ref.dx;
    g[1] = h->cpp.dy / h->ref.dy;
    g[2] = h->cpp.dz / h->ref.dz;
    return g[0] == 5.f && g[1] == 5.f && g[2] == 5.f;
}

void op_spline_field(nrh_f3d *h) {
    ensure_field(h);
    float g[3];
    const int lut = lut_rule(h, g) ? 1 : 0;
    // every voxel's 4x4x4 support must lie inside the grid (the reference would extrapolate
    // through get_SlidedValues for a grid that does not cover the image)
    const int dims[3] = { h->ref.nx, h->ref.ny, h->ref.nz }, gd[3] = { h->cpp.nx, h->cpp.ny, h->cpp.nz };
    for (int i = 0; i < 3; ++i) {
        const int c = dims[i] - 1;
        const int pre = lut ? c / 5 : (int)((float)c / g[i]);
        NRH_REQUIRE(pre + 3 < gd[i], NRH_ERR_UNSUPPORTED, "control point grid does not cover the reference image");
    }
    h->velFieldVersion = 0;  // the field no longer holds a velocity exponentiation
    h->touch();
    hipLaunchKernelGGL(k_spline_field, dim3(blocks_for(h->N)), dim3(kBlock), 0, h->stream, h->ref.nx, h->ref.ny,
                       h->ref.nz, h->cpp.nx, h->cpp.ny, h->G, h->cppPos.p, h->mask.p, g[0], g[1], g[2], lut,
                       h->params.field_order, h->field.p, h->N);
    NRH_HIP(hipGetLastError());
}

void op_resample(nrh_f3d *h) {
    h->touch();
    ensure_warped(h);
    NRH_REQUIRE(!h->field.empty(), NRH_ERR_STATE, "resample before the deformation field");
    NRH_REQUIRE(!h->floImg.empty(), NRH_ERR_UNSUPPORTED, "per-operation resampling needs float32 image storage");
    hipLaunchKernelGGL(k_resample_linear, dim3(blocks_for(h->N)), dim3(kBlock), 0, h->stream, h->field.p, h->N,
                       h->mask.p, h->floImg.p, h->flo.nx, h->flo.ny, h->flo.nz, to_affine(h->flo.ijk),
                       h->params.padding, h->warped.p);
    NRH_HIP(hipGetLastError());
}

void op_image_gradient(nrh_f3d *h) {
    ensure_warped_grad(h);
    NRH_REQUIRE(!h->field.empty(), NRH_ERR_STATE, "image gradient before the deformation field");
    NRH_REQUIRE(!h->floImg.empty(), NRH_ERR_UNSUPPORTED, "per-operation gradient needs float32 image storage");
    hipLaunchKernelGGL(k_image_gradient_linear, dim3(blocks_for(h->N)), dim3(kBlock), 0, h->stream, h->field.p,
                       h->N, h->mask.p, h->floImg.p, h->flo.nx, h->flo.ny, h->flo.nz, to_affine(h->flo.ijk),
                       h->params.padding, h->warpedGrad.p);
    NRH_HIP(hipGetLastError());
}

void op_joint_histogram(nrh_f3d *h, const float *warped) {
    h->touch();
    const int rb = h->params.ref_bins, fb = h->params.flo_bins;
    // histCount is zero here: allocation zeroes it and every finalisation consumes it
    const unsigned b = std::min(blocks_for(h->N), 2048u);
    hipLaunchKernelGGL(k_joint_histogram, dim3(b), dim3(kBlock), (size_t)rb * fb * sizeof(uint32_t), h->stream,
                       ref_ptr(h), warped, h->mask.p, h->N, rb, fb, h->histCount.p);
    NRH_HIP(hipGetLastError());
}

void op_nmi_finalize(nrh_f3d *h, float *kTab, const double *pubS1, int pubN1, int bePartials) {
    h->kTabCurrent = kTab != nullptr && h->totalBins() <= kFinLds;
    NRH_REQUIRE(pubN1 < 0 || (h->totalBins() <= kFinLds && pubN1 <= 10), NRH_ERR_ARG, "finalisation cannot publish");
    if (h->totalBins() <= kFinLds) {
        const bool pub = pubN1 >= 0;
        hipLaunchKernelGGL(k_nmi_finalize_lds, dim3(1), dim3(1024), 0, h->stream, h->histCount.p, h->params.ref_bins,
                           h->params.flo_bins, h->histPro.p, h->histLog.p, h->histLogF.p, h->ent.p,
                           h->kTabCurrent ? kTab : nullptr, bePartials > 0 ? (const double *)h->partials.p : nullptr,
                           bePartials, 1.0 / (double)(3 * h->G), h->scalars.p + 0, pub ? h->publishedDev : nullptr, pubS1,
                           pub ? pubN1 : 0, pub ? ++h->publishSeq : (uint64_t)0);
    } else {
        hipLaunchKernelGGL(k_nmi_finalize, dim3(1), dim3(1024), 0, h->stream, h->histCount.p, h->params.ref_bins,
                           h->params.flo_bins, h->histPro.p, h->histLog.p, h->histLogF.p, h->ent.p);
        if (bePartials > 0) op_bending_energy_sum(h, bePartials, h->scalars.p + 0);
    }
    NRH_HIP(hipGetLastError());
}

void op_nmi_voxel_gradient(nrh_f3d *h, double weight) {
    ensure_voxel_grad(h);
    NRH_REQUIRE(!h->warped.empty() && !h->warpedGrad.empty(), NRH_ERR_STATE,
                "NMI voxel gradient needs the warped image and its gradient");
    const size_t logBytes = (size_t)h->totalBins() * sizeof(double);
    if (logBytes <= 64 * 1024) {
        // four workgroups per CU on 256 CUs, each staging the log histogram once
        const unsigned grid = std::min(blocks_for(h->N), 1024u);
        hipLaunchKernelGGL(k_nmi_voxel_gradient_lds, dim3(grid), dim3(kBlock), logBytes, h->stream, ref_ptr(h),
                           h->warped.p, h->warpedGrad.p, h->mask.p, h->N, h->params.ref_bins, h->params.flo_bins,
                           h->histLog.p, h->ent.p, weight, h->voxelGrad.p);
    } else {
        hipLaunchKernelGGL(k_nmi_voxel_gradient, dim3(blocks_for(h->N)), dim3(kBlock), 0, h->stream, ref_ptr(h),
                           h->warped.p, h->warpedGrad.p, h->mask.p, h->N, h->params.ref_bins, h->params.flo_bins,
                           h->histLog.p, h->ent.p, weight, h->voxelGrad.p);
    }
    NRH_HIP(hipGetLastError());
}

void op_nmi_voxel_gradient_eval(nrh_f3d *h) {
    const size_t bytes = (size_t)h->params.ref_bins * h->params.flo_bins * sizeof(double);
    if (bytes > 64 * 1024) {
        zero_voxel_gradient(h);
        op_nmi_voxel_gradient(h, 1.0);
        return;
    }
    ensure_voxel_grad(h);
    NRH_REQUIRE(!h->warped.empty() && !h->warpedGrad.empty(), NRH_ERR_STATE,
                "NMI voxel gradient needs the warped image and its gradient");
    h->voxelGradPending = false;
    // four workgroups per CU on 256 CUs, each staging the table once
    hipLaunchKernelGGL(k_nmi_voxel_gradient_eval, dim3(std::min(blocks_for(h->N), 1024u)), dim3(kBlock), bytes, h->stream,
                       ref_ptr(h), h->warped.p, h->warpedGrad.p, h->mask.p, h->N, h->params.ref_bins, h->params.flo_bins,
                       h->histLog.p, h->ent.p, h->voxelGrad.p);
    NRH_HIP(hipGetLastError());
}

// Cubic B-spline kernel of reg_tools_kernelConvolution (reg-lib/cpu/_reg_tools.cpp:868-904)
int convolution_kernel(float spacing, float pixdim, std::vector<float>& kern) {
    const double temp = (double)(spacing / pixdim);
    const int radius = (int)(temp * 2.0f);
    kern.resize(2 * radius + 1);
    for (int i = -radius; i <= radius; ++i) {
        const double rel = std::fabs(i / temp);
        float kv = 0.f;
        if (rel < 1.0) kv = (float)(2.0 / 3.0 - rel * rel + 0.5 * rel * rel * rel);
        else if (rel < 2.0) kv = (float)(-((rel - 2.0) * (rel - 2.0) * (rel - 2.0)) / 6.0);
        kern[i + radius] = kv;
    }
    return radius;
}

void zero_voxel_gradient(nrh_f3d *h) {
    ensure_voxel_grad(h);
    NRH_HIP(hipMemsetAsync(h->voxelGrad.p, 0, h->voxelGrad.bytes(), h->stream));
    h->voxelGradPending = false;
}

void op_convolve_voxel_gradient(nrh_f3d *h) {
    NRH_REQUIRE(!h->voxelGrad.empty(), NRH_ERR_STATE, "no voxel-based gradient to convolve");
    const size_t N = h->N;
    h->convTmp.alloc(N);
    h->convDens.alloc(N);
    h->convDensTmp.alloc(N);
    h->convNan.alloc(N);
    const int dims[3] = { h->ref.nx, h->ref.ny, h->ref.nz };
    const float pix[3] = { h->ref.dx, h->ref.dy, h->ref.dz };
    const float sp[3] = { h->cpp.dx, h->cpp.dy, h->cpp.dz };
    for (int axis = 0; axis < 3; ++axis) {
        std::vector<float> kern;
        const int radius = convolution_kernel(sp[axis], pix[axis], kern);
        if (radius > 0) {
            h->convKernel.alloc(std::max<size_t>(kern.size(), 64));
            NRH_HIP(hipMemcpyAsync(h->convKernel.p, kern.data(), kern.size() * sizeof(float), hipMemcpyHostToDevice, h->stream));
        }
        for (int comp = 0; comp < 3; ++comp) {
            float *d = h->voxelGrad.p + comp * N;
            hipLaunchKernelGGL(k_conv_prepare, dim3(blocks_for(N)), dim3(kBlock), 0, h->stream, d, (const int *)nullptr,
                               N, h->convDens.p, h->convNan.p);
            if (radius > 0 && dims[axis] > 1) {
                hipLaunchKernelGGL(k_conv_axis, dim3(blocks_for(N)), dim3(kBlock), 0, h->stream, d, h->convDens.p,
                                   dims[0], dims[1], dims[2], axis, h->convKernel.p, radius, h->convTmp.p, h->convDensTmp.p,
                                   h->params.field_order);
                NRH_HIP(hipMemcpyAsync(d, h->convTmp.p, N * sizeof(float), hipMemcpyDeviceToDevice, h->stream));
                hipLaunchKernelGGL(k_conv_normalise, dim3(blocks_for(N)), dim3(kBlock), 0, h->stream, d, h->convDensTmp.p,
                                   h->convNan.p, N);
            } else {
                hipLaunchKernelGGL(k_conv_normalise, dim3(blocks_for(N)), dim3(kBlock), 0, h->stream, d, h->convDens.p,
                                   h->convNan.p, N);
            }
        }
    }
    NRH_HIP(hipGetLastError());
}

static Affine mat_mul_affine(const float *a, const float *b) {
    // mat44 product in double stored in float (reg-lib/cpu/Maths.hpp:235-245)
    Affine r;
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 4; ++j)
            r.m[i * 4 + j] = (float)((double)a[i * 4 + 0] * (double)b[0 * 4 + j] + (double)a[i * 4 + 1] * (double)b[1 * 4 + j] +
                                     (double)a[i * 4 + 2] * (double)b[2 * 4 + j] + (double)a[i * 4 + 3] * (double)b[3 * 4 + j]);
    return r;
}

float node_weight_ratio(const nrh_f3d *h, float weight) {
    // weight *= node spacing / voxel spacing per axis (reg-lib/cpu/_reg_localTrans.cpp:1595-1604)
    const float pd[3] = { h->ref.dx, h->ref.dy, h->ref.dz };
    const float gd[3] = { h->cpp.dx, h->cpp.dy, h->cpp.dz };
    for (int i = 0; i < 3; ++i) {
        float r = gd[i];
        if (h->cpp.sform) {
            const float *m = h->cpp.xyz;
            r = std::sqrt(m[i * 4 + 0] * m[i * 4 + 0] + m[i * 4 + 1] * m[i * 4 + 1] + m[i * 4 + 2] * m[i * 4 + 2]);
        }
        r /= pd[i];
        weight *= r;
    }
    return weight;
}

void node_transforms(const nrh_f3d *h, Affine& T, Affine& R) {
    T = mat_mul_affine(h->ref.ijk, h->cpp.xyz);
    R = to_affine(h->flo.ijk);
    if (h->velocity && h->velExt0) {
        // the grid's extension 0 maps the grid into the reference space (reg-lib/cpu/
        // _reg_localTrans.cpp:1568-1592): inverse(A) between the grid and the image, and
        // inverse(A)'s 3x3 times the floating orientation in the reorientation
        float inv[16], gridToRef[16];
        nifti_inverse(h->velExt0M, inv);
        mat44_product(inv, h->cpp.xyz, gridToRef);
        T = mat_mul_affine(h->ref.ijk, gridToRef);
        M33 a, o;
        for (int i = 0; i < 3; ++i)
            for (int j = 0; j < 3; ++j) {
                a.m[i][j] = h->velExt0M[i * 4 + j];
                o.m[i][j] = h->flo.ijk[i * 4 + j];
            }
        const M33 r = m33_mul(m33_inverse(a), o);
        for (int i = 0; i < 3; ++i)
            for (int j = 0; j < 3; ++j) R.m[i * 4 + j] = r.m[i][j];
    }
}

void op_voxel_to_node(nrh_f3d *h, float weight) {
    NRH_REQUIRE(!h->voxelGrad.empty(), NRH_ERR_STATE, "no voxel-based gradient");
    Affine T, R;
    node_transforms(h, T, R);
    const float w = node_weight_ratio(h, weight);
    hipLaunchKernelGGL(k_voxel_to_node, dim3(blocks_for(h->G)), dim3(kBlock), 0, h->stream, h->voxelGrad.p, h->ref.nx,
                       h->ref.ny, h->ref.nz, h->cpp.nx, h->cpp.ny, h->cpp.nz, T, R, w, h->nodeGrad.p);
    NRH_HIP(hipGetLastError());
}

static BrickGrid brick_grid(const nrh_f3d *h) { return be_brick_grid(h->cpp.nx, h->cpp.ny, h->cpp.nz); }

void op_bending_energy(nrh_f3d *h, double *out_device) {
    const BrickGrid bg = brick_grid(h);
    const unsigned nb = (unsigned)(bg.bx * bg.by * bg.bz);
    h->partials.alloc(std::max<size_t>(h->partials.n, 3 * (size_t)nb));
    hipLaunchKernelGGL(k_be_value, dim3(nb, 3), dim3(256), 0, h->stream, h->cppPos.p, h->cpp.nx, h->cpp.ny, h->cpp.nz, bg,
                       h->partials.p);
    NRH_HIP(hipGetLastError());
    op_bending_energy_sum(h, (int)(3 * nb), out_device);
}

void op_bending_energy_sum(nrh_f3d *h, int n, double *out_device) {
    hipLaunchKernelGGL(k_be_sum, dim3(1), dim3(256), 0, h->stream, (const double *)h->partials.p, n,
                       1.0 / (double)(3 * h->G), out_device);
    NRH_HIP(hipGetLastError());
}

void op_bending_energy_gradient(nrh_f3d *h, float weight, bool trackMax) {
    const BrickGrid bg = brick_grid(h);
    if (trackMax) op_fill_u32(h->maxBits.p, 1, 0u, h->stream);
    h->beGrad.alloc(3 * h->G);
    hipLaunchKernelGGL(k_be_gradient, dim3((unsigned)(bg.bx * bg.by * bg.bz), 3), dim3(256), 0, h->stream, h->cppPos.p,
                       h->cpp.nx, h->cpp.ny, h->cpp.nz, bg, to_affine(h->cpp.xyz), h->beGrad.p);
    hipLaunchKernelGGL(k_be_apply, dim3(blocks_for(h->G)), dim3(256), 0, h->stream, h->cppPos.p, h->cpp.nx, h->cpp.ny,
                       h->cpp.nz, to_affine(h->cpp.xyz), (const float *)h->beGrad.p, weight / (float)h->G, h->nodeGrad.p,
                       trackMax ? h->maxBits.p : nullptr);
    NRH_HIP(hipGetLastError());
    h->cppVersion++;  // the round trip may have changed the last bit of some points
}

namespace {

float sig6(double v) {
    if (v == 0) return 0.f;
    const double a = std::fabs(v);
    const int e = (int)std::floor(std::log10(a));
    const double scale = std::pow(10.0, 5 - e);
    const double r = std::floor(a * scale + 0.5) / scale;
    return (float)(v < 0 ? -r : r);
}

// set_first_order_basis_values 3-D (reg-lib/cpu/_reg_splineBasis.cpp:182-290): the reference writes
// the tensor products of the B-spline first derivative {-1/2, 0, 1/2} and value {1/6, 2/3, 1/6} as
// 6-significant-digit literals; they are regenerated here.
LeBasis make_le_basis() {
    const double v[3] = { 1.0 / 6.0, 2.0 / 3.0, 1.0 / 6.0 }, d1[3] = { -0.5, 0.0, 0.5 };
    LeBasis B;
    int i = 0;
    for (int c = 0; c < 3; ++c)
        for (int b = 0; b < 3; ++b)
            for (int a = 0; a < 3; ++a, ++i) {
                B.b[0][i] = sig6(d1[a] * v[b] * v[c]);
                B.b[1][i] = sig6(v[a] * d1[b] * v[c]);
                B.b[2][i] = sig6(v[a] * v[b] * d1[c]);
            }
    return B;
}

M33 grid_reorientation(const nrh_f3d *h) {
    M33 r;
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) r.m[i][j] = h->cpp.ijk[i * 4 + j];
    return r;
}

// nifti_mat33_inverse on the host, with the long double reciprocal of niftilib.
M33 host_m33_inverse(const M33& R) {
    const double r11 = R.m[0][0], r12 = R.m[0][1], r13 = R.m[0][2];
    const double r21 = R.m[1][0], r22 = R.m[1][1], r23 = R.m[1][2];
    const double r31 = R.m[2][0], r32 = R.m[2][1], r33 = R.m[2][2];
    double deti = r11 * r22 * r33 - r11 * r32 * r23 - r21 * r12 * r33 + r21 * r32 * r13 + r31 * r12 * r23 -
                  r31 * r22 * r13;
    if (deti != 0.0L) deti = (double)(1.0L / (long double)deti);
    M33 Q;
    Q.m[0][0] = (float)(deti * (r22 * r33 - r32 * r23));
    Q.m[0][1] = (float)(deti * (-r12 * r33 + r32 * r13));
    Q.m[0][2] = (float)(deti * (r12 * r23 - r22 * r13));
    Q.m[1][0] = (float)(deti * (-r21 * r33 + r31 * r23));
    Q.m[1][1] = (float)(deti * (r11 * r33 - r31 * r13));
    Q.m[1][2] = (float)(deti * (-r11 * r23 + r21 * r13));
    Q.m[2][0] = (float)(deti * (r21 * r32 - r31 * r22));
    Q.m[2][1] = (float)(deti * (-r11 * r32 + r31 * r12));
    Q.m[2][2] = (float)(deti * (r11 * r22 - r21 * r12));
    return Q;
}

}  // namespace

void op_linear_energy(nrh_f3d *h, double *out_device, bool keepDiag) {
    static const LeBasis B = make_le_basis();
    const unsigned nb = blocks_for(h->G);
    h->leDiag.alloc(3 * h->G);
    h->partials.alloc(std::max<size_t>(h->partials.n, 2 * (size_t)nb + 64));
    hipLaunchKernelGGL(k_le_terms, dim3(nb), dim3(kBlock), 0, h->stream, h->cppPos.p, h->cpp.nx, h->cpp.ny, h->cpp.nz,
                       B, grid_reorientation(h), h->leDiag.p, h->partials.p + nb + 32, h->maxBits.p + 7,
                       1.0 / (double)(3 * h->G), out_device);
    NRH_HIP(hipGetLastError());
    h->leDiagVersion = keepDiag ? h->cppVersion : 0;
}

void op_linear_energy_gradient(nrh_f3d *h, float weight, bool trackMax) {
    static const LeBasis B = make_le_basis();
    if (h->leDiagVersion != h->cppVersion || h->leDiag.empty())
        op_linear_energy(h, h->scalars.p + 7, true);  // the per-node diagonal of the current points
    if (trackMax) op_fill_u32(h->maxBits.p, 1, 0u, h->stream);
    const float ratio = weight / (float)h->G;
    hipLaunchKernelGGL(k_le_grad, dim3(blocks_for(h->G)), dim3(kBlock), 0, h->stream, h->leDiag.p, h->cpp.nx,
                       h->cpp.ny, h->cpp.nz, B, host_m33_inverse(grid_reorientation(h)), ratio, h->nodeGrad.p,
                       trackMax ? h->maxBits.p : nullptr);
    NRH_HIP(hipGetLastError());
}

void op_max_length(nrh_f3d *h) {
    op_fill_u32(h->maxBits.p, 1, 0u, h->stream);
    const unsigned b = std::min(blocks_for(h->G), 1024u);
    hipLaunchKernelGGL(k_max_length, dim3(b), dim3(kBlock), 0, h->stream, h->nodeGrad.p, h->G, h->maxBits.p);
    hipLaunchKernelGGL(k_max_to_scalar, dim3(1), dim3(64), 0, h->stream, h->maxBits.p, h->scalars.p + 1);
    NRH_HIP(hipGetLastError());
}

void op_normalise(nrh_f3d *h, double max_length) {
    if (max_length == 0) return;
    hipLaunchKernelGGL(k_normalise, dim3(blocks_for(3 * h->G)), dim3(kBlock), 0, h->stream, h->nodeGrad.p, 3 * h->G,
                       1.0 / max_length);
    NRH_HIP(hipGetLastError());
}

void op_normalise_from_bits(nrh_f3d *h) {
    hipLaunchKernelGGL(k_normalise_bits, dim3(blocks_for(3 * h->G)), dim3(kBlock), 0, h->stream, h->nodeGrad.p,
                       3 * h->G, (const uint32_t *)h->maxBits.p, h->scalars.p + 1);
    NRH_HIP(hipGetLastError());
}

void op_max_length_bits(nrh_f3d *h) {
    op_fill_u32(h->maxBits.p, 1, 0u, h->stream);
    const unsigned b = std::min(blocks_for(h->G), 1024u);
    hipLaunchKernelGGL(k_max_length, dim3(b), dim3(kBlock), 0, h->stream, h->nodeGrad.p, h->G, h->maxBits.p);
    NRH_HIP(hipGetLastError());
}

void op_normalise_device(nrh_f3d *h) {
    hipLaunchKernelGGL(k_normalise_dev, dim3(blocks_for(3 * h->G)), dim3(kBlock), 0, h->stream, h->nodeGrad.p,
                       3 * h->G, (const double *)(h->scalars.p + 1));
    NRH_HIP(hipGetLastError());
}

void op_rescale(nrh_f3d *h, float *data, size_t n, float lo, float hi) {
    const uint32_t init[2] = { 0xffffffffu, 0u };
    NRH_HIP(hipMemcpyAsync(h->maxBits.p + 2, init, sizeof init, hipMemcpyHostToDevice, h->stream));
    const unsigned b = std::min(blocks_for(n), 2048u);
    hipLaunchKernelGGL(k_minmax, dim3(b), dim3(kBlock), 0, h->stream, data, n, h->maxBits.p + 2);
    hipLaunchKernelGGL(k_rescale, dim3(blocks_for(n)), dim3(kBlock), 0, h->stream, data, n, h->maxBits.p + 2, lo, hi);
    NRH_HIP(hipGetLastError());
}

void op_cg(nrh_f3d *h, int first) {
    const size_t n = 3 * h->G;
    if (first) {
        hipLaunchKernelGGL(k_cg_init, dim3(blocks_for(n)), dim3(kBlock), 0, h->stream, h->nodeGrad.p, h->cgG.p, h->cgH.p, n);
    } else {
        const unsigned nb = std::min(blocks_for(n), 512u);
        h->partials.alloc(std::max<size_t>(h->partials.n, 2 * (size_t)nb + 64));
        hipLaunchKernelGGL(k_cg_dots, dim3(nb), dim3(kBlock), 0, h->stream, h->nodeGrad.p, h->cgG.p, h->cgH.p, n, h->partials.p);
        hipLaunchKernelGGL(k_cg_gamma, dim3(1), dim3(1024), 0, h->stream, h->partials.p, (int)nb, h->scalars.p + 2);
        hipLaunchKernelGGL(k_cg_apply, dim3(blocks_for(n)), dim3(kBlock), 0, h->stream, h->nodeGrad.p, h->cgG.p, h->cgH.p,
                           n, (const double *)(h->scalars.p + 2));
    }
    NRH_HIP(hipGetLastError());
}

// The symmetric conjugate-gradient update (reg-lib/Optimiser.cpp:231-310): both directions'
// dot products summed before one gamma updates both; launched on fw's stream after bw's work.
__global__ void __launch_bounds__(1024)
k_cg_gamma_pair(const double *__restrict__ pf, int nf, const double *__restrict__ pb, int nb, double *__restrict__ gf,
                double *__restrict__ gb) {
    __shared__ double red[16];
    double g[2][2];
    const double *parts[2] = { pf, pb };
    const int counts[2] = { nf, nb };
    for (int d = 0; d < 2; ++d) {
        double gg = 0, dgg = 0;
        for (int i = threadIdx.x; i < counts[d]; i += blockDim.x) {
            gg += parts[d][2 * i];
            dgg += parts[d][2 * i + 1];
        }
        gg = block_sum_double(gg, red);
        __syncthreads();
        dgg = block_sum_double(dgg, red);
        __syncthreads();
        g[d][0] = gg;
        g[d][1] = dgg;
    }
    if (threadIdx.x == 0) *gf = *gb = (g[0][1] + g[1][1]) / (g[0][0] + g[1][0]);
}

void op_cg_pair(nrh_f3d *fw, nrh_f3d *bw, int first) {
    // bw's arrays are updated on fw's stream: wait for bw's queued work first
    NRH_HIP(hipStreamSynchronize(bw->stream));
    hipStream_t s = fw->stream;
    const size_t nf = 3 * fw->G, nb = 3 * bw->G;
    if (first) {
        hipLaunchKernelGGL(k_cg_init, dim3(blocks_for(nf)), dim3(kBlock), 0, s, fw->nodeGrad.p, fw->cgG.p, fw->cgH.p, nf);
        hipLaunchKernelGGL(k_cg_init, dim3(blocks_for(nb)), dim3(kBlock), 0, s, bw->nodeGrad.p, bw->cgG.p, bw->cgH.p, nb);
    } else {
        const unsigned bf = std::min(blocks_for(nf), 512u), bb = std::min(blocks_for(nb), 512u);
        fw->partials.alloc(std::max<size_t>(fw->partials.n, 2 * (size_t)bf + 64));
        bw->partials.alloc(std::max<size_t>(bw->partials.n, 2 * (size_t)bb + 64));
        hipLaunchKernelGGL(k_cg_dots, dim3(bf), dim3(kBlock), 0, s, fw->nodeGrad.p, fw->cgG.p, fw->cgH.p, nf,
                           fw->partials.p);
        hipLaunchKernelGGL(k_cg_dots, dim3(bb), dim3(kBlock), 0, s, bw->nodeGrad.p, bw->cgG.p, bw->cgH.p, nb,
                           bw->partials.p);
        hipLaunchKernelGGL(k_cg_gamma_pair, dim3(1), dim3(1024), 0, s, fw->partials.p, (int)bf, bw->partials.p, (int)bb,
                           fw->scalars.p + 2, bw->scalars.p + 2);
        hipLaunchKernelGGL(k_cg_apply, dim3(blocks_for(nf)), dim3(kBlock), 0, s, fw->nodeGrad.p, fw->cgG.p, fw->cgH.p,
                           nf, (const double *)(fw->scalars.p + 2));
        hipLaunchKernelGGL(k_cg_apply, dim3(blocks_for(nb)), dim3(kBlock), 0, s, bw->nodeGrad.p, bw->cgG.p, bw->cgH.p,
                           nb, (const double *)(bw->scalars.p + 2));
    }
    NRH_HIP(hipGetLastError());
    NRH_HIP(hipStreamSynchronize(s));
}

void op_update_dof(nrh_f3d *h, float scale) {
    const size_t n = 3 * h->G;
    hipLaunchKernelGGL(k_update_dof, dim3(blocks_for(n)), dim3(kBlock), 0, h->stream, h->cppPos.p, h->best.p,
                       h->nodeGrad.p, scale, n);
    NRH_HIP(hipGetLastError());
    h->cppVersion++;
}

namespace {
// The values, then (after a system-scope fence) the sequence number in slot 15, which the host
// polls: a reader that sees the number sees the values.
__global__ void k_publish(double *__restrict__ dst, const double *__restrict__ s0, int n0,
                          const double *__restrict__ s1, int n1, const double *__restrict__ s2, int n2,
                          uint64_t seq) {
    const int i = threadIdx.x;
    if (i < n0) dst[i] = s0[i];
    else if (i < n0 + n1) dst[i] = s1[i - n0];
    else if (i < n0 + n1 + n2) dst[i] = s2[i - n0 - n1];
    __threadfence_system();
    __syncthreads();
    if (i == 0) __hip_atomic_store((uint64_t *)(dst + 15), seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
}  // namespace

void op_publish(nrh_f3d *h, const double *s0, int n0, const double *s1, int n1, const double *s2, int n2) {
    NRH_REQUIRE(n0 + n1 + n2 <= 15, NRH_ERR_ARG, "too many scalars to publish");
    hipLaunchKernelGGL(k_publish, dim3(1), dim3(64), 0, h->stream, h->publishedDev, s0, n0, s1, n1, s2, n2,
                       ++h->publishSeq);
    NRH_HIP(hipGetLastError());
}

void wait_published(nrh_f3d *h) {
    // poll the sequence number the publish kernel writes last (a driver synchronisation costs
    // tens of microseconds of wake-up); every 256 polls ask the stream for an error, and once it
    // reports completion the number must be there
    const volatile uint64_t *seq = (const volatile uint64_t *)(h->published + 15);
    for (unsigned spins = 1;; ++spins) {
        if (__atomic_load_n((const uint64_t *)seq, __ATOMIC_ACQUIRE) == h->publishSeq) return;
        if (spins % 256 == 0) {
            const hipError_t e = hipStreamQuery(h->stream);
            if (e == hipSuccess) {
                NRH_REQUIRE(__atomic_load_n((const uint64_t *)seq, __ATOMIC_ACQUIRE) == h->publishSeq, NRH_ERR_HIP,
                            "the stream completed without publishing its results");
                return;
            }
            if (e != hipErrorNotReady) NRH_HIP(e);
        }
    }
}

double read_scalar(nrh_f3d *h, const double *dev) {
    op_publish(h, dev, 1);
    wait_published(h);
    return h->published[0];
}

// ------------------------------------------------------------------ batches of pairs
namespace {

// The objective terms of each active pair (a workgroup each) into results[8 q ..]: NMI, H_r, H_f,
// H_rf, total, the bending energy, the weighted value (reg_f3d::GetObjectiveFunctionValue with the
// linear energy off), and the current max gradient length; mirrored into coherent host memory.
// sumBe: the bending energy is summed from the partials of the launch before.
__global__ void __launch_bounds__(256)
k_batch_values(const PairOps *__restrict__ P, const int *active, int sumBe, const float *__restrict__ w,
               double *__restrict__ res, double *__restrict__ host) {
#pragma clang fp contract(off)
    __shared__ double red[16];
    const int q = blockIdx.x;
    if (skip_pair(active, q)) return;
    const PairOps& o = P[q];
    double be = 0;
    if (sumBe) {
        const double t = sum_partials_256(o.partials, 3 * o.beBlocks, red);
        if (threadIdx.x == 0) *o.beOut = be = t * o.beScale;
    } else if (threadIdx.x == 0) {
        be = *o.beOut;
    }
    if (threadIdx.x != 0) return;
    const double simW = (double)w[2 * q], beW = (double)w[2 * q + 1];
    double r[kBatchResults];
    r[0] = o.ent[4];
    for (int k = 0; k < 4; ++k) r[1 + k] = o.ent[k];
    r[5] = beW > 0 ? be : 0.0;
    const double wMeasure = simW > 0 ? simW * r[0] : 0.0;
    const double wBE = beW > 0 ? beW * r[5] : 0.0;
    r[6] = wMeasure - wBE;
    r[7] = *o.maxLen;
    for (int k = 0; k < kBatchResults; ++k) {
        res[q * kBatchResults + k] = r[k];
        host[q * kBatchResults + k] = r[k];
    }
}

}  // namespace

void batch_ops_setup(nrh_batch *b) {
    std::vector<PairOps> ops(b->P);
    std::vector<int2> itBE, itG3, itCg;
    std::vector<float> w(2 * b->P);
    for (int q = 0; q < b->P; ++q) {
        nrh_f3d *h = b->pairs[q];
        NRH_REQUIRE(h->params.measure == NRH_MEASURE_NMI && h->params.le_weight == 0.f && h->mask.empty(),
                    NRH_ERR_UNSUPPORTED, "batched pairs use NMI, no linear energy and no mask");
        NRH_REQUIRE(h->totalBins() <= kFinLds, NRH_ERR_UNSUPPORTED, "too many histogram bins for a batch");
        const BrickGrid bg = brick_grid(h);
        const int nb = bg.bx * bg.by * bg.bz;
        const size_t n3 = 3 * h->G;
        const int cgBlocks = (int)std::min(blocks_for(n3), 512u);
        h->partials.alloc(std::max(h->partials.n, std::max(3 * (size_t)nb, 2 * (size_t)cgBlocks + 64)));
        h->beGrad.alloc(3 * h->G);
        PairOps o{};
        o.cpp = h->cppPos.p;
        o.best = h->best.p;
        o.grad = h->nodeGrad.p;
        o.cgG = h->cgG.p;
        o.cgH = h->cgH.p;
        o.gnx = h->cpp.nx;
        o.gny = h->cpp.ny;
        o.gnz = h->cpp.nz;
        o.G = h->G;
        o.xyz = to_affine(h->cpp.xyz);
        o.bg = bg;
        o.beBlocks = nb;
        o.cgBlocks = cgBlocks;
        o.beScale = 1.0 / (double)(3 * h->G);
        o.partials = h->partials.p;
        o.beGrad = h->beGrad.p;
        o.beOut = h->scalars.p + 0;
        o.maxBits = h->maxBits.p;
        o.maxLen = h->scalars.p + 1;
        o.gam = h->scalars.p + 2;
        o.counts = h->histCount.p;
        o.pro = h->histPro.p;
        o.logh = h->histLog.p;
        o.logf = h->histLogF.p;
        o.ent = h->ent.p;
        o.rb = h->params.ref_bins;
        o.fb = h->params.flo_bins;
        ops[q] = o;
        w[2 * q] = h->params.similarity_weight;
        w[2 * q + 1] = h->params.be_weight;
        for (int k = 0; k < nb; ++k) itBE.push_back(make_int2(q, k));
        for (unsigned k = 0; k < blocks_for(n3); ++k) itG3.push_back(make_int2(q, (int)k));
        for (int k = 0; k < cgBlocks; ++k) itCg.push_back(make_int2(q, k));
    }
    b->pairOps.alloc(ops.size() * sizeof(PairOps));
    NRH_HIP(hipMemcpyAsync(b->pairOps.p, ops.data(), ops.size() * sizeof(PairOps), hipMemcpyHostToDevice, b->stream));
    b->weights.alloc(w.size());
    NRH_HIP(hipMemcpyAsync(b->weights.p, w.data(), w.size() * sizeof(float), hipMemcpyHostToDevice, b->stream));
    auto up = [&](DevBuf<int2>& dst, const std::vector<int2>& v, int& n) {
        dst.alloc(v.size());
        NRH_HIP(hipMemcpyAsync(dst.p, v.data(), v.size() * sizeof(int2), hipMemcpyHostToDevice, b->stream));
        n = (int)v.size();
    };
    up(b->itBE, itBE, b->nBE);
    up(b->itG3, itG3, b->nG3);
    up(b->itCg, itCg, b->nCg);
    b->results.alloc((size_t)kBatchResults * b->P);
    NRH_HIP(hipMemsetAsync(b->results.p, 0, b->results.bytes(), b->stream));
    NRH_HIP(hipStreamSynchronize(b->stream));
}

void batch_finalize(nrh_batch *b, const int *active) {
    hipLaunchKernelGGL(k_nmi_finalize_batch, dim3(b->P), dim3(1024), 0, b->stream, (const PairOps *)b->pairOps.p,
                       active);
    NRH_HIP(hipGetLastError());
}

void batch_be_value(nrh_batch *b, const int *active) {
    hipLaunchKernelGGL(k_be_value_batch, dim3(b->nBE, 3), dim3(256), 0, b->stream, (const PairOps *)b->pairOps.p,
                       b->itBE.p, active);
    NRH_HIP(hipGetLastError());
}

void batch_be_gradient(nrh_batch *b, const int *active) {
    const PairOps *P = (const PairOps *)b->pairOps.p;
    hipLaunchKernelGGL(k_zero_max_bits_batch, dim3((b->P + 255) / 256), dim3(256), 0, b->stream, P, b->P, active);
    hipLaunchKernelGGL(k_be_gradient_batch, dim3(b->nBE, 3), dim3(256), 0, b->stream, P, b->itBE.p, active);
    NRH_HIP(hipGetLastError());
}

void batch_normalise(nrh_batch *b, const int *active) {
    hipLaunchKernelGGL(k_normalise_batch, dim3(b->nG3), dim3(kBlock), 0, b->stream, (const PairOps *)b->pairOps.p,
                       b->itG3.p, active);
    NRH_HIP(hipGetLastError());
}

void batch_cg(nrh_batch *b, const int *active, const int *first) {
    const PairOps *P = (const PairOps *)b->pairOps.p;
    hipLaunchKernelGGL(k_cg_init_batch, dim3(b->nG3), dim3(kBlock), 0, b->stream, P, b->itG3.p, active, first);
    hipLaunchKernelGGL(k_cg_dots_batch, dim3(b->nCg), dim3(kBlock), 0, b->stream, P, b->itCg.p, active, first);
    hipLaunchKernelGGL(k_cg_gamma_batch, dim3(b->P), dim3(1024), 0, b->stream, P, active, first);
    hipLaunchKernelGGL(k_cg_apply_batch, dim3(b->nG3), dim3(kBlock), 0, b->stream, P, b->itG3.p, active, first);
    NRH_HIP(hipGetLastError());
}

void batch_update(nrh_batch *b, const int *active, const float *scales) {
    hipLaunchKernelGGL(k_update_dof_batch, dim3(b->nG3), dim3(kBlock), 0, b->stream, (const PairOps *)b->pairOps.p,
                       b->itG3.p, active, scales);
    NRH_HIP(hipGetLastError());
}

void batch_copy_dof(nrh_batch *b, const int *active, bool toBest) {
    hipLaunchKernelGGL(k_copy_dof_batch, dim3(b->nG3), dim3(kBlock), 0, b->stream, (const PairOps *)b->pairOps.p,
                       b->itG3.p, active, toBest ? 1 : 0);
    NRH_HIP(hipGetLastError());
}

void batch_values(nrh_batch *b, const int *active, bool sumBe) {
    hipLaunchKernelGGL(k_batch_values, dim3(b->P), dim3(256), 0, b->stream, (const PairOps *)b->pairOps.p, active,
                       sumBe ? 1 : 0, b->weights.p, b->results.p, b->publishedDev);
    NRH_HIP(hipGetLastError());
}

}  // namespace nrh

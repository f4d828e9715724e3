// Helpers shared by the F3D and Aladin drivers; no device use except by the pyramid.
#pragma once

#include <vector>
#include "common.hpp"

namespace nrh {

// nifti_mat44_inverse (reg-io/niftilib/nifti1_io.c:1680-1717)
void mat44_inverse(const float *R, float *Q);
// reg_createControlPointGrid<float> (reg-lib/cpu/_reg_localTrans.cpp:21-128)
void create_grid(const nrh_geom& ref, const float spacing[3], nrh_geom& grid, float *identity);

// reg_createSymmetricControlPointGrids<float> without an affine (reg-lib/cpu/_reg_localTrans.cpp:132-358)
void symmetric_grids(const nrh_geom& ref, const nrh_geom& flo, const float spacing[3], nrh_geom& grid, float *fw,
                     float *bw, const float *halfFw = nullptr, const float *halfBw = nullptr);
// operator*(mat44, mat44) of reg-lib/cpu/Maths.hpp:237-246 (double sums, float results)
void mat44_product(const float *A, const float *B, float *R);
// reg_createSymmetricControlPointGrids's half affines; 1 when the grids carry them as extensions
int half_affines(const float A[16], float hf[16], float hb[16]);

// Geometry of reg_downsampleImage<float>'s result with the flagged axes halved
// (reg-lib/cpu/_reg_tools.cpp:1343-1467)
void downsampled_geometry(const nrh_geom& g, const bool axes[3], nrh_geom& out);

// One level of an image pyramid on the device.
struct DevLevel {
    nrh_geom geom{};
    DevBuf<float> img;
};

// reg_createImagePyramid<float> (reg-lib/cpu/_reg_tools.cpp:1705-1733) on the current device
// (pyramid.hip): the finest level is the input; each coarser level halves the axes whose half-size
// is still >= 32 voxels.  `data` is host memory; returns with the levels complete.
std::vector<DevLevel> device_pyramid(const nrh_geom& g, const float *data, int levels, int toPerform,
                                     hipStream_t stream);

// A stream of its own for work outside any handle; drained, then destroyed.
struct ScopedStream {
    hipStream_t s = nullptr;
    ScopedStream() { NRH_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking)); }
    ~ScopedStream() {
        (void)hipStreamSynchronize(s);
        (void)hipStreamDestroy(s);
    }
    ScopedStream(const ScopedStream&) = delete;
    ScopedStream& operator=(const ScopedStream&) = delete;
};

}  // namespace nrh

"""The evaluation's convolution at the nodes only against the per-operation calls.

On grids whose nodes lie off the voxels, objective / gradient convolve the voxel gradient only at
the voxels that the nodes read.  The node gradient must equal the one of the per-operation calls
(whole-image convolution, then node extraction) bit for bit, and the voxel gradient read after the
evaluation must be the convolved one.  The grid spacings lie on both sides of the rule that keeps
the full convolution (about 3.1 voxels), on anisotropic, oblique and short images.
"""
import numpy as np
import pytest

from niftyreg_amd import _lib, phantoms
from niftyreg_amd.f3d import F3dContent, default_params
from niftyreg_amd.geometry import Geom, create_control_point_grid

pytestmark = pytest.mark.gpu


def _geom(dims, oblique):
    m = np.eye(4, dtype=np.float32)
    th = 0.25 if oblique else 0.0
    rot = np.array([[np.cos(th), -np.sin(th), 0], [np.sin(th), np.cos(th), 0], [0, 0, 1]])
    m[:3, :3] = (rot @ np.diag([1.1, 0.95, 1.2])).astype(np.float32)
    m[:3, 3] = [4.0, -3.0, 2.0]
    return Geom(dims, m)


@pytest.mark.parametrize("order", [_lib.FIELD_ORDER_SCALAR, _lib.FIELD_ORDER_SSE])
@pytest.mark.parametrize("dims,spacing,oblique", [
    ((40, 37, 33), 5.0, True),
    ((41, 30, 35), 3.6, False),   # near the rule's line
    ((24, 26, 22), 2.4, True),    # below it: the full convolution
    ((17, 9, 12), 13.0, False),   # kernels longer than the lines
])
def test_node_gradient_equals_per_operation_chain(gpu, dims, spacing, oblique, order):
    g = _geom(dims, oblique)
    ref = phantoms.blob_phantom(dims, 1).ravel()
    flo = phantoms.blob_phantom(dims, 2).ravel()
    cg, cpp = create_control_point_grid(g, [spacing] * 3)
    cpp = (cpp + np.random.default_rng(3).uniform(-1, 1, cpp.size)).astype(np.float32)
    p = default_params(similarity_weight=0.999, be_weight=0.001, field_order=order)
    h = F3dContent(g, ref, g, flo, cg, cpp, params=p)
    h.rescale_intensities((2, 65), (2, 65))
    h.objective()
    h.gradient()
    got, conv = h.node_gradient(), h.voxel_gradient()
    h.set_control_points(cpp)
    h.GetDeformationField()
    h.ResampleImage()
    h.GetImageGradient()
    h.ZeroVoxelBasedMeasureGradient()
    h.GetSimilarityMeasureValue()
    h.GetVoxelBasedSimilarityMeasureGradient(1.0)
    h.ConvolveImage()
    h.VoxelCentricToNodeCentric(0.999)
    h.ApproxBendingEnergyGradient(0.001)
    assert np.array_equal(conv, h.voxel_gradient(), equal_nan=True)
    assert np.array_equal(got, h.node_gradient(), equal_nan=True)
    assert np.isfinite(got).all() and np.abs(got).max() > 0
    h.close()

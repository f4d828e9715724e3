"""The LNCC evaluation's passes against the per-operation measure.

objective / gradient form the same sums as the per-operation calls, every product rounded to float, in
fewer passes: the value and the voxel gradient are equal bit for bit, and so is the node gradient on a
grid off the voxels.  The projection onto nodes that lie on voxels is separable where the calls convolve
the image axis by axis (1e-5, float sums of a few hundred terms).
"""
import numpy as np
import pytest

from niftyreg_amd import _lib, phantoms
from niftyreg_amd.f3d import F3dContent, default_params
from niftyreg_amd.geometry import Geom, create_control_point_grid

pytestmark = pytest.mark.gpu


def _chain(h, cpp, weight):
    h.set_control_points(cpp)
    h.GetDeformationField()
    h.ResampleImage()
    value = h.GetLnccValue()
    h.GetImageGradient()
    h.ZeroVoxelBasedMeasureGradient()
    h.GetVoxelBasedLnccGradient(1.0)
    voxel = h.voxel_gradient()
    h.ConvolveImage()
    h.VoxelCentricToNodeCentric(weight)
    h.ApproxBendingEnergyGradient(1.0 - weight)
    return value, voxel, h.node_gradient()


@pytest.mark.parametrize("dims,spacing,sigma,masked,nans,voxel", [
    ((64, 32, 32), 5.0, -5.0, False, False, (1, 1, 1)),       # whole tiles
    ((65, 33, 41), 5.0, -5.0, True, False, (1, 1, 1)),        # one past them, masked
    ((23, 70, 12), 4.0, -5.0, False, True, (1, 1, 1)),        # lines shorter than the kernel, NaN voxels
    ((40, 36, 34), 5.0, 4.5, False, False, (1.0, 1.2, 20.0)), # no smoothing along z (radius 0)
    ((41, 37, 35), 5.0, -10.0, False, False, (1, 1, 1)),      # the longest tiled kernel (radius 30)
    ((41, 37, 35), 5.0, -1.0, False, False, (1, 1, 1)),       # fewer taps than a chunk
    ((36, 34, 30), 4.6, -3.0, True, True, (1, 1, 1)),         # nodes off the voxels
    ((36, 34, 30), 4.6, -11.0, False, False, (1, 1, 1)),      # and too long a kernel
])
def test_evaluation_matches_per_operation_measure(gpu, dims, spacing, sigma, masked, nans, voxel):
    g = Geom.identity(dims, spacing=voxel)
    rng = np.random.default_rng(sum(dims))
    ref = phantoms.blob_phantom(dims, 1).ravel()
    flo = phantoms.blob_phantom(dims, 2).ravel()
    if nans:
        ref[rng.integers(0, ref.size, 20)] = np.nan
        flo[rng.integers(0, flo.size, 20)] = np.nan
    cg, cpp = create_control_point_grid(g, [spacing * p for p in g.pixdim])
    cpp = (cpp + rng.uniform(-1, 1, cpp.size)).astype(np.float32)
    mask = (rng.uniform(size=g.nvox) > 0.2).astype(np.int32) - 1 if masked else None
    p = default_params(similarity_weight=0.99, be_weight=0.01, measure=_lib.MEASURE_LNCC, lncc_sigma=sigma)
    h = F3dContent(g, ref, g, flo, cg, cpp, mask=mask, params=p)
    h.rescale_intensities((0, 1), (0, 1))
    value, terms = h.objective()
    h.gradient()
    got, vox = h.node_gradient(), h.voxel_gradient()
    h.set_control_points(cpp)
    h.gradient()  # without the objective: the same gradient
    assert np.array_equal(got, h.node_gradient())
    want_value, want_voxel, want = _chain(h, cpp, 0.99)
    h.close()
    assert terms[0] == float(np.float32(0.99)) * want_value
    assert np.isfinite(got).all() and np.isfinite(vox).all() and np.abs(want).max() > 0
    if spacing == 4.6:
        assert np.array_equal(got, want)
    else:
        assert np.array_equal(vox, want_voxel)
        assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)


@pytest.mark.parametrize("huge", [0.0, 3e15, 1e25, 3e38, np.inf])
def test_evaluation_of_signed_and_huge_intensities(gpu, huge):
    """Negative values, and values whose squares grow large or overflow, as they are (no rescaling)."""
    dims = (41, 37, 35)
    g = Geom.identity(dims)
    rng = np.random.default_rng(11)
    ref = phantoms.blob_phantom(dims, 1).ravel() - np.float32(0.4)
    flo = phantoms.blob_phantom(dims, 2).ravel() - np.float32(0.6)
    if huge:
        ref[rng.integers(0, ref.size, 2)] = [huge, -huge]
        flo[rng.integers(0, flo.size, 2)] = [-huge, huge]
    cg, cpp = create_control_point_grid(g, [5.0] * 3)
    cpp = (cpp + rng.uniform(-1, 1, cpp.size)).astype(np.float32)
    p = default_params(similarity_weight=0.99, be_weight=0.01, measure=_lib.MEASURE_LNCC, lncc_sigma=-2.0)
    h = F3dContent(g, ref, g, flo, cg, cpp, params=p)
    value, terms = h.objective()
    h.gradient()
    vox = h.voxel_gradient()
    want_value, want_voxel, _ = _chain(h, cpp, 0.99)
    h.close()
    assert terms[0] == float(np.float32(0.99)) * want_value
    assert np.abs(want_voxel).max() > 0
    assert np.array_equal(vox, want_voxel, equal_nan=True)


@pytest.mark.parametrize("dims,spacing,masked", [
    ((65, 33, 41), 5.0, True),    # the tabulated spacing: masked voxels of the field are not written
    ((64, 40, 32), 4.0, True),    # zeros there
    ((66, 37, 35), 6.0, False),
])
def test_evaluation_warps_as_the_per_operation_chain(gpu, dims, spacing, masked):
    """The field and the warped image behind a value and a gradient: those of the per-operation calls,
    bit for bit, on grids that the fused sweeps take too."""
    g = Geom.identity(dims)
    rng = np.random.default_rng(sum(dims))
    ref = phantoms.blob_phantom(dims, 1).ravel()
    flo = phantoms.blob_phantom(dims, 2).ravel()
    cg, cpp = create_control_point_grid(g, [spacing] * 3)
    cpp = (cpp + rng.uniform(-1.5, 1.5, cpp.size)).astype(np.float32)
    mask = (rng.uniform(size=g.nvox) > 0.2).astype(np.int32) - 1 if masked else None
    keep = mask > -1 if masked else np.ones(g.nvox, bool)
    p = default_params(similarity_weight=0.99, be_weight=0.01, measure=_lib.MEASURE_LNCC, lncc_sigma=-3.0)
    h = F3dContent(g, ref, g, flo, cg, cpp, mask=mask, params=p)
    h.rescale_intensities((0, 1), (0, 1))
    got = []
    for call in (h.objective, h.gradient):
        h.set_control_points(cpp)
        call()
        got.append((h.deformation_field().reshape(3, -1), h.warped().ravel()))
    h.set_control_points(cpp)
    h.GetDeformationField()
    h.ResampleImage()
    field, warped = h.deformation_field().reshape(3, -1), h.warped().ravel()
    h.close()
    for f, w in got:
        assert np.array_equal(f[:, keep], field[:, keep])
        assert np.array_equal(w[keep], warped[keep], equal_nan=True)
        if masked and spacing != 5.0:
            assert not f[:, ~keep].any()

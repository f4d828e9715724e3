"""The voxel gradient of an evaluation (one FP64 table, written in place) against the operation's own
form of the reference's sums, over images whose intensities sit inside the histogram, on its edges,
outside it, on integers and undefined, with a mask: equal to float rounding of FP64 sums of 16 terms.
"""
import numpy as np
import pytest

from niftyreg_amd import phantoms
from niftyreg_amd.f3d import F3dContent, default_params
from niftyreg_amd.geometry import Geom, create_control_point_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bins", [8, 64, 90])
@pytest.mark.parametrize("span", [(2, 3), (0, 1), (-3, -2)])  # first bin, and bins left free at the end
def test_chain_gradient(gpu, bins, span):
    dims = (31, 29, 27)
    g = Geom.identity(dims)
    cg, cpp = create_control_point_grid(g, [4.6] * 3)  # nodes off the voxels: the per-operation chain
    rng = np.random.default_rng(bins)
    cpp = (cpp + rng.uniform(-1, 1, cpp.size)).astype(np.float32)
    lo, hi = span[0], bins + 4 - span[1]
    ref = phantoms.blob_phantom(dims, 1).ravel()
    flo = phantoms.blob_phantom(dims, 8).ravel()
    ref, flo = [(lo + (a - a.min()) / (a.max() - a.min()) * (hi - lo)).astype(np.float32) for a in (ref, flo)]
    ref[::5] = np.round(ref[::5])
    ref[::101] = np.nan
    flo[::97] = np.nan
    mask = (rng.uniform(size=g.nvox) > 0.2).astype(np.int32) - 1
    h = F3dContent(g, ref, g, flo, cg, cpp, mask=mask, params=default_params(bins=bins, similarity_weight=1.0, be_weight=0.0))
    try:
        assert not h.fused_available()
        h.objective()
        h.gradient()
        got = h.node_gradient()
        h.GetDeformationField()
        h.ResampleImage()
        h.GetSimilarityMeasureValue()
        h.GetImageGradient()
        h.ZeroVoxelBasedMeasureGradient()
        h.GetVoxelBasedSimilarityMeasureGradient(1.0)
        h.ConvolveImage()
        h.ZeroTransformationGradient()
        h.VoxelCentricToNodeCentric(1.0)
        want = h.node_gradient()
        scale = np.abs(want[np.isfinite(want)]).max()
        assert np.array_equal(np.isfinite(got), np.isfinite(want))
        # a voxel's value differs by a few roundings of a float (6e-8 each); a node sums hundreds with
        # weights of sum 1
        assert np.nanmax(np.abs(got - want)) <= 1e-6 * scale
    finally:
        h.close()

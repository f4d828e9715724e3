"""The symmetric pair's objective and gradient against its chain of per-operation calls, the two images
of different sizes: exponentiated fields, warps, measures, voxel gradients, their exponentiation along
the opposite grid, convolution, node extraction, penalty gradients and the shared normalisation.

Off the voxels the evaluation convolves only what the nodes read, with the calls' sums: LNCC gradients
are equal bit for bit.  The NMI evaluation takes its derivative from one FP64 table (a few FP64 roundings
before a voxel's value is rounded to float), and where the nodes lie on voxels the projection is
separable: 1e-6 and 1e-5.
"""
import numpy as np
import pytest

from niftyreg_amd import _lib, phantoms
from niftyreg_amd.f3d import F3d2Pair, F3dContent, default_params
from niftyreg_amd.geometry import Geom, create_symmetric_control_point_grids
from test_gpu_pyramid import _oblique

pytestmark = pytest.mark.gpu
BE, LE = 0.001, 0.01


def _pair(rg, fg, measure):
    ref, flo = phantoms.blob_phantom(rg.dims, 1).ravel(), phantoms.blob_phantom(fg.dims, 4).ravel()
    spacing = [5.0 * (a + b) / 2 for a, b in zip(rg.pixdim, fg.pixdim)]
    cg, fw, bw = create_symmetric_control_point_grids(rg, fg, spacing)
    rng = np.random.default_rng(5)
    fw, bw = [(p + rng.uniform(-1.5, 1.5, p.size)).astype(np.float32) for p in (fw, bw)]
    p = [default_params(similarity_weight=1 - BE - LE, be_weight=BE, le_weight=LE, measure=measure, lncc_sigma=-3.0)
         for _ in range(2)]
    hf = F3dContent(rg, ref, fg, flo, cg, fw, params=p[0])
    hb = F3dContent(fg, flo, rg, ref, cg, bw, params=p[1])
    span = (0, 1) if measure == _lib.MEASURE_LNCC else (2, 65)
    hf.rescale_intensities(span, span)
    hb.rescale_intensities(span, span)
    return F3d2Pair(hf, hb, steps=6), fw, bw


@pytest.mark.parametrize("measure", [_lib.MEASURE_NMI, _lib.MEASURE_LNCC])
@pytest.mark.parametrize("rg,fg", [
    (Geom.identity((40, 36, 32)), Geom.identity((40, 36, 32))),
    (Geom.identity((40, 36, 32)), Geom.identity((37, 41, 30))),
    (_oblique((36, 34, 30)), Geom.identity((34, 38, 28), (1.1, 1.0, 1.2), (-2.0, 1.0, 3.0))),
])
def test_evaluation_equals_the_calls(gpu, measure, rg, fg):
    lncc = measure == _lib.MEASURE_LNCC
    pair, fw, bw = _pair(rg, fg, measure)
    hf, hb = pair.fw, pair.bw
    try:
        value, terms = pair.objective()
        length = pair.gradient(normalise=True)
        got = [h.node_gradient() for h in (hf, hb)]
        points = [h.get_control_points() for h in (hf, hb)]
        # the gradient without an objective before it: from the same points, the same
        hf.set_control_points(fw)
        hb.set_control_points(bw)
        assert pair.gradient(normalise=True) == length
        for h, g in zip((hf, hb), got):
            assert np.array_equal(h.node_gradient(), g)

        hf.set_control_points(fw)
        hb.set_control_points(bw)
        hf.velocity_steps = 6
        hf.GetDefFieldFromVelocityGrid(True)
        hb.velocity_steps = hf.velocity_steps
        hb.GetDefFieldFromVelocityGrid(False)
        sim = []
        for h in (hf, hb):
            h.ResampleImage()
            sim.append(h.GetLnccValue() if lncc else h.GetSimilarityMeasureValue()[0])
        be = [h.ApproxBendingEnergy() for h in (hf, hb)]
        le = [h.ApproxLinearEnergy() for h in (hf, hb)]
        for h in (hf, hb):
            h.GetImageGradient()
            h.ZeroVoxelBasedMeasureGradient()
            h.GetVoxelBasedLnccGradient(1.0) if lncc else h.GetVoxelBasedSimilarityMeasureGradient(1.0)
        raw = [h.voxel_gradient() for h in (hf, hb)]
        hf.ExponentiateGradient(hb)
        hb.set_voxel_gradient(raw[1])
        hb.ExponentiateGradient(hf)
        w = np.float32(1 - BE - LE)
        for h in (hf, hb):
            h.ConvolveImage()
            h.VoxelCentricToNodeCentric(w)
            h.ApproxBendingEnergyGradient(np.float32(BE))
            h.ApproxLinearEnergyGradient(np.float32(LE))
        longest = max(h.GetMaximalLength() for h in (hf, hb))
        for h in (hf, hb):
            h.NormaliseGradient(longest)
        want = [h.node_gradient() for h in (hf, hb)]
        for t, x, wt in zip(terms, (sim, be, le), (w, np.float32(BE), np.float32(LE))):
            assert abs(t - float(wt) * sum(x)) <= 1e-12 * abs(t)
        assert abs(value - (terms[0] - terms[1] - terms[2])) <= 1e-15
        for h, p in zip((hf, hb), points):
            assert np.array_equal(h.get_control_points(), p)
        for h, g, x in zip((hf, hb), got, want):
            assert np.isfinite(x).all() and np.abs(x).max() > 0.1
            off = rg.dims == (36, 34, 30)
            if off and lncc:
                assert length == longest and np.array_equal(g, x)
            else:
                assert abs(length - longest) <= 1e-6 * longest
                assert np.linalg.norm(g - x) <= (1e-6 if off else 1e-5) * np.linalg.norm(x)
    finally:
        pair.close()

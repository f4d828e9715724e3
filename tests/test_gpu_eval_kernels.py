"""The small kernels of an evaluation at the edges of their work splits: the bending energy, a
workgroup per component of a brick of 8 x 8 x 4 nodes, at grids that end on, one short of and one past
a brick; the histogram's finalisation, 1024 threads with each entry in a register, at bin counts from
a few entries to the largest that fit the LDS and past them.
"""
import numpy as np
import pytest

import oracles as O
from niftyreg_amd import phantoms
from niftyreg_amd.f3d import F3dContent, default_params
from niftyreg_amd.geometry import Geom, create_control_point_grid

pytestmark = pytest.mark.gpu


def content(dims, rb=68, fb=68, seed=0):
    g = Geom.identity(dims)
    cg, cpp = create_control_point_grid(g, [5.0] * 3)
    cpp = (cpp + np.random.default_rng(seed).uniform(-2, 2, cpp.size)).astype(np.float32)
    p = default_params()
    p.ref_bins, p.flo_bins = rb, fb
    h = F3dContent(g, phantoms.blob_phantom(dims, seed).ravel(), g, phantoms.blob_phantom(dims, seed + 7).ravel(), cg, cpp,
                   params=p)
    h.rescale_intensities((2, rb - 3), (2, fb - 3))
    return h, g, cg, cpp


# images whose grids have 5 .. 17 nodes along an axis
@pytest.mark.parametrize("dims", [(8, 8, 8), (16, 21, 6), (20, 25, 16), (21, 26, 21), (56, 61, 26), (66, 11, 31)])
def test_bending_energy_at_brick_edges(gpu, dims):
    h, g, cg, cpp = content(dims)
    try:
        want = O.orc_be(cg, cpp)
        assert abs(h.ApproxBendingEnergy() - want) <= 1e-12 * abs(want)
        start = np.random.default_rng(1).normal(size=3 * cg.nvox).astype(np.float32)
        h.set_node_gradient(start)
        h.ApproxBendingEnergyGradient(0.01)
        grad = O.orc_be_grad(cg, cpp, 0.01, start)
        assert np.array_equal(h.node_gradient(), grad)
        assert h.GetMaximalLength() == float(O.orc().orc_max_length(O.fp(grad), cg.nvox))
        h.set_control_points(cpp)
        _, terms = h.objective()  # its bending energy comes from the exact pass's launch
        assert abs(terms[1] - np.float32(0.001) * want) <= 1e-9 * want
        length = h.gradient(normalise=True)
        one = h.node_gradient()
        assert np.isclose(float(O.orc().orc_max_length(O.fp(one), cg.nvox)), 1.0, rtol=1e-6) and length > 0
    finally:
        h.close()


@pytest.mark.parametrize("bins", [24, 68])
def test_published_bending_energy_follows_the_points(gpu, bins):
    """The finalisation sums the bending energy and publishes it from the same address: each objective
    has the energy of its own points, not of the last ones."""
    h, g, cg, cpp = content((40, 36, 32), bins, bins)
    try:
        for scale in (1.0, 3.0, 0.25, 2.0):
            points = (cpp * np.float32(scale)).astype(np.float32)
            h.set_control_points(points)
            want = O.orc_be(cg, points)
            assert abs(h.objective()[1][1] - np.float32(0.001) * want) <= 1e-9 * want
    finally:
        h.close()


@pytest.mark.parametrize("rb,fb", [(8, 8), (9, 113), (113, 9), (32, 32), (33, 31), (64, 65), (88, 88), (87, 89), (90, 90)])
def test_finalisation_over_bins(gpu, rb, fb):
    h, g, cg, cpp = content((23, 22, 21), rb, fb)
    try:
        h.GetDeformationField()
        h.ResampleImage()
        nmi, ent = h.GetSimilarityMeasureValue()
        ref, _ = h.get_images()
        v, pro, logh, ent_o = O.orc_nmi(ref, h.warped(), rb, fb, None)
        # FP64 sums of up to 8100 terms in another order
        assert abs(nmi - v) <= 1e-12 * abs(v)
        assert np.allclose(ent, ent_o, rtol=1e-12, atol=0)
        p, l = h.histogram()
        assert np.allclose(p, pro, rtol=1e-12, atol=1e-18)
        assert np.allclose(l, logh, rtol=1e-12, atol=1e-15)
        if rb * fb + rb + fb > 7936:  # past the LDS the objective needs a linear-energy term
            p = default_params(le_weight=0.01)
            p.ref_bins, p.flo_bins = rb, fb
            h.set_params(p)
        _, terms = h.objective()
        be = O.orc_be(cg, cpp)
        assert abs(terms[0] / np.float32(0.999) - v) <= 1e-6 * v
        assert abs(terms[1] - np.float32(0.001) * be) <= 1e-9 * be
    finally:
        h.close()

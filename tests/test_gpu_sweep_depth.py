"""The sweeps' tile depth: a pair's own sweeps take 2, 4 or 8 slices a tile by the image's size, a
batch's always 8.  Objective, node gradient and length of a pair alone and in a batch are equal
bit for bit whatever the depth; the sizes lie on both sides of the rule's lines (320, 640, 1024 and 1600
tiles of 64 x 8 x 8) and end in partial tiles."""
import numpy as np
import pytest

from niftyreg_amd import phantoms
from niftyreg_amd.f3d import F3dBatch, F3dContent, default_params
from niftyreg_amd.geometry import Geom, create_control_point_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [
    (65, 9, 3),        # one shallow tile past each edge
    (128, 128, 77),    # 320 tiles: depth 2
    (128, 128, 81),    # 352: depth 4, the last tile one slice
    (128, 157, 121),   # 640: depth 4
    (190, 143, 95),    # 648: depth 8
    (250, 121, 125),   # 1024: depth 8
    (190, 171, 123),   # 1056: depth 4
    (190, 176, 187),   # 1584: depth 4
    (190, 176, 193),   # 1650: depth 8, the last tile one slice
])
@pytest.mark.parametrize("storage", [0, 1])
def test_depths_agree(gpu, dims, storage):
    g = Geom.identity(dims)
    rng = np.random.default_rng(sum(dims))
    ref = phantoms.shell_phantom(dims, 1).ravel()
    flo = phantoms.shell_phantom(dims, 2).ravel()
    cg, cpp = create_control_point_grid(g, [5.0] * 3)
    cpp = (cpp + rng.uniform(-1, 1, cpp.size)).astype(np.float32)
    h = F3dContent(g, ref, g, flo, cg, cpp, params=default_params(image_storage=storage))
    h.rescale_intensities((2, 65), (2, 65))
    value, terms = h.objective()
    length = h.gradient(normalise=True)
    grad = h.node_gradient()
    h.set_control_points(cpp)
    b = F3dBatch([h])
    bv, _ = b.objective()
    bl = b.gradient(normalise=True)
    assert bv[0] == value and bl[0] == length
    assert np.array_equal(h.node_gradient(), grad)
    assert np.isfinite(grad).all() and np.abs(grad).max() > 0
    b.close()
    h.close()

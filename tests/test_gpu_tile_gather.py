"""The gradient resampling through LDS (and the field composition) at the edges of their tiles: sizes
below, on and past a tile of 32 x 8 x 2 or 4 voxels, fields that are the identity, whose boxes fit,
whose boxes do not, that leave the image, and single undefined positions; against the oracle, bit for
bit.
"""
import numpy as np
import pytest

import oracles as O
from niftyreg_amd.f3d import F3dContent
from niftyreg_amd.geometry import Geom, create_control_point_grid

pytestmark = pytest.mark.gpu

SIZES = [(2, 2, 2), (31, 7, 3), (32, 8, 2), (33, 9, 8), (65, 17, 5), (70, 40, 31), (128, 129, 65)]


def positions(dims, rng, amplitude, smooth):
    z, y, x = np.meshgrid(*[np.arange(n, dtype=np.float32) for n in dims[::-1]], indexing="ij")
    p = np.stack([x, y, z])
    if smooth:
        d = [amplitude * np.sin((x * a + y * b + z * c) / 9.0 + a) for a, b, c in ((1, 2, 1), (2, 1, 3), (1, 1, 2))]
        return (p + np.stack(d)).astype(np.float32)
    return (p + rng.uniform(-amplitude, amplitude, p.shape)).astype(np.float32)


@pytest.mark.parametrize("dims", SIZES)
@pytest.mark.parametrize("amplitude,smooth", [(0.0, True), (0.4, True), (4.0, True), (0.7, False), (30.0, False)])
def test_tiles(gpu, dims, amplitude, smooth):
    rng = np.random.default_rng(sum(dims))
    g = Geom.identity(dims)
    cg, cpp = create_control_point_grid(g, [5.0] * 3)
    img = rng.uniform(size=g.nvox).astype(np.float32)
    h = F3dContent(g, img, g, img, cg, cpp)
    try:
        pos = positions(dims, rng, amplitude, smooth)
        pos[:, dims[2] // 2, dims[1] // 2, dims[0] // 2] += 1e6  # one position far outside
        grad = rng.normal(size=3 * g.nvox).astype(np.float32)
        h.set_voxel_gradient(grad)
        h.set_deformation_field(pos)
        assert np.array_equal(h.ResampleGradient(1, 0.5), O.orc_resample_gradient(g, grad, pos.ravel(), 0.5))
        field = positions(dims, rng, 1.5, False)
        h.DefFieldCompose(g, field)
        assert np.array_equal(h.deformation_field(), O.orc_def_compose(g, field.ravel(), pos.ravel()))
    finally:
        h.close()

"""Block matching at the edges of its work split: one active block a workgroup to 1536 of them, five
above (whole and partial last workgroups), the short way for blocks whose values are all defined and the
checked one beside it, against the oracle, bit for bit.
"""
import numpy as np
import pytest

import oracles as O
from niftyreg_amd import phantoms
from niftyreg_amd.aladin import AladinContent
from niftyreg_amd.geometry import Geom

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(8, 8, 4), (12, 12, 8), (16, 20, 8), (17, 19, 9), (24, 20, 24), (40, 33, 31),
                                  (64, 64, 48), (60, 60, 56), (61, 57, 55), (64, 61, 53)])
@pytest.mark.parametrize("holes", [0, 1, 40, "half"])
def test_block_matching(gpu, dims, holes):
    g = Geom.identity(dims)
    rng = np.random.default_rng(sum(dims))
    ref = phantoms.blob_phantom(dims, 5).ravel().astype(np.float32) + rng.normal(0, 0.01, g.nvox).astype(np.float32)
    warped = np.roll(ref, 1) + rng.normal(0, 0.02, g.nvox).astype(np.float32)
    if holes == "half":
        warped.reshape(dims[::-1])[:, :, : dims[0] // 2] = np.nan
    elif holes:
        warped[rng.integers(0, g.nvox, holes)] = np.nan
        ref[rng.integers(0, g.nvox, holes)] = np.nan
    tb, n = O.orc_active_blocks(g, ref, 50, None)
    h = AladinContent(g, ref, g, ref)
    try:
        assert h.active_blocks == n
        h.set_warped(warped)
        h.BlockMatching()
        rp, wp, d = h.positions()
        orp, owp, od = O.orc_block_matching(g, ref, warped, tb, n, None)
        assert d == od
        assert np.array_equal(rp, orp)
        assert np.array_equal(wp, owp, equal_nan=True)
    finally:
        h.close()

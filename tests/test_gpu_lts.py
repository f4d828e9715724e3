"""The trimmed fit at the edges of its work split (one point a thread, the sizes of its LDS variants and
past them, ragged last chunks), with undefined correspondences and with residuals that tie at the
threshold, against the oracle.
"""
import numpy as np
import pytest

import oracles as O
from niftyreg_amd import aladin, phantoms
from test_gpu_aladin import LTS_RTOL, _points

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("affine", [True, False])
@pytest.mark.parametrize("n", [16, 63, 64, 65, 1023, 1024, 1025, 4095, 4096, 4097, 16384, 32768, 32769])
def test_lts_sizes(gpu, n, affine):
    A = phantoms.random_affine(9, scale=(0.97, 1.03) if affine else (1.0, 1.0), shear=0.02 if affine else 0.0)
    rp, wp = _points(n, n, A.astype(np.float64), outliers=0.3 if n > 100 else 0.0)
    wp = wp + np.random.default_rng(n).normal(0, 0.05, wp.size).astype(np.float32)
    if n > 1000:
        wp.reshape(-1, 3)[::17] = np.nan
    got = aladin.lts(rp, wp, 50, affine)
    assert np.allclose(got, O.orc_lts(rp, wp, 50, affine), rtol=LTS_RTOL, atol=LTS_RTOL)


@pytest.mark.parametrize("n", [512, 5000])
def test_lts_ties(gpu, n):
    """Points and displacements on a coarse lattice: many residuals are equal, at the threshold too."""
    rng = np.random.default_rng(n)
    rp = rng.integers(-6, 7, (n, 3)).astype(np.float32) * 4
    wp = rp + rng.integers(-1, 2, (n, 3)).astype(np.float32)
    for percent in (30, 50, 100):
        got = aladin.lts(rp.ravel(), wp.ravel(), percent, True)
        assert np.allclose(got, O.orc_lts(rp.ravel(), wp.ravel(), percent, True), rtol=LTS_RTOL, atol=LTS_RTOL)

"""A registration's levels: where their images come from.

With one level the pyramid's only image is the input, so a registration without a pyramid (the images
uploaded for the level) must end on the same points, bit for bit: one pair, a batch, a symmetric pair.
A symmetric registration that performs only the coarser of two levels must equal a one-level one on the
images that the host downsamples, at twice the spacing (penalty weights 0: they scale with the levels).
"""
import numpy as np
import pytest

from niftyreg_amd import _lib, phantoms
from niftyreg_amd.f3d import register, register_batch, register_symmetric
from niftyreg_amd.geometry import Geom
from test_gpu_pyramid import _down, _oblique

pytestmark = pytest.mark.gpu


def _pair(rd, fd, oblique=False):
    rg = _oblique(rd) if oblique else Geom.identity(rd)
    fg = Geom.identity(fd, (1.1, 1.0, 1.2), (-2.0, 1.0, 3.0)) if oblique else Geom.identity(fd)
    return rg, phantoms.blob_phantom(rd, 1).ravel(), fg, phantoms.blob_phantom(fd, 4).ravel()


@pytest.mark.parametrize("measure", [_lib.MEASURE_NMI, _lib.MEASURE_LNCC])
@pytest.mark.parametrize("oblique", [False, True])
def test_one_level_without_a_pyramid(gpu, measure, oblique):
    p = _pair((40, 36, 34), (38, 40, 32), oblique)
    opt = dict(levels=1, maxit=6, measure=measure, lncc_sigma=-3.0)
    for run in (register, register_symmetric):
        a, b = run(*p, **opt, use_pyramid=True), run(*p, **opt, use_pyramid=False)
        assert a[0].dims == b[0].dims and a[-2:] == b[-2:] and a[-1] > 0
        for u, v in zip(a[1:-2], b[1:-2]):
            assert np.isfinite(u).all() and np.array_equal(u, v)


def test_one_level_batch_without_a_pyramid(gpu):
    pairs = [_pair(d, d) for d in ((40, 36, 34), (33, 44, 30))]
    a, _ = register_batch(pairs, levels=1, maxit=6, use_pyramid=True)
    b, _ = register_batch(pairs, levels=1, maxit=6, use_pyramid=False)
    for u, v in zip(a, b):
        assert np.isfinite(u[1]).all() and np.array_equal(u[1], v[1]) and u[2:] == v[2:]


def test_two_levels_without_a_pyramid(gpu):
    """The second level uploads the images again: it starts from the first level's points and gains."""
    p = _pair((40, 36, 34), (38, 40, 32))
    for run in (register, register_symmetric):
        one = run(*p, levels=1, spacing=10.0, be=0.0, le=0.0, maxit=6, use_pyramid=False)
        two = run(*p, levels=2, spacing=5.0, be=0.0, le=0.0, maxit=3, use_pyramid=False)
        assert all(np.isfinite(u).all() for u in two[1:-2]) and two[-2] > one[-2]


@pytest.mark.parametrize("measure", [_lib.MEASURE_NMI, _lib.MEASURE_LNCC])
@pytest.mark.parametrize("rd,fd,oblique", [((67, 70, 66), (70, 66, 64), False), ((66, 81, 40), (72, 64, 43), True)])
def test_symmetric_coarse_level_equals_host_downsampling(gpu, measure, rd, fd, oblique):
    rg, ref, fg, flo = _pair(rd, fd, oblique)
    opt = dict(be=0.0, le=0.0, maxit=4, measure=measure, lncc_sigma=-3.0)
    whole = register_symmetric(rg, ref, fg, flo, levels=2, levels_to_perform=1, spacing=5.0, **opt)
    (rc, rimg), (fc, fimg) = _down(rg, ref), _down(fg, flo)
    coarse = register_symmetric(rc, rimg, fc, fimg, levels=1, spacing=10.0, **opt)
    assert whole[0].dims == coarse[0].dims and whole[3:] == coarse[3:] and whole[4] > 0
    for u, v in zip(whole[1:3], coarse[1:3]):
        assert np.isfinite(u).all() and np.array_equal(u, v)

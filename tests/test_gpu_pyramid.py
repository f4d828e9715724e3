"""The device pyramid against the host's nrh_downsample_image.

A registration that performs only its coarsest level on a full-resolution image must equal, bit for
bit, a one-level registration on the image downsampled on the host: odd sizes, an axis too short
to halve, an oblique geometry and NaN voxels (also at a decimated voxel).  For lines of fewer
voxels than the smoothing kernel's five taps, the starting NMI of the two.
"""
import ctypes

import numpy as np
import pytest

from niftyreg_amd import _lib, aladin
from niftyreg_amd.f3d import register
from niftyreg_amd.geometry import Geom

pytestmark = pytest.mark.gpu


def _down(g, img):
    axes = np.array([n // 2 >= 32 for n in g.dims], np.int32)
    gc, out = g.to_c(), _lib.nrh_geom()
    _lib.call("nrh_downsample_image", ctypes.byref(gc), _lib.fptr(img), _lib.iptr(axes), ctypes.byref(out), None)
    og = Geom.from_c(out)
    res = np.empty(og.nvox, np.float32)
    _lib.call("nrh_downsample_image", ctypes.byref(gc), _lib.fptr(img), _lib.iptr(axes), ctypes.byref(out),
              _lib.fptr(res))
    return og, res


def _oblique(dims):
    th = 0.25
    m = np.eye(4, dtype=np.float32)
    rot = np.array([[np.cos(th), -np.sin(th), 0], [np.sin(th), np.cos(th), 0], [0, 0, 1]])
    m[:3, :3] = (rot @ np.diag([1.1, 0.95, 1.2])).astype(np.float32)
    m[:3, 3] = [4.0, -3.0, 2.0]
    return Geom(dims, m)


@pytest.mark.parametrize("dims,oblique,nans,levels", [
    ((64, 64, 64), False, False, 2),
    ((67, 81, 40), True, False, 2),     # the z axis is not halved
    ((129, 65, 64), False, True, 3),
])
def test_coarse_level_equals_host_downsampling(gpu, dims, oblique, nans, levels):
    g = _oblique(dims) if oblique else Geom.identity(dims)
    rng = np.random.default_rng(sum(dims))
    z, y, x = np.meshgrid(*[np.arange(n) for n in dims[::-1]], indexing="ij")
    base = np.sin(x / 5.0) + np.cos(y / 7.0 + x / 11.0) + np.sin(z / 4.0 + y / 9.0)
    ref = (base + rng.normal(0, 0.05, base.shape)).astype(np.float32).reshape(-1)
    flo = (np.roll(base, (0, 1, 1), (0, 1, 2)) + rng.normal(0, 0.05, base.shape)).astype(np.float32).reshape(-1)
    if nans:
        ref[rng.integers(0, ref.size, 200)] = np.nan
        flo[rng.integers(0, flo.size, 200)] = np.nan
        flo[0] = ref[0] = np.nan
    opt = dict(levels_to_perform=1, rigid=False, align_centre=False, maxit=2)
    whole = aladin.register(g, ref, g, flo, levels=levels, **opt)
    rg, fg = (g, ref), (g, flo)
    for _ in range(levels - 1):
        rg, fg = _down(*rg), _down(*fg)
    coarse = aladin.register(rg[0], rg[1], fg[0], fg[1], levels=1, **opt)
    assert np.isfinite(whole).all()
    assert np.array_equal(whole, coarse)


@pytest.mark.parametrize("nz", [2, 3, 4])
def test_short_lines(gpu, nz):
    g = Geom.identity((70, 66, nz))
    rng = np.random.default_rng(nz)
    ref = rng.uniform(0, 1, g.nvox).astype(np.float32)
    flo = (ref ** 2 + rng.normal(0, 0.05, g.nvox)).astype(np.float32)
    opt = dict(be=0.0, le=0.0, maxit=0, levels_to_perform=1)
    whole = register(g, ref, g, flo, levels=2, spacing=5.0, **opt)
    rg, fg = _down(g, ref), _down(g, flo)
    coarse = register(rg[0], rg[1], fg[0], fg[1], levels=1, spacing=10.0, **opt)
    assert whole[2] == coarse[2] and whole[2] > 1.0

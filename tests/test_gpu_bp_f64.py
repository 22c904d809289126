"""All-FP64 backprojection at the edges of its tiles and pulse splits."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle
from uncc_sar_focusing_amd import _lib
from uncc_sar_focusing_amd.scenes import ImageGrid, circular_aperture

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
# An ulp of the range (1.8e-12 m at 12.5 km) is 7e-10 rad of phase at 9.6 GHz,
# independent from pulse to pulse and pixel to pixel.
TOL = 1e-9


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _case(Np, nfft, Nx, Ny, spacing, x0):
    rng = np.random.default_rng(Np * 1000 + Nx)
    geom = circular_aperture(Np, max(8, nfft // 4))
    prof = rng.standard_normal((Np, nfft)) + 1j * rng.standard_normal((Np, nfft))
    grid = ImageGrid(Nx, Ny, x0, 0.3, spacing * (Nx - 1), spacing * (Ny - 1))
    return geom, prof, grid


# one pixel block and its neighbours, one pulse, split counts 1, 2, 4 and 32; the
# last two reach past both ends of the profiles
@pytest.mark.parametrize("Np,nfft,Nx,Ny,spacing,x0", [
    (1, 2, 2, 2, 0.1, 0.0), (1, 64, 32, 16, 0.1, 0.0), (31, 256, 33, 17, 0.1, 2.0),
    (32, 256, 31, 15, 0.1, 0.0), (65, 100, 64, 33, 0.05, 0.0), (520, 512, 40, 70, 0.1, -3.0),
    (40, 128, 50, 61, 0.4, 0.0), (70, 64, 20, 300, 0.2, 0.0)])
def test_matches_oracle(ctx, Np, nfft, Nx, Ny, spacing, x0):
    geom, prof, grid = _case(Np, nfft, Nx, Ny, spacing, x0)
    args = (_dev(prof), _dev(geom.ant), _dev(geom.r0), _dev(geom.f0), grid, geom.maxWr)
    img = ctx.backproject(*args, precision="f64")
    ref = oracle.bp_f64(prof, geom.ant, geom.r0, geom.f0, grid, geom.maxWr)
    assert oracle.rel_l2(img.cpu().numpy(), ref) <= TOL
    # added to an image, and without allocating
    twice = ctx.backproject(*args, precision="f64", out=img.clone(), accumulate=True)
    assert oracle.rel_l2(twice.cpu().numpy(), 2 * ref) <= TOL
    d = _lib.BpDesc(grid.Nx, grid.Ny, nfft, Np, grid.x0, grid.y0, grid.Wx, grid.Wy, geom.maxWr,
                    _lib.SARF_BP_F64, 0, 0, 0, 0.0, 0.0)
    out = torch.empty_like(img)
    _lib.check(ctx.lib.sarf_backproject_noalloc(
        ctx._h, C.byref(d), *(C.c_void_p(t.data_ptr()) for t in args[:4]),
        C.c_void_p(out.data_ptr()), ctx._stream()))
    assert torch.equal(out, img)

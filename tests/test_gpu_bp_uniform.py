"""Tile 15's image-formation engine on each of its paths: fast pulses, pulses
gated at the swath's ends or by the carrier, pulses near enough or without a
carrier for the direct form, and windows on either side of what its LDS holds."""
import numpy as np
import pytest
import torch

import oracle
from uncc_sar_focusing_amd.scenes import Geometry, ImageGrid, circular_aperture

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
# rel-L2 1e-4 is the engine's bound against the oracle; at X band and these
# extents (at most 13 m across, 0.4 m along the line of sight) phases of some ten
# revolutions round at 1e-6: below 1e-5.
TOL = 1e-5


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _check(ctx, geom, nfft, grid, max_wr, tol=TOL, split=0):
    rng = np.random.default_rng(nfft + grid.Nx)
    n = geom.Np
    prof = (rng.standard_normal((n, nfft)) + 1j * rng.standard_normal((n, nfft))).astype(np.complex64)
    args = (_dev(prof), _dev(geom.ant), _dev(geom.r0), _dev(geom.f0), grid, max_wr)
    img = ctx.backproject(*args, tile=15, pulse_split=split)
    ref = oracle.bp_f64(prof, geom.ant, geom.r0, geom.f0, grid, max_wr)
    assert oracle.rel_l2(img.cpu().numpy(), ref) <= tol
    # the engine of the gradient's forward image and of the candidate batches
    old = ctx.backproject(*args, tile=15, pulse_split=split, for_gradient=True)
    assert oracle.rel_l2(old.cpu().numpy(), ref) <= 2 * tol


# pulses: one, around the chunk of 64, several splits; tile edges in x and y
@pytest.mark.parametrize("Np,Nx,Ny,split", [(1, 2, 2, 0), (63, 256, 8, 1), (64, 255, 9, 0),
                                            (65, 257, 7, 1), (130, 300, 21, 3)])
def test_fast_pulses(ctx, Np, Nx, Ny, split):
    geom = circular_aperture(Np, 200)
    grid = ImageGrid(Nx, Ny, 0.3, -0.2, 0.05 * (Nx - 1), 0.05 * (Ny - 1))
    _check(ctx, geom, 1024, grid, geom.maxWr, split=split)


def test_gated_at_both_ends_of_the_swath(ctx):
    """A 6 m swath under an 8 m image: pixels before, in and past the profile
    (the interpolated samples are white, so an edge pixel's gate decides)."""
    geom = circular_aperture(70, 200)
    grid = ImageGrid(200, 161, 0.0, 0.0, 0.05 * 199, 0.05 * 160)
    _check(ctx, geom, 512, grid, 6.0)


def test_gated_by_the_carrier(ctx):
    """400 revolutions per metre over 0.85 m from the tile's centre: past the 250
    of the fast path.  Phases of up to 340 revolutions round at 3e-5 of one
    (ulp), rms 8e-5 rad with two roundings."""
    geom = circular_aperture(20, 200, f0=60e9, center_deg=82.0)
    grid = ImageGrid(256, 16, 0.0, 0.0, 0.05 * 255, 0.05 * 15)
    _check(ctx, geom, 1024, grid, geom.maxWr, tol=2e-4)


def test_near_range(ctx):
    """100 m from the scene, where the cubic term along the pixel axis passes a
    millionth of a revolution.  What the expansion itself leaves out, t^2 / (8
    R^3), is 5e-6 m at a tile's corner 2.6 m from its centre: 2e-3 rad."""
    near = circular_aperture(12, 200, ground_range=80.0, altitude=60.0)
    _check(ctx, near, 512, ImageGrid(64, 24, 0.0, 0.0, 0.02 * 63, 0.02 * 23), near.maxWr, tol=2e-3)


def test_without_a_carrier(ctx):
    """Pulses with a start frequency of zero, and a negative one."""
    g = circular_aperture(12, 200)
    f0 = g.f0.copy()
    f0[::3] = 0.0
    f0[1] = -f0[1]
    mixed = Geometry(ant=g.ant, r0=g.r0, f0=f0, df=g.df, K=g.K)
    _check(ctx, mixed, 1024, ImageGrid(256, 16, 0.0, 0.0, 0.05 * 255, 0.05 * 15), g.maxWr)


@pytest.mark.parametrize("bins_per_m", [115.0, 118.0, 150.0])
def test_window_capacity(ctx, bins_per_m):
    """The worst-case window of a 256 x 8 tile at 0.05 m on either side of the
    1536 bins of the smaller LDS, with the line of sight along the tile (the
    widest windows a pulse can need): phases of up to 330 revolutions (8e-5 rad
    as above) and window positions of up to 1500 bins (ulp 1.2e-4 of a bin, rms
    5e-5 of white samples)."""
    geom = circular_aperture(9, 200, center_deg=5.0)
    nfft = 4096
    grid = ImageGrid(256, 16, 0.0, 0.0, 0.05 * 255, 0.05 * 15)
    _check(ctx, geom, nfft, grid, nfft / bins_per_m, tol=3e-4)

"""Candidate batches on either side of the size from which their kernel is the one
for five waves per SIMD: a candidate's entropy does not depend on the batch."""
import numpy as np
import pytest
import torch

from uncc_sar_focusing_amd import autofocus
from uncc_sar_focusing_amd.scenes import ImageGrid, circular_aperture

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# 8 tiles (256 x 8), 8 (128 x 16) and 8 (64 x 32): 2400 work items, and 8 x 37 at a time
@pytest.mark.parametrize("tile,Nx,Ny", [(15, 256, 64), (16, 250, 62), (13, 130, 64), (5, 127, 61)])
def test_entropy_does_not_depend_on_the_batch(ctx, tile, Nx, Ny):
    geom = circular_aperture(40, 100)
    rng = np.random.default_rng(tile)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    prof = dev((rng.standard_normal((40, 512)) + 1j * rng.standard_normal((40, 512))).astype(np.complex64))
    grid = ImageGrid(Nx, Ny, 0.0, 0.0, 0.05 * (Nx - 1), 0.05 * (Ny - 1))
    basis = dev(autofocus.detrended_basis(autofocus.poly_basis(40)))
    direction = dev(autofocus.los_directions(geom.ant))
    coefs = dev(rng.uniform(-0.3, 0.3, (300, 3)))
    args = (prof, dev(geom.ant), dev(geom.r0), dev(geom.f0), grid, geom.maxWr)
    whole = ctx.batch_entropy(*args, coefs, basis, direction, tile=tile)
    parts = torch.cat([ctx.batch_entropy(*args, c.contiguous(), basis, direction, tile=tile)
                       for c in coefs.split(37)])
    assert torch.equal(whole, parts)
    # and not one value for all
    assert whole.unique().numel() > 250

"""A start frequency below zero: its phases need the same reduction before the
sine/cosine unit (|x| <= 256 revolutions) as those of a positive one."""
import numpy as np
import pytest
import torch

import oracle
from uncc_sar_focusing_amd.scenes import ImageGrid, circular_aperture

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("tile", [5, 13, 15])
@pytest.mark.parametrize("f0", [60e9, -60e9])
def test_phases_past_the_unit(ctx, tile, f0):
    """400 revolutions per metre, rows 0.3 m apart along the line of sight: 336
    revolutions and more over half of a tile's 8 to 32 rows.  Local ranges of up
    to 3.8 m (ulp 2.4e-7 m) and phases of up to 1500 revolutions (ulp 1.2e-4)
    round at 3e-5 revolutions rms each, ten of them 6e-4 rad."""
    geom = circular_aperture(20, 200, f0=f0)
    grid = ImageGrid(256, 64, 0.0, 0.0, 0.01 * 255, 0.3 * 63)
    rng = np.random.default_rng(5)
    prof = (rng.standard_normal((20, 1024)) + 1j * rng.standard_normal((20, 1024))).astype(np.complex64)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    args = (dev(prof), dev(geom.ant), dev(geom.r0), dev(geom.f0), grid, geom.maxWr)
    ref = oracle.bp_f64(prof, geom.ant, geom.r0, geom.f0, grid, geom.maxWr)
    for gradient in (False, True):
        img = ctx.backproject(*args, tile=tile, for_gradient=gradient)
        assert oracle.rel_l2(img.cpu().numpy(), ref) <= 2e-3, gradient

"""Mixed backprojection of a near aperture: windows wider than the linear bound of
the tile, whose curvature term only the antenna's distance sets."""
import numpy as np
import pytest
import torch

import oracle
from uncc_sar_focusing_amd.scenes import ImageGrid, circular_aperture

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("gradient", [False, True])
def test_window_of_a_near_aperture(ctx, gradient):
    """256 x 8 pixels at 0.05 m seen along x from 30 m: the linear bound is 1530
    bins, the window 1643.  The range expansion leaves out 3e-3 revolutions rms
    at 9.6 GHz, 3e-4 (2e-3 rad) at 1 GHz, and 4e-5 m, 5e-3 of a bin of white samples
    (7e-3 of them): below 2e-2 together with its largest parts.  A window cut
    to 1536 bins loses 28 bins of pixels, 2 % of the image's energy."""
    geom = circular_aperture(12, 200, f0=1e9, ground_range=30.0, altitude=0.3, center_deg=3.0)
    grid = ImageGrid(256, 16, 0.0, 0.0, 0.05 * 255, 0.05 * 15)
    nfft = 4096
    bins_per_m = 1522 / (0.05 * (255 + 7))
    rng = np.random.default_rng(8)
    prof = (rng.standard_normal((12, nfft)) + 1j * rng.standard_normal((12, nfft))).astype(np.complex64)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    img = ctx.backproject(dev(prof), dev(geom.ant), dev(geom.r0), dev(geom.f0), grid,
                          nfft / bins_per_m, tile=15, pulse_split=1, for_gradient=gradient)
    ref = oracle.bp_f64(prof, geom.ant, geom.r0, geom.f0, grid, nfft / bins_per_m)
    assert oracle.rel_l2(img.cpu().numpy(), ref) <= 2e-2

"""Tile 15's engine at carriers of many range bins per revolution, where a window
position taken from the phase would magnify the phase's rounding."""
import numpy as np
import pytest
import torch

import oracle
from uncc_sar_focusing_amd.scenes import ImageGrid, circular_aperture

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# 17500, 1750, 88, 8.7, 7.3 and 0.55 bins per revolution: the direct form, positions by
# themselves down to 8, from the phase below
@pytest.mark.parametrize("f0", [3e5, 3e6, 6e7, 6e8, 7.2e8])
@pytest.mark.parametrize("max_wr", [None, 12.0])
def test_low_carrier(ctx, f0, max_wr):
    """0.1 m pixels: positions of up to 60 bins (ulp 3.8e-6 of one, rms 1.1e-6) after
    four roundings, of white samples (slope 1.4): 3e-6, the phases beside it
    small.  A swath of 12 m under a 20 m image gates pulses at both its ends."""
    geom = circular_aperture(70, 500, f0=f0)
    grid = ImageGrid(300, 200, 0.0, 0.0, 0.1 * 299, 0.1 * 199)
    wr = max_wr if max_wr else geom.maxWr
    nfft = 4096 if max_wr is None else 420
    rng = np.random.default_rng(3)
    prof = (rng.standard_normal((70, nfft)) + 1j * rng.standard_normal((70, nfft))).astype(np.complex64)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    img = ctx.backproject(dev(prof), dev(geom.ant), dev(geom.r0), dev(geom.f0), grid, wr, tile=15)
    ref = oracle.bp_f64(prof, geom.ant, geom.r0, geom.f0, grid, wr)
    assert oracle.rel_l2(img.cpu().numpy(), ref) <= 5e-6

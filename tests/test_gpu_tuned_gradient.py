"""A launch shape tuned for plain images leaves the pulse groups, and with them the
bits, of the image that a gradient is taken of alone."""
import numpy as np
import pytest
import torch

from uncc_sar_focusing_amd.api import Context
from uncc_sar_focusing_amd.scenes import ImageGrid, circular_aperture

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def test_tuned_groups():
    geom = circular_aperture(200, 100)
    rng = np.random.default_rng(1)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    prof = dev((rng.standard_normal((200, 512)) + 1j * rng.standard_normal((200, 512))).astype(np.complex64))
    grid = ImageGrid(130, 64, 0.0, 0.0, 0.1 * 129, 0.1 * 63)
    args = (prof, dev(geom.ant), dev(geom.r0), dev(geom.f0), grid, geom.maxWr)
    ctx = Context(0)
    # tile 1 is not the one a hint along y would pick, so it is the tuned one below
    for_gradient = ctx.backproject(*args, tile=1, for_gradient=True)
    explicit = ctx.backproject(*args, tile=1, pulse_split=3)
    los = geom.los()
    entry = dict(Nx=130, Ny=64, Np=200, Nfft=512, dx=grid.Wx / 129, dy=grid.Wy / 63,
                 maxWr=geom.maxWr, los_x=los[0], los_y=los[1], tile=1, pulse_split=3)
    ctx.load_tune_table([entry])
    assert torch.equal(ctx.backproject(*args, los=los), explicit)
    assert torch.equal(ctx.backproject(*args, los=los, for_gradient=True), for_gradient)
    assert not torch.equal(for_gradient, explicit)
    ctx.close()

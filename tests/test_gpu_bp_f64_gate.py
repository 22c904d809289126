"""All-FP64 backprojection: a pulse whose range is no number, infinite
or far past FP32, is outside the swath gate of every pixel and leaves the other
pulses' image alone."""
import numpy as np
import pytest
import torch

import oracle
from uncc_sar_focusing_amd.scenes import ImageGrid, circular_aperture

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
# an ulp of the range (1.8e-12 m at 12.5 km) is 7e-10 rad of phase at 9.6 GHz
TOL = 1e-9


# one workgroup for all pulses, and pulse groups
@pytest.mark.parametrize("Np,Nx,Ny", [(9, 33, 17), (70, 40, 61)])
def test_pulses_outside_the_gate(ctx, Np, Nx, Ny):
    rng = np.random.default_rng(Np)
    geom = circular_aperture(Np, 64)
    prof = rng.standard_normal((Np, 256)) + 1j * rng.standard_normal((Np, 256))
    grid = ImageGrid(Nx, Ny, 0.0, 0.0, 0.1 * (Nx - 1), 0.1 * (Ny - 1))
    ant, r0, f0 = geom.ant.copy(), geom.r0.copy(), geom.f0.copy()
    ant[1, 0] = np.nan
    r0[3], r0[4] = np.inf, -np.inf
    r0[6] += 1e6
    f0[6] = np.nan
    ant[7, 0], r0[7] = 1e21, 0.0
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    img = ctx.backproject(dev(prof), dev(ant), dev(r0), dev(f0), grid, geom.maxWr,
                          precision="f64").cpu().numpy()
    keep = np.ones(Np, dtype=bool)
    keep[[1, 3, 4, 6, 7]] = False
    ref = oracle.bp_f64(prof[keep], geom.ant[keep], geom.r0[keep], geom.f0[keep], grid, geom.maxWr)
    assert oracle.rel_l2(img, ref) <= TOL

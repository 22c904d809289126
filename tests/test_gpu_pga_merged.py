"""Batches whose images need several transform lengths: their row steps share
launches, and results equal those of every image by itself bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _image(nx, ny, seed):
    rng = np.random.default_rng(seed)
    a = (rng.standard_normal((nx, ny)) + 1j * rng.standard_normal((nx, ny))) * 0.05
    a[rng.integers(nx // 3, nx - nx // 3, ny), np.arange(ny)] += 1.0
    return torch.from_numpy(a.astype(np.complex64)).to(DEV)


# transform lengths 2^5 .. 2^13: all of them; two merged ones; one merged and the
# longest, which has launches of its own; one length only; the merge's limits
# (Nx = 256 and 257: the last row by radix 2 in LDS and the first in registers)
@pytest.mark.parametrize("sizes", [
    [(2, 3), (16, 1), (17, 9), (64, 5), (100, 33), (200, 7), (256, 6), (257, 5), (512, 3),
     (513, 2), (1024, 5), (1025, 3), (2048, 2), (2049, 1)],
    [(300, 41), (900, 17)], [(2049, 3), (700, 9)], [(600, 8), (700, 5)], [(256, 1), (257, 1)]])
def test_equals_single_images(ctx, sizes):
    imgs = [_image(nx, ny, 7 * i) for i, (nx, ny) in enumerate(sizes)]
    singles = [i.clone() for i in imgs]
    got = ctx.pga_scenes(imgs, 3)
    for img, one, (af, rms) in zip(imgs, singles, got):
        af1, rms1 = ctx.pga(one, 3)
        assert torch.equal(img, one)
        assert torch.equal(af, af1) and torch.equal(rms, rms1)

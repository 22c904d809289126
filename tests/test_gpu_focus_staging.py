"""Uploads of the host-buffer path in pieces through the pinned staging: the
pageable call against the page-locked one, which sends each pulse group in one
copy.  The kernels and pulse groups are the same, so the images are equal to
the last bit."""
import numpy as np
import pytest
import torch

from uncc_sar_focusing_amd.api import Context
from uncc_sar_focusing_amd.scenes import ImageGrid, circular_aperture

pytestmark = pytest.mark.gpu


# rows of 4 KiB: 512 pulses are one piece of 2 MiB; 2100 pulses are groups of
# 262, 919 and 919, the latter of two pieces each
@pytest.mark.parametrize("sizes", [(1,), (511, 512, 513), (1025, 2), (2100, 600, 2100)])
def test_pageable_upload_in_pieces_equals_one_copy(sizes):
    ctx = Context(0)
    grid = ImageGrid(24, 20, 0.1, -0.2, 5.0, 4.0)
    for Np in sizes:
        rng = np.random.default_rng(Np)
        geom = circular_aperture(Np, 512)
        pin = torch.empty((Np, 512), dtype=torch.complex64, pin_memory=True)
        ph = (rng.standard_normal((Np, 512)) + 1j * rng.standard_normal((Np, 512))).astype(np.complex64)
        pin.copy_(torch.from_numpy(ph))
        args = (geom.ant, geom.r0, geom.f0, grid, 512, geom.maxWr)
        ref = ctx.focus_host(pin.numpy(), *args)
        img = ctx.focus_host(ph, *args)
        assert np.abs(ref).min() > 0
        assert np.array_equal(img, ref), Np

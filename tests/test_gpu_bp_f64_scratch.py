"""All-FP64 backprojection where it has no scratch for partial images: the same
bits as with it."""
import ctypes as C
from contextlib import closing

import numpy as np
import pytest
import torch

from uncc_sar_focusing_amd import _lib
from uncc_sar_focusing_amd.api import Context
from uncc_sar_focusing_amd.scenes import ImageGrid, circular_aperture

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _inputs(Np, Nx, Ny, seed):
    rng = np.random.default_rng(seed)
    geom = circular_aperture(Np, 64)
    prof = rng.standard_normal((Np, 256)) + 1j * rng.standard_normal((Np, 256))
    grid = ImageGrid(Nx, Ny, 0.0, 0.0, 0.1 * (Nx - 1), 0.1 * (Ny - 1))
    return (_dev(prof), _dev(geom.ant), _dev(geom.r0), _dev(geom.f0), grid, geom.maxWr)


def test_first_call_under_capture():
    """A context whose first FP64 image is captured: nothing to allocate."""
    args = _inputs(130, 50, 41, 1)
    with closing(Context(0)) as warm:
        ref = warm.backproject(*args, precision="f64")
        twice = warm.backproject(*args, precision="f64", out=ref.clone(), accumulate=True)
    with closing(Context(0)) as ctx:
        out = torch.empty_like(ref)
        g = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(g):
            ctx.backproject(*args, precision="f64", out=out)
        for _ in range(3):
            out.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, ref)
        g2 = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g2):
            ctx.backproject(*args, precision="f64", out=out, accumulate=True)
        g2.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, twice)
        # an eager call afterwards has its scratch
        assert torch.equal(ctx.backproject(*args, precision="f64"), ref)


def test_allocation_free_calls_that_overlap():
    """Two contexts on two streams: the allocation-free entry shares no scratch in
    FP64."""
    cases = [_inputs(256, 150, 130, 2), _inputs(200, 170, 140, 3)]
    ctxs = [Context(0), Context(0)]
    refs = [c.backproject(*a, precision="f64") for c, a in zip(ctxs, cases)]
    outs = [torch.empty_like(r) for r in refs]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for _ in range(5):
        for o in outs:
            o.zero_()
        torch.cuda.synchronize()
        for c, a, o, st in zip(ctxs, cases, outs, streams):
            grid = a[4]
            d = _lib.BpDesc(grid.Nx, grid.Ny, a[0].shape[1], a[0].shape[0], grid.x0, grid.y0,
                            grid.Wx, grid.Wy, a[5], _lib.SARF_BP_F64, 0, 0, 0, 0.0, 0.0)
            _lib.check(c.lib.sarf_backproject_noalloc(
                c._h, C.byref(d), *(C.c_void_p(t.data_ptr()) for t in a[:4]),
                C.c_void_p(o.data_ptr()), C.c_void_p(st.cuda_stream)))
        torch.cuda.synchronize()
        for o, r in zip(outs, refs):
            assert torch.equal(o, r)
    for c in ctxs:
        c.close()

"""Rounding of range compression against long double: through global memory no more
than that of radix-4 passes with every twiddle from a table, at lengths that are no
power of two no more than that of the longer convolution."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _error(ctx, Np, K, nfft, dtype):
    rng = np.random.default_rng(nfft)
    ph = (rng.standard_normal((Np, K)) + 1j * rng.standard_normal((Np, K))).astype(dtype)
    got = ctx.range_compress(torch.from_numpy(ph).to("cuda:0"), nfft).cpu().numpy()
    ref = np.fft.fftshift(np.fft.ifft(ph.astype(np.clongdouble), n=nfft, axis=1), axes=1)
    d = got.astype(np.clongdouble) - ref
    return float(np.sqrt(np.sum(np.abs(d) ** 2) / np.sum(np.abs(ref) ** 2)))


# The same operations on the host give rel-L2 1.23e-7 at 2^16 (radix-4 passes 1.28e-7)
# and 1.32e-7 at 2^17 (1.32e-7).
@pytest.mark.parametrize("nfft,tol", [(65536, 1.31e-7), (131072, 1.36e-7)])
def test_fp32(ctx, nfft, tol):
    assert _error(ctx, 5, 6000, nfft, np.complex64) <= tol


# On the host 1.20e-16 at 32 (radix-4 passes 1.21e-16), 2.75e-16 at 1024 (2.79e-16) and
# 2.97e-16 at 4096 (3.35e-16).
@pytest.mark.parametrize("Np,K,nfft,tol", [(2000, 3, 32, 1.25e-16), (200, 102, 1024, 2.84e-16),
                                           (50, 410, 4096, 3.2e-16)])
def test_fp64(ctx, Np, K, nfft, tol):
    assert _error(ctx, Np, K, nfft, np.complex128) <= tol


# Lengths that are no power of two.  The bounds are the errors of plain transforms of the
# length for 2 N - 1, whatever K, in the register-resident kernel and in radix-4 passes.
@pytest.mark.parametrize("N,K,tol", [(37, 28, 1.30e-7), (65, 64, 1.62e-7), (300, 213, 1.79e-7),
                                     (1025, 1024, 2.35e-7), (3000, 731, 2.77e-7),
                                     (4097, 4096, 4.2e-7), (20011, 3000, 1.73e-7)])
def test_fp32_other_lengths(ctx, N, K, tol):
    assert _error(ctx, 400 if N < 2000 else 20, K, N, np.complex64) <= tol


@pytest.mark.parametrize("N,K,tol", [(3000, 700, 6.8e-16)])
def test_fp64_other_lengths(ctx, N, K, tol):
    assert _error(ctx, 20, K, N, np.complex128) <= tol

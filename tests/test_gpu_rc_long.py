"""Range compression through global-memory passes: every number of passes and
every radix, in both precisions, with more pulses than one slab holds."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
# FP32: each of the log2 N butterfly levels and each twiddle rounds at 6e-8,
# growing as the square root: below 5e-7 at 2^20; a Bluestein length takes two
# transforms of twice the length.  FP64 the same with 1.1e-16.
TOL = {np.complex64: 1e-6, np.complex128: 4e-15}


def _check(ctx, Np, K, nfft, dtype, taper, ramp, tol):
    rng = np.random.default_rng(nfft + Np)
    ph = (rng.standard_normal((Np, K)) + 1j * rng.standard_normal((Np, K))).astype(dtype)
    w = np.hamming(K).astype(np.float32) if taper else None
    fr = (9.6e9 + 1e6 * np.arange(Np), 12500.0 + 0.37 * np.arange(Np)) if ramp else None
    dev = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    prof = ctx.range_compress(dev(ph), nfft, taper=dev(w) if taper else None,
                              ramp=tuple(dev(a) for a in fr) if ramp else None).cpu().numpy()
    x = ph.astype(np.complex128) * (w.astype(np.float64) if taper else 1.0)
    ref = np.fft.fftshift(np.fft.ifft(x, n=nfft, axis=1), axes=1)
    if ramp:
        ref = ref * np.exp(-4j * np.pi / 299792458.0 * fr[0] * fr[1])[:, None]
    assert oracle.rel_l2(prof, ref) <= tol, (nfft, K)


@pytest.mark.parametrize("log2n", [1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 12, 14, 15, 16, 17, 19])
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_powers_of_two(ctx, log2n, dtype):
    n = 1 << log2n
    for Np, K in ((1, n), (5, max(1, n // 3)), (37 if log2n < 12 else 3, max(1, n // 2 + 1) if n > 2 else 1)):
        # the ramp is formed in FP64: its argument of 1e6 radians rounds at 1e-10
        _check(ctx, Np, K, n, dtype, log2n % 2 == 0, False, TOL[dtype])


@pytest.mark.parametrize("nfft", [3, 60, 129, 1000, 5001])
def test_other_lengths_f64(ctx, nfft):
    for Np, K in ((1, nfft), (9, max(1, nfft // 3))):
        _check(ctx, Np, K, nfft, np.complex128, True, False, 1e-14)


@pytest.mark.parametrize("nfft", [8193, 20011, 100000])
def test_other_lengths_f32(ctx, nfft):
    for Np, K in ((1, nfft), (6, nfft // 4)):
        _check(ctx, Np, K, nfft, np.complex64, False, True, 2e-6)


# the convolution length follows N + K - 1: the last K of one power of two and the
# first of the next, in the register-resident and the global-memory form
@pytest.mark.parametrize("nfft,K,dtype", [
    (3000, 1097, np.complex64), (3000, 1098, np.complex64), (37, 28, np.complex64),
    (37, 29, np.complex64), (5000, 3193, np.complex64), (8191, 2, np.complex64),
    (8191, 1, np.complex64), (9000, 7385, np.complex64), (9000, 7386, np.complex64),
    (1000, 25, np.complex128), (1000, 26, np.complex128), (3, 1, np.complex128)])
def test_convolution_length(ctx, nfft, K, dtype):
    single = dtype == np.complex64
    for Np in (1, 6):
        _check(ctx, Np, K, nfft, dtype, True, single, 2e-6 if single else 1e-14)


# 128 MB of rows a slab: 256 pulses of 2^16 bins, 128 of 2^17 (three passes),
# 512 of a Bluestein length of 2^15
@pytest.mark.parametrize("Np,K,nfft", [(259, 30, 65536), (130, 500, 131072), (515, 77, 16001)])
def test_more_pulses_than_a_slab(ctx, Np, K, nfft):
    _check(ctx, Np, K, nfft, np.complex64, True, True, 2e-6)

"""Chirp-z lengths, real kinds, inverse, on spectra that no transform of this
library made: against the inverse DFT on the host.  The smallest and the largest
length of every compiled convolution length, as in test_gpu_chirp.py.

Expected values straight from the definition (numpy, 64 bits), without the pair
pre-process of half-length transforms (signalsmith-fft.h:478-492):
  RealFFT          the unnormalised inverse of bins 0 ... N/2, bin 0 holding the
                   two real ones (DC, Nyquist)
  ModifiedRealFFT  x[t] = 2 Re sum_k X[k] e^{2 pi i t (k + 1/2) / N}
Tolerances are those of the forward real kinds there: rel L2 1e-6 in FP32, 2e-13
in FP64."""
import numpy as np
import pytest
import torch

import fft_amd
from fft_amd import _lib as L
from fft_amd import synth
from oracle import pyoracle as po
from tests.test_gpu_chirp import M32, M64, S32, S64, _edges

CASES = [(L.F32, n) for _, n in _edges(M32) + S32] + [(L.F64, n) for _, n in _edges(M64) + S64]


def _inverse(s, shifted):
    """N reals of N / 2 bins (rows), N = 2 n."""
    n = s.shape[-1]
    if not shifted:
        full = np.concatenate([s, np.zeros_like(s[..., :1])], -1)
        full[..., 0], full[..., n] = s[..., 0].real, s[..., 0].imag
        return np.fft.irfft(full, 2 * n) * (2 * n)
    y = np.fft.ifft(s, 2 * n, norm="forward")  # zeros for the mirrored bins
    return 2 * (y * np.exp(1j * np.pi * np.arange(2 * n) / (2 * n))).real


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [L.R2C, L.R2C_HALFSHIFT])
@pytest.mark.parametrize("prec,n", CASES)
def test_inverse_of_any_spectrum(prec, n, kind):
    cdt, rdt, tol = ((np.complex64, torch.float32, 1e-6) if prec == L.F32 else
                     (np.complex128, torch.float64, 2e-13))
    batch = 37 if n < 400 else 3
    s = synth.complex_uniform(n + 1, (batch, n), cdt)
    sd = torch.from_numpy(s).cuda()
    y = torch.empty(batch, 2 * n, dtype=rdt, device="cuda")
    fft_amd.Plan(2 * n, kind, prec).execute_ptr(
        sd.data_ptr(), y.data_ptr(), batch, L.INVERSE, torch.cuda.current_stream().cuda_stream)
    want = _inverse(s.astype(np.complex128), kind == L.R2C_HALFSHIFT)
    got = y.cpu().numpy()
    for row in {0, batch - 1}:
        assert po.rel_l2(got[row], want[row]) <= tol
    assert po.rel_l2(got, want) <= tol


@pytest.mark.parametrize("shifted", [False, True])
@pytest.mark.parametrize("n", [17, 50])
def test_expected_values_are_the_oracles(n, shifted):
    s = synth.complex_uniform(n, (n,), np.complex128)
    assert po.rel_l2(_inverse(s, shifted), po.real_ifft(s, half_shift=shifted)) <= 1e-12

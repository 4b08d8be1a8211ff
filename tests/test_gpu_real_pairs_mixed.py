"""Two-pass real transforms through the paired and the rotating column passes, at
the compiled mixed-radix column lengths of FP64 and the FP32 ones from 576 on: each
length as the first pass and as the second, beside 135 or 150 columns (odd and
even counts: without and with a middle column that pairs within itself; tiles of 4
to 32 columns that do not divide them), both kinds, both directions, in batches.

Expected values straight from the definition (numpy, 64 bits).  Tolerance: rel L2
1e-6 in FP32, 1e-12 in FP64, as for every two-pass length; a value that took
another partner or rotation would be off by its own size, so the largest error of
a bin is held to 1e-4 (FP32) and 1e-10 of the root mean square too."""
import numpy as np
import pytest
import torch

import fft_amd
from fft_amd import _lib as L
from fft_amd import synth

pytestmark = pytest.mark.gpu

F32_LENGTHS = [576, 600, 625, 640, 648, 675, 720, 729, 750, 768, 800, 810, 864, 900, 960, 972,
               1000]
F64_LENGTHS = [81, 125, 144, 162, 180, 192, 200, 216, 225, 240, 243, 250, 270, 288, 300, 320, 324,
               360, 375, 384, 400, 405, 432, 450, 480, 486, 500, 540] + F32_LENGTHS
# (precision, first-pass length, second-pass length)
CASES = [(p, n1, n2) for p, lengths in ((L.F32, F32_LENGTHS), (L.F64, F64_LENGTHS))
         for i, n in enumerate(lengths)
         for n1, n2 in ((n, (135, 150)[i % 2]), ((150, 135)[i % 2], n))]


def _forward(x, shifted):
    n = x.shape[-1]
    if shifted:
        return np.fft.fft(x * np.exp(-1j * np.pi * np.arange(n) / n))[..., : n // 2]
    y = np.fft.rfft(x)
    y[..., 0] += 1j * y[..., n // 2].real
    return y[..., : n // 2]


def _inverse(s, shifted):
    h = s.shape[-1]
    if shifted:
        y = np.fft.ifft(s, 2 * h, norm="forward")
        return 2 * (y * np.exp(1j * np.pi * np.arange(2 * h) / (2 * h))).real
    full = np.concatenate([s, 1j * s[..., :1]], -1)
    full[..., 0], full[..., h] = s[..., 0].real, s[..., 0].imag
    return np.fft.irfft(full, 2 * h) * (2 * h)


def _check(got, want, prec):
    tol, peak = (1e-6, 1e-4) if prec == L.F32 else (1e-12, 1e-10)
    e = np.abs(got.cpu().numpy() - want)
    rms = np.sqrt(np.mean(np.abs(want) ** 2))
    assert np.sqrt(np.mean(e ** 2)) <= tol * rms and e.max() <= peak * rms


@pytest.mark.parametrize("prec,n1,n2", CASES)
def test_column_lengths(prec, n1, n2):
    rdt, cdt = (np.float32, np.complex64) if prec == L.F32 else (np.float64, np.complex128)
    h, batch = n1 * n2, 2
    x = synth.real_uniform(h, (batch, 2 * h), rdt)
    s = synth.complex_uniform(h + 1, (batch, h), cdt)
    xd, sd = torch.from_numpy(x).cuda(), torch.from_numpy(s).cuda()
    y, z = torch.empty_like(sd), torch.empty_like(xd)
    stream = torch.cuda.current_stream().cuda_stream
    for kind in (L.R2C, L.R2C_HALFSHIFT):
        plan = fft_amd.Plan(2 * h, kind, prec, split=n1)
        plan.execute_ptr(xd.data_ptr(), y.data_ptr(), batch, 0, stream)
        plan.execute_ptr(sd.data_ptr(), z.data_ptr(), batch, 1, stream)
        _check(y, _forward(x.astype(np.float64), kind == L.R2C_HALFSHIFT), prec)
        _check(z, _inverse(s.astype(np.complex128), kind == L.R2C_HALFSHIFT), prec)

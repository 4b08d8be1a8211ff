"""Accuracy of chirp-z lengths in one launch and in three: forward, inverse and
round trip against the DFT in more bits than the plan has.

Bounds: the errors that the separate launches of bluestein.hip (the smallest
2^a 3^b 5^c convolution length, kernel transformed in the working precision)
have at these lengths on such inputs, and 2 % for the choice of the inputs.
With the convolution kernel transformed in the working precision the compiled
convolution lengths are up to 1.33 times above them."""
import numpy as np
import pytest
import scipy.fft
import torch

import fft_amd
from fft_amd import _lib as L
from fft_amd import synth

pytestmark = pytest.mark.gpu

# (precision, n, rel L2 forward, inverse, round trip)
BOUNDS = [
    (L.F32, 97, 1.73e-7, 1.73e-7, 2.48e-7),
    (L.F32, 691, 2.07e-7, 2.08e-7, 2.93e-7),
    (L.F32, 1904, 2.19e-7, 2.18e-7, 3.05e-7),
    (L.F32, 1999, 2.36e-7, 2.34e-7, 3.50e-7),
    (L.F32, 17895, 2.63e-7, 2.64e-7, 3.77e-7),
    (L.F32, 287163, 2.88e-7, 2.87e-7, 4.08e-7),
    (L.F32, 1013754, 2.93e-7, 2.93e-7, 4.14e-7),
    (L.F64, 191, 4.64e-16, 4.67e-16, 5.78e-16),
    (L.F64, 3063, 5.23e-16, 5.23e-16, 6.74e-16),
    (L.F64, 129838, 5.86e-16, 5.85e-16, 7.98e-16),
]


def _rel(y, want):
    e = y.cpu().numpy().astype(want.dtype) - want
    return float(np.linalg.norm(np.abs(e)) / np.linalg.norm(np.abs(want)))


@pytest.mark.parametrize("prec,n,fwd,inv,both", BOUNDS)
def test_no_less_exact_than_separate_launches(prec, n, fwd, inv, both):
    cdt, wide = ((np.complex64, np.complex128) if prec == L.F32 else
                 (np.complex128, np.clongdouble))
    x = synth.complex_normal(n, (max(1, 32768 // n), n), cdt)
    plan = fft_amd.Plan(n, L.C2C, prec)
    stream = torch.cuda.current_stream().cuda_stream

    def run(a, d):
        y = torch.empty_like(a)
        plan.execute_ptr(a.data_ptr(), y.data_ptr(), a.shape[0], d, stream)
        return y

    xd, xw = torch.from_numpy(x).cuda(), x.astype(wide)
    y = run(xd, 0)
    assert _rel(y, scipy.fft.fft(xw)) <= 1.02 * fwd
    assert _rel(run(xd, 1), scipy.fft.ifft(xw, norm="forward")) <= 1.02 * inv
    assert _rel(run(y, 1), xw * n) <= 1.02 * both

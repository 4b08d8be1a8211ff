"""Compiled single passes and 16-bit / F32X column passes of mixed-radix lengths:
the smallest and largest of each type, lengths whose last butterflies leave
threads idle, batches that leave part of the last block empty.  Against the
runtime-planned kernels (the same bits where the radices are the same), alone
and in place, and against the oracle (signalsmith-fft.h:295-315, :446-502).

Tolerance (oracle): rel L2 1e-6 in FP32, 1e-7 in F32X, 1e-12 in FP64; 16-bit
storage the rounding of the ideal result, twice that where an intermediate is
stored too."""
import numpy as np
import pytest
import torch

import fft_amd
from fft_amd import _lib as L
from fft_amd import synth
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

HALF = {L.F16: torch.float16, L.BF16: torch.bfloat16}
TOL = {L.F32: 1e-6, L.F32X: 1e-7, L.F64: 1e-12}

# (kind, precision, length): reals for the real kinds
CASES = (
    [(L.C2C, L.F32, n) for n in (72, 81, 100, 375, 675, 3375, 9000, 9375, 9720, 13824, 15000,
                                 15625)]
    + [(k, L.F32, 2 * h) for k in (L.R2C, L.R2C_HALFSHIFT)
       for h in (81, 90, 100, 243, 375, 500, 1620, 3375, 4374, 8748, 9000, 13122, 15000, 15625)]
    + [(L.C2C, L.F64, n) for n in (64, 100, 500, 2500, 4500, 6750, 8100, 9000)]
    + [(k, L.F64, 2 * h) for k in (L.R2C, L.R2C_HALFSHIFT)
       for h in (64, 75, 81, 135, 300, 729, 1125, 2187, 3125, 5625, 7290, 7680, 8192)]
    + [(L.C2C, p, n) for p in (L.F16, L.BF16)
       for n in (64, 81, 135, 375, 1125, 2187, 3125, 8100, 9375, 11250, 13122, 15625, 16000,
                 # two passes
                 135 * 125, 243 * 162, 360 * 375, 729 * 486, 810 * 1000, 675 * 640)]
    + [(L.C2C, L.F32X, n) for n in (64, 81, 135, 375, 1125, 2187, 3125, 6561, 7500, 7680,
                                    135 * 125, 243 * 162, 360 * 375, 729 * 486, 810 * 1000)])


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _c128(t, prec):
    v = t.float().cpu().numpy().astype(np.float64) if prec in HALF else t.cpu().numpy()
    return v[..., 0] + 1j * v[..., 1] if prec in HALF else v


def _data(kind, prec, n, batch, d):
    """Input of direction d and an output of its shape."""
    dt64 = prec == L.F64
    cdt = np.complex128 if dt64 else np.complex64
    if prec in HALF:
        g = torch.Generator(device="cpu").manual_seed(n + d)
        x = torch.randn(batch, n, 2, generator=g).to(HALF[prec]).cuda()
        return x, torch.empty_like(x)
    if kind == L.C2C:
        x = torch.from_numpy(synth.complex_normal(n + d, (batch, n), cdt)).cuda()
        return x, torch.empty_like(x)
    r = torch.from_numpy(synth.real_uniform(n, (batch, n),
                                            np.float64 if dt64 else np.float32)).cuda()
    c = torch.from_numpy(synth.complex_uniform(n, (batch, n // 2), cdt)).cuda()
    return (c, torch.empty_like(r)) if d else (r, torch.empty_like(c))


def _run(plan, x, y, d):
    plan.execute_ptr(x.data_ptr(), y.data_ptr(), x.shape[0], d, _stream())
    torch.cuda.synchronize()
    return y


def _bytes(t):
    return t.contiguous().view(torch.uint8).flatten()


@pytest.mark.parametrize("kind,prec,n", CASES)
def test_compiled_length(kind, prec, n):
    batch = 67 if n < 4000 else 5
    plan = fft_amd.Plan(n, kind, prec)
    plain = fft_amd.Plan(n, kind, prec, variant=-2)
    same = plan.info()["radices"] == plain.info()["radices"]
    for d in (0, 1):
        x, y = _data(kind, prec, n, batch, d)
        _run(plan, x, y, d)
        ref = _run(plain, x, torch.empty_like(y), d)
        if same:
            assert torch.equal(_bytes(y), _bytes(ref))
        one = _run(plan, x[batch - 2:batch - 1].clone(), torch.empty_like(y[:1]), d)
        assert torch.equal(_bytes(one), _bytes(y[batch - 2:batch - 1]))
        buf = x.clone()
        _run(plan, buf, buf, d)
        assert torch.equal(_bytes(buf), _bytes(y))
        xv, yv = _c128(x[batch - 1], prec), _c128(y[batch - 1], prec)
        if kind == L.C2C:
            xv = xv.astype(np.complex128)
            want = po.ifft(xv) if d else po.fft(xv)
        elif d:
            want = po.real_ifft(xv.astype(np.complex128), half_shift=kind == L.R2C_HALFSHIFT)
        else:
            want = po.real_fft(xv.astype(np.float64), half_shift=kind == L.R2C_HALFSHIFT)
        err = po.rel_l2(yv, want)
        if prec in HALF:
            w = torch.from_numpy(np.stack([want.real, want.imag], -1).astype(np.float32))
            ideal = po.rel_l2(_c128(w.to(HALF[prec]), prec), want)
            tol = (2.0 if plan.info()["passes"] == 2 else 1.05) * ideal + 1e-6
        else:
            tol = TOL[prec]
        assert err <= tol, (err, tol)

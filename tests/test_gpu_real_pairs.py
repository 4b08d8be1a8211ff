"""Two-pass real transforms whose pair sums run inside the column passes
(paired tiles): bitwise the same as the runtime-planned passes with the
separate post-process, at column counts that leave part of the last tile empty,
odd and even (with and without a middle column that pairs within itself), both
kinds, both directions, batched, strided and in place; and the oracle.

Tolerance (oracle): rel L2 1e-6 in FP32, 1e-12 in FP64, as for every two-pass
length."""
import ctypes

import numpy as np
import pytest
import torch

import fft_amd
from fft_amd import _lib as L
from fft_amd import synth
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

# (precision, half length h, first-pass column length N1): the second pass has
# N1 columns of length h / N1, the first h / N1 columns of length N1
CASES = [
    (L.F32, 16384 * 2, 128), (L.F32, 48000, 240), (L.F32, 46875, 375), (L.F32, 50625, 225),
    (L.F32, 18225, 135), (L.F32, 19683, 243), (L.F32, 32805, 243), (L.F32, 31250, 250),
    (L.F32, 81000, 450), (L.F32, 91125, 729), (L.F32, 1 << 17, 512), (L.F32, 1 << 20, 1024),
    (L.F32, 1 << 21, 1024), (L.F32, 625 * 125, 625), (L.F32, 17280, 160),
    (L.F64, 1 << 18, 512), (L.F64, 1 << 20, 1024),
]


def _stream():
    return torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("kind", [L.R2C, L.R2C_HALFSHIFT])
@pytest.mark.parametrize("prec,h,n1", CASES)
def test_paired_passes(prec, h, n1, kind):
    rdt, cdt = (torch.float32, torch.complex64) if prec == L.F32 else (torch.float64,
                                                                      torch.complex128)
    n, batch = 2 * h, 3
    plan = fft_amd.Plan(n, kind, prec, split=n1)
    plain = fft_amd.Plan(n, kind, prec, split=n1, variant=-2)  # no compiled kernels
    assert plan.info()["passes"] == 2
    x = torch.from_numpy(synth.real_uniform(
        h, (batch, n), np.float32 if prec == L.F32 else np.float64)).cuda()
    spec = torch.from_numpy(synth.complex_uniform(
        h + 1, (batch, h), np.complex64 if prec == L.F32 else np.complex128)).cuda()
    y = torch.empty(batch, h, dtype=cdt, device="cuda")
    z = torch.empty(batch, n, dtype=rdt, device="cuda")
    y0, z0 = torch.empty_like(y), torch.empty_like(z)
    same = plan.info()["radices"] == plain.info()["radices"]
    for p, a, b in ((plan, y, z), (plain, y0, z0)):
        p.execute_ptr(x.data_ptr(), a.data_ptr(), batch, 0, _stream())
        p.execute_ptr(spec.data_ptr(), b.data_ptr(), batch, 1, _stream())
    torch.cuda.synchronize()
    if same:
        assert torch.equal(y, y0) and torch.equal(z, z0)
    tol = 1e-6 if prec == L.F32 else 1e-12
    assert po.rel_l2(y[1].cpu().numpy(), y0[1].cpu().numpy()) <= tol
    mod = kind == L.R2C_HALFSHIFT
    want = po.real_fft(x[2].cpu().numpy().astype(np.float64), half_shift=mod)
    assert po.rel_l2(y[2].cpu().numpy(), want) <= tol
    want = po.real_ifft(spec[2].cpu().numpy().astype(np.complex128), half_shift=mod)
    assert po.rel_l2(z[2].cpu().numpy(), want) <= tol
    # alone, in place and with gaps: the same bits
    for d, src, dst in ((0, x, y), (1, spec, z)):
        buf = src.clone()
        plan.execute_ptr(buf.data_ptr(), buf.data_ptr(), batch, d, _stream())
        torch.cuda.synchronize()
        assert torch.equal(buf.view(torch.uint8).flatten(), dst.view(torch.uint8).flatten())
        one = torch.empty_like(dst[:1])
        plan.execute_ptr(src[1:2].contiguous().data_ptr(), one.data_ptr(), 1, d, _stream())
        assert torch.equal(one[0], dst[1])
        gi, go = src.shape[1] + 6, dst.shape[1] + 10
        wide = torch.zeros(batch, gi, dtype=src.dtype, device="cuda")
        wide[:, : src.shape[1]] = src
        out = torch.full((batch, go), 5, dtype=dst.dtype, device="cuda")
        L.check(L.lib().sfft_execute_strided(plan.handle, ctypes.c_void_p(wide.data_ptr()), gi,
                                             ctypes.c_void_p(out.data_ptr()), go, batch, d,
                                             ctypes.c_void_p(_stream())))
        torch.cuda.synchronize()
        assert torch.equal(out[:, : dst.shape[1]].contiguous(), dst)
        assert bool((out[:, dst.shape[1]:] == 5).all())

"""Chirp-z transforms that run in one launch or three: the smallest and the
largest length of every compiled convolution length (three launches: of every
column length, at the shortest and at longer rows, and the ends of the range),
all kinds and both directions, batches that leave part of a block idle, strided
and in place.

Expected values: the DFT in 64 bits (numpy).  Tolerances are those of every
length: rel L2 1e-6 in FP32, and in FP64 1e-13 for the complex kind; the real
kinds add a twiddled pair sum on top, for which 2e-13 is taken."""
import ctypes

import numpy as np
import pytest
import torch

import fft_amd
from fft_amd import _lib as L
from fft_amd import synth
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

M32 = [64, 128, 192, 256, 320, 384, 448, 512, 640, 768, 1024, 1536, 2048, 3072, 4096, 5120, 6144,
       8192, 9216, 10240, 16384]
M64 = [64, 128, 192, 256, 320, 384, 512, 640, 768, 1024, 1280, 1536, 2048, 2560, 3072, 3840, 4096,
       5120, 6144, 8192]


def _direct(n):
    for p in (2, 3, 5, 7, 11, 13):
        while n % p == 0:
            n //= p
    return n == 1


def _edges(ms):
    """(M, n): the smallest and the largest chirp-z length n of each M."""
    out, low = [], 17
    for m in ms:
        own = [n for n in range(low, (m + 1) // 2 + 1) if not _direct(n)]
        out += [(m, n) for n in sorted({own[0], own[-1]})]
        low = (m + 1) // 2 + 1
    return out


N1 = [128, 144, 160, 176, 192, 208, 240]
# (M, n) of plans of three launches: the largest chirp-z n of N1 x 128 and of
# N1 x 1024 (F64: 64 and 512), the first one past one launch, one of each row
# length of eight elements a thread, and the ends
S32 = _edges([16384] + [c * 128 for c in N1[1:]])[2:] + \
    [(c * 1024, _edges([c * 1024])[-1][1]) for c in N1[::2]] + \
    [(m, _edges([m])[-1][1]) for m in (208 * 2048, 208 * 4096)] + \
    [(240 << 14, 1966080 - 1)]
S64 = _edges([8192] + [c * 64 for c in N1[1:]])[2:] + \
    [(c * 512, _edges([c * 512])[-1][1]) for c in N1[1::2]] + \
    [(m, _edges([m])[-1][1]) for m in (208 * 1024, 208 * 2048)] + [(240 << 13, 983040 - 1)]


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _spectrum(x, n, shifted):
    turn = np.exp(-1j * np.pi * np.arange(n) / n) if shifted else 1.0
    y = np.fft.fft(x * turn)
    out = y[..., : n // 2].copy()
    if not shifted:
        out[..., 0] = y[..., 0].real + 1j * y[..., n // 2].real
    return out


@pytest.mark.parametrize("prec,m,n", [(L.F32, m, n) for m, n in _edges(M32) + S32] +
                         [(L.F64, m, n) for m, n in _edges(M64) + S64])
def test_edges_of_each_convolution_length(prec, m, n):
    cdt = np.complex64 if prec == L.F32 else np.complex128
    rdt = np.float32 if prec == L.F32 else np.float64
    tol, tol_real = (1e-6, 1e-6) if prec == L.F32 else (1e-13, 2e-13)
    batch = 37 if n < 400 else 3  # not a multiple of the transforms per block
    plan = fft_amd.Plan(n, L.C2C, prec)
    assert plan.info()["chirp_length"] == m
    x = synth.complex_uniform(n, (batch, n), cdt)
    for d in (0, 1):
        xd = torch.from_numpy(x).cuda()
        yd = torch.empty_like(xd)
        plan.execute_ptr(xd.data_ptr(), yd.data_ptr(), batch, d, _stream())
        x64 = x.astype(np.complex128)
        want = np.fft.ifft(x64, norm="forward") if d else np.fft.fft(x64)
        assert np.array_equal(xd.cpu().numpy(), x), "input was changed"
        assert po.rel_l2(yd.cpu().numpy(), want) <= tol, (n, d)
        plan.execute_ptr(xd.data_ptr(), xd.data_ptr(), batch, d, _stream())
        assert torch.equal(xd, yd), "in place differs"
    for kind in (L.R2C, L.R2C_HALFSHIFT):
        rp = fft_amd.Plan(2 * n, kind, prec)
        r = synth.real_uniform(n, (batch, 2 * n), rdt)
        rd = torch.from_numpy(r).cuda()
        sd = torch.empty(batch, n, dtype=torch.complex64 if prec == L.F32 else torch.complex128,
                         device="cuda")
        back = torch.empty_like(rd)
        rp.execute_ptr(rd.data_ptr(), sd.data_ptr(), batch, 0, _stream())
        rp.execute_ptr(sd.data_ptr(), back.data_ptr(), batch, 1, _stream())
        want = _spectrum(r.astype(np.float64), 2 * n, kind == L.R2C_HALFSHIFT)
        assert po.rel_l2(sd.cpu().numpy(), want) <= tol_real, (n, kind)
        assert po.rel_l2(back.cpu().numpy(), 2 * n * r.astype(np.float64)) <= 2 * tol_real
        # the inverse on spectra of its own, against the oracle's pair pre-process
        s = synth.complex_uniform(n + 1, (1, n), cdt)
        st = torch.from_numpy(s).cuda()
        rp.execute_ptr(st.data_ptr(), back.data_ptr(), 1, 1, _stream())
        mid = fft_amd.Plan(2 * n, kind, L.F64)
        s64 = torch.from_numpy(s.astype(np.complex128)).cuda()
        b64 = torch.empty(1, 2 * n, dtype=torch.float64, device="cuda")
        mid.execute_ptr(s64.data_ptr(), b64.data_ptr(), 1, 1, _stream())
        assert po.rel_l2(back[0].cpu().numpy(), b64[0].cpu().numpy()) <= tol_real


def test_launch_sequence_past_three_launches():
    """The first length whose convolution has no compiled split."""
    n = 1966080 + 1
    plan = fft_amd.Plan(n, L.C2C, L.F32)
    assert plan.info()["chirp_length"] > 240 << 14
    x = synth.complex_uniform(n, (1, n), np.complex64)
    xd = torch.from_numpy(x).cuda()
    yd = torch.empty_like(xd)
    plan.execute_ptr(xd.data_ptr(), yd.data_ptr(), 1, 0, _stream())
    assert po.rel_l2(yd.cpu().numpy(), np.fft.fft(x.astype(np.complex128))) <= 1e-6


@pytest.mark.parametrize("n", [17, 1009, 8191, 50021])
def test_strided_and_workspace_rules(n):
    """Explicit distances leave the gaps alone, and the workspace a caller is
    asked for is still 2 rows of the smallest 2^a 3^b 5^c length >= 2 n - 1."""
    plan = fft_amd.Plan(n, L.C2C, L.F32)
    x = torch.from_numpy(synth.complex_uniform(n, (5, n), np.complex64)).cuda()
    y = torch.empty_like(x)
    plan.execute_ptr(x.data_ptr(), y.data_ptr(), 5, 0, _stream())
    xs = torch.zeros(5, n + 3, dtype=torch.complex64, device="cuda")
    xs[:, :n] = x
    ys = torch.full((5, n + 11), 7 + 7j, dtype=torch.complex64, device="cuda")
    L.check(L.lib().sfft_execute_strided(plan.handle, ctypes.c_void_p(xs.data_ptr()), n + 3,
                                         ctypes.c_void_p(ys.data_ptr()), n + 11, 5, 0,
                                         ctypes.c_void_p(_stream())))
    torch.cuda.synchronize()
    assert torch.equal(ys[:, :n].contiguous(), y)
    assert bool((ys[:, n:] == 7 + 7j).all())
    row = plan.workspace_size(1, False) // 16
    assert row >= 2 * n - 1 and set(_factors(row)) <= {2, 3, 5}
    assert plan.workspace_size(6, False) == 6 * 16 * row


def _factors(n):
    p, out = 2, []
    while n > 1:
        while n % p == 0:
            out.append(p)
            n //= p
        p += 1
    return out

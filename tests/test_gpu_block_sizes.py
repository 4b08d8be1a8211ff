"""Single passes whose blocks hold fewer transforms than 256 threads would, or
run the persistent schedule: batches that end before, at and after a block, and
past the resident blocks, alone and in place; the bits of the runtime-planned
pass where it has the same radices, and the definition (numpy) at the last
transform."""
import numpy as np
import pytest
import torch

import fft_amd
from fft_amd import _lib as L

pytestmark = pytest.mark.gpu

TOL = {L.F32: 1e-6, L.F64: 1e-12, L.F32X: 1e-7}
REAL = (L.R2C, L.R2C_HALFSHIFT)
CASES = (
    [(L.C2C, L.F32, n) for n in (162, 256, 512, 648, 800, 1600, 2048, 7680)]
    + [(L.C2C, L.F64, n) for n in (75, 90, 125, 162, 200, 225, 256, 288, 375, 384, 400, 405, 480,
                                   500, 512, 640, 720, 810, 960, 972, 1024, 1080, 1125, 1200,
                                   1250, 1728, 1920, 2048, 2160, 2187, 2500, 3000, 3125, 3240,
                                   3375, 3600, 3840, 4320)]
    + [(L.C2C, L.F32X, 1280)]
    + [(k, L.F32, 2 * h) for k in REAL for h in (512, 800, 1296, 2187, 2400, 2560, 6480)]
    + [(k, L.F64, 2 * h) for k in REAL for h in (300, 320, 1280, 2048)])


def _bits(t):
    return t.contiguous().view(torch.uint8).flatten()


def _want(v, kind, n, d):
    """The definition in FP64 (numpy) of one transform."""
    if kind == L.C2C:
        return np.fft.ifft(v, norm="forward") if d else np.fft.fft(v)
    if kind == L.R2C:
        full = np.fft.rfft(v)
        out = full[:n // 2].copy()
        out[0] = full[0].real + 1j * full[n // 2].real
        return out
    return np.fft.fft(v * np.exp(-1j * np.pi / n * np.arange(n)))[:n // 2]


@pytest.mark.parametrize("kind,prec,n", CASES)
def test_blocks(kind, prec, n):
    f64 = prec == L.F64
    cdt, rdt = (torch.complex128, torch.float64) if f64 else (torch.complex64, torch.float32)
    cn = n if kind == L.C2C else n // 2
    plan = fft_amd.Plan(n, kind, prec)
    plain = fft_amd.Plan(n, kind, prec, variant=-2)
    assert plan.info()["passes"] == 1
    same = plan.info()["radices"] == plain.info()["radices"]
    stream = torch.cuda.current_stream().cuda_stream
    top = 2100 if cn < 1000 else 1100  # more groups than blocks stay resident
    batches = (1, 2, 3, 5, 13, 33, top)
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(top, n, dtype=cdt if kind == L.C2C else rdt, device="cuda", generator=g)
    for d in (0, 1):
        real_out = kind != L.C2C and d == 1
        y = torch.empty(top, n if real_out else cn, dtype=rdt if real_out else cdt, device="cuda")
        plan.execute_ptr(x.data_ptr(), y.data_ptr(), top, d, stream)
        if same:
            ref = torch.empty_like(y)
            plain.execute_ptr(x.data_ptr(), ref.data_ptr(), top, d, stream)
            assert torch.equal(_bits(y), _bits(ref))
        for b in batches:
            part = torch.full((b + 1, y.shape[1]), 7, dtype=y.dtype, device="cuda")
            plan.execute_ptr(x[top - b:].data_ptr(), part.data_ptr(), b, d, stream)
            assert torch.equal(_bits(part[:b]), _bits(y[top - b:])), (b, d)
            assert bool((part[b] == 7).all()), (b, d)
        if kind == L.C2C:
            buf = x.clone()
            plan.execute_ptr(buf.data_ptr(), buf.data_ptr(), top, d, stream)
            assert torch.equal(_bits(buf), _bits(y))
        got = y[top - 1].cpu().numpy().astype(np.float64 if real_out else np.complex128)
        if not real_out:
            v = x[top - 1].cpu().numpy().astype(np.complex128 if kind == L.C2C else np.float64)
            want = _want(v, kind, n, d)
        else:
            want = n * last
        err = np.linalg.norm(got - want) / np.linalg.norm(want)
        # (the inverse of the kept spectra adds the forward error to its own)
        assert err <= (2 if real_out else 1) * TOL[prec], (err, d)
        if kind != L.C2C and d == 0:
            last = x[top - 1].cpu().numpy().astype(np.float64)
            x = y  # the spectra are the inverse's input

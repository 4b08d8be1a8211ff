"""Compiled column passes of two-pass plans at their dispatch edges: wide tiles
(taken once every CU has one), the column lengths 576 to 1000, FP64 and F32X.
A transform has the same bits alone, below and above the wide tiles' threshold,
in place and with gaps; it matches the runtime-planned passes of the same split
and the oracle (signalsmith-fft.h:295-315, :374-386).

Tolerance (oracle): rel L2 1e-6 in FP32, 1e-7 in F32X (the rounding of the
result), 1e-12 in FP64, as for every two-pass length; 16-bit storage twice the
rounding of the ideal result (result and stored intermediate)."""
import ctypes
import math

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


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _input(prec, batch, n):
    if prec in HALF:
        g = torch.Generator(device="cpu").manual_seed(n)
        return torch.randn(batch, n, 2, generator=g).to(HALF[prec]).cuda()
    dt = np.complex128 if prec == L.F64 else np.complex64
    return torch.from_numpy(synth.complex_normal(n, (batch, n), dt)).cuda()


def _c128(t, prec):
    if prec in HALF:
        v = t.float().cpu().numpy().astype(np.float64)
        return v[..., 0] + 1j * v[..., 1]
    return t.cpu().numpy().astype(np.complex128)


def _oracle_ok(x, y, prec, inverse):
    want = po.ifft(_c128(x, prec)) if inverse else po.fft(_c128(x, prec))
    err = po.rel_l2(_c128(y, prec), want)
    if prec in HALF:
        w = torch.from_numpy(np.stack([want.real, want.imag], -1).astype(np.float32))
        tol = 2.0 * po.rel_l2(_c128(w.to(HALF[prec]), prec), want) + 1e-6
    else:
        tol = TOL[prec]
    assert err <= tol, (err, tol)


def _run(plan, x, y, d):
    plan.execute_ptr(x.data_ptr(), y.data_ptr(), x.shape[0], d, _stream())
    torch.cuda.synchronize()
    return y


# (precision, n, transforms below the threshold of a pass, transforms above)
WIDE = [
    (L.F32, 1 << 20, 3, 4),    # 1024 x 1024, 16 columns a tile in both passes
    (L.F32, 1 << 22, 1, 2),    # 4096 (8 columns) x 1024
    (L.F32, 1 << 24, 1, 2),    # 4096 x 4096, two-level four-step table
    (L.F16, 1 << 21, 3, 5),    # 2048 (16 columns) x 1024
    (L.BF16, 1 << 21, 3, 5),
    (L.F16, 1 << 22, 1, 3),    # 4096 (8 columns) x 1024
    (L.F32X, 1 << 20, 3, 5),   # 4096 (4 columns) x 256
]


@pytest.mark.parametrize("prec,n,lo,hi", WIDE)
def test_wide_tiles(prec, n, lo, hi):
    plan = fft_amd.Plan(n, L.C2C, prec)
    plain = fft_amd.Plan(n, L.C2C, prec, variant=-2)
    x = _input(prec, hi, n)
    for d in (0, 1):
        y = _run(plan, x, torch.empty_like(x), d)
        few = _run(plan, x[:lo].contiguous(), torch.empty_like(x[:lo]), d)
        assert torch.equal(few, y[:lo])
        last = _run(plan, x[hi - 1:].clone(), torch.empty_like(x[:1]), d)
        assert torch.equal(last[0], y[hi - 1])
        ref = _run(plain, x, torch.empty_like(x), d)
        if plan.info()["radices"] == plain.info()["radices"]:
            assert torch.equal(ref, y)
        _oracle_ok(x[hi - 1], y[hi - 1], prec, d)
        buf = x.clone()
        assert torch.equal(_run(plan, buf, buf, d), y)
        gap = torch.zeros((hi, n + 12) + x.shape[2:], dtype=x.dtype, device="cuda")
        gap[:, :n] = x
        out = torch.full((hi, n + 6) + x.shape[2:], 5, dtype=x.dtype, device="cuda")
        L.check(L.lib().sfft_execute_strided(
            plan.handle, ctypes.c_void_p(gap.data_ptr()), n + 12,
            ctypes.c_void_p(out.data_ptr()), n + 6, hi, d, ctypes.c_void_p(_stream())))
        torch.cuda.synchronize()
        assert torch.equal(out[:, :n], y) and bool((out[:, n:] == 5).all())


# both passes of each length: 45 columns leave part of the last tile empty
LARGE = [576, 600, 640, 648, 675, 720, 750, 768, 800, 810, 864, 900, 960, 972, 1000]


@pytest.mark.parametrize("prec", [L.F32, L.F64])
@pytest.mark.parametrize("length", LARGE)
def test_large_columns(length, prec):
    n, batch = 45 * length, 3
    x = _input(prec, batch, n)
    for split in (length, 45):
        plan = fft_amd.Plan(n, L.C2C, prec, split=split)
        plain = fft_amd.Plan(n, L.C2C, prec, split=split, variant=-2)
        assert plan.info()["passes"] == 2
        for d in (0, 1):
            y = _run(plan, x, torch.empty_like(x), d)
            ref = _run(plain, x, torch.empty_like(x), d)
            if plan.info()["radices"] == plain.info()["radices"]:
                assert torch.equal(y, ref)
            _oracle_ok(x[2], y[2], prec, d)
            buf = x.clone()
            assert torch.equal(_run(plan, buf, buf, d), y)
            one = _run(plan, x[1:2].clone(), torch.empty_like(x[:1]), d)
            assert torch.equal(one[0], y[1])


# F32X: one pass (compiled singles) and two
@pytest.mark.parametrize("n", [256, 512, 1024, 2048, 4096, 8192, 1 << 15, 1 << 17, 1 << 19])
def test_f32x_compiled(n):
    x = _input(L.F32X, 5, n)
    plan = fft_amd.Plan(n, L.C2C, L.F32X)
    plain = fft_amd.Plan(n, L.C2C, L.F32X, variant=-2)
    for d in (0, 1):
        y = _run(plan, x, torch.empty_like(x), d)
        ref = _run(plain, x, torch.empty_like(x), d)
        # FP64 arithmetic: another factorisation may differ in the last FP32 bit
        assert po.rel_l2(_c128(y, L.F32X), _c128(ref, L.F32X)) <= 1e-7
        _oracle_ok(x[4], y[4], L.F32X, d)
        one = _run(plan, x[3:4].clone(), torch.empty_like(x[:1]), d)
        assert torch.equal(one[0], y[3])


# lengths whose best split is one of two compiled column lengths, and lengths
# without one (factors 7, 11, 13): the plan, the same split asked for, and the
# runtime-planned passes agree
@pytest.mark.parametrize("prec", [L.F32, L.F64])
@pytest.mark.parametrize("n", [262440, 331776, 360000, 500000, 703125, 746496, 1000000,
                               11 * 31250, 13 * 13 * 2048, 7 * 49152])
def test_planned_split(n, prec):
    plan = fft_amd.Plan(n, L.C2C, prec)
    plain = fft_amd.Plan(n, L.C2C, prec, variant=-2)
    x = _input(prec, 2, n)
    assert plan.info()["passes"] == plain.info()["passes"] == 2
    n1 = math.prod(plan.info()["radices"])
    assert n1 == math.prod(plain.info()["radices"])
    for d in (0, 1):
        y = _run(plan, x, torch.empty_like(x), d)
        asked = _run(fft_amd.Plan(n, L.C2C, prec, split=n1), x, torch.empty_like(x), d)
        assert torch.equal(y, asked)
        ref = _run(plain, x, torch.empty_like(x), d)
        assert po.rel_l2(_c128(y, prec), _c128(ref, prec)) <= TOL[prec]
        _oracle_ok(x[1], y[1], prec, d)

"""First column passes of 128, 144 and 625 in two tile widths: launches of less
than a tile per CU (625: per two) take the narrower one.  Batches on both sides of
that line, one transform, and strided: every transform has the bits of the
runtime-planned pass, and matches the oracle (signalsmith-fft.h:295-315,
:446-502)."""
import ctypes

import numpy as np
import pytest
import torch

import fft_amd
from fft_amd import _lib as L
from fft_amd import synth
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

# (complex length, first-pass length, columns of its wide tile, CUs per tile)
CASES = [(128 * 125, 128, 64, 1), (144 * 125, 144, 64, 1), (144 * 243, 144, 64, 1),
         (625 * 125, 625, 16, 2)]


def _lines(n, n1, wide, cus):
    """Largest batch of the narrow tile, and the smallest of the wide one."""
    tiles = torch.cuda.get_device_properties(0).multi_processor_count // cus
    edge = -(-tiles * wide // (n // n1))
    return edge - 1, edge


@pytest.mark.parametrize("kind", [L.C2C, L.R2C])
@pytest.mark.parametrize("n,n1,wide,cus", CASES)
def test_widths_agree(n, n1, wide, cus, kind):
    size = n if kind == L.C2C else 2 * n
    plan = fft_amd.Plan(size, kind, L.F32, split=n1)
    plain = fft_amd.Plan(size, kind, L.F32, split=n1, variant=-2)
    assert plan.info()["radices"] == plain.info()["radices"]
    stream = torch.cuda.current_stream().cuda_stream
    last, first = _lines(n, n1, wide, cus)
    if kind == L.C2C:
        x = torch.from_numpy(synth.complex_normal(n, (first, n), np.complex64)).cuda()
    else:
        x = torch.from_numpy(synth.real_uniform(n, (first, size), np.float32)).cuda()
    ref = torch.empty(first, n, dtype=torch.complex64, device="cuda")
    plain.execute_ptr(x.data_ptr(), ref.data_ptr(), first, 0, stream)
    for batch in (1, last, first):
        y = torch.empty_like(ref[:batch])
        plan.execute_ptr(x.data_ptr(), y.data_ptr(), batch, 0, stream)
        torch.cuda.synchronize()
        assert torch.equal(y, ref[:batch]), batch
    gi, go = size + 6, n + 10
    xs = torch.zeros(3, gi, dtype=x.dtype, device="cuda")
    xs[:, :size] = x[:3]
    ys = torch.full((3, go), 5, dtype=torch.complex64, device="cuda")
    L.check(L.lib().sfft_execute_strided(plan.handle, ctypes.c_void_p(xs.data_ptr()), gi,
                                         ctypes.c_void_p(ys.data_ptr()), go, 3, 0,
                                         ctypes.c_void_p(stream)))
    torch.cuda.synchronize()
    assert torch.equal(ys[:, :n].contiguous(), ref[:3]) and bool((ys[:, n:] == 5).all())
    xh = x[first - 1].cpu().numpy()
    want = po.fft(xh.astype(np.complex128)) if kind == L.C2C else po.real_fft(
        xh.astype(np.float64))
    assert po.rel_l2(ref[first - 1].cpu().numpy(), want) <= 1e-6

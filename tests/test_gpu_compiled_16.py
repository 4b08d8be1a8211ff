"""16-bit storage, single pass: a plan computes what its runtime-planned pass
computes, at every 2^a 3^b 5^c length that one pass holds.  Exceptions by name:
the powers of two 512 and 8192 and six lengths whose compiled kernels have
radices of their own.  Bits at the lengths where the 512-thread blocks of the
16-bit pass lead to other radices than 1024 threads would, batched and strided
(strided calls run the runtime-planned pass)."""
import ctypes

import pytest
import torch

import fft_amd
from fft_amd import _lib as L

pytestmark = pytest.mark.gpu

HALF = {L.F16: torch.float16, L.BF16: torch.bfloat16}
OWN = {512, 8192, 6561, 8100, 11250, 13500, 14400, 15360}
BITS = [4860, 5832, 6480, 6912, 7290, 7776, 8000, 8640, 9000, 9600, 9720, 10000, 10240, 10935,
        11664, 12000, 12150, 12500, 12800, 12960, 13122, 13824, 14580]


def _smooth(lo, hi):
    out = {2 ** a * 3 ** b * 5 ** c for a in range(15) for b in range(9) for c in range(7)}
    return sorted(n for n in out if lo <= n <= hi)


@pytest.mark.parametrize("prec", list(HALF))
def test_radices(prec):
    other = []
    for n in _smooth(64, 16384):
        plan, plain = fft_amd.Plan(n, L.C2C, prec), fft_amd.Plan(n, L.C2C, prec, variant=-2)
        a, b = plan.info(), plain.info()
        if a["passes"] == b["passes"] == 1 and a["radices"] != b["radices"]:
            other.append(n)
    assert set(other) <= OWN, other


@pytest.mark.parametrize("prec", list(HALF))
@pytest.mark.parametrize("n", BITS)
def test_bits(n, prec):
    batch, gap = 5, 8
    stream = torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device="cpu").manual_seed(n)
    x = (torch.randn(batch, n + gap, 2, generator=g) / 64).to(HALF[prec]).cuda()
    xc = x[:, :n].contiguous()
    plan, plain = fft_amd.Plan(n, L.C2C, prec), fft_amd.Plan(n, L.C2C, prec, variant=-2)
    for d in (0, 1):
        y, ref, ys = torch.empty_like(xc), torch.empty_like(xc), torch.full_like(x, 3)
        plan.execute_ptr(xc.data_ptr(), y.data_ptr(), batch, d, stream)
        plain.execute_ptr(xc.data_ptr(), ref.data_ptr(), batch, d, stream)
        L.check(L.lib().sfft_execute_strided(plan.handle, ctypes.c_void_p(x.data_ptr()), n + gap,
                                             ctypes.c_void_p(ys.data_ptr()), n + gap, batch, d,
                                             ctypes.c_void_p(stream)))
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), ref.view(torch.int16))
        assert torch.equal(ys[:, :n].contiguous().view(torch.int16), y.view(torch.int16))
        assert bool((ys[:, n:] == 3).all())

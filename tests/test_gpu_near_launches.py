"""Two-pass launches whose data fits the L2 caches number their column tiles
XCD by XCD: the same bits as one transform at a time, on either side of the
rule's edges (8 and 16 transforms, 14 and 34 MB) and with tile counts that 8
does not divide, and the definition (numpy) at the last transform."""
import numpy as np
import pytest
import torch

import fft_amd
from fft_amd import _lib as L

pytestmark = pytest.mark.gpu

TOL = {L.F32: 1e-6, L.F64: 1e-12}
MB = 1 << 20
# (kind, precision, length, batches): 17496 = 108 x 162, 27000 = 150 x 180,
# 32768 = 128 x 256, 40960 reals = 128 x 160
CASES = [(L.C2C, L.F32, 27000, (7, 8, 15, 16, 17, 65, 66, 165, 166)),
         (L.C2C, L.F64, 17496, (7, 8, 16, 17, 52, 53, 127, 128)),
         (L.C2C, L.F64, 32768, (8, 17, 67, 69)),
         (L.R2C, L.F32, 40960, (8, 17, 89, 217, 218)),
         (L.R2C_HALFSHIFT, L.F64, 40960, (8, 17, 44, 45, 109))]


@pytest.mark.parametrize("kind,prec,n,batches", CASES)
def test_bits(kind, prec, n, batches):
    cdt = torch.complex128 if prec == L.F64 else torch.complex64
    rdt = torch.float64 if prec == L.F64 else torch.float32
    cn = n if kind == L.C2C else n // 2
    # the batches lie on both sides of 34 MB
    assert any(b * cn * cdt.itemsize > 34 * MB for b in batches)
    assert any(b * cn * cdt.itemsize <= 34 * MB for b in batches)
    plan = fft_amd.Plan(n, kind, prec)
    assert plan.info()["passes"] == 2
    stream = torch.cuda.current_stream().cuda_stream
    top = max(batches)
    for d in (0, 1):
        g = torch.Generator(device="cuda").manual_seed(n + d)
        real_in, real_out = kind != L.C2C and d == 0, kind != L.C2C and d == 1
        x = torch.randn(top, n if real_in else cn, dtype=rdt if real_in else cdt, device="cuda",
                        generator=g)
        y = torch.empty(top, n if real_out else cn, dtype=rdt if real_out else cdt, device="cuda")
        one = torch.empty_like(y)
        for i in range(top):
            plan.execute_ptr(x[i].data_ptr(), one[i].data_ptr(), 1, d, stream)
        for b in batches:
            y.zero_()
            plan.execute_ptr(x.data_ptr(), y.data_ptr(), b, d, stream)
            assert torch.equal(y[:b], one[:b]), (d, b)
            assert not bool(torch.count_nonzero(y[b:])), (d, b)
            z = x.clone()  # in place, through the workspace
            if not (real_in or real_out):
                plan.execute_ptr(z.data_ptr(), z.data_ptr(), b, d, stream)
                assert torch.equal(z[:b], one[:b]), (d, b)
        if kind == L.C2C:
            v = x[top - 1].cpu().numpy().astype(np.complex128)
            want = np.fft.ifft(v, norm="forward") if d else np.fft.fft(v)
            got = one[top - 1].cpu().numpy().astype(np.complex128)
            assert np.linalg.norm(got - want) <= TOL[prec] * np.linalg.norm(want)

"""Workspace of chirp-z lengths: the library reserves what a call uses, none in
one launch and M values a transform in three, for its own callers (the
no-allocation entry point, uneven batches, the server).  What the C ABI asks a
caller for is unchanged (sfft_plan_workspace_size: two rows a transform)."""
import ctypes

import pytest
import torch

import fft_amd
from fft_amd import _lib as L
from fft_amd import synth
from fft_amd.serving import Server

pytestmark = pytest.mark.gpu


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _input(n, batch):
    return torch.from_numpy(synth.complex_uniform(n, (batch, n), "complex64")).cuda()


# 1009: one launch; 100003: three, M = 208 x 1024 values of 8 bytes a transform
@pytest.mark.parametrize("n,batch", [(1009, 4096), (100003, 39)])
def test_noalloc_takes_what_the_call_uses(n, batch):
    plan = fft_amd.Plan(n)
    assert plan.workspace_size(batch, False) > 64 << 20  # more than the array holds
    x = _input(n, batch)
    for d in (0, 1):
        y, want = torch.empty_like(x), torch.empty_like(x)
        rc = L.lib().sfft_execute_noalloc(plan.handle, ctypes.c_void_p(x.data_ptr()),
                                          ctypes.c_void_p(y.data_ptr()), batch, d,
                                          ctypes.c_void_p(_stream()))
        assert rc == L.SFFT_OK, L.lib().sfft_last_error()
        plan.execute_ptr(x.data_ptr(), want.data_ptr(), batch, d, _stream())
        torch.cuda.synchronize()
        assert torch.equal(y, want)


def test_noalloc_refuses_more():
    n, batch = 100003, 40  # 40 x 212992 x 8 bytes > 64 MiB
    plan = fft_amd.Plan(n)
    x = torch.zeros(batch, n, dtype=torch.complex64, device="cuda")
    y = torch.empty_like(x)
    rc = L.lib().sfft_execute_noalloc(plan.handle, ctypes.c_void_p(x.data_ptr()),
                                      ctypes.c_void_p(y.data_ptr()), batch, 0,
                                      ctypes.c_void_p(_stream()))
    assert rc == L.SFFT_ERR_BUDGET


@pytest.mark.parametrize("n", [1009, 100003])
def test_callers_workspace_rule(n):
    plan = fft_amd.Plan(n)
    x = _input(n, 3)
    y = torch.empty_like(x)
    ws = torch.empty(plan.workspace_size(3, False), dtype=torch.uint8, device="cuda")

    def call(w, size):
        return L.lib().sfft_execute_workspace(
            plan.handle, ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(y.data_ptr()), 3, 0,
            ctypes.c_void_p(w), size, ctypes.c_void_p(_stream()))

    assert call(None, 0) == L.SFFT_ERR_INVALID_ARG
    assert call(ws.data_ptr(), ws.numel() - 1) == L.SFFT_ERR_INVALID_ARG
    assert call(x.data_ptr(), ws.numel()) == L.SFFT_ERR_ALIASING
    assert call(ws.data_ptr(), ws.numel()) == L.SFFT_OK
    want = torch.empty_like(x)
    plan.execute_ptr(x.data_ptr(), want.data_ptr(), 3, 0, _stream())
    torch.cuda.synchronize()
    assert torch.equal(y, want)


def _batch(items):
    arr = (L.BatchItem * len(items))()
    off = 0
    for i, (n, count) in enumerate(items):
        arr[i] = L.BatchItem(n, L.C2C, i % 2, count, off, off)
        off += n * count * 8
    h = ctypes.c_void_p()
    L.check(L.lib().sfft_batch_create(ctypes.byref(h), arr, len(items), L.F32))
    return h, off // 8


def test_uneven_batch_reserves_nothing_for_one_launch():
    fft_amd.Plan(1009)
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    h, _ = _batch([(1009, 20000)])  # two rows of 2025 values a transform: 648 MB
    used = free0 - torch.cuda.mem_get_info()[0]
    L.lib().sfft_batch_destroy(h)
    assert used < 100 << 20, used


def test_uneven_batch_of_both():
    items = [(1009, 7), (100003, 3), (4096, 2), (5003, 4)]
    h, total = _batch(items)
    x = _input(total, 1)[0]
    y = torch.empty_like(x)
    for _ in range(2):  # captured, then replayed
        L.check(L.lib().sfft_batch_execute(h, ctypes.c_void_p(x.data_ptr()),
                                           ctypes.c_void_p(y.data_ptr()),
                                           ctypes.c_void_p(_stream())))
        torch.cuda.synchronize()
        off = 0
        for i, (n, count) in enumerate(items):
            part = x[off:off + n * count].clone()
            want = torch.empty_like(part)
            fft_amd.Plan(n).execute_ptr(part.data_ptr(), want.data_ptr(), count, i % 2, _stream())
            torch.cuda.synchronize()
            assert torch.equal(y[off:off + n * count], want), n
            off += n * count
        y.zero_()
    L.lib().sfft_batch_destroy(h)


def test_server_budget_is_what_the_request_uses():
    """Input and output of 4096 transforms of 1009 are 66 MB, and two rows a
    transform would be another 133."""
    n, batch = 1009, 4096
    with Server(budget_bytes=80 << 20) as srv:
        srv.submit(1, n, L.C2C, 0, batch, seed=3, retain=True)
        srv.drain()
        rec = srv.poll()
        assert rec["status"][0] == L.SFFT_OK
        got = torch.from_numpy(srv.fetch(1, n * batch * 8).copy()).view(torch.complex64)
        srv.release(1)
    x = torch.empty(batch, n, dtype=torch.complex64, device="cuda")
    fft_amd.fill(x, seed=3)
    y = torch.empty_like(x)
    fft_amd.Plan(n).execute_ptr(x.data_ptr(), y.data_ptr(), batch, 0, _stream())
    assert torch.equal(got.view(batch, n), y.cpu())

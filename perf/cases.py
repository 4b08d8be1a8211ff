"""The workloads by which this engine's speed is measured.

Each case is one pass through the public entry points (FFT, RealFFT,
ModifiedRealFFT, Plan, UnevenBatch) over data that is resident in HBM.  A
case is a dict of plain values:

    kind   "c2c", "real", "shifted" (ModifiedRealFFT), "frames" (the mixed
           batch of bench.py) or "uneven" (many sizes in one launch)
    prec   "f32", "f64", or the storage variants "f32x", "f16", "bf16"
    n      transform length (reals for the real kinds)
    batch  transforms per call ("uneven": transforms in the batch)

Every pass runs both directions: forward on the input, and the unnormalised
inverse on the spectra that the forward call wrote.  The storage variants
take a second input for the inverse instead, because N x overflows 16 bits.
"""
import math

import numpy as np
import torch

import fft_amd
from fft_amd import _lib as L

# bench.py's step: complex sizes of one batch each, and real frames
FRAME_SIZES = (1920, 3000, 16384)
FRAME_REAL = 2048

CPLX = {"f32": torch.complex64, "f64": torch.complex128}
REAL = {"f32": torch.float32, "f64": torch.float64}
STORED = {"f32x": (torch.float32, L.F32X), "f16": (torch.float16, L.F16),
          "bf16": (torch.bfloat16, L.BF16)}


def listed():
    return [
        # one transform at a time, as a caller of the reference's fft()/ifft()
        # does it: latency and launches
        {"name": "single_4096", "kind": "c2c", "prec": "f32", "n": 4096, "batch": 1},
        # bench.py's step: audio-sized and power-of-two blocks, 8192 of each,
        # and 16384 real frames; the largest case
        {"name": "frames_8192", "kind": "frames", "prec": "f32", "n": 16384, "batch": 8192},
        # a queue of requests of every fast size up to 65536, both directions
        {"name": "uneven_20000", "kind": "uneven", "prec": "f32", "n": 65536, "batch": 20000},
        # long signals, and the same size in IEEE half storage
        {"name": "long_2p20", "kind": "c2c", "prec": "f32", "n": 1 << 20, "batch": 16},
        {"name": "long_2p20_f16", "kind": "c2c", "prec": "f16", "n": 1 << 20, "batch": 16},
        # one very long signal
        {"name": "long_2p24", "kind": "c2c", "prec": "f32", "n": 1 << 24, "batch": 1},
        # FFT<double>, the type the reference publishes its figures for
        {"name": "f64_65536", "kind": "c2c", "prec": "f64", "n": 65536, "batch": 256},
        # a batch just above what one workgroup holds in LDS
        {"name": "c2c_32768", "kind": "c2c", "prec": "f32", "n": 32768, "batch": 1024},
        # one second of 96 kHz audio per real transform
        {"name": "real_96000", "kind": "real", "prec": "f32", "n": 96000, "batch": 512},
        # ModifiedRealFFT frames (bins at k + 1/2), an ordinary block size
        {"name": "shifted_4096", "kind": "shifted", "prec": "f32", "n": 4096, "batch": 2048},
        # lengths with large prime factors, which the reference takes as well
        {"name": "prime_1009", "kind": "c2c", "prec": "f32", "n": 1009, "batch": 4096},
        {"name": "prime_100003", "kind": "c2c", "prec": "f32", "n": 100003, "batch": 64},
    ]


def _smooth(lo, hi):
    """All 2^a 3^b 5^c in [lo, hi]."""
    out = []
    p2 = 1
    while p2 <= hi:
        p3 = p2
        while p3 <= hi:
            p5 = p3
            while p5 <= hi:
                if p5 >= lo:
                    out.append(p5)
                p5 *= 5
            p3 *= 3
        p2 *= 2
    return sorted(out)


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["c2c", "c2c", "c2c", "c2c", "real", "real", "shifted", "uneven"])
    if kind == "uneven":
        return {"kind": kind, "prec": "f32", "n": 65536,
                "batch": int(_log_uniform(rng, 500, 10000))}
    prec = rng.choice(["f32", "f32", "f32", "f64"])
    if kind == "c2c" and rng.random() < 0.25:
        prec = rng.choice(["f32x", "f16", "bf16"])
    if prec not in STORED and rng.random() < 0.3:
        # any length; almost all of these have a large prime factor
        n = int(_log_uniform(rng, 64, 200000)) | 1
    else:
        n = rng.choice(_smooth(64, 1 << 20))
    if kind != "c2c":
        n *= 2
    # 64 KiB to 512 MiB of input per call
    size = {"f64": 16, "f16": 4, "bf16": 4}.get(prec, 8) * n // (1 if kind == "c2c" else 2)
    batch = max(1, int(_log_uniform(rng, 1 << 16, 1 << 29)) // size)
    return {"kind": kind, "prec": prec, "n": n, "batch": batch}


def _queue(count, hi):
    """Sizes (log-uniform over the fast sizes in [64, hi]) and directions of
    an uneven batch: the same for every seed, as a plan is."""
    fast = np.array(_smooth(64, hi))
    r = np.random.RandomState(count % 65521 + 3)
    logn = r.uniform(math.log(64), math.log(hi), count)
    edges = (np.log(fast[1:]) + np.log(fast[:-1])) / 2
    return fast[np.searchsorted(edges, logn)], r.randint(0, 2, count)


def _inputs(case, seed):
    """The input tensors, on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed * 1000003 + 17)

    def randn(*shape, dtype=torch.float32):
        return torch.randn(*shape, dtype=dtype, device="cuda", generator=g)

    kind, prec, n, batch = (case[k] for k in ("kind", "prec", "n", "batch"))
    if kind == "uneven":
        total = int(_queue(batch, n)[0].sum())
        return [torch.rand(total, 2, device="cuda", generator=g).mul_(2).sub_(1)]
    if kind == "frames":
        xs = [randn(batch, m, dtype=torch.complex64) for m in FRAME_SIZES]
        return xs + [randn(2 * batch, FRAME_REAL)]
    if prec in STORED:
        return [randn(batch, n, 2).to(STORED[prec][0]) for _ in range(2)]
    if kind == "c2c":
        return [randn(batch, n, dtype=CPLX[prec])]
    return [randn(batch, n, dtype=REAL[prec])]


def prepare(case, seed):
    kind, prec, n, batch = (case[k] for k in ("kind", "prec", "n", "batch"))
    xs = _inputs(case, seed)
    state = {"kind": kind, "batch": batch}
    if kind == "uneven":
        sizes, dirs = _queue(batch, n)
        state["queue"] = fft_amd.UnevenBatch([int(s) for s in sizes], [int(d) for d in dirs])
        state["x"] = xs[0]
        state["y"] = torch.empty_like(xs[0])
        return state
    if prec in STORED:
        state["kind"] = "stored"
        state["plan"] = fft_amd.Plan(n, L.C2C, STORED[prec][1])
        state["pairs"] = [(x, torch.empty_like(x)) for x in xs]
        return state
    if kind == "frames":
        calls = [(fft_amd.FFT(m), x) for m, x in zip(FRAME_SIZES, xs)]
        calls.append((fft_amd.RealFFT(FRAME_REAL), xs[-1]))
    elif kind == "c2c":
        calls = [(fft_amd.FFT(n, dtype=CPLX[prec]), xs[0])]
    elif kind == "real":
        calls = [(fft_amd.RealFFT(n, dtype=REAL[prec]), xs[0])]
    else:
        calls = [(fft_amd.ModifiedRealFFT(n, dtype=REAL[prec]), xs[0])]
    state["calls"] = []
    for f, x in calls:
        if x.is_complex():
            y = torch.empty_like(x)
        else:
            cplx = torch.complex64 if x.dtype == torch.float32 else torch.complex128
            y = torch.empty(x.shape[0], x.shape[1] // 2, dtype=cplx, device="cuda")
        state["calls"].append((f, x, y, torch.empty_like(x)))
    return state


def run(state):
    if state["kind"] == "uneven":
        return state["queue"].execute(state["x"], state["y"])
    if state["kind"] == "stored":
        stream = torch.cuda.current_stream().cuda_stream
        for direction, (x, y) in zip((L.FORWARD, L.INVERSE), state["pairs"]):
            state["plan"].execute_ptr(x.data_ptr(), y.data_ptr(), state["batch"], direction,
                                      stream)
        return [y for _, y in state["pairs"]]
    out = []
    for f, x, y, z in state["calls"]:
        f.fft(x, y)
        f.ifft(y, z)
        out += [y, z]
    return out


def work(case):
    kind, prec, n, batch = (case[k] for k in ("kind", "prec", "n", "batch"))
    if kind == "uneven":
        sizes = _queue(batch, n)[0].astype(np.float64)
        return {"bytes": 16 * float(sizes.sum()),
                "flops": float((5 * sizes * np.log2(sizes)).sum())}
    if kind == "frames":
        parts = [(16 * m, 5 * m * math.log2(m), batch) for m in FRAME_SIZES]
        parts.append((8 * FRAME_REAL, 2.5 * FRAME_REAL * math.log2(FRAME_REAL), 2 * batch))
    else:
        value = {"f64": 16, "f16": 4, "bf16": 4}.get(prec, 8)
        m = n if kind == "c2c" else n // 2
        parts = [(2 * value * m, 5 * m * math.log2(n), batch)]
    return {"bytes": 2.0 * sum(b * c for b, _, c in parts),
            "flops": 2.0 * sum(f * c for _, f, c in parts)}


def exact(case, seed):
    """The same results in 64 bits, from torch's own FFT on the host."""
    kind, prec, n, batch = (case[k] for k in ("kind", "prec", "n", "batch"))
    xs = [x.cpu() for x in _inputs(case, seed)]
    if kind == "uneven":
        sizes, dirs = _queue(batch, n)
        x = torch.view_as_complex(xs[0].double())
        y = torch.empty_like(x)
        ends = np.cumsum(sizes)
        for m in np.unique(sizes):
            for d in (0, 1):
                at = torch.from_numpy(ends[(sizes == m) & (dirs == d)] - m)
                if not len(at):
                    continue
                rows = at[:, None] + torch.arange(int(m))[None, :]
                part = x[rows]
                y[rows] = torch.fft.ifft(part, norm="forward") if d else torch.fft.fft(part)
        return torch.view_as_real(y)
    if prec in STORED:
        x, w = (torch.view_as_complex(v.double()) for v in xs)
        return [torch.view_as_real(torch.fft.fft(x)),
                torch.view_as_real(torch.fft.ifft(w, norm="forward"))]
    out = []
    for x in xs:
        if x.is_complex():
            x = x.to(torch.complex128)
            out += [torch.fft.fft(x), x.shape[-1] * x]
            continue
        x = x.double()
        m = x.shape[-1]
        if kind == "shifted":
            # bins at k + 1/2: the spectrum of x e^{-i pi t / N}
            turn = torch.polar(torch.ones(m, dtype=torch.float64),
                               -math.pi / m * torch.arange(m, dtype=torch.float64))
            y = torch.fft.fft(x * turn)[..., :m // 2]
        else:
            full = torch.fft.rfft(x)
            y = full[..., :m // 2].clone()
            y[..., 0] = torch.complex(full[..., 0].real, full[..., m // 2].real)
        out += [y, m * x]
    return out

"""The transforms that a program asks of this library, as cases that can be timed and checked.

Each case is a call (or a short run of calls) of the public Python API on buffers that live on
the GPU, with inputs of zero mean and unit variance.  Kinds:

  vector  fft, then ifft, of one short vector: a call's latency
  rows    a batch of equal smooth lengths in one call (direct lines and four-step lengths)
  conv    a batch of rows whose length is prime or has a large prime factor (Rader, Bluestein)
  uneven  one plan over many transforms of different lengths
  served  a burst of requests of mixed lengths through the continuous-batching server
  real    rfft of real rows, then irfft of the spectra
  nd      a multi-dimensional transform of one array
  half    a batch of ComplexF16 rows
"""
import math
import os
import sys
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "catabrafft.jl_amd"))
import catabrafft as C  # noqa: E402

CALLS = {"fft": C.fft, "ifft": C.ifft, "bfft": C.bfft}


def listed():
    return [
        # one vector there and back, as a caller that transforms signal by signal does
        {"name": "vector 1024 F64", "kind": "vector", "n": 1024, "dtype": "complex128"},
        # the benchmark's short rows: a mixed-radix length, in both precisions and directions
        {"name": "rows 2520 x 4096 F32", "kind": "rows", "n": 2520, "batch": 4096,
         "dtype": "complex64", "call": "fft"},
        {"name": "rows 2520 x 4096 F64", "kind": "rows", "n": 2520, "batch": 4096,
         "dtype": "complex128", "call": "ifft"},
        # the benchmark's long rows, the largest arrays here
        {"name": "rows 2^20 x 64 F32", "kind": "rows", "n": 1 << 20, "batch": 64,
         "dtype": "complex64", "call": "fft"},
        {"name": "rows 2^20 x 64 F64", "kind": "rows", "n": 1 << 20, "batch": 64,
         "dtype": "complex128", "call": "bfft"},
        # prime lengths of the benchmark's Rader section: one whose convolution fits a workgroup,
        # and the longest
        {"name": "prime 4099 x 4093 F32", "kind": "conv", "n": 4099, "batch": 4093,
         "dtype": "complex64", "call": "fft"},
        {"name": "prime 1048573 x 16 F32", "kind": "conv", "n": 1048573, "batch": 16,
         "dtype": "complex64", "call": "fft"},
        # a tenth of the benchmark's uneven batch, with its mix of lengths
        {"name": "uneven 1000 F32", "kind": "uneven", "count": 1000, "lo": 64, "hi": 1 << 18,
         "dtype": "complex64", "call": "fft"},
        # requests that arrive together at the server, lengths as the serving benchmark's
        {"name": "served 48", "kind": "served", "count": 48, "lo": 64, "hi": 1 << 18},
        # one-second frames of audio at 48 kHz: spectra and back
        {"name": "real 48000 x 512 F32", "kind": "real", "n": 48000, "batch": 512,
         "dtype": "float32"},
        # a cubic volume, as spectral solvers and filters transform it
        {"name": "volume 256^3 F32", "kind": "nd", "n0": 256, "n1": 256, "n2": 256,
         "dtype": "complex64", "call": "fft"},
        # half-precision storage of medium rows
        {"name": "half 65536 x 256", "kind": "half", "n": 65536, "batch": 256, "call": "fft"},
    ]


# ------------------------------------------------------------------------------ lengths
def _smooth(n, primes=(2, 3, 5, 7)):
    for p in primes:
        while n % p == 0:
            n //= p
    return n == 1


def _prime(n):
    return n >= 2 and all(n % p for p in range(2, math.isqrt(n) + 1))


def _nearest(n, pred, lo=2):
    d = 0
    while True:
        for c in (n - d, n + d):
            if c >= lo and pred(c):
                return c
        d += 1


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mixed_length(rng, lo, hi):
    """Log-uniform, snapped to a 7-smooth (70 %), other composite (20 %) or prime (10 %) length."""
    n, u = _log_uniform(rng, lo, hi), rng.uniform(0, 1)
    if u < 0.7:
        return _nearest(n, _smooth)
    if u < 0.9:
        return _nearest(n, lambda m: not _smooth(m) and not _prime(m))
    return _nearest(n, _prime)


class _Uniform:
    """random.Random.uniform on a numpy generator, for lengths made from a case's own fields."""

    def __init__(self, seed):
        self.g = np.random.Generator(np.random.PCG64(seed))

    def uniform(self, a, b):
        return float(self.g.uniform(a, b))


def _uneven_lengths(case):
    rng = _Uniform(1000003 * case["count"] + case["lo"] + case["hi"])
    return [_mixed_length(rng, case["lo"], case["hi"]) for _ in range(case["count"])]


def _requests(case):
    """(length, rows, dtype) of each request: rows geometric with mean 16, one in ten F64."""
    rng = _Uniform(999983 * case["count"] + case["lo"] + case["hi"])
    out = []
    for _ in range(case["count"]):
        n = _mixed_length(rng, case["lo"], case["hi"])
        rows = 1 + int(math.log(1.0 - rng.uniform(0, 1)) / math.log(1.0 - 1.0 / 16.0))
        rows = max(1, min(rows, 256, (1 << 20) // n))
        out.append((n, rows, "complex128" if rng.uniform(0, 1) < 0.1 else "complex64"))
    return out


def draw(rng):
    kind = rng.choice(["vector", "rows", "rows", "rows", "conv", "conv", "uneven", "served",
                       "real", "nd", "half"])
    dtype = rng.choice(["complex64", "complex128"])
    call = rng.choice(["fft", "ifft", "bfft"])
    wide = dtype == "complex128"
    if kind == "vector":
        n = _log_uniform(rng, 16, 8192)
        return {"kind": kind, "n": _nearest(n, _smooth), "dtype": dtype}
    if kind == "rows":
        n = _nearest(_log_uniform(rng, 64, 1 << 20), _smooth)
        if rng.random() < 0.3:
            n = 1 << max(6, round(math.log2(n)))
        total = _log_uniform(rng, 1 << 18, 1 << (24 if wide else 25))
        return {"kind": kind, "n": n, "batch": max(1, total // n), "dtype": dtype, "call": call}
    if kind == "conv":
        n = _log_uniform(rng, 17, (1 << 18) if wide else (1 << 20) - 3)
        prime = rng.random() < 0.5
        n = _nearest(n, _prime if prime else lambda m: not _smooth(m, (2, 3, 5, 7, 11, 13)), 17)
        total = _log_uniform(rng, 1 << 18, 1 << (21 if wide else 23))
        return {"kind": kind, "n": n, "batch": max(1, total // n), "dtype": dtype, "call": call}
    if kind == "uneven":
        return {"kind": kind, "count": rng.randrange(50, 500), "lo": rng.choice([16, 64, 256]),
                "hi": rng.choice([1 << 14, 1 << 16, 1 << 17]), "dtype": dtype, "call": call}
    if kind == "served":
        return {"kind": kind, "count": rng.randrange(8, 60), "lo": 64,
                "hi": rng.choice([1 << 12, 1 << 15, 1 << 18])}
    if kind == "real":
        n = _log_uniform(rng, 64, 1 << 19)
        even = rng.random() < 0.8
        n = _nearest(n, lambda m: _smooth(m) and m % 2 == (0 if even else 1))
        total = _log_uniform(rng, 1 << 18, 1 << 23)
        return {"kind": kind, "n": n, "batch": max(1, total // n),
                "dtype": "float64" if wide else "float32"}
    if kind == "nd":
        if rng.random() < 0.5:
            n0, n1, n2 = (_nearest(_log_uniform(rng, 64, 2048), _smooth) for _ in range(3))
            n0 = 1
        else:
            n0, n1, n2 = (_nearest(_log_uniform(rng, 16, 200), _smooth) for _ in range(3))
        return {"kind": kind, "n0": n0, "n1": n1, "n2": n2, "dtype": dtype, "call": call}
    n = _nearest(_log_uniform(rng, 64, 1 << 18), _smooth)
    total = _log_uniform(rng, 1 << 18, 1 << 24)
    return {"kind": "half", "n": n, "batch": max(1, total // n), "call": rng.choice(["fft", "ifft"])}


# ------------------------------------------------------------------------------ inputs
def _randn(shape, dtype, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(shape, dtype=getattr(torch, dtype), device="cuda", generator=g)


def _inputs(case, seed):
    kind = case["kind"]
    if kind == "vector":
        return _randn((case["n"],), case["dtype"], seed)
    if kind in ("rows", "conv", "real"):
        return _randn((case["batch"], case["n"]), case["dtype"], seed)
    if kind == "nd":
        return _randn((case["n0"], case["n1"], case["n2"]), case["dtype"], seed)
    if kind == "half":  # (re, im) float16 pairs, scaled so that a spectrum stays in range
        x = _randn((case["batch"], 2 * case["n"]), "float32", seed) * 0.7
        return x.to(torch.float16).view(torch.complex32)
    if kind == "uneven":
        return _randn((sum(_uneven_lengths(case)),), case["dtype"], seed)
    return [_randn((b, n), d, seed + 7919 * i) for i, (n, b, d) in enumerate(_requests(case))]


def prepare(case, seed):
    x = _inputs(case, seed)
    state = {"case": case, "x": x}
    if case["kind"] == "uneven":
        lengths = _uneven_lengths(case)
        offsets = np.concatenate([[0], np.cumsum(lengths)[:-1]]).astype(np.int64)
        state["plan"] = C.UnevenPlan(lengths, offsets, np.dtype(case["dtype"]))
        state["y"] = torch.empty_like(x)
    elif case["kind"] == "served":
        state["server"] = C.Server()
        state["y"] = [torch.empty_like(v) for v in x]
    return state


def run(state):
    case, x = state["case"], state["x"]
    kind = case["kind"]
    if kind == "vector":
        y = C.fft(x)
        return y, C.ifft(y)
    if kind in ("rows", "conv"):
        return CALLS[case["call"]](x)
    if kind == "uneven":
        fwd = case["call"] == "fft"
        return state["plan"].exec_torch(x, out=state["y"], direction=C.FORWARD if fwd else C.BACKWARD,
                                        normalize=case["call"] == "ifft")
    if kind == "served":
        server = state["server"]
        tickets = [server.submit(a, b) for a, b in zip(x, state["y"])]
        return [server.wait(t) for t in tickets]
    if kind == "real":
        spectra = C.rfft(x)
        return spectra, C.irfft(spectra, case["n"])
    if kind == "nd":
        axes = None if case["n0"] > 1 else (1, 2)
        return {"fft": C.fftn, "ifft": C.ifftn, "bfft": C.bfftn}[case["call"]](x, axes)
    return CALLS[case["call"]](x).view(torch.float16)


# ------------------------------------------------------------------------------ bounds
_SIZE = {"complex64": 8, "complex128": 16, "float32": 4, "float64": 8}


def _work1(n, rows, size):
    return 2.0 * n * rows * size, 5.0 * n * rows * math.log2(max(n, 2))


def work(case):
    """Each input read once and each output written once; 5 n log2 n operations a transform."""
    kind = case["kind"]
    if kind == "vector":
        b, f = _work1(case["n"], 1, _SIZE[case["dtype"]])
        return {"bytes": 2 * b, "flops": 2 * f}
    if kind in ("rows", "conv"):
        b, f = _work1(case["n"], case["batch"], _SIZE[case["dtype"]])
        return {"bytes": b, "flops": f}
    if kind == "half":
        b, f = _work1(case["n"], case["batch"], 4)
        return {"bytes": b, "flops": f}
    if kind == "uneven":
        each = [_work1(n, 1, _SIZE[case["dtype"]]) for n in _uneven_lengths(case)]
    elif kind == "served":
        each = [_work1(n, b, _SIZE[d]) for n, b, d in _requests(case)]
    elif kind == "real":  # rows read, spectra written, spectra read, rows written
        n, rows, size = case["n"], case["batch"], _SIZE[case["dtype"]]
        return {"bytes": 2.0 * rows * size * (n + 2 * (n // 2 + 1)),
                "flops": 5.0 * n * rows * math.log2(n)}
    else:
        total = case["n0"] * case["n1"] * case["n2"]
        return {"bytes": 2.0 * total * _SIZE[case["dtype"]], "flops": 5.0 * total * math.log2(total)}
    return {"bytes": sum(e[0] for e in each), "flops": sum(e[1] for e in each)}


# ------------------------------------------------------------------------------ 64-bit values
def _rows64(x, call):
    """numpy's transform of each row, the work split over threads; F64 rows in long double."""
    wide = np.clongdouble if x.dtype == np.complex128 and x.size <= 1 << 27 else np.complex128
    fn = np.fft.fft if call == "fft" else np.fft.ifft
    x = x.reshape(-1, x.shape[-1])
    scale = x.shape[-1] if call == "bfft" else 1
    y = np.empty(x.shape, np.complex128)
    rows = max(1, (1 << 18) // x.shape[-1])

    def part(r):
        v = fn(x[r:r + rows].astype(wide), axis=-1)
        y[r:r + rows] = v * scale if scale != 1 else v

    with ThreadPoolExecutor(min(16, os.cpu_count() or 1)) as ex:
        list(ex.map(part, range(0, x.shape[0], rows)))
    return y


def exact(case, seed):
    kind, x = case["kind"], _inputs(case, seed)
    if kind == "served":
        return [torch.from_numpy(_rows64(v.cpu().numpy(), "fft").reshape(v.shape)) for v in x]
    if kind == "half":
        x = x.view(torch.float16).float().view(torch.complex64)
    x = x.cpu().numpy()
    if kind == "vector":
        return torch.from_numpy(_rows64(x[None], "fft")[0]), torch.from_numpy(x.astype(np.complex128))
    if kind in ("rows", "conv"):
        return torch.from_numpy(_rows64(x, case["call"]))
    if kind == "half":
        return torch.view_as_real(torch.from_numpy(_rows64(x, case["call"]))).reshape(x.shape[0], -1)
    if kind == "uneven":
        y, lengths = np.empty(x.shape, np.complex128), _uneven_lengths(case)
        ends = np.cumsum(lengths)

        def one(k):
            y[ends[k] - lengths[k]:ends[k]] = _rows64(x[None, ends[k] - lengths[k]:ends[k]],
                                                      case["call"])[0]

        with ThreadPoolExecutor(min(16, os.cpu_count() or 1)) as ex:
            list(ex.map(one, range(len(lengths))))
        return torch.from_numpy(y)
    if kind == "real":
        spectra = np.empty((x.shape[0], x.shape[1] // 2 + 1), np.complex128)
        rows = max(1, (1 << 18) // x.shape[1])

        def part(r):
            spectra[r:r + rows] = np.fft.rfft(x[r:r + rows].astype(np.float64), axis=-1)

        with ThreadPoolExecutor(min(16, os.cpu_count() or 1)) as ex:
            list(ex.map(part, range(0, x.shape[0], rows)))
        return torch.from_numpy(spectra), torch.from_numpy(x.astype(np.float64))
    axes = (0, 1, 2) if case["n0"] > 1 else (1, 2)
    y = x.astype(np.complex128)
    y = np.fft.fftn(y, axes=axes) if case["call"] == "fft" else np.fft.ifftn(y, axes=axes)
    return torch.from_numpy(y * (np.prod([y.shape[a] for a in axes]) if case["call"] == "bfft" else 1))

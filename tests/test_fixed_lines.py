"""Kernels of lines whose radices are compile-time constants (csrc/fixed_line.h).

A fixed line performs the operations of the run-time pass table in the same order, so the default
plan of a length must give, bit for bit, what the same length gives with its shape forced through
wisdom (a forced E runs the run-time kernels): every length that has a kernel of its own, both
precisions, both directions, batches that leave a workgroup partly filled, rows with gaps, in
place.  The CPU tests run the emulation build, whose list is a sample of the lengths.
"""
import ctypes
import os
import re

import numpy as np
import pytest

from conftest import ROOT, seeded_complex

TABLE = os.path.join(ROOT, "catabrafft.jl_amd", "csrc", "fixed_table.h")


def _lengths(prefix):
    """The lengths of the lists whose macro name is prefix or prefix with a part number."""
    out, on = set(), False
    with open(TABLE) as f:
        for line in f:
            if line.startswith("#define"):
                on = line.split()[1].split("(")[0] == prefix
            m = re.match(r"\s+X\(([\d, ]+)\)", line)
            if on and m:
                out.add(int(np.prod([int(v) for v in m.group(1).split(",")])))
    return sorted(out)


FEW = _lengths("CFFT_ROW_LINES_FEW")
ALL = sorted(set(_lengths("CFFT_ROW_LINES_0")) | set(_lengths("CFFT_ROW_LINES_1")))


def test_every_short_smooth_length_is_listed():
    def smooth(n):
        for p in (2, 3, 5, 7):
            while n % p == 0:
                n //= p
        return n == 1

    assert ALL == [n for n in range(16, 8193) if smooth(n)] and set(FEW) <= set(ALL)


@pytest.fixture(scope="module")
def emu():
    import sys

    sys.path.insert(0, os.path.join(ROOT, "tests", "emu"))
    import build_emu
    import catabrafft._lib as L

    return L._sig(ctypes.CDLL(build_emu.build()))


def _desc(lib, p):
    buf = ctypes.create_string_buffer(4096)
    lib.cfft_plan_describe(p, buf, len(buf))
    return buf.value.decode()


def _run_time_row(n, dt, desc):
    """Short F64 lines of radix 16 and one more pass, and long F32 powers of two, keep the run-time
    kernel."""
    if dt == np.complex128:
        return n < 192 and re.search(r"direct \[16,\d+\]", desc) is not None
    return n >= 4096 and n & (n - 1) == 0


@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
@pytest.mark.parametrize("n", FEW)
def test_emulated_fixed_rows_match_the_run_time_kernel(emu, tmp_path, n, dt):
    code, batch = (0 if dt == np.complex64 else 1), 7
    idist, odist = n + 3, n + 1
    w = tmp_path / "w.txt"
    w.write_text(f"{n} {batch} {idist} {odist} {code} 1 : 16 64 0 0 0 -1 0 0\n")
    ctx = ctypes.c_void_p()
    assert emu.cfft_init(0, ctypes.byref(ctx)) == 0
    assert emu.cfft_wisdom_import(ctx, str(w).encode()) == 0
    x = seeded_complex(idist, batch=batch, seed=n, dtype=dt)
    got = {}
    for flags in (0, 1):
        p = ctypes.c_void_p()
        assert emu.cfft_plan_1d(ctx, n, batch, idist, odist, code, flags, ctypes.byref(p)) == 0
        d = _desc(emu, p)
        assert ("fixed" in d) == (flags == 0 and not _run_time_row(n, dt, d)), d
        got[flags] = []
        for direction, norm in ((-1, 0), (1, 1)):
            y = np.full((batch, odist), 7, dtype=dt)
            assert emu.cfft_exec(p, x.ctypes.data, y.ctypes.data, direction, norm, None) == 0
            assert np.all(y[:-1, n:] == 7)
            got[flags].append(y)
        emu.cfft_plan_destroy(p)
    for a, b in zip(got[0], got[1]):
        assert np.array_equal(a, b)
    emu.cfft_finalize(ctx)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
def test_fixed_rows_match_the_run_time_kernel(gpu_ready, tmp_path, dt):
    import torch

    import catabrafft as C

    code, batch = (0 if dt == np.complex64 else 1), 7
    w = tmp_path / "w.txt"
    w.write_text("".join(f"{n} {batch} {n} {n} {code} 1 : 16 64 0 0 0 -1 0 0\n" for n in ALL))
    C.import_wisdom(str(w))
    for n in ALL:
        print(f"fixed rows n={n} {np.dtype(dt)}", flush=True)
        x = torch.from_numpy(seeded_complex(n, batch=batch, seed=n, dtype=dt)).cuda()
        p, q = C.Plan(n, batch, dt), C.Plan(n, batch, dt, flags=C.MEASURE)
        fixed = not _run_time_row(n, dt, p.describe())
        assert ("fixed" in p.describe()) == fixed and "fixed" not in q.describe(), (
            p.describe(), q.describe())
        for direction, norm in ((-1, False), (1, True)):
            a = p.exec_torch(x, direction=direction, normalize=norm)
            b = q.exec_torch(x, direction=direction, normalize=norm)
            assert torch.equal(torch.view_as_real(a), torch.view_as_real(b)), (n, direction)
        z = x.clone()
        p.exec_torch(z, z)
        assert torch.equal(torch.view_as_real(z), torch.view_as_real(p.exec_torch(x)))
        ref = torch.fft.fft(x.cpu().to(torch.complex128)).cuda()
        err = float((z - ref).norm() / ref.norm())
        # four roundings of eps / 2 a pass and one for the table, as in the parity tests
        assert err < (1e-6 if code == 0 else 4 * np.finfo(float).eps * np.log2(n)), (n, err)


@pytest.mark.parametrize("threads", [64, 256, 512, 1024])
@pytest.mark.parametrize("n,dt", [(16, np.complex64), (1024, np.complex128), (720, np.complex64),
                                  (2520, np.complex64), (2520, np.complex128)])
def test_emulated_fixed_rows_at_any_thread_count(emu, tmp_path, n, dt, threads):
    """A plan that asks for the default capacity and its own thread count: kernels of 1 to 64
    lines a workgroup, on both sides of one line per workgroup."""
    code, batch = (0 if dt == np.complex64 else 1), 70
    w = tmp_path / "w.txt"
    w.write_text(f"{n} {batch} {n} {n} {code} 1 : 0 {threads} 0 0 0 -1 0 0\n")
    ctx, p = ctypes.c_void_p(), ctypes.c_void_p()
    assert emu.cfft_init(0, ctypes.byref(ctx)) == 0
    assert emu.cfft_wisdom_import(ctx, str(w).encode()) == 0
    assert emu.cfft_plan_1d(ctx, n, batch, n, n, code, 1, ctypes.byref(p)) == 0
    d = _desc(emu, p)
    tt, c = map(int, re.search(r"fixed Tt=(\d+) C=(\d+)", d).groups())
    # the kernels' launch bounds: 256 threads, or one line of more
    assert 1 <= c and (c == 1 if tt > 128 else c * tt <= 256), d
    x = seeded_complex(n, batch=batch, seed=n, dtype=dt)
    y = np.zeros_like(x)
    assert emu.cfft_exec(p, x.ctypes.data, y.ctypes.data, -1, 0, None) == 0
    ref = np.fft.fft(x.astype(np.clongdouble))
    bound = 1e-6 if code == 0 else 4 * np.finfo(float).eps * np.log2(n)
    assert float(np.linalg.norm(y - ref) / np.linalg.norm(ref)) < bound, d
    emu.cfft_plan_destroy(p)
    emu.cfft_finalize(ctx)


# ------------------------------------------------------------------------------ four-step passes
FS_FEW = _lengths("CFFT_FS_LINES_FEW")
FS_ALL = _lengths("CFFT_FS_LINES")
FORCED = "16 64 {n1} 2 2 -1 0 0 pr=0"  # the run-time kernels, one line per thread
OWN = "0 64 {n1} 0 0 -1 -1 0"          # the lines' own kernels, at their tiles


def _emu_four_step(emu, tmp_path, n1, n2, batch, dt, fields, dist, shift):
    """A four-step of n1 x n2 in the emulation, its rows `dist` apart and its buffers `shift`
    elements past a 16-byte boundary: forward out of place, inverse in place."""
    n, code = n1 * n2, (0 if dt == np.complex64 else 1)
    w = tmp_path / "w.txt"
    w.write_text(f"{n} {batch} {dist} {dist} {code} 1 : {fields.format(n1=n1)}\n")
    ctx, p = ctypes.c_void_p(), ctypes.c_void_p()
    assert emu.cfft_init(0, ctypes.byref(ctx)) == 0
    assert emu.cfft_wisdom_import(ctx, str(w).encode()) == 0
    assert emu.cfft_plan_1d(ctx, n, batch, dist, dist, code, 1, ctypes.byref(p)) == 0
    x = np.zeros(batch * dist + 2, dtype=dt)[shift:][:batch * dist]
    x[:] = seeded_complex(batch * dist, seed=n, dtype=dt)
    y = np.zeros(batch * dist + 2, dtype=dt)[shift:][:batch * dist]
    assert emu.cfft_exec(p, x.ctypes.data, y.ctypes.data, -1, 0, None) == 0
    assert emu.cfft_exec(p, x.ctypes.data, x.ctypes.data, 1, 1, None) == 0
    d = _desc(emu, p)
    emu.cfft_plan_destroy(p)
    emu.cfft_finalize(ctx)
    return d, y, x


@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
@pytest.mark.parametrize("n2", [16, 35])  # an even and an odd number of lines side by side
@pytest.mark.parametrize("n1", FS_FEW)
def test_emulated_fixed_four_step_matches_the_run_time_kernels(emu, tmp_path, n1, n2, dt):
    for a, b, dist, shift in ((n1, n2, n1 * n2, 0), (n2, n1, n1 * n2 + 1, 1)):
        if n2 == 35 and n2 not in FS_FEW and a == n2:
            continue
        d0, y0, x0 = _emu_four_step(emu, tmp_path, a, b, 3, dt, FORCED, dist, shift)
        d1, y1, x1 = _emu_four_step(emu, tmp_path, a, b, 3, dt, OWN, dist, shift)
        assert "fixed" not in d0 and "fixed=" in d1, (d0, d1)
        assert np.array_equal(y0, y1) and np.array_equal(x0, x1), (a, b, dist)


@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
@pytest.mark.parametrize("ca,cb", [(2, 0), (0, 8), (8, 4)])
def test_emulated_four_step_keeps_the_tiles_it_is_given(emu, tmp_path, dt, ca, cb):
    """Tiles asked for through wisdom at the default capacity are the ones that run, with the
    default tiles' bits."""
    n1, n2 = 256, 128
    d0, y0, x0 = _emu_four_step(emu, tmp_path, n1, n2, 2, dt, OWN, n1 * n2, 0)
    d1, y1, x1 = _emu_four_step(emu, tmp_path, n1, n2, 2, dt, f"0 64 {{n1}} {ca} {cb} -1 -1 0",
                                n1 * n2, 0)
    assert "fixed=AB" in d0 and "fixed" not in d1, (d0, d1)
    assert (not ca or f" CA={ca} " in d1) and (not cb or f" CB={cb} " in d1), d1
    assert np.array_equal(y0, y1) and np.array_equal(x0, x1)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
def test_fixed_four_step_matches_the_run_time_kernels(gpu_ready, tmp_path, dt):
    import torch

    import catabrafft as C

    code, batch = (0 if dt == np.complex64 else 1), 2
    for line in FS_ALL:
        for n1, n2 in ((line, 16), (48, line), (line, 15)):
            n = n1 * n2
            got = []
            for fields in (FORCED, OWN):
                w = tmp_path / "w.txt"
                w.write_text(f"{n} {batch} {n} {n} {code} 1 : {fields.format(n1=n1)}\n")
                C.import_wisdom(str(w))
                p = C.Plan(n, batch, dt, flags=C.MEASURE)
                print(f"{np.dtype(dt)} {p.describe()}", flush=True)
                own = "A" if n2 == 15 else "AB"
                assert ("fixed=" + own in p.describe()) == (fields is OWN), p.describe()
                x = torch.from_numpy(seeded_complex(n, batch=batch, seed=n, dtype=dt)).cuda()
                y = p.exec_torch(x, direction=1, normalize=True)
                p.exec_torch(x, x)
                got.append((torch.view_as_real(y), torch.view_as_real(x)))
            assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]), (n1, n2)


# ------------------------------------------------------------------------------ strided axes
STRIDED_FEW = _lengths("CFFT_STRIDED_LINES_FEW")
STRIDED = _lengths("CFFT_STRIDED_LINES")


def _nd_reference(x):
    return np.fft.fft(x.astype(np.clongdouble), axis=0)


@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
@pytest.mark.parametrize("n", STRIDED_FEW + [64, 80, 176, 1000])
@pytest.mark.parametrize("inner", [18, 5])  # line pairs, and an odd number of lines
def test_emulated_strided_axes(emu, n, inner, dt):
    """A strided axis on both sides of the range whose sequences have no radix 16."""
    ctx, p, code = ctypes.c_void_p(), ctypes.c_void_p(), (0 if dt == np.complex64 else 1)
    assert emu.cfft_init(0, ctypes.byref(ctx)) == 0
    dims = (ctypes.c_int64 * 2)(n, inner)
    assert emu.cfft_plan_nd(ctx, 2, dims, 1, code, 0, ctypes.byref(p)) == 0
    d = _desc(emu, p)
    if n in STRIDED_FEW and (code == 0 or n < 512):
        assert "fixed" in d, d
    x = seeded_complex(n * inner, seed=n, dtype=dt).reshape(n, inner)
    y = np.zeros_like(x)
    assert emu.cfft_exec(p, x.ctypes.data, y.ctypes.data, -1, 0, None) == 0
    want = _nd_reference(x)
    assert float(np.linalg.norm(y - want) / np.linalg.norm(want)) < _bound(n, dt), d
    emu.cfft_plan_destroy(p)
    emu.cfft_finalize(ctx)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
def test_strided_axes(gpu_ready, dt):
    import torch

    import catabrafft as C

    for n in STRIDED + [64, 1000, 1024]:
        for inner in (40, 5):
            print(f"{np.dtype(dt)} strided n={n} x {inner}", flush=True)
            x = seeded_complex(2 * n * inner, seed=n, dtype=dt).reshape(2, n, inner)
            y = C.fftn(torch.from_numpy(x).cuda(), (1,)).cpu().numpy()
            want = np.fft.fft(x.astype(np.clongdouble), axis=1)
            err = float(np.linalg.norm(y - want) / np.linalg.norm(want))
            assert err < _bound(n, dt), (n, inner, err)


# ------------------------------------------------------------------------------ convolutions
def _factor_smooth(n, primes=(2, 3, 5, 7, 11, 13)):
    for p in primes:
        while n % p == 0:
            n //= p
    return n == 1


def _prime(n):
    return n > 1 and all(n % d for d in range(2, int(n ** 0.5) + 1))


def _conv_lengths(lines):
    """Per convolution length L: the longest prime whose padded convolution fits it (Rader) and the
    longest length with a large prime factor that does (Bluestein)."""
    out, prev = [], 0
    for L in lines:
        for need, ok in ((lambda n: 2 * (n - 1) - 1, lambda n: _prime(n) and not _factor_smooth(n - 1)),
                         (lambda n: 2 * n - 1, lambda n: not _prime(n) and not _factor_smooth(n))):
            n = L // 2 + 2
            while n > 2 and not (prev < need(n) <= L and ok(n)):
                n -= 1
            if n > 2:
                out.append((L, n))
        prev = L
    return out


CONV = {np.complex64: _conv_lengths(_lengths("CFFT_CONV_LINES")),
        np.complex128: _conv_lengths(_lengths("CFFT_CONV_LINES_F64"))}


def _bound(n, dt):
    """The parity bounds: ComplexF32 1e-6, ComplexF64 4 eps log2 n (relative L2)."""
    return 1e-6 if dt == np.complex64 else 4 * np.finfo(float).eps * max(1.0, np.log2(n))


@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
def test_emulated_fixed_convolutions(emu, dt):
    ctx, code, batch = ctypes.c_void_p(), (0 if dt == np.complex64 else 1), 5
    assert emu.cfft_init(0, ctypes.byref(ctx)) == 0
    for L, n in [(16, 17), (256, 257)] + CONV[dt][::5]:
        p = ctypes.c_void_p()
        assert emu.cfft_plan_1d(ctx, n, batch, n, n, code, 0, ctypes.byref(p)) == 0
        assert f"fused L={L} " in _desc(emu, p) and "fixed" in _desc(emu, p), _desc(emu, p)
        x = seeded_complex(n, batch=batch, seed=n, dtype=dt)
        y, z = np.zeros_like(x), x.copy()
        assert emu.cfft_exec(p, x.ctypes.data, y.ctypes.data, -1, 0, None) == 0
        assert emu.cfft_exec(p, z.ctypes.data, z.ctypes.data, 1, 1, None) == 0
        for got, ref in ((y, np.fft.fft(x.astype(np.clongdouble))),
                         (z, np.fft.ifft(x.astype(np.clongdouble)))):
            err = float(np.linalg.norm(got - ref) / np.linalg.norm(ref))
            assert err < _bound(n, dt), (n, L, err)
        emu.cfft_plan_destroy(p)
    emu.cfft_finalize(ctx)


@pytest.mark.parametrize("threads", [64, 512, 1024])
@pytest.mark.parametrize("n,dt", [(19, np.complex64), (239, np.complex128), (1013, np.complex64)])
def test_emulated_fixed_convolutions_at_any_thread_count(emu, tmp_path, n, dt, threads):
    """A plan that asks for the default capacity and its own thread count keeps to the workgroups
    its kernel is compiled for (512 threads in a work list, 1024 of a longer line)."""
    code, batch = (0 if dt == np.complex64 else 1), 40 if n > 100 else 1000
    w = tmp_path / "w.txt"
    w.write_text(f"{n} {batch} {n} {n} {code} 1 : 0 {threads} 0 0 0 -1 0 0\n")
    ctx, p = ctypes.c_void_p(), ctypes.c_void_p()
    assert emu.cfft_init(0, ctypes.byref(ctx)) == 0
    assert emu.cfft_wisdom_import(ctx, str(w).encode()) == 0
    assert emu.cfft_plan_1d(ctx, n, batch, n, n, code, 1, ctypes.byref(p)) == 0
    d = _desc(emu, p)
    c, tt = map(int, re.search(r" C=(\d+) fixed Tt=(\d+)", d).groups())
    assert 1 <= c and (c == 1 or c * tt <= 512), d
    x = seeded_complex(n, batch=batch, seed=n, dtype=dt)
    y = np.zeros_like(x)
    assert emu.cfft_exec(p, x.ctypes.data, y.ctypes.data, -1, 0, None) == 0
    ref = np.fft.fft(x.astype(np.clongdouble))
    assert float(np.linalg.norm(y - ref) / np.linalg.norm(ref)) < _bound(n, dt), d
    emu.cfft_plan_destroy(p)
    emu.cfft_finalize(ctx)


def _next_smooth(m):
    while not _factor_smooth(m, (2, 3, 5, 7)):
        m += 1
    return m


@pytest.mark.parametrize("n,dt", [(1031, np.complex64), (4099, np.complex64), (239, np.complex128),
                                  (34, np.complex128), (8209, np.complex128)])
@pytest.mark.parametrize("knobs", ["16 64 0 0 0 -1 0 0", "8 128 0 0 0 -1 0 0",
                                   "0 64 0 0 0 -1 -1 0 wv=1 fc=0"])
def test_emulated_forced_convolutions_pad_as_little_as_they_can(emu, tmp_path, n, dt, knobs):
    """Shapes forced through wisdom run the run-time kernels, at the shortest smooth length: the
    longer lengths of the kernels with compile-time radices are no gain there."""
    code = 0 if dt == np.complex64 else 1
    w = tmp_path / "w.txt"
    w.write_text(f"{n} 2 {n} {n} {code} 1 : {knobs}\n")
    ctx, p = ctypes.c_void_p(), ctypes.c_void_p()
    assert emu.cfft_init(0, ctypes.byref(ctx)) == 0
    assert emu.cfft_wisdom_import(ctx, str(w).encode()) == 0
    assert emu.cfft_plan_1d(ctx, n, 2, n, n, code, 1, ctypes.byref(p)) == 0
    d = _desc(emu, p)
    L = _next_smooth(2 * (n - 1) - 1 if _prime(n) else 2 * n - 1)
    assert f" L={L} " in d and "fixed" not in d, (L, d)
    x = seeded_complex(n, batch=2, seed=n, dtype=dt)
    y = np.zeros_like(x)
    assert emu.cfft_exec(p, x.ctypes.data, y.ctypes.data, -1, 0, None) == 0
    ref = np.fft.fft(x.astype(np.clongdouble))
    assert float(np.linalg.norm(y - ref) / np.linalg.norm(ref)) < _bound(n, dt), d
    emu.cfft_plan_destroy(p)
    emu.cfft_finalize(ctx)


@pytest.mark.parametrize("n,dt", [(34, np.complex128), (137, np.complex128), (310, np.complex128),
                                  (317, np.complex64), (383, np.complex64), (1111, np.complex64),
                                  (1523, np.complex64)])
def test_emulated_padded_convolutions_are_as_accurate_as_the_shortest(emu, tmp_path, n, dt):
    """The padded length of a default plan is chosen for its rounding errors too: they are no larger
    than at the shortest smooth length, which a forced shape runs at.  Bound: the lengths' errors
    are within 4 % (one standard deviation) of the model that chooses, so two of them within
    1 + 2 sqrt(2) 0.04."""
    code, batch = (0 if dt == np.complex64 else 1), max(8, 32768 // n)
    x = seeded_complex(n, batch=batch, seed=n, dtype=dt)
    ref = np.fft.fft(x.astype(np.clongdouble))
    w = tmp_path / "w.txt"
    w.write_text(f"{n} {batch} {n} {n} {code} 1 : 16 64 0 0 0 -1 0 0\n")
    ctx, err = ctypes.c_void_p(), []
    assert emu.cfft_init(0, ctypes.byref(ctx)) == 0
    assert emu.cfft_wisdom_import(ctx, str(w).encode()) == 0
    for flags in (0, 1):
        p, y = ctypes.c_void_p(), np.zeros_like(x)
        assert emu.cfft_plan_1d(ctx, n, batch, n, n, code, flags, ctypes.byref(p)) == 0
        assert ("fixed" in _desc(emu, p)) == (flags == 0), _desc(emu, p)
        assert emu.cfft_exec(p, x.ctypes.data, y.ctypes.data, -1, 0, None) == 0
        err.append(float(np.linalg.norm(y - ref) / np.linalg.norm(ref)))
        emu.cfft_plan_destroy(p)
    assert err[0] < (1 + 2 * np.sqrt(2) * 0.04) * err[1], (n, err)
    emu.cfft_finalize(ctx)


@pytest.mark.parametrize("n,dt", [(25087, np.complex64), (100351, np.complex128), (129023, np.complex128),
                                  (156734, np.complex128)])
def test_emulated_large_convolutions_are_as_accurate_as_the_shortest(emu, tmp_path, n, dt):
    """The same for convolutions of two lines, and the same bound: 100351 and 129023, whose shortest
    length has kernels of its own, and 156734, whose shortest length has none."""
    code = 0 if dt == np.complex64 else 1
    x = seeded_complex(n, batch=2, seed=n, dtype=dt)
    ref = np.fft.fft(x.astype(np.clongdouble))
    w = tmp_path / "w.txt"
    w.write_text(f"{n} 2 {n} {n} {code} 1 : 16 64 0 0 0 -1 0 0\n")
    ctx, err, L = ctypes.c_void_p(), [], []
    assert emu.cfft_init(0, ctypes.byref(ctx)) == 0
    assert emu.cfft_wisdom_import(ctx, str(w).encode()) == 0
    for flags in (0, 1):
        p, y = ctypes.c_void_p(), np.zeros_like(x)
        assert emu.cfft_plan_1d(ctx, n, 2, n, n, code, flags, ctypes.byref(p)) == 0
        L.append(int(_desc(emu, p).split(" L=")[1].split()[0]))
        assert emu.cfft_exec(p, x.ctypes.data, y.ctypes.data, -1, 0, None) == 0
        err.append(float(np.linalg.norm(y - ref) / np.linalg.norm(ref)))
        emu.cfft_plan_destroy(p)
    assert (L[0] == L[1]) == (n != 156734), L
    assert err[0] < (1 + 2 * np.sqrt(2) * 0.04) * err[1], (n, L, err)
    emu.cfft_finalize(ctx)


@pytest.mark.parametrize("n,L", [(88607, 1 << 16 | 1 << 17), (119101, 1 << 18)])
def test_emulated_large_convolutions_prefer_few_large_factors(emu, n, L):
    """2^16 3 before 2^12 45 and 2^18 before 2^14 15, which are shorter and slower."""
    ctx, p = ctypes.c_void_p(), ctypes.c_void_p()
    assert emu.cfft_init(0, ctypes.byref(ctx)) == 0
    assert emu.cfft_plan_1d(ctx, n, 1, n, n, 0, 0, ctypes.byref(p)) == 0
    assert f" L={L} " in _desc(emu, p)
    emu.cfft_plan_destroy(p)
    emu.cfft_finalize(ctx)


SHORT_PRIMES = [n for n in range(17, 2050) if _prime(n) and _factor_smooth(n - 1)]


@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
def test_emulated_short_primes_convolve_without_padding(emu, dt):
    """A prime n up to 2049 whose n - 1 is a product of radices: a convolution of n - 1 points on a
    kernel of its own, alone and in a work list of all of them."""
    ctx, code = ctypes.c_void_p(), (0 if dt == np.complex64 else 1)
    assert emu.cfft_init(0, ctypes.byref(ctx)) == 0
    lens = np.array(SHORT_PRIMES, dtype=np.int64)
    offs = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int64)
    P, u = ctypes.POINTER(ctypes.c_int64), ctypes.c_void_p()
    x = seeded_complex(int(lens.sum()), seed=7, dtype=dt)
    y = np.zeros_like(x)
    assert emu.cfft_plan_many_uneven(ctx, len(lens), lens.ctypes.data_as(P),
                                     offs.ctypes.data_as(P), code, 0, ctypes.byref(u)) == 0
    assert emu.cfft_exec(u, x.ctypes.data, y.ctypes.data, -1, 0, None) == 0
    for n, o in zip(lens.tolist(), offs.tolist()):
        p = ctypes.c_void_p()
        assert emu.cfft_plan_1d(ctx, n, 3, n, n, code, 0, ctypes.byref(p)) == 0
        d = _desc(emu, p)
        assert f"rader-fused L={n - 1} " in d and "fixed" in d, d
        rows = np.stack([x[o:o + n]] * 3)
        assert emu.cfft_exec(p, rows.ctypes.data, rows.ctypes.data, -1, 0, None) == 0
        assert all(np.array_equal(r, y[o:o + n]) for r in rows), n
        ref = np.fft.fft(x[o:o + n].astype(np.clongdouble))
        err = float(np.linalg.norm(rows[0] - ref) / np.linalg.norm(ref))
        assert err < _bound(n, dt), (n, err)
        emu.cfft_plan_destroy(p)
    emu.cfft_plan_destroy(u)
    emu.cfft_finalize(ctx)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
def test_short_primes_convolve_without_padding(gpu_ready, dt):
    import torch

    import catabrafft as C

    lens = np.array(SHORT_PRIMES, dtype=np.int64)
    offs = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int64)
    x = torch.from_numpy(seeded_complex(int(lens.sum()), seed=7, dtype=dt)).cuda()
    y = C.UnevenPlan(lens, offs, dt).exec_torch(x, torch.zeros_like(x))
    for n, o in zip(lens.tolist(), offs.tolist()):
        p = C.Plan(n, 67, dt)
        print(f"{np.dtype(dt)} {p.describe()}", flush=True)
        rows = torch.stack([x[o:o + n]] * 67)
        p.exec_torch(rows, rows)
        assert all(torch.equal(torch.view_as_real(r), torch.view_as_real(y[o:o + n])) for r in rows)
        ref = np.fft.fft(x[o:o + n].cpu().numpy().astype(np.clongdouble))
        err = float(np.linalg.norm(rows[-1].cpu().numpy() - ref) / np.linalg.norm(ref))
        assert err < _bound(n, dt), (n, err)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
def test_fixed_convolutions(gpu_ready, dt):
    """Each length against numpy in long double, and one work list of all of them against the
    plans alone, bit for bit."""
    import torch

    import catabrafft as C

    lens = [17, 257] + [n for _, n in CONV[dt]]
    offs = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int64)
    x = torch.from_numpy(seeded_complex(int(np.sum(lens)), seed=3, dtype=dt)).cuda()
    u = C.UnevenPlan(lens, offs, dt)
    y = u.exec_torch(x, torch.zeros_like(x))
    for n, o in zip(lens, offs):
        p = C.Plan(n, 1, dt)
        print(f"{np.dtype(dt)} {p.describe()}", flush=True)
        assert "fixed" in p.describe(), p.describe()
        a = p.exec_torch(x[o:o + n])
        assert torch.equal(torch.view_as_real(a), torch.view_as_real(y[o:o + n])), n
        rows = torch.from_numpy(seeded_complex(n, batch=67, seed=n, dtype=dt)).cuda()
        q = C.Plan(n, 67, dt)
        got = q.exec_torch(rows, direction=1, normalize=True).cpu().numpy()
        ref = np.fft.ifft(rows.cpu().numpy().astype(np.clongdouble))
        err = float(np.linalg.norm(got - ref) / np.linalg.norm(ref))
        assert err < _bound(n, dt), (n, err)


# ------------------------------------------------------------------------------ large convolutions
def _convl_lengths(lo, hi, count):
    """Lengths spread over [lo, hi]: primes (Rader, padded or not) and composites with a large
    prime factor (Bluestein) in turn, 65537 = 2^16 + 1 among them where it falls in the range."""
    out = [65537] if lo <= 65537 <= hi else []
    for i in range(count):
        n = int(lo * (hi / lo) ** (i / (count - 1)))
        while not ((_prime(n) and not _factor_smooth(n - 1)) if i % 2 else
                   (not _prime(n) and not _factor_smooth(n))):
            n += 1
        out.append(n)
    return out


@pytest.mark.parametrize("dt,lo,hi,count", [(np.complex64, 8200, 140000, 9),
                                            (np.complex128, 5200, 40000, 7)])
def test_emulated_fixed_large_convolutions(emu, dt, lo, hi, count):
    ctx, code = ctypes.c_void_p(), (0 if dt == np.complex64 else 1)
    assert emu.cfft_init(0, ctypes.byref(ctx)) == 0
    lens = np.array(_convl_lengths(lo, hi, count), dtype=np.int64)
    offs = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int64)
    P, u = ctypes.POINTER(ctypes.c_int64), ctypes.c_void_p()
    x = seeded_complex(int(lens.sum()), seed=5, dtype=dt)
    y = np.zeros_like(x)
    assert emu.cfft_plan_many_uneven(ctx, len(lens), lens.ctypes.data_as(P),
                                     offs.ctypes.data_as(P), code, 0, ctypes.byref(u)) == 0
    assert emu.cfft_exec(u, x.ctypes.data, y.ctypes.data, 1, 1, None) == 0
    for n, o in zip(lens.tolist(), offs.tolist()):
        p = ctypes.c_void_p()
        assert emu.cfft_plan_1d(ctx, n, 1, n, n, code, 0, ctypes.byref(p)) == 0
        assert "fused3" in _desc(emu, p) and "fixed" in _desc(emu, p), _desc(emu, p)
        z = x[o:o + n].copy()
        assert emu.cfft_exec(p, z.ctypes.data, z.ctypes.data, 1, 1, None) == 0
        assert np.array_equal(z, y[o:o + n]), n
        ref = np.fft.ifft(x[o:o + n].astype(np.clongdouble))
        err = float(np.linalg.norm(z - ref) / np.linalg.norm(ref))
        assert err < _bound(n, dt), (n, err)
        emu.cfft_plan_destroy(p)
    emu.cfft_plan_destroy(u)
    emu.cfft_finalize(ctx)


@pytest.mark.parametrize("n,dt", [(8219, np.complex64), (3 * 2803, np.complex64),
                                  (5003, np.complex128), (3 * 1801, np.complex128)])
def test_emulated_large_convolution_tables(emu, n, dt):
    """Spectra longer than the host transforms (4096 points), in both precisions and both orders (fused
    and two-line), and blocked permutations whose last tile is partly filled: rows of a batch, forward
    and backward."""
    ctx, p, code = ctypes.c_void_p(), ctypes.c_void_p(), (0 if dt == np.complex64 else 1)
    assert emu.cfft_init(0, ctypes.byref(ctx)) == 0
    assert emu.cfft_plan_1d(ctx, n, 2, n, n, code, 0, ctypes.byref(p)) == 0
    assert "fixed" in _desc(emu, p), _desc(emu, p)
    x = seeded_complex(n, batch=2, seed=n, dtype=dt)
    for direction, ref in ((-1, np.fft.fft), (1, np.fft.ifft)):
        y, want = np.zeros_like(x), ref(x.astype(np.clongdouble))
        assert emu.cfft_exec(p, x.ctypes.data, y.ctypes.data, direction, int(direction > 0), None) == 0
        assert float(np.linalg.norm(y - want) / np.linalg.norm(want)) < _bound(n, dt), _desc(emu, p)
    emu.cfft_plan_destroy(p)
    emu.cfft_finalize(ctx)


@pytest.mark.gpu
@pytest.mark.parametrize("dt,lo,hi,count", [(np.complex64, 8200, 1500000, 40),
                                            (np.complex128, 5200, 1500000, 40)])
def test_fixed_large_convolutions(gpu_ready, dt, lo, hi, count):
    import torch

    import catabrafft as C

    lens = _convl_lengths(lo, hi, count)
    offs = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int64)
    x = torch.from_numpy(seeded_complex(int(np.sum(lens)), seed=3, dtype=dt)).cuda()
    y = C.UnevenPlan(lens, offs, dt).exec_torch(x, torch.zeros_like(x))
    for n, o in zip(lens, offs):
        for batch in (1, 3):
            p = C.Plan(n, batch, dt)
            print(f"{np.dtype(dt)} {p.describe()}", flush=True)
            assert "fixed" in p.describe(), p.describe()
            rows = torch.stack([x[o:o + n]] * batch)
            a = p.exec_torch(rows)
            for r in range(batch):
                assert torch.equal(torch.view_as_real(a[r]), torch.view_as_real(y[o:o + n])), n
        p.exec_torch(rows, rows, direction=1, normalize=True)
        ref = np.fft.ifft(x[o:o + n].cpu().numpy().astype(np.clongdouble))
        err = float(np.linalg.norm(rows[-1].cpu().numpy() - ref) / np.linalg.norm(ref))
        assert err < _bound(n, dt), (n, err)


# ------------------------------------------------------------------------------ real input
def _check_real(n, batch, dt, forward, backward):
    """rfft and irfft of `batch` rows against numpy in long double, at the parity bounds."""
    rng = np.random.Generator(np.random.PCG64(n))
    x = rng.standard_normal((batch, n)).astype(dt)
    bound = 1e-6 if dt == np.float32 else 4 * np.finfo(float).eps * np.log2(n)
    ref = np.fft.rfft(x.astype(np.longdouble), axis=-1)
    got = forward(x)
    assert float(np.linalg.norm(got - ref) / np.linalg.norm(ref)) < bound, n
    # the transform of a spectrum whose ends are real, as numpy takes them to be
    X = (rng.standard_normal(got.shape) + 1j * rng.standard_normal(got.shape)).astype(got.dtype)
    X[:, 0] = X[:, 0].real
    X[:, -1] = X[:, -1].real
    ref = np.fft.irfft(X.astype(np.clongdouble), n, axis=-1)
    got = backward(X)
    assert float(np.linalg.norm(got - ref) / np.linalg.norm(ref)) < bound, n


@pytest.mark.parametrize("n,dt", [(2 * 1024 * 256, np.float32), (2 * 1024 * 128, np.float64)])
def test_emulated_real_four_step_ends(emu, tmp_path, n, dt):
    ctx, p, batch = ctypes.c_void_p(), ctypes.c_void_p(), 2
    cdt = np.complex64 if dt == np.float32 else np.complex128
    assert emu.cfft_init(0, ctypes.byref(ctx)) == 0
    assert emu.cfft_plan_1d_real(ctx, n, batch, n, n // 2 + 1, 0 if dt == np.float32 else 1, 0,
                                 ctypes.byref(p)) == 0
    assert "fused ends" in _desc(emu, p), _desc(emu, p)

    def run(a, out, direction):
        assert emu.cfft_exec(p, a.ctypes.data, out.ctypes.data, direction, 1, None) == 0
        return out

    _check_real(n, batch, dt, lambda x: run(x, np.zeros((batch, n // 2 + 1), cdt), -1),
                lambda X: run(X, np.zeros((batch, n), dt), 1))
    emu.cfft_plan_destroy(p)
    emu.cfft_finalize(ctx)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_real_four_step_ends(gpu_ready, dt):
    import torch

    import catabrafft as C

    for m in (16807, 19683, 24000, 32768, 34300, 46656, 50625, 65536, 78125, 131072, 10 ** 6,
              1 << 20, 2 * 3 ** 12):
        p = C.RealPlan(2 * m, 3, dt)
        print(p.describe(), flush=True)
        assert "fused ends" in p.describe(), p.describe()
        _check_real(2 * m, 3, dt,
                    lambda x: p.forward_torch(torch.from_numpy(x).cuda()).cpu().numpy(),
                    lambda X: p.backward_torch(torch.from_numpy(X).cuda(), True).cpu().numpy())

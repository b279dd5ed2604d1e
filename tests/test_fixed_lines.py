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
        assert ("fixed" in d) == (flags == 0), d
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
        assert "fixed" in p.describe() and "fixed" not in q.describe(), (p.describe(), q.describe())
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

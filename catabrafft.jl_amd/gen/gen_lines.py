#!/usr/bin/env python3
"""Generates csrc/fixed_table.h: the lines that have kernels of their own (fixed_line.h).

    python gen_lines.py [out.h]

A line is a length and its radix sequence, the one the planner takes by default for that length
(line_radices in library.cpp).  The rows kernels cover every 7-smooth length from 16 to 8192: the
lengths a workgroup holds in both precisions.  The four-step passes cover every 7-smooth length
from 16 to 2048, and 4096: the factors of the lengths up to 2^22 and of 2^24.  The lists are split in parts so that several
translation units compile them in parallel; the _FEW list is the part that the CPU emulation
build of the tests compiles.
"""
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
PARTS = 2


def line_radices(n):
    """16s (with one 8, 4 or 2 for the remainder), 9s and a 3, then 7s and 5s; largest first."""
    cnt = {}
    m = n
    for p in (2, 3, 5, 7):
        while m % p == 0:
            cnt[p] = cnt.get(p, 0) + 1
            m //= p
    if m != 1:
        return None
    r = []
    q, rem = divmod(cnt.get(2, 0), 4)
    if rem == 1 and q >= 1:
        r += [16] * (q - 1) + [8, 4]
    else:
        r += [16] * q + {0: [], 1: [2], 2: [4], 3: [8]}[rem]
    r += [9] * (cnt.get(3, 0) // 2) + [3] * (cnt.get(3, 0) % 2)
    r += [7] * cnt.get(7, 0) + [5] * cnt.get(5, 0)
    return sorted(r, reverse=True)


def fourstep_radices(n):
    """Powers of two: the fewest passes, the bits spread evenly, smallest radix first; others as
    line_radices (fourstep_line_radices in library.cpp)."""
    if n & (n - 1):
        return line_radices(n)
    k = n.bit_length() - 1
    passes = (k + 3) // 4
    base, extra = divmod(k, passes)
    return [1 << (base + (i >= passes - extra)) for i in range(passes)]


def macro(name, lines):
    out = [f"#define {name}(X) \\"]
    out += [f"    X({', '.join(map(str, r))}) \\" for r in lines]
    out[-1] = out[-1][:-2]
    return "\n".join(out)


def main():
    out = sys.argv[1] if len(sys.argv) > 1 else os.path.join(HERE, "..", "csrc", "fixed_table.h")
    rows = [line_radices(n) for n in range(16, 8193) if line_radices(n)]
    parts = [
        "// fixed_table.h -- GENERATED by gen/gen_lines.py; do not edit by hand.",
        "// Radix sequences of the lines with kernels of their own: X(r0, r1, ...).",
        "#pragma once",
        macro("CFFT_ROW_LINES_FEW", [r for i, r in enumerate(rows) if i % 24 == 5]
              + [line_radices(n) for n in (16, 64, 720, 1024, 2520)]),
    ]
    for k in range(PARTS):
        parts.append(macro(f"CFFT_ROW_LINES_{k}", rows[k::PARTS]))
    fs = [fourstep_radices(n) for n in list(range(16, 2049)) + [4096] if line_radices(n)]
    fs += [[2, 8, 8], [4, 8, 8]]  # the strided axes of N-D transforms: no radix 16
    parts.append(macro("CFFT_FS_LINES_FEW", [r for i, r in enumerate(fs) if i % 16 == 3]
                       + [fourstep_radices(n) for n in (16, 128, 256, 1024)] + fs[-2:]))
    parts.append(macro("CFFT_FS_LINES", fs))
    with open(out, "w") as f:
        f.write("\n".join(parts) + "\n")
    print(f"wrote {os.path.normpath(out)}: {len(rows)} row lines, {len(fs)} four-step lines")


if __name__ == "__main__":
    main()

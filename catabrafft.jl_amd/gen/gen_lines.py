#!/usr/bin/env python3
"""Generates csrc/fixed_table.h: the lines that have kernels of their own (fixed_line.h).

    python gen_lines.py [out.h]

A line is a length and its radix sequence, the one the planner takes by default for that length
(line_radices in library.cpp).  The rows kernels cover every 7-smooth length from 16 to 8192: the
lengths a workgroup holds in both precisions.  The four-step passes cover every 7-smooth length
from 16 to 2048, and 4096: the factors of the lengths up to 2^22 and of 2^24; strided axes have
sequences of their own under 1024 points.  The fused convolutions pad to
the lengths of conv_lines (and those of short primes that need no padding have the lengths of
conv_exact_lines), the large ones to products of two of convl_lines.  The lists are split in parts
so that several translation units compile them in parallel; the _FEW list is the part that the CPU
emulation build of the tests compiles.
"""
import math
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


# Direct lines whose threads fixed_rows.h's rule does not suit: length: (threads, lines a workgroup),
# the fastest of 2 to 12 thread counts (capacities 6 to 21, and those that the butterflies of the last
# pass fill) and of workgroups of about 64, 128 and 256 threads, on MI355X over batches of 240 MB in
# each of input and output.  They are the lengths that ran more than 2 % slower by the rule than on
# the run-time rows kernel.
ROW_SHAPES_F32 = {
    30: (15, 4), 50: (25, 10), 70: (35, 7), 90: (15, 17), 98: (49, 2), 120: (24, 10),
    126: (21, 12), 135: (45, 2), 150: (30, 8), 162: (27, 9), 225: (45, 5), 245: (49, 5),
    280: (40, 3), 315: (63, 1), 324: (41, 6), 336: (24, 5), 378: (63, 1), 560: (40, 3),
    600: (40, 6), 625: (125, 2), 648: (81, 3), 729: (81, 3), 784: (56, 1), 1792: (128, 2),
    2048: (128, 2), 3200: (320, 1), 3584: (448, 1), 3840: (240, 1), 5488: (392, 1),
    6272: (448, 1), 6400: (400, 1), 6720: (480, 1), 7168: (448, 1), 7680: (512, 1),
}
ROW_SHAPES_F64 = {
    25: (5, 51), 30: (15, 17), 32: (8, 32), 50: (25, 10), 70: (35, 7), 75: (25, 10), 98: (49, 2),
    100: (25, 10), 105: (35, 7), 140: (35, 3), 147: (49, 5), 196: (49, 5), 2048: (256, 1),
    3024: (252, 1),
}


def strided_radices(n):
    """The strided axes of N-D transforms: no radix 16, the powers of two in the fewest passes of up to
    8, largest first (strided_line_radices in library.cpp); None where the four-step's sequence stays."""
    r = fourstep_radices(n)
    if r is None or 16 not in r or not 80 <= n < 1024:
        return None
    k = (n & -n).bit_length() - 1
    passes = (k + 2) // 3
    base, extra = divmod(k, passes)
    two = [1 << (base + (i < extra)) for i in range(passes)]
    return sorted(two + [q for q in line_radices(n >> k) or []], reverse=True)


# Squared rounding error that a pass adds to a convolution, by its radix, in units of the square of
# half an epsilon; REPEATED more for the square of the number of passes of such a radix (the roundings
# of its constants add up in step).  Fitted to the errors of the convolutions of 2600
# lengths from 17 to 16,000 in both precisions; a length's error is within 4 % of the root of the
# sum, one standard deviation.
NOISE = {16: 3.0, 13: 3.7, 11: 3.3, 9: 3.3, 8: 2.5, 7: 1.7, 5: 2.2, 4: 1.8, 3: 1.9, 2: 1.3}
REPEATED = {16: 0.1, 9: 0.4, 7: 0.6}


def noise(r):
    return sum(NOISE[k] for k in r) + sum(c * r.count(k) ** 2 for k, c in REPEATED.items())


def conv_lines():
    """Convolution lengths 2^a m from 80 (the shortest padded convolutions, of n = 34, need 67 points)
    to 16384, 16s first and the odd radices last: those that no longer length beats in both cost
    (length x (passes + 0.3)) and rounding noise, nor one up to 6 % longer in noise."""
    cand = []
    for a in range(1, 15):
        for m in (1, 3, 5, 7, 9, 15, 21, 25, 27, 35, 45, 49, 63, 75, 81):
            if not 80 <= m << a <= 16384:
                continue
            q, rem = divmod(a, 4)
            r = [16] * q
            if rem == 1 and q:
                r = r[:-1] + [8, 4]
            elif rem:
                r.append(1 << rem)
            for p in (9, 7, 5, 3):
                while m % p == 0:
                    r.append(p)
                    m //= p
            cand.append(r)

    def cost(r):
        return math.prod(r) * (len(r) + 0.3)

    keep = []
    for r in sorted(cand, key=lambda r: -math.prod(r)):
        if not any(noise(k) <= noise(r) and (cost(k) <= cost(r) or math.prod(k) < 1.06 * math.prod(r))
                   for k in keep):
            keep.append(r)
    return keep[::-1]


def conv_exact_lines():
    """The other lengths n - 1 of primes n from 17 to 2049 whose factors are radices: the convolution of
    such a prime needs no padding.  Powers of two first and the odd radices last, as above (4 %
    faster than largest first, MI355X, 8 million elements; errors the same on average), but largest
    first under 64 points, where the order adds 8 % to the F32 errors of n = 31 and 61."""
    def prime(n):
        return all(n % d for d in range(2, math.isqrt(n) + 1))

    out, have = [], {math.prod(r) for r in conv_lines()}
    for L in range(16, 2049):
        if not prime(L + 1) or L in have:
            continue
        a = (L & -L).bit_length() - 1
        q, rem = divmod(a, 4)
        r, m = [16] * q, L >> a
        if rem == 1 and q:
            r = r[:-1] + [8, 4]
        elif rem:
            r.append(1 << rem)
        for p in (13, 11, 9, 7, 5, 3):
            while m % p == 0:
                r.append(p)
                m //= p
        if m == 1:
            out.append(r if L >= 64 else sorted(r, reverse=True))
    return out


def convl_lines():
    """Lines of the large convolutions: 2^a {1, 3, 5, 7, 9} from 64 to 2048 points."""
    return sorted({m << a for m in (1, 3, 5, 7, 9) for a in range(3, 12) if 64 <= m << a <= 2048})


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
    parts.append("// Direct lines with threads and lines a workgroup of their own (gen_lines.py: ROW_SHAPES_*).")
    parts.append("struct RowShape {\n    int n, threads, lines;\n};")
    for name, of in (("kRowShapesF32", ROW_SHAPES_F32), ("kRowShapesF64", ROW_SHAPES_F64)):
        parts.append(f"constexpr RowShape {name}[] = {{\n    "
                     + "\n    ".join(f"{{{n}, {t}, {c}}}," for n, (t, c) in of.items()) + "\n};")
    fs = [fourstep_radices(n) for n in list(range(16, 2049)) + [4096] if line_radices(n)]
    parts.append(macro("CFFT_FS_LINES_FEW", [r for i, r in enumerate(fs) if i % 16 == 3]
                       + [fourstep_radices(n) for n in (16, 128, 256, 1024)]))
    parts.append(macro("CFFT_FS_LINES", fs))
    strided = [strided_radices(n) for n in range(16, 1024) if strided_radices(n)]
    parts.append(macro("CFFT_STRIDED_LINES_FEW", [r for i, r in enumerate(strided) if i % 8 == 1]
                       + [strided_radices(n) for n in (128, 256)]))
    parts.append(macro("CFFT_STRIDED_LINES", strided))
    parts.append(macro("CFFT_STRIDED_LINES_F64", [r for r in strided if math.prod(r) < 512]))
    parts.append("// Squared rounding errors of the passes of a convolution by radix (gen_lines.py: noise).")
    for name, of in (("kPassNoise", NOISE), ("kRepeatedNoise", REPEATED)):
        parts.append(f"constexpr double {name}[17] = {{"
                     + ", ".join(str(of.get(r, 0.0)) for r in range(17)) + "};")
    conv = conv_lines()
    parts.append(macro("CFFT_CONV_LINES", conv))
    parts.append(macro("CFFT_CONV_LINES_F64", [r for r in conv if math.prod(r) <= 8192]))
    exact = conv_exact_lines()
    parts.append(macro("CFFT_CONV_EXACT_LINES", exact))
    two = []
    for n in convl_lines():
        q = fourstep_radices(n)
        two.append([f"CFFT_Q({', '.join(map(str, r))})" for r in (q, sorted(q, reverse=True))])
    parts.append("// X(radices of launch A, radices of launches BA and C), CFFT_Q(...) a sequence")
    parts.append("#define CFFT_Q(...) Rad<__VA_ARGS__>")
    parts.append(macro("CFFT_CONVL_LINES", two))
    with open(out, "w") as f:
        f.write("\n".join(parts) + "\n")
    print(f"wrote {os.path.normpath(out)}: {len(rows)} row lines, {len(fs)} four-step lines, "
          f"{len(conv)} + {len(exact)} convolution lengths, {len(two)} lines of large convolutions")


if __name__ == "__main__":
    main()

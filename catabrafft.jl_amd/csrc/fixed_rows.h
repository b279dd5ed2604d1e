// fixed_rows.h -- rows kernels of fixed lines (fixed_line.h) and their table entries, compiled by
// kernels_fixed_rows_*.hip from the lists of fixed_table.h.
#pragma once
#include "fixed_line.h"
#include "fixed_table.h"
#include "kernels_impl.h"
#include "kernels_prec.h"

namespace cfft {

template <typename T>
struct FixedRowSrc {
    const V_t<T>* p;
    T sg;
    template <int STEP>
    __device__ __forceinline__ V_t<T> at(int e, int j) const {
        V_t<T> v = load_stream<T>((p + j * STEP)[e]);
        v.y *= sg;
        return v;
    }
};
template <typename T>
struct FixedRowDst {
    V_t<T>* p;
    T sx, sy;
    template <int STEP>
    __device__ __forceinline__ void put_at(int e, int k, V_t<T> v) const {
        store_stream<T>((p + k * STEP)[e], V_t<T>{v.x * sx, v.y * sy});
    }
};

// Elements per thread.  Timed on MI355X over 15 lengths from 128 to 4096, 10.5 million elements
// each, for capacities 6 to 18 (the run-time kernel in brackets): 12 is best or within 4 % of the
// best except where a power of two or an F64 line has a radix 16, whose other passes then pair
// their butterflies: F32 512 30.6 us at 16 against 36.4 at 12 (37.0), 2048 33.5 against 35.9
// (37.9); F64 1920 65.7 against 70.9 (101.8), 3840 74.6 against 80.6 (110.7).  At 12: F32 2520
// 37.4 us (45.5), 720 34.7 (45.8), 3000 41.5 (65.7); F64 2520 79.9 (105.1), 360 61.7 (108.8).
//
// Batches larger than the Infinity Cache (30 x 2^20 elements in F32, 15 in F64) are less forgiving:
// - lines under 192 points take 8, as many threads as the run-time kernel, whose stores run over
//   more lanes: F32 64 144 us (208 at 12; run-time 149), 96 92 (148; 97); F64 48 119 (141; 119);
// - F32 lines of radix 16 take 8 where 12 leaves more than a tenth of the waves' lanes without a
//   thread: 384 125 us (149 at 12; run-time 128), 640 106 (126; 115), 960 96 (115; 107), 720 105
//   (116; 127); where it does not, 12 stays better: 320 99 (142 at 8; 143), 1280 103 (117; 114).
constexpr int lanes_percent(int TT) {
    return TT <= 64 ? 64 / TT * TT * 100 / 64 : TT * 100 / ((TT + 63) / 64 * 64);
}
template <typename T, class Q>
constexpr int fixed_row_capacity() {
    if (Q::N < 192) return 8;
    if (sizeof(T) == 8 && Q::has(16)) return 16;
    if (Q::threads(12) > 1024) return 16;
    if (sizeof(T) == 8) return 12;
    if ((Q::N & (Q::N - 1)) == 0) return Q::N >= 512 ? 16 : 12;
    const int t8 = Q::threads(8), t12 = Q::threads(12);
    return Q::has(16) && t8 <= 1024 && lanes_percent(t12) < 90 &&
                   lanes_percent(t8) > lanes_percent(t12)
               ? 8
               : 12;
}

// Lengths that these capacities do not suit have threads and lines a workgroup from a list, and ran
// 2-24 % slower by the rule than on the run-time kernel (240 MB batches; by the rule, now, run-time):
// F32 50 256, 122, 219 us, 126 168, 118, 153, 280 124, 101, 109, 560 129, 104, 118, 600 142, 110, 121,
// 7168 155, 117, 125; F64 30 242, 102, 200, 100 132, 89, 122, 3024 136, 98, 126.  Most are lines of whose
// last butterflies the rule's threads leave a part for another round, which stores short runs.
template <typename T>
constexpr RowShape row_shape(int n) {
    if constexpr (sizeof(T) == 4) {
        for (const RowShape& s : kRowShapesF32)
            if (s.n == n) return s;
    } else {
        for (const RowShape& s : kRowShapesF64)
            if (s.n == n) return s;
    }
    return RowShape{n, 0, 0};
}

// a.C lines per workgroup, a.Tt = TT threads and a.Ls LDS elements each.  Bound by HBM: 2520 x
// 4096 moves 4.4 TB/s in F32 and 4.2 in F64 (the run-time kernel 3.6 and 3.2), 1024 x 16384 F64
// 5.8 (5.2).
template <typename T, class Q, int TT>
__global__ void __launch_bounds__(TT > 256 ? TT : 256)
k_rows_fixed(const V_t<T>* __restrict__ in, V_t<T>* __restrict__ out, RowsArgs a,
             const V_t<T>* __restrict__ tw) {
    CFFT_DYN_LDS(smem);
    const int tid = threadIdx.x;
    const int c = TT > 128 ? 0 : tid / TT;
    const int t = tid - c * TT;
    const int64_t line = (int64_t)blockIdx.x * a.C + c;
    const bool active = line < a.nlines && c < a.C;
    const int64_t l = active ? line : 0;
    FixedRowSrc<T> src{in + l * a.idist, (T)a.sgn_in};
    FixedRowDst<T> dst{out + l * a.odist, (T)a.scale, (T)(a.scale * a.sgn_in)};
    const FixedLds<T, fixed_pad<Q>()> lds{reinterpret_cast<V_t<T>*>(smem) + c * a.Ls};
    fixed_line<T, Q, TT>(t, active, tw, src, dst, lds);
}

template <typename T, class Q>
struct FixedRowOf {
    static constexpr RowShape shape = row_shape<T>(Q::N);
    static constexpr int TT =
        shape.threads ? shape.threads : Q::threads(fixed_row_capacity<T, Q>());
    static constexpr int Ls = fixed_line_elems<Q>() | 1;  // odd: lines start in different banks
    // what k_rows_fixed is compiled for: one line where TT > 128, else up to 256 threads
    static constexpr int max_lines = TT > 128 ? 1 : 256 / TT;
    // by default: workgroups of 64 threads
    static constexpr int lines = shape.lines ? shape.lines : TT < 64 ? 64 / TT : 1;
    static_assert(lines <= max_lines, "a listed shape exceeds the kernel's launch bounds");
    static_assert(TT <= 1024, "a line runs on one workgroup");
    static hipError_t launch(const void* in, void* out, const RowsArgs& a, const void* tw,
                             hipStream_t st) {
        if (a.C < 1 || a.C > max_lines) return hipErrorInvalidValue;
        const size_t lds = sizeof(V_t<T>) * (size_t)a.C * Ls;
        const int64_t blocks = (a.nlines + a.C - 1) / a.C;
        hipLaunchKernelGGL((k_rows_fixed<T, Q, TT>), dim3((unsigned)blocks), dim3(a.C * TT), lds,
                           st, (const V_t<T>*)in, (V_t<T>*)out, a, (const V_t<T>*)tw);
        return hipGetLastError();
    }
    static void prepare() { detail::allow_big_lds(k_rows_fixed<T, Q, TT>); }
    static FixedRow row() { return FixedRow{Q::r, Q::np, Q::N, TT, Ls, lines, max_lines, launch, prepare}; }
};

}  // namespace cfft

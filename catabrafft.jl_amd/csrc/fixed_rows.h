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
template <typename T, class Q>
constexpr int fixed_row_capacity() {
    if (sizeof(T) == 8 && Q::has(16)) return 16;
    if (Q::threads(12) > 1024) return 16;
    return sizeof(T) == 4 && (Q::N & (Q::N - 1)) == 0 && Q::N >= 512 ? 16 : 12;
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
    static constexpr int TT = Q::threads(fixed_row_capacity<T, Q>());
    static constexpr int Ls = fixed_line_elems<Q>() | 1;  // odd: lines start in different banks
    static_assert(TT <= 1024, "a line runs on one workgroup");
    static hipError_t launch(const void* in, void* out, const RowsArgs& a, const void* tw,
                             hipStream_t st) {
        const size_t lds = sizeof(V_t<T>) * (size_t)a.C * Ls;
        const int64_t blocks = (a.nlines + a.C - 1) / a.C;
        hipLaunchKernelGGL((k_rows_fixed<T, Q, TT>), dim3((unsigned)blocks), dim3(a.C * TT), lds,
                           st, (const V_t<T>*)in, (V_t<T>*)out, a, (const V_t<T>*)tw);
        return hipGetLastError();
    }
    static void prepare() { detail::allow_big_lds(k_rows_fixed<T, Q, TT>); }
    static FixedRow row() { return FixedRow{Q::r, Q::np, Q::N, TT, Ls, launch, prepare}; }
};

}  // namespace cfft

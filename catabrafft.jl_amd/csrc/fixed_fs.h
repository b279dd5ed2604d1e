// fixed_fs.h -- four-step passes A and B of fixed lines (fixed_line.h) and their table entries,
// compiled by kernels_fixed_fs_*.hip from the lists of fixed_table.h.
//
// The tiles, the mapping of lanes (line first) and the operations are those of k_fs_a / k_fs_b
// (T = float, double) and of k_fs_a_pair / k_fs_b_pair (T = f2p, two adjacent ComplexF32 lines per
// thread), hence the same bits.  G is the storage of the plan's input (pass A) or output (pass B):
// ComplexF16 lines are converted at the one end that touches them, the middle stays float.
#pragma once
#include "fixed_line.h"
#include "fixed_table.h"
#include "kernels_impl.h"
#include "kernels_prec.h"

namespace cfft {

// Element at a byte offset of fewer than 2^32 from a pointer that is uniform across the wave (one
// scalar base and one 32-bit offset per lane instead of a 64-bit address per lane).
template <typename G>
__device__ __forceinline__ const G& at_byte(const G* p, unsigned off) {
    return *reinterpret_cast<const G*>(reinterpret_cast<const char*>(p) + off);
}
template <typename G>
__device__ __forceinline__ G& at_byte(G* p, unsigned off) {
    return *reinterpret_cast<G*>(reinterpret_cast<char*>(p) + off);
}

// Two adjacent elements of storage G as one access.
struct alignas(16) fx_c32x2 {
    float r0, i0, r1, i1;
};
struct alignas(8) fx_c16x2 {
    ch16 a, b;
};

// How T reads and writes storage G across adjacent lines: kWidth lines per thread.
template <typename T, typename G>
struct FsAccess {
    static constexpr int kWidth = 1;
    using E = T;  // scalar of one line
    static __device__ __forceinline__ V_t<T> load(const G* p, unsigned off) {
        return load_elem<T>(at_byte(p, off));
    }
    static __device__ __forceinline__ void store(G* p, unsigned off, V_t<T> v) {
        store_elem<T>(at_byte(p, off), v);
    }
};
template <>
struct FsAccess<f2p, float2> {
    static constexpr int kWidth = 2;
    using E = float;
    static __device__ __forceinline__ cp2 load(const float2* p, unsigned off) {
        const fx_c32x2 g = at_byte(reinterpret_cast<const fx_c32x2*>(p), off);
        return cp2{f2p(g.r0, g.r1), f2p(g.i0, g.i1)};
    }
    static __device__ __forceinline__ void store(float2* p, unsigned off, cp2 v) {
        at_byte(reinterpret_cast<fx_c32x2*>(p), off) = fx_c32x2{v.x.a, v.y.a, v.x.b, v.y.b};
    }
};
template <>
struct FsAccess<f2p, ch16> {
    static constexpr int kWidth = 2;
    using E = float;
    static __device__ __forceinline__ cp2 load(const ch16* p, unsigned off) {
        const fx_c16x2 g = at_byte(reinterpret_cast<const fx_c16x2*>(p), off);
        const float2 a = load_elem<float>(g.a), b = load_elem<float>(g.b);
        return cp2{f2p(a.x, b.x), f2p(a.y, b.y)};
    }
    static __device__ __forceinline__ void store(ch16* p, unsigned off, cp2 v) {
        fx_c16x2 g;
        store_elem<float>(g.a, float2{v.x.a, v.y.a});
        store_elem<float>(g.b, float2{v.x.b, v.y.b});
        at_byte(reinterpret_cast<fx_c16x2*>(p), off) = g;
    }
};

template <typename T> struct FsScalar { using type = T; };
template <> struct FsScalar<f2p> { using type = float; };

// v with its imaginary part(s) times sg.
template <typename T, typename S>
__device__ __forceinline__ V_t<T> fx_conj(V_t<T> v, S sg) {
    if constexpr (std::is_same<T, f2p>::value) v.y *= f2p(sg, sg);
    else v.y *= sg;
    return v;
}

// Lines with elements `stride` elements of G apart: element e of the thread's line at byte
// col + e * step of p.
template <typename T, typename G, typename S>
struct FsColSrc {
    const G* p;       // uniform
    unsigned col, step;
    S sg;
    template <int STEP>
    __device__ __forceinline__ V_t<T> at(int e, int j) const {
        const char* q = reinterpret_cast<const char*>(p) + (uint64_t)((unsigned)(j * STEP)) * step;
        return fx_conj<T>(FsAccess<T, G>::load(reinterpret_cast<const G*>(q), col + (unsigned)e * step), sg);
    }
};

// Pass A output: line c's elements contiguous at byte row of p (the second line of a pair `next`
// bytes on), streaming.
template <typename T, typename F>
struct FsMidDst {
    F* p;             // uniform; F = float2 / double2
    unsigned row, next;
    template <int STEP>
    __device__ __forceinline__ void put_at(int e, int k, V_t<T> v) const {
        F* q = p + k * STEP;
        const unsigned o = row + (unsigned)e * (unsigned)sizeof(F);
        if constexpr (std::is_same<T, f2p>::value) {
            store_stream<float>(at_byte(q, o), float2{v.x.a, v.y.a});
            store_stream<float>(at_byte(q, o + next), float2{v.x.b, v.y.b});
        } else {
            store_stream<T>(at_byte(q, o), v);
        }
    }
};

// Pass B input: as FsColSrc, then times the four-step twiddle w_n^{e k1} (of both lines of a pair).
template <typename T, typename F, typename S>
struct FsTwSrc {
    const F* p;
    unsigned col, step;
    const F* t3;      // LDS (nullptr: no twiddle)
    int tbits, k1;
    S sg;
    template <int STEP>
    __device__ __forceinline__ V_t<T> at(int e, int j) const {
        const char* q = reinterpret_cast<const char*>(p) + (uint64_t)((unsigned)(j * STEP)) * step;
        return FsAccess<T, F>::load(reinterpret_cast<const F*>(q), col + (unsigned)e * step);
    }
    template <int STEP>
    __device__ __forceinline__ V_t<T> post_at(int e, int j, V_t<T> v) const {
        const int x = (e + j * STEP) * k1;
        if (t3) {
            if constexpr (std::is_same<T, f2p>::value) {
                const float2 a = cmul(float2{v.x.a, v.y.a}, tw3_get<float>(t3, tbits, x));
                const float2 b =
                    cmul(float2{v.x.b, v.y.b}, tw3_get<float>(t3, tbits, x + (e + j * STEP)));
                v = cp2{f2p(a.x, b.x), f2p(a.y, b.y)};
            } else {
                v = cmul(v, tw3_get<T>(t3, tbits, x));
            }
        }
        return fx_conj<T>(v, sg);
    }
};

// Pass B output: element e of the thread's line(s) at byte col + e * step of p, scaled.
template <typename T, typename G, typename S>
struct FsColDst {
    G* p;
    unsigned col, step;
    S sx, sy;
    template <int STEP>
    __device__ __forceinline__ void put_at(int e, int k, V_t<T> v) const {
        char* q = reinterpret_cast<char*>(p) + (uint64_t)((unsigned)(k * STEP)) * step;
        if constexpr (std::is_same<T, f2p>::value)
            v = cp2{v.x * f2p(sx, sx), v.y * f2p(sy, sy)};
        else
            v = V_t<T>{v.x * sx, v.y * sy};
        FsAccess<T, G>::store(reinterpret_cast<G*>(q), col + (unsigned)e * step, v);
    }
};

// Most threads of a workgroup: short lines, and pairs whose first pass is a radix 16, keep to 512,
// which leaves a thread up to 256 registers (a pair's radix 16 holds 64 of data and its twiddles;
// at 1024 threads it spills to scratch memory).
template <typename T, class Q, int TT>
constexpr int fixed_fs_threads() {
    return TT <= 128 || (std::is_same<T, f2p>::value && Q::r[0] == 16) ? 512 : 1024;
}

// a.C lines per tile, a.Tt = TT threads per line (pair) and a.Ls LDS elements per line (pair).
template <typename T, typename G, class Q, int TT>
__global__ void __launch_bounds__((fixed_fs_threads<T, Q, TT>()))
k_fs_a_fixed(const G* __restrict__ in, void* __restrict__ out_, FourStepAArgs a,
             const typename Vec2<typename FsScalar<T>::type>::type* __restrict__ tw) {
    CFFT_DYN_LDS(smem);
    using S = typename FsScalar<T>::type;
    using F = typename Vec2<S>::type;
    constexpr int W = FsAccess<T, G>::kWidth;
    const int tiles = (a.N2 + a.C - 1) / a.C;
    const int bid = xcd_block(a.xcd);
    const int64_t bt = bid / tiles;
    const int j20 = (bid - (int)(bt * tiles)) * a.C;
    const int Cp = a.C / W;
    const int c = threadIdx.x & (Cp - 1);
    const int t = threadIdx.x >> (__ffs(Cp) - 1);
    const bool active = j20 + W * c < a.N2;
    const unsigned j2 = active ? W * c : 0;  // within the tile
    FsColSrc<T, G, S> src{in + bt * a.idist + j20, j2 * (unsigned)sizeof(G),
                          (unsigned)a.N2 * (unsigned)sizeof(G), (S)a.sgn_in};
    FsMidDst<T, F> dst{(F*)out_ + bt * a.odist + (int64_t)j20 * Q::N,
                       j2 * (unsigned)(Q::N * sizeof(F)), (unsigned)(Q::N * sizeof(F))};
    const FixedLds<T, fixed_pad<Q>()> lds{reinterpret_cast<V_t<T>*>(smem) + c * a.Ls};
    fixed_line<T, Q, TT>(t, active, tw, src, dst, lds);
}

template <typename T, typename G, class Q, int TT>
__global__ void __launch_bounds__((fixed_fs_threads<T, Q, TT>()))
k_fs_b_fixed(const void* in_, G* out, FourStepBArgs a,
             const typename Vec2<typename FsScalar<T>::type>::type* __restrict__ tw) {
    CFFT_DYN_LDS(smem);
    using S = typename FsScalar<T>::type;
    using F = typename Vec2<S>::type;
    constexpr int W = FsAccess<T, G>::kWidth;
    const int tiles = (a.N1 + a.C - 1) / a.C;
    const int bid = xcd_block(a.xcd);
    const int64_t bt = bid / tiles;
    const int k10 = (bid - (int)(bt * tiles)) * a.C;
    const int Cp = a.C / W;
    F* t3 = reinterpret_cast<F*>(smem + fsb_tw_offset(sizeof(T), Cp, a.Ls));
    if (a.tw3) {
        stage_table<S>((const F*)a.tw3, t3, tw3_entries(a.tbits, a.tnc));
        __syncthreads();
    }
    const int c = threadIdx.x & (Cp - 1);
    const int t = threadIdx.x >> (__ffs(Cp) - 1);
    const bool active = k10 + W * c < a.N1;
    const unsigned kc = active ? W * c : 0;  // within the tile
    FsTwSrc<T, F, S> src{(const F*)in_ + bt * a.idist + k10, kc * (unsigned)sizeof(F),
                         (unsigned)a.N1 * (unsigned)sizeof(F), a.tw3 ? t3 : nullptr, a.tbits,
                         k10 + (int)kc, (S)a.sgn_in};
    FsColDst<T, G, S> dst{out + bt * a.odist + k10, kc * (unsigned)sizeof(G),
                          (unsigned)a.N1 * (unsigned)sizeof(G), (S)a.scale,
                          (S)(a.scale * a.sgn_out)};
    const FixedLds<T, fixed_pad<Q>()> lds{reinterpret_cast<V_t<T>*>(smem) + c * a.Ls};
    fixed_line<T, Q, TT, 0, Q::np == 1>(t, active, tw, src, dst, lds);
}

// Elements per thread: 8 for powers of two and short lines, 12 for others of 512 points or more,
// whose radices then pair their butterflies (1000 = 8 5 5 5, 10^6 x 32 F64: 516 us against 620;
// 768 = 16 16 3, 786,432 x 32 F32: 205 against 233; but 160 and 125, 20,000 x 512 F64: 146 against
// 134).
template <typename T, class Q>
constexpr int fixed_fs_capacity() {
    if (Q::threads(8) > 512) return 16;
    return (Q::N & (Q::N - 1)) == 0 || Q::N < 512 ? 8 : 12;
}

template <typename T, typename G, class Q>
struct FixedFsOf {
    using S = typename FsScalar<T>::type;
    using F = typename Vec2<S>::type;
    static constexpr int TT = Q::threads(fixed_fs_capacity<T, Q>());
    static constexpr int W = FsAccess<T, G>::kWidth;
    static hipError_t launch_a(const void* in, void* out, const FourStepAArgs& a, const void* tw,
                               hipStream_t st) {
        const int64_t blocks = (int64_t)((a.N2 + a.C - 1) / a.C) * a.batch;
        hipLaunchKernelGGL((k_fs_a_fixed<T, G, Q, TT>), dim3((unsigned)blocks), dim3(a.C / W * TT),
                           fsb_tw_offset(sizeof(T), a.C / W, a.Ls), st, (const G*)in, out, a,
                           (const F*)tw);
        return hipGetLastError();
    }
    static hipError_t launch_b(const void* in, void* out, const FourStepBArgs& a, const void* tw,
                               hipStream_t st) {
        const int64_t blocks = (int64_t)((a.N1 + a.C - 1) / a.C) * a.batch;
        const size_t lds = fsb_tw_offset(sizeof(T), a.C / W, a.Ls) +
                           (a.tw3 ? (size_t)tw3_entries(a.tbits, a.tnc) * sizeof(F) : 0);
        hipLaunchKernelGGL((k_fs_b_fixed<T, G, Q, TT>), dim3((unsigned)blocks), dim3(a.C / W * TT),
                           lds, st, in, (G*)out, a, (const F*)tw);
        return hipGetLastError();
    }
    static void prepare() {
        detail::allow_big_lds(k_fs_a_fixed<T, G, Q, TT>);
        detail::allow_big_lds(k_fs_b_fixed<T, G, Q, TT>);
    }
    // pass B alone: the strided axes' sequences
    static FixedFs strided_entry() {
        FixedFs f = FixedFs{Q::r, Q::np, Q::N, TT, fixed_fs_threads<T, Q, TT>(), W, (int)sizeof(V_t<T>),
                            fixed_pad<Q>(), nullptr, launch_b, nullptr};
        f.prepare = [] { detail::allow_big_lds(k_fs_b_fixed<T, G, Q, TT>); };
        return f;
    }
    static FixedFs entry() {
        return FixedFs{Q::r, Q::np, Q::N, TT, fixed_fs_threads<T, Q, TT>(), W, (int)sizeof(V_t<T>), fixed_pad<Q>(),
                       launch_a, launch_b, prepare};
    }
};

}  // namespace cfft

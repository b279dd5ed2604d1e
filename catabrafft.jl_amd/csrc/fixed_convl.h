// fixed_convl.h -- the three launches of a large convolution (ConvLArgs in kernels.h) over lines
// whose radices are compile-time constants: A and C run fixed lines of N1 points (fixed_line.h), BA
// the in-place pair of FFTs of N2 points with the product in registers (fixed_conv.h).  Ti:
// precision of x and y; Tc: precision of the convolution.
//
// What bounds them: A and C the gather and the scatter by the primitive root (8-byte elements all
// over a line), BA the two work lines and K, 16 L bytes each in F64, and one workgroup a CU: F64 lines
// with a radix 16 take 132 registers, where 128 would let a second one in (LDS would: a tile is two
// lines of 2048).  n = 1048573 x 16 lines (ComplexF32, convolved in F64, L = 2^21): 387 +
// 438 + 456 us on the run-time kernels, 327 + 533 + 352 here.  Short lines, whose index arithmetic
// weighs more, gain more: n = 20011 x 512 in ComplexF32 406 us -> 326, x 256 in F64 354 -> 279.
//
// Tables in the order the kernels read them, so that a wave's loads are contiguous:
//   perm, iperm  [(tile N1 + e) C + c]: element (A: input, C: output) e of line c of the tile
//   K            [((tile R + k) N2 / R + b) C + c]: output k of butterfly b of line c's last
//                forward pass (radix R)
#pragma once
#include "fixed_conv.h"
#include "fixed_fs.h"

namespace cfft {

// The lines: A takes the four-step sequence of its length (powers of two smallest radix first, so
// that every thread gathers), BA and C the same radices largest first: BA's middle pass then holds
// few elements, and all of C's threads scatter (with a radix 16 last, half of them scattered twice
// as much each, and C took 650 us instead of 521 for 16 lines of L = 2^21).
template <class Q>
constexpr int convl_threads() { return Q::threads(fixed_fs_capacity<float, Q>()); }
// Most threads of a workgroup: 512 where they fit (F64 lines of 256 threads come two at a time),
// which leaves a thread up to 256 registers.
template <typename Tc>
constexpr int convl_block(int TT) { return TT <= (sizeof(Tc) == 8 ? 256 : 128) ? 512 : 1024; }

// A's input: element e of the thread's column, gathered.
template <typename Ti, typename Tc>
struct FxGatherCol {
    const V_t<Ti>* x;
    const int* perm;          // Rader: the tile's block, at line c
    const V_t<Tc>* chirp;
    int C, N2, j2, live;      // element e is there where e N2 + j2 < live
    bool rader;
    Tc sg;
    template <int STEP>
    __device__ __forceinline__ V_t<Tc> at(int e, int j) const {
        const int el = e + j * STEP, i = el * N2 + j2;
        if (rader) {
            const V_t<Ti> u = x[perm[i < live ? el * C : 0]];
            return i < live ? V_t<Tc>{(Tc)u.x, (Tc)u.y * sg} : V_t<Tc>{0, 0};
        }
        const int ic = i < live ? i : live - 1;
        const V_t<Ti> u = x[ic];
        const V_t<Tc> v = cmul(V_t<Tc>{(Tc)u.x, (Tc)u.y * sg}, chirp[ic]);
        return i < live ? v : V_t<Tc>{0, 0};
    }
};

// A's and BA's output: the thread's line, contiguous.
template <typename T>
struct FxLineDst {
    V_t<T>* p;
    template <int STEP>
    __device__ __forceinline__ void put_at(int e, int k, V_t<T> v) const { (p + k * STEP)[e] = v; }
};

// C's output.  Where an element goes (Rader) or what it is multiplied by (Bluestein) is loaded
// ahead of the butterflies.
template <typename Ti, typename Tc>
struct FxScatterDst {
    struct Prep {
        V_t<Tc> w;
        int dst;
    };
    V_t<Ti>* y;
    const int* iperm;
    const V_t<Tc>* chirp;
    int C, N2, k1, live;
    bool rader;
    V_t<Tc> x0;
    Tc invL, sx, sy;
    template <int STEP>
    __device__ __forceinline__ Prep prep_at(int e, int k) const {
        const int el = e + k * STEP, i = el * N2 + k1;
        Prep r;
        if (rader) {
            r.dst = iperm[i < live ? el * C : 0];
            r.dst = i < live ? r.dst : -1;
            r.w = V_t<Tc>{0, 0};
        } else {
            r.dst = i < live ? i : -1;
            r.w = chirp[i < live ? i : live - 1];
        }
        return r;
    }
    template <int STEP>
    __device__ __forceinline__ void put_at(int, int, V_t<Tc> v, const Prep& r) const {
        const V_t<Tc> cv = V_t<Tc>{v.x * invL, -v.y * invL};
        const V_t<Tc> o = rader ? V_t<Tc>{x0.x + cv.x, x0.y + cv.y} : cmul(cv, r.w);
        if (r.dst >= 0) y[r.dst] = V_t<Ti>{(Ti)(o.x * sx), (Ti)(o.y * sy)};
    }
};

template <typename Ti, typename Tc, class Q>
__device__ __forceinline__ void fixed_convl_a_body(unsigned char* smem, const ConvLArgs& a,
                                                   int tile, const V_t<Ti>* xl, V_t<Tc>* m1,
                                                   V_t<Tc>* slot, const V_t<Tc>* tw) {
    constexpr int TT = convl_threads<Q>();
    const int C = a.CA, c = threadIdx.x & (C - 1), t = threadIdx.x >> (__ffs(C) - 1);
    const int j2 = tile * C + c;
    const bool active = t < TT && j2 < a.N2, rader = a.mode == (int)ConvMode::Rader;
    const int tv = t < TT ? t : 0, j2c = active ? j2 : 0;
    if (rader && tile == 0 && threadIdx.x == 0) {
        const V_t<Ti> u0 = xl[0];
        slot[1] = V_t<Tc>{(Tc)u0.x, (Tc)u0.y * (Tc)a.sgn};
    }
    FxGatherCol<Ti, Tc> src{xl, a.perm + ((int64_t)tile * Q::N * C + c), (const V_t<Tc>*)a.chirp, C,
                            a.N2, j2c, (int)a.n - (rader ? 1 : 0), rader, (Tc)a.sgn};
    FxLineDst<Tc> dst{m1 + (int64_t)j2c * Q::N};
    const FixedLds<Tc, fixed_pad<Q>()> lds{reinterpret_cast<V_t<Tc>*>(smem) + c * a.LsA};
    fixed_line<Tc, Q, TT>(tv, active, tw, src, dst, lds);
}

template <typename Tc, class Q>
__device__ __forceinline__ void fixed_convl_ba_body(unsigned char* smem, const ConvLArgs& a,
                                                    int tile, const V_t<Tc>* m1, V_t<Tc>* m2,
                                                    V_t<Tc>* slot, const V_t<Tc>* tw) {
    constexpr int TT = convl_threads<Q>();
    const int C = a.CB, k10 = tile * C;
    V_t<Tc>* t3 = reinterpret_cast<V_t<Tc>*>(smem + fsb_tw_offset(sizeof(Tc), C, a.LsB));
    stage_table<Tc>((const V_t<Tc>*)a.tw3, t3, tw3_entries(a.tbits, a.tnc));
    __syncthreads();
    const int c = threadIdx.x & (C - 1), t = threadIdx.x >> (__ffs(C) - 1);
    const bool active = t < TT && k10 + c < a.N1;
    const int tv = t < TT ? t : 0, cc = active ? c : 0;
    FsTwSrc<Tc, V_t<Tc>, Tc> src{m1 + k10, cc * (unsigned)sizeof(V_t<Tc>),
                                 (unsigned)a.N1 * (unsigned)sizeof(V_t<Tc>), t3, a.tbits, k10 + cc,
                                 (Tc)1};
    FxLineDst<Tc> dst{m2 + (int64_t)(k10 + cc) * Q::N};
    const FixedLds<Tc, conv_pad<Q>()> lds{reinterpret_cast<V_t<Tc>*>(smem) + c * a.LsB};
    // the slot {A^[0]} of line k1 = 0; other lines' go to an LDS word nobody reads
    V_t<Tc>* dump = t3 + tw3_entries(a.tbits, a.tnc);
    conv_run<Tc, Q, TT, false, false>(tv, active, tw,
                                      (const V_t<Tc>*)a.K + (int64_t)tile * Q::N * C + cc,
                                      k10 + cc == 0 ? slot : dump, src, dst, lds, C);
}

template <typename Ti, typename Tc, class Q>
__device__ __forceinline__ void fixed_convl_c_body(unsigned char* smem, const ConvLArgs& a,
                                                   int tile, const V_t<Tc>* m2, V_t<Ti>* yl,
                                                   const V_t<Tc>* slots, const V_t<Tc>* tw) {
    constexpr int TT = convl_threads<Q>();
    const int C = a.CC, k10 = tile * C;
    V_t<Tc>* t3 = reinterpret_cast<V_t<Tc>*>(smem + fsb_tw_offset(sizeof(Tc), C, a.LsC));
    stage_table<Tc>((const V_t<Tc>*)a.tw3, t3, tw3_entries(a.tbits, a.tnc));
    __syncthreads();
    const int c = threadIdx.x & (C - 1), t = threadIdx.x >> (__ffs(C) - 1);
    const bool active = t < TT && k10 + c < a.N2, rader = a.mode == (int)ConvMode::Rader;
    const int tv = t < TT ? t : 0, cc = active ? c : 0;
    const Tc invL = (Tc)(1.0 / ((double)Q::N * a.N2));
    const Tc sx = (Tc)a.scale, sy = (Tc)(a.scale * a.sgn);
    const V_t<Tc> x0 = rader ? slots[1] : V_t<Tc>{0, 0};
    if (rader && tile == 0 && threadIdx.x == 0) {
        const V_t<Tc> d0 = slots[0];
        yl[0] = V_t<Ti>{(Ti)((x0.x + d0.x) * sx), (Ti)((x0.y + d0.y) * sy)};
    }
    FsTwSrc<Tc, V_t<Tc>, Tc> src{m2 + k10, cc * (unsigned)sizeof(V_t<Tc>),
                                 (unsigned)a.N2 * (unsigned)sizeof(V_t<Tc>), t3, a.tbits, k10 + cc,
                                 (Tc)1};
    FxScatterDst<Ti, Tc> dst{yl, a.iperm + ((int64_t)tile * Q::N * C + cc),
                             (const V_t<Tc>*)a.chirp, C, a.N2, k10 + cc, (int)a.n - (rader ? 1 : 0), rader, x0, invL,
                             sx, sy};
    const FixedLds<Tc, fixed_pad<Q>()> lds{reinterpret_cast<V_t<Tc>*>(smem) + c * a.LsC};
    fixed_line<Tc, Q, TT>(tv, active, tw, src, dst, lds);
}

template <typename Ti, typename Tc, class Q>
__global__ void __launch_bounds__((convl_block<Tc>(convl_threads<Q>())))
k_convl_a_fixed(const V_t<Ti>* __restrict__ x, ConvLArgs a, const V_t<Tc>* __restrict__ tw) {
    CFFT_DYN_LDS(smem);
    int64_t line;
    int tile;
    convl_tile((a.N2 + a.CA - 1) / a.CA, line, tile);
    fixed_convl_a_body<Ti, Tc, Q>(smem, a, tile, x + line * a.idist,
                                  (V_t<Tc>*)a.m1 + line * ((int64_t)Q::N * a.N2),
                                  (V_t<Tc>*)a.dc + 2 * line, tw);
}
template <typename Tc, class Q>
__global__ void __launch_bounds__((convl_block<Tc>(convl_threads<Q>())))
k_convl_ba_fixed(ConvLArgs a, const V_t<Tc>* __restrict__ tw) {
    CFFT_DYN_LDS(smem);
    int64_t line;
    int tile;
    convl_tile((a.N1 + a.CB - 1) / a.CB, line, tile);
    const int64_t L = (int64_t)a.N1 * Q::N;
    fixed_convl_ba_body<Tc, Q>(smem, a, tile, (const V_t<Tc>*)a.m1 + line * L,
                               (V_t<Tc>*)a.m2 + line * L, (V_t<Tc>*)a.dc + 2 * line, tw);
}
template <typename Ti, typename Tc, class Q>
__global__ void __launch_bounds__((convl_block<Tc>(convl_threads<Q>())))
k_convl_c_fixed(V_t<Ti>* __restrict__ y, ConvLArgs a, const V_t<Tc>* __restrict__ tw) {
    CFFT_DYN_LDS(smem);
    int64_t line;
    int tile;
    convl_tile((a.N2 + a.CC - 1) / a.CC, line, tile);
    fixed_convl_c_body<Ti, Tc, Q>(smem, a, tile,
                                  (const V_t<Tc>*)a.m2 + line * ((int64_t)Q::N * a.N2),
                                  y + line * a.odist, (const V_t<Tc>*)a.dc + 2 * line, tw);
}

// LDS bytes: C lines of Ls elements, then (BA, C) the three-level table and one element.
inline size_t convl_fixed_lds(size_t elem, int C, int Ls, size_t table) {
    return fsb_tw_offset(elem, C, Ls) + (table ? (table + 1) * 2 * elem : 0);
}

template <typename Ti, typename Tc, class Q, class QB>
struct FixedConvLOf {
    static constexpr int TT = convl_threads<Q>(), TB = convl_threads<QB>();
    static_assert(Q::N == QB::N && TT <= 1024 && TB <= 1024, "one length, one workgroup");
    static hipError_t launch_a(const void* x, const ConvLArgs& a, const void* tw, hipStream_t st) {
        const int64_t g = (int64_t)((a.N2 + a.CA - 1) / a.CA) * a.nlines;
        hipLaunchKernelGGL((k_convl_a_fixed<Ti, Tc, Q>), dim3((unsigned)g), dim3(a.CA * TT),
                           convl_fixed_lds(sizeof(Tc), a.CA, a.LsA, 0), st, (const V_t<Ti>*)x, a,
                           (const V_t<Tc>*)tw);
        return hipGetLastError();
    }
    static hipError_t launch_ba(const ConvLArgs& a, const void* tw, hipStream_t st) {
        const int64_t g = (int64_t)((a.N1 + a.CB - 1) / a.CB) * a.nlines;
        hipLaunchKernelGGL((k_convl_ba_fixed<Tc, QB>), dim3((unsigned)g), dim3(a.CB * TB),
                           convl_fixed_lds(sizeof(Tc), a.CB, a.LsB, tw3_entries(a.tbits, a.tnc)),
                           st, a, (const V_t<Tc>*)tw);
        return hipGetLastError();
    }
    static hipError_t launch_c(void* y, const ConvLArgs& a, const void* tw, hipStream_t st) {
        const int64_t g = (int64_t)((a.N2 + a.CC - 1) / a.CC) * a.nlines;
        hipLaunchKernelGGL((k_convl_c_fixed<Ti, Tc, QB>), dim3((unsigned)g), dim3(a.CC * TB),
                           convl_fixed_lds(sizeof(Tc), a.CC, a.LsC, tw3_entries(a.tbits, a.tnc)),
                           st, (V_t<Ti>*)y, a, (const V_t<Tc>*)tw);
        return hipGetLastError();
    }
    static void prepare() {
        detail::allow_big_lds(k_convl_a_fixed<Ti, Tc, Q>);
        detail::allow_big_lds(k_convl_ba_fixed<Tc, QB>);
        detail::allow_big_lds(k_convl_c_fixed<Ti, Tc, QB>);
    }
    static FixedConvL row() {
        return FixedConvL{Q::r, QB::r, Q::np, Q::N, TT, TB, fixed_pad<Q>(), conv_pad<QB>(),
                          fixed_pad<QB>(), convl_block<Tc>(TT), convl_block<Tc>(TB), launch_a, launch_ba, launch_c, prepare};
    }
};

}  // namespace cfft

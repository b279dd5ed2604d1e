// fixed_conv.h -- Rader and Bluestein transforms whose convolution length has compile-time radices
// (fixed_line.h): the whole transform in one workgroup's LDS, as conv_body, with another order of
// the two FFTs.
//
// The forward FFT_L decimates in frequency in place and leaves its output in digit-reversed order;
// the kernel spectrum is stored in that order; the second FFT_L decimates in time and takes it
// from there to natural order.  So
//   - a pass writes the LDS elements its own threads read: one barrier a pass instead of two;
//   - the last forward pass, the product with the spectrum and the first pass of the second
//     FFT_L use the same elements and stay in registers: 2 np - 1 passes instead of 2 np, and no
//     pass of its own for the product.
// What bounds it: VALU issue and the LDS exchanges of those passes (HBM moves 2 n elements a line),
// and, where a line takes more than 512 threads, that the 120 or so registers of the middle pass leave
// a CU one workgroup, whose barriers nothing hides.
// n = 4099 x 4093 lines in ComplexF32, 269 MB: 516 us on the run-time kernel (L = 8232, 10 passes
// and a product), 275 us here (L = 8960, 7 passes of 560 threads).
#pragma once
#include "fixed_line.h"
#include "fixed_table.h"
#include "kernels_impl.h"
#include "kernels_prec.h"

namespace cfft {

// LDS padding: the middle pass reads runs of the last radix (an odd one spreads them by itself).
template <class Q>
constexpr int conv_pad() { return Q::r[Q::np - 1] % 2 ? -1 : 4; }

// Butterfly b of pass I in place: p = b mod n1 and the position of its first element; its R
// elements are n1 apart.
template <class Q, int I>
struct InPlace {
    static constexpr int R = Q::r[I], g = Q::N / Q::stride(I), n1 = g / R, nb = Q::N / R;
    static __device__ __forceinline__ int p(int b) { return I == 0 ? b : (int)((unsigned)b % n1); }
    static __device__ __forceinline__ int base(int b) {
        return I == 0 ? b : (int)((unsigned)b / n1) * g + (int)((unsigned)b % n1);
    }
};

// Pass I with its twiddles after (forward, decimation in frequency) or before (second FFT_L,
// decimation in time) the butterfly.  src(e, j, n1) reads and dst(e, k, n1, v) writes element
// e + j n1; BAR: a barrier between the reads and the writes.
template <typename T, class Q, int TT, int I, bool DIT, bool BAR, typename W, class SRC, class DST>
__device__ __forceinline__ void conv_pass(const int t, const bool active, const W* __restrict__ tw,
                                          const SRC& src, const DST& dst) {
    using V = typename Vec2<T>::type;
    using P = InPlace<Q, I>;
    constexpr int R = P::R, nb = P::nb, MB = (nb + TT - 1) / TT;
    constexpr bool full = nb % TT == 0, twiddled = P::n1 > 1;
    constexpr int VW = (int)(sizeof(V) / 4);
    constexpr int KP0 = tw_prefetch_vgprs(MB * R * VW) / (MB * VW);
    constexpr int KP = !twiddled ? 0 : (R - 1) < KP0 ? (R - 1) : KP0;
    const W* __restrict__ tp = tw + Q::twoff(I);
    W w[MB][KP > 0 ? KP : 1];
    V v[MB][R];
    if constexpr (KP > 0) {
#pragma unroll
        for (int ib = 0; ib < MB; ++ib) {
            const int bt = t + ib * TT;
            const unsigned o = (unsigned)P::p(full || bt < nb ? bt : nb - 1) * (R - 1);
#pragma unroll
            for (int k = 0; k < KP; ++k) w[ib][k] = tp[o + k];
        }
    }
#pragma unroll
    for (int ib = 0; ib < MB; ++ib) {
        const int b = t + ib * TT;
        if (active && (full || b < nb)) {
            const int e = P::base(b);
#pragma unroll
            for (int j = 0; j < R; ++j) v[ib][j] = src.template at<P::n1>(e, j);
        }
    }
    if constexpr (HasPostAt<SRC>::value) {
#pragma unroll
        for (int ib = 0; ib < MB; ++ib) {
            const int b = t + ib * TT;
            if (active && (full || b < nb)) {
#pragma unroll
                for (int j = 0; j < R; ++j)
                    v[ib][j] = src.template post_at<P::n1>(P::base(b), j, v[ib][j]);
            }
        }
    }
    if constexpr (BAR) __syncthreads();
#pragma unroll
    for (int ib = 0; ib < MB; ++ib) {
        const int b = t + ib * TT;
        if (active && (full || b < nb)) {
            const int e = P::base(b), p = P::p(b);
            auto twiddle = [&] {
                if constexpr (twiddled) {
#pragma unroll
                    for (int k = 1; k <= KP; ++k) v[ib][k] = cmul(v[ib][k], w[ib][k - 1]);
#pragma unroll
                    for (int k = KP + 1; k < R; ++k)
                        v[ib][k] = cmul(v[ib][k], tp[p * (R - 1) + k - 1]);
                }
            };
            if constexpr (DIT) twiddle();
            Dft<R>::run(v[ib]);
            if constexpr (!DIT) twiddle();
#pragma unroll
            for (int k = 0; k < R; ++k) dst.template put_at<P::n1>(e, k, v[ib][k]);
        }
    }
}

// The last forward pass, conj(X K) and the first pass of the second FFT_L, in registers.  The
// spectrum of butterfly b's output k is K[(k nb + b) kc]; *dc = X[0].
template <typename T, class Q, int TT, bool BAR, class SRC, class DST>
__device__ __forceinline__ void conv_middle(const int t, const bool active,
                                            const typename Vec2<T>::type* __restrict__ K,
                                            typename Vec2<T>::type* dc, const SRC& src,
                                            const DST& dst, const int kc) {
    using V = typename Vec2<T>::type;
    constexpr int I = Q::np - 1, R = Q::r[I], nb = Q::N / R, MB = (nb + TT - 1) / TT;
    constexpr bool full = nb % TT == 0;
    // spectrum values loaded ahead of the first butterfly; the rest load after it
    constexpr int KP = R <= 8 ? R : 8;
#pragma unroll
    for (int ib = 0; ib < MB; ++ib) {
        const int b = t + ib * TT;
        V v[R], kv[KP];
        const bool live = active && (full || b < nb);
        if (live) {
#pragma unroll
            for (int k = 0; k < KP; ++k) kv[k] = (K + k * nb * kc)[b * kc];
#pragma unroll
            for (int j = 0; j < R; ++j) v[j] = src.template at<1>(b * R, j);
        }
        if constexpr (BAR) __syncthreads();
        if (live) {
            Dft<R>::run(v);
            if (b == 0) *dc = v[0];
#pragma unroll
            for (int k = 0; k < R; ++k)
                v[k] = cconj(cmul(v[k], k < KP ? kv[k < KP ? k : 0]
                                             : (K + k * nb * kc)[b * kc]));
            Dft<R>::run(v);
#pragma unroll
            for (int k = 0; k < R; ++k) dst.template put_at<1>(b * R, k, v[k]);
        }
    }
}

template <typename T, class Q, int TT, int I, typename W, class LDS>
__device__ __forceinline__ void conv_down(const int t, const bool active, const W* tw,
                                          const LDS& lds) {
    if constexpr (I < Q::np - 1) {
        conv_pass<T, Q, TT, I, false, false>(t, active, tw, lds, lds);
        __syncthreads();
        conv_down<T, Q, TT, I + 1>(t, active, tw, lds);
    }
}
template <typename T, class Q, int TT, int I, typename W, class LDS>
__device__ __forceinline__ void conv_up(const int t, const bool active, const W* tw,
                                        const LDS& lds) {
    if constexpr (I > 0) {
        conv_pass<T, Q, TT, I, true, false>(t, active, tw, lds, lds);
        __syncthreads();
        conv_up<T, Q, TT, I - 1>(t, active, tw, lds);
    }
}

// conj(FFT_L(conj(K FFT_L(src)))): src and dst hold natural order; SB: src reads the line's own
// LDS, DB: dst writes it; kc: the spectra interleaved (lines side by side in one table).
template <typename T, class Q, int TT, bool SB, bool DB, class SRC, class DST, class LDS>
__device__ __forceinline__ void conv_run(const int t, const bool active,
                                         const typename Vec2<T>::type* __restrict__ tw,
                                         const typename Vec2<T>::type* __restrict__ K,
                                         typename Vec2<T>::type* dc, const SRC& src,
                                         const DST& dst, const LDS& lds, const int kc = 1) {
    if constexpr (Q::np == 1) {
        conv_middle<T, Q, TT, SB || DB>(t, active, K, dc, src, dst, kc);
    } else {
        conv_pass<T, Q, TT, 0, false, SB>(t, active, tw, src, lds);
        __syncthreads();
        conv_down<T, Q, TT, 1>(t, active, tw, lds);
        conv_middle<T, Q, TT, false>(t, active, K, dc, lds, lds, kc);
        __syncthreads();
        conv_up<T, Q, TT, Q::np - 2>(t, active, tw, lds);
        conv_pass<T, Q, TT, 0, true, DB>(t, active, tw, lds, dst);
    }
}

// ------------------------------------------------------------------------------ the two ends
template <typename T, class LDS>
struct FxRaderSrc {  // a[e] = x[g^e] from the staged input
    LDS X;
    const int* perm;
    int live;  // n - 1
    template <int STEP>
    __device__ __forceinline__ V_t<T> at(int e, int j) const {
        const int i = e + j * STEP;
        if (i >= live) return V_t<T>{0, 0};
        return X.template at<0>(perm[i], 0);
    }
};
template <typename T, class LDS>
struct FxRaderDst {  // X[g^-k] = x0 + conj(v) / L
    LDS X;
    const int* iperm;
    V_t<T> x0;
    T invL;
    int live;
    template <int STEP>
    __device__ __forceinline__ void put_at(int e, int k, V_t<T> v) const {
        const int i = e + k * STEP;
        if (i < live)
            X.template put_at<0>(iperm[i], 0, V_t<T>{x0.x + v.x * invL, x0.y - v.y * invL});
    }
};
template <typename T>
struct FxChirpSrc {  // x[e] chirp[e] from global memory
    const V_t<T>* x;
    const V_t<T>* chirp;
    T sg;
    int n;
    template <int STEP>
    __device__ __forceinline__ V_t<T> at(int e, int j) const {
        const int i = e + j * STEP;
        if (i >= n) return V_t<T>{0, 0};
        V_t<T> v = x[i];
        v.y *= sg;
        return cmul(v, chirp[i]);
    }
};
template <typename T>
struct FxChirpDst {  // y[k] = chirp[k] conj(v) / L, scaled
    V_t<T>* y;
    const V_t<T>* chirp;
    T invL, sx, sy;
    int n;
    template <int STEP>
    __device__ __forceinline__ void put_at(int e, int k, V_t<T> v) const {
        const int i = e + k * STEP;
        if (i >= n) return;
        const V_t<T> r = cmul(V_t<T>{v.x * invL, -v.y * invL}, chirp[i]);
        y[i] = V_t<T>{r.x * sx, r.y * sy};
    }
};

// Threads of a line: one radix-16 butterfly each, the other passes up to 21 elements.
template <typename T, class Q>
constexpr int fixed_conv_threads() { return Q::has(16) ? Q::N / 16 : Q::threads(16); }
template <typename T, class Q>
constexpr int fixed_conv_block() { return fixed_conv_threads<T, Q>() > 512 ? 1024 : 512; }

// One workgroup's lines: line c of `nl` on threads [c TT, (c + 1) TT); LDS: C lines of Ls
// elements, then C slots {A^[0]}.
template <typename T, class Q, class LINES>
__device__ __forceinline__ void fixed_conv_body(unsigned char* smem, const LINES& lines, int nl,
                                                int n, int C, int Ls, int mode, int sgn,
                                                double scale, const int* perm, const int* iperm,
                                                const V_t<T>* chirp, const V_t<T>* K,
                                                const V_t<T>* tw) {
    constexpr int TT = fixed_conv_threads<T, Q>();
    using LDS = FixedLds<T, conv_pad<Q>()>;
    const int tid = threadIdx.x;
    // a work-list launch may have more threads than the item's lines: those stay idle, on a valid
    // thread index (the passes load twiddles ahead for every thread)
    const int c = tid / TT;
    const int t = tid - c * TT;
    const bool active = c < C && c < nl;
    const int cc = active ? c : 0;
    V_t<T>* const xs = reinterpret_cast<V_t<T>*>(smem);
    V_t<T>* const dc = xs + C * Ls + cc;
    const LDS L{xs + cc * Ls};
    const T sg = (T)sgn, invL = (T)(1.0 / Q::N), sx = (T)scale, sy = (T)(scale * sgn);
    const V_t<T>* const in = lines.in(cc);
    V_t<T>* const out = lines.out(cc);
    if (mode == (int)ConvMode::Rader) {
        if (active)
            batched_for<kStageLoadU>(t, TT, n, [&](int i) { return in[i]; },
                                     [&](int i, V_t<T> v) {
                                         v.y *= sg;
                                         L.template put_at<0>(i, 0, v);
                                     });
        __syncthreads();
        const V_t<T> x0 = L.template at<0>(0, 0);
        FxRaderSrc<T, LDS> src{L, perm, n - 1};
        FxRaderDst<T, LDS> dst{L, iperm, x0, invL, n - 1};
        conv_run<T, Q, TT, true, true>(t, active, tw, K, dc, src, dst, L);
        // every pass barrier lies between the slot's write and this read, except that a line of
        // one pass has only the barrier before its writes
        if constexpr (Q::np == 1) __syncthreads();
        if (active && t == 0) L.template put_at<0>(0, 0, V_t<T>{x0.x + dc->x, x0.y + dc->y});
        __syncthreads();
        if (active)
            batched_for<kStageU>(t, TT, n, [&](int i) { return L.template at<0>(i, 0); },
                                 [&](int i, V_t<T> v) { out[i] = V_t<T>{v.x * sx, v.y * sy}; });
    } else {
        FxChirpSrc<T> src{in, chirp, sg, n};
        FxChirpDst<T> dst{out, chirp, invL, sx, sy, n};
        conv_run<T, Q, TT, false, false>(t, active, tw, K, dc, src, dst, L);
    }
}

template <typename T, class Q>
__global__ void __launch_bounds__((fixed_conv_block<T, Q>()))
k_conv_fixed(const V_t<T>* __restrict__ in, V_t<T>* __restrict__ out, ConvSmallArgs a,
             const V_t<T>* __restrict__ tw) {
    CFFT_DYN_LDS(smem);
    const int64_t line0 = (int64_t)blockIdx.x * a.C;
    const int nl = (int)((a.nlines - line0) < a.C ? (a.nlines - line0) : a.C);
    UniformLines<T> lines{in + line0 * a.idist, out + line0 * a.odist, a.idist, a.odist, nullptr};
    fixed_conv_body<T, Q>(smem, lines, nl, a.n, a.C, a.Ls, a.mode, a.sgn_in, a.scale, a.perm,
                          a.iperm, (const V_t<T>*)a.chirp, (const V_t<T>*)a.K, tw);
}

template <typename T, class Q>
struct FixedConvOf {
    static constexpr int TT = fixed_conv_threads<T, Q>();
    static constexpr int SH = conv_pad<Q>();
    static_assert(TT <= 1024, "a line runs on one workgroup");
    static hipError_t launch(const void* in, void* out, const ConvSmallArgs& a, const void* tw,
                             hipStream_t st) {
        const size_t lds = sizeof(V_t<T>) * (size_t)a.C * (a.Ls + 1);
        const int64_t blocks = (a.nlines + a.C - 1) / a.C;
        hipLaunchKernelGGL((k_conv_fixed<T, Q>), dim3((unsigned)blocks), dim3(a.C * TT), lds, st,
                           (const V_t<T>*)in, (V_t<T>*)out, a, (const V_t<T>*)tw);
        return hipGetLastError();
    }
    static void prepare() { detail::allow_big_lds(k_conv_fixed<T, Q>); }
    // unpadded: of the list of exact lengths
    static FixedConv row(bool unpadded = false) {
        return FixedConv{Q::r, Q::np, Q::N, TT, SH, fixed_conv_block<T, Q>(), unpadded, launch,
                         prepare};
    }
};

}  // namespace cfft

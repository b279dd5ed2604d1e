// fixed_line.h -- the Stockham passes of engine.h for lines whose radices are known at compile
// time, and so their length, strides, twiddle offsets, threads and LDS layout too.
//
// The run-time pass table of engine.h costs a line about 40 % of its vector instructions (index
// arithmetic of every LDS and twiddle access, bounds of every butterfly), the scalar loads of the
// table between passes, and the registers of the largest radix of its switch.  Here addresses are
// one base and constants, and a kernel holds the registers of its own radices: 42-112 registers
// per lane instead of 60-128.  The operations on the data and their order are those of
// stockham_pass, so a line's bits do not depend on which of the two ran it.
#pragma once
#include "engine.h"

namespace cfft {

// The radix sequence of a line.
template <int... R>
struct Rad {
    static constexpr int np = (int)sizeof...(R);
    static constexpr int r[np] = {R...};
    static constexpr int N = (R * ...);
    // product of the radices before pass i
    static constexpr int stride(int i) {
        int s = 1;
        for (int k = 0; k < i; ++k) s *= r[k];
        return s;
    }
    // pass i's block of the twiddle table (engine.h: PassTable::twoff)
    static constexpr int twoff(int i) {
        int o = 0, s = 1;
        for (int k = 0; k < i; ++k) {
            o += N / (s * r[k]) * (r[k] - 1);
            s *= r[k];
        }
        return o;
    }
    // threads of a line whose threads hold at most E elements (at least one butterfly) in a pass
    static constexpr int threads(int E) {
        int t = 1;
        for (int k = 0; k < np; ++k) {
            const int nb = N / r[k], mb = bfly_per_thread(E, r[k]);
            const int n = (nb + mb - 1) / mb;
            t = n > t ? n : t;
        }
        return t;
    }
    static constexpr bool has(int radix) {
        for (int k = 0; k < np; ++k)
            if (r[k] == radix) return true;
        return false;
    }
};

// LDS layout of a fixed line: one pad element per 2^SH elements, SH < 0 none.  The first pass
// writes runs of r[0] elements: an odd r[0] spreads them over the banks by itself.
template <class Q>
constexpr int fixed_pad() { return Q::r[0] % 2 ? -1 : 4; }
template <int SH>
__host__ __device__ constexpr int fixed_at(int e) { return SH < 0 ? e : e + (e >> (SH < 0 ? 0 : SH)); }
template <class Q>
constexpr int fixed_line_elems() { return fixed_at<fixed_pad<Q>()>(Q::N - 1) + 1; }

// LDS position of element e + j STEP, as that of element e plus a constant where the padding
// allows it.
template <int SH, int STEP>
__device__ __forceinline__ int fixed_at(int e, int j) {
    if constexpr (SH < 0) {
        return e + j * STEP;
    } else if constexpr (STEP % (1 << SH) == 0) {
        return e + (e >> SH) + j * (STEP + (STEP >> SH));
    } else {
        const int x = e + j * STEP;
        return x + (x >> SH);
    }
}

// One line in LDS, elements (re, im) together.
template <typename T, int SH>
struct FixedLds {
    using V = typename Vec2<T>::type;
    V* p;
    template <int STEP>
    __device__ __forceinline__ V at(int e, int j) const { return p[fixed_at<SH, STEP>(e, j)]; }
    template <int STEP>
    __device__ __forceinline__ void put_at(int e, int k, V v) const { p[fixed_at<SH, STEP>(e, k)] = v; }
};

// A destination may load ahead what its stores need (HasPrepAt): prep_at<STEP>(e, k) before the
// butterflies, handed back to put_at.
template <class D, class = void>
struct HasPrepAt : std::false_type {};
template <class D>
struct HasPrepAt<D, std::void_t<typename D::Prep>> : std::true_type {};

// Pass I of line Q with TT threads: src.at<STEP>(e, j) is element e + j STEP of its input,
// dst.put_at<STEP>(e, k, v) stores element e + k STEP of its output.  BAR: a barrier between the
// reads and the writes (both go to the same LDS).  Twiddles load first, and a source's post_at
// runs once all of the pass's loads are issued, as in stockham_pass.
template <class S, class = void>
struct HasPostAt : std::false_type {};
template <class S>
struct HasPostAt<S, std::void_t<decltype(&S::template post_at<1>)>> : std::true_type {};

template <typename T, class Q, int TT, int I, bool BAR, typename W, class SRC, class DST>
__device__ __forceinline__ void fixed_pass(const int t, const bool active,
                                           const W* __restrict__ tw, const SRC& src,
                                           const DST& dst) {
    using V = typename Vec2<T>::type;
    constexpr int R = Q::r[I], s = Q::stride(I), nb = Q::N / R, MB = (nb + TT - 1) / TT;
    constexpr bool full = nb % TT == 0, twiddled = s * R < Q::N;
    constexpr int VW = (int)(sizeof(V) / 4), WW = (int)(sizeof(W) / 4);
    constexpr int KP0 = tw_prefetch_vgprs(MB * R * VW) / (MB * WW);
    constexpr int KP = !twiddled ? 0 : (R - 1) < KP0 ? (R - 1) : KP0;
    const W* __restrict__ tp = tw + Q::twoff(I);
    W w[MB][KP > 0 ? KP : 1];
    V v[MB][R];
    if constexpr (KP > 0) {
#pragma unroll
        for (int ib = 0; ib < MB; ++ib) {
            const int bt = t + ib * TT;
            const int b = full || bt < nb ? bt : nb - 1;
            const unsigned o = (unsigned)b / s * (R - 1);
#pragma unroll
            for (int k = 0; k < KP; ++k) w[ib][k] = tp[o + k];
        }
    }
#pragma unroll
    for (int ib = 0; ib < MB; ++ib) {
        const int b = t + ib * TT;
        if (active && (full || b < nb)) {
#pragma unroll
            for (int j = 0; j < R; ++j) v[ib][j] = src.template at<nb>(b, j);
        }
    }
    if constexpr (HasPostAt<SRC>::value) {
#pragma unroll
        for (int ib = 0; ib < MB; ++ib) {
            const int b = t + ib * TT;
            if (active && (full || b < nb)) {
#pragma unroll
                for (int j = 0; j < R; ++j) v[ib][j] = src.template post_at<nb>(b, j, v[ib][j]);
            }
        }
    }
    if constexpr (BAR) __syncthreads();
#pragma unroll
    for (int ib = 0; ib < MB; ++ib) {
        const int b = t + ib * TT;
        if (active && (full || b < nb)) {
            const int p = (int)((unsigned)b / s), q = b - p * s;
            if constexpr (HasPrepAt<DST>::value) {
                static_assert(!twiddled, "a last pass");
                // (8 at a time: a radix 16 would hold as many registers again)
                constexpr int H = R <= 8 ? R : 8;
                typename DST::Prep pr[H];
#pragma unroll
                for (int k = 0; k < H; ++k) pr[k] = dst.template prep_at<s>(q + s * R * p, k);
                Dft<R>::run(v[ib]);
#pragma unroll
                for (int k = 0; k < H; ++k)
                    dst.template put_at<s>(q + s * R * p, k, v[ib][k], pr[k]);
#pragma unroll
                for (int k = H; k < R; ++k) pr[k - H] = dst.template prep_at<s>(q + s * R * p, k);
#pragma unroll
                for (int k = H; k < R; ++k)
                    dst.template put_at<s>(q + s * R * p, k, v[ib][k], pr[k - H]);
            } else {
                Dft<R>::run(v[ib]);
                if constexpr (twiddled) {
#pragma unroll
                    for (int k = 1; k <= KP; ++k) v[ib][k] = cmul(v[ib][k], w[ib][k - 1]);
#pragma unroll
                    for (int k = KP + 1; k < R; ++k)
                        v[ib][k] = cmul(v[ib][k], tp[p * (R - 1) + k - 1]);
                }
                const int base = q + s * R * p;
#pragma unroll
                for (int k = 0; k < R; ++k) dst.template put_at<s>(base, k, v[ib][k]);
            }
        }
    }
}

// The passes of line Q from src through lds to dst.  ALIAS: the last pass writes what it or its
// source reads -- dst is the line's LDS, or a line of one pass works in place (a barrier between the
// two).
template <typename T, class Q, int TT, int I = 0, bool ALIAS = false, typename W, class SRC,
          class DST, class LDS>
__device__ __forceinline__ void fixed_line(const int t, const bool active,
                                           const W* __restrict__ tw, const SRC& src,
                                           const DST& dst, const LDS& lds) {
    constexpr bool first = I == 0, last = I == Q::np - 1;
    if constexpr (first && last) {
        fixed_pass<T, Q, TT, I, ALIAS>(t, active, tw, src, dst);
    } else if constexpr (first) {
        fixed_pass<T, Q, TT, I, false>(t, active, tw, src, lds);
    } else if constexpr (last) {
        fixed_pass<T, Q, TT, I, ALIAS>(t, active, tw, lds, dst);
    } else {
        fixed_pass<T, Q, TT, I, true>(t, active, tw, lds, lds);
    }
    if constexpr (!last) {
        __syncthreads();
        fixed_line<T, Q, TT, I + 1>(t, active, tw, src, dst, lds);
    }
}

}  // namespace cfft

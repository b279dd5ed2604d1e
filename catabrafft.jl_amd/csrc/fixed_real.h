// fixed_real.h -- the real-input ends of a four-step on fixed lines (fixed_fs.h): n = 2 m reals as m
// complex values, m = N1 x N2 (r2c_pair / C2RSrc in kernels_impl.h give the identities).
//
//   k_fs_b_real  pass B that untangles its spectrum before it stores it.  Output k = k1 + N1 k2
//                needs Z[m - k], which lies on line N1 - k1: a tile holds the lines k1 and N1 - k1
//                of its half range, leaves them in LDS and stores X from there.
//   k_fs_a_real  pass A that builds its input Z'[k] from X[k] and X[m - k] as it loads it.
//
// Each takes the place of an elementwise pass over the whole batch (a read and a write of m
// complex values a row) beside the two passes of the four-step.  Bound by memory like those: rfft
// and brfft of 512 rows of 48000 reals in F32 (98 MB of reals, 98 MB of spectra) take 237 us
// together instead of 287; k_fs_b_real 73 us where pass B and the untangling pass took 43 + 58,
// k_fs_a_real 66 where the tangling pass and pass A took 43 + 44.
#pragma once
#include "fixed_fs.h"

namespace cfft {

// X[k] from Z[k] and Z[m - k]; wk = w^k for 2 k <= m, else w^{m - k} (w^k = -conj(w^{m - k})).
template <typename T>
__device__ __forceinline__ V_t<T> untangle(V_t<T> zk, V_t<T> zj, V_t<T> wk, bool low) {
    V_t<T> x;
    r2c_pair<T>(zk, zj, low ? wk : V_t<T>{-wk.x, wk.y}, x);
    return x;
}

// a.C lines per tile: a.C / 2 values of k1 <= N1 / 2 and their partners.  a.odist: complex elements
// between the spectra of m + 1; rw[k] = e^{-2 pi i k / n}.
template <typename T, class Q, int TT>
__global__ void __launch_bounds__((fixed_fs_threads<T, Q, TT>()))
k_fs_b_real(const V_t<T>* __restrict__ in, V_t<T>* __restrict__ out, FourStepBArgs a,
            const V_t<T>* __restrict__ rw, const V_t<T>* __restrict__ tw) {
    CFFT_DYN_LDS(smem);
    const int N1 = a.N1, half = a.C / 2, last = N1 / 2;
    const int tiles = (last + half) / half;  // last + 1 values of k1
    const int bid = xcd_block(a.xcd);
    const int64_t bt = bid / tiles;
    const int a0 = (bid - (int)(bt * tiles)) * half;
    V_t<T>* t3 = reinterpret_cast<V_t<T>*>(smem + fsb_tw_offset(sizeof(T), a.C, a.Ls));
    stage_table<T>((const V_t<T>*)a.tw3, t3, tw3_entries(a.tbits, a.tnc));
    __syncthreads();
    const int c = threadIdx.x & (a.C - 1);
    const int t = threadIdx.x >> (__ffs(a.C) - 1);
    const int q = a0 + (c & (half - 1));  // the pair: lines q and N1 - q
    const bool upper = c >= half, active = q <= last;
    const int k1 = !active ? 0 : !upper ? q : (q ? N1 - q : 0);
    FsTwSrc<T, V_t<T>, T> src{in + bt * a.idist, (unsigned)k1 * (unsigned)sizeof(V_t<T>),
                              (unsigned)N1 * (unsigned)sizeof(V_t<T>), t3, a.tbits, k1, (T)1};
    V_t<T>* const lines = reinterpret_cast<V_t<T>*>(smem);
    const FixedLds<T, fixed_pad<Q>()> lds{lines + c * a.Ls}, mate{lines + (c ^ half) * a.Ls};
    fixed_line<T, Q, TT, 0, true>(t, active, tw, src, lds, lds);
    __syncthreads();
    // lines 0 and N1 / 2 are their own partners: the upper copy stores nothing
    if (!active || (upper && (q == 0 || 2 * q == N1))) return;
    V_t<T>* const X = out + bt * a.odist;
    const int m = N1 * Q::N;
    constexpr int U = 4;
    for (int e0 = t; e0 < Q::N; e0 += U * TT) {
        V_t<T> w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = e0 + u * TT, k = k1 + N1 * (e < Q::N ? e : 0);
            w[u] = rw[2 * k <= m ? k : m - k];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = e0 + u * TT;
            if (e >= Q::N) break;
            const int k = k1 + N1 * e;
            const int ej = k1 ? Q::N - 1 - e : (e ? Q::N - e : 0);
            const V_t<T> zk = lds.template at<0>(e, 0), zj = mate.template at<0>(ej, 0);
            X[k] = untangle<T>(zk, zj, w[u], 2 * k <= m);
            if (k == 0) X[m] = untangle<T>(zk, zj, w[u], false);
        }
    }
}

// Element k = e N2 + j2 of conj(Z'), scaled, from the spectrum X of m + 1 values.
template <typename T>
struct FsRealSrc {
    const V_t<T>* X;
    const V_t<T>* rw;
    int N2, j2, m;
    T s;
    template <int STEP>
    __device__ __forceinline__ V_t<T> at(int e, int j) const {
        const int k = (e + j * STEP) * N2 + j2;
        const V_t<T> xk = X[k], cxj = cconj(X[m - k]);
        const V_t<T> p = V_t<T>{xk.x + cxj.x, xk.y + cxj.y};
        const V_t<T> d = V_t<T>{xk.x - cxj.x, xk.y - cxj.y};
        const V_t<T> wd = cmul(cconj(rw[k]), d);
        return V_t<T>{(p.x - wd.y) * s, -((p.y + wd.x) * s)};
    }
};

// a.idist: complex elements between the spectra; scale goes into the loaded values.
template <typename T, class Q, int TT>
__global__ void __launch_bounds__((fixed_fs_threads<T, Q, TT>()))
k_fs_a_real(const V_t<T>* __restrict__ in, V_t<T>* __restrict__ out, FourStepAArgs a, double scale,
            const V_t<T>* __restrict__ rw, const V_t<T>* __restrict__ tw) {
    CFFT_DYN_LDS(smem);
    const int tiles = (a.N2 + a.C - 1) / a.C;
    const int bid = xcd_block(a.xcd);
    const int64_t bt = bid / tiles;
    const int j20 = (bid - (int)(bt * tiles)) * a.C;
    const int c = threadIdx.x & (a.C - 1);
    const int t = threadIdx.x >> (__ffs(a.C) - 1);
    const bool active = j20 + c < a.N2;
    const unsigned j2 = active ? c : 0;
    FsRealSrc<T> src{in + bt * a.idist, rw, a.N2, j20 + (int)j2, Q::N * a.N2, (T)scale};
    FsMidDst<T, V_t<T>> dst{out + bt * a.odist + (int64_t)j20 * Q::N,
                            j2 * (unsigned)(Q::N * sizeof(V_t<T>)),
                            (unsigned)(Q::N * sizeof(V_t<T>))};
    const FixedLds<T, fixed_pad<Q>()> lds{reinterpret_cast<V_t<T>*>(smem) + c * a.Ls};
    fixed_line<T, Q, TT>(t, active, tw, src, dst, lds);
}

template <typename T, class Q>
struct FixedRealOf {
    static constexpr int TT = Q::threads(fixed_fs_capacity<T, Q>());
    static hipError_t launch_b(const void* in, void* out, const FourStepBArgs& a, const void* rw,
                               const void* tw, hipStream_t st) {
        const int half = a.C / 2;
        const int64_t blocks = (int64_t)((a.N1 / 2 + half) / half) * a.batch;
        const size_t lds = fsb_tw_offset(sizeof(T), a.C, a.Ls) +
                           (size_t)tw3_entries(a.tbits, a.tnc) * sizeof(V_t<T>);
        hipLaunchKernelGGL((k_fs_b_real<T, Q, TT>), dim3((unsigned)blocks), dim3(a.C * TT), lds, st,
                           (const V_t<T>*)in, (V_t<T>*)out, a, (const V_t<T>*)rw,
                           (const V_t<T>*)tw);
        return hipGetLastError();
    }
    static hipError_t launch_a(const void* in, void* out, const FourStepAArgs& a, double scale,
                               const void* rw, const void* tw, hipStream_t st) {
        const int64_t blocks = (int64_t)((a.N2 + a.C - 1) / a.C) * a.batch;
        hipLaunchKernelGGL((k_fs_a_real<T, Q, TT>), dim3((unsigned)blocks), dim3(a.C * TT),
                           fsb_tw_offset(sizeof(T), a.C, a.Ls), st, (const V_t<T>*)in,
                           (V_t<T>*)out, a, scale, (const V_t<T>*)rw, (const V_t<T>*)tw);
        return hipGetLastError();
    }
    static void prepare() {
        detail::allow_big_lds(k_fs_a_real<T, Q, TT>);
        detail::allow_big_lds(k_fs_b_real<T, Q, TT>);
    }
    static FixedReal entry() {
        return FixedReal{Q::r, Q::np, Q::N, TT, fixed_fs_threads<T, Q, TT>(), (int)sizeof(V_t<T>),
                         fixed_pad<Q>(), launch_b, launch_a, prepare};
    }
};

}  // namespace cfft

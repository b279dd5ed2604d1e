// kernels_plan.hip -- the tables of a convolution, put on the device into the order and the precision
// that its kernels read.  Bound by memory, and by far less than the way through the host: planning
// n = 1048573 (L = 2^21) took 69 ms with the spectrum copied to the host, reordered there and copied
// back, and the permutations blocked there, 40 ms here (without any order, 39).
#include "kernels.h"
#include "kernels_impl.h"

namespace cfft {
// out[((tile N2 + x) C + c)] = F[k + N1 freq[x]], k = tile C + c (0 past the last line)
template <typename T>
__global__ void __launch_bounds__(256)
k_order_spectrum(const double2* __restrict__ F, V_t<T>* __restrict__ out,
                 const int* __restrict__ freq, int N1, int N2, int C, int64_t count) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= count) return;
    const int c = (int)(i % C);
    const int64_t r = i / C;
    const int64_t k = r / N2 * C + c;
    const double2 v = k < N1 ? F[k + (int64_t)N1 * freq[r % N2]] : double2{0, 0};
    out[i] = V_t<T>{(T)v.x, (T)v.y};
}

// out[((tile N1 + e) C + c)] = perm[e N2 + j], j = tile C + c (0 past the end)
__global__ void __launch_bounds__(256)
k_block_perm(const int* __restrict__ perm, int* __restrict__ out, int N1, int N2, int C,
             int64_t live, int64_t count) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= count) return;
    const int c = (int)(i % C);
    const int64_t r = i / C;
    const int64_t j = r / N1 * C + c, at = r % N1 * N2 + j;
    out[i] = j < N2 && at < live ? perm[at] : 0;
}

hipError_t launch_order_spectrum(Prec pc, const void* F, void* out, const int* freq, int N1, int N2,
                                 int C, int64_t count, hipStream_t st) {
    const dim3 grid((unsigned)((count + 255) / 256));
    if (pc == Prec::F32)
        hipLaunchKernelGGL(k_order_spectrum<float>, grid, dim3(256), 0, st, (const double2*)F,
                           (float2*)out, freq, N1, N2, C, count);
    else
        hipLaunchKernelGGL(k_order_spectrum<double>, grid, dim3(256), 0, st, (const double2*)F,
                           (double2*)out, freq, N1, N2, C, count);
    return hipGetLastError();
}
hipError_t launch_block_perm(const int* perm, int* out, int N1, int N2, int C, int64_t live,
                             int64_t count, hipStream_t st) {
    hipLaunchKernelGGL(k_block_perm, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, perm,
                       out, N1, N2, C, live, count);
    return hipGetLastError();
}
}  // namespace cfft

// kernels_fixed_conv_multi_f64.hip -- the work-list kernels of the fixed fused convolutions
// (fixed_conv.h) in F64: an item runs the body of its plan's length.  Lines of more than 512
// threads have a kernel of their own (Block = 1024), so that the others may hold more registers
// than a workgroup of 1024 threads allows.
#include "fixed_conv.h"

namespace cfft {
template <int Block>
__global__ void __launch_bounds__(Block)
k_conv_fixed_multi_f64(MultiArgs ma, const MItem* __restrict__ items,
                       const MPlan* __restrict__ plans) {
    CFFT_DYN_LDS(smem);
    const MItem it = items[blockIdx.x];
    const MPlan* P = plans + it.plan;
    int sgn;
    double scale;
    item_direction(it, P->n, ma, sgn, scale);
    ItemLines<double> lines{ma.in_base, ma.out_base, &it};
#define CFFT_CONV(...)                                                                          \
    case Rad<__VA_ARGS__>::N:                                                                   \
        if constexpr (fixed_conv_block<double, Rad<__VA_ARGS__>>() == Block)                        \
            fixed_conv_body<double, Rad<__VA_ARGS__>>(                                              \
                smem, lines, it.count, P->n, P->C, P->Ls, P->mode, sgn, scale, P->perm,         \
                P->iperm, (const V_t<double>*)P->chirp, (const V_t<double>*)P->K,                     \
                (const V_t<double>*)P->line.tw);                                                   \
        break;
    switch (P->L) {
        CFFT_CONV_LINES_F64(CFFT_CONV)
        default: break;
    }
}

hipError_t conv_fixed_multi_f64(const MultiLaunch& L, const MultiArgs& ma, hipStream_t st) {
    if ((MultiKernel)L.kernel == MultiKernel::ConvFixedWide)
        hipLaunchKernelGGL(k_conv_fixed_multi_f64<1024>, dim3((unsigned)L.nitems), dim3(L.block),
                           L.lds, st, ma, L.items, L.plans);
    else
        hipLaunchKernelGGL(k_conv_fixed_multi_f64<512>, dim3((unsigned)L.nitems), dim3(L.block),
                           L.lds, st, ma, L.items, L.plans);
    return hipGetLastError();
}
void init_kernels_fixed_conv_multi_f64() {
    detail::allow_big_lds(k_conv_fixed_multi_f64<512>);
    detail::allow_big_lds(k_conv_fixed_multi_f64<1024>);
}
}  // namespace cfft

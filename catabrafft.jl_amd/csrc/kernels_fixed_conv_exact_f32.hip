// kernels_fixed_conv_exact_f32.hip -- fixed fused convolutions (fixed_conv.h) of the lengths n - 1 of
// short primes n, in F32: alone, and the work-list kernel in which an item runs the body of its
// plan's length.
#include "fixed_conv.h"

namespace cfft {
#define CFFT_CONV(...) rows.push_back(FixedConvOf<float, Rad<__VA_ARGS__>>::row(true));
void fixed_conv_exact_f32(std::vector<FixedConv>& rows) {
    CFFT_CONV_EXACT_LINES(CFFT_CONV)
}
#undef CFFT_CONV

__global__ void __launch_bounds__(512)
k_conv_exact_multi_f32(MultiArgs ma, const MItem* __restrict__ items,
                      const MPlan* __restrict__ plans) {
    CFFT_DYN_LDS(smem);
    const MItem it = items[blockIdx.x];
    const MPlan* P = plans + it.plan;
    int sgn;
    double scale;
    item_direction(it, P->n, ma, sgn, scale);
    ItemLines<float> lines{ma.in_base, ma.out_base, &it};
#define CFFT_CONV(...)                                                                          \
    case Rad<__VA_ARGS__>::N:                                                                   \
        static_assert(fixed_conv_block<float, Rad<__VA_ARGS__>>() == 512, "short lines");      \
        fixed_conv_body<float, Rad<__VA_ARGS__>>(                                              \
            smem, lines, it.count, P->n, P->C, P->Ls, P->mode, sgn, scale, P->perm, P->iperm,   \
            (const V_t<float>*)P->chirp, (const V_t<float>*)P->K, (const V_t<float>*)P->line.tw); \
        break;
    switch (P->L) {
        CFFT_CONV_EXACT_LINES(CFFT_CONV)
        default: break;
    }
}

hipError_t conv_exact_multi_f32(const MultiLaunch& L, const MultiArgs& ma, hipStream_t st) {
    hipLaunchKernelGGL(k_conv_exact_multi_f32, dim3((unsigned)L.nitems), dim3(L.block), L.lds, st, ma,
                       L.items, L.plans);
    return hipGetLastError();
}
void init_kernels_fixed_conv_exact_f32() { detail::allow_big_lds(k_conv_exact_multi_f32); }
}  // namespace cfft

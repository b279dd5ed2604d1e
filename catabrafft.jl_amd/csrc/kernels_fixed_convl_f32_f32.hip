// kernels_fixed_convl_f32_f32.hip -- large convolutions over fixed lines (fixed_convl.h): data in
// F32, convolution in F32; alone, and as the work-list kernels in which an item runs the body of
// its plan's line.
#include "fixed_convl.h"

namespace cfft {
#define CFFT_ROW(QA, QB) rows.push_back(FixedConvLOf<float, float, QA, QB>::row());
void fixed_convl_f32_f32(std::vector<FixedConvL>& rows) { CFFT_CONVL_LINES(CFFT_ROW) }

// Block: 512 or 1024, the most threads of the lines' workgroups (convl_block).
template <int Phase, int Block>
__global__ void __launch_bounds__(Block)
k_convl_fixed_multi_f32_f32(MultiArgs ma, const MItem* __restrict__ items,
                            const MPlan* __restrict__ plans) {
    CFFT_DYN_LDS(smem);
    const MItem it = items[xcd_item()];
    const MPlan* P = plans + it.plan;
    int sgn;
    double scale;
    item_direction(it, P->n, ma, sgn, scale);
    const ConvLArgs a = convl_args_of(*P, sgn, scale);
    const int so = (it.flags >> kSelOutShift) & 15, si = it.flags & kSelInMask;
    V_t<float>* const dc = reinterpret_cast<V_t<float>*>(it.dc);
#define CFFT_CASE(QA, QB)                                                                       \
    case QA::N:                                                                                 \
        if constexpr (Phase == 0 && convl_block<float>(convl_threads<QA>()) == Block)                   \
            fixed_convl_a_body<float, float, QA>(                                                  \
                smem, a, it.count, mptr<const V_t<float>>(it.in, si, ma.in_base, ma.out_base),    \
                mptr<V_t<float>>(it.out, so, ma.in_base, ma.out_base), dc,                        \
                (const V_t<float>*)P->la.tw);                                                     \
        if constexpr (Phase == 1 && convl_block<float>(convl_threads<QB>()) == Block)                   \
            fixed_convl_ba_body<float, QB>(                                                       \
                smem, a, it.count, mptr<const V_t<float>>(it.in, si, ma.in_base, ma.out_base),    \
                mptr<V_t<float>>(it.out, so, ma.in_base, ma.out_base), dc,                        \
                (const V_t<float>*)P->lb.tw);                                                     \
        if constexpr (Phase == 2 && convl_block<float>(convl_threads<QB>()) == Block)                   \
            fixed_convl_c_body<float, float, QB>(                                                  \
                smem, a, it.count, mptr<const V_t<float>>(it.in, si, ma.in_base, ma.out_base),    \
                mptr<V_t<float>>(it.out, so, ma.in_base, ma.out_base), dc,                        \
                (const V_t<float>*)P->line.tw);                                                   \
        break;
    switch (Phase == 1 ? P->N2 : P->N1) {
        CFFT_CONVL_LINES(CFFT_CASE)
        default: break;
    }
}

template <int Phase>
static hipError_t launch_f32_f32(const MultiLaunch& L, const MultiArgs& ma, hipStream_t st) {
    if (L.block <= 512)
        hipLaunchKernelGGL((k_convl_fixed_multi_f32_f32<Phase, 512>), dim3((unsigned)L.nitems),
                           dim3(L.block), L.lds, st, ma, L.items, L.plans);
    else
        hipLaunchKernelGGL((k_convl_fixed_multi_f32_f32<Phase, 1024>), dim3((unsigned)L.nitems),
                           dim3(L.block), L.lds, st, ma, L.items, L.plans);
    return hipGetLastError();
}
hipError_t convl_fixed_multi_f32_f32(const MultiLaunch& L, const MultiArgs& ma, hipStream_t st) {
    switch ((MultiKernel)L.kernel) {
        case MultiKernel::ConvFA: return launch_f32_f32<0>(L, ma, st);
        case MultiKernel::ConvFBA: return launch_f32_f32<1>(L, ma, st);
        default: return launch_f32_f32<2>(L, ma, st);
    }
}
void init_kernels_fixed_convl_multi_f32_f32() {
    detail::allow_big_lds(k_convl_fixed_multi_f32_f32<0, 512>);
    detail::allow_big_lds(k_convl_fixed_multi_f32_f32<0, 1024>);
    detail::allow_big_lds(k_convl_fixed_multi_f32_f32<1, 512>);
    detail::allow_big_lds(k_convl_fixed_multi_f32_f32<1, 1024>);
    detail::allow_big_lds(k_convl_fixed_multi_f32_f32<2, 512>);
    detail::allow_big_lds(k_convl_fixed_multi_f32_f32<2, 1024>);
}
}  // namespace cfft

// kernels_fixed_conv_f32.hip -- fixed fused convolutions (fixed_conv.h) in F32.
#include "fixed_conv.h"

namespace cfft {
#define CFFT_CONV(...) rows.push_back(FixedConvOf<float, Rad<__VA_ARGS__>>::row());
void fixed_conv_f32(std::vector<FixedConv>& rows) {
    CFFT_CONV_LINES(CFFT_CONV)
}
}  // namespace cfft

// kernels_fixed_conv_f64.hip -- fixed fused convolutions (fixed_conv.h) in F64.
#include "fixed_conv.h"

namespace cfft {
#define CFFT_CONV(...) rows.push_back(FixedConvOf<double, Rad<__VA_ARGS__>>::row());
void fixed_conv_f64(std::vector<FixedConv>& rows) {
    CFFT_CONV_LINES_F64(CFFT_CONV)
}
}  // namespace cfft

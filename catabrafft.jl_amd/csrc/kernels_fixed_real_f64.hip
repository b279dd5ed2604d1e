// kernels_fixed_real_f64.hip -- real-input four-step passes on fixed lines (fixed_real.h) in F64.
#include "fixed_real.h"

namespace cfft {
#ifdef CFFT_EMU_LANES
#define CFFT_LINES CFFT_FS_LINES_FEW
#else
#define CFFT_LINES CFFT_FS_LINES
#endif
#define CFFT_FS(...) rows.push_back(FixedRealOf<double, Rad<__VA_ARGS__>>::entry());
void fixed_real_f64(std::vector<FixedReal>& rows) {
    CFFT_LINES(CFFT_FS)
}
}  // namespace cfft

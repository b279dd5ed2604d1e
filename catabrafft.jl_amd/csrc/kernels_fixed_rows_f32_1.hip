// kernels_fixed_rows_f32_1.hip -- part 1 of the fixed-line rows kernels (fixed_rows.h) in F32.
#include "fixed_rows.h"

namespace cfft {
#ifdef CFFT_EMU_LANES
#define CFFT_LINES(X)
#else
#define CFFT_LINES CFFT_ROW_LINES_1
#endif
#define CFFT_ROW(...) rows.push_back(FixedRowOf<float, Rad<__VA_ARGS__>>::row());
void fixed_rows_f32_1(std::vector<FixedRow>& rows) {
    (void)rows;
    CFFT_LINES(CFFT_ROW)
}
}  // namespace cfft

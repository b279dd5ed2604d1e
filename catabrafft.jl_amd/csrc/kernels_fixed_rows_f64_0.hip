// kernels_fixed_rows_f64_0.hip -- part 0 of the fixed-line rows kernels (fixed_rows.h) in F64.
#include "fixed_rows.h"

namespace cfft {
#ifdef CFFT_EMU_LANES
#define CFFT_LINES CFFT_ROW_LINES_FEW
#else
#define CFFT_LINES CFFT_ROW_LINES_0
#endif
#define CFFT_ROW(...) rows.push_back(FixedRowOf<double, Rad<__VA_ARGS__>>::row());
void fixed_rows_f64_0(std::vector<FixedRow>& rows) {
    (void)rows;
    CFFT_LINES(CFFT_ROW)
}
}  // namespace cfft

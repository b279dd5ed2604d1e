// kernels_fixed_fs_f32.hip -- fixed four-step passes (fixed_fs.h) with T = float and lines stored
// as float2.
#include "fixed_fs.h"

namespace cfft {
#ifdef CFFT_EMU_LANES
#define CFFT_LINES CFFT_FS_LINES_FEW
#define CFFT_STRIDED CFFT_STRIDED_LINES_FEW
#else
#define CFFT_LINES CFFT_FS_LINES
#define CFFT_STRIDED CFFT_STRIDED_LINES
#endif
#define CFFT_FS(...) rows.push_back(FixedFsOf<float, float2, Rad<__VA_ARGS__>>::entry());
#define CFFT_B(...) rows.push_back(FixedFsOf<float, float2, Rad<__VA_ARGS__>>::strided_entry());
void fixed_fs_f32(std::vector<FixedFs>& rows) {
    CFFT_LINES(CFFT_FS)
    CFFT_STRIDED(CFFT_B)
}
}  // namespace cfft

// kernels_fixed_fs_pair.hip -- fixed four-step passes (fixed_fs.h) with T = f2p and lines stored
// as float2.
#include "fixed_fs.h"

namespace cfft {
#ifdef CFFT_EMU_LANES
#define CFFT_LINES CFFT_FS_LINES_FEW
#else
#define CFFT_LINES CFFT_FS_LINES
#endif
#define CFFT_FS(...) rows.push_back(FixedFsOf<f2p, float2, Rad<__VA_ARGS__>>::entry());
void fixed_fs_pair(std::vector<FixedFs>& rows) {
    CFFT_LINES(CFFT_FS)
}
}  // namespace cfft

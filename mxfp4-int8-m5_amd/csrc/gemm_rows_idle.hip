// The larger tiles of gemm_rows.hip for launches that leave CUs idle: 32x32x32 MFMAs.
#include "gemm_tile.h"

namespace scmx {

void launch_rows_idle(const GemmArgs& a, int bmode, int tile, hipStream_t s) {
    const int rows256 = (a.M + 255) / 256, rows128 = (a.M + 127) / 128;
    switch (tile) {
        case 0: return launch_tile<256, 256, 64, 2, 4, 1, 2, false, false, 1, 0, 32>(a, bmode, rows256, s);
        case 1: return launch_tile<256, 128, 128, 4, 2, 1, 3, false, false, 1, 0, 32>(a, bmode, rows256, s);
        case 2: return launch_tile<128, 128, 128, 4, 2, 1, 3, false, false, 1, 0, 32>(a, bmode, rows128, s);
        default: return launch_tile<128, 64, 128, 4, 2, 4, 2, false, false, 1, 0, 32>(a, bmode, rows128, s);
    }
}

}  // namespace scmx

// The dense GEMM's tiles that read activations by rows (ROW_TILES in gemm.hip, by their index there).
#include "gemm_tile.h"

namespace scmx {

// As with blocked activations (gemm_blocked.hip) a launch that leaves CUs idle multiplies with 32x32x32.  Time with
// 16x16x64 over that with 32x32x32, same tile, geometric mean up to three quarters of a tile per CU / above, 104
// problems: 256x256 1.04 / 0.98, 256x128 1.05 / 0.97, 128x128 1.03 / 0.98, 128x64 1.02 / 0.99 (896 x 12288 at 5824 rows
// 85.5 -> 79.5 us); the tiles with K groups 0.99.
void launch_rows(const GemmArgs& a, int bmode, int tile, hipStream_t s) {
    const int rows256 = (a.M + 255) / 256, rows128 = (a.M + 127) / 128, rows64 = (a.M + 63) / 64;
    const long long columns = (a.N + (tile == 0 ? 255 : tile == 3 ? 63 : 127)) / (tile == 0 ? 256 : tile == 3 ? 64 : 128);
    if (tile <= 3 && 4 * columns * (tile <= 1 ? rows256 : rows128) <= 3 * device_cus()) return launch_rows_idle(a, bmode, tile, s);
    switch (tile) {
        case 0: return launch_tile<256, 256, 64, 2, 4, 1, 2>(a, bmode, rows256, s);
        case 1: return launch_tile<256, 128, 128, 4, 2, 1, 3>(a, bmode, rows256, s);
        case 2: return launch_tile<128, 128, 128, 4, 2, 1, 3>(a, bmode, rows128, s);
        case 3: return launch_tile<128, 64, 128, 4, 2, 4>(a, bmode, rows128, s);
        case 5: return launch_tile<64, 64, 128, 2, 2, 1, 2, false, false, 2>(a, bmode, rows64, s);
        case 6: return launch_tile<64, 32, 128, 2, 1, 1, 2, false, false, 4>(a, bmode, rows64, s);
        default: return launch_tile<64, 64, 128, 2, 2, 3>(a, bmode, rows64, s);
    }
}

}  // namespace scmx

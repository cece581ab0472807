// The dense GEMM's tiles that read blocked activations (BLOCKED_TILES in gemm.hip, by their index there).
#include "gemm_tile.h"

namespace scmx {

// A launch that leaves CUs idle is far from the power limit that 16x16x64 MFMAs were chosen for (gemm_tile.h), and
// 32x32x32 takes half the instructions.  Eight waves on 256x128, time with 16x16x64 over that with 32x32x32, geometric
// mean by tiles on 256 CUs: up to 64 1.08, 65 ... 128 1.07, 129 ... 160 1.05, 161 ... 192 1.01, 193 and more 0.99 (4096
// x 12288 at 1280 rows, 160 tiles, 74.4 -> 71.0 us); table decode, which the vector ALU bounds, at every count 1.03 (40
// problems; 6144 x 4864 at 1408 rows 138.6 -> 133.8).  256x256 is a tile for one wave that leaves CUs idle; with
// 16x16x64 its registers hold one buffer of activations less (1.05 ... 1.2 times slower).
void launch_blocked(const GemmArgs& a, int bmode, int tile, hipStream_t s) {
    const int rows256 = (a.M + 255) / 256, cus = device_cus();
    switch (tile) {
        case 0: return launch_tile<256, 128, 64, 4, 1, 2, 2, false, false, 1, 1, 16, FP4_MODES>(a, bmode, rows256, s);
        case 1: return launch_tile<256, 256, 64, 4, 2, 1, 2, false, false, 1, 1, 32, FP4_MODES>(a, bmode, rows256, s);
        case 2:
        case 3:
            if (bmode == B_PACKED_GENERIC || 8LL * rows256 * ((a.N + 127) / 128) <= 5 * cus)
                return launch_tile<256, 128, 128, 8, 1, 1, 2, false, false, 1, 1, 32, PACKED_MODES>(a, bmode, rows256, s);
            return launch_tile<256, 128, 128, 8, 1, 1, 2, false, false, 1, 1, 16, FP4_MODES>(a, bmode, rows256, s);
        case 4: return launch_tile<256, 64, 128, 8, 1, 1, 2, false, false, 1, 1, 16, PACKED_MODES>(a, bmode, rows256, s);
        case 5: return launch_tile<128, 64, 128, 4, 1, 2, 2, false, false, 1, 1, 16, PACKED_MODES>(a, bmode, (a.M + 127) / 128, s);
        default: return launch_tile<64, 64, 128, 2, 2, 2, 2, false, false, 1, 1, 16, PACKED_MODES>(a, bmode, (a.M + 63) / 64, s);
    }
}

}  // namespace scmx

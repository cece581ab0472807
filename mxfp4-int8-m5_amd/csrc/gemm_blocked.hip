// The dense GEMM's tiles that read blocked activations (BLOCKED_TILES in gemm.hip, by their index there).
#include "gemm_tile.h"

namespace scmx {

void launch_blocked(const GemmArgs& a, int bmode, int tile, hipStream_t s) {
    switch (tile) {
        case 0: return launch_tile<256, 128, 64, 4, 1, 2, 2, false, false, 1, 1, 16, FP4_MODES>(a, bmode, (a.M + 255) / 256, s);
        case 1: return launch_tile<256, 128, 128, 8, 1, 1, 2, false, false, 1, 1, 16, PACKED_MODES>(a, bmode, (a.M + 255) / 256, s);
        case 2: return launch_tile<256, 64, 128, 8, 1, 1, 2, false, false, 1, 1, 16, PACKED_MODES>(a, bmode, (a.M + 255) / 256, s);
        case 3: return launch_tile<128, 64, 128, 4, 1, 2, 2, false, false, 1, 1, 16, PACKED_MODES>(a, bmode, (a.M + 127) / 128, s);
        default: return launch_tile<64, 64, 128, 2, 2, 2, 2, false, false, 1, 1, 16, PACKED_MODES>(a, bmode, (a.M + 63) / 64, s);
    }
}

}  // namespace scmx

// The grouped GEMM's tiles (expert segments of a sorted batch) and which of them a launch takes.
#include "gemm_tile.h"

namespace scmx {

void launch_grouped(const GemmArgs& a, int bmode, int tm, hipStream_t s) {
    const int max_tiles = (a.M + tm - 1) / tm + a.n_experts;   // e2e/sc_moe.py:155
    // 256-row tiles, activations staged in LDS, from 256 rows per expert on: the fewest LDS bytes per MFMA.  Below that 128-row
    // ones (two to a slot where the segments are cut into 256): workgroups of four waves whose activation fragments come
    // straight from the gathered rows, two of them on a CU.  64 experts of 2048 x 2048 / 2048 x 1024, 125 rows each: 67 + 37
    // us for 86 + 51 (64-row tiles 74 + 41); 375 rows each 155 + 83 for 153 + 85.
    if (tm == 256 && a.M / a.n_experts >= 256 && (a.N % 256 == 0 || a.N >= 1024))
        launch_tile<256, 256, 64, 2, 4, 1, 2, true>(a, bmode, max_tiles, s);
    else if (tm >= 128) {
        GemmArgs b = a;
        b.sub_log2 = tm == 256 ? 1 : 0;
        launch_tile<128, 128, 128, 4, 1, 2, 2, false, false, 1, 2>(b, bmode, max_tiles << b.sub_log2, s);
    }
    else if (bmode != B_INT8 && bmode != B_PACKED_GENERIC && a.K % 256 == 0 && a.N % 128 == 0 &&
             reinterpret_cast<uintptr_t>(a.bcodes) % 8 == 0) {
        // Few rows per expert: the pass streams the expert weights, and what it pays per weight is the staging.  The packed
        // tile writes and reads half the weight bytes in LDS, its waves sit side by side along N (every fragment is decoded
        // once) and two or three workgroups share a CU.  Its lanes read the block codes of two K steps with one aligned
        // load of 2, 4 or 8 bytes, hence the conditions on K and on the pointer.  Bound by the vector ALU: 64 codes a lane
        // and step to decode (10 instructions per 8) beside 8 MFMAs.  Skewed routing, 70 rows an expert on average, us packed
        // / staged INT8: 257 experts of 1024 x 2048, published format 100.5 / 108, 16-blocks 104 / 117, MXFP4 105.5 / 114,
        // e2m1/B16/M1..10 111 / 120; 64 of 2048 x 1024 30.4 / 31.2, 30.5 / 32.1, 30.9 / 32.0, 31.1 / 33.2.
        // A reduction of four steps at most is mostly prologue and epilogue: eight waves on 256 columns, four a SIMD, share
        // them.  257 experts of 2048 x 512, 70 rows, us 256 / 128 columns: 63.3 / 67.2, 61.6 / 69.9, 64.6 / 70.1, 64.9 / 71.0;
        // 64 of 4096 x 256 23.5 / 24.6; K = 768 the other way round, 29.9 / 26.5.
        if (a.K <= 512 && a.N % 256 == 0)
            launch_tile<64, 256, 128, 1, 8, 4, 2, false, true, 1, 0, 32, FP4_MODES>(a, bmode, max_tiles, s);
        else
            launch_tile<64, 128, 128, 1, 4, 2, 2, false, true, 1, 0, 32, FP4_MODES>(a, bmode, max_tiles, s);
    } else
        launch_tile<64, 128, 128, 2, 4>(a, bmode, max_tiles, s);
}

}  // namespace scmx

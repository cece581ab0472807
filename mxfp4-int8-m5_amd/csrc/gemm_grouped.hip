// The grouped GEMM's tiles (expert segments of a sorted batch) and which of them a launch takes.
#include "gemm_tile.h"

namespace scmx {

// 128x128 tiles, one or (sub_log2) two to a slot: four waves whose activation fragments come straight from the gathered
// rows, two workgroups a CU; eight waves on activations staged in LDS where there is less than a tile for every other
// CU (published format, 95 rows: 8 experts of 2048 x 4096 24.0 / 21.9 us, 4096 x 2048 24.1 / 26.8; 16 of 768 x 1024 8.6
// / 8.1).  Table decode does not fit the registers of four waves and stays with eight up to four tiles a CU (60 rows, 8
// experts of 4096 x 2048 42.9 / 28.5; 64 of 2048 x 1024 66.9 / 72.2).
static void launch_128(const GemmArgs& a, int bmode, int slots, hipStream_t s) {
    const int row_tiles = slots << a.sub_log2;
    const long long tiles = (long long)a.n_experts * ((a.N + 127) / 128), cus = device_cus();
    if (tiles <= cus / 2 || (bmode == B_PACKED_GENERIC && tiles < 4 * cus))
        launch_tile<128, 128, 128, 4, 2, 1, 3, false, false, 1, 0, 32>(a, bmode, row_tiles, s);
    else
        launch_tile<128, 128, 128, 4, 1, 2, 2, false, false, 1, 2>(a, bmode, row_tiles, s);
}

// A 256-row slot goes to one 256x256 tile (the fewest LDS bytes per MFMA, 16-row blocks past the segment skipped), one
// 256x128 tile or two of 128x128.  What decides is how the tiles fill the chip.  `tiles` = the 256x256 ones if no
// expert had more than 256 rows; real counts are uneven: at 100 rows on average hardly any has, at 180 a quarter more.
// Skewed routing, us 256x256 / 256x128 / pairs of 128x128, published format unless named:
// - two tiles a CU and more, or 256 rows and more: 256x256.  64 experts of 2048 x 2048, 128 / 200 rows 89.9 / 92.8 /
//   92.9, 105 / 100 / 115; 257 of 1024 x 2048 152 / 178 / 193, 195 / 213 / 240.
// - one wave that nearly fills the chip, under 128 rows: 256x256.  64 of 1024 x 1024, 100 rows 22.2 / 24.4 / 26.6; 16
//   of 4096 x 4096 60.7 / 68.6 / 76.3.
// - fewer tiles than two a CU, up to 200 rows: pairs, spread over more of the chip (32 of 1024 x 2048, 140 rows 38.8 /
//   35.9 / 32.2; 64 of 1024 x 1024 34.9 / 32.6 / 31.3; 48 of 1536 x 2048 68.9 / 57.2 / 59.3), on long reductions that
//   fill a wave 256x128 (32 of 2048 x 2048 59.1 / 55.4 / 56.4; 16 of 4096 x 4096 90.7 / 92.0 / 95.5); beyond 200 rows
//   256x128: 32 of 2048 x 2048, 220 rows 68.3 / 60.3 / 70.5; 64 of 512 x 2048 39.9 / 39.4 / 43.9.
// - a handful of tiles: pairs (16 of 768 x 1024, 100 ... 180 rows - / 11 / 8.6).
// INT8 weights are cheaper to stage, so that 256x256 loses less: pairs only up to 140 rows and half a chip (16 of
// 2048 x 2048, 140 rows 33.1 / 36.5 / 30.1; 32 of 1024 x 2048, 180 rows 34.1 / 38.5 / 38.1).  Table decode: 256x128, a
// row group's decode shared by the most rows a wave can hold (64 of 2048 x 2048, 128 rows 182 / 154 / 241; 8 of
// 2048 x 4096, 95 rows 117 / 55 / 85).
static void launch_256(const GemmArgs& a, int bmode, int slots, hipStream_t s) {
    const bool wide = a.N % 256 == 0 || a.N >= 1024, fp4 = bmode != B_INT8 && bmode != B_PACKED_GENERIC;
    const int rows = a.M / a.n_experts;
    const long long tiles = (long long)a.n_experts * ((a.N + 255) / 256), cus = device_cus();
    const bool few = rows < 256 && tiles < 2 * cus, one_wave = tiles > cus / 2 && tiles <= cus;
    const bool pairs = few && (fp4               ? (rows <= 200 && !(one_wave && (rows < 128 || a.K >= 2048))) || tiles <= cus / 4
                               : bmode == B_INT8 ? (rows <= 140 && tiles <= cus / 2) || tiles <= cus / 4
                                                 : false);
    if (pairs) {
        GemmArgs b = a;
        b.sub_log2 = 1;
        launch_128(b, bmode, slots, s);
    } else if (!wide || bmode == B_PACKED_GENERIC || (few && fp4 && !(one_wave && rows < 128))) {
        launch_tile<256, 128, 128, 4, 2, 1, 3, false, false, 1, 0, 32>(a, bmode, slots, s);
    } else if (tiles <= cus && (bmode == B_INT8 || bmode == B_PACKED_B16M)) {
        // CUs idle, no power limit (gemm_tile.h): 32x32x32, 4 per cent faster with INT8 weights, 2 with
        // e2m1/B16/M1..10, level with the other formats (32 of 1024 x 2048, 180 rows 36.8 -> 34.1, 42.1 -> 40.1,
        // published 39.1 -> 38.7)
        launch_tile<256, 256, 64, 2, 4, 1, 2, true, false, 1, 0, 32, 1u << B_INT8 | 1u << B_PACKED_B16M>(a, bmode, slots, s);
    } else {
        launch_tile<256, 256, 64, 2, 4, 1, 2, true, false, 1, 0, 16, ALL_MODES & ~(1u << B_PACKED_GENERIC)>(a, bmode, slots, s);
    }
}

void launch_grouped(const GemmArgs& a, int bmode, int tm, hipStream_t s) {
    const int max_tiles = (a.M + tm - 1) / tm + a.n_experts;   // e2e/sc_moe.py:155
    if (a.blocked)
        // Slots of blocked activations: the dense GEMM's 256x128 tile of four waves, two workgroups a CU, whose waves take
        // the tile's 16-row blocks in turn, so that a slot's missing rows are missing from all four SIMDs.  Bound like the
        // dense tile (matrix pipe 39 per cent busy, vector ALU 36, LDS 46) and by what a tile costs beyond its K loop.
        // Published format, skewed routing, us by rows (launch_256) / from slots: 64 experts of 2048 x 2048, 8000 rows 76.5
        // / 64.7, 24000 159.3 / 131.7; of 2048 x 1024 43.0 / 37.5, 88.2 / 73.5; 257 of 1024 x 2048, 54000 rows 197 / 192.5.
        return launch_tile<256, 128, 64, 4, 1, 2, 2, true, false, 1, 1, 16, FP4_MODES>(a, bmode, max_tiles, s);
    const bool fp4 = bmode != B_INT8 && bmode != B_PACKED_GENERIC;
    if (tm == 256) {
        launch_256(a, bmode, max_tiles, s);
    } else if (tm == 128) {
        launch_128(a, bmode, max_tiles, s);
    } else if (fp4 && a.K % 256 == 0 && a.N % 128 == 0 &&
             reinterpret_cast<uintptr_t>(a.bcodes) % 8 == 0) {
        // Few rows per expert: the pass streams the expert weights, and what it pays per weight is the staging.  The
        // packed tile writes and reads half the weight bytes in LDS, its waves sit side by side along N (every fragment
        // is decoded once) and two or three workgroups share a CU.  Its lanes read the block codes of two K steps with
        // one aligned load of 2, 4 or 8 bytes, hence the conditions on K and on the pointer.  Bound by the vector ALU:
        // 64 codes a lane and step to decode (10 instructions per 8) beside 8 MFMAs.  Skewed routing, 70 rows an expert
        // on average, us packed / staged INT8: 257 experts of 1024 x 2048, published format 100.5 / 108, 16-blocks 104
        // / 117, MXFP4 105.5 / 114, e2m1/B16/M1..10 111 / 120; 64 of 2048 x 1024 30.4 / 31.2, 30.5 / 32.1, 30.9 / 32.0,
        // 31.1 / 33.2.  A reduction of four steps at most is mostly prologue and epilogue: eight waves on 256 columns,
        // four a SIMD, share them.  257 experts of 2048 x 512, 70 rows, us 256 / 128 columns: 63.3 / 67.2, 61.6 / 69.9,
        // 64.6 / 70.1, 64.9 / 71.0; 64 of 4096 x 256 23.5 / 24.6; K = 768 the other way round, 29.9 / 26.5.
        // The four-wave tile leaves out the MFMAs and LDS traffic of a half without rows: 257 experts of 1024 x 2048, 70
        // rows each 115 -> 113 us (e2m1/B16/M1..10), 104 -> 102 (published), 25 rows 67.6 -> 64.3, 4 rows 54.3 -> 51.0;
        // level at K = 1024.  Eight waves have no registers for it (63 -> 73).
        if (a.K <= 512 && a.N % 256 == 0)
            launch_tile<64, 256, 128, 1, 8, 4, 2, false, true, 1, 0, 32, FP4_MODES>(a, bmode, max_tiles, s);
        else
            launch_tile<64, 128, 128, 1, 4, 2, 2, true, true, 1, 0, 32, FP4_MODES>(a, bmode, max_tiles, s);
    } else
        launch_tile<64, 128, 128, 2, 4, 4>(a, bmode, max_tiles, s);
}

}  // namespace scmx

// What the GEMM kernels are launched with: the dense and grouped tiles (gemm_*.hip) and the few-row kernel (gemm_skinny.hip).
#pragma once
#include "scmx_common.h"

namespace scmx {

struct GemmArgs {
    const int8_t* xq;        // activations INT8 [rows, K] (blocked: 32 x 32 blocks in MFMA operand order, see AD)
    const float* xscale;     // [rows]
    const int32_t* gather;   // optional: logical row r reads xq[gather[r]], xscale[gather[r]]
    const uint32_t* codes;   // packed weights [E][N*K/8]
    const uint8_t* bcodes;   // [E][N][bc_row_bytes]
    const int8_t* wq;        // INT8 weights [E*N, K] when the tile is fed from unpacked weights
    const float* wscale;     // [E][N]
    const uint16_t* res;     // [M, N] residual (epilogue 2)
    void* out;
    int M, N, K;             // M = number of logical rows (R for the grouped GEMM)
    int bc_row_bytes;
    int epi;
    const int32_t* off;      // grouped: expert segment offsets [E+1]; dense: NULL
    const uint16_t* silu;    // SwiGLU epilogue: the table of the rounded sigmoid
    const int32_t* tstart;   // grouped: first row tile of each expert [E+1]
    int n_experts;
    int sub_log2;            // grouped: a segment's row tile is 1 << sub_log2 of the kernel's
    int blocked;             // dense: xq is in the blocked layout (FEW_ROWS: and the few-row kernel takes it)
    DevFormat fmt;
};

// B_PACKED_DEFAULT / B_PACKED_B16: the published codebook with power-of-two shifts on 32- / 16-element blocks (decoded
// with the FP4 conversion); B_PACKED_B16M: that codebook on 16-element blocks with 4-bit codes for consecutive integer
// multipliers (FP4 conversion, then one fused multiply-add); B_PACKED_GENERIC: any member of the format family (table
// decode).
// B_PACKED_E8M0: a standard MXFP4 tensor in place -- B_PACKED_DEFAULT's decode with the block's shift taken from its
// E8M0 byte minus the row's lowest one (which the row scale carries).
enum { FEW_ROWS = 2 };   // GemmArgs::blocked
enum { B_INT8 = 0, B_PACKED_DEFAULT = 1, B_PACKED_GENERIC = 2, B_PACKED_B16 = 3, B_PACKED_B16M = 4, B_PACKED_E8M0 = 5 };

constexpr int SKINNY_MAX_ROWS = 128;
// The few-row kernel's time (us) on a dense problem of up to SKINNY_MAX_ROWS rows, activations in the blocked layout.
float skinny_time(int M, int N, int K, int cus, int most = SKINNY_MAX_ROWS / 16);
void launch_skinny(const GemmArgs& a, int bmode, hipStream_t s);
void launch_rows(const GemmArgs& a, int bmode, int tile, hipStream_t s);
void launch_rows_idle(const GemmArgs& a, int bmode, int tile, hipStream_t s);
void launch_blocked(const GemmArgs& a, int bmode, int tile, hipStream_t s);
void launch_grouped(const GemmArgs& a, int bmode, int tm, hipStream_t s);

}  // namespace scmx

// out = x W^T for a few bf16 rows x [M, K] and a bf16 matrix W [N, K]: the output head of a prompt's last token and the
// router of a decode step, the two linears of a model that stay bf16.
//
// Bound: HBM, W is read once.  A tile is 16 rows of W; the eight waves of a workgroup split its columns in turns of 64, so
// that a wave asks for both halves of a 128-byte line of each row together.  Two workgroups per CU walk the tiles, each
// wave's next loads (the next tile's, where a wave's share of a row is one batch) in flight while the current ones are
// multiplied: a workgroup per tile spent most of its time on its first loads (151936 x 896: 107 us against 46).  The
// matrix instruction does the products at up to 16 rows of x for the price of one (columns beyond M repeat row 0 and are
// dropped), sums in float32; the waves' partial sums meet in LDS in wave order, in two buffers by turns: one barrier a tile.
#include <algorithm>

#include "scmx_common.h"

namespace scmx {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int LB_WAVES = 8, LB_CHUNK = 64, LB_DEPTH = 4;   // chunks of 64 columns, up to four per batch of loads

// DEPTH: chunks per wave and batch.  ONE: a row is one batch, whose fragments of x stay in registers.
template <int DEPTH, bool ONE>
__global__ __launch_bounds__(LB_WAVES * 64, 4) void linear_bf16_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                                       uint16_t* __restrict__ out, int M, int N, int K) {
    __shared__ f32x4 part[2][LB_WAVES][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int tiles = N / 16 + (N % 16 != 0), chunks = K / LB_CHUNK;
    const int batches = ONE ? 1 : (chunks + LB_WAVES * DEPTH - 1) / (LB_WAVES * DEPTH);
    // matrix operands: lane holds 8 consecutive columns 8 g .. of row r (of W; of x)
    const uint16_t* xp = x + size_t(r < M ? r : 0) * K + 8 * g;
    auto load = [&](const uint16_t* p, int b, u32x4 (&v)[2 * DEPTH]) {
#pragma unroll
        for (int i = 0; i < DEPTH; ++i) {   // chunks beyond the row repeat its last one and are not multiplied
            const size_t col = size_t(min((b * DEPTH + i) * LB_WAVES + wave, chunks - 1)) * LB_CHUNK;
            v[2 * i] = *reinterpret_cast<const u32x4*>(p + col);
            v[2 * i + 1] = *reinterpret_cast<const u32x4*>(p + col + 32);
        }
    };
    auto weights = [&](int t) { return w + size_t(min(t * 16 + r, N - 1)) * K + 8 * g; };
    u32x4 xv[2 * DEPTH], cur[2 * DEPTH], nxt[2 * DEPTH];
    if (ONE) load(xp, 0, xv);
    load(weights(int(blockIdx.x)), 0, cur);
    int turn = 0;
    for (int t = int(blockIdx.x); t < tiles; t += int(gridDim.x), turn ^= 1) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int b = 0; b < batches; ++b) {
            const bool last = b + 1 == batches;
            if (!ONE) load(xp, b, xv);
            if (!last || tiles - t > int(gridDim.x)) load(weights(last ? t + int(gridDim.x) : t), last ? 0 : b + 1, nxt);
#pragma unroll
            for (int i = 0; i < DEPTH; ++i)
                if ((b * DEPTH + i) * LB_WAVES + wave < chunks) {   // the same for the whole wave
#pragma unroll
                    for (int s = 0; s < 2; ++s)
                        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, cur[2 * i + s]),
                                                                      __builtin_bit_cast(bf16x8, xv[2 * i + s]), acc, 0, 0, 0);
                }
#pragma unroll
            for (int i = 0; i < 2 * DEPTH; ++i) cur[i] = nxt[i];
        }
        part[turn][wave][lane] = acc;
        __syncthreads();   // the other buffer is written again only behind the next tile's barrier
        // register i of lane (r, g) is row 16 t + 4 g + i of W times row r of x
        const int row = int(threadIdx.x) >> 4, j = int(threadIdx.x) & 15, n = t * 16 + j;
        if (row < M && n < N) {
            float s = 0.0f;
#pragma unroll
            for (int v = 0; v < LB_WAVES; ++v) s += part[turn][v][(j >> 2) * 16 + row][j & 3];
            out[size_t(row) * N + n] = f32_to_bf16(s);
        }
    }
}

}  // namespace scmx

using namespace scmx;

extern "C" int scmx_linear_bf16(const uint16_t* x, const uint16_t* w, uint16_t* out, int M, int N, int K, void* stream) {
    if (!x || !w || !out || (uintptr_t(x) | uintptr_t(w)) % 16) {
        set_error("linear_bf16: null or misaligned pointer (x and w: 16 bytes)");
        return SCMX_ERR_ARG;
    }
    if (M < 0 || M > 16 || N < 1 || N > 0x7FFFFFF0 || K < LB_CHUNK || K % LB_CHUNK) {
        set_error("linear_bf16: need 0 <= M <= 16, N >= 1 and K %% %d == 0 (M=%d N=%d K=%d)", LB_CHUNK, M, N, K);
        return SCMX_ERR_ARG;
    }
    if (M == 0) return SCMX_OK;
    const unsigned tiles = (unsigned(N) + 15u) / 16u;
    const dim3 grid(std::min(tiles, 2u * unsigned(device_cus()))), block(LB_WAVES * 64);
    hipStream_t st = (hipStream_t)stream;
    const int turns = (K / LB_CHUNK + LB_WAVES - 1) / LB_WAVES;   // chunks of a row per wave
    if (turns == 1) linear_bf16_kernel<1, true><<<grid, block, 0, st>>>(x, w, out, M, N, K);
    else if (turns == 2) linear_bf16_kernel<2, true><<<grid, block, 0, st>>>(x, w, out, M, N, K);
    else if (turns == 3) linear_bf16_kernel<3, true><<<grid, block, 0, st>>>(x, w, out, M, N, K);
    else if (turns == 4) linear_bf16_kernel<4, true><<<grid, block, 0, st>>>(x, w, out, M, N, K);
    else linear_bf16_kernel<4, false><<<grid, block, 0, st>>>(x, w, out, M, N, K);
    return check_launch("linear_bf16");
}

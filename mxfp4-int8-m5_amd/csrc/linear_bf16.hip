// out = x W^T for a few bf16 rows x [M, K] and a bf16 matrix W [N, K]: the output head of a prompt's last token and the
// router of a decode step, the two linears of a model that stay bf16.
//
// Bound: HBM, W is read once.  A tile is 16 rows of W; the eight waves of a workgroup split its columns in turns of 64, so
// that a wave asks for both halves of a 128-byte line of each row together.  Two workgroups per CU walk the tiles, each
// wave's next loads (the next tile's, where a wave's share of a row is one batch) in flight while the current ones are
// multiplied: a workgroup per tile spent most of its time on its first loads (151936 x 896: 107 us against 50).  The
// matrix instruction does the products at up to 16 rows of x for the price of one (columns beyond M repeat row 0 and are
// dropped), sums in float32; the waves' partial sums meet in LDS in wave order, in two buffers by turns: one barrier a tile.
//
// A row that does not fill its batches (RAGGED) is read through a buffer that ends with it: the chunks beyond cost neither
// traffic nor a branch.  Loading them from the row's end cost as much as real ones, and with batches of four chunks a wave
// where three do one of two batches was nearly empty.  One row, weights from HBM, us before / after: 50304 x 576 17.5 / 14.2,
// x 1088 23.8 / 20.6, x 2304 67.0 / 47.9, x 3072 70.3 / 56.4, 32000 x 5120 67.6 / 63.1, 151936 x 2560 197.5 / 140.9.  Rows that
// fill them keep plain loads, which take 4 % less there (57344 x 2048: 43.1 us, through a buffer 44.8).
#include <algorithm>
#include <type_traits>

#include "scmx_common.h"

namespace scmx {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int LB_WAVES = 8, LB_CHUNK = 64, LB_DEPTH = 4;   // chunks of 64 columns, up to four per batch of loads

// DEPTH: chunks per wave and batch.  ONE: a row is one batch, whose fragments of x stay in registers.
template <int DEPTH, bool ONE, bool RAGGED>
__global__ __launch_bounds__(LB_WAVES * 64, 4) void linear_bf16_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                                       uint16_t* __restrict__ out, int M, int N, int K) {
    __shared__ f32x4 part[2][LB_WAVES][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int tiles = N / 16 + (N % 16 != 0), chunks = K / LB_CHUNK;
    const int batches = ONE ? 1 : (chunks + LB_WAVES * DEPTH - 1) / (LB_WAVES * DEPTH);
    // matrix operands: lane holds 8 consecutive columns 8 g .. of row r (of W; of x); p: `rows` rows.  RAGGED: a buffer, past
    // whose end reads give zeros without touching memory
    auto load = [&](const uint16_t* p, int rows, int row, int b, u32x4 (&v)[2 * DEPTH]) {
        [[maybe_unused]] const __amdgpu_buffer_rsrc_t buf =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p), 0, rows * K * 2, 0x00020000);
#pragma unroll
        for (int i = 0; i < DEPTH; ++i) {   // chunks beyond the row are not multiplied
            const int chunk = (b * DEPTH + i) * LB_WAVES + wave;
            if (RAGGED) {
                const int at = chunk < chunks ? (row * K + chunk * LB_CHUNK + 8 * g) * 2 : 0x7FFFFF00;
                v[2 * i] = __builtin_amdgcn_raw_buffer_load_b128(buf, at, 0, 0);
                v[2 * i + 1] = __builtin_amdgcn_raw_buffer_load_b128(buf, at + 64, 0, 0);
            } else {
                const uint16_t* at = p + size_t(min(row, rows - 1)) * K + size_t(min(chunk, chunks - 1)) * LB_CHUNK + 8 * g;
                v[2 * i] = *reinterpret_cast<const u32x4*>(at);
                v[2 * i + 1] = *reinterpret_cast<const u32x4*>(at + 32);
            }
        }
    };
    auto load_w = [&](int t, int b, u32x4 (&v)[2 * DEPTH]) { load(w + size_t(t) * 16 * K, min(16, N - t * 16), r, b, v); };
    auto load_x = [&](int b, u32x4 (&v)[2 * DEPTH]) { load(x, M, r < M ? r : 0, b, v); };
    u32x4 xv[2 * DEPTH], cur[2 * DEPTH], nxt[2 * DEPTH];
    if (ONE) load_x(0, xv);
    load_w(int(blockIdx.x), 0, cur);
    int turn = 0;
    for (int t = int(blockIdx.x); t < tiles; t += int(gridDim.x), turn ^= 1) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int b = 0; b < batches; ++b) {
            const bool last = b + 1 == batches;
            if (!ONE) load_x(b, xv);
            if (!last || tiles - t > int(gridDim.x)) load_w(last ? t + int(gridDim.x) : t, last ? 0 : b + 1, nxt);
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
    // chunks of a row per wave, in batches as even as can be
    const int turns = (K / LB_CHUNK + LB_WAVES - 1) / LB_WAVES;
    const int batches = (turns + LB_DEPTH - 1) / LB_DEPTH, depth = (turns + batches - 1) / batches;
    const bool ragged = K % (LB_CHUNK * LB_WAVES * depth) != 0 && K <= 1 << 25;   // (16 rows within a buffer's 32-bit offsets)
    auto go = [&](auto d, auto one) {
        constexpr int D = decltype(d)::value;
        constexpr bool ONE = decltype(one)::value;
        if (ragged) linear_bf16_kernel<D, ONE, true><<<grid, block, 0, st>>>(x, w, out, M, N, K);
        else linear_bf16_kernel<D, ONE, false><<<grid, block, 0, st>>>(x, w, out, M, N, K);
    };
    using std::integral_constant;
    if (turns == 1) go(integral_constant<int, 1>{}, std::true_type{});
    else if (turns == 2) go(integral_constant<int, 2>{}, std::true_type{});
    else if (turns == 3) go(integral_constant<int, 3>{}, std::true_type{});
    else if (turns == 4) go(integral_constant<int, 4>{}, std::true_type{});
    else if (depth == 3) go(integral_constant<int, 3>{}, std::false_type{});
    else go(integral_constant<int, 4>{}, std::false_type{});
    return check_launch("linear_bf16");
}

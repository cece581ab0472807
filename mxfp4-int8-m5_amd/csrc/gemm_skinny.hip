// Dense W4A8 GEMM for few activation rows (a short prompt, sequences decoding together): M up to 128.
//
// Such a problem streams the weights once and is over: what it needs is every CU loading at once, not operand reuse.  A
// workgroup owns 16 weight rows and all M activation rows (or, on layers of so few columns that CUs would idle, some of the
// 16-row tiles of them: row_groups); its waves split K (wave w of NW takes the 128-wide steps w,
// w + NW, ...), decode the weights in registers and multiply with v_mfma_i32_16x16x64_i8, weights as the row operand.
// Nothing passes through LDS but the waves' INT32 partial sums at the end, which add up exactly in any order.
//
// Which k a lane's operand bytes stand for is free as long as both operands agree: lane (row r = l % 16, group g = l / 16)
// loads the 16 bytes of codes of weights 32 g ... 32 g + 31 of a step -- one 32-block, or two 16-blocks -- and the 32
// activation bytes of the same k; the first 16 of them are the operand bytes of one MFMA, the other 16 of a second.
// A lane ends with 4 consecutive output columns of one activation row, the unit of the epilogues.
//
// The activations come in the blocked layout: read by rows, the 16 rows of a fragment lie K bytes apart, which for K a
// multiple of 1024 is the same few L2 channels for every workgroup at once (2048 x 2048 at M = 64: 13.2 us by rows, 4.6
// blocked).
#include <type_traits>

#include "gemm_args.h"

namespace scmx {

template <int TILES, int BMODE, int NW, int DW>
__global__ __launch_bounds__(NW * 64) void skinny_kernel(const GemmArgs a) {
    __shared__ v4i part[NW][TILES][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int K = a.K, N = a.N, M = a.M, steps = K / 128, n0 = int(blockIdx.x) * 16;
    const int tile0 = int(blockIdx.y) * TILES;   // first 16-row tile of this workgroup's activation rows
    const size_t wrow = size_t(min(n0 + r, N - 1));
    const uint8_t* cp = reinterpret_cast<const uint8_t*>(a.codes) + wrow * (K / 2) + 16 * g;
    const uint8_t* bp = a.bcodes + wrow * a.bc_row_bytes;
    [[maybe_unused]] const uint32_t rmin = BMODE == B_PACKED_E8M0 ? e8m0_row_min(a.wscale[wrow]) : 0u;
    // activations in the blocked layout (rows padded to whole 32-row blocks): block (m / 32, k / 32), 16-byte halves of k
    const int8_t* ap[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t)   // (a tile past M: any block)
        ap[t] = a.xq + (size_t(min(tile0 + t, (M - 1) / 16) >> 1) * (K / 32) + g) * 1024 + (16 * ((tile0 + t) & 1) + r) * 16;

    struct Weights {
        u32x4 w;
        uint32_t bc;
    };
    struct Acts {
        v4i x[TILES][2];
    };
    auto load_w = [&](Weights& d, int s) {
        if (s >= steps) return;   // wave-uniform
        d.w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(cp + size_t(s) * 64));
        if (BMODE == B_PACKED_DEFAULT) d.bc = bp[s];
        else if (BMODE == B_PACKED_B16) d.bc = bp[2 * s + (g >> 1)];
        else if (BMODE != B_PACKED_GENERIC) d.bc = bp[4 * s + g];
    };
    auto load_x = [&](Acts& d, int s) {
        if (s >= steps) return;
        const size_t at = size_t(s) * 4096;
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            d.x[t][0] = *reinterpret_cast<const v4i*>(ap[t] + at);
            d.x[t][1] = *reinterpret_cast<const v4i*>(ap[t] + at + 512);
        }
    };
    v4i acc[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) acc[t] = v4i{0, 0, 0, 0};
    auto compute = [&](const Weights& d, const Acts& x, int s) {
        uint32_t o[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t w = d.w[j];
            if (BMODE == B_PACKED_DEFAULT) {
                decode_word_fp4(w, fp4_scale((d.bc >> (2 * g)) & 3u), o[2 * j], o[2 * j + 1]);
            } else if (BMODE == B_PACKED_E8M0) {
                decode_word_fp4(w, fp4_scale((d.bc - rmin) & 0x7Fu), o[2 * j], o[2 * j + 1]);
            } else if (BMODE == B_PACKED_B16) {
                decode_word_fp4(w, fp4_scale((d.bc >> (4 * (g & 1) + 2 * (j >> 1))) & 3u), o[2 * j], o[2 * j + 1]);
            } else if (BMODE == B_PACKED_B16M) {
                const _Float16 m = _Float16(float((a.fmt.mult[0] & 0xFFu) + ((d.bc >> (4 * (j >> 1))) & 15u)));
                decode_word_fp4_mul(w, half2_t{m, m}, o[2 * j], o[2 * j + 1]);
            } else {
                const uint32_t blk = uint32_t(128 * s + 32 * g + 8 * j) >> a.fmt.block_log2;
                const BlockLut lut = scaled_lut_mul(a.fmt.lut_lo, a.fmt.lut_hi,
                                                    mult_of(a.fmt, block_code(bp, blk, a.fmt.bc_bits)));
                decode_word(w, lut, o[2 * j], o[2 * j + 1]);
            }
        }
        const v4i w0 = v4i{int(o[0]), int(o[1]), int(o[2]), int(o[3])}, w1 = v4i{int(o[4]), int(o[5]), int(o[6]), int(o[7])};
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w0, x.x[t][0], acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1, x.x[t][1], acc[t], 0, 0, 0);
        }
    };
    // DW steps of weights (from HBM) and two of activations (from the L2) in flight; nothing is requested past the last step
    constexpr int DX = 2;
    Weights wb[DW];
    Acts xb[DX];
#pragma unroll
    for (int u = 0; u < DW; ++u) load_w(wb[u], wave + NW * u);
#pragma unroll
    for (int u = 0; u < DX; ++u) load_x(xb[u], wave + NW * u);
    for (int s0 = wave; s0 < steps; s0 += NW * DW) {
#pragma unroll
        for (int u = 0; u < DW; ++u) {
            const int s = s0 + NW * u;
            if (s < steps) compute(wb[u], xb[u % DX], s);   // wave-uniform
            load_w(wb[u], s + NW * DW);
            load_x(xb[u % DX], s + NW * DX);
        }
    }

    // ---- the waves' partial sums, then the epilogue: one v4i (four columns of one row) per thread and turn ------------
#pragma unroll
    for (int t = 0; t < TILES; ++t) part[wave][t][lane] = acc[t];
    __syncthreads();
    for (int e = threadIdx.x; e < TILES * 64; e += NW * 64) {
        const int t = e >> 6, l = e & 63;
        const int m = 16 * (tile0 + t) + (l & 15), n = n0 + 4 * (l >> 4);
        if (m >= M || n >= N) continue;   // N % 4 == 0
        v4i tot = part[0][t][l];
#pragma unroll
        for (int w = 1; w < NW; ++w) tot += part[w][t][l];
        if (a.epi == SCMX_EPI_I32) {
            *reinterpret_cast<v4i*>(reinterpret_cast<int32_t*>(a.out) + size_t(m) * N + n) = tot;
            continue;
        }
        const float xs = a.xscale[m];
        const f32x4 ws = *reinterpret_cast<const f32x4*>(a.wscale + n);
        float y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = __fmul_rn(__fmul_rn(float(tot[i]), xs), ws[i]);
        uint16_t* out = reinterpret_cast<uint16_t*>(a.out);
        if (a.epi == SCMX_EPI_SWIGLU) {   // rows (g, g, u, u)
            *reinterpret_cast<uint32_t*>(out + size_t(m) * (N / 2) + n / 2) = swiglu_lut2(a.silu, y[0], y[1], y[2], y[3]);
            continue;
        }
        if (a.epi == SCMX_EPI_RES) {
            const u32x2 rr = *reinterpret_cast<const u32x2*>(a.res + size_t(m) * N + n);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float rv = __uint_as_float(i & 1 ? (rr[i >> 1] & 0xFFFF0000u) : (rr[i >> 1] << 16));
                y[i] = __fadd_rn(rv, round_bf16(y[i]));
            }
        }
        *reinterpret_cast<u32x2*>(out + size_t(m) * N + n) = u32x2{f32_to_bf16x2(y[0], y[1]), f32_to_bf16x2(y[2], y[3])};
    }
}

// Groups that the 16-row tiles are cut into, a workgroup each: as many as the CUs that a workgroup per 16 columns leaves idle
// allow.  What a workgroup takes beyond the latency of its loads is its activations through the vector L1 (48 rows of 6144:
// 295 KB at 64 bytes a clock); the weights that several then decode come from one L2 where the groups of a column land on
// one XCD, which they do with a multiple of eight columns of workgroups (2048, 1152 and 896 wide layers, not 1376).  us
// with one group / several: 2048 x 6144 at 40 rows 7.5 / 6.8 (two), 64 8.3 / 6.9, 128 11.3 / 8.5; 896 x 4864 at 40 rows 6.4
// / 5.3 (three), 128 9.6 / 5.9 (four); 2048 x 2048 at 128 5.6 / 4.5.  Groups beyond that share CUs: 4096 x 4096 at 40 rows
// 6.6 / 9.1, 2048 x 6144 in three 9.5.
static int row_groups(int tiles, int columns, int cus) {
    const int room = max(1, cus / columns), per = (tiles + room - 1) / room;
    return (tiles + per - 1) / per;
}

// Its time in us beside what any launch costs.  A CU runs `turns` = ceil(N / 16 / CUs) workgroups, each of which walks its
// weights and the rows of activations of its group (five row tiles run as six, seven as eight); groups of more than `most`
// tiles are taken for one.  The coefficients were fitted to one group (1002 problems, weights from HBM); with weights in the
// L2, as a loop over one layer has them, a launch takes 2.3 us and 0.8 of this, 5 per cent off on average and 13 at the
// 95th percentile, in one group and in several alike (963 problems: 13 widths 512 ... 24576, 12 reductions 512 ... 12288,
// 16 ... 128 rows).
float skinny_time(int M, int N, int K, int cus, int most) {
    const int columns = (N + 15) / 16, turns = columns <= cus ? 1 : (columns + cus - 1) / cus;
    const int rows16 = (M + 15) / 16, groups = row_groups(rows16, columns, cus), share = (rows16 + groups - 1) / groups;
    const int tiles = share > most ? rows16 : share;
    const float more = 16.0f * float((tiles == 5 ? 6 : tiles == 7 ? 8 : tiles) - 1), k = float(K);
    return K <= 2048 ? 0.33f + 1.6e-5f * k + float(turns) * k * (5.6e-4f + 1.19e-5f * more)
                     : 1.31e-4f * k - 0.3f + float(turns) * k * (6.8e-4f + 1.03e-5f * more);
}

void launch_skinny(const GemmArgs& args, int bmode, hipStream_t s) {
    GemmArgs a = args;
    if (a.epi == SCMX_EPI_SWIGLU) a.silu = silu_table_device();   // (the argument check has seen that it is there)
    const int columns = (a.N + 15) / 16, rows16 = (a.M + 15) / 16, groups = row_groups(rows16, columns, device_cus());
    const dim3 grid(columns, groups);
    // Waves per workgroup: four with four steps each where that is all of K (fewer partial sums to add: 2048 x 2048 at M = 40
    // 4.3 against 4.4 us, 12288 x 2048 at 32 7.9 against 10), else eight with six steps in flight (2048 x 6144 7.6 against 9.9).
    auto tiles = [&](auto bm) {
        constexpr int BM = decltype(bm)::value;
        auto go = [&](auto tl) {
            constexpr int T = decltype(tl)::value;
            if (a.K <= 2048) skinny_kernel<T, BM, 4, 4><<<grid, dim3(256), 0, s>>>(a);
            else skinny_kernel<T, BM, 8, 6><<<grid, dim3(512), 0, s>>>(a);
        };
        switch ((rows16 + groups - 1) / groups) {   // (several groups: of at most four tiles)
            case 1: return go(std::integral_constant<int, 1>{});
            case 2: return go(std::integral_constant<int, 2>{});
            case 3: return go(std::integral_constant<int, 3>{});
            case 4: return go(std::integral_constant<int, 4>{});
            case 5:
            case 6: return go(std::integral_constant<int, 6>{});
            default: return go(std::integral_constant<int, 8>{});
        }
    };
    switch (bmode) {
        case B_PACKED_DEFAULT: return tiles(std::integral_constant<int, B_PACKED_DEFAULT>{});
        case B_PACKED_B16: return tiles(std::integral_constant<int, B_PACKED_B16>{});
        case B_PACKED_B16M: return tiles(std::integral_constant<int, B_PACKED_B16M>{});
        case B_PACKED_E8M0: return tiles(std::integral_constant<int, B_PACKED_E8M0>{});
        default: return tiles(std::integral_constant<int, B_PACKED_GENERIC>{});
    }
}

}  // namespace scmx

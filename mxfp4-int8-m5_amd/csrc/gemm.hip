// W4A8 GEMM: the C entry points and the choice of a dense problem's tile.
#include <atomic>

#include "gemm_args.h"

namespace scmx {

static int packed_mode(const DevFormat& f) {
    return is_mxfp4_e8m0_format(f)     ? B_PACKED_E8M0
           : is_default_format(f)      ? B_PACKED_DEFAULT
           : is_pow2_block16_format(f) ? B_PACKED_B16
           : is_block16_range_format(f) ? B_PACKED_B16M
                                        : B_PACKED_GENERIC;
}

// Dense: one launch, with the tile a cost model makes fastest.  A launch runs its tiles in waves of (CUs x workgroups
// that share a CU); a wave costs f + s per 128 of K and not less than w, all three by the number of co-resident
// workgroups, and a last wave that leaves CUs idle costs a part of a full one.  Both tables are fitted to 334 problems
// (widths 896 ... 24576, reductions 896 ... 12288, 33 ... 8192 rows, every tile timed): the choice costs 0.24 per cent
// over the fastest blocked tile on average, 0.46 over the fastest row tile.
struct Cand {
    int bm, bn, occ;
    float f[4], s[4], w[4];   // per wave, by co-resident workgroups 1..occ: fixed us, us per 128 of K, least us
    float low, mid;           // a wave on half of the CUs or fewer / on three quarters of them costs this part of a full one
    int waves;                // ONE, SEVERAL: only for launches of that many
};
enum { ONE = 1, SEVERAL = 2 };
// Activations by rows, staged in LDS.  What the table encodes: 256x256 moves the fewest LDS bytes per MFMA; the small
// tiles share a CU and lose less to a ragged tile count; with no more 64x64 tiles than CUs two K groups per tile put
// eight waves on a CU, and with no more 64x32 tiles than CUs four K groups of two waves do.  (Three 64x64 tiles on a
// CU: fitted apart to single waves of 513 ... 768 of them, 2048 x 2048 at 1152 rows 14.3 us where the first fit gave
// 11.8 and 128x128 takes 12.9.)
static const Cand ROW_TILES[7] = {
    {256, 256, 1, {9.46f}, {1.772f}, {18.9f}, 0.78f, 0.86f},
    {256, 128, 1, {5.97f}, {0.857f}, {11.5f}, 0.865f, 0.93f},
    {128, 128, 1, {4.18f}, {0.513f}, {6.4f}, 0.98f, 1.04f},
    {128, 64, 2, {3.9f, 2.64f}, {0.364f, 0.649f}, {2.26f, 8.32f}, 0.945f, 1.015f},
    {64, 64, 3, {3.39f, 3.82f, 4.6f}, {0.322f, 0.462f, 0.607f}, {3.94f, 2.12f, 3.0f}, 0.975f, 1.01f},
    {64, 64, 1, {2.51f}, {0.233f}, {4.81f}, 1.0f, 1.05f},    // two K groups
    {64, 32, 1, {2.41f}, {0.157f}, {4.145f}, 1.0f, 1.05f},   // four K groups
};
// Blocked activations, read by the waves themselves.  Workgroups of four waves share a CU (two of 256x128, three of
// 128x64, four of 64x64): their barriers and epilogues do not coincide, which eight waves of one workgroup cannot
// avoid.  Eight waves on one tile are faster where the launch has no more than a tile per CU.  The one-wave entries are
// fitted to 741 problems in which such launches are many (each tile timed; 200 of them with 120 ... 260 tiles, five
// times in turn): the choice costs 0.37 per cent over the fastest tile on average there, 1.05 without 256x256 and with
// the entry for several waves (1024 x 6144 x 4096, MXFP4, 34.5 us for 28.6).
static const Cand BLOCKED_TILES[7] = {
    {256, 128, 2, {6.11f, 8.34f}, {0.966f, 1.498f}, {4.2f, 2.3f}, 0.914f, 0.96f},
    {256, 256, 1, {12.7f}, {1.46f}, {18.7f}, 0.813f, 0.856f, ONE},
    {256, 128, 1, {5.51f}, {0.805f}, {11.5f}, 0.9f, 0.85f, ONE},       // eight waves
    {256, 128, 1, {5.51f}, {0.805f}, {11.5f}, 0.85f, 0.93f, SEVERAL},  // eight waves
    {256, 64, 1, {3.945f}, {0.416f}, {2.4f}, 0.98f, 1.05f},            // eight waves
    {128, 64, 3, {3.78f, 4.09f, 2.62f}, {0.34f, 0.498f, 0.806f}, {3.83f, 5.3f, 3.0f}, 0.925f, 0.98f},
    {64, 64, 4, {3.15f, 3.54f, 3.58f, 1.83f}, {0.294f, 0.419f, 0.618f, 0.782f}, {5.49f, 4.07f, 2.67f, 3.0f}, 0.95f, 1.0f},
};
struct TileChoice {
    int index;
    float us;   // its modelled time, a launch included
};
// Asked for on every call of a layer: shifts where the sizes are powers of two, no division for less than one wave.
static TileChoice fastest_tile(const Cand* cand, int first, int last, long M, long N, long K, long cus) {
    const float steps = float(K) / 128.0f;
    TileChoice best = {-1, 1e30f};
    for (int c = first; c <= last; ++c) {   // from the largest tile down: a tie goes to the larger one
        const Cand& k = cand[c];
        const long n = ((M + k.bm - 1) >> __builtin_ctz(k.bm)) * ((N + k.bn - 1) >> __builtin_ctz(k.bn));
        if (cand == ROW_TILES && c >= 5 && (n > cus || K % (c == 5 ? 256 : 512))) continue;   // K groups
        const long cap = cus * k.occ;
        if (k.waves && (n <= cap) != (k.waves == ONE)) continue;
        const long full = n < cap ? 0 : n / cap, rest = n - full * cap;
        float t = float(full) * fmaxf(k.f[k.occ - 1] + steps * k.s[k.occ - 1], k.w[k.occ - 1]);
        if (rest) {
            const int r = rest <= cus ? 1 : int((rest + cus - 1) / cus);   // workgroups per CU in the last wave
            float w = fmaxf(k.f[r - 1] + steps * k.s[r - 1], k.w[r - 1]);
            if (r == 1) {   // CUs idle
                const float fill = float(rest) / float(cus);
                w *= fill <= 0.5f    ? k.low
                     : fill <= 0.75f ? k.low + (k.mid - k.low) * (fill - 0.5f) * 4.0f
                                     : k.mid + (1.0f - k.mid) * (fill - 0.75f) * 4.0f;
            }
            t += w;
        }
        if (t < best.us) best = {c, t};
    }
    return best;
}

// The layout a dense layer's activations are quantized into, and with it the kernel: the blocked tiles, the few-row
// kernel (blocked as well) or the row tiles, by their models.  The quantizer takes 0.3 us longer for blocks.  Beyond
// the few-row kernel's range only the row tiles with K groups were ever the fastest of all (up to 1.4 times, narrow
// layers); within it the blocked tiles have to be a tenth faster (wide layers at 100 rows and more are: 128 x 12288 x
// 2048 9.3 us for 10.7). The few-row kernel's model takes no launch in.  On 334 drawn problems of 9 ... 128 rows (512 ...
// 12400 columns and reductions, three formats, weights from HBM) whole linears cost 0.2 per cent over the fastest form on
// average, 6.5 at most.  Formats whose codes are looked up: a tile's weights
// are decoded again by each of its row groups, once by the few-row kernel, which is worth half as much again. No table
// gives less than `least`, so the smallest calls, which the host bounds, look no further.  The four-wave 256x128 tile,
// which some formats do not take (launch_dense), never decides: the same layout with and without it on 250 000 drawn
// problems.
enum { BY_ROWS = 0, BLOCKED = 1 };   // and FEW_ROWS
static int dense_layout(const scmx_format* fmt, int M, int N, int K, int most = SKINNY_MAX_ROWS / 16) {
    const int cus = device_cus();
    const bool small = M <= SKINNY_MAX_ROWS, candidate = small && long(M + 15) / 16 * 16 * N <= 480000;   // (beyond: not measured)
    const float few = candidate ? 1.0f + 0.9f * skinny_time(M, N, K, cus, most) : 1e30f;
    const float least = fmaxf(3.8f, 2.41f + 0.157f / 128.0f * float(K));
    if (few < least) return FEW_ROWS;
    const float rows = fastest_tile(ROW_TILES, small ? 0 : 5, 6, M, N, K, cus).us;
    const float blocks = (0.3f + fastest_tile(BLOCKED_TILES, 0, 6, M, N, K, cus).us) * (small ? 1.1f : 1.0f);
    const float tile = fminf(rows, blocks);
    if (few < tile) return FEW_ROWS;
    DevFormat f;
    if (fmt && few < 1.5f * tile && make_dev_format(fmt, &f) == SCMX_OK && packed_mode(f) == B_PACKED_GENERIC) return FEW_ROWS;
    return blocks < rows ? BLOCKED : BY_ROWS;
}

static void launch_dense(const GemmArgs& a, int bmode, hipStream_t s) {
    if (a.blocked == FEW_ROWS) return launch_skinny(a, bmode, s);
    if (a.blocked) {
        // The four-wave 256x128 tile and the 256x256 one read K in steps of 64.  With a byte per 32 weights and a row
        // of those 128 bytes or longer they read a cache line per weight row and step for two of them, and the vector
        // L1 does not hold the lines until the next step: four waves on 6001 x 6144 x 4096 161 us against 152 of the
        // eight waves (2-bit codes 144 / 148; K = 2048 66.6 / 68.8); 256x256 against the fastest other tile 0.98 times
        // as fast with more than 192 tiles, 1.02 with fewer.  Table decode does not fit the registers of the four
        // waves, and 256x256 is 1.07 times slower with it (40 problems; 12288 x 4096 at 896 rows 123 us, 108 on
        // 256x64).
        const bool wide_codes = (bmode == B_PACKED_E8M0 || bmode == B_PACKED_B16M) && a.K >= 4096;
        const bool many = 4LL * ((a.M + 255) / 256) * ((a.N + 255) / 256) > 3 * device_cus();
        const int first = bmode == B_PACKED_GENERIC || (wide_codes && many) ? 2 : wide_codes ? 1 : 0;
        return launch_blocked(a, bmode, fastest_tile(BLOCKED_TILES, first, 6, a.M, a.N, a.K, device_cus()).index, s);
    }
    launch_rows(a, bmode, fastest_tile(ROW_TILES, 0, 6, a.M, a.N, a.K, device_cus()).index, s);
}

static int check_gemm_common(const char* who, int M, int N, int K, int epi, bool need_scales, const void* xq,
                             const float* xscale, const float* wscale, const uint16_t* res, const void* out) {
    if (M < 0 || N <= 0 || K <= 0 || K % 128 || N % 4) {
        set_error("%s: need M >= 0, N %% 4 == 0 and K %% 128 == 0 (M=%d N=%d K=%d)", who, M, N, K);
        return SCMX_ERR_ARG;
    }
    if (uint64_t(M) * uint64_t(K) > 0xFFFFFFFFull || uint64_t(N) * uint64_t(K) > 0x7FFFFFFFull) {
        set_error("%s: operands beyond the 32-bit offsets of the kernel (M*K = %llu, N*K = %llu)", who,
                  (unsigned long long)(uint64_t(M) * K), (unsigned long long)(uint64_t(N) * K));
        return SCMX_ERR_ARG;
    }
    if (epi < 0 || epi > 3) {
        set_error("%s: unknown epilogue %d", who, epi);
        return SCMX_ERR_ARG;
    }
    if (!xq || !out || (need_scales && epi != SCMX_EPI_I32 && (!xscale || !wscale)) || (epi == SCMX_EPI_RES && !res)) {
        set_error("%s: null pointer argument", who);
        return SCMX_ERR_ARG;
    }
    if (uintptr_t(xq) % 16 || uintptr_t(out) % 16 || uintptr_t(wscale) % 16 || uintptr_t(res) % 8) {
        set_error("%s: xq / out / wscale must be 16-byte aligned (res 8-byte)", who);
        return SCMX_ERR_ARG;
    }
    if (epi == SCMX_EPI_SWIGLU && N % 8) {
        set_error("%s: the SwiGLU epilogue needs N %% 8 == 0", who);
        return SCMX_ERR_ARG;
    }
    if (epi == SCMX_EPI_SWIGLU && !silu_table_device()) {
        set_error("%s: the SiLU table of the SwiGLU epilogue could not be located on the device", who);
        return SCMX_ERR_LAUNCH;
    }
    return SCMX_OK;
}

}  // namespace scmx

using namespace scmx;

extern "C" {

int scmx_mm_epi(const int8_t* xq, const int8_t* wq, const float* xscale, const float* wscale, const uint16_t* res,
                void* out, int epi, int M, int N, int K, void* stream) {
    if (int rc = check_gemm_common("mm_epi", M, N, K, epi, true, xq, xscale, wscale, res, out)) return rc;
    if (!wq || uintptr_t(wq) % 16) {
        set_error("mm_epi: wq must be non-null and 16-byte aligned");
        return SCMX_ERR_ARG;
    }
    if (M == 0) return SCMX_OK;
    GemmArgs a = {};
    a.xq = xq; a.xscale = xscale; a.wq = wq; a.wscale = wscale; a.res = res; a.out = out;
    a.M = M; a.N = N; a.K = K; a.epi = epi;
    launch_dense(a, B_INT8, (hipStream_t)stream);
    return check_launch("mm_epi");
}

int scmx_mm_i8_i32(const int8_t* xq, const int8_t* wq, int32_t* acc, int M, int N, int K, void* stream) {
    return scmx_mm_epi(xq, wq, nullptr, nullptr, nullptr, acc, SCMX_EPI_I32, M, N, K, stream);
}

static int mm_w4a8(const scmx_format* fmt, const int8_t* xq, const float* xscale, const uint32_t* codes,
                   const uint8_t* bcodes, const float* wscale, const uint16_t* res, void* out, int epi, int M, int N,
                   int K, int blocked, void* stream) {
    DevFormat f;
    if (int rc = make_dev_format(fmt, &f)) return rc;
    if (int rc = check_gemm_common("mm_w4a8", M, N, K, epi, true, xq, xscale, wscale, res, out)) return rc;
    if (!codes || !bcodes || uintptr_t(codes) % 16 || K % f.block || (K / f.block * f.bc_bits) % 8) {
        set_error("mm_w4a8: codes must be 16-byte aligned, K a multiple of the block with whole block-code bytes per row");
        return SCMX_ERR_ARG;
    }
    if (f.e8m0 && !wscale) {
        set_error("mm_w4a8: the E8M0 form decodes with the row scales; wscale must not be NULL");
        return SCMX_ERR_ARG;
    }
    if (M == 0) return SCMX_OK;
    GemmArgs a = {};
    a.xq = xq; a.xscale = xscale; a.codes = codes; a.bcodes = bcodes; a.wscale = wscale; a.res = res; a.out = out;
    a.M = M; a.N = N; a.K = K; a.epi = epi; a.fmt = f;
    a.bc_row_bytes = K / f.block * f.bc_bits / 8;
    a.blocked = blocked;
    launch_dense(a, packed_mode(f), (hipStream_t)stream);
    return check_launch("mm_w4a8");
}

int scmx_mm_w4a8(const scmx_format* fmt, const int8_t* xq, const float* xscale, const uint32_t* codes,
                 const uint8_t* bcodes, const float* wscale, const uint16_t* res, void* out, int epi, int M, int N,
                 int K, void* stream) {
    return mm_w4a8(fmt, xq, xscale, codes, bcodes, wscale, res, out, epi, M, N, K, 0, stream);
}

int scmx_mm_w4a8_blocked(const scmx_format* fmt, const int8_t* xq, const float* xscale, const uint32_t* codes,
                         const uint8_t* bcodes, const float* wscale, const uint16_t* res, void* out, int epi, int M,
                         int N, int K, void* stream) {
    if (uintptr_t(xq) % 16) {
        set_error("mm_w4a8_blocked: xq must be 16-byte aligned");
        return SCMX_ERR_ARG;
    }
    if (M > 0 && K > 0 && ((uint64_t(M) + 31) & ~uint64_t(31)) * uint64_t(K) > 0xFFFFFFFFull) {
        set_error("mm_w4a8_blocked: the activations' whole 32-row blocks lie beyond the 32-bit offsets of the kernel (M=%d K=%d)", M, K);
        return SCMX_ERR_ARG;
    }
    const bool few = M > 0 && N > 0 && K > 0 && dense_layout(fmt, M, N, K) == FEW_ROWS;
    return mm_w4a8(fmt, xq, xscale, codes, bcodes, wscale, res, out, epi, M, N, K, few ? FEW_ROWS : BLOCKED, stream);
}

int scmx_mm_w4a8_prefers_blocked(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 128) return 0;
    // Callers keep the answer they have had for 97 ... 128 rows on 1376 ... 2048 columns and K beyond 3000, by rows (2048 x 4096
    // at 128 rows 8.3 us and 2.8 for the quantization), from before the few-row kernel cut such rows into groups of four tiles
    // (6.5 and 3.3); the whole linear, which lays its rows out itself, and who hands over blocks get the groups.
    return dense_layout(nullptr, M, N, K, 3) != BY_ROWS;
}

// The fused layer quantizes into whichever layout suits the shape (dense_layout).  Both layouts take (M rounded up to
// 32) x K bytes at most.
static int quantize_and_multiply(const scmx_format* fmt, const uint16_t* x, int8_t* xq, float* xs, bool room_for_blocks,
                                 const uint32_t* codes, const uint8_t* bcodes, const float* wscale, const uint16_t* res,
                                 void* out, int epi, int M, int N, int K, void* stream) {
    const long long Mp = (static_cast<long long>(M) + 31) & ~31LL;
    int blocked = BY_ROWS;
    if (room_for_blocks && M > 0 && N > 0 && K > 0 && K % 128 == 0 && uint64_t(Mp) * uint64_t(K) <= 0xFFFFFFFFull)
        blocked = dense_layout(fmt, M, N, K);
    if (blocked) {
        if (int rc = scmx_act_quant_blocked(x, xq, xs, M, int(Mp), K, stream)) return rc;
    } else {
        if (int rc = scmx_act_quant(x, xq, xs, M, M, K, stream)) return rc;
    }
    return mm_w4a8(fmt, xq, xs, codes, bcodes, wscale, res, out, epi, M, N, K, blocked, stream);
}

size_t scmx_linear_w4a8_workspace(int M, int K) {
    if (M <= 0 || K <= 0) return 0;
    const size_t Mp = (size_t(M) + 31) & ~size_t(31);   // whole 32-row blocks of the blocked layout
    const size_t q = (Mp * size_t(K) + 255) & ~size_t(255);
    return q + Mp * sizeof(float);
}

int scmx_linear_w4a8(const scmx_format* fmt, const uint16_t* x, const uint32_t* codes, const uint8_t* bcodes,
                     const float* wscale, const uint16_t* res, void* out, int epi, int M, int N, int K,
                     void* workspace, size_t workspace_bytes, void* stream) {
    if (M < 0 || K <= 0) {
        set_error("linear_w4a8: bad shape M=%d K=%d", M, K);
        return SCMX_ERR_ARG;
    }
    if (!workspace || workspace_bytes < scmx_linear_w4a8_workspace(M, K) || uintptr_t(workspace) % 256) {
        set_error("linear_w4a8: workspace must be 256-byte aligned and hold %zu bytes",
                  scmx_linear_w4a8_workspace(M, K));
        return SCMX_ERR_WORKSPACE;
    }
    int8_t* xq = reinterpret_cast<int8_t*>(workspace);
    const size_t Mp = (size_t(M) + 31) & ~size_t(31);
    float* xs = reinterpret_cast<float*>(xq + ((Mp * size_t(K) + 255) & ~size_t(255)));
    return quantize_and_multiply(fmt, x, xq, xs, true, codes, bcodes, wscale, res, out, epi, M, N, K, stream);
}

// ---- the dense layer for callers that cannot allocate ------------------------------------------------------------
// The INT8 activations and their scales, which scmx_linear_w4a8 keeps in the caller's workspace, live here in a fixed
// array of the library's device image (every GPU the library runs on holds its own copy until the process ends).
// `scratch` is a host-side stand-in in host code, not a device address: the address on the current device comes from
// hipGetSymbolAddress, once per device, and only that pointer is handed to kernels.
constexpr size_t STATIC_XQ_BYTES = size_t(16) << 20;   // M * K <= 16 Mi elements, e.g. 2048 x 8192 or 8192 x 2048
constexpr int STATIC_MAX_ROWS = 16384;                 // M <= 16384 scales
constexpr size_t STATIC_SCRATCH_BYTES = STATIC_XQ_BYTES + size_t(STATIC_MAX_ROWS) * sizeof(float);
static __device__ __align__(256) uint8_t scratch[STATIC_SCRATCH_BYTES];

// Device address of `scratch` on the current device (NULL with the error text set when it cannot be resolved).
static uint8_t* static_scratch_device() {
    static std::atomic<uint8_t*> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
        set_error("linear_w4a8_static: no current device (or a device index beyond 63)");
        return nullptr;
    }
    uint8_t* p = cached[dev].load(std::memory_order_acquire);
    if (!p) {
        void* addr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !addr) {
            set_error("linear_w4a8_static: hipGetSymbolAddress(scratch) failed on device %d: %s", dev, hipGetErrorString(e));
            return nullptr;
        }
        p = reinterpret_cast<uint8_t*>(addr);
        cached[dev].store(p, std::memory_order_release);
    }
    return p;
}

int scmx_init(void) {
    if (!static_scratch_device()) return SCMX_ERR_LAUNCH;
    if (!silu_table_device()) {
        set_error("init: the SiLU table of the SwiGLU epilogue could not be located on the current device");
        return SCMX_ERR_LAUNCH;
    }
    return SCMX_OK;
}

size_t scmx_linear_w4a8_static_max_elements(void) { return STATIC_XQ_BYTES; }
int scmx_linear_w4a8_static_max_rows(void) { return STATIC_MAX_ROWS; }

int scmx_linear_w4a8_static(const scmx_format* fmt, const uint16_t* x, const uint32_t* codes, const uint8_t* bcodes,
                            const float* wscale, const uint16_t* res, void* out, int epi, int M, int N, int K,
                            void* stream) {
    if (M < 0 || K <= 0) {
        set_error("linear_w4a8_static: bad shape M=%d K=%d", M, K);
        return SCMX_ERR_ARG;
    }
    if (size_t(M) * size_t(K) > STATIC_XQ_BYTES || M > STATIC_MAX_ROWS) {
        set_error("linear_w4a8_static: M*K = %zu elements or M = %d rows beyond the built-in scratch (%zu elements, %d "
                  "rows); use scmx_linear_w4a8 with a workspace", size_t(M) * size_t(K), M, STATIC_XQ_BYTES,
                  STATIC_MAX_ROWS);
        return SCMX_ERR_WORKSPACE;
    }
    uint8_t* base = static_scratch_device();
    if (!base) return SCMX_ERR_LAUNCH;
    int8_t* xq = reinterpret_cast<int8_t*>(base);
    float* xs = reinterpret_cast<float*>(base + STATIC_XQ_BYTES);
    // every byte of xq and xs[M] that the GEMM reads is written by the quantization first (in the blocked layout: the
    // whole last 32-row block, rows past M as zeros): nothing has to start at zero, whatever the previous call left
    // behind
    const size_t Mp = (size_t(M) + 31) & ~size_t(31);
    const bool room = Mp * size_t(K) <= STATIC_XQ_BYTES && Mp <= size_t(STATIC_MAX_ROWS);
    return quantize_and_multiply(fmt, x, xq, xs, room, codes, bcodes, wscale, res, out, epi, M, N, K, stream);
}

static int moe_common(const char* who, const int8_t* xq, const float* xscale, const int32_t* gather, int R,
                      const float* wscale, const int32_t* off, const int32_t* tstart, int n_experts, int tm, int N,
                      int K, int epi, void* out, GemmArgs* a) {
    if (epi == SCMX_EPI_RES) {
        set_error("%s: the grouped GEMM has no residual epilogue", who);
        return SCMX_ERR_ARG;
    }
    if (int rc = check_gemm_common(who, R, N, K, epi, true, xq, xscale, wscale, nullptr, out)) return rc;
    if (!off || !tstart || n_experts < 1 || n_experts > (1 << 20) || !(tm == 64 || tm == 128 || tm == 256)) {
        set_error("%s: need off / tstart, 1 <= n_experts <= 2^20 and a row tile of 64, 128 or 256 (got %d)", who, tm);
        return SCMX_ERR_ARG;
    }
    *a = GemmArgs{};
    a->xq = xq; a->xscale = xscale; a->gather = gather; a->wscale = wscale; a->out = out;
    a->M = R; a->N = N; a->K = K; a->epi = epi; a->off = off; a->tstart = tstart; a->n_experts = n_experts;
    return SCMX_OK;
}

static int moe_mm(const scmx_format* fmt, const int8_t* xq, const float* xscale, const int32_t* gather, int R,
                  const uint32_t* codes, const uint8_t* bcodes, const float* wscale, const int32_t* off, const int32_t* tstart,
                  int n_experts, int tm, int N, int K, int epi, void* out, int blocked, void* stream) {
    DevFormat f;
    if (int rc = make_dev_format(fmt, &f)) return rc;
    GemmArgs a;
    if (int rc = moe_common("moe_mm", xq, xscale, gather, R, wscale, off, tstart, n_experts, tm, N, K, epi, out, &a))
        return rc;
    if (!codes || !bcodes || uintptr_t(codes) % 16 || K % f.block || (K / f.block * f.bc_bits) % 8) {
        set_error("moe_mm: codes must be 16-byte aligned, K a multiple of the block with whole block-code bytes per row");
        return SCMX_ERR_ARG;
    }
    if (f.e8m0 && !wscale) {
        set_error("moe_mm: the E8M0 form decodes with the row scales; wscale must not be NULL");
        return SCMX_ERR_ARG;
    }
    if (R == 0) return SCMX_OK;
    a.codes = codes; a.bcodes = bcodes; a.fmt = f;
    a.bc_row_bytes = K / f.block * f.bc_bits / 8;
    a.blocked = blocked;
    launch_grouped(a, packed_mode(f), tm, (hipStream_t)stream);
    return check_launch("moe_mm");
}

int scmx_moe_mm(const scmx_format* fmt, const int8_t* xq, const float* xscale, const int32_t* gather, int R,
                const uint32_t* codes, const uint8_t* bcodes, const float* wscale, const int32_t* off,
                const int32_t* tstart, int n_experts, int tm, int N, int K, int epi, void* out, void* stream) {
    return moe_mm(fmt, xq, xscale, gather, R, codes, bcodes, wscale, off, tstart, n_experts, tm, N, K, epi, out, 0, stream);
}

int scmx_moe_mm_takes_slots(const scmx_format* fmt, int R, int n_experts, int K) {
    DevFormat f;
    return R >= 0 && n_experts >= 1 && n_experts <= (1 << 20) && K > 0 && K % 128 == 0 && K <= 12288 &&
           (uint64_t(R) / 256 + 1 + uint64_t(n_experts)) * 256 * uint64_t(K) <= 0xFFFFFFFFull &&
           make_dev_format(fmt, &f) == SCMX_OK && packed_mode(f) != B_PACKED_GENERIC;
}

int scmx_moe_mm_blocked(const scmx_format* fmt, const int8_t* xq, const float* xscale, int R, const uint32_t* codes,
                        const uint8_t* bcodes, const float* wscale, const int32_t* off, const int32_t* tstart, int n_experts,
                        int N, int K, int epi, void* out, void* stream) {
    DevFormat f;
    if (int rc = make_dev_format(fmt, &f)) return rc;
    if (!scmx_moe_mm_takes_slots(fmt, R, n_experts, K)) {
        set_error("moe_mm_blocked: need a format that decodes with the FP4 conversion, 1 <= n_experts <= 2^20, K a multiple of 128 up to "
                  "12288 and slots within 2^32 bytes (R=%d K=%d, %d experts)", R, K, n_experts);
        return packed_mode(f) == B_PACKED_GENERIC ? SCMX_ERR_FORMAT : SCMX_ERR_ARG;
    }
    return moe_mm(fmt, xq, xscale, nullptr, R, codes, bcodes, wscale, off, tstart, n_experts, 256, N, K, epi, out, 1, stream);
}

int scmx_moe_mm_i8(const int8_t* xq, const float* xscale, const int32_t* gather, int R, const int8_t* wq,
                   const float* wscale, const int32_t* off, const int32_t* tstart, int n_experts, int tm, int N,
                   int K, int epi, void* out, void* stream) {
    GemmArgs a;
    if (int rc = moe_common("moe_mm_i8", xq, xscale, gather, R, wscale, off, tstart, n_experts, tm, N, K, epi, out, &a))
        return rc;
    if (!wq || uintptr_t(wq) % 16) {
        set_error("moe_mm_i8: wq must be non-null and 16-byte aligned");
        return SCMX_ERR_ARG;
    }
    if (R == 0) return SCMX_OK;
    a.wq = wq;
    launch_grouped(a, B_INT8, tm, (hipStream_t)stream);
    return check_launch("moe_mm_i8");
}

}  // extern "C"

// Library plumbing (errors, format validation) and the small memory-bound kernels: weight unpack, activation
// quantization, standard-MXFP4 scale conversion.
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <atomic>
#include <type_traits>

#include "scmx_common.h"

namespace scmx {

static thread_local char g_err[512] = "";

void set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

int check_launch(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("%s: %s", what, hipGetErrorString(e));
        return SCMX_ERR_LAUNCH;
    }
    return SCMX_OK;
}

// Compute units of the current device, asked once per device (256 on MI355X; the fallback when the query fails).
int device_cus() {
    static std::atomic<int> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    int n = cached[dev].load(std::memory_order_relaxed);
    if (n <= 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

int make_dev_format(const scmx_format* f, DevFormat* out) {
    if (!f) {
        set_error("format is NULL");
        return SCMX_ERR_ARG;
    }
    const int b = f->block;
    if (!(b == 8 || b == 16 || b == 32 || b == 64 || b == 128)) {
        set_error("format: block %d not in {8,16,32,64,128}", b);
        return SCMX_ERR_FORMAT;
    }
    if (b == 32 && f->bc_bits == 8 && f->n_mult == 0) {   // standard MXFP4: E8M0 bytes in place of block codes
        const int mag[8] = {0, 1, 2, 3, 4, 6, 8, 12};
        for (int i = 0; i < 8; ++i)
            if (f->code_mag[i] != mag[i]) {
                set_error("format: the E8M0 form takes the E2M1 code magnitudes 0,1,2,3,4,6,8,12");
                return SCMX_ERR_FORMAT;
            }
        DevFormat d;
        memset(&d, 0, sizeof(d));
        d.lut_lo = 0x03020100u;
        d.lut_hi = 0x0C080604u;
        d.mult[0] = 0x08040201u;
        d.block = 32;
        d.block_log2 = 5;
        d.bc_bits = 8;
        d.pow2 = 1;
        d.e8m0 = 1;
        *out = d;
        return SCMX_OK;
    }
    if (!(f->bc_bits == 1 || f->bc_bits == 2 || f->bc_bits == 4 || f->bc_bits == 8) || f->n_mult < 1 ||
        f->n_mult > 16 || f->n_mult > (1 << f->bc_bits)) {
        set_error("format: bc_bits %d / n_mult %d unsupported (need bc_bits in {1,2,4,8}, n_mult <= min(16, 2^bc_bits))",
                  f->bc_bits, f->n_mult);
        return SCMX_ERR_FORMAT;
    }
    int mag_max = 0, mult_max = 0;
    for (int i = 0; i < 8; ++i) {
        if (f->code_mag[i] < 0 || f->code_mag[i] > 127) {
            set_error("format: code_mag[%d] = %d outside 0..127", i, f->code_mag[i]);
            return SCMX_ERR_FORMAT;
        }
        mag_max = f->code_mag[i] > mag_max ? f->code_mag[i] : mag_max;
    }
    for (int i = 0; i < f->n_mult; ++i) {
        if (f->mult[i] < 1 || f->mult[i] > 127) {
            set_error("format: mult[%d] = %d outside 1..127", i, f->mult[i]);
            return SCMX_ERR_FORMAT;
        }
        mult_max = f->mult[i] > mult_max ? f->mult[i] : mult_max;
    }
    if (mag_max * mult_max > 127) {
        set_error("format: max(code_mag) * max(mult) = %d does not fit INT8", mag_max * mult_max);
        return SCMX_ERR_FORMAT;
    }
    DevFormat d;
    memset(&d, 0, sizeof(d));
    for (int i = 0; i < 4; ++i) {
        d.lut_lo |= uint32_t(f->code_mag[i]) << (8 * i);
        d.lut_hi |= uint32_t(f->code_mag[4 + i]) << (8 * i);
    }
    d.pow2 = 1;
    for (int i = 0; i < f->n_mult; ++i) {
        d.mult[i >> 2] |= uint32_t(f->mult[i]) << (8 * (i & 3));
        if (f->mult[i] != (1 << i)) d.pow2 = 0;
    }
    d.block = b;
    d.block_log2 = b == 8 ? 3 : b == 16 ? 4 : b == 32 ? 5 : b == 64 ? 6 : 7;
    d.bc_bits = f->bc_bits;
    *out = d;
    return SCMX_OK;
}

// ---- unpack_i8: one thread per 16-byte group of codes (32 weights) ---------------------------------------------
__global__ __launch_bounds__(256) void unpack_i8_kernel(DevFormat f, const u32x4* __restrict__ codes,
                                                        const uint8_t* __restrict__ bcodes, u32x4* __restrict__ wq,
                                                        int64_t n_groups, int groups_per_row, int bc_row_bytes) {
    const int64_t g = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (g >= n_groups) return;
    const int64_t row = g / groups_per_row;
    const uint32_t k0 = uint32_t(g % groups_per_row) * 32u;
    const u32x4 w = codes[g];
    const uint8_t* row_bc = bcodes + row * bc_row_bytes;
    uint32_t o[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t bc = block_code(row_bc, (k0 + 8u * j) >> f.block_log2, f.bc_bits);
        const BlockLut t = scaled_lut_mul(f.lut_lo, f.lut_hi, mult_of(f, bc));
        decode_word(w[j], t, o[2 * j], o[2 * j + 1]);
    }
    wq[2 * g] = u32x4{o[0], o[1], o[2], o[3]};
    wq[2 * g + 1] = u32x4{o[4], o[5], o[6], o[7]};
}

// Fallback for K not a multiple of 32: one thread per code word (8 weights).
__global__ __launch_bounds__(256) void unpack_i8_word_kernel(DevFormat f, const uint32_t* __restrict__ codes,
                                                             const uint8_t* __restrict__ bcodes,
                                                             u32x2* __restrict__ wq, int64_t n_words,
                                                             int words_per_row, int bc_row_bytes) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n_words) return;
    const int64_t row = i / words_per_row;
    const uint32_t k0 = uint32_t(i % words_per_row) * 8u;
    const uint32_t bc = block_code(bcodes + row * bc_row_bytes, k0 >> f.block_log2, f.bc_bits);
    const BlockLut t = scaled_lut_mul(f.lut_lo, f.lut_hi, mult_of(f, bc));
    uint32_t a, b;
    decode_word(codes[i], t, a, b);
    wq[i] = u32x2{a, b};
}

// The largest magnitude of eight bf16 values and m; their INT8 codes.
__device__ __forceinline__ float amax8(const u32x4& v, float m) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        m = fmaxf(m, fabsf(__uint_as_float(v[e] << 16)));
        m = fmaxf(m, fabsf(__uint_as_float(v[e] & 0xFFFF0000u)));
    }
    return m;
}
__device__ __forceinline__ u32x2 codes8(const u32x4& v, float qi) {
    uint32_t o[2] = {0u, 0u};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int q0 = quant_code(__uint_as_float(v[e] << 16), qi);
        const int q1 = quant_code(__uint_as_float(v[e] & 0xFFFF0000u), qi);
        o[e >> 1] |= (uint32_t(q0) & 0xFFu) << (16 * (e & 1));
        o[e >> 1] |= (uint32_t(q1) & 0xFFu) << (16 * (e & 1) + 8);
    }
    return u32x2{o[0], o[1]};
}

// ---- act_quant: one workgroup per token row ---------------------------------------------------------------------
// Lanes read 8 bf16 (16 bytes) per step; the row maximum goes through LDS; the second sweep re-reads the row
// (cache hit) and writes 8 codes per lane.
__global__ __launch_bounds__(256) void act_quant_kernel(const uint16_t* __restrict__ x, int8_t* __restrict__ xq,
                                                        float* __restrict__ xs, int M, int K) {
    __shared__ float red[4];
    const int row = blockIdx.x, tid = threadIdx.x;
    u32x2* qrow = reinterpret_cast<u32x2*>(xq + size_t(row) * K);
    if (row >= M) {
        for (int c = tid; c < K / 8; c += 256) qrow[c] = u32x2{0u, 0u};
        if (tid == 0) xs[row] = 0.0f;
        return;
    }
    const u32x4* xrow = reinterpret_cast<const u32x4*>(x + size_t(row) * K);
    float amax = 0.0f;
    for (int c = tid; c < K / 8; c += 256) {
        amax = amax8(xrow[c], amax);
    }
    amax = wave_max(amax);
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float s = __fdiv_rn(amax, 127.0f);
    const float qi = s > 0.0f ? __fdiv_rn(1.0f, s) : 0.0f;
    for (int c = tid; c < K / 8; c += 256) {
        qrow[c] = codes8(xrow[c], qi);
    }
    if (tid == 0) xs[row] = s;
}

// The same with the row held in registers: one wave per row, lane l owns the 16-byte pieces l, l + 64, ... (up to CH of
// them, K <= 512 * CH, K % 32 == 0), so the row is read once and the only reduction is inside the wave.  Four rows per
// workgroup.
// BLK: xq leaves in the blocked layout of the dense GEMM's large tiles (32 x 32 blocks in MFMA operand order, described at
// act_quant_blocked_kernel below; Mp % 32 == 0): eight rows per workgroup, whose codes meet in LDS -- the 16 bytes of row
// r, k 16 c ... at slot c * 8 + (r + c / 2) % 8 -- and are stored as whole 128-byte lines (8 rows x 16 bytes are adjacent
// in a block).  The loads stay what they are by rows: 16 contiguous bytes per lane.
// (Registers are held to what lets four waves share a SIMD up to 6144 values, three up to 8192: 4000 rows x 6144 blocked 16.6
// us at three, 13.0 at four.  Whole rows of up to 6144 in the row layout fit without it and are given fewer registers then:
// 4096 values 76 for 82, six waves a SIMD for five, 3 - 6 per cent at 257 ... 1500 rows.)
// SORT (BLK): the rows of x are sorted by expert and those of xq are the slots of the grouped GEMM, 256 rows each: row p of
// a slot holds row p of that slot's part of the segment.  Of the rows past a segment only those of its last eight are
// written (as zeros).
struct SortedRows {
    const int32_t *off, *tstart;   // as for the grouped GEMM
    int n_experts;
    // Workgroup b's 2^LOG rows, aligned in their slot: the first one and the segment's end among the sorted rows, and the
    // first one's place in the slots; false: none.  Expert e's groups start at off[e] / 2^LOG + e, room enough for a cut one
    // each, so R / 2^LOG + E workgroups cover every segment.  (A grid over the rows of all slots idles where experts have
    // few: 8000 x 1024 over 64 experts 8.5 us for 5.9, 54000 x 512 over 257 30.5 for 20.4.)
    template <int LOG>
    __device__ bool rows(int b, int* first, int* end, int* place) const {
        const int e = last_started(n_experts, b, [&](int i) { return (off[i] >> LOG) + i; });
        const int o = off[e], r = (b - (o >> LOG) - e) << LOG;
        *first = o + r;
        *end = off[e + 1];
        *place = (tstart[e] << 8) + r;
        return *first < *end;
    }
};
template <int CH, bool BLK, bool WHOLE, bool SORT = false>
__global__ __launch_bounds__(BLK ? 512 : 256, !BLK && WHOLE && CH <= 12 ? 1 : CH <= 12 ? 4 : CH <= 16 ? 3 : 1) void act_quant_wave_kernel(
    const uint16_t* __restrict__ x, int8_t* __restrict__ xq, float* __restrict__ xs, int M, int Mp, int K_any, SortedRows sort) {
    const int K = WHOLE ? 512 * CH : K_any;   // WHOLE: every lane has all of its CH pieces
    constexpr int RPW = BLK ? 8 : 4;
    constexpr int TURN = CH > 16 ? CH / 2 : CH;   // pieces whose codes are in LDS at once (at most 64 KB)
    __shared__ u32x2 tile[BLK ? TURN * 64 * 8 : 1];
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int row0 = blockIdx.x * RPW, row = row0 + wid;   // of xq; of x and xs
    if constexpr (SORT) {
        if (!sort.rows<3>(blockIdx.x, &row, &M, &row0)) return;
        row += wid;
    }
    auto gather_store = [&](int j0) {   // BLK: the codes of pieces j0 .. j0 + TURN - 1 of every row, after all are in LDS
        __syncthreads();
        int8_t* const blk = xq + (size_t(row0 >> 5) * size_t(K >> 5)) * 1024;
        const u32x4* t16 = reinterpret_cast<const u32x4*>(tile);
#pragma unroll
        for (int j = 0; j < TURN / 2 + TURN % 2; ++j) {   // 32 TURN chunks of 16 k x 8 rows, 512 per pass
            const int idx = int(threadIdx.x) + 512 * j, cl = idx >> 3, r = idx & 7, c = cl + 32 * j0;
            if ((WHOLE && TURN % 2 == 0) || (cl < 32 * TURN && c < K / 16))
                *reinterpret_cast<u32x4*>(blk + size_t(c >> 1) * 1024 + (c & 1) * 512 + ((row0 + r) & 31) * 16) =
                    t16[cl * 8 + ((r + (cl >> 1)) & 7)];
        }
        if (TURN < CH) __syncthreads();
    };
    // piece p (8 codes, counted from the turn's first) of this wave's row: half p % 2 of the 16-byte slot of chunk p / 2
    auto slot = [&](int p) { return ((p >> 1) * 8 + ((wid + (p >> 2)) & 7)) * 2 + (p & 1); };
    auto mine = [&](int j) { return WHOLE || lane + 64 * j < K / 8; };
    if (!BLK && row >= Mp) return;
    u32x2* qrow = reinterpret_cast<u32x2*>(xq + size_t(row) * K);
    if (row >= M) {
#pragma unroll
        for (int j0 = 0; j0 < CH; j0 += TURN) {
#pragma unroll
            for (int j = j0; j < j0 + TURN; ++j)
                if (mine(j)) {
                    if (BLK) tile[slot(lane + 64 * (j - j0))] = u32x2{0u, 0u}; else qrow[lane + 64 * j] = u32x2{0u, 0u};
                }
            if (BLK) gather_store(j0);
        }
        if (!SORT && lane == 0) xs[row] = 0.0f;
        return;
    }
    const u32x4* xrow = reinterpret_cast<const u32x4*>(x + size_t(row) * K);
    u32x4 v[CH];
#pragma unroll
    for (int j = 0; j < CH; ++j) v[j] = mine(j) ? xrow[lane + 64 * j] : u32x4{0u, 0u, 0u, 0u};
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < CH; ++j) amax = amax8(v[j], amax);
    amax = wave_max(amax);
    const float s = __fdiv_rn(amax, 127.0f);
    const float qi = s > 0.0f ? __fdiv_rn(1.0f, s) : 0.0f;
#pragma unroll
    for (int j0 = 0; j0 < CH; j0 += TURN) {
#pragma unroll
        for (int j = j0; j < j0 + TURN; ++j) {
            const u32x2 o = codes8(v[j], qi);
            if (mine(j)) {
                if (BLK) tile[slot(lane + 64 * (j - j0))] = o; else qrow[lane + 64 * j] = o;
            }
        }
        if (BLK) gather_store(j0);
    }
    if (lane == 0) xs[row] = s;
}

// ---- act_quant into the blocked layout ---------------------------------------------------------------------------
// xq as the large dense GEMM tiles take it: blocks of 32 rows x 32 k (1 KB), block (m / 32, k / 32) at
// ((m / 32) * (K / 32) + k / 32) KB, and inside a block the 16 bytes of row r, k half h at (32 h + r) * 16 -- the order
// in which the 64 lanes of a wave hold a 32x32x32 MFMA operand, so that a wave fetches one block with one coalesced load.
// Rows of K <= 12288 go through act_quant_wave_kernel above, few rows (up to 16384 values) through act_quant_row_kernel below;
// this is the kernel for longer rows and for many of more than 12288 values: one wave per row, eight rows per workgroup, the
// row read twice, every lane writing the 16 bytes of its own 16 elements.  Same codes and scales as act_quant_kernel: the row maximum does not depend on the order it is
// taken in.
__global__ __launch_bounds__(512) void act_quant_blocked_kernel(const uint16_t* __restrict__ x, int8_t* __restrict__ xq,
                                                                float* __restrict__ xs, int M, int Mp, int K) {
    const int row = blockIdx.x * 8 + (threadIdx.x >> 6), lane = threadIdx.x & 63;   // Mp % 32 == 0: whole groups of 8 rows
    const int pieces = K / 16;
    // piece c of the row (k = 16 c ...): k slice c / 2, half c % 2
    int8_t* const dst = xq + (size_t(row >> 5) * size_t(K >> 5)) * 1024 + size_t(row & 31) * 16;
    auto at = [&](int c) { return reinterpret_cast<u32x4*>(dst + size_t(c >> 1) * 1024 + (c & 1) * 512); };
    if (row >= M) {
        for (int c = lane; c < pieces; c += 64) *at(c) = u32x4{0u, 0u, 0u, 0u};
        if (lane == 0) xs[row] = 0.0f;
        return;
    }
    const u32x4* xrow = reinterpret_cast<const u32x4*>(x + size_t(row) * K);
    float amax = 0.0f;
    for (int c = lane; c < pieces; c += 64) amax = amax8(xrow[2 * c + 1], amax8(xrow[2 * c], amax));
    amax = wave_max(amax);
    const float s = __fdiv_rn(amax, 127.0f);
    const float qi = s > 0.0f ? __fdiv_rn(1.0f, s) : 0.0f;
    for (int c = lane; c < pieces; c += 64) {
        const u32x2 lo = codes8(xrow[2 * c], qi), hi = codes8(xrow[2 * c + 1], qi);
        *at(c) = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
    if (lane == 0) xs[row] = s;
}

// Either layout for few rows and, by rows, for rows too long for a wave's registers: a workgroup of WAVES waves per row, P pieces of 16 values per thread in registers (K % 32 == 0, K <= 1024 * WAVES * P).  A
// handful of rows is a matter of latency: with a wave per row the rounding of 6144 values is a chain of 96 per lane (40 rows
// blocked: 4.6 us, 2.9 here), and rows of 12288 values were read twice (9.0, 3.7).
template <int WAVES, int P, bool BLK>
__global__ __launch_bounds__(WAVES * 64) void act_quant_row_kernel(const uint16_t* __restrict__ x, int8_t* __restrict__ xq,
                                                                   float* __restrict__ xs, int M, int K) {
    __shared__ float red[WAVES];
    const int row = blockIdx.x, tid = threadIdx.x, pieces = K / 16;
    int8_t* const dst = BLK ? xq + (size_t(row >> 5) * size_t(K >> 5)) * 1024 + size_t(row & 31) * 16 : xq + size_t(row) * K;
    auto at = [&](int c) { return reinterpret_cast<u32x4*>(BLK ? dst + size_t(c >> 1) * 1024 + (c & 1) * 512 : dst + 16 * c); };
    if (row >= M) {
        for (int c = tid; c < pieces; c += WAVES * 64) *at(c) = u32x4{0u, 0u, 0u, 0u};
        if (tid == 0) xs[row] = 0.0f;
        return;
    }
    const u32x4* xrow = reinterpret_cast<const u32x4*>(x + size_t(row) * K);
    u32x4 v[P][2];
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const int c = tid + j * WAVES * 64;
        v[j][0] = v[j][1] = u32x4{0u, 0u, 0u, 0u};
        if (c < pieces) {
            v[j][0] = xrow[2 * c];
            v[j][1] = xrow[2 * c + 1];
        }
    }
#pragma unroll
    for (int j = 0; j < P; ++j) amax = amax8(v[j][1], amax8(v[j][0], amax));
    amax = wave_max(amax);
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WAVES; ++w) amax = fmaxf(amax, red[w]);
    const float s = __fdiv_rn(amax, 127.0f);
    const float qi = s > 0.0f ? __fdiv_rn(1.0f, s) : 0.0f;
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const int c = tid + j * WAVES * 64;
        if (c >= pieces) break;
        const u32x2 lo = codes8(v[j][0], qi), hi = codes8(v[j][1], qi);
        *at(c) = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
    if (tid == 0) xs[row] = s;
}

// ---- rows of xq, sorted by expert, into the grouped GEMM's blocked slots -------------------------------------------
// A workgroup per 32-row block of a slot, its waves in turn on 512 of K: loads of 128 contiguous bytes of each of 8 rows,
// stored as pieces of 8 rows x 16 bytes, whole 128-byte lines of the blocks.  Bound by the stores: 24000 rows of 2048
// (every row eight times), 49 MB written, 16.8 us, the launch and four dependent trips to memory in it.
__global__ __launch_bounds__(256) void moe_gather_blocked_kernel(const int8_t* __restrict__ xq, const float* __restrict__ xscale,
                                                                 const int32_t* __restrict__ gather, SortedRows sort, int K,
                                                                 int8_t* __restrict__ out, float* __restrict__ out_scale) {
    const int lane = threadIdx.x & 63;
    int first, end, place;
    if (!sort.rows<5>(blockIdx.x, &first, &end, &place)) return;
    const int r8 = lane >> 3, c = lane & 7;   // row within eight, 16-byte piece within 128 bytes
    const int8_t* src[4];
    bool live[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const int r = first + 8 * g + r8;
        live[g] = r < end;
        const int from = gather[min(r, end - 1)];
        src[g] = xq + size_t(from) * K + c * 16;
        if (threadIdx.x < 64 && c == 0 && live[g]) out_scale[r] = xscale[from];
    }
    int8_t* const dst = out + size_t(place >> 5) * size_t(K >> 5) * 1024 + (c >> 1) * 1024 + (c & 1) * 512 + r8 * 16;
    for (int k = (threadIdx.x >> 6) * 512; k < K; k += 2048) {
        u32x4 v[4][4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                if (k + 128 * q < K) v[q][g] = *reinterpret_cast<const u32x4*>(src[g] + k + 128 * q);
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                if (k + 128 * q < K && live[g]) *reinterpret_cast<u32x4*>(dst + size_t((k >> 5) + 4 * q) * 1024 + g * 128) = v[q][g];
    }
}

// ---- rot_quant: randomized Hadamard rotation of every 32-wide block, then per-token INT8 ---------------------------
// Thread t owns 4 consecutive values; 8 consecutive lanes hold one block.  Butterfly order as in the host
// formulation: two stages inside the thread, then strides 1, 2, 4 across lanes (lower = lower + upper,
// upper = lower - upper); the result times 1/sqrt(32) is rounded to bf16 before the row maximum is taken.
__global__ __launch_bounds__(256) void rot_quant_kernel(const uint16_t* __restrict__ x, const float* __restrict__ signs,
                                                        int8_t* __restrict__ xq, float* __restrict__ xs, int M, int K) {
    __shared__ float red[4];
    constexpr int MAXJ = 8;   // K <= 8192
    const int row = blockIdx.x, tid = threadIdx.x;
    const int J = K / 1024, rem = K % 1024;   // whole sweeps of 256 threads x 4 values, then a partial one
    float v[MAXJ + 1][4];
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j <= MAXJ; ++j) {
        const int p = 4 * (j * 256 + tid);
        const bool in = j < J || (j == J && p < K);
        if (j > J || (j == J && rem == 0)) break;
        float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f, a3 = 0.0f;
        if (in && row < M) {
            const u32x2 w = *reinterpret_cast<const u32x2*>(x + size_t(row) * K + p);
            const f32x4 sg = *reinterpret_cast<const f32x4*>(signs + p);
            a0 = __fmul_rn(__uint_as_float(w[0] << 16), sg[0]);
            a1 = __fmul_rn(__uint_as_float(w[0] & 0xFFFF0000u), sg[1]);
            a2 = __fmul_rn(__uint_as_float(w[1] << 16), sg[2]);
            a3 = __fmul_rn(__uint_as_float(w[1] & 0xFFFF0000u), sg[3]);
        }
        float b[4] = {__fadd_rn(a0, a1), __fsub_rn(a0, a1), __fadd_rn(a2, a3), __fsub_rn(a2, a3)};
        float a[4] = {__fadd_rn(b[0], b[2]), __fadd_rn(b[1], b[3]), __fsub_rn(b[0], b[2]), __fsub_rn(b[1], b[3])};
#pragma unroll
        for (int h = 1; h < 8; h <<= 1)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float c = __shfl_xor(a[i], h, WAVE);
                a[i] = (tid & h) ? __fsub_rn(c, a[i]) : __fadd_rn(a[i], c);
            }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[j][i] = round_bf16(__fmul_rn(a[i], 0.17677669529663687f));
            if (in) amax = fmaxf(amax, fabsf(v[j][i]));
        }
    }
    amax = wave_max(amax);
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float s = __fdiv_rn(amax, 127.0f);
    const float qi = s > 0.0f ? __fdiv_rn(1.0f, s) : 0.0f;
#pragma unroll
    for (int j = 0; j <= MAXJ; ++j) {
        const int p = 4 * (j * 256 + tid);
        if (j > J || (j == J && rem == 0)) break;
        if (j < J || p < K) {
            uint32_t o = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) o |= (uint32_t(quant_code(v[j][i], qi)) & 0xFFu) << (8 * i);
            *reinterpret_cast<uint32_t*>(xq + size_t(row) * K + p) = o;
        }
    }
    if (tid == 0) xs[row] = row < M ? s : 0.0f;
}

// ---- standard MXFP4 -> block codes + row scale: one wave per row -----------------------------------------------
__global__ __launch_bounds__(256) void mxfp4_to_sc_kernel(const uint8_t* __restrict__ e8m0,
                                                          uint8_t* __restrict__ bcodes, float* __restrict__ wscale,
                                                          int32_t* __restrict__ status, int64_t N, int nb) {
    const int64_t row = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= N) return;
    const uint8_t* e = e8m0 + row * nb;
    int lo = 255, hi = 0;
    for (int b = lane; b < nb; b += 64) {
        lo = min(lo, int(e[b]));
        hi = max(hi, int(e[b]));
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        lo = min(lo, __shfl_xor(lo, off, WAVE));
        hi = max(hi, __shfl_xor(hi, off, WAVE));
    }
    if (hi - lo > 3 && lane == 0) atomicOr(status, 1);
    // exponent bytes 0 (a scale below every normal float's) and 255 (NaN in the MX specification) cannot be read in place
    if ((lo < 1 || hi > 254) && lane == 0) atomicOr(status, 2);
    for (int byte = lane; bcodes && byte < nb / 4; byte += 64) {
        uint32_t v = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) v |= (uint32_t(min(int(e[4 * byte + j]) - lo, 3))) << (2 * j);
        bcodes[row * (nb / 4) + byte] = uint8_t(v);
    }
    // wscale = 2^(lo - 127 - 1); exponents below the normal range give the exact subnormal (or zero) value
    if (lane == 0) wscale[row] = ldexpf(1.0f, lo - 128);
}

}  // namespace scmx

using namespace scmx;

// A workgroup per row while the rows are few (by rows from 2049 values on: 8 rows x 2048 2.2 us with a wave per row, 2.4 with
// a workgroup; 4096 2.6 and 2.4), and for rows beyond a wave's registers (4000 rows x 12288 by rows: 36 us read twice, 23).
// Blocked, its 16-byte stores of a single row fill no line: the wave kernel then, up to 12288 values (4000
// rows x 12288: 40 us read twice, 29), and beyond, from 1024 rows on, the one that reads them twice (14336 values: 600 rows as
// fast either way, 1500 21.6 us and 22.8 by row workgroups, 4000 47.8 and 55.6).
static bool act_quant_rows_fit(int Mp, int K, bool blocked) {
    if (K % 32 || K > 16384) return false;
    if (K <= 2048) return blocked && Mp <= 128 && K > 512;
    return Mp <= (blocked && K > 12288 ? 1024 : 256) || (!blocked && K > 8192);
}
template <bool BLK>
static void launch_act_quant_rows(const uint16_t* x, int8_t* xq, float* xs, int M, int Mp, int K, hipStream_t st) {
    if (K <= 1024) act_quant_row_kernel<1, 1, BLK><<<dim3(Mp), dim3(64), 0, st>>>(x, xq, xs, M, K);
    else if (K <= 4096) act_quant_row_kernel<4, 1, BLK><<<dim3(Mp), dim3(256), 0, st>>>(x, xq, xs, M, K);
    else if (K <= 8192) act_quant_row_kernel<8, 1, BLK><<<dim3(Mp), dim3(512), 0, st>>>(x, xq, xs, M, K);
    else act_quant_row_kernel<8, 2, BLK><<<dim3(Mp), dim3(512), 0, st>>>(x, xq, xs, M, K);
}
// A wave per row: the smallest number of register pieces that holds it.  False: the row is too long (or K % 32 != 0).
template <bool BLK, bool SORT = false>
static bool launch_act_quant_waves(const uint16_t* x, int8_t* xq, float* xs, int M, int Mp, int K, hipStream_t st, SortedRows sort = {}) {
    if (K % 32 || K > (BLK ? 12288 : 8192)) return false;
    const dim3 grid(SORT ? unsigned(M) / 8u + unsigned(sort.n_experts) : BLK ? unsigned(Mp) / 8u : (unsigned(Mp) + 3u) / 4u);
    const dim3 block(BLK ? 512 : 256);
    auto go = [&](auto ch) {
        constexpr int CH = decltype(ch)::value;
        if (K == 512 * CH) act_quant_wave_kernel<CH, BLK, true, SORT><<<grid, block, 0, st>>>(x, xq, xs, M, Mp, K, sort);
        else act_quant_wave_kernel<CH, BLK, false, SORT><<<grid, block, 0, st>>>(x, xq, xs, M, Mp, K, sort);
    };
    const int ch = (K + 511) / 512;
    if (ch <= 1) go(std::integral_constant<int, 1>{});
    else if (ch <= 2) go(std::integral_constant<int, 2>{});
    else if (ch <= 3) go(std::integral_constant<int, 3>{});
    else if (ch <= 4) go(std::integral_constant<int, 4>{});
    else if (ch <= 6) go(std::integral_constant<int, 6>{});
    else if (ch <= 8) go(std::integral_constant<int, 8>{});
    else if (ch <= 10) go(std::integral_constant<int, 10>{});
    else if (ch <= 12) go(std::integral_constant<int, 12>{});
    else if (ch <= 16) go(std::integral_constant<int, 16>{});
    else if constexpr (BLK) go(std::integral_constant<int, 24>{});
    return true;
}

extern "C" {

#ifndef SCMX_BUILD_ID
#define SCMX_BUILD_ID "unknown"
#endif
// "scmx <version> (gfx950) <source revision the library was built from>"
const char* scmx_version(void) { return "scmx 0.2 (gfx950) " SCMX_BUILD_ID; }
const char* scmx_last_error(void) { return g_err; }

void scmx_mxfp4_format(scmx_format* f) {
    scmx_default_format(f);
    f->bc_bits = 8;
    f->n_mult = 0;
    for (int i = 0; i < 16; ++i) f->mult[i] = 0;
}

void scmx_default_format(scmx_format* f) {
    memset(f, 0, sizeof(*f));
    f->block = 32;
    f->bc_bits = 2;
    f->n_mult = 4;
    const int mag[8] = {0, 1, 2, 3, 4, 6, 8, 12};
    for (int i = 0; i < 8; ++i) f->code_mag[i] = mag[i];
    for (int i = 0; i < 4; ++i) f->mult[i] = 1 << i;
}

int scmx_unpack_i8(const scmx_format* fmt, const uint32_t* codes, const uint8_t* bcodes, int8_t* wq, int64_t n_rows,
                   int64_t K, void* stream) {
    DevFormat f;
    if (int rc = make_dev_format(fmt, &f)) return rc;
    if (f.e8m0) {
        set_error("unpack_i8: the E8M0 form needs the row scales to place a block; convert with scmx_mxfp4_to_sc first");
        return SCMX_ERR_FORMAT;
    }
    if (!codes || !bcodes || !wq || n_rows < 0 || K <= 0 || K % f.block || (K / f.block * f.bc_bits) % 8) {
        set_error("unpack_i8: need non-null pointers, K (%lld) a multiple of block %d and whole block-code bytes per row",
                  (long long)K, f.block);
        return SCMX_ERR_ARG;
    }
    if (K > (int64_t(1) << 30) || n_rows > (int64_t(1) << 40) / K) {   // keeps every count below 2^40 and the grid below 2^32
        set_error("unpack_i8: %lld x %lld weights are more than one launch takes (2^40)", (long long)n_rows, (long long)K);
        return SCMX_ERR_ARG;
    }
    if (n_rows == 0) return SCMX_OK;
    const int bc_row_bytes = int(K / f.block * f.bc_bits / 8);
    hipStream_t s = (hipStream_t)stream;
    if (K % 32 == 0 && (uintptr_t(codes) % 16 == 0) && (uintptr_t(wq) % 16 == 0)) {
        const int64_t groups = n_rows * (K / 32);
        unpack_i8_kernel<<<dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, s>>>(
            f, (const u32x4*)codes, bcodes, (u32x4*)wq, groups, int(K / 32), bc_row_bytes);
    } else {
        if (uintptr_t(wq) % 8) {
            set_error("unpack_i8: output must be 8-byte aligned");
            return SCMX_ERR_ARG;
        }
        const int64_t words = n_rows * (K / 8);
        unpack_i8_word_kernel<<<dim3((unsigned)((words + 255) / 256)), dim3(256), 0, s>>>(
            f, codes, bcodes, (u32x2*)wq, words, int(K / 8), bc_row_bytes);
    }
    return check_launch("unpack_i8");
}

int scmx_act_quant_blocked(const uint16_t* x, int8_t* xq, float* xs, int M, int Mp, int K, void* stream) {
    if (!x || !xq || !xs || M < 0 || Mp < M || Mp % 32 || Mp > (1 << 30) || K <= 0 || K % 32 || uintptr_t(x) % 16 ||
        uintptr_t(xq) % 16) {
        set_error("act_quant_blocked: need M <= Mp <= 2^30 with Mp %% 32 == 0 (Mp = %d), K %% 32 == 0 (K = %d), x and xq "
                  "16-byte aligned", Mp, K);
        return SCMX_ERR_ARG;
    }
    if (Mp == 0) return SCMX_OK;
    hipStream_t st = (hipStream_t)stream;
    if (act_quant_rows_fit(Mp, K, true)) launch_act_quant_rows<true>(x, xq, xs, M, Mp, K, st);
    else if (!launch_act_quant_waves<true>(x, xq, xs, M, Mp, K, st))
        act_quant_blocked_kernel<<<dim3(unsigned(Mp) / 8u), dim3(512), 0, st>>>(x, xq, xs, M, Mp, K);
    return check_launch("act_quant_blocked");
}

int scmx_act_quant(const uint16_t* x, int8_t* xq, float* xs, int M, int Mp, int K, void* stream) {
    if (!x || !xq || !xs || M < 0 || Mp < M || Mp > (1 << 30) || K <= 0 || K % 8 || uintptr_t(x) % 16 || uintptr_t(xq) % 8) {
        set_error("act_quant: need M <= Mp <= 2^30, K %% 8 == 0 (K = %d), x 16-byte and xq 8-byte aligned", K);
        return SCMX_ERR_ARG;
    }
    if (Mp == 0) return SCMX_OK;
    hipStream_t st = (hipStream_t)stream;
    if (uintptr_t(xq) % 16 == 0 && act_quant_rows_fit(Mp, K, false)) launch_act_quant_rows<false>(x, xq, xs, M, Mp, K, st);
    else if (!launch_act_quant_waves<false>(x, xq, xs, M, Mp, K, st))
        act_quant_kernel<<<dim3(Mp), dim3(256), 0, st>>>(x, xq, xs, M, K);
    return check_launch("act_quant");
}

static int check_sorted(const char* who, const int32_t* off, const int32_t* tstart, int n_experts, int R, int K, SortedRows* s) {
    if (!off || !tstart || n_experts < 1 || n_experts > (1 << 20) || R < 0 || K <= 0 || K % 128 ||
        (uint64_t(R) / 256 + 1 + uint64_t(n_experts)) * 256 * uint64_t(K) > 0xFFFFFFFFull) {
        set_error("%s: need off / tstart, 1 <= n_experts <= 2^20 (%d), K %% 128 == 0 (K = %d) and slots within 2^32 bytes (R = %d)", who,
                  n_experts, K, R);
        return SCMX_ERR_ARG;
    }
    *s = SortedRows{off, tstart, n_experts};
    return SCMX_OK;
}

int scmx_moe_gather_blocked(const int8_t* xq, const float* xscale, const int32_t* gather, const int32_t* off, const int32_t* tstart,
                            int n_experts, int R, int K, int8_t* out, float* out_scale, void* stream) {
    SortedRows s;
    if (int rc = check_sorted("moe_gather_blocked", off, tstart, n_experts, R, K, &s)) return rc;
    if (!xq || !xscale || !gather || !out || !out_scale || uintptr_t(xq) % 16 || uintptr_t(out) % 16) {
        set_error("moe_gather_blocked: null pointer argument, or xq / out not 16-byte aligned");
        return SCMX_ERR_ARG;
    }
    if (R == 0) return SCMX_OK;
    const dim3 grid(unsigned(R) / 32u + unsigned(n_experts));
    moe_gather_blocked_kernel<<<grid, dim3(256), 0, (hipStream_t)stream>>>(xq, xscale, gather, s, K, out, out_scale);
    return check_launch("moe_gather_blocked");
}

int scmx_act_quant_sorted(const uint16_t* x, const int32_t* off, const int32_t* tstart, int n_experts, int R, int K, int8_t* xq, float* xs,
                          void* stream) {
    SortedRows s;
    if (int rc = check_sorted("act_quant_sorted", off, tstart, n_experts, R, K, &s)) return rc;
    if (!x || !xq || !xs || uintptr_t(x) % 16 || uintptr_t(xq) % 16 || K > 12288) {
        set_error("act_quant_sorted: need x, xq and xs, x and xq 16-byte aligned, K <= 12288 (K = %d)", K);
        return SCMX_ERR_ARG;
    }
    if (R == 0) return SCMX_OK;
    launch_act_quant_waves<true, true>(x, xq, xs, R, R, K, (hipStream_t)stream, s);
    return check_launch("act_quant_sorted");
}

int scmx_rot_quant(const uint16_t* x, const float* signs, int8_t* xq, float* xs, int M, int Mp, int K, void* stream) {
    if (!x || !signs || !xq || !xs || M < 0 || Mp < M || K <= 0 || K % 32 || K > 8192) {
        set_error("rot_quant: null pointer, Mp < M, or K not a multiple of 32 in 32..8192 (M=%d Mp=%d K=%d)", M, Mp, K);
        return SCMX_ERR_ARG;
    }
    if (uintptr_t(x) % 8 || uintptr_t(signs) % 16 || uintptr_t(xq) % 4) {
        set_error("rot_quant: x must be 8-byte, signs 16-byte, xq 4-byte aligned");
        return SCMX_ERR_ARG;
    }
    if (Mp == 0) return SCMX_OK;
    rot_quant_kernel<<<dim3(Mp), dim3(256), 0, (hipStream_t)stream>>>(x, signs, xq, xs, M, K);
    return check_launch("rot_quant");
}

int scmx_mxfp4_to_sc(const uint8_t* e8m0, uint8_t* bcodes, float* wscale, int32_t* status, int64_t N, int64_t K,
                     void* stream) {
    if (!e8m0 || !wscale || !status || N < 0 || N > (int64_t(1) << 32) || K <= 0 || K % 128 || K > (int64_t(1) << 30)) {
        set_error("mxfp4_to_sc: need non-null pointers, N <= 2^32 and K %% 128 == 0, K <= 2^30 (K = %lld)", (long long)K);
        return SCMX_ERR_ARG;
    }
    if (N == 0) return SCMX_OK;
    mxfp4_to_sc_kernel<<<dim3((unsigned)((N + 3) / 4)), dim3(256), 0, (hipStream_t)stream>>>(e8m0, bcodes, wscale,
                                                                                               status, N, int(K / 32));
    return check_launch("mxfp4_to_sc");
}

}  // extern "C"

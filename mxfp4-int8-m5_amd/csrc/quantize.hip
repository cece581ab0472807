// SC-MXFP4 weight quantizer on the device: float weights -> packed codes, block codes and row scales.
//
// Restates, bit for bit, sim/mx_int8.py:39-109 (block exponent search, spread constraint, E2M1 rounding, INT8
// embedding) followed by the packing of sim/make_testcase.py:26-44 and e2e/sc_format.py:93-111.  A thread owns one
// block: its weights stay in registers from the search to the packing, sums over a block need no cross-lane traffic,
// and a workgroup takes as many whole rows as give its 256 threads a block each.
//
// The host decides between exponents by a strict "<" on float64 sums taken in a fixed order.  Here the sums are formed
// in float32 first (which scaling by powers of two leaves exact up to the sums' own rounding), and only where two of
// them are too close for float32 to tell apart is the block summed again in float64 in the host's order: eight running
// sums r[j] = ((a[j] + a[8+j]) + a[16+j]) + a[24+j], then ((r0+r1)+(r2+r3)) + ((r4+r5)+(r6+r7)).
#include <climits>
#include <type_traits>

#include "scmx_common.h"

namespace scmx {

constexpr int QNT = 256;
constexpr int MAX_SPREAD = 3;   // sim/mx_int8.py:18

__device__ __forceinline__ double pow2_f64(int e) { return __longlong_as_double((long long)(1023 + e) << 52); }

// Index of the E2M1 level nearest to |x| (saturating at 6); a midpoint goes to the lower level (sim/mx_int8.py:23-25).
__device__ __forceinline__ int e2m1_index(double x) {
    const double a = fmin(fabs(x), 6.0);
    return int(a > 0.25) + int(a > 0.75) + int(a > 1.25) + int(a > 1.75) + int(a > 2.5) + int(a > 3.5) + int(a > 5.0);
}
__device__ __forceinline__ double e2m1_level(int idx) {   // 0, .5, 1, 1.5, 2, 3, 4, 6
    return idx <= 4 ? 0.5 * idx : (idx == 5 ? 3.0 : (idx == 6 ? 4.0 : 6.0));
}

// Squared error of BLOCK consecutive weights quantized at exponent e (sim/mx_int8.py:34-36), in float64 and summed in
// the host's order.  Reads the weights again: it decides near ties only.
template <int BLOCK, typename W>
__device__ double block_sq_err(W&& weight, int e) {
    double r[8];
#pragma unroll 1
    for (int i = 0; i < BLOCK; i += 8) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const double b = double(weight(i + j));
            const double x = b * pow2_f64(-e);
            const double q = e2m1_level(e2m1_index(x));
            const double d = (x < 0.0 ? -q : q) * pow2_f64(e) - b;
            r[j] = i == 0 ? d * d : r[j] + d * d;
        }
    }
    return ((r[0] + r[1]) + (r[2] + r[3])) + ((r[4] + r[5]) + (r[6] + r[7]));
}

// The same with a lane per weight b, the block's lanes side by side: the sum in the first of them, by the same additions.
template <int BLOCK>
__device__ double lane_sq_err(double b, int e) {
    const double x = b * pow2_f64(-e);
    const double q = e2m1_level(e2m1_index(x));
    const double d = (x < 0.0 ? -q : q) * pow2_f64(e) - b;
    const double sq = d * d;
    double r = sq + __shfl_down(sq, 8, BLOCK);
    if (BLOCK == 32) {
        r = r + __shfl_down(sq, 16, BLOCK);
        r = r + __shfl_down(sq, 24, BLOCK);
    }
    r = r + __shfl_xor(r, 1, BLOCK);
    r = r + __shfl_xor(r, 2, BLOCK);
    return r + __shfl_xor(r, 4, BLOCK);
}

// BLOCK consecutive weights into registers; vec: the address is 16-byte aligned.
template <int BLOCK, bool BF16>
__device__ __forceinline__ void load_block(const void* __restrict__ w, size_t at, bool vec, float (&v)[BLOCK]) {
    if (BF16) {
        const uint16_t* p = reinterpret_cast<const uint16_t*>(w) + at;
        if (vec) {
#pragma unroll
            for (int i = 0; i < BLOCK / 8; ++i) {
                const u32x4 u = reinterpret_cast<const u32x4*>(p)[i];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    v[8 * i + 2 * j] = __uint_as_float(u[j] << 16);
                    v[8 * i + 2 * j + 1] = __uint_as_float(u[j] & 0xFFFF0000u);
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < BLOCK; ++i) v[i] = bf16_to_f32(p[i]);
        }
    } else {
        const float* p = reinterpret_cast<const float*>(w) + at;
        if (vec) {
#pragma unroll
            for (int i = 0; i < BLOCK / 4; ++i) {
                const f32x4 u = reinterpret_cast<const f32x4*>(p)[i];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[4 * i + j] = u[j];
            }
        } else {
#pragma unroll
            for (int i = 0; i < BLOCK; ++i) v[i] = p[i];
        }
    }
}

// The code words of a block leave in 16- or 8-byte stores where the pointer allows it.
template <int BLOCK>
__device__ __forceinline__ void store_codes(uint32_t* __restrict__ dst, bool vec, const uint32_t (&c)[BLOCK / 8]) {
    if (BLOCK == 32 && vec) {
        *reinterpret_cast<u32x4*>(dst) = u32x4{c[0], c[1], c[BLOCK / 8 - 2], c[BLOCK / 8 - 1]};
    } else if (vec) {
        *reinterpret_cast<u32x2*>(dst) = u32x2{c[0], c[1]};
    } else {
#pragma unroll
        for (int i = 0; i < BLOCK / 8; ++i) dst[i] = c[i];
    }
}

typedef float f32x2_t __attribute__((ext_vector_type(2)));

// Squared error, in units of the square of 2^e0, of the block x * 2^e0 at exponent e0 + log2(scale).  The FP4 conversion
// does the rounding: it takes a tie to the even code where the host takes the lower one, which is the same distance away.
template <int BLOCK>
__device__ __forceinline__ float fp4_sq_err(const float (&x)[BLOCK], float scale) {
    float r0 = 0.0f, r1 = 0.0f;
#pragma unroll
    for (int i = 0; i < BLOCK; i += 2) {
        const uint32_t c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, x[i], x[i + 1], scale, 0);
        const f32x2_t v = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, scale, 0);
        const float d0 = v[0] - x[i], d1 = v[1] - x[i + 1];   // exact: the difference fits 24 bits
        r0 = __builtin_fmaf(d0, d0, r0);
        r1 = __builtin_fmaf(d1, d1, r1);
    }
    return r0 + r1;
}

// The same for weights born in bf16, as half-precision pairs: two conversions, a packed difference and a dot product per
// two weights, two instructions a weight for three.  Scaled to magnitudes below 8 their eight bits fit half precision
// down to 2^-17.  A difference is a multiple of its weight's last bit and no larger than the weight (or below 5 at a last
// bit of 2^-5, where it saturates), so it is exact too, and the dot product adds exact squares in float32.  What is
// smaller rounds to zero at every exponent tried, as all below 1/8 does: it adds the same to all three sums, whatever is
// left of it.  The others' squares are multiples of 2^-20: two sums differ by that or not at all.
template <int BLOCK>
__device__ __forceinline__ float fp4_sq_err_half(const half2_t (&x)[BLOCK / 2], float scale) {
    float r0 = 0.0f, r1 = 0.0f;
#pragma unroll
    for (int i = 0; i < BLOCK / 2; i += 4) {   // the conversion writes one byte and keeps the others: four share a register
        uint32_t c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(0u, x[i], scale, 0);
        c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(c, x[i + 1], scale, 1);
        c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(c, x[i + 2], scale, 2);
        c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(c, x[i + 3], scale, 3);
        const half2_t d0 = half2_t(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(c, scale, 0)) - x[i];
        const half2_t d1 = half2_t(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(c, scale, 1)) - x[i + 1];
        const half2_t d2 = half2_t(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(c, scale, 2)) - x[i + 2];
        const half2_t d3 = half2_t(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(c, scale, 3)) - x[i + 3];
        r0 = __builtin_amdgcn_fdot2(d0, d0, r0, false);
        r1 = __builtin_amdgcn_fdot2(d1, d1, r1, false);
        r0 = __builtin_amdgcn_fdot2(d2, d2, r0, false);
        r1 = __builtin_amdgcn_fdot2(d3, d3, r1, false);
    }
    return r0 + r1;
}

// Eight weights' codes at a power-of-two scale, signs included: a word of the packed layout.
__device__ __forceinline__ uint32_t fp4_word(const float* x, float scale) {
    uint32_t c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, x[0], x[1], scale, 0);
    c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(c, x[2], x[3], scale, 1);
    c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(c, x[4], x[5], scale, 2);
    return __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(c, x[6], x[7], scale, 3);
}
// A zero code has no sign.
__device__ __forceinline__ uint32_t unsigned_zeros(uint32_t c) {
    const uint32_t m = c & 0x77777777u;
    return m | (c & (m + 0x77777777u) & 0x88888888u);
}

// nb = K / BLOCK blocks per row, `rows` rows per workgroup.  Bound: vector ALU: three trial roundings with their error
// sums. The codes come from the conversion, which takes a midpoint to the even code where the host takes the lower one.
// bf16 weights have eight bits: 2^-12 smaller, one on a midpoint lies below it and no other changes sides.  float32
// weights are converted as they are and 2^-23 smaller: where both agree so does the host (a midpoint whose even code is
// the lower one, or none near); the others' blocks take the arithmetic.  That arithmetic for every weight took 28.8 us
// where the conversion's 22.2 stood beside it, near ties summed by one lane of the wave 44, a lane per weight and every
// candidate in float64 across lanes 234 (12288 x 2048, bf16, 32-blocks).
// Registers decide how many waves hide the conversions' latency: four a SIMD need 128 a thread.  16-blocks are held to
// that, at the price of 40 spilled registers (most around the float64 sums of near ties, which few blocks take); bf16
// 32-blocks fit only if the weights are read again for their codes (L2 has them) instead of kept over the barrier; float32
// 32-blocks fit neither way.  us, before / with half-precision trials / so bounded, 12288 x 2048: bf16
// 32-blocks 24.3 / 23.9 / 21.8 (bounded without reading again 24.7; five or six waves 29), 16-blocks 47.7 / 47.8 / 31.6;
// float32 32-blocks 28.9 (bounded 32.3, read again 31.5), 16-blocks 50.4 / - / 35.9.  4096 x 12288: bf16 47.1 -> 39.7
// and 70.8 -> 50.2, float32 16-blocks 76.3 -> 67.3.
template <int BLOCK, bool BF16>
__global__ __launch_bounds__(QNT, BLOCK == 16 || BF16 ? 4 : 1) void quantize_sc_kernel(
    const void* __restrict__ w, uint32_t* __restrict__ codes, uint8_t* __restrict__ bcodes, float* __restrict__ wscale,
    int64_t N, int K, int rows, bool vec) {
    constexpr bool AGAIN = BLOCK == 32 && BF16;   // the weights are read again for their codes
    extern __shared__ int s_e[];   // rows x nb block exponents, then the rows' smallest allowed and lowest exponents
    const int nb = K / BLOCK;
    const size_t row0 = size_t(blockIdx.x) * rows;
    const int live = int(min(int64_t(rows), N - int64_t(row0)));
    const int total = live * nb, tid = threadIdx.x, lane = tid & 63;
    int* s_floor = s_e + rows * nb;
    int* s_lo = s_floor + rows;
    constexpr int EMPTY = INT_MIN;   // an all-zero block: the host's -inf
    const size_t base = row0 * K;

    // ---- exponent of every block (sim/mx_int8.py:39-65, rule "search") --------------------------------------------
    float v[BLOCK];
    for (int b0 = tid & ~63; b0 < total; b0 += QNT) {   // whole waves, for the ties
        const int b = b0 + lane;
        const size_t at = base + size_t(b) * BLOCK;
        int chosen = EMPTY, e0 = 0;
        bool tie = false;
        auto weight = [&](size_t i) -> float {
            if (BF16) return bf16_to_f32(reinterpret_cast<const uint16_t*>(w)[i]);
            return reinterpret_cast<const float*>(w)[i];
        };
        if (b < total) {
            load_block<BLOCK, BF16>(w, at, vec, v);
            float amax = 0.0f;
#pragma unroll
            for (int i = 0; i < BLOCK; ++i) amax = fmaxf(amax, fabsf(v[i]));
            if (amax > 0.0f) {
                // floor(log2 amax) of a float32-born value is its binary exponent
                e0 = int((__double_as_longlong(double(amax)) >> 52) & 0x7FF) - 1023 - 2;
                float s0, sm, sp;
                if constexpr (BF16) {
                    half2_t x[BLOCK / 2];
#pragma unroll
                    for (int i = 0; i < BLOCK; i += 2)
                        x[i / 2] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(__builtin_amdgcn_ldexpf(v[i], -e0),
                                                                                         __builtin_amdgcn_ldexpf(v[i + 1], -e0)));
                    s0 = fp4_sq_err_half<BLOCK>(x, 1.0f), sm = fp4_sq_err_half<BLOCK>(x, 0.5f), sp = fp4_sq_err_half<BLOCK>(x, 2.0f);
                } else {
                    float x[BLOCK];
#pragma unroll
                    for (int i = 0; i < BLOCK; ++i) x[i] = __builtin_amdgcn_ldexpf(v[i], -e0);
                    s0 = fp4_sq_err<BLOCK>(x, 1.0f), sm = fp4_sq_err<BLOCK>(x, 0.5f), sp = fp4_sq_err<BLOCK>(x, 2.0f);
                }
                // A float32 sum of 32 squares of exact differences is within 32 half-ulps (2e-6) of the exact one, the
                // host's float64 sum within 1e-14: apart by more than 1e-5, the sums order alike.  (Below 1e-30 squares
                // underflow.)
                auto close = [](float a, float b) { return !(fabsf(a - b) > 1e-5f * fmaxf(a, b)) || fmaxf(a, b) < 1e-30f; };
                const float s1 = sm < s0 ? sm : s0;
                tie = close(sm, s0) || close(sp, s1);
                chosen = sp < s1 ? e0 + 1 : sm < s0 ? e0 - 1 : e0;
            }
        }
        // Near ties in float64.  A few of them the wave takes one after the other, a lane per weight (about 1.5 us
        // each); where many lanes have one, each sums its own (15 us in all, as one does: a matrix of a few rows waited
        // for its one tie).
        uint64_t ties = __ballot(tie);
        auto decide = [&](double t0, double tm, double tp) {
            double best = t0;
            int e = e0;
            if (tm < best) {
                best = tm;
                e = e0 - 1;
            }
            return tp < best ? e0 + 1 : e;
        };
        if (__popcll(ties) > 8) {
            if (tie) {
                auto mine = [&](int i) { return weight(at + i); };
                chosen = decide(block_sq_err<BLOCK>(mine, e0), block_sq_err<BLOCK>(mine, e0 - 1), block_sq_err<BLOCK>(mine, e0 + 1));
            }
        } else {
            while (ties) {
                const int src = __ffsll((unsigned long long)ties) - 1;
                ties &= ties - 1;
                const int e = __shfl(e0, src, WAVE), group = lane / BLOCK;
                const double a = double(weight(base + size_t(b0 + src) * BLOCK + lane % BLOCK));
                // lane group 0: exponent e, group 1: e - 1, the others e + 1 (of 32 lanes there are two groups: once
                // more)
                const double first = lane_sq_err<BLOCK>(a, group == 0 ? e : group == 1 ? e - 1 : e + 1);
                const double third = BLOCK == 16 ? first : lane_sq_err<BLOCK>(a, e + 1);
                const double t0 = __shfl(first, 0, WAVE), tm = __shfl(first, BLOCK, WAVE);
                const double tp = __shfl(third, BLOCK == 16 ? 32 : 0, WAVE);
                if (lane == src) chosen = decide(t0, tm, tp);
            }
        }
        if (b < total) s_e[b] = chosen;
    }
    __syncthreads();

    // ---- row constraint (sim/mx_int8.py:68-81) and the row's lowest exponent (sim/mx_int8.py:92-109): as many lanes per row, a
    // wave at most, as let the rows go side by side (a wave each, 64 rows took 16 turns: 64 x 128 13 us) ---------------------
    int per = 64;
    while (per * rows > QNT && per > 1) per >>= 1;
    for (int r = tid / per; r < live; r += QNT / per) {
        const int l = tid & (per - 1);
        int top = EMPTY;
        for (int i = l; i < nb; i += per) top = max(top, s_e[r * nb + i]);
        for (int off = per >> 1; off >= 1; off >>= 1) top = max(top, __shfl_xor(top, off, WAVE));
        if (top == EMPTY) top = 0;   // all-zero row
        const int floor_e = top - MAX_SPREAD;
        int lo = INT_MAX;
        for (int i = l; i < nb; i += per) lo = min(lo, max(s_e[r * nb + i], floor_e));
        for (int off = per >> 1; off >= 1; off >>= 1) lo = min(lo, __shfl_xor(lo, off, WAVE));
        if (l == 0) {
            s_floor[r] = floor_e;
            s_lo[r] = lo;
            wscale[row0 + r] = float(pow2_f64(lo - 1));   // 2^(E_lo - 1), sim/mx_int8.py:101
        }
    }
    __syncthreads();

    // ---- codes (sim/make_testcase.py:36-39, e2e/sc_format.py:72-73) ------------------------------------------------
    for (int b = tid; b < total; b += QNT) {
        const size_t at = base + size_t(b) * BLOCK;
        if (AGAIN || total > QNT) load_block<BLOCK, BF16>(w, at, vec, v);   // (or more than one block per thread)
        const int e = max(s_e[b], s_floor[b / nb]);
        uint32_t c[BLOCK / 8], open = 1u;
        if (e > -100 && e < 120) {   // (its scale is an ordinary float32)
            const float scale = __uint_as_float(uint32_t(127 + e) << 23);
            float y[BLOCK], sum = 0.0f;
#pragma unroll
            for (int i = 0; i < BLOCK; ++i) {
                y[i] = v[i] * (BF16 ? 1.0f - 0x1p-12f : 1.0f - 0x1p-23f);
                sum += y[i];
            }
            open = uint32_t(!(fabsf(sum) < 3e38f));   // infinities and NaN
#pragma unroll
            for (int q = 0; q < BLOCK / 8; ++q) {
                c[q] = fp4_word(y + 8 * q, scale);
                if (!BF16) open |= c[q] ^ fp4_word(v + 8 * q, scale);
                c[q] = unsigned_zeros(c[q]);
            }
        }
        if (open) {
#pragma unroll
            for (int i = 0; i < BLOCK / 8; ++i) c[i] = 0u;
#pragma unroll
            for (int i = 0; i < BLOCK; ++i) {
                // index of the E2M1 level nearest to a = |w| 2^-e, saturating at 7, a midpoint to the lower level
                // (sim/mx_int8.py:23-25): levels are t / 2 apart from t = 2^max(floor(log2 a), 0) on, so the index is
                // ceil(2 a / t - 1/2) plus two per octave above the first
                const float a = fabsf(__builtin_amdgcn_ldexpf(v[i], -e));
                const uint32_t t = max(__float_as_uint(a) & 0x7F800000u, 0x3F800000u);
                const float m = ceilf(__builtin_fmaf(a, __uint_as_float(0x7F800000u - t), -0.5f));
                const int idx = min(int(m) + 2 * (int(t >> 23) - 127), 7);
                c[i >> 3] |= (uint32_t(idx) | ((v[i] < 0.0f && idx > 0) ? 8u : 0u)) << (4 * (i & 7));
            }
        }
        store_codes<BLOCK>(codes + at / 8, vec, c);
    }
    // block codes: shift = e - lo in 0..3, 2 bits each, four blocks per byte (e2e/sc_format.py:14)
    for (int j = tid; j < total / 4; j += QNT) {
        const int r = 4 * j / nb;
        uint32_t byte = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) byte |= uint32_t(max(s_e[4 * j + i], s_floor[r]) - s_lo[r]) << (2 * i);
        bcodes[row0 * (nb / 4) + j] = uint8_t(byte);
    }
}

// ---- the integer-exact format family: w = base[row] * mult[block] * sign * code ------------------------------------
// Restates sim/formats.py:64-107 in float32, as the host computes it: the largest row base is
// peak / (largest multiplier * largest code); 8 bases per octave below it are tried in descending order, each with
// the per-block multiplier of least squared error (first minimum), and a candidate replaces the best so far only
// when its total error over the row is strictly smaller.  Block errors and row totals are summed in the order of
// the host's pairwise reduction.  A thread owns one block and keeps its magnitudes in registers over all trials.
struct FamilyArgs {
    float cb[8];      // code magnitudes
    float cut[7];     // midpoints between neighbouring magnitudes
    float mult[16];
    float half_inv[16];   // 0.5 / mult
    int n_mult, bc_bits;
};

// numpy's pairwise sum of n contiguous float32 values (n <= 128: eight strided running sums, a fixed tree, then the
// n % 8 tail; longer inputs are split in two at a multiple of 8 below the middle).  DEPTH splits at most: four bring
// any n <= 1024 down to 128.
template <int DEPTH>
__device__ __forceinline__ float np_pairwise_sum(const float* a, int n) {
    if constexpr (DEPTH > 0) {
        if (n > 128) {
            int n2 = n / 2;
            n2 -= n2 % 8;
            const float lower = np_pairwise_sum<DEPTH - 1>(a, n2);
            return __fadd_rn(lower, np_pairwise_sum<DEPTH - 1>(a + n2, n - n2));
        }
    }
    if (n < 8) {
        float r = 0.0f;
        for (int i = 0; i < n; ++i) r = __fadd_rn(r, a[i]);
        return r;
    }
    float r[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) r[j] = a[j];
    int i = 8;
    for (; i < n - (n % 8); i += 8) {
#pragma unroll
        for (int j = 0; j < 8; ++j) r[j] = __fadd_rn(r[j], a[i + j]);
    }
    float res = __fadd_rn(__fadd_rn(__fadd_rn(r[0], r[1]), __fadd_rn(r[2], r[3])),
                          __fadd_rn(__fadd_rn(r[4], r[5]), __fadd_rn(r[6], r[7])));
    for (; i < n; ++i) res = __fadd_rn(res, a[i]);
    return res;
}

__device__ __forceinline__ int family_index(const FamilyArgs& f, float x) {   // nearest code, ties to the lower one
    const float a = fminf(fabsf(x), f.cb[7]);
    int idx = 0;
#pragma unroll
    for (int i = 0; i < 7; ++i) idx += int(a > f.cut[i]);
    return idx;
}
// sign(a) times its magnitude, for a >= 0: a zero has no sign and costs nothing, also where the smallest magnitude is
// not 0 (in the E2M1 codebook it is).
template <bool E2M1>
__device__ __forceinline__ float family_level(const FamilyArgs& f, float a) {
    float v = !E2M1 && a > 0.0f ? f.cb[0] : 0.0f;
#pragma unroll
    for (int i = 0; i < 7; ++i) v = a > f.cut[i] ? f.cb[i + 1] : v;
    return v;
}

// Squared error of the block of magnitudes aw at scale sc, as the host evaluates it (float32, its order of sums).
template <int BLOCK, bool E2M1>
__device__ __forceinline__ float family_sq_err(const FamilyArgs& f, const float (&aw)[BLOCK], float sc) {
    float r[8];
#pragma unroll
    for (int i = 0; i < BLOCK; ++i) {
        const float v = family_level<E2M1>(f, __fdiv_rn(aw[i], sc));
        const float d = __fsub_rn(__fmul_rn(v, sc), aw[i]);
        const float sq = __fmul_rn(d, d);
        r[i & 7] = i < 8 ? sq : __fadd_rn(r[i & 7], sq);
    }
    return __fadd_rn(__fadd_rn(__fadd_rn(r[0], r[1]), __fadd_rn(r[2], r[3])),
                     __fadd_rn(__fadd_rn(r[4], r[5]), __fadd_rn(r[6], r[7])));
}

// The same for the E2M1 codebook (0, 1, 2, 3, 4, 6, 8, 12 = twice the FP4 values) through the FP4 conversion: about 13
// instructions per weight instead of 40.  The quotient is formed twice with an approximate reciprocal, 2^-20 too large
// and 2^-20 too small: where both round to the same code so does the correctly rounded quotient, whose error lies
// between; where they differ (a quotient next to a midpoint) *same is cleared and the caller takes the form above.
template <int BLOCK>
__device__ __forceinline__ float family_sq_err_e2m1(const float (&aw)[BLOCK], float sc, bool* same) {
    const float h = 0.5f * __builtin_amdgcn_rcpf(sc);
    const float up = h * 1.00000095367431640625f, dn = h * 0.99999904632568359375f;
    float r[8];
    uint32_t diff = 0;
#pragma unroll
    for (int i = 0; i < BLOCK; i += 2) {
        const uint32_t cu = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, aw[i] * up, aw[i + 1] * up, 1.0f, 0);
        const uint32_t cd = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, aw[i] * dn, aw[i + 1] * dn, 1.0f, 0);
        diff |= cu ^ cd;
        const f32x2_t v = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(cd, 2.0f, 0);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const float d = __fsub_rn(__fmul_rn(v[k], sc), aw[i + k]);
            const float sq = __fmul_rn(d, d);
            r[(i + k) & 7] = i < 8 ? sq : __fadd_rn(r[(i + k) & 7], sq);
        }
    }
    *same = diff == 0u;
    return __fadd_rn(__fadd_rn(__fadd_rn(r[0], r[1]), __fadd_rn(r[2], r[3])),
                     __fadd_rn(__fadd_rn(r[4], r[5]), __fadd_rn(r[6], r[7])));
}

// That error to within the bound below, at 4 instructions per weight: one quotient, the conversion there and back, two
// fused multiply-adds.
template <int BLOCK>
__device__ __forceinline__ float family_sq_err_near(const float (&aw)[BLOCK], float sc, float h) {   // h = 0.5 / sc
    float r0 = 0.0f, r1 = 0.0f;
    auto add = [&](int i, f32x2_t v) {
        const float d0 = __builtin_fmaf(v[0], sc, -aw[i]), d1 = __builtin_fmaf(v[1], sc, -aw[i + 1]);
        r0 = __builtin_fmaf(d0, d0, r0);
        r1 = __builtin_fmaf(d1, d1, r1);
    };
#pragma unroll
    for (int i = 0; i < BLOCK; i += 8) {   // the conversion writes one byte and keeps the others: four share a register
        uint32_t c = 0u;
        c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(c, aw[i] * h, aw[i + 1] * h, 1.0f, 0);
        c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(c, aw[i + 2] * h, aw[i + 3] * h, 1.0f, 1);
        c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(c, aw[i + 4] * h, aw[i + 5] * h, 1.0f, 2);
        c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(c, aw[i + 6] * h, aw[i + 7] * h, 1.0f, 3);
        add(i, __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, 2.0f, 0));
        add(i + 2, __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, 2.0f, 1));
        add(i + 4, __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, 2.0f, 2));
        add(i + 6, __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, 2.0f, 3));
    }
    return r0 + r1;
}
// How far the root of that sum can be from the root of the host's, twice (the two sides of a comparison), in parts of
// the norm of the weights summed over.  With D_i the distance of weight i to the nearest level, D_i <= |w_i| (zero is a
// level): the level taken is the nearest to a quotient 2^-21.4 off at most, so the difference to it exceeds D_i by
// 2^-20.4 |w_i| at most; seventeen additions are 2^-20 of the sum, 2^-20.9 of its root.  The host's own roundings are
// 2^-21 of the norm.  By the triangle inequality 1.75 x 2^-20 in all, twice 2^-18.2; for a row, whose sum of block
// errors rounds by 2^-20.4 of its root on either side, 2^-17.3.
constexpr float NEAR = 7.62939453125e-6f;   // 2^-17

constexpr int FAM_ROWS = 4;   // rows per workgroup at most: more are needed only for K < 1024, and their tables cost LDS

// Bound: vector ALU.  In the E2M1 codebook a trial is first evaluated to 2^-19 (family_sq_err_near): that settles
// nearly every multiplier of a block and base, and all but one or two of a row's bases; only what it leaves open is
// evaluated as the host does. Multipliers run from the largest down and end where clipping the block's largest weight
// alone costs more than the best so far, in every lane.  2048 x 2048 bf16, ten multipliers: 67 us; 130 with every trial
// as the host evaluates it (13 instructions a weight), 520 with a lane per weight, a correctly rounded division per
// trial and the sums across lanes.
// BASES: 1 where there are fewer blocks than lanes, each of which would run all trials of one (64 x 128, ten
// multipliers 27 -> 11 us). In the E2M1 codebook 4 beyond that: twice the waves to hide the conversions' latency and
// the uneven number of trials (600 x 2048 44 us with all eight in a thread, 34 with four; 4096 x 2048 114 and 116).
template <int BLOCK, bool BF16, bool E2M1, int BASES>   // bases per thread
__global__ __launch_bounds__(QNT) void quantize_family_kernel(const void* __restrict__ w, uint32_t* __restrict__ codes,
                                                             uint8_t* __restrict__ bcodes, float* __restrict__ wscale,
                                                             int64_t N, int K, int rows, bool vec, const FamilyArgs f) {
    extern __shared__ float s_f[];   // per row: 8 x nb block errors; then 8 x nb multiplier indices per row
    __shared__ uint32_t s_peak[FAM_ROWS];
    __shared__ float s_tot[FAM_ROWS][8];
    __shared__ int s_best[FAM_ROWS];
    __shared__ float s_norm[FAM_ROWS];     // sum of squares of the row
    __shared__ uint32_t s_open[FAM_ROWS];  // bases whose totals have to be summed as the host does
    const int nb = K / BLOCK;
    float* s_err = s_f;
    uint8_t* s_mi = reinterpret_cast<uint8_t*>(s_f + size_t(rows) * 8 * nb);
    const size_t row0 = size_t(blockIdx.x) * rows;
    const int live = int(min(int64_t(rows), N - int64_t(row0)));
    const int total = live * nb, tid = threadIdx.x;
    const size_t wbase = row0 * K;
    // row peaks (bit patterns of non-negative floats order like the floats)
    if (tid < FAM_ROWS) {
        s_peak[tid] = 0u;
        s_norm[tid] = 0.0f;
        s_open[tid] = 0u;
    }
    __syncthreads();
    float v[BLOCK];
    for (int b = tid; b < total; b += QNT) {
        load_block<BLOCK, BF16>(w, wbase + size_t(b) * BLOCK, vec, v);
        float amax = 0.0f;
#pragma unroll
        for (int i = 0; i < BLOCK; ++i) amax = fmaxf(amax, fabsf(v[i]));
        atomicMax(&s_peak[b / nb], __float_as_uint(amax));
    }
    __syncthreads();
    // 2^(-j/8) rounded to float32: the candidate ladder of one octave
    const float ladder[8] = {1.0f, 0.9170040488243103f, 0.8408964276313782f, 0.7711054086685181f, 0.7071067690849304f,
                             0.6484197974205017f, 0.5946035385131836f, 0.5452538728713989f};
    auto row_top = [&](int r) {
        float peak = __uint_as_float(s_peak[r]);
        if (peak == 0.0f) peak = 1.0f;
        return __fdiv_rn(peak, __fmul_rn(f.mult[f.n_mult - 1], f.cb[7]));
    };

    // ---- per candidate base and block: the best multiplier and its error ------------------------------------------
    // The trial of one scale as the host evaluates it (a scale near the ends of the float32 range leaves its reciprocal
    // no room).
    auto in_range = [](float sc) { return sc > 1e-30f && sc < 1e30f; };
    auto trial = [&](const float (&aw)[BLOCK], float sc) {
        bool same = false;
        float e = 0.0f;
        if (E2M1 && in_range(sc)) e = family_sq_err_e2m1<BLOCK>(aw, sc, &same);
        if (!same) e = family_sq_err<BLOCK, E2M1>(f, aw, sc);
        return e;
    };
    for (int t = tid; t < total * (8 / BASES); t += QNT) {
        const int b = t / (8 / BASES), j0 = t % (8 / BASES) * BASES;
        if (BASES < 8 || total > QNT) load_block<BLOCK, BF16>(w, wbase + size_t(b) * BLOCK, vec, v);
        const int r = b / nb, kb = b - r * nb;
        const float top = row_top(r);
        float aw[BLOCK], amax = 0.0f, norm2 = 0.0f;
#pragma unroll
        for (int i = 0; i < BLOCK; ++i) {
            aw[i] = fabsf(v[i]);
            amax = fmaxf(amax, aw[i]);
            norm2 = __builtin_fmaf(aw[i], aw[i], norm2);
        }
        // the bounds hold away from the ends of the float32 range; a block of zeros costs nothing at any scale
        const bool near = E2M1 && ((norm2 > 1e-20f && norm2 < 1e20f) || (norm2 == 0.0f && amax == 0.0f)) &&
                          in_range(top * ladder[7] * f.mult[0]) && in_range(top * f.mult[f.n_mult - 1]);
        const float width = NEAR * __builtin_amdgcn_sqrtf(norm2);
        if (E2M1) {
            if (j0 == 0) atomicAdd(&s_norm[r], norm2);
            if (!near) atomicOr(&s_open[r], 0xFFu);
        }
#pragma unroll 1
        for (int j = j0; j < j0 + BASES; ++j) {
            const float base = __fmul_rn(top, ladder[j]);
            float best = __builtin_inff();
            int best_i = 0;
            bool all = true;   // every multiplier as the host evaluates it
            if (near) {
                float second = __builtin_inff(), third = __builtin_inff();
                int second_i = 0;
                const float inv = __builtin_amdgcn_rcpf(base);
#pragma unroll 1
                for (int i = f.n_mult - 1; i >= 0; --i) {
                    const float sc = __fmul_rn(base, f.mult[i]);
                    const float clip = amax - f.cb[7] * sc;
                    if (!__any(!(clip * (1.0f - NEAR) > __builtin_amdgcn_sqrtf(best) + width))) break;   // of the lanes in the loop
                    const float e = family_sq_err_near<BLOCK>(aw, sc, inv * f.half_inv[i]);
                    const bool first = e < best, next = e < second;
                    third = fminf(third, first ? second : fmaxf(e, second));
                    second_i = first ? best_i : next ? i : second_i;
                    second = first ? best : next ? e : second;
                    best_i = first ? i : best_i;
                    best = first ? e : best;
                }
                if (norm2 == 0.0f) best_i = 0;   // first of equals
                const float limit = __builtin_amdgcn_sqrtf(best) + width;
                all = norm2 != 0.0f && !(__builtin_amdgcn_sqrtf(third) > limit);
                if (norm2 != 0.0f && !all && !(__builtin_amdgcn_sqrtf(second) > limit)) {   // one of two, the lower one of equals
                    const int lo = min(best_i, second_i), hi = max(best_i, second_i);
                    const float el = trial(aw, __fmul_rn(base, f.mult[lo])), eh = trial(aw, __fmul_rn(base, f.mult[hi]));
                    best_i = eh < el ? hi : lo;
                }
            }
            if (all) {
#pragma unroll 1
                for (int i = 0; i < f.n_mult; ++i) {
                    const float e = trial(aw, __fmul_rn(base, f.mult[i]));
                    if (i == 0 || e < best) {
                        best = e;
                        best_i = i;
                    }
                }
            }
            s_err[(r * 8 + j) * nb + kb] = best;
            s_mi[(r * 8 + j) * nb + kb] = uint8_t(best_i);
        }
    }
    __syncthreads();
    if (tid < 8 * live) s_tot[tid >> 3][tid & 7] = np_pairwise_sum<4>(s_err + tid * nb, nb);
    __syncthreads();
    if constexpr (E2M1) {   // the bases that these totals leave open: their blocks' errors once more, as the host sums them
        if (tid < live) {
            float least = __builtin_inff();
            for (int j = 0; j < 8; ++j) least = fminf(least, s_tot[tid][j]);
            const float limit = __builtin_amdgcn_sqrtf(least) + NEAR * __builtin_amdgcn_sqrtf(s_norm[tid]);
            uint32_t open = s_open[tid];
            for (int j = 0; j < 8; ++j)
                if (!(__builtin_amdgcn_sqrtf(s_tot[tid][j]) > limit)) open |= 1u << j;
            s_open[tid] = open;
        }
        __syncthreads();
        for (int t = tid; t < total * (8 / BASES); t += QNT) {
            const int b = t / (8 / BASES), j0 = t % (8 / BASES) * BASES, r = b / nb, kb = b - r * nb;
            uint32_t open = s_open[r];
            if ((open & (open - 1u)) == 0u) continue;   // settled
            open &= ((1u << BASES) - 1u) << j0;
            if (open == 0u) continue;
            if (BASES < 8 || total > QNT) load_block<BLOCK, BF16>(w, wbase + size_t(b) * BLOCK, vec, v);
            float aw[BLOCK];
#pragma unroll
            for (int i = 0; i < BLOCK; ++i) aw[i] = fabsf(v[i]);
            for (; open; open &= open - 1u) {
                const int j = __builtin_ctz(open);
                const float sc = __fmul_rn(__fmul_rn(row_top(r), ladder[j]), f.mult[s_mi[(r * 8 + j) * nb + kb]]);
                s_err[(r * 8 + j) * nb + kb] = trial(aw, sc);
            }
        }
        __syncthreads();
        if (tid < 8 * live) {
            const uint32_t open = s_open[tid >> 3];
            if ((open & (open - 1u)) != 0u && ((open >> (tid & 7)) & 1u))
                s_tot[tid >> 3][tid & 7] = np_pairwise_sum<4>(s_err + tid * nb, nb);
        }
        __syncthreads();
    }
    if (tid < live) {
        float best = __builtin_inff();
        int bj = 0;
        for (int j = 0; j < 8; ++j)
            if ((!E2M1 || ((s_open[tid] >> j) & 1u)) && s_tot[tid][j] < best) {
                best = s_tot[tid][j];
                bj = j;
            }
        s_best[tid] = bj;
        wscale[row0 + tid] = __fmul_rn(row_top(tid), ladder[bj]);
    }
    __syncthreads();

    // ---- codes ----------------------------------------------------------------------------------------------------
    for (int b = tid; b < total; b += QNT) {
        if (BASES < 8 || total > QNT) load_block<BLOCK, BF16>(w, wbase + size_t(b) * BLOCK, vec, v);
        const int r = b / nb, kb = b - r * nb, bj = s_best[r];
        const float base = __fmul_rn(row_top(r), ladder[bj]);
        const bool dead = base == 0.0f;   // a vanishing row underflows its base: it is exactly zero (e2e/pack_format.py:55-58)
        const float sc = __fmul_rn(base, f.mult[s_mi[(r * 8 + bj) * nb + kb]]);
        uint32_t c[BLOCK / 8];
#pragma unroll
        for (int i = 0; i < BLOCK / 8; ++i) c[i] = 0u;
        uint32_t open = 1u;   // quotients that two sides of a reciprocal round to different codes (as in family_sq_err_e2m1)
        if (E2M1 && !dead && in_range(sc)) {
            const float h = 0.5f * __builtin_amdgcn_rcpf(sc);
            const float up = h * 1.00000095367431640625f, dn = h * 0.99999904632568359375f;
            open = 0u;
#pragma unroll
            for (int q = 0; q < BLOCK / 8; ++q) {
                const float* x = v + 8 * q;
                float below[8], above[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    below[i] = x[i] * dn;
                    above[i] = x[i] * up;
                }
                c[q] = fp4_word(below, 1.0f);
                open |= c[q] ^ fp4_word(above, 1.0f);
                c[q] = unsigned_zeros(c[q]);
#pragma unroll
                for (int i = 0; i < 8; ++i) open |= uint32_t(!(fabsf(x[i]) < 3e38f));   // infinities and NaN
            }
        }
        if (!dead && open) {
#pragma unroll
            for (int i = 0; i < BLOCK / 8; ++i) c[i] = 0u;
#pragma unroll
            for (int i = 0; i < BLOCK; ++i) {
                const float x = __fdiv_rn(v[i], sc);
                const bool minus = x < 0.0f && family_level<E2M1>(f, fabsf(x)) > 0.0f;
                c[i >> 3] |= (uint32_t(family_index(f, x)) | (minus ? 8u : 0u)) << (4 * (i & 7));
            }
        }
        store_codes<BLOCK>(codes + (wbase + size_t(b) * BLOCK) / 8, vec, c);
    }
    // block codes: index into the multiplier table, bc_bits each (e2e/sc_format.py:14); a dead row takes multiplier 1
    const int per_byte = 8 / f.bc_bits, row_bytes = nb / per_byte;
    int one = 0;
    for (int i = 0; i < f.n_mult; ++i)
        if (f.mult[i] == 1.0f) one = i;
    for (int q = tid; q < live * row_bytes; q += QNT) {
        const int r = q / row_bytes, kb = (q - r * row_bytes) * per_byte, bj = s_best[r];
        const bool dead = __fmul_rn(row_top(r), ladder[bj]) == 0.0f;
        uint32_t byte = 0;
        for (int i = 0; i < per_byte; ++i)
            byte |= uint32_t(dead ? one : s_mi[(r * 8 + bj) * nb + kb + i]) << (f.bc_bits * i);
        bcodes[row0 * row_bytes + q] = uint8_t(byte);
    }
}

// fn(block width, is bf16) as compile-time constants.
template <typename Fn>
static void by_block_and_type(int block, int bf16, Fn&& fn) {
    using B32 = std::integral_constant<int, 32>;
    using B16 = std::integral_constant<int, 16>;
    if (block == 32) bf16 ? fn(B32{}, std::true_type{}) : fn(B32{}, std::false_type{});
    else bf16 ? fn(B16{}, std::true_type{}) : fn(B16{}, std::false_type{});
}

// Rows per workgroup: as many whole rows as give each of its threads one block, which then stays in registers.
static int rows_per_group(int nb, int most) { return nb >= QNT ? 1 : (QNT / nb < most ? QNT / nb : most); }

}  // namespace scmx

using namespace scmx;

extern "C" int scmx_quantize_family(const scmx_format* fmt, const void* w, int w_is_bf16, int64_t N, int K,
                                    uint32_t* codes, uint8_t* bcodes, float* wscale, void* stream) {
    DevFormat df;
    if (int rc = make_dev_format(fmt, &df)) return rc;
    if (!w || !codes || !bcodes || !wscale || N < 0 || N > 0x7FFFFFFF || K <= 0) {
        set_error("quantize_family: null pointer or bad shape (N=%lld K=%d)", (long long)N, K);
        return SCMX_ERR_ARG;
    }
    const int block = fmt->block, per_byte = 8 / fmt->bc_bits;
    if ((block != 16 && block != 32) || K % (block * per_byte) || K > 16384) {
        set_error("quantize_family: block must be 16 or 32 and K a multiple of %d blocks, at most 16384 (block=%d K=%d)",
                  per_byte, block, K);
        return SCMX_ERR_ARG;
    }
    FamilyArgs f = {};
    for (int i = 0; i < 8; ++i) f.cb[i] = float(fmt->code_mag[i]);
    for (int i = 0; i < 7; ++i) {
        if (fmt->code_mag[i + 1] < fmt->code_mag[i]) {
            set_error("quantize_family: code magnitudes must ascend");
            return SCMX_ERR_FORMAT;
        }
        f.cut[i] = (f.cb[i + 1] + f.cb[i]) / 2.0f;
    }
    for (int i = 0; i < fmt->n_mult; ++i) {
        if (i && fmt->mult[i] <= fmt->mult[i - 1]) {
            set_error("quantize_family: block multipliers must ascend");
            return SCMX_ERR_FORMAT;
        }
        f.mult[i] = float(fmt->mult[i]);
        f.half_inv[i] = 0.5f / f.mult[i];
    }
    f.n_mult = fmt->n_mult;
    f.bc_bits = fmt->bc_bits;
    if (N == 0) return SCMX_OK;
    const int nb = K / block;
    // us, a thread per block and base / four bases a thread, bf16 in 16-blocks with ten multipliers: 640 x 896 22 / 26,
    // 1000 x 896 25 / 28, 600 x 2048 35 / 33.  Other codebooks (a thread per base / per block): 269 x 896 42 / 56, 1000
    // x 896 66 / 56.
    const bool e2m1 = df.lut_lo == 0x03020100u && df.lut_hi == 0x0C080604u, spread = long(N) * nb <= (e2m1 ? 65536 : 32768);
    const int rows = rows_per_group(spread ? 8 * nb : e2m1 ? 2 * nb : nb, FAM_ROWS);
    const size_t smem = size_t(rows) * 8 * nb * (sizeof(float) + 1);
    const dim3 grid((unsigned)((N + rows - 1) / rows)), wg(QNT);
    const bool vec = uintptr_t(w) % 16 == 0 && uintptr_t(codes) % 16 == 0;
    auto go = [&](auto kernel) {
        kernel<<<grid, wg, smem, (hipStream_t)stream>>>(w, codes, bcodes, wscale, N, K, rows, vec, f);
    };
    auto typed = [&](auto blk, auto bf) {
        constexpr int B = decltype(blk)::value;
        constexpr bool BF = decltype(bf)::value;
        if (e2m1) spread ? go(quantize_family_kernel<B, BF, true, 1>) : go(quantize_family_kernel<B, BF, true, 4>);
        else spread ? go(quantize_family_kernel<B, BF, false, 1>) : go(quantize_family_kernel<B, BF, false, 8>);
    };
    by_block_and_type(block, w_is_bf16, typed);
    return check_launch("quantize_family");
}

extern "C" int scmx_quantize_sc(const void* w, int w_is_bf16, int64_t N, int K, int block, uint32_t* codes,
                                uint8_t* bcodes, float* wscale, void* stream) {
    if (!w || !codes || !bcodes || !wscale || N < 0 || K <= 0) {
        set_error("quantize_sc: null pointer or bad shape (N=%lld K=%d)", (long long)N, K);
        return SCMX_ERR_ARG;
    }
    if ((block != 16 && block != 32) || K % (4 * block) || K > 131072) {
        set_error("quantize_sc: block must be 16 or 32 and K a multiple of 4 blocks, at most 131072 (block=%d K=%d)",
                  block, K);
        return SCMX_ERR_ARG;
    }
    if (N > 0x7FFFFFFF) {
        set_error("quantize_sc: more than 2^31 - 1 rows");
        return SCMX_ERR_ARG;
    }
    if (N == 0) return SCMX_OK;
    const int nb = K / block, rows = rows_per_group(nb, QNT / 4);
    const dim3 grid((unsigned)((N + rows - 1) / rows)), wg(QNT);
    const size_t smem = size_t(rows) * (nb + 2) * sizeof(int);
    const bool vec = uintptr_t(w) % 16 == 0 && uintptr_t(codes) % 16 == 0;
    by_block_and_type(block, w_is_bf16, [&](auto blk, auto bf) {
        quantize_sc_kernel<decltype(blk)::value, decltype(bf)::value>
            <<<grid, wg, smem, (hipStream_t)stream>>>(w, codes, bcodes, wscale, N, K, rows, vec);
    });
    return check_launch("quantize_sc");
}

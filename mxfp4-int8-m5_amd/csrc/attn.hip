// Single-token attention against a KV cache (decode): out[h] = softmax(q[h] . K^T * scale) V for every query head.
//
// The linear layers are the product here; this kernel exists so that a decode step is a fixed, short sequence of
// launches that a HIP graph can replay: it reads the number of valid cache rows from device memory, so the same
// captured launch serves every position.  One workgroup per query head.  A row of K or V (d bf16 values) is read by
// d / 8 lanes, 16 bytes each; such a lane group walks every (groups)-th row with a running maximum, sum and
// weighted value chunk (one pass over K and V, the rows of a few steps in flight together and one rescaling for all of
// them), and the groups' partial results are merged, those of a wave across its lanes and the waves' through LDS.
// Accumulation is float32, the output bf16.  For long contexts the rows of a head are cut into several ranges, one
// workgroup each (16 workgroups alone read a long cache at a fraction of the memory bandwidth), and a small second kernel
// merges the ranges' results.  Where two query heads share a KV head, a workgroup then serves both of them from one
// reading of the rows.
#include <type_traits>

#include "scmx_common.h"

namespace scmx {

constexpr int ANT = 512;
constexpr int ATTN_SINGLE_MAX = 128;   // rows up to which a split launch falls back to one workgroup per head: one turn of its loads

// A launch of this many ranges may serve the query heads of a KV head two at a time (kernel below), and does so with more
// rows than these.  16 heads of 128 over 8 KV heads, sixteen caches in turn, attention and merge in a graph, us with 32 ranges
// two heads at a time / 16 ranges one at a time (in the grid of 32): 300 rows 7.7 / 6.8, 1000 8.2 / 7.4, 2000 8.4 / 7.8, 3000
// 9.0 / 8.9; against a launch of 16 ranges 4096 10.2 / 12.1, 6000 11.9 / 14.9, 12000 15.8 / 21.4.
constexpr int ATTN_PAIR_RANGES = 32, ATTN_PAIR_MIN = 3072;

// What the fused variant needs besides the attention operands: the token's q|k|v row as the qkv projection wrote it,
// the per-head norm weights and the rotary frequencies.
struct QkvArgs {
    const uint16_t* y;        // bf16 [(hq + 2 hk) * d]: q heads, k heads, v heads
    const uint16_t* qn;       // bf16 [d]
    const uint16_t* kn;       // bf16 [d]
    const float* inv_freq;    // [d / 2]
    float eps;
};

// Sum over the LPR lanes of a group (LPR a power of two from 8 on, groups aligned), in every lane: data-parallel-primitive
// additions inside a row of 16 lanes.
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int LPR>
__device__ __forceinline__ float group_sum(float v) {
    static_assert(LPR == 8 || LPR == 16 || LPR == 32, "8, 16 or 32 lanes");
    v = dpp_add<0xB1>(v);    // quad_perm 1 0 3 2
    v = dpp_add<0x4E>(v);    // quad_perm 2 3 0 1
    v = dpp_add<0x141>(v);   // row_half_mirror: the other quad of eight
    if (LPR >= 16) v = dpp_add<0x140>(v);   // row_mirror: the other eight of sixteen
    if (LPR >= 32) v += __shfl_xor(v, 16, WAVE);
    return v;
}

// FUSED: the workgroup first normalises and rotates its own q heads and its KV head's new k (as the row kernel
// qkv_headnorm_kernel does, same arithmetic), keeps them and the new v in LDS, and attends over the cache rows below
// the position plus that new row; the first query head of every KV group appends the new k and v to the cache.  No
// workgroup reads what another writes in the same launch.
// Bound by latency up to some thousand rows (the launch, the position, the rows, the merge: a chain of trips to memory),
// then by reading the cache.
template <int D, bool FUSED>
struct AttnDecode {
    static constexpr int LPR = D / 8;              // lanes per cache row
    static constexpr int GROUPS = ANT / LPR;       // lane groups per workgroup, each walking its own rows
    static constexpr int WAVES = ANT / 64, UN = 4; // UN: rows in flight per lane group
    struct Shared {
        float m[WAVES][2], l[WAVES][2], acc[WAVES][2][D];
        float sin[FUSED ? D / 2 : 1], cos[FUSED ? D / 2 : 1];
        __attribute__((aligned(16))) uint16_t knew[FUSED ? 2 : 1][D], qnew[FUSED ? 2 : 1][D];   // this token's k, v and q heads (bf16)
    };

    static constexpr int PER = D / 64, FREQ = (D + 127) / 128;   // a lane's elements of a head; its frequencies
    // FUSED: what a wave works on before the rows: waves 0 / 1 / 2 (and 4, a second q) the q / k / v head of this token,
    // wave 3 the rotation.  Requested first of all: memory returns a wave's loads in order, behind the cache rows they
    // would come last.
    struct Token {
        uint16_t y[PER], w[PER];   // the lane's elements of the head and their norm weights
        float freq[FREQ];
        bool q, any;
    };
    static __device__ __forceinline__ Token token(int head, int other, int hq, int hk, const QkvArgs& x) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, kvh = head / (hq / hk);
        Token t;
        t.q = wave == 0 || (wave == 4 && other >= 0);
        t.any = t.q || wave == 1 || wave == 2;
        if (t.any) {
            const int g = wave == 0 ? head : wave == 4 ? other : wave == 1 ? hq + kvh : hq + hk + kvh;
            const uint16_t* w = t.q ? x.qn : x.kn;
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                t.y[i] = x.y[size_t(g) * D + PER * lane + i];
                t.w[i] = w[PER * lane + i];
            }
        } else if (wave == 3) {
#pragma unroll
            for (int j = 0; j < FREQ; ++j)
                if (lane + 64 * j < D / 2) t.freq[j] = x.inv_freq[lane + 64 * j];
        }
        return t;
    }

    // The query head `head` (HEADS = 2: and `other`, of the same KV head), cache rows [row0, row1) of n; whole: they are all
    // of them, the output is written; else the unnormalised results, maxima and sums go to `part` (and part_other).
    template <int HEADS>
    static __device__ __forceinline__ void run(Shared& s, const uint16_t* __restrict__ q, uint16_t* __restrict__ kc,
                                               uint16_t* __restrict__ vc, int head, int other, int hq, int hk, int rows, int n,
                                               int row0, int row1, bool append, float scale, const QkvArgs& x, const Token& token,
                                               bool whole, uint16_t* __restrict__ out, float* part, float* part_other) {
        const int tid = threadIdx.x, grp = tid / LPR, c = tid % LPR, lane = tid & 63, wave = tid >> 6;
        const int kvh = head / (hq / hk);
        const uint16_t* kbase = kc + size_t(kvh) * rows * D + 8 * c;
        const uint16_t* vbase = vc + size_t(kvh) * rows * D + 8 * c;
        // Every lane of the workgroup runs the same number of trips (rows beyond row1 are skipped by predication), so the
        // cross-lane sums below always see whole groups.
        const int trips = (max(row1 - row0, 0) + GROUPS - 1) / GROUPS;
        u32x4 kw[UN], vw[UN];
        auto load_trips = [&](int t0) {
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                if (u > 0 && t0 + u >= trips) break;
                const int j = row0 + (t0 + u) * GROUPS + grp;
                const size_t ro = size_t(j < row1 ? j : 0) * D;
                kw[u] = *reinterpret_cast<const u32x4*>(kbase + ro);
                vw[u] = *reinterpret_cast<const u32x4*>(vbase + ro);
            }
        };
        load_trips(0);   // on their way while the fused variant prepares q and the new row

        if (FUSED) {
            const int newrow = n - 1;   // the position of the token being decoded
            float nv[PER];
            const bool live = token.any && (HEADS == 2 || wave < 3);
            if (wave == 3) {
#pragma unroll
                for (int j = 0; j < FREQ; ++j) {
                    const int i = lane + 64 * j;
                    if (i < D / 2) sincosf(float(int64_t(newrow)) * token.freq[j], &s.sin[i], &s.cos[i]);
                }
            } else if (live) {
                float yv[PER];
                float ss = 0.0f;
#pragma unroll
                for (int i = 0; i < PER; ++i) {
                    yv[i] = bf16_to_f32(token.y[i]);
                    ss = __fadd_rn(ss, __fmul_rn(yv[i], yv[i]));
                }
                if (wave != 2) {
                    head_norm(yv, ss, PER, D, [&](int i) { return bf16_to_f32(token.w[i]); }, x.eps, nv);
                } else {
#pragma unroll
                    for (int i = 0; i < PER; ++i) nv[i] = yv[i];
                }
            }
            __syncthreads();
            if (live) {
                uint16_t* dst = (wave == 1 ? kc : vc) + (size_t(kvh) * rows + newrow) * D + PER * lane;
                uint16_t* here = token.q ? s.qnew[wave >> 2] : s.knew[wave - 1];
                auto emit = [&](int i, uint16_t b) {
                    here[PER * lane + i] = b;
                    if (append && !token.q) dst[i] = b;
                };
                head_rope(nv, PER, lane, D, wave != 2 ? s.sin : nullptr, s.cos, emit);   // v passes through unrotated
            }
            __syncthreads();
        }

        float qv[HEADS][8];
#pragma unroll
        for (int h = 0; h < HEADS; ++h) {
            const u32x4 w = FUSED ? *reinterpret_cast<const u32x4*>(&s.qnew[h][8 * c])
                                  : *reinterpret_cast<const u32x4*>(q + size_t(h ? other : head) * D + 8 * c);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                qv[h][2 * i] = bf16_lo(w[i]) * scale;
                qv[h][2 * i + 1] = bf16_hi(w[i]) * scale;
            }
        }
        float m[HEADS], l[HEADS], acc[HEADS][8];
#pragma unroll
        for (int h = 0; h < HEADS; ++h) {
            m[h] = -3.0e38f;
            l[h] = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[h][i] = 0.0f;
        }
        for (int t0 = 0; t0 < trips; t0 += UN) {
            if (t0 > 0) load_trips(t0);
            float sc[HEADS][UN];
            bool ok[UN];
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const int j = row0 + (t0 + u) * GROUPS + grp;
                ok[u] = j < row1;
                if (u > 0 && t0 + u >= trips) {   // (wave-uniform)
#pragma unroll
                    for (int h = 0; h < HEADS; ++h) sc[h][u] = -3.0e38f;
                    continue;
                }
                if (FUSED && j == n - 1) {   // the new row comes from LDS, not from the cache being appended to
                    kw[u] = *reinterpret_cast<const u32x4*>(&s.knew[0][8 * c]);
                    vw[u] = *reinterpret_cast<const u32x4*>(&s.knew[1][8 * c]);
                }
                float kf[8];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    kf[2 * i] = bf16_lo(kw[u][i]);
                    kf[2 * i + 1] = bf16_hi(kw[u][i]);
                }
#pragma unroll
                for (int h = 0; h < HEADS; ++h) {
                    float a = qv[h][0] * kf[0], b = qv[h][1] * kf[1];
#pragma unroll
                    for (int i = 1; i < 4; ++i) {
                        a = __builtin_fmaf(qv[h][2 * i], kf[2 * i], a);
                        b = __builtin_fmaf(qv[h][2 * i + 1], kf[2 * i + 1], b);
                    }
                    sc[h][u] = group_sum<LPR>(a + b);
                }
            }
#pragma unroll
            for (int h = 0; h < HEADS; ++h) {
                float mn = m[h];
#pragma unroll
                for (int u = 0; u < UN; ++u) mn = ok[u] ? fmaxf(mn, sc[h][u]) : mn;
                const float alpha = __expf(m[h] - mn);
                m[h] = mn;
                l[h] *= alpha;
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[h][i] *= alpha;
#pragma unroll
                for (int u = 0; u < UN; ++u) {
                    sc[h][u] = ok[u] ? __expf(sc[h][u] - mn) : 0.0f;
                    l[h] += sc[h][u];
                }
            }
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                if (u > 0 && t0 + u >= trips) break;
                float vf[8];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    vf[2 * i] = bf16_lo(vw[u][i]);
                    vf[2 * i + 1] = bf16_hi(vw[u][i]);
                }
                if (!ok[u]) continue;   // (0 times a row that is not part of the context could be NaN)
#pragma unroll
                for (int h = 0; h < HEADS; ++h)
#pragma unroll
                    for (int i = 0; i < 8; ++i) acc[h][i] = __builtin_fmaf(sc[h][u], vf[i], acc[h][i]);
            }
        }
        // the groups of a wave meet across its lanes, the waves in LDS
#pragma unroll
        for (int h = 0; h < HEADS; ++h) {
            float mx = m[h];
#pragma unroll
            for (int off = LPR; off < 64; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off, WAVE));
            const float w = __expf(m[h] - mx);   // groups that saw no row have l = 0 and contribute nothing
            l[h] *= w;
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[h][i] *= w;
#pragma unroll
            for (int off = LPR; off < 64; off <<= 1) {
                l[h] += __shfl_xor(l[h], off, WAVE);
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[h][i] += __shfl_xor(acc[h][i], off, WAVE);
            }
            if (lane < LPR) {
                *reinterpret_cast<f32x4*>(&s.acc[wave][h][8 * c]) = f32x4{acc[h][0], acc[h][1], acc[h][2], acc[h][3]};
                *reinterpret_cast<f32x4*>(&s.acc[wave][h][8 * c + 4]) = f32x4{acc[h][4], acc[h][5], acc[h][6], acc[h][7]};
                if (c == 0) {
                    s.m[wave][h] = mx;
                    s.l[wave][h] = l[h];
                }
            }
        }
        __syncthreads();
        if (tid >= HEADS * D) return;
        const int h = tid / D, e = tid % D;   // element e of head h
        float mx = s.m[0][h];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) mx = fmaxf(mx, s.m[w][h]);
        float num = 0.0f, den = 0.0f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float f = __expf(s.m[w][h] - mx);
            num += f * s.acc[w][h][e];
            den += f * s.l[w][h];
        }
        if (whole) {
            out[size_t(h ? other : head) * D + e] = f32_to_bf16(num / den);
        } else {   // num and den are relative to mx; a range without rows leaves mx = -3e38, den = 0
            float* pw = h ? part_other : part;
            pw[e] = num;
            if (e == 0) {
                pw[D] = mx;
                pw[D + 1] = den;
            }
        }
    }
};

// PAIR (ATTN_PAIR_RANGES ranges or more, an even number of them, and of query heads to a KV head): blockIdx.x counts pairs
// of heads.  Up to ATTN_PAIR_MIN rows, blockIdx.y % 2 says which of the two a workgroup serves, in half as many ranges; the
// grid is the same either way, so a captured launch serves every position.
template <int D, bool FUSED, bool PAIR>
__global__ __launch_bounds__(ANT) void attn_decode_kernel(const uint16_t* __restrict__ q, uint16_t* __restrict__ kc,
                                                         uint16_t* __restrict__ vc,
                                                         const int64_t* __restrict__ pos_dev, int n0,
                                                         uint16_t* __restrict__ out, int hq, int hk, int rows, float scale,
                                                         const QkvArgs x, float* __restrict__ partial) {
    using A = AttnDecode<D, FUSED>;
    __shared__ typename A::Shared s;
    const int head = PAIR ? 2 * blockIdx.x + (blockIdx.y & 1) : blockIdx.x, other = PAIR ? head ^ 1 : -1;
    typename A::Token token;
    if constexpr (FUSED) token = A::token(head, other, hq, hk, x);
    // A device-resident position outside the cache (the host cannot see it) touches no cache row: the output is
    // zero and nothing is appended.
    const int64_t n64 = pos_dev ? pos_dev[0] + 1 : int64_t(n0);
    int range = PAIR ? blockIdx.y >> 1 : blockIdx.y;   // one head at a time
    if (n64 < 1 || n64 > rows) {
        if (range == 0)
            for (int e = threadIdx.x; e < D; e += ANT) out[size_t(head) * D + e] = 0;
        return;
    }
    const int n = int(n64);
    // gridDim.y > 1: the valid rows are cut into equal ranges, one per workgroup of a head; every workgroup leaves its
    // unnormalised result, maximum and sum in `partial` and a second kernel merges them. A context of at most
    // ATTN_SINGLE_MAX rows is read fastest by one workgroup per head (16 heads of a long cache, us, single / 16 ranges with
    // the merge: 128 rows 6.1 / 6.2, 160 - / 6.3): range 0 then takes all of it and writes the output, the other
    // workgroups leave at once and the merge kernel finds nothing to do.
    const bool whole = gridDim.y == 1 || n <= ATTN_SINGLE_MAX, both = PAIR && n > ATTN_PAIR_MIN;
    if (whole && range > 0) return;
    int ranges = whole ? 1 : PAIR ? gridDim.y >> 1 : gridDim.y;
    if (both) {
        ranges = gridDim.y;
        range = blockIdx.y;
    }
    const int chunk = (n + ranges - 1) / ranges;
    const int row0 = range * chunk, row1 = min(n, row0 + chunk);   // this workgroup's rows [row0, row1)
    const auto part = [&](int h) { return partial + (size_t(h) * gridDim.y + range) * (D + 2); };
    const bool append = range == 0 && (both ? min(head, other) : head) % (hq / hk) == 0;
    if constexpr (PAIR) {
        if (both) {
            A::template run<2>(s, q, kc, vc, head, other, hq, hk, rows, n, row0, row1, append, scale, x, token, false, out, part(head),
                               part(other));
            return;
        }
    }
    A::template run<1>(s, q, kc, vc, head, other, hq, hk, rows, n, row0, row1, append, scale, x, token, whole, out, part(head), nullptr);
}

// Merge of the per-range results of one head: out = sum_s w_s num_s / sum_s w_s den_s with w_s = exp(m_s - max m).
// Bound: one trip to memory behind a launch.  Everything is requested at once, and before the position is known; a wave's
// lanes hold the ranges' maxima and sums (one each), and the ranges' results are dealt to MERGE_NT / D parts of the
// workgroup.
constexpr int MERGE_NT = 512;
template <int D, int RANGES>   // up to RANGES ranges
__global__ __launch_bounds__(MERGE_NT) void attn_merge_kernel(const float* __restrict__ partial, uint16_t* __restrict__ out,
                                                            int slots, bool pair, const int64_t* __restrict__ pos_dev, int n0, int rows) {
    constexpr int PARTS = MERGE_NT / D, PER = RANGES / PARTS;
    static_assert(RANGES <= 64 && RANGES % PARTS == 0, "a lane per range");
    __shared__ float s_num[PARTS][D];
    const int head = blockIdx.x, part = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / D), e = threadIdx.x % D, lane = threadIdx.x & 63;
    const float* pw = partial + size_t(head) * slots * (D + 2);
    const float pm = pw[min(lane, slots - 1) * (D + 2) + D], pl = pw[min(lane, slots - 1) * (D + 2) + D + 1];
    float pn[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) pn[u] = pw[min(part + u * PARTS, slots - 1) * (D + 2) + e];
    const int64_t n64 = pos_dev ? pos_dev[0] + 1 : int64_t(n0);
    if (n64 <= ATTN_SINGLE_MAX || n64 > rows) return;   // range 0 wrote the output itself (zeros for a position outside the cache)
    const int splits = pair && n64 <= ATTN_PAIR_MIN ? slots >> 1 : slots;   // of the slots, those that hold a range
    const float mx = wave_max(lane < splits ? pm : -3.0e38f);   // (over the whole wave)
    const float w = lane < splits ? __expf(pm - mx) : 0.0f, den = wave_sum(lane < splits ? w * pl : 0.0f);
    float num = 0.0f;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const float f = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), part + u * PARTS));
        if (part + u * PARTS < splits) num += f * pn[u];
    }
    s_num[part][e] = num;
    __syncthreads();
    if (part > 0) return;
#pragma unroll
    for (int p = 1; p < PARTS; ++p) num += s_num[p][e];
    out[size_t(head) * D + e] = f32_to_bf16(num / den);
}

template <bool FUSED>
static void launch_attn(int d, hipStream_t st, const uint16_t* q, uint16_t* kc, uint16_t* vc, const int64_t* pos_dev, int n,
                        uint16_t* out, int hq, int hk, int rows, float scale, const QkvArgs& x, float* partial, int splits) {
    const auto go = [&](auto dim) {
        constexpr int D = decltype(dim)::value;
        const bool pair = splits >= ATTN_PAIR_RANGES && splits % 2 == 0 && hq / hk % 2 == 0;
        if (pair)
            attn_decode_kernel<D, FUSED, true><<<dim3(hq / 2, splits), dim3(ANT), 0, st>>>(q, kc, vc, pos_dev, n, out, hq, hk, rows, scale,
                                                                                           x, partial);
        else
            attn_decode_kernel<D, FUSED, false><<<dim3(hq, splits), dim3(ANT), 0, st>>>(q, kc, vc, pos_dev, n, out, hq, hk, rows, scale, x,
                                                                                        partial);
        if (splits > 32) attn_merge_kernel<D, 64><<<dim3(hq), dim3(MERGE_NT), 0, st>>>(partial, out, splits, pair, pos_dev, n, rows);
        else if (splits > 16) attn_merge_kernel<D, 32><<<dim3(hq), dim3(MERGE_NT), 0, st>>>(partial, out, splits, pair, pos_dev, n, rows);
        else if (splits > 1) attn_merge_kernel<D, 16><<<dim3(hq), dim3(MERGE_NT), 0, st>>>(partial, out, splits, pair, pos_dev, n, rows);
    };
    if (d == 64) go(std::integral_constant<int, 64>{});
    else if (d == 128) go(std::integral_constant<int, 128>{});
    else go(std::integral_constant<int, 256>{});
}

// The row ranges of a split launch: `workspace` holds splits * hq * (d + 2) floats.
static int check_split(const char* who, const float* workspace, int splits) {
    if (splits < 1 || splits > 64 || (splits > 1 && (!workspace || uintptr_t(workspace) % 4))) {
        set_error("%s: splits must be 1..64 and need a float workspace of splits * hq * (d + 2) entries", who);
        return SCMX_ERR_ARG;
    }
    return SCMX_OK;
}

}  // namespace scmx

using namespace scmx;

static int check_attn(const char* who, int hq, int hk, int d, int cache_rows) {
    if (hq < 1 || hk < 1 || hq > 65535 || hq % hk || cache_rows < 1) {
        set_error("%s: bad head counts or cache size (hq=%d hk=%d rows=%d)", who, hq, hk, cache_rows);
        return SCMX_ERR_ARG;
    }
    if (d != 64 && d != 128 && d != 256) {
        set_error("%s: head dim must be 64, 128 or 256 (d=%d)", who, d);
        return SCMX_ERR_ARG;
    }
    return SCMX_OK;
}

extern "C" int scmx_attn_decode(const uint16_t* q, const uint16_t* kcache, const uint16_t* vcache, const int64_t* pos_dev,
                                int n, uint16_t* out, int hq, int hk, int d, int cache_rows, float scale,
                                float* workspace, int splits, void* stream) {
    if (!q || !kcache || !vcache || !out) {
        set_error("attn_decode: null pointer argument");
        return SCMX_ERR_ARG;
    }
    if (int rc = check_attn("attn_decode", hq, hk, d, cache_rows)) return rc;
    if (uintptr_t(q) % 16 || uintptr_t(kcache) % 16 || uintptr_t(vcache) % 16) {
        set_error("attn_decode: q and the caches must be 16-byte aligned");
        return SCMX_ERR_ARG;
    }
    if (!pos_dev && (n < 1 || n > cache_rows)) {
        set_error("attn_decode: %d valid rows outside 1..%d", n, cache_rows);
        return SCMX_ERR_ARG;
    }
    if (int rc = check_split("attn_decode", workspace, splits)) return rc;
    launch_attn<false>(d, (hipStream_t)stream, q, const_cast<uint16_t*>(kcache), const_cast<uint16_t*>(vcache), pos_dev, n,
                       out, hq, hk, cache_rows, scale, QkvArgs{}, workspace, splits);
    return check_launch("attn_decode");
}

extern "C" int scmx_attn_decode_qkv(const uint16_t* y, const uint16_t* qn, const uint16_t* kn, float eps,
                                    const float* inv_freq, const int64_t* pos_dev, int64_t pos0, uint16_t* kcache,
                                    uint16_t* vcache, uint16_t* out, int hq, int hk, int d, int cache_rows, float scale,
                                    float* workspace, int splits, void* stream) {
    if (!y || !qn || !kn || !inv_freq || !kcache || !vcache || !out) {
        set_error("attn_decode_qkv: null pointer argument");
        return SCMX_ERR_ARG;
    }
    if (int rc = check_attn("attn_decode_qkv", hq, hk, d, cache_rows)) return rc;
    if (uintptr_t(kcache) % 16 || uintptr_t(vcache) % 16) {
        set_error("attn_decode_qkv: caches must be 16-byte aligned");
        return SCMX_ERR_ARG;
    }
    if (!pos_dev && (pos0 < 0 || pos0 >= cache_rows)) {
        set_error("attn_decode_qkv: position %lld outside a cache of %d rows", (long long)pos0, cache_rows);
        return SCMX_ERR_ARG;
    }
    if (int rc = check_split("attn_decode_qkv", workspace, splits)) return rc;
    launch_attn<true>(d, (hipStream_t)stream, nullptr, kcache, vcache, pos_dev, int(pos0) + 1, out, hq, hk, cache_rows, scale,
                      QkvArgs{y, qn, kn, inv_freq, eps}, workspace, splits);
    return check_launch("attn_decode_qkv");
}

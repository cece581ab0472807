// W4A8 GEMM on CDNA4 INT8 MFMA: the tile kernel of dense prefill (gemm_rows*.hip, gemm_blocked.hip) and of grouped
// mixture-of-experts (gemm_grouped.hip).
//
// One workgroup computes a BM x BN tile of  acc[m, n] = sum_k xq[m, k] * q[n, k]  in INT32.  Per K step of BK the
// workgroup stages BM x BK activation bytes and BN x BK weight bytes in LDS; the weight bytes are produced in
// registers from the packed 4-bit codes (16 bytes of codes = one run of 32 weights per thread) right before they
// are written to LDS, so the INT8 form of the weights exists only there.  Waves then read 16-byte operand
// fragments and issue v_mfma_i32_16x16x64_i8 (MF = 16) or v_mfma_i32_32x32x32_i8 (MF = 32) with the weights as the row
// operand: each lane ends up with groups of 4 consecutive output columns n of one token row m, which is the unit every
// epilogue works on.
// LDS holds three stages of the K loop; global loads run four steps ahead in two register sets, and the decode and
// LDS writes of step i+2 are issued between the MFMAs of step i, with one barrier per step.
#pragma once
#include <type_traits>

#include "gemm_args.h"

namespace scmx {

// MF, the shape of the MFMA.  At the chip's power limit (all-zero operands run a third faster) and on INT8 operands as
// they occur, a loop of MFMAs alone reaches 4420 TOP/s with 16x16x64 and 3740 with 32x32x32 (half the accumulator
// traffic per multiply-add): gate|up of 12288 x 2048 at 8192 rows, same tile, 208 us with the latter and 199 with the
// former.  A launch bound elsewhere is far from that limit, and 32x32x32 takes half the instructions: the packed tile
// (bound by the vector ALU that decodes its weights) uses it, 16-block power-of-two format, 64 experts of 2048 x 2048 /
// 257 of 1024 x 2048, 70 rows each: 50.2 -> 47.7 and 109 -> 104 us.
//
// FD = number of register buffers of the split operand's fragments: fetched FD - 1 phases (half k slices) ahead of
// their MFMAs.
// SKIP (grouped launches): a row tile that ends inside its expert's segment multiplies only the 16-row blocks that hold
// valid rows.  The two waves that share a SIMD then own the same columns and different row halves of the tile, so that
// a half-empty tile halves the MFMA work of every SIMD instead of idling two of the four.
// (PK: the halves of 32 rows; the waves sit side by side along the columns and skip alike.)
// PK (the FP4-conversion formats, K steps of 128): the weights stay packed in LDS -- 64 bytes of codes per row and K
// step plus the step's block-code bytes -- and every wave decodes its own fragments after reading them.  Half the
// weight bytes through LDS in both directions, paid with one decode per wave row that shares the fragment.
// KG > 1 (small problems: fewer tiles than CUs): KG groups of WGM x WGN waves share the tile, each multiplies its own K
// / KG of the reduction out of LDS stages of its own, and the INT32 partial sums meet in LDS before the epilogue
// (exact: integer addition is associative).  A CU then runs KG times the waves on the same tile count.
// AD (ADM 1, dense: activations in the blocked layout; ADM 2, grouped: rows, gathered): the activation tile does not
// pass through LDS; every wave loads the fragments of its own rows from memory, two K steps ahead: four runs of 256
// bytes from the blocked layout, sixteen of 64 from rows.  Waves must then not share rows (WGN = 1, or few column
// groups), and only the weight rows of a stage exist in LDS.
//
// OCC: waves a SIMD that the tile's registers and LDS leave room for at least, and with them the workgroups that share a CU.
template <int BM, int BN, int BK, int WGM, int WGN, int BMODE, int OCC = 1, int FD = 2, bool SKIP = false, bool PK = false,
          int KG = 1, int ADM = 0, int MF = 16>
__global__ __launch_bounds__(WGM* WGN* KG * 64, OCC) void gemm_kernel(const GemmArgs a) {
    constexpr bool AD = ADM != 0, ADR = ADM == 2;   // activation fragments straight from memory; from the row layout
    constexpr bool DEAL = SKIP && AD;   // the tile's MF-row blocks are dealt to the waves in turn
    constexpr int NSTAGE = 3;   // LDS stages: one being read, one ready, one being written
    constexpr int NT = WGM * WGN * 64;   // threads of one K group
    constexpr int WTM = BM / WGM, WTN = BN / WGN;
    constexpr int MI = WTM / MF, NI = WTN / MF;   // MF-row / MF-column blocks of a wave's tile
    constexpr int ACC16 = WTM * WTN / 256;        // its accumulators, in 16 x 16 blocks
    static_assert(WTM % 32 == 0 && WTN % 32 == 0 && (BK == 64 || BK == 128), "tile must be whole 32x32 blocks");
    static_assert(MF == 32 || (MF == 16 && !PK), "MFMA shapes 32x32x32 and, weights staged as INT8, 16x16x64");
    static_assert(MF == 16 || ADM != 2, "activation fragments from gathered rows: 64-wide slices");
    constexpr int CPR = BK / 16;             // 16-byte chunks per LDS row
    constexpr int RPB = 256 / BK;            // rows per 256 bytes, i.e. per sweep of the 64 LDS banks
    constexpr int A_CHUNKS = AD ? 0 : BM * CPR;   // 16-byte pieces of the activation tile
    constexpr int A_PER = AD ? 1 : (A_CHUNKS + NT - 1) / NT;
    constexpr int A_BYTES = AD ? 0 : BM * BK;     // the activation rows of a stage
    // packed weights are staged in runs of 8 * WPC weights (WPC code words) per thread: 32 when that keeps every
    // thread busy, else 16
    constexpr int WPC = BN * BK / 32 >= NT ? 4 : 2;
    constexpr int B_CHUNKS = BMODE == B_INT8 ? BN * CPR : BN * BK / (8 * WPC);
    constexpr int B_PER = (B_CHUNKS + NT - 1) / NT;
    // PK: block-code bytes per weight row and K step
    constexpr int BCB = BMODE == B_PACKED_B16M || BMODE == B_PACKED_E8M0 ? 4 : BMODE == B_PACKED_B16 ? 2 : 1;
    constexpr int BCR = BCB == 4 ? 2 : 1;   // registers for those of two steps
    static_assert(!PK || (BK == 128 && WPC == 4 && BMODE != B_INT8 && BMODE != B_PACKED_GENERIC),
                  "packed weights in LDS: K steps of 128, 16-byte runs, FP4-conversion formats");
    // bytes per stage: BM activation rows, then BN weight rows (PK: 64 code bytes each)
    constexpr int STAGE = A_BYTES + (PK ? BN * (BK / 2) : BN * BK);
    static_assert(STAGE % 16 == 0, "stages keep 16-byte alignment");

    // Rows are BK bytes with no padding; the 16-byte chunk c of row r sits at chunk c ^ ((r / RPB) % CPR), which
    // spreads the 16 rows a b128 fragment read touches per pass over all 64 banks.
    // The epilogue reuses the buffer for one [WTM x (row bytes + 16)] output tile per wave; when the bf16 tiles
    // need more than the stages and still fit the CU, the buffer is sized for them.
    constexpr int EPI_BYTES = WGM * WGN * WTM * (WTN * 2 + 16);
    static_assert(KG == 1 || (!PK && !SKIP), "K groups: staged dense tiles");
    static_assert(!AD || (!PK && KG == 1), "activation fragments from memory: staged tiles");
    constexpr int GROUP_BYTES = NSTAGE * STAGE;
    // after the K loop: group 0's output tiles (the widest epilogue's) from 0, then the other groups' partial sums
    constexpr int PART_BYTES = NT * ACC16 * 16;
    constexpr int PART_BASE = WGM * WGN * WTM * (WTN * 4 + 16);
    constexpr int KG_BYTES = PART_BASE + (KG - 1) * PART_BYTES > KG * GROUP_BYTES ? PART_BASE + (KG - 1) * PART_BYTES : KG * GROUP_BYTES;
    static_assert(KG == 1 || KG_BYTES <= 160 * 1024, "stages and partial sums fit the CU's LDS");
    constexpr int SMEM_BYTES =
        KG > 1 ? KG_BYTES : (EPI_BYTES > NSTAGE * STAGE && EPI_BYTES <= 150 * 1024) ? EPI_BYTES : NSTAGE * STAGE;
    __shared__ __attribute__((aligned(16))) int8_t smem[SMEM_BYTES];
    // scales of the tile's rows and columns, fetched before the K loop so that the epilogue does not start with a
    // round trip to memory
    __shared__ __attribute__((aligned(16))) float s_xs[BM], s_ws[BN];
    // SwiGLU: the sigmoid's table (8 KB), copied to LDS while the first operands are on their way, where the CU then still
    // holds the workgroups that OCC counts on.  The others (three packed expert tiles fill the CU's LDS, as do two staged
    // ones of 64x128, two of 128x64 and three of 64x64) copy it over their stages once the K loop is done, behind the
    // waves' output tiles: one trip to the L2 and a barrier, hidden by the other workgroups (SIG_LATE).  A wave's 64 gates
    // lie in some 30 cache lines, which the vector L1 would serve one after the other.
    // With the 65536-entry table of silu(g) in memory, two conversions and one lookup at a time instead of two, 12288 x
    // 2048 at 2048 rows took 57.3 us for 53.0, at 1500 51.1 for 49.4, at 256 12.0 for 11.1; 6144 x 4096 at 6000 rows 152.5
    // for 148.4.  A sparse block of 257 experts, 2000 tokens, whose gate|up runs packed tiles: 257.5 with the lookups in
    // memory, 253.3 with the late copy.  An early copy that takes a workgroup from the CU costs every epilogue, us early /
    // late, scaled output and SwiGLU: 64x128 with table decode, 257 experts of 1024 x 2048, 60 rows each, 329 / 234 and
    // 334 / 238, with INT8 weights 145 / 128 and 149 / 128; 128x64, 12288 x 1152 at 160 rows, 11.5 / 9.3 and 12.5 / 10.2;
    // 64x64, 49152 x 1024 at 50 rows, 10.4 / 8.8 and 10.7 / 9.2.
    constexpr int SIG_BYTES = int(sizeof(uint16_t)) * 2 * int(SIGMOID_ENTRIES);
    constexpr int CU_WGS = OCC * 4 * 64 / (NT * KG) > 1 ? OCC * 4 * 64 / (NT * KG) : 1;
    constexpr int CU_SHARE = 160 * 1024 / CU_WGS, LDS_BYTES = SMEM_BYTES + (BM + BN) * 4;
    static_assert(LDS_BYTES <= CU_SHARE, "the workgroups that OCC counts on fit the CU's LDS");
    constexpr bool SIG = !PK && LDS_BYTES + SIG_BYTES <= CU_SHARE;
    __shared__ __attribute__((aligned(16))) uint16_t s_sig[SIG ? 2 * SIGMOID_ENTRIES : 8];
    constexpr int SIG_AT = WGM * WGN * WTM * (WTN + 16);   // behind the waves' output tiles
    constexpr bool SIG_LATE = !SIG && KG == 1 && SIG_AT + SIG_BYTES <= SMEM_BYTES;
    uint16_t* const sig = SIG ? s_sig : reinterpret_cast<uint16_t*>(smem + (SIG_LATE ? SIG_AT : 0));
    auto swz = [](int row, int chunk) { return row * BK + ((chunk ^ ((row / RPB) & (CPR - 1))) << 4); };
    // packed weight rows (64 bytes, 4 chunks): 4 rows per sweep of the banks, chunk c of row r at c ^ ((r / 4) % 4)
    auto swzp = [](int row, int chunk) { return row * (BK / 2) + ((chunk ^ ((row >> 2) & 3)) << 4); };

    const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(int(threadIdx.x) / NT);   // K group (wave-uniform)
    const int tid = KG == 1 ? int(threadIdx.x) : int(threadIdx.x) % NT, lane = tid & 63, wave = tid >> 6;
    int8_t* const sm = smem + kg * GROUP_BYTES;   // this group's stages
    const int wm = SKIP ? wave / WGN : wave % WGM, wn = SKIP ? wave % WGN : wave / WGM;

    // tile row of row r of this wave's tile (r counts whole MF-row blocks of the wave)
    auto tile_row = [&](int r) { return DEAL ? (r / MF * WGM + wm) * MF + r % MF : wm * WTM + r; };

    // ---- which tile ------------------------------------------------------------------------------------------
    const int num_n = (a.N + BN - 1) / BN;
    int m0, n0, row_end, expert = 0;
    [[maybe_unused]] int ablk0;   // first 32-row block of the tile's activations in the blocked layout
    if (a.tstart) {   // grouped: row tiles of BM inside expert segments
        // Workgroup b runs on XCD b % 8: inside every chunk of 8 row tiles each XCD takes one row tile with all of
        // its column tiles, so an activation panel is fetched into one L2 only.  The segments' row tiles (slots) may be
        // taller than this kernel's: then a slot is 1 << sub_log2 of them.
        const int j = blockIdx.x % (8 * num_n);
        const int tile = blockIdx.x / (8 * num_n) * 8 + (j & 7), slot = tile >> a.sub_log2;
        n0 = (j >> 3) * BN;
        const int E = a.n_experts;
        if (slot >= a.tstart[E]) return;
        expert = last_started(E, slot, [&](int e) { return a.tstart[e]; });   // the expert the slot belongs to
        m0 = a.off[expert] + (((slot - a.tstart[expert]) << a.sub_log2) + (tile & ((1 << a.sub_log2) - 1))) * BM;
        row_end = a.off[expert + 1];
        if (m0 >= row_end) return;   // the last slot's spare tiles
        ablk0 = tile * (BM / 32);    // blocked: slots are whole, one after the other
    } else {
        const int num_m = (a.M + BM - 1) / BM;
        int pid = blockIdx.x;
        const int total = num_m * num_n;
        if ((total & 7) == 0) pid = (pid & 7) * (total >> 3) + (pid >> 3);   // neighbours in tile order share an XCD
        // Tile order: bands of 4 row tiles, inside a band column by column.  The 32 to 128 workgroups
        // an XCD runs at once (one to four a CU) then share 4 activation panels and 8 to 32 weight panels however large
        // M is.  (Four was measured with one workgroup a CU.)
        constexpr int GM = 4;
        const int band = pid / (GM * num_n), r = pid % (GM * num_n);
        const int rows_in_band = min(GM, num_m - band * GM);
        n0 = (r / rows_in_band) * BN;
        m0 = (band * GM + r % rows_in_band) * BM;
        row_end = a.M;
        ablk0 = m0 / 32;
    }
    const int K = a.K;
    const int KL = K / KG;         // length of this group's part of the reduction
    const int kbase = kg * KL;     // and its first k (a multiple of 128)
    // MF-row blocks of this wave's tile that hold rows of the segment (wave-uniform)
    const int mi_active =
        DEAL   ? __builtin_amdgcn_readfirstlane(min(MI, max(0, ((row_end - m0 + MF - 1) / MF - wm + WGM - 1) / WGM)))
        : SKIP ? __builtin_amdgcn_readfirstlane(min(MI, max(0, (row_end - (m0 + wm * WTM) + MF - 1) / MF)))
               : MI;
    // The tile's scales are REQUESTED here, before the first operand loads, and stored to LDS after those have been
    // issued: memory returns a wave's loads in order, so scales requested first arrive first and their wait does not
    // cover the operand loads (fetched and stored up front they cost every tile two serial round trips to memory).
    constexpr int XS_PER = (BM + NT - 1) / NT, WS_PER = (BN + NT - 1) / NT;
    float xs_reg[XS_PER], ws_reg[WS_PER];
    int xs_row[XS_PER];
#pragma unroll
    for (int j = 0; j < XS_PER; ++j) {   // the scale's row: through the gather list when there is one (loaded with the
        const int m = m0 + tid + j * NT;   // operand rows' entries below, one wait for all of them)
        xs_row[j] = (a.xscale && tid + j * NT < BM && m < row_end) ? (a.gather ? a.gather[m] : m) : -1;
    }

    // ---- per-thread staging assignments (fixed over the K loop) ------------------------------------------------
    // Global operands are read with buffer loads: a per-thread byte offset fixed for the whole K loop plus a scalar
    // offset that advances with k, so the loop spends no vector instructions on addresses.
    const auto rsrc = [](const void* p, size_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, int(bytes), 0x00020000);
    };
    const size_t erow = size_t(expert) * a.N;   // first weight row of this expert
    const __amdgpu_buffer_rsrc_t ra = rsrc(a.xq, 0xFFFFFFFFu);
    const __amdgpu_buffer_rsrc_t rb = BMODE == B_INT8 ? rsrc(a.wq + erow * K, size_t(a.N) * K)
                                                      : rsrc(reinterpret_cast<const uint8_t*>(a.codes) + erow * (K / 2), size_t(a.N) * (K / 2));
    const __amdgpu_buffer_rsrc_t rbc = rsrc(a.bcodes + erow * a.bc_row_bytes, size_t(a.N) * a.bc_row_bytes);
    int a_src[A_PER], a_dst[A_PER];
    uint32_t a_live = 0;   // SKIP: the chunks of rows inside the segment (the others are neither written to LDS nor used)
#pragma unroll
    for (int j = 0; j < A_PER; ++j) {
        if (AD) { a_src[j] = a_dst[j] = 0; continue; }
        const int c = tid + j * NT;
        const int row = c / CPR, kc = c % CPR;
        if (m0 + row < row_end) a_live |= 1u << j;
        int gr = min(m0 + row, row_end - 1);   // rows past the segment re-read its last row: one cache line, not a row each
        if (a.gather) gr = a.gather[gr];
        a_src[j] = int(uint32_t(gr) * uint32_t(K) + kc * 16 + kbase);
        a_dst[j] = swz(row, kc);
    }
    int b_src[B_PER], b_bc[B_PER], b_dst[B_PER], b_dst2[B_PER], b_k[B_PER];
    [[maybe_unused]] uint32_t b_rmin[B_PER];   // B_PACKED_E8M0: lowest exponent byte of the thread's weight row
#pragma unroll
    for (int j = 0; j < B_PER; ++j) {
        const int c = tid + j * NT;
        if (BMODE == B_INT8) {
            const int row = c / CPR, kc = c % CPR;
            const int gn = min(n0 + row, a.N - 1);
            b_src[j] = gn * K + kc * 16 + kbase;
            b_dst[j] = A_BYTES + swz(row, kc);
            b_dst2[j] = 0;
            b_bc[j] = 0;
            b_k[j] = 0;
        } else {
            constexpr int RUNS = BK / (8 * WPC);   // runs per tile row
            const int row = c / RUNS, kb = c % RUNS;
            const int gn = min(n0 + row, a.N - 1);
            b_src[j] = gn * (K / 2) + kb * 4 * WPC + kbase / 2;
            // the block-code byte of the run: 4 blocks per byte, i.e. 128 weights (one byte per K step at most) or 64
            // (two 4-bit codes per byte: 32)
            b_bc[j] = gn * a.bc_row_bytes + (BMODE == B_PACKED_B16      ? (kbase + kb * 8 * WPC) >> 6
                                             : BMODE == B_PACKED_B16M   ? (kbase + kb * 8 * WPC) >> 5
                                             : BMODE == B_PACKED_E8M0   ? (kbase + kb * 8 * WPC) >> 5
                                             : BMODE == B_PACKED_DEFAULT ? kbase >> 7
                                                                        : 0);
            if (BMODE == B_PACKED_E8M0) b_rmin[j] = e8m0_row_min(a.wscale[erow + gn]);
            if (PK) {   // the run's 16 code bytes as they are
                b_dst[j] = A_BYTES + swzp(row, kb);
                b_dst2[j] = 0;
            } else {
                b_dst[j] = A_BYTES + swz(row, kb * WPC / 2);
                b_dst2[j] = A_BYTES + swz(row, kb * WPC / 2 + 1);
            }
            b_k[j] = kb * 8 * WPC;
        }
    }

#pragma unroll
    for (int j = 0; j < XS_PER; ++j) xs_reg[j] = xs_row[j] >= 0 ? a.xscale[xs_row[j]] : 0.0f;
#pragma unroll
    for (int j = 0; j < WS_PER; ++j) {
        const int c = tid + j * NT;
        ws_reg[j] = (a.xscale && c < BN && n0 + c < a.N) ? a.wscale[size_t(expert) * a.N + n0 + c] : 0.0f;
    }

    constexpr int SIG_PIECES = SIG_BYTES / 16, SIG_PER = (SIG_PIECES + NT * KG - 1) / (NT * KG);   // pieces a thread copies
    [[maybe_unused]] u32x4 sig_reg[SIG_PER];
    static_assert(alignof(silu_ce::Table) % sizeof(u32x4) == 0, "the table is read in whole pieces");
    auto load_sig = [&] {
#pragma unroll
        for (int j = 0; j < SIG_PER; ++j)
            sig_reg[j] = reinterpret_cast<const u32x4*>(a.silu)[min(int(threadIdx.x) + j * NT * KG, SIG_PIECES - 1)];
    };
    auto store_sig = [&](uint16_t* to) {
#pragma unroll
        for (int j = 0; j < SIG_PER; ++j)
            if (int(threadIdx.x) + j * NT * KG < SIG_PIECES) reinterpret_cast<u32x4*>(to)[int(threadIdx.x) + j * NT * KG] = sig_reg[j];
    };
    const bool sig_copy = SIG && a.epi == SCMX_EPI_SWIGLU, late_sig = SIG_LATE && a.epi == SCMX_EPI_SWIGLU;
    if (sig_copy) load_sig();

    // Two register sets hold the global loads of two K steps in flight.
    struct Staged {
        u32x4 a[A_PER], b[B_PER];
        uint8_t bc[B_PER];   // kept as loaded: widening it here would make the compiler wait for the load at once
    };
    Staged r0, r1;

    // Loads past the last K step re-read the last step (never consumed): every iteration issues the same loads, so
    // the wait before a register set is used covers exactly that set and not the younger one.
    // The loads of one K step are issued in NKK slices (activation chunks j with j % NKK == q in slice q, the
    // weight words in the last one) so that the K loop can spread them between its MFMAs.
    constexpr int NKK = BK / 32;
    auto load_slice = [&](Staged& r, int k0, int q) {
#pragma unroll
        for (int j = 0; j < A_PER; ++j)
            if (!AD && j % NKK == q && (A_CHUNKS % NT == 0 || tid + j * NT < A_CHUNKS))
                r.a[j] = __builtin_amdgcn_raw_buffer_load_b128(ra, a_src[j], k0, 0);
        if (q != NKK - 1) return;
#pragma unroll
        for (int j = 0; j < B_PER; ++j)
            if (B_CHUNKS % NT == 0 || tid + j * NT < B_CHUNKS) {
                if (BMODE == B_INT8) {
                    r.b[j] = __builtin_amdgcn_raw_buffer_load_b128(rb, b_src[j], k0, 0);
                } else {
                    if (WPC == 4) {
                        r.b[j] = __builtin_amdgcn_raw_buffer_load_b128(rb, b_src[j], k0 >> 1, 0);
                    } else {
                        const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rb, b_src[j], k0 >> 1, 0);
                        r.b[j][0] = v[0];
                        r.b[j][1] = v[1];
                    }
                    if (PK) continue;   // block codes go straight to the lanes that decode
                    if (BMODE == B_PACKED_DEFAULT)   // 32-blocks, 2-bit codes, 4 blocks per byte: keep the raw byte
                        r.bc[j] = __builtin_amdgcn_raw_buffer_load_b8(rbc, b_bc[j], k0 >> 7, 0);
                    if (BMODE == B_PACKED_B16)       // 16-blocks: a byte covers 64 weights
                        r.bc[j] = __builtin_amdgcn_raw_buffer_load_b8(rbc, b_bc[j], k0 >> 6, 0);
                    if (BMODE == B_PACKED_B16M)      // 16-blocks, 4-bit codes: 32 weights
                        r.bc[j] = __builtin_amdgcn_raw_buffer_load_b8(rbc, b_bc[j], k0 >> 5, 0);
                    if (BMODE == B_PACKED_E8M0)      // one exponent byte per 32 weights
                        r.bc[j] = __builtin_amdgcn_raw_buffer_load_b8(rbc, b_bc[j], k0 >> 5, 0);
                }
            }
    };
    auto load_global = [&](Staged& r, int k0) {
        k0 = min(k0, KL - BK);
#pragma unroll
        for (int q = 0; q < NKK; ++q) load_slice(r, k0, q);
    };

    // Staging work of one K step, cut into NKK slices so that it can be issued in the shadow of the MFMAs of the
    // step being multiplied: slice q writes the activation chunks j with j % NKK == q and decodes the weight code
    // words w with w * NKK / 4 == q; the last slice writes the decoded weights.
    auto stage_slice = [&](const Staged& r, int8_t* st, int k0, int q, uint32_t (&o)[B_PER][8]) {
        k0 += kbase;   // block indices below count from the row's first weight
#pragma unroll
        for (int j = 0; j < A_PER; ++j)
            if (!AD && j % NKK == q && (A_CHUNKS % NT == 0 || tid + j * NT < A_CHUNKS) && (!SKIP || ((a_live >> j) & 1u)))
                *reinterpret_cast<u32x4*>(st + a_dst[j]) = r.a[j];
#pragma unroll
        for (int j = 0; j < B_PER; ++j)
            if (B_CHUNKS % NT == 0 || tid + j * NT < B_CHUNKS) {
                if (BMODE == B_INT8) {
                    if (q == 0) *reinterpret_cast<u32x4*>(st + b_dst[j]) = r.b[j];
                } else if (PK) {
                    if (q == j % NKK) *reinterpret_cast<u32x4*>(st + b_dst[j]) = r.b[j];
                } else {
#pragma unroll
                    for (int w = 0; w < WPC; ++w) {
                        if (w * NKK / WPC != q) continue;
                        if (BMODE == B_PACKED_DEFAULT) {
                            const uint32_t blk = uint32_t(k0 + b_k[j]) >> 5;
                            decode_word_fp4(r.b[j][w], fp4_scale((uint32_t(r.bc[j]) >> (2 * (blk & 3))) & 3u), o[j][2 * w],
                                            o[j][2 * w + 1]);
                        } else if (BMODE == B_PACKED_E8M0) {   // the run lies inside one block
                            decode_word_fp4(r.b[j][w], fp4_scale((uint32_t(r.bc[j]) - b_rmin[j]) & 0x7Fu), o[j][2 * w],
                                            o[j][2 * w + 1]);
                        } else if (BMODE == B_PACKED_B16) {
                            const uint32_t blk = uint32_t(k0 + b_k[j] + 8 * w) >> 4;
                            decode_word_fp4(r.b[j][w], fp4_scale((uint32_t(r.bc[j]) >> (2 * (blk & 3))) & 3u), o[j][2 * w],
                                            o[j][2 * w + 1]);
                        } else if (BMODE == B_PACKED_B16M) {
                            const uint32_t blk = uint32_t(k0 + b_k[j] + 8 * w) >> 4;
                            const _Float16 m = _Float16(int(((uint32_t(r.bc[j]) >> (4 * (blk & 1))) & 15u) + (a.fmt.mult[0] & 0xFFu)));
                            decode_word_fp4_mul(r.b[j][w], half2_t{m, m}, o[j][2 * w], o[j][2 * w + 1]);
                        } else {
                            const uint32_t blk = uint32_t(k0 + b_k[j] + 8 * w) >> a.fmt.block_log2;
                            const uint32_t bc = block_code(a.bcodes + erow * a.bc_row_bytes + b_bc[j], blk, a.fmt.bc_bits);
                            const BlockLut t = scaled_lut_mul(a.fmt.lut_lo, a.fmt.lut_hi, mult_of(a.fmt, bc));
                            decode_word(r.b[j][w], t, o[j][2 * w], o[j][2 * w + 1]);
                        }
                    }
                    if (q == (WPC - 1) * NKK / WPC) {
                        *reinterpret_cast<u32x4*>(st + b_dst[j]) = u32x4{o[j][0], o[j][1], o[j][2], o[j][3]};
                        if (WPC == 4) *reinterpret_cast<u32x4*>(st + b_dst2[j]) = u32x4{o[j][4], o[j][5], o[j][6], o[j][7]};
                    }
                }
            }
    };
    auto store_lds = [&](const Staged& r, int stage, int k0) {
        k0 = min(k0, KL - BK);
        uint32_t o[B_PER][8];
#pragma unroll
        for (int q = 0; q < NKK; ++q) stage_slice(r, sm + stage * STAGE, k0, q, o);
    };

    constexpr int AG = MF == 32 ? 4 : 1;   // groups of four columns of a row that a lane holds of a block
    std::conditional_t<MF == 32, v16i, v4i> acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
            for (int r = 0; r < 4 * AG; ++r) acc[i][j][r] = 0;

    // fragment addresses: lane l supplies row l % MF and the 16 k-bytes of part l / MF of a k slice (64 wide in four
    // parts, or 32 in two); block origins are multiples of MF rows, so the swizzle term depends on the lane only
    constexpr int PARTS = 64 / MF, KS = BK / (16 * PARTS);   // k slices of a step
    const int lr = lane % MF, part = lane / MF;
    const int sw = (lr / RPB) & (CPR - 1);
    int koff[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) koff[s] = ((PARTS * s + part) ^ sw) << 4;
    const int a_frag = (wm * WTM + lr) * BK;
    const int b_frag = A_BYTES + (wn * WTN + lr) * BK;

    const int KT = KL / BK;
    // Pipeline.  Iteration kt: barrier; multiply step kt out of its LDS stage while the register set holding step
    // kt+2 is decoded and written into its stage, one slice per 32-wide k slice of MFMAs; then reissue that set's
    // global loads for step kt+4.  A stage is rewritten two barriers after its last read and readable one barrier
    // after it was written, so the first fragments of step kt+1 are fetched at the end of iteration kt, ahead of the
    // barrier that opens kt+1.  The stage indices are compile-time constants (the loop is unrolled over the
    // 3 stages x 2 register sets), which keeps every LDS address an immediate offset from a fixed register.
    // PK: block codes of the current / the next two K steps, one register per weight row (two in the formats with a byte
    // or a 4-bit code per block: a register per step)
    [[maybe_unused]] uint32_t bcc[NI][BCR], bcn[NI][BCR];
    [[maybe_unused]] int bc_src[NI];
#pragma unroll
    for (int j = 0; j < NI; ++j) bc_src[j] = min(n0 + wn * WTN + j * MF + lr, a.N - 1) * a.bc_row_bytes;
    // block codes of K steps s and s + 1 (s even); past the end the last pair of steps again (never consumed)
    auto load_bc = [&](int s, uint32_t (&f)[NI][BCR]) {
        const int so = min(s, (K / BK - 1) & ~1) * BCB;
#pragma unroll
        for (int j = 0; j < NI; ++j)
            if constexpr (BCR == 2) {
                const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rbc, bc_src[j], so, 0);
                f[j][0] = v[0];
                f[j][1] = v[1];
            } else {
                f[j][0] = BCB == 2 ? uint32_t(__builtin_amdgcn_raw_buffer_load_b32(rbc, bc_src[j], so, 0))
                                   : uint32_t(__builtin_amdgcn_raw_buffer_load_b16(rbc, bc_src[j], so, 0));
            }
    };
    // PK, E8M0: lowest exponent byte of the lane's weight rows
    [[maybe_unused]] uint32_t w_rmin[NI];
    if constexpr (PK && BMODE == B_PACKED_E8M0) {
#pragma unroll
        for (int j = 0; j < NI; ++j) w_rmin[j] = e8m0_row_min(a.wscale[erow + min(n0 + wn * WTN + j * MF + lr, a.N - 1)]);
    }
    // AD: the activations come in 32-row x 32-k blocks of 1 KB, 16 bytes of a row per piece, piece (row % 32, k / 16 %
    // 2) at (k / 16 % 2) * 512 + (row % 32) * 16, block (m / 32, k / 32) at ((m / 32) * (K / 32) + k / 32) KB.  A
    // fragment (16 rows x 64 k) is then four runs of 256 bytes.  Every wave loads the fragments of its own rows
    // straight into registers, two K steps ahead, in three buffers that rotate with the LDS stages (two where the largest
    // wave tile leaves no registers for a third): the activation tile never passes through LDS.
    constexpr int NAB = MF == 16 && ACC16 > 16 ? 2 : NSTAGE;   // the largest wave tiles have registers for two buffers only (below)
    [[maybe_unused]] v4i fad[NAB][KS][MI];
    [[maybe_unused]] int ad_src[ADR || DEAL ? MI : WTM / 32];
    if constexpr (ADR) {
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            int gr = min(m0 + tile_row(i * 16 + lr), row_end - 1);
            if (a.gather) gr = a.gather[gr];
            ad_src[i] = int(uint32_t(gr) * uint32_t(K) + uint32_t(part) * 16u);
        }
    } else if constexpr (DEAL) {   // blocks past the segment: the wave's last one (or the tile's first) again
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int b = mi_active ? min(i, mi_active - 1) * WGM + wm : 0;   // MF-row block of the tile
            ad_src[i] = int(uint32_t(ablk0 + (MF == 32 ? b : b >> 1)) * uint32_t(K >> 5) * 1024u + uint32_t(MF == 32 ? 0 : b & 1) * 256u +
                            uint32_t(part) * 512u + uint32_t(lr) * 16u);
        }
    } else if constexpr (AD) {
        const int last_block = (a.M + 31) / 32 - 1;
#pragma unroll
        for (int i = 0; i < WTM / 32; ++i)
            ad_src[i] = int(uint32_t(min((m0 + wm * WTM) / 32 + i, last_block)) * uint32_t(K >> 5) * 1024u +
                            uint32_t(part) * 512u + uint32_t(lr) * 16u + uint32_t(kbase) * 32u);
    }
    auto load_ad = [&](int buf, int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                // a block of 32 rows holds an MF = 32 fragment, or those of an even i and the next
                const int at = ADR               ? ad_src[i] + s * 64
                               : DEAL || MF == 32 ? ad_src[i] + s * (MF == 32 ? 1024 : 2048)
                                                  : ad_src[i / 2] + s * 2048 + (i & 1) * 256;
                const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(ra, at, ADR ? k0 : k0 * 32, 0);
                fad[buf][s][i] = v4i{int(v[0]), int(v[1]), int(v[2]), int(v[3])};
            }
    };
    if constexpr (PK) load_bc(0, bcc);   // ahead of the operand loads, like the scales
    load_global(r0, 0);
    load_global(r1, BK);
    if (a.xscale) {   // published by the barrier that opens the K loop
#pragma unroll
        for (int j = 0; j < XS_PER; ++j)
            if (tid + j * NT < BM) s_xs[tid + j * NT] = xs_reg[j];
#pragma unroll
        for (int j = 0; j < WS_PER; ++j)
            if (tid + j * NT < BN) s_ws[tid + j * NT] = ws_reg[j];
    }
    if (sig_copy) store_sig(s_sig);
    if constexpr (AD) load_ad(0, 0);
    store_lds(r0, 0, 0);
    store_lds(r1, 1, BK);
    load_global(r0, 2 * BK);
    // The loads stay apart, in the order the K loop issues them (activations of a step, then the weights two steps
    // ahead of them): the loop's first copy has two predecessors (this code and the loop's end) and waits for the fewer
    // outstanding loads of the two -- interleaved here, that wait covered the younger set as well, in every trip
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (AD) {
        load_ad(1, min(BK, KL - BK));
        __builtin_amdgcn_sched_barrier(0);
    }
    load_global(r1, 3 * BK);
    // ---- PK: fragments of packed weights ------------------------------------------------------------------------
    // The k positions of a 64-wide pair of MFMA slices are dealt so that a lane's packed codes are one 16-byte read: lane
    // half h supplies k = 64 p + 32 h + 16 s + (0..15) to slice s of pair p, i.e. 32 consecutive activation bytes (two
    // 16-byte reads) and 32 consecutive codes (one), the latter one block of 32 or two of 16.
    // Three things are in flight per wave: the MFMAs of pair p, the decode of pair p + 1 (its codes were read during pair
    // p - 1) and the LDS reads of pair p + 1's activations and pair p + 2's codes.
    // The block codes do not pass through LDS: the lane that decodes row n reads the codes of two K steps of that row
    // (2 * BCB bytes) from memory every second step, two steps ahead.
    constexpr int NKP = NKK / 2, PMI = PK ? MI : 1, PNI = PK ? NI : 1;
    [[maybe_unused]] v4i pa[2][2][PMI];   // activation fragments [pair parity][slice][row block]
    [[maybe_unused]] v4i pw[2][PNI];      // 32 codes per weight row as read from LDS [pair parity]
    [[maybe_unused]] v4i px[2][2][PNI];   // decoded INT8 operands [pair parity][slice][column block]
    [[maybe_unused]] const int w_frag = A_BYTES + (wn * WTN + lr) * (BK / 2);
    auto load_pa = [&](const int8_t* src, int kp, v4i (&f)[2][PMI]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PMI; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (!SKIP || i < mi_active)
                    f[h][i] = *reinterpret_cast<const v4i*>(src + a_frag + i * 32 * BK + (((4 * kp + 2 * part + h) ^ sw) << 4));
    };
    auto load_pw = [&](const int8_t* src, int kp, v4i (&f)[PNI]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < PNI; ++j)
            f[j] = *reinterpret_cast<const v4i*>(src + w_frag + j * 32 * (BK / 2) + (((2 * kp + part) ^ ((lr >> 2) & 3)) << 4));
    };
    // 32 codes -> the INT8 operands of the pair's two slices; `odd` = the K step's parity (which half of the block codes)
    auto decode_pair = [&](const v4i (&f)[PNI], const uint32_t (&bc)[NI][BCR], int odd, int kp,
                           v4i (&x)[2][PNI]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < PNI; ++j) {
            uint32_t o[8];
            if constexpr (BMODE == B_PACKED_B16M) {   // blocks 4 kp + 2 h and the next one of the step's 8, 4 bits each
                const uint32_t t = bc[j][odd] >> (16 * kp + 8 * part);
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const _Float16 m = _Float16(int(((t >> (4 * (w >> 1))) & 15u) + (a.fmt.mult[0] & 0xFFu)));
                    decode_word_fp4_mul(uint32_t(f[j][w]), half2_t{m, m}, o[2 * w], o[2 * w + 1]);
                }
            } else {
                float s0, s1;
                if constexpr (BMODE == B_PACKED_B16) {   // the same, 2 bits each
                    const uint32_t t = bc[j][0] >> (16 * odd + 8 * kp + 4 * part);
                    s0 = fp4_scale(t & 3u);
                    s1 = fp4_scale((t >> 2) & 3u);
                } else if constexpr (BMODE == B_PACKED_E8M0) {   // byte 2 kp + h of the step's 4
                    s0 = s1 = fp4_scale((((bc[j][odd] >> (16 * kp + 8 * part)) & 0xFFu) - w_rmin[j]) & 0x7Fu);
                } else {                                 // block 2 kp + h of the step's 4
                    s0 = s1 = fp4_scale((bc[j][0] >> (8 * odd + 4 * kp + 2 * part)) & 3u);
                }
                decode_word_fp4(uint32_t(f[j][0]), s0, o[0], o[1]);
                decode_word_fp4(uint32_t(f[j][1]), s0, o[2], o[3]);
                decode_word_fp4(uint32_t(f[j][2]), s1, o[4], o[5]);
                decode_word_fp4(uint32_t(f[j][3]), s1, o[6], o[7]);
            }
            x[0][j] = v4i{int(o[0]), int(o[1]), int(o[2]), int(o[3])};
            x[1][j] = v4i{int(o[4]), int(o[5]), int(o[6]), int(o[7])};
        }
    };
    auto iteration_pk = [&](auto step_tag, auto parity_tag, Staged& r, int kt) __attribute__((always_inline)) {
        constexpr int rd = decltype(step_tag)::value;
        constexpr int odd = decltype(parity_tag)::value;   // kt % 2
        constexpr int wr = (rd + 2) % NSTAGE;
        constexpr int nx = (rd + 1) % NSTAGE;
        __syncthreads();
        const int8_t* src = smem + rd * STAGE;
        const int8_t* nxt = smem + nx * STAGE;
        int8_t* dst = smem + wr * STAGE;
        const int k2 = min((kt + 2) * BK, K - BK);
        const int k4 = min((kt + 4) * BK, K - BK);
        uint32_t o[B_PER][8];
        if (!odd) load_bc(kt + 2, bcn);
#pragma unroll
        for (int kp = 0; kp < NKP; ++kp) {
            const int cur = kp % 2, oth = (kp + 1) % 2;   // NKP is even: pair 0 of every step has parity 0
            load_pa(kp + 1 < NKP ? src : nxt, (kp + 1) % NKP, pa[oth]);
            if (kp + 1 == NKP && odd) {   // the next pair belongs to step kt + 1
#pragma unroll
                for (int j = 0; j < NI; ++j)
#pragma unroll
                    for (int q = 0; q < BCR; ++q) bcc[j][q] = bcn[j][q];
            }
            decode_pair(pw[oth], bcc, kp + 1 < NKP ? odd : 1 - odd, (kp + 1) % NKP, px[oth]);
            load_pw(nxt, kp, pw[cur]);   // pair kp + 2 = pair kp of the next step; pw[cur] was decoded a pair ago
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int i = 0; i < PMI; ++i) {
                    if (SKIP && i >= mi_active) break;
#pragma unroll
                    for (int j = 0; j < PNI; ++j)
                        if constexpr (PK) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(px[cur][h][j], pa[cur][h][i], acc[i][j], 0, 0, 0);
                }
                stage_slice(r, dst, k2, 2 * kp + h, o);
            }
        }
        load_global(r, k4);
    };
    static_assert(!PK || NKP == 2, "the pair buffers return to phase 0 every K step");

    // MF = 16: a step runs in phases, two per 64-wide k slice: the operand with more 16-row blocks in the wave's tile
    // is split, one half of its fragments per phase, and fetched FD - 1 phases ahead into FD rotating register buffers;
    // the other operand's fragments are held for the slice and fetched one slice ahead, half of them in each phase.
    // The fragments fetched at the end of an iteration belong to the next step's stage.
    // MF = 32: a phase is a 32-wide k slice with the fragments of all of the wave's rows and columns.
    constexpr bool F16 = MF == 16;
    constexpr bool SPLITN = AD || NI >= MI;                 // the split operand: weights (columns) or activations (rows)
    constexpr int SF = F16 ? (SPLITN ? NI : MI) / 2 : 1, HF = F16 ? (SPLITN ? MI : NI) : 1;
    constexpr int AHEAD = FD - 1;
    static_assert(AHEAD >= 1 && AHEAD <= NKK, "fragment prefetch distance");
    [[maybe_unused]] v4i fs[FD][SF], fh[2][HF];
    auto load_split = [&](const int8_t* src, int phase, v4i (&x)[SF]) __attribute__((always_inline)) {
        if (SKIP && mi_active == 0) return;
#pragma unroll
        for (int f = 0; f < SF; ++f) {
            const int blk = (phase & 1) * SF + f;
            if (!SPLITN && SKIP && blk >= mi_active) continue;
            x[f] = *reinterpret_cast<const v4i*>(src + (SPLITN ? b_frag : a_frag) + blk * 16 * BK + koff[phase >> 1]);
        }
    };
    auto load_held = [&](const int8_t* src, int s, int part, v4i (&x)[HF]) __attribute__((always_inline)) {
        if (AD || (SKIP && mi_active == 0)) return;
#pragma unroll
        for (int f = 0; f < HF; ++f) {
            if (f / ((HF + 1) / 2) != part) continue;
            if (SPLITN && SKIP && f >= mi_active) continue;
            x[f] = *reinterpret_cast<const v4i*>(src + (SPLITN ? a_frag : b_frag) + f * 16 * BK + koff[s]);
        }
    };
    constexpr int AI = F16 ? 1 : MI, BI = F16 ? 1 : NI;
    [[maybe_unused]] v4i fa[FD][AI], fb[FD][BI];
    auto load_frags = [&](const int8_t* src, int kk, v4i (&xa)[AI], v4i (&xb)[BI]) __attribute__((always_inline)) {
        if (SKIP && mi_active == 0) return;
#pragma unroll
        for (int i = 0; i < AI; ++i)
            if (!AD && (!SKIP || i < mi_active)) xa[i] = *reinterpret_cast<const v4i*>(src + a_frag + i * 32 * BK + koff[kk]);
#pragma unroll
        for (int j = 0; j < BI; ++j) xb[j] = *reinterpret_cast<const v4i*>(src + b_frag + j * 32 * BK + koff[kk]);
    };
    __syncthreads();
    if constexpr (PK) {
        load_pa(smem, 0, pa[0]);
        load_pw(smem, 0, pw[0]);
        load_pw(smem, 1, pw[1]);
        decode_pair(pw[0], bcc, 0, 0, px[0]);
    } else if constexpr (!F16) {
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) load_frags(sm, q, fa[q], fb[q]);
    } else {
        load_held(sm, 0, 0, fh[0]);
        load_held(sm, 0, 1, fh[0]);
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) load_split(sm, q, fs[q]);
    }
    // The k slices of an iteration are fenced against each other for the scheduler: left alone, the compiler sinks every
    // LDS write of the step to its end, in front of the barrier (32x32x32 MFMAs, M = 8192: 442 -> 429 us over the four
    // layers with the fences on the 256x256 tile; M = 128 ... 1024 on the small tiles: 2-3 %).
    auto iteration_staged = [&](auto step_tag, auto parity_tag, auto stage_tag, Staged& r, int kt) __attribute__((always_inline)) {
        constexpr int rd = decltype(step_tag)::value;        // kt % 3: stage of step kt
        constexpr bool ST = decltype(stage_tag)::value;      // false in the last two steps: nothing left to stage
        constexpr int wr = (rd + 2) % NSTAGE;                // stage of step kt + 2
        constexpr int nx = (rd + 1) % NSTAGE;                // stage of step kt + 1
        constexpr int ph = (NKK * rd) % FD;                  // buffer of phase 0 of this step (FD divides 6 * NKK)
        constexpr int hp = KS == 1 ? int(decltype(parity_tag)::value) : 0;   // held buffer of slice 0 (kt % 2 if odd counts)
        __syncthreads();
        const int8_t* src = sm + rd * STAGE;
        const int8_t* nxt = sm + nx * STAGE;
        int8_t* dst = sm + wr * STAGE;
        const int k2 = min((kt + 2) * BK, KL - BK);      // past the end: rewrites a stage nobody reads again
        const int k4 = min((kt + 4) * BK, KL - BK);
        uint32_t o[B_PER][8];
        constexpr int ab = NAB == 2 ? int(decltype(parity_tag)::value) : rd;   // activation buffer of this step
        if constexpr (AD && ST && NAB == 3) load_ad(wr, k2);
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk) {
            const int s = F16 ? kk >> 1 : kk, h = kk & 1, now = (ph + kk) % FD, then = (ph + kk + AHEAD) % FD;
            if constexpr (F16) {
                load_split(kk + AHEAD < NKK ? src : nxt, (kk + AHEAD) % NKK, fs[then]);
                load_held(s + 1 < KS ? src : nxt, (s + 1) % KS, h, fh[(hp + s + 1) % 2]);
            } else {
                load_frags(kk + AHEAD < NKK ? src : nxt, (kk + AHEAD) % NKK, fa[then], fb[then]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int x = 0; x < (F16 && !SPLITN ? SF : MI); ++x) {
                const int i = F16 && !SPLITN ? h * SF + x : x;
                if (SKIP && i >= mi_active) continue;
#pragma unroll
                for (int y = 0; y < (F16 && SPLITN ? SF : NI); ++y) {
                    const int j = F16 && SPLITN ? h * SF + y : y;
                    if constexpr (F16) {
                        const v4i act = AD ? fad[ab][s][i] : SPLITN ? fh[(hp + s) % 2][i] : fs[now][x];
                        const v4i wgt = SPLITN ? fs[now][y] : fh[(hp + s) % 2][j];
                        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wgt, act, acc[i][j], 0, 0, 0);
                    } else {
                        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[now][j], AD ? fad[ab][s][i] : fa[now][i], acc[i][j], 0, 0, 0);
                    }
                }
            }
            if constexpr (ST) stage_slice(r, dst, k2, kk, o);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (AD && ST && NAB == 2) load_ad(ab, k2);   // into the buffer just multiplied
        if constexpr (ST) load_global(r, k4);
    };
    auto iteration = [&](auto step_tag, auto parity_tag, Staged& r, int kt) __attribute__((always_inline)) {
        if constexpr (PK) iteration_pk(step_tag, parity_tag, r, kt); else iteration_staged(step_tag, parity_tag, std::true_type{}, r, kt);
    };
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    using S2 = std::integral_constant<int, 2>;
    // Whole trips of 6 steps run without an exit inside; the remaining steps are nested so that every copy of the
    // iteration has exactly one predecessor.  (With merging paths the compiler must assume the fewest outstanding
    // loads of any path when it places its waits, and ends up waiting for loads issued one step ago.)
    int kt = 0;
    using Even = std::integral_constant<int, 0>;
    using Odd = std::integral_constant<int, 1>;
    if constexpr (PK) {
        for (; kt + 6 <= KT; kt += 6) {   // kt stays even here: the parity of every copy is fixed
            iteration(S0{}, Even{}, r0, kt);
            iteration(S1{}, Odd{}, r1, kt + 1);
            iteration(S2{}, Even{}, r0, kt + 2);
            iteration(S0{}, Odd{}, r1, kt + 3);
            iteration(S1{}, Even{}, r0, kt + 4);
            iteration(S2{}, Odd{}, r1, kt + 5);
        }
        if (kt < KT) {
            iteration(S0{}, Even{}, r0, kt);
            if (kt + 1 < KT) {
                iteration(S1{}, Odd{}, r1, kt + 1);
                if (kt + 2 < KT) {
                    iteration(S2{}, Even{}, r0, kt + 2);
                    if (kt + 3 < KT) {
                        iteration(S0{}, Odd{}, r1, kt + 3);
                        if (kt + 4 < KT) iteration(S1{}, Even{}, r0, kt + 4);
                    }
                }
            }
        }
    } else {
        // The last two steps find their stages written and have nothing to stage or load: they run as copies without
        // that work.  Small wave tiles append them at each exit of the staged steps (one predecessor each); larger
        // ones, with few registers to spare for the copies that so many joins cost, select them by the stage reached;
        // the largest (128 accumulators, 256x256) keeps every step alike and stages past the end.
        constexpr bool INLINE_TAIL = ACC16 <= 8, NO_TAIL = ACC16 > 16;
        static_assert(!F16 || (AD ? NAB == 3 || NO_TAIL : KS == 2 || NO_TAIL), "the copies without staging do not know their step's parity");
        const int KM = NO_TAIL ? KT : max(KT - 2, 0);   // steps that stage step kt + 2
        auto last_two = [&](auto s_first, auto s_second) __attribute__((always_inline)) {
            iteration_staged(s_first, Even{}, std::false_type{}, r0, 0);
            if (KT >= 2) iteration_staged(s_second, Even{}, std::false_type{}, r0, 0);
        };
        auto tail = [&](auto s_first, auto s_second) __attribute__((always_inline)) {
            if constexpr (INLINE_TAIL) last_two(s_first, s_second);
        };
        for (; kt + 6 <= KM; kt += 6) {
            iteration(S0{}, Even{}, r0, kt);
            iteration(S1{}, Odd{}, r1, kt + 1);
            iteration(S2{}, Even{}, r0, kt + 2);
            iteration(S0{}, Odd{}, r1, kt + 3);
            iteration(S1{}, Even{}, r0, kt + 4);
            iteration(S2{}, Odd{}, r1, kt + 5);
        }
        if (kt < KM) {
            iteration(S0{}, Even{}, r0, kt);
            if (kt + 1 < KM) {
                iteration(S1{}, Odd{}, r1, kt + 1);
                if (kt + 2 < KM) {
                    iteration(S2{}, Even{}, r0, kt + 2);
                    if (kt + 3 < KM) {
                        iteration(S0{}, Odd{}, r1, kt + 3);
                        if (kt + 4 < KM) {
                            iteration(S1{}, Even{}, r0, kt + 4);
                            tail(S2{}, S0{});
                        } else {
                            tail(S1{}, S2{});
                        }
                    } else {
                        tail(S0{}, S1{});
                    }
                } else {
                    tail(S2{}, S0{});
                }
            } else {
                tail(S1{}, S2{});
            }
        } else {
            tail(S0{}, S1{});
        }
        if constexpr (!INLINE_TAIL && !NO_TAIL) {
            switch (KM % 3) {
                case 0: last_two(S0{}, S1{}); break;
                case 1: last_two(S1{}, S2{}); break;
                default: last_two(S2{}, S0{}); break;
            }
        }
    }

    // ---- epilogue ---------------------------------------------------------------------------------------------
    // Lane holds acc[i][j][r] = (m = i*16 + lane%16, n = j*16 + 4(lane/16) + r) of its wave tile: 4 consecutive
    // columns of one row, the unit every epilogue works on.  Results go through a per-wave LDS tile so that global
    // stores are 16 bytes per lane over whole contiguous row segments.
    const int N = a.N;
    if (late_sig) load_sig();
    __syncthreads();   // every wave is done reading the staging buffers
    if (late_sig) {
        store_sig(sig);
        __syncthreads();
    }
    if constexpr (KG > 1) {   // the groups' partial sums meet in group 0 (register r of thread t at word r * NT + t)
        if (kg > 0) {
            int32_t* sums = reinterpret_cast<int32_t*>(smem + PART_BASE + (kg - 1) * PART_BYTES);
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j)
#pragma unroll
                    for (int r = 0; r < 4 * AG; ++r) sums[((i * NI + j) * 4 * AG + r) * NT + tid] = acc[i][j][r];
        }
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int g = 1; g < KG; ++g) {
            const int32_t* other = reinterpret_cast<const int32_t*>(smem + PART_BASE + (g - 1) * PART_BYTES);
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j)
#pragma unroll
                    for (int r = 0; r < 4 * AG; ++r) acc[i][j][r] += other[((i * NI + j) * 4 * AG + r) * NT + tid];
        }
    }
    auto epilogue = [&](auto epi_tag) {
    constexpr int epi = decltype(epi_tag)::value;
    constexpr int esize = epi == SCMX_EPI_I32 ? 4 : 2;
    constexpr int ocols = epi == SCMX_EPI_SWIGLU ? WTN / 2 : WTN;     // output columns of the wave tile
    const int on = epi == SCMX_EPI_SWIGLU ? N / 2 : N;            // output row length
    constexpr int rowb = ocols * esize;                                // bytes per tile row
    constexpr int rsb = rowb + 16;                                     // padded LDS row stride
    constexpr bool fits = WGM * WGN * WTM * rsb <= SMEM_BYTES;   // per-wave tiles reuse the staging LDS
    int8_t* wtile = smem + (fits ? wave * (WTM * rsb) : 0);
    const int wn0 = n0 + wn * WTN;            // wave tile origin (input column index)
    const bool wide = fits && (size_t(on) * esize) % 16 == 0 && reinterpret_cast<uintptr_t>(a.out) % 16 == 0 &&
                      (epi != SCMX_EPI_RES || reinterpret_cast<uintptr_t>(a.res) % 16 == 0);

    float xsv[MI];
    f32x4 wsv[NI][AG];
    if (epi != SCMX_EPI_I32) {
#pragma unroll
        for (int i = 0; i < MI; ++i) xsv[i] = s_xs[tile_row(i * MF + lr)];
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
            for (int g = 0; g < AG; ++g) wsv[j][g] = *reinterpret_cast<const f32x4*>(&s_ws[wn * WTN + j * MF + 8 * g + 4 * part]);
    }
    auto emit = [&](auto wide_tag) __attribute__((always_inline)) {
    constexpr bool W = decltype(wide_tag)::value;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int row = i * MF + lr;
        const int m = m0 + tile_row(row);
        if (SKIP && i >= mi_active) break;
        const float xs = epi != SCMX_EPI_I32 ? xsv[i] : 0.0f;
#pragma unroll
        for (int jg = 0; jg < NI * AG; ++jg) {
            const int j = jg / AG, g = jg % AG;
            const int col = j * MF + 8 * g + 4 * part;
            const int n = wn0 + col;
            if (epi == SCMX_EPI_I32) {
                const v4i v = v4i{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
                if (W)
                    *reinterpret_cast<v4i*>(wtile + row * rsb + col * 4) = v;
                else if (m < row_end && n < N)
                    *reinterpret_cast<v4i*>(reinterpret_cast<int32_t*>(a.out) + size_t(m) * N + n) = v;
                continue;
            }
            const f32x4 w4 = wsv[j][g];
            float y[4];
#pragma unroll
            for (int r = 0; r < 4; ++r)
                y[r] = __fmul_rn(__fmul_rn(float(acc[i][j][4 * g + r]), xs), w4[r]);
            uint16_t* out = reinterpret_cast<uint16_t*>(a.out);
            if (epi == SCMX_EPI_SWIGLU) {   // (g, g, u, u) -> two outputs
                const uint32_t o = swiglu_lut2(SIG || SIG_LATE ? sig : a.silu, y[0], y[1], y[2], y[3]);
                if (W)
                    *reinterpret_cast<uint32_t*>(wtile + row * rsb + col) = o;
                else if (m < row_end && n < N)
                    *reinterpret_cast<uint32_t*>(out + size_t(m) * on + n / 2) = o;
                continue;
            }
            u32x2 o;
            o[0] = f32_to_bf16x2(y[0], y[1]);
            o[1] = f32_to_bf16x2(y[2], y[3]);
            if (W) {
                *reinterpret_cast<u32x2*>(wtile + row * rsb + col * 2) = o;   // the residual is added on the way out
            } else if (m < row_end && n < N) {
                if (epi == SCMX_EPI_RES) {
                    const u32x2 rr = *reinterpret_cast<const u32x2*>(a.res + size_t(m) * N + n);
#pragma unroll
                    for (int r = 0; r < 2; ++r) {
                        const float lo = __fadd_rn(__uint_as_float(rr[r] << 16), __uint_as_float(o[r] << 16));
                        const float hi = __fadd_rn(__uint_as_float(rr[r] & 0xFFFF0000u), __uint_as_float(o[r] & 0xFFFF0000u));
                        o[r] = f32_to_bf16x2(lo, hi);
                    }
                }
                *reinterpret_cast<u32x2*>(out + size_t(m) * N + n) = o;
            }
        }
    }
    };
    if (wide) emit(std::true_type{}); else emit(std::false_type{});
    if (!wide) return;
    __builtin_amdgcn_wave_barrier();   // LDS operations of one wave complete in order: the tile is visible to its lanes

    // read the tile back 16 bytes per lane, whole rows at a time, and store
    constexpr int ppr = rowb / 16;                 // 16-byte pieces per tile row (2, 4, 8 or 16)
    constexpr int epp = 16 / esize;                // output elements per piece
    const int ocol0 = epi == SCMX_EPI_SWIGLU ? wn0 / 2 : wn0;
    // In batches of eight pieces per lane: all LDS reads (and residual loads) of a batch are in flight before the first
    // is used, instead of one round trip per piece.
    constexpr int NP = WTM * ppr / 64, NB = NP < 8 ? NP : 8;
    static_assert(WTM * ppr % 64 == 0 && NP % NB == 0, "whole batches of pieces per lane");
#pragma unroll 1
    for (int p0 = lane; p0 < (SKIP ? mi_active * MF : WTM) * ppr; p0 += 64 * NB) {
        u32x4 v[NB], rr[NB];
        bool ok[NB], full[NB];
        int8_t* dst[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int p = p0 + 64 * i;
            const int row = p / ppr, pc = p % ppr;
            const int m = m0 + tile_row(row), c = ocol0 + pc * epp;
            ok[i] = m < row_end && c < on;
            full[i] = c + epp <= on;
            dst[i] = reinterpret_cast<int8_t*>(a.out) + (size_t(m) * on + c) * esize;
            v[i] = *reinterpret_cast<const u32x4*>(wtile + row * rsb + pc * 16);
            if (epi == SCMX_EPI_RES) {
                rr[i] = u32x4{0u, 0u, 0u, 0u};
                if (ok[i]) {
                    if (full[i]) {
                        rr[i] = *reinterpret_cast<const u32x4*>(a.res + size_t(m) * on + c);
                    } else {
                        const u32x2 r2 = *reinterpret_cast<const u32x2*>(a.res + size_t(m) * on + c);
                        rr[i][0] = r2[0];
                        rr[i][1] = r2[1];
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            if (!ok[i]) continue;
            if (epi == SCMX_EPI_RES) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float lo = __fadd_rn(__uint_as_float(rr[i][r] << 16), __uint_as_float(v[i][r] << 16));
                    const float hi = __fadd_rn(__uint_as_float(rr[i][r] & 0xFFFF0000u), __uint_as_float(v[i][r] & 0xFFFF0000u));
                    v[i][r] = f32_to_bf16x2(lo, hi);
                }
            }
            if (full[i])
                // streaming store: the tile is not read again by this kernel, and lines that never sit dirty in the L2
                // do not have to be written back when the kernel ends
                __builtin_nontemporal_store(v[i], reinterpret_cast<u32x4*>(dst[i]));
            else   // the row ends inside this piece: rows are multiples of 4 elements, so exactly half of it is valid
                *reinterpret_cast<u32x2*>(dst[i]) = u32x2{v[i][0], v[i][1]};
        }
    }
    };
    switch (a.epi) {
        case SCMX_EPI_I32: epilogue(std::integral_constant<int, SCMX_EPI_I32>{}); break;
        case SCMX_EPI_SCALE: epilogue(std::integral_constant<int, SCMX_EPI_SCALE>{}); break;
        case SCMX_EPI_RES: epilogue(std::integral_constant<int, SCMX_EPI_RES>{}); break;
        default: epilogue(std::integral_constant<int, SCMX_EPI_SWIGLU>{}); break;
    }
}

// ---- launch ----------------------------------------------------------------------------------------------------

// The weight modes a tile is built for: what callers never ask of it is not compiled.
constexpr unsigned ALL_MODES = 63u, PACKED_MODES = ALL_MODES & ~(1u << B_INT8), FP4_MODES = PACKED_MODES & ~(1u << B_PACKED_GENERIC);

template <int BM, int BN, int BK, int WGM, int WGN, int OCC = 1, int FD = 2, bool SKIP = false, bool PK = false, int KG = 1,
          int ADM = 0, int MF = 16, unsigned MODES = ALL_MODES>
static void launch_tile(const GemmArgs& a_in, int bmode, int row_tiles, hipStream_t s) {
    GemmArgs a = a_in;
    if (a.epi == SCMX_EPI_SWIGLU) a.silu = silu_table_device();
    const int num_n = (a.N + BN - 1) / BN;
    if (a.tstart) row_tiles = (row_tiles + 7) & ~7;   // grouped: whole chunks of 8 row-tile slots (spare slots exit at once)
    const dim3 grid(unsigned(row_tiles) * unsigned(num_n)), block(WGM * WGN * KG * 64);
    const auto go = [&](auto mode) {
        constexpr int B = decltype(mode)::value;
        if constexpr ((MODES >> B) & 1u) gemm_kernel<BM, BN, BK, WGM, WGN, B, OCC, FD, SKIP, PK, KG, ADM, MF><<<grid, block, 0, s>>>(a);
    };
    switch (bmode) {
        case B_INT8: return go(std::integral_constant<int, B_INT8>{});
        case B_PACKED_DEFAULT: return go(std::integral_constant<int, B_PACKED_DEFAULT>{});
        case B_PACKED_B16: return go(std::integral_constant<int, B_PACKED_B16>{});
        case B_PACKED_B16M: return go(std::integral_constant<int, B_PACKED_B16M>{});
        case B_PACKED_E8M0: return go(std::integral_constant<int, B_PACKED_E8M0>{});
        default: return go(std::integral_constant<int, B_PACKED_GENERIC>{});
    }
}

}  // namespace scmx

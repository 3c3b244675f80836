// GEMM on fp32 operands with the bf16 matrix cores: x = hi + lo with hi = bf16(x), lo = bf16(x - hi), and
// a @ b = a_hi b_hi + a_hi b_lo + a_lo b_hi in fp32 (everything but a_lo b_lo: about 16 mantissa bits).
//
// The operands are read as fp32 and split in registers between the LDS and the matrix cores.  Splitting them in
// a pass of their own first costs that pass (1000 x 4096 x 2048: 23 us) and makes the product read six bytes per
// element (hi, hi, lo) where four are enough; what one compute unit can take in bounds these shapes (gemm_ks.hip).
//
// Tiles, waves and the sum of the two k halves are those of gemm_ks.hip: 128 x 128, a wavefront owns 64 x 128 for
// half of the k.  A stage is 32 k of fp32 (rows of 128 bytes); the two wavefronts of a pair take alternate stages, so
// a step is two stages (64 k) and 96 v_mfma_f32_16x16x32_bf16 per wavefront: three products of 32 blocks.
// A fragment is two 16-byte pieces of a row (pieces q and 4 + q of the eight for lane group q: both operands use
// this order of the k, and each read touches all banks once); its eight values become one hi and one lo operand with
// 16 vector instructions (v_dot2_f32_bf16 subtracts a hi half without unpacking it; 24 with shifts and subtractions
// are 5 % slower over the whole product).
// Measured, split pass + bf16 product of 3K before, now: 1000 x 4096 x 2048 row-major B 87 -> 62 us, transposed B 94 -> 59;
// 16 x 4096 x 2048 45 -> 22; 1024 x 4096 x 8192 transposed 299 -> 211.  A step takes 1.5 us: 0.85 for its MFMAs alone
// (the clock is then at 1.8 GHz), 0.3 for what the loads add, 0.3 for splitting and fragment reads between the MFMAs of
// the one wavefront a SIMD holds.
#include "gemm_common.h"

namespace kr {

namespace {

constexpr int BT = 128;                        // tile rows and columns
constexpr int BKS = 32;                        // k of a stage
constexpr int kOper = BT * BKS * 4;            // bytes of one operand in a stage: 16 KiB
constexpr int kStage = 2 * kOper;              // A, then B
constexpr int kRing = 5;                       // stages
constexpr int kLds = kRing * kStage;           // 160 KiB
constexpr int kWaves = 4;
constexpr int kLoadsA = kOper / 1024 / kWaves;       // LDS-DMA loads (1 KiB) of A per wave and stage: 4, and 4 of B
constexpr int kLoads = 2 * kLoadsA;
constexpr int kEpWave = 32 * (BT + 4) * 4;
static_assert(kEpWave * kWaves <= kLds, "epilogue patch must fit in the stages");

// schedule of a step's 96 MFMA slots (see k_step below)
constexpr int kBar = 8, kReadGap = 3, kConv0 = 32, kLoadGap = 5;
static_assert(kBar + 1 + kLoadGap * (2 * kLoads - 1) < 96 && kConv0 + 48 <= 96 && kBar + 1 + kReadGap * 11 < kConv0 + 4 * 11 - 8, "step schedule");

typedef const __attribute__((address_space(3))) f32x4* lds_f4;
typedef const __attribute__((address_space(3))) float* lds_f1;
typedef __attribute__((address_space(3))) f32x4* lds_f32x4;

constexpr int vmcnt_lgkm0_imm(int n) { return (n & 15) | (7 << 4) | (0 << 8) | ((n >> 4) << 14); }

// EVEN: M and N are multiples of 128, K of 64.
template <bool B_NT, bool EVEN>
__global__ __launch_bounds__(kWaves * 64) void gemm_f32_kernel(const GemmArgs g) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // starts at LDS address 0
    const float* A = (const float*)g.A;
    const float* B = (const float*)g.B;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int mh = wave >> 1, kh = wave & 1;   // rows 64 mh .. +63 of the tile, stage kh of a step
    int tile_m, tile_n;
    tile_of(g, blockIdx.x, 0, tile_m, tile_n);
    const int m0 = tile_m * BT, n0 = tile_n * BT;
    // steps of this workgroup (64 k each): all of them, or the share of split blockIdx.y
    const int kt_all = (g.K + 2 * BKS - 1) / (2 * BKS);
    const int kt_begin = g.k_splits > 1 ? (int)((int64_t)kt_all * blockIdx.y / g.k_splits) : 0;
    const int kt_total = g.k_splits > 1 ? (int)((int64_t)kt_all * (blockIdx.y + 1) / g.k_splits) - kt_begin : kt_all;
    const int k_begin = kt_begin * 2 * BKS;
    const float* a_tile = A + (int64_t)m0 * g.lda + k_begin;

    // ---- LDS-DMA addressing -------------------------------------------------------------------
    // A (and transposed B): a load fills 8 rows: lane l -> row l/8, slot l%8 holds piece slot ^ ((row >> 1) & 7);
    // wave w takes the row groups w, w+4, w+8, w+12
    const int sw = (4 * (wave & 1) + (lane >> 4)) & 7;
    const int piece = (lane & 7) ^ sw;
    const uint32_t a_voff = (uint32_t)(((int64_t)(lane >> 3) * g.lda + piece * 4) * 4);
    uint32_t b_voff[2];
    if (B_NT) {
        b_voff[0] = b_voff[1] = (uint32_t)(((int64_t)(lane >> 3) * g.ldb + piece * 4) * 4);
    } else {
        // row-major B: a load fills 2 k-rows of 512 bytes: lane l -> k-row l/32, slot l%32 holds piece
        // slot ^ 4*((k >> 2) & 3); wave w takes the groups w, w+4, w+8, w+12 of the stage's 16, whose (k >> 2) & 3
        // is w/2 for the even ones and w/2 + 2 for the odd ones
#pragma unroll
        for (int o = 0; o < 2; ++o)
            b_voff[o] = (uint32_t)(((int64_t)(lane >> 5) * g.ldb + (((lane & 31) ^ (4 * ((wave >> 1) + 2 * o))) << 2)) * 4);
    }
    // stages at or past K: the pieces past K are requested out of range, which writes zeros
    // (row-major B: its k-rows past K lie past the matrix' end)
    const int s_all = 2 * kt_total;                         // stages of this workgroup
    const int s_tail = (g.K - k_begin) / BKS;               // first stage of the workgroup that is not full (or past its end)
    constexpr uint32_t kOob = 0x80000000u;
    const bool in_k = EVEN || s_tail * BKS + piece * 4 < g.K - k_begin;
    const uint32_t a_tail = in_k ? a_voff : kOob, b_tail = in_k ? b_voff[0] : kOob;
    const int rows_a = EVEN ? BT : min(BT, g.M - m0), rows_b = EVEN ? BT : min(BT, g.N - n0);
    const i32x4 a_rsrc = raw_rsrc(a_tile, EVEN ? (int64_t)0x7fffffff : ((int64_t)(rows_a - 1) * g.lda + (g.K - k_begin)) * 4);
    const i32x4 bt_rsrc = raw_rsrc(B + (int64_t)n0 * g.ldb + k_begin,
                                   EVEN ? (int64_t)0x7fffffff : ((int64_t)(rows_b - 1) * g.ldb + (g.K - k_begin)) * 4);
    // load q of stage s into LDS offset `stage`; past the last stage nothing is needed, but the count per step must
    // not change (the waits below count loads), so all lanes re-read the first 16 bytes of the last one
    auto issue_load = [&](int s, uint32_t stage, int q) __attribute__((always_inline)) {
        const bool live = s < s_all;
        const int ss = min(s, s_all - 1), k0 = ss * BKS;
        const bool tail = !EVEN && ss == s_tail, past = !EVEN && ss > s_tail;
        const int rg = wave + 4 * (q % kLoadsA);
        if (q < kLoadsA) {
            lds_dma_b128(a_rsrc, stage + rg * 1024, !live ? 0u : past ? kOob : tail ? a_tail : a_voff, (int)(((int64_t)8 * rg * g.lda + k0) * 4));
        } else if (B_NT) {
            lds_dma_b128(bt_rsrc, stage + kOper + rg * 1024, !live ? 0u : past ? kOob : tail ? b_tail : b_voff[0], (int)(((int64_t)8 * rg * g.ldb + k0) * 4));
        } else {
            const int64_t kb = k_begin + k0;
            lds_dma_b128(raw_rsrc(B + kb * g.ldb + n0, EVEN ? (int64_t)0x7fffffff : ((g.K - 1 - kb) * g.ldb + (g.N - n0)) * 4),
                         stage + kOper + rg * 1024, live ? b_voff[q & 1] : 0u, (int)((int64_t)2 * rg * g.ldb * 4));
        }
    };

    // ---- fragments --------------------------------------------------------------------------------
    // lane -> row p = lane%16 of a 16-row block, pieces gq and 4 + gq of the row (gq = lane/16).  A's four blocks are
    // taken in the order 0 1 2 3 by the first wave of a pair and 2 3 0 1 by the second (see gemm_ks.hip).
    const int p = lane & 15, gq = lane >> 4;
    const uint32_t f0 = (uint32_t)(p * 128 + ((gq ^ ((p >> 1) & 7)) << 4)), f1 = (uint32_t)(p * 128 + (((4 + gq) ^ ((p >> 1) & 7)) << 4));
    const uint32_t ab[2] = {(uint32_t)(mh * 64 * 128 + kh * 32 * 128), (uint32_t)(mh * 64 * 128 + (kh ^ 1) * 32 * 128)};
    uint32_t fb[B_NT ? 1 : 4];   // row-major B: k-row 4 gq, column p of the 16-column block 4c + r at fb[r] + c * 256
    if (!B_NT) {
#pragma unroll
        for (int r = 0; r < 4; ++r) fb[B_NT ? 0 : r] = kOper + (uint32_t)(4 * gq * 512 + (((4 * r + (p >> 2)) ^ (4 * gq)) << 4) + (p & 3) * 4);
    } else {
        fb[0] = kOper;
    }
    // fragment f of a step: 0 .. 7 the column blocks of B, 8 .. 11 the row blocks of A
    float raw[12][8];
    u32x4 hi[2][12], lo[2][12];
    auto read_frag = [&](int f, uint32_t stage) __attribute__((always_inline)) {
        if (!B_NT && f < 8) {
            const uint32_t a = fb[B_NT ? 0 : f & 3] + stage + (f >> 2) * 256;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                raw[f][e] = *(lds_f1)(size_t)(a + e * 512);
                raw[f][4 + e] = *(lds_f1)(size_t)(a + (16 + e) * 512);
            }
        } else {
            const uint32_t a = stage + (f < 8 ? fb[0] + f * 2048 : ab[(f - 8) >> 1] + ((f - 8) & 1) * 2048);
            const f32x4 x = *(lds_f4)(size_t)(f0 + a), y = *(lds_f4)(size_t)(f1 + a);
            raw[f][0] = x.x; raw[f][1] = x.y; raw[f][2] = x.z; raw[f][3] = x.w;
            raw[f][4] = y.x; raw[f][5] = y.y; raw[f][6] = y.z; raw[f][7] = y.w;
        }
    };
    // values 2e and 2e+1 of fragment f.  (The factors (-1, 0) and (0, -1) are kept from the compiler: it would encode
    // the first as the inline constant -1.0, which the instruction reads as (0, -1) too.)
    uint32_t sel0 = 0x0000bf80u, sel1 = 0xbf800000u;
    asm("" : "+s"(sel0));
    asm("" : "+s"(sel1));
    auto split2 = [&](int buf, int f, int e) __attribute__((always_inline)) {
        const uint32_t h = pack_bf16(raw[f][2 * e], raw[f][2 * e + 1]);
        const bf16x2 hb = __builtin_bit_cast(bf16x2, h);
        hi[buf][f][e] = h;   // x - hi is exact
        lo[buf][f][e] = pack_bf16(__builtin_amdgcn_fdot2_f32_bf16(hb, __builtin_bit_cast(bf16x2, sel0), raw[f][2 * e], false),
                                  __builtin_amdgcn_fdot2_f32_bf16(hb, __builtin_bit_cast(bf16x2, sel1), raw[f][2 * e + 1], false));
    };

    f32x4 acc[4][8];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#define KR_SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)
    auto pin = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j) asm volatile("" : "+a"(acc[i][j]));
    };
    pin();
    // stages 0 .. 4 are requested before the loop; wait for stages 0 and 1
#pragma unroll
    for (int st = 0; st < kRing; ++st)
#pragma unroll
        for (int q = 0; q < kLoads; ++q) issue_load(st, st * kStage, q);
    __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm((kRing - 2) * kLoads));
    __builtin_amdgcn_s_barrier();
    KR_SCHED_FENCE();
#pragma unroll
    for (int f = 0; f < 12; ++f) read_frag(f, kh * kStage);
#pragma unroll
    for (int f = 0; f < 12; ++f)
#pragma unroll
        for (int e = 0; e < 4; ++e) split2(0, f, e);
    KR_SCHED_FENCE();

    // ---- k loop ------------------------------------------------------------------------------------
    // Step t: 96 MFMAs on the operands split during step t-1 (hi hi, then b_lo a_hi, then b_hi a_lo over the 32
    // blocks, so that an accumulator is used once in 32 slots).  Behind slot kBar the wave waits for its fragment
    // reads of step t and for stages 2t+2 and 2t+3 (stage 2t+4 stays outstanding) and meets the others; then the
    // fragments of step t+1 are read, one per kReadGap slots, and split from slot kConv0 on, two values per slot; the
    // stages of step t are free, and the loads of stages 2t+5 and 2t+6 go out, one per kLoadGap slots.
    uint32_t st_next = 2 * kStage + kh * kStage, st_load = 0;
    auto wrap = [](uint32_t s) __attribute__((always_inline)) { return s >= (uint32_t)kLds ? s - kLds : s; };
    auto k_step = [&](int t, auto buf_c) __attribute__((always_inline)) {
        constexpr int cur = decltype(buf_c)::value, nxt = cur ^ 1;
        const uint32_t st_load2 = wrap(st_load + kStage);
#pragma unroll
        for (int s = 0; s < 96; ++s) {
            const int pr = s / 32, i = (s % 32) / 8, j = s % 8;
            asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                         : "+a"(acc[i][j])
                         : "v"(pr == 1 ? lo[cur][j] : hi[cur][j]), "v"(pr == 2 ? lo[cur][8 + i] : hi[cur][8 + i]));
            if (s == kBar) {
                KR_SCHED_FENCE();
                __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm(kLoads));
                __builtin_amdgcn_s_barrier();
            }
            if (s > kBar) {
                const int u = s - kBar - 1;
                if (u % kReadGap == 0 && u / kReadGap < 12) read_frag(u / kReadGap, st_next);
                if (u % kLoadGap == 0 && u / kLoadGap < 2 * kLoads)
                    issue_load(2 * t + kRing + u / kLoadGap / kLoads, u / kLoadGap < kLoads ? st_load : st_load2, u / kLoadGap % kLoads);
            }
            if (s >= kConv0 && s - kConv0 < 48) split2(nxt, (s - kConv0) / 4, (s - kConv0) % 4);
            KR_SCHED_FENCE();
        }
        st_load = wrap(st_load + 2 * kStage);
        st_next = wrap(st_next + 2 * kStage);
    };
    int t = 0;
#pragma nounroll
    for (; t + 2 <= kt_total; t += 2) {
        k_step(t, std::integral_constant<int, 0>{});
        k_step(t + 1, std::integral_constant<int, 1>{});
    }
    pin();
    if (t < kt_total) k_step(t, std::integral_constant<int, 0>{});
    __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm(0));
    __syncthreads();
    pin();

    // ---- sum of the two halves of the k: a wave keeps its first two block rows and hands over the others ------
    const uint32_t mine = (uint32_t)(wave * 16384 + lane * 16), other = (uint32_t)((wave ^ 1) * 16384 + lane * 16);
    f32x4 sum[2][8];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) *(lds_f32x4)(size_t)(mine + (i * 8 + j) * 1024) = acc[2 + i][j];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const f32x4 x = *(lds_f32x4)(size_t)(other + (i * 8 + j) * 1024);
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[i][j][e] = acc[i][j][e] + x[e];
        }
    __syncthreads();
    gemm_epilogue<BT, 32, BT, 1, 4, EVEN, kEpWave>(g, g.n_peers, g.bias, sum, smem, m0, n0, 2 * mh + kh, 0, lane, wave);
}
#undef KR_SCHED_FENCE

}  // namespace

hipError_t launch_gemm_f32(const GemmArgs& g, bool b_nt, hipStream_t st) {
    const bool even = g.M % BT == 0 && g.N % BT == 0 && g.K % (2 * BKS) == 0;
    const dim3 grid((unsigned)(g.tiles_m * g.tiles_n), (unsigned)g.k_splits), block(kWaves * 64);
    static std::atomic<uint64_t> opted[4];
#define KR_LAUNCH(NT, EV)                                                                                               \
    do {                                                                                                                \
        if (hipError_t e = lds_opt_in((const void*)gemm_f32_kernel<NT, EV>, kLds, opted[2 * NT + EV]); e != hipSuccess) \
            return e;                                                                                                   \
        hipLaunchKernelGGL((gemm_f32_kernel<NT, EV>), grid, block, kLds, st, g);                                        \
    } while (0)
    if (b_nt) {
        if (even) KR_LAUNCH(true, true); else KR_LAUNCH(true, false);
    } else {
        if (even) KR_LAUNCH(false, true); else KR_LAUNCH(false, false);
    }
#undef KR_LAUNCH
    return hipGetLastError();
}

}  // namespace kr

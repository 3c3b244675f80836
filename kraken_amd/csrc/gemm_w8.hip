// Product of fp8 (e4m3fn) operands whose sums keep all 24 bits: the operands stay fp8 in memory and in LDS and are widened
// to bf16 (exactly) in registers, between LDS and the bf16 matrix cores.  The fp8 matrix-core instruction keeps about 16
// bits of a sum, so shapes that promise 24 used to take two conversion passes, a bf16 product with an fp32 result
// and a third pass: 4000 x 6656 x 4096 in 257 us, now 139 (135 to 146 on different cards); 64 x 8192 x 8192 96 -> 37; 700 x 7168 x 8192 164 -> 78.
//
// Bound by the bf16 matrix cores.  Tile, waves, LDS stages and loads are those of the 256x256 kernel (gemm_dtl.hip):
// 256 rows, four wavefronts of 128 x 16 NB, rows of 128 bytes per stage -- 128 k here, so a stage lasts four sub-steps of
// 32 k instead of two, and half the bytes per flop come through LDS and L2.  What is added is one
// v_cvt_scalef32_pk_bf16_fp8 (two values) per matrix-core instruction of 16 cycles.
//
// A 16-byte LDS read gives a lane 16 k of a row: its low eight k are the operand of one sub-step, the high eight that of
// the next (both operands take their k in this same order, which is all a sum needs).  Sub-steps alternate between two
// sets of widened fragments; while one runs, the other set is formed from the raw fragments, and as soon as a raw fragment
// has given both its halves it is read again from LDS for the next 64 k.
//
// Tiles of two widths in one launch: the first columns as 256-column tiles in whole rounds of the 256 compute units, the rest
// as narrower ones (plan_w8 in gemm.hip) that divide what is left evenly.
#include "gemm_common.h"

namespace kr {

namespace {

constexpr int BM = 256, kWaves = 4;
constexpr int kRowB = 128;                     // bytes (= k) of a row in a stage
constexpr int A_ST = BM * kRowB;               // 32 KiB
constexpr uint32_t B_BASE = 2 * A_ST;          // two stages of A, then two of B
constexpr int B_ST = 256 * kRowB;
constexpr int kLds = 2 * (A_ST + B_ST);
constexpr int NA = 8;                          // 16-row blocks of a wave
constexpr int LOADS_A = A_ST / 1024 / kWaves;  // LDS-DMA loads (1 KiB) per wave and step

typedef const __attribute__((address_space(3))) i32x4* lds_raw;

constexpr int vmcnt_imm(int n) { return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14); }
constexpr int kLgkm0 = 0xc07f;

// two fp8 of a word (its low or high half) as two bf16, exactly
template <bool HIGH_HALF>
__device__ __forceinline__ uint32_t widen2(int w) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, HIGH_HALF));
}

// One tile: rows tile_m * 256, columns n0 .. n0 + 32 NB - 1.  PART: k-steps kt_begin .. kt_begin + kt_total - 1 only, the
// accumulators go to `part` in register order (gemm_dtl_tail_finish_kernel sums and rounds them).
template <int NB, bool PART>
__device__ __forceinline__ void w8_tile(const GemmArgs& g, unsigned char* smem, int tile_m, int n0, int kt_begin, int kt_total, f32x4* part) {
    constexpr int LOADS_B = NB, LOADS = LOADS_A + LOADS_B;
    constexpr int NF = NB + NA;                // fragments: B blocks, then A blocks
    constexpr int NM = NA * NB;                // MFMAs of a sub-step
    // (nothing is outstanding at entry; see gemm_dtl_tile)
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = tile_m * BM;
    // operands in units of two bytes: g.K, g.lda and g.ldb are halved
    const int kt_all = (g.K + kRowB / 2 - 1) / (kRowB / 2);
    const int k_begin = kt_begin * (kRowB / 2);
    const uint16_t* a_tile;
    int64_t lda;
    gathered_a_tile(g, m0, BM, a_tile, lda);
    a_tile = (const uint16_t*)wave_uniform((int64_t)a_tile) + k_begin;
    lda = wave_uniform(lda);

    // ---- LDS-DMA addressing (as in gemm_dtl_tile) ---------------------------------------------
    const int sw = (4 * (wave & 1) + (lane >> 4)) & 7;
    const int piece = (lane & 7) ^ sw;
    const uint32_t a_voff = (uint32_t)(((int64_t)(lane >> 3) * lda + piece * 8) * 2);
    const uint32_t b_voff = (uint32_t)(((int64_t)(lane >> 3) * g.ldb + piece * 8) * 2);
    // pieces past K of a last k-step that is not full are requested out of range, which writes zeros
    const bool in_k = (kt_all - 1) * (kRowB / 2) + piece * 8 < g.K;
    const uint32_t a_tail = in_k ? a_voff : 0x80000000u, b_tail = in_k ? b_voff : 0x80000000u;
    const int t_tail = kt_all - 1 - kt_begin;
    // rows past M and columns past N are out of range as well
    const int rows_a = min(BM, g.M - m0), rows_b = min(32 * NB, g.N - n0);
    const i32x4 a_rsrc = raw_rsrc(a_tile, ((int64_t)(rows_a - 1) * lda + (g.K - k_begin)) * 2);
    const i32x4 b_rsrc = raw_rsrc(g.B + (int64_t)n0 * g.ldb + k_begin, ((int64_t)(rows_b - 1) * g.ldb + (g.K - k_begin)) * 2);
    auto issue_load = [&](int t, uint32_t stage, int q) __attribute__((always_inline)) {
        // (past the end the count per step must not change: all lanes re-read the first 16 bytes of the last step)
        const bool live = t < kt_total, tail = t == t_tail;
        const int k0 = min(t, kt_total - 1) * (kRowB / 2);
        if (q < LOADS_A) {
            const int ch = wave + 4 * q;
            lds_dma_b128(a_rsrc, stage * A_ST + ch * 1024, !live ? 0u : tail ? a_tail : a_voff, (int)(((int64_t)8 * ch * lda + k0) * 2));
        } else {
            const int ch = wave + 4 * (q - LOADS_A);
            lds_dma_b128(b_rsrc, B_BASE + stage * B_ST + ch * 1024, !live ? 0u : tail ? b_tail : b_voff, (int)(((int64_t)8 * ch * g.ldb + k0) * 2));
        }
    };

    // ---- fragments ----------------------------------------------------------------------------
    // lane -> row lane%16 of a 16-row block, the 16 k of piece 4h + lane/16 (h: half of the stage's 128 k)
    const int p = lane & 15, gq = lane >> 4;
    uint32_t fa[2], fb[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t pc = (uint32_t)(((4 * h + gq) ^ ((p >> 1) & 7)) << 4);
        fa[h] = (uint32_t)((wm * 128 + p) * kRowB) + pc;
        fb[h] = B_BASE + (uint32_t)((wn * 16 * NB + p) * kRowB) + pc;
    }
    i32x4 raw[NF];
    u32x4 frag[2][NF];
    auto read_raw = [&](int r, int h, uint32_t stage) __attribute__((always_inline)) {
        const uint32_t a = r < NB ? fb[h] + stage * B_ST + r * 2048 : fa[h] + stage * A_ST + (r - NB) * 2048;
        raw[r] = *(lds_raw)(size_t)a;
    };
    // conversion c of a set: word c % 4 of fragment c / 4, from half `half` of its raw fragment
    auto widen = [&](auto half_c, int c) __attribute__((always_inline)) {
        constexpr int half = decltype(half_c)::value;
        const int r = c / 4, w = c % 4;
        const int src = raw[r][2 * half + w / 2];
        frag[half][r][w] = (w & 1) ? widen2<true>(src) : widen2<false>(src);
    };
    f32x4 acc[NA][NB];
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto pin = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NA; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) asm volatile("" : "+a"(acc[i][j]));
    };
    pin();
#define KR_SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)

    // ---- k loop ---------------------------------------------------------------------------------
    // Sub-steps of a step (128 k): s = 0, 1 multiply the low and high halves of the stage's first 64 k, s = 2, 3 those of the
    // second.  Even sub-steps form the high halves and read the raw fragments of the next 64 k behind them; odd ones form
    // the low halves of those.  All LDS reads of a stage have been issued by the end of sub-step 0: barrier (a) behind
    // slot kBarA of sub-step 1 frees the stage for the loads of step t+2, kGap slots apart through the rest of the step;
    // barrier (b) in front of sub-step 2 waits for the loads of step t+1.
    constexpr int kBarA = 10;
    constexpr int kLoad0 = NM + kBarA + 1;                            // slot of the step's first load
    constexpr int kGap = (4 * NM - 1 - kLoad0) / (LOADS - 1);
    constexpr int kBeforeB = (2 * NM - 1 - kLoad0) / kGap + 1;        // loads in slots < 2 NM
    static_assert(kGap >= 4 && kLoad0 + kGap * (LOADS - 1) < 4 * NM && kBeforeB < LOADS, "step schedule");
    constexpr int NC = 4 * NF;                                         // conversions of a sub-step
#pragma unroll
    for (int q = 0; q < LOADS; ++q) issue_load(0, 0, q);
#pragma unroll
    for (int q = 0; q < LOADS; ++q) issue_load(1, 1, q);
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(LOADS));
    __builtin_amdgcn_s_barrier();
    KR_SCHED_FENCE();
#pragma unroll
    for (int r = 0; r < NF; ++r) read_raw(r, 0, 0);
#pragma unroll
    for (int c = 0; c < NC; ++c) widen(std::integral_constant<int, 0>{}, c);
    KR_SCHED_FENCE();
    auto k_step = [&](int t, auto stage_c) __attribute__((always_inline)) {
        constexpr uint32_t cur = decltype(stage_c)::value, nxt = cur ^ 1u;
#pragma unroll
        for (int u = 0; u < 4 * NM; ++u) {
            const int s = u / NM, v = u % NM;        // sub-step, slot in it
            const int i = v / NB, j = v % NB;
            if (u == 2 * NM) {
                __builtin_amdgcn_s_waitcnt(vmcnt_imm(kBeforeB));
                __builtin_amdgcn_s_barrier();
                KR_SCHED_FENCE();
            }
            // (the accumulator tied to its AGPRs, as in gemm_dtl_tile's k_step16)
            asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(frag[s & 1][j]), "v"(frag[s & 1][NB + i]));
#pragma unroll
            for (int c = v * NC / NM; c < (v + 1) * NC / NM; ++c) {
                if (s & 1) {
                    widen(std::integral_constant<int, 0>{}, c);
                } else {
                    widen(std::integral_constant<int, 1>{}, c);
                    if (c % 4 == 3) read_raw(c / 4, s == 0 ? 1 : 0, s == 0 ? cur : nxt);
                }
            }
            if (u == NM + kBarA) {
                KR_SCHED_FENCE();
                __builtin_amdgcn_s_waitcnt(kLgkm0);
                __builtin_amdgcn_s_barrier();
            }
            if (u >= kLoad0 && (u - kLoad0) % kGap == 0 && (u - kLoad0) / kGap < LOADS) issue_load(t + 2, cur, (u - kLoad0) / kGap);
            KR_SCHED_FENCE();
        }
    };
    int t = 0;
#pragma nounroll
    for (; t + 2 <= kt_total; t += 2) {
        k_step(t, std::integral_constant<uint32_t, 0>{});
        k_step(t + 1, std::integral_constant<uint32_t, 1>{});
    }
    pin();
    if (t < kt_total) k_step(t, std::integral_constant<uint32_t, 0>{});
    // drain the surplus loads before the LDS is reused
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    __syncthreads();
    pin();
#undef KR_SCHED_FENCE
    if constexpr (PART) {
        const int rows = n0 + wn * 16 * NB < g.N ? g.M - m0 - wm * 128 : 0;   // (blocks outside the matrix are not read either)
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            if (16 * i >= rows) break;
#pragma unroll
            for (int j = 0; j < NB; ++j) __builtin_nontemporal_store(acc[i][j], part + (i * NB + j) * (kWaves * 64) + threadIdx.x);
        }
    } else {
        const int row0 = m0 + wm * 128, col0 = n0 + wn * 16 * NB;
        uint8_t* dst = (uint8_t*)g.out + (int64_t)row0 * g.N + col0;
        store_tile_fp8_blocks<NB, true>(acc, smem, dst, g.N, lane, wave, g.M - row0, g.N - col0);
    }
}

// Tile order: the first g.wide_panels column panels as 256-column tiles, then the other columns in tiles of 32 NB2 (NB2 = 0:
// there are none).  Each region is dealt to the XCDs and walked like a launch of its own (tile_schedule).
template <int NB2>
__global__ __launch_bounds__(kWaves * 64) void gemm_w8_kernel(const GemmArgs g) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // starts at LDS address 0
    const int kt_all = (g.K + kRowB / 2 - 1) / (kRowB / 2);
    const int wide = g.tiles_m * g.wide_panels;
    int tile_m, tile_n;
    if (NB2 == 0 || (int)blockIdx.x < wide) {
        tile_in_order(xcd_position(blockIdx.x, wide), g.tiles_m, g.wide_panels, g.group_n, g.pivot_tiles, tile_m, tile_n);
        w8_tile<8, false>(g, smem, tile_m, tile_n * 256, 0, kt_all, nullptr);
    } else if constexpr (NB2 != 0) {
        const int narrow_panels = g.tiles_n - g.wide_panels;
        tile_in_order(xcd_position(blockIdx.x - wide, g.tiles_m * narrow_panels), g.tiles_m, narrow_panels, g.group_n, g.pivot_tiles, tile_m, tile_n);
        w8_tile<NB2, false>(g, smem, tile_m, g.wide_panels * 256 + tile_n * 32 * NB2, 0, kt_all, nullptr);
    }
}

// Few tiles: g.k_splits workgroups share the K loop of each (256 columns all), the accumulators go to the workspace
// (g.out) as [tile][part][quad][thread].
__global__ __launch_bounds__(kWaves * 64) void gemm_w8_part_kernel(const GemmArgs g) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int kt_all = (g.K + kRowB / 2 - 1) / (kRowB / 2);
    const int split = (int)(blockIdx.x % (unsigned)g.k_splits), index = (int)(blockIdx.x / (unsigned)g.k_splits);
    const int kt0 = (int)((int64_t)kt_all * split / g.k_splits), kt1 = (int)((int64_t)kt_all * (split + 1) / g.k_splits);
    int tile_m, tile_n;
    tile_schedule(g, schedule_position(g, index, 0), tile_m, tile_n);
    w8_tile<8, true>(g, smem, tile_m, tile_n * 256, kt0, kt1 - kt0, (f32x4*)g.out + ((int64_t)index * g.k_splits + split) * (64 * kWaves * 64));
}

}  // namespace

// g: operands in units of two bytes (K, lda, ldb halved); g.wide_panels panels of 256 columns and g.tiles_n - g.wide_panels
// of 32 nb2; with g.tail_tiles (all tiles, 256 columns) the K loops are shared and the parts meet in `workspace`.
hipError_t launch_gemm_w8(const GemmArgs& g, int nb2, hipStream_t st, void* workspace) {
    const dim3 block(kWaves * 64);
    static std::atomic<uint64_t> opted[6];
    if (g.tail_tiles > 0) {
        if (hipError_t e = lds_opt_in((const void*)gemm_w8_part_kernel, kLds, opted[5]); e != hipSuccess) return e;
        GemmArgs gs = g;
        gs.out = workspace;
        hipLaunchKernelGGL(gemm_w8_part_kernel, dim3((unsigned)(g.tail_tiles * g.k_splits)), block, kLds, st, gs);
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
        return launch_tail_finish(g, st, workspace);
    }
    const dim3 grid((unsigned)(g.tiles_m * g.tiles_n));
#define KR_LAUNCH(NB2, SLOT)                                                                                                  \
    do {                                                                                                                      \
        if (hipError_t e = lds_opt_in((const void*)gemm_w8_kernel<NB2>, kLds, opted[SLOT]); e != hipSuccess) return e;        \
        hipLaunchKernelGGL(gemm_w8_kernel<NB2>, grid, block, kLds, st, g);                                                    \
    } while (0)
    switch (nb2) {
        case 0: KR_LAUNCH(0, 0); break;
        case 4: KR_LAUNCH(4, 1); break;
        case 5: KR_LAUNCH(5, 2); break;
        case 6: KR_LAUNCH(6, 3); break;
        case 7: KR_LAUNCH(7, 4); break;
        default: return hipErrorInvalidValue;
    }
#undef KR_LAUNCH
    return hipGetLastError();
}

}  // namespace kr

// bf16 GEMM for shapes with few output tiles: 128x128 tiles, a deep ring of LDS stages, and the k of a stage
// divided between two wavefronts.
//
// With a few hundred tiles of 128 x 128 there is one workgroup per compute unit, so nothing hides what its own
// pipeline does not.  Two things bound it.  (1) The LDS: with the usual 2 x 2 arrangement (64 x 64 of C per
// wavefront) a k-step of 64 reads 64 KiB of fragments and writes 32 KiB of operands, 768 cycles for 512 cycles
// of MFMAs.  Here a wavefront owns 64 x 128 of C for half of the k (fragments 48 KiB, 640 cycles), and pairs of
// wavefronts add their halves through LDS once at the end (64 KiB).  (2) The latency of the operands: every
// line comes from the last-level cache or HBM once per XCD, and all its workgroups wait for it together.  Five
// stages of 64 k (160 KiB, the whole LDS) keep the loads of four steps in flight.
//
// Stage: A and transposed-contiguous B as rows of 128 bytes (64 k), the eight 16-byte pieces XOR-swizzled with
// (row >> 1) & 7 as in the 256x256 kernel (gemm_dtl.hip); row-major B as k-rows of 256 bytes, pieces swizzled
// with the k-row so that a transposing read touches all banks once.  The fragments of step t+1 are read into a
// second set of registers during step t.
#include "gemm_common.h"

namespace kr {

namespace {

constexpr int BT = 128;                        // tile rows and columns
constexpr int BKS = 64;                        // k of a stage
constexpr int kOper = BT * BKS * 2;            // bytes of one operand in a stage: 16 KiB
constexpr int kStage = 2 * kOper;              // A, then B
constexpr int kRing = 5;                       // stages
constexpr int kLds = kRing * kStage;           // 160 KiB
constexpr int kWaves = 4;
constexpr int kLoadsA = kOper / 1024 / kWaves;       // LDS-DMA loads (1 KiB) of A per wave and step: 4, and 4 of B
constexpr int kLoads = 2 * kLoadsA;
constexpr int kEpWave = 32 * (BT + 4) * 4;
static_assert(kEpWave * kWaves <= kLds, "epilogue patch must fit in the stages");

// schedule of a step's 32 MFMA slots (see k_step below)
constexpr int kBar = 6, kLoadGap = 3;
static_assert(kBar + 1 + kLoadGap * (kLoads - 1) < 32 && kBar + 12 < 32, "step schedule");

typedef const __attribute__((address_space(3))) bf16x8* lds_frag;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4* lds_tr;
typedef __attribute__((address_space(3))) f32x4* lds_f32x4;

constexpr int vmcnt_lgkm0_imm(int n) { return (n & 15) | (7 << 4) | (0 << 8) | ((n >> 4) << 14); }

// EVEN: M and N are multiples of 128, K of 64.
template <bool B_NT, bool EVEN>
__global__ __launch_bounds__(kWaves * 64) void gemm_ks_kernel(const GemmArgs g) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // starts at LDS address 0
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int mh = wave >> 1, kh = wave & 1;   // rows 64 mh .. +63 of the tile, k 32 kh .. +31 of a stage
    int tile_m, tile_n;
    // (no band region here, and 0.2 us less than tile_of: 256 x 4096 x 2048 with one peer 23.4 / 23.2 us, 512 x 5120 x 1536 19.0 / 18.8)
    tile_schedule(g, schedule_position(g, blockIdx.x), tile_m, tile_n);
    const int m0 = tile_m * BT, n0 = tile_n * BT;
    // k-steps of this workgroup: all of them, or the share of split blockIdx.y
    const int kt_all = (g.K + BKS - 1) / BKS;
    const int kt_begin = g.k_splits > 1 ? (int)((int64_t)kt_all * blockIdx.y / g.k_splits) : 0;
    const int kt_total = g.k_splits > 1 ? (int)((int64_t)kt_all * (blockIdx.y + 1) / g.k_splits) - kt_begin : kt_all;
    const int k_begin = kt_begin * BKS;
    const uint16_t* a_tile;
    int64_t lda;
    gathered_a_tile(g, m0, BT, a_tile, lda);
    a_tile = (const uint16_t*)wave_uniform((int64_t)a_tile) + k_begin;
    lda = wave_uniform(lda);

    // ---- LDS-DMA addressing -------------------------------------------------------------------
    // A (and transposed B): a load fills 8 rows: lane l -> row l/8, slot l%8 holds piece
    // slot ^ ((row >> 1) & 7); wave w takes the row groups w, w+4, w+8, w+12, whose parity is the wave's, so
    // the lane part of the address is computed once.
    const int sw = (4 * (wave & 1) + (lane >> 4)) & 7;
    const int piece = (lane & 7) ^ sw;
    const uint32_t a_voff = (uint32_t)(((int64_t)(lane >> 3) * lda + piece * 8) * 2);
    uint32_t b_voff;
    if (B_NT) {
        b_voff = (uint32_t)(((int64_t)(lane >> 3) * g.ldb + piece * 8) * 2);
    } else {
        // row-major B: a load fills 4 k-rows of 256 bytes: lane l -> k-row l/16, slot l%16 holds piece
        // slot ^ 2*((k & 3) + 4*((k >> 3) & 1)); wave w takes the groups w, w+4, ... of the stage's 16
        b_voff = (uint32_t)(((int64_t)(lane >> 4) * g.ldb + (((lane & 15) ^ (2 * ((lane >> 4) + 4 * ((wave >> 1) & 1)))) << 3)) * 2);
    }
    // A last k-step that is not full: pieces at or past K are requested out of range, which writes zeros
    // (row-major B: its k-rows past K lie past the matrix' end).
    const int t_tail = kt_all - 1 - kt_begin;
    constexpr uint32_t kOob = 0x80000000u;
    const bool in_k = EVEN || (kt_all - 1) * BKS + piece * 8 < g.K;
    const uint32_t a_tail = in_k ? a_voff : kOob, b_tail = in_k ? b_voff : kOob;
    const int rows_a = EVEN ? BT : min(BT, g.M - m0), rows_b = EVEN ? BT : min(BT, g.N - n0);
    const i32x4 a_rsrc = raw_rsrc(a_tile, EVEN ? (int64_t)0x7fffffff : ((int64_t)(rows_a - 1) * lda + (g.K - k_begin)) * 2);
    const i32x4 bt_rsrc = raw_rsrc(g.B + (int64_t)n0 * g.ldb + k_begin,
                                   EVEN ? (int64_t)0x7fffffff : ((int64_t)(rows_b - 1) * g.ldb + (g.K - k_begin)) * 2);
    // load q of step t into the stage at LDS offset `stage`; past the last step nothing is needed, but the count
    // per step must not change (the waits below count loads), so all lanes re-read the first 16 bytes of the last one
    auto issue_load = [&](int t, uint32_t stage, int q) __attribute__((always_inline)) {
        const bool live = t < kt_total;
        const int tt = min(t, kt_total - 1), k0 = tt * BKS;
        const bool tail = !EVEN && tt == t_tail;
        const int rg = wave + 4 * (q % kLoadsA);
        if (q < kLoadsA) {
            lds_dma_b128(a_rsrc, stage + rg * 1024, !live ? 0u : tail ? a_tail : a_voff, (int)(((int64_t)8 * rg * lda + k0) * 2));
        } else if (B_NT) {
            lds_dma_b128(bt_rsrc, stage + kOper + rg * 1024, !live ? 0u : tail ? b_tail : b_voff, (int)(((int64_t)8 * rg * g.ldb + k0) * 2));
        } else {
            const int64_t kb = k_begin + k0;
            lds_dma_b128(raw_rsrc(g.B + kb * g.ldb + n0, EVEN ? (int64_t)0x7fffffff : ((g.K - 1 - kb) * g.ldb + (g.N - n0)) * 2),
                         stage + kOper + rg * 1024, live ? b_voff : 0u, (int)((int64_t)4 * rg * g.ldb * 2));
        }
    };

    // ---- fragment addressing ----------------------------------------------------------------------
    // lane -> row p = lane%16 of a 16-row block, 8 k at piece 4 kh + lane/16 of the row.  A's four blocks are taken
    // in the order 0 1 2 3 by the first wave of a pair and 2 3 0 1 by the second: each then keeps the sums of
    // its first two and hands over the other two.
    const int p = lane & 15, gq = lane >> 4;
    const uint32_t fl = (uint32_t)(p * 128 + (((4 * kh + gq) ^ ((p >> 1) & 7)) << 4));
    const uint32_t fa0 = fl + (uint32_t)(mh * 64 * 128 + kh * 32 * 128), fa1 = fl + (uint32_t)(mh * 64 * 128 + (kh ^ 1) * 32 * 128);
    uint32_t fb[B_NT ? 1 : 8];
    if (B_NT) {
        fb[0] = kOper + fl;
    } else {
        // transposing reads: group gq reads k-rows 32 kh + 8 gq + p/4 (and 4 further on), columns 16j + 4(p%4) .. +3
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int pc = (2 * j + ((p & 3) >> 1)) ^ (2 * ((p >> 2) + 4 * (gq & 1)));
            fb[j] = kOper + (uint32_t)((32 * kh + 8 * gq + (p >> 2)) * 256 + pc * 16 + (p & 1) * 8);
        }
    }
    bf16x8 af[2][4], bf[2][8];
    // fragment r of a step in the order its MFMAs need them: A block 0, all of B, the other A blocks
    auto read_frag = [&](int buf, int r, uint32_t stage) __attribute__((always_inline)) {
        if (r == 0 || r > 8) {
            const int i = r == 0 ? 0 : r - 8;
            af[buf][i] = *(lds_frag)(size_t)((i < 2 ? fa0 : fa1) + stage + (i & 1) * 2048);
        } else if (B_NT) {
            bf[buf][r - 1] = *(lds_frag)(size_t)(fb[0] + stage + (r - 1) * 2048);
        } else {
            const uint32_t a = fb[B_NT ? 0 : r - 1] + stage;
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(size_t)a);
            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(size_t)(a + 1024));
            bf[buf][r - 1] = __builtin_bit_cast(bf16x8, (s16x8){lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w});
        }
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
    // stages 0 .. 3 are requested before the loop; wait for stage 0
#pragma unroll
    for (int st = 0; st < kRing - 1; ++st)
#pragma unroll
        for (int q = 0; q < kLoads; ++q) issue_load(st, st * kStage, q);
    __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm((kRing - 2) * kLoads));
    __builtin_amdgcn_s_barrier();
    KR_SCHED_FENCE();
#pragma unroll
    for (int r = 0; r < 12; ++r) read_frag(0, r, 0);

    // ---- k loop ------------------------------------------------------------------------------------
    // Step t: 32 MFMAs on the fragments read during step t-1.  Behind slot kBar the wave waits for its fragment
    // reads of step t and its loads of step t+1 (those of t+2 and t+3 stay outstanding) and meets the others:
    // stage t+1 is then complete, and its fragments are read, one per slot; stage t is free in every wave, and
    // the loads of step t+4, which take the slot of stage t-1, go out one per kLoadGap slots.
    uint32_t st_next = kStage, st_load = (kRing - 1) * kStage;   // LDS offsets of stages t+1 and t+4
    auto k_step = [&](int t, auto buf_c) __attribute__((always_inline)) {
        constexpr int cur = decltype(buf_c)::value, nxt = cur ^ 1;
#pragma unroll
        for (int s = 0; s < 32; ++s) {
            const int i = s / 8, j = s % 8;
            asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(bf[cur][j]), "v"(af[cur][i]));
            if (s == kBar) {
                KR_SCHED_FENCE();
                __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm((kRing - 3) * kLoads));
                __builtin_amdgcn_s_barrier();
            }
            if (s > kBar) {
                const int u = s - kBar - 1;
                if (u < 12) read_frag(nxt, u, st_next);
                if (u % kLoadGap == 0 && u / kLoadGap < kLoads) issue_load(t + kRing - 1, st_load, u / kLoadGap);
            }
            KR_SCHED_FENCE();
        }
        st_load = st_load == (kRing - 1) * kStage ? 0u : st_load + kStage;
        st_next = st_next == (kRing - 1) * kStage ? 0u : st_next + kStage;
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

// Loads the file's device code for the current device (code objects are loaded on first use, which moves
// device memory).
hipError_t load_gemm_ks() {
    hipFuncAttributes a;
    return hipFuncGetAttributes(&a, (const void*)gemm_ks_kernel<true, true>);
}

hipError_t launch_gemm_ks(const GemmArgs& g, bool b_nt, hipStream_t st) {
    const bool even = g.M % BT == 0 && g.N % BT == 0 && g.K % BKS == 0;
    const dim3 grid((unsigned)(g.tiles_m * g.tiles_n), (unsigned)g.k_splits), block(kWaves * 64);
    static std::atomic<uint64_t> opted[4];
#define KR_LAUNCH(NT, EV)                                                                                              \
    do {                                                                                                               \
        if (hipError_t e = lds_opt_in((const void*)gemm_ks_kernel<NT, EV>, kLds, opted[2 * NT + EV]); e != hipSuccess) \
            return e;                                                                                                  \
        hipLaunchKernelGGL((gemm_ks_kernel<NT, EV>), grid, block, kLds, st, g);                                        \
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

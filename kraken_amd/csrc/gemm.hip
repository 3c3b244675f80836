// bf16 GEMM on the gfx950 matrix cores with a fused reduce(+bias) epilogue.
//
//   C = A[M,K] @ B[K,N]                      (fp32 accumulate, v_mfma_f32_32x32x16_bf16)
//   out  = C[band] + sum_j peers[j] + bias   (rows of the band; one store, no C round trip)
//   c_full[rows outside the band] = bf16(C)
//
// Workgroup tile BM x BN x 64, WM x WN wavefronts, each owning a
// (BM/WM) x (BN/WN) block of C as 32x32 MFMA accumulators.  A and B tiles are
// staged in LDS as [row][64 k] bf16 (128-byte rows) with the 16-byte chunks of
// a row XOR-swizzled by the row index, so that the 128-bit fragment reads of 8
// consecutive rows land in 8 different bank groups.  Two LDS stages: the
// global loads of k-step t+1 are issued before the MFMAs of step t and written
// to the other stage afterwards (one workgroup barrier per k-step).
// Row-major B ([K,N], N contiguous) is transposed on its way into LDS: a
// thread loads an 8(k) x 8(n) block with eight 128-bit loads, transposes it in
// registers with byte permutes and writes eight 128-bit [n][8 k] chunks.
// Epilogue (shared with the LDS-DMA kernel for 256x256 tiles): accumulators go
// through a per-wave LDS patch to turn the MFMA layout into row-contiguous
// 8-element vectors, so peers, bias and output are all moved with 128-bit
// accesses covering whole row segments.  This file also holds the C entry point
// and the choice between the two kernels.
#include <stdlib.h>

#include <type_traits>

#include <algorithm>
#include <cmath>
#include <mutex>

#include "gemm_common.h"

namespace kr {


constexpr int BK = 64;            // k extent of one LDS stage
constexpr int kRowBytes = BK * 2; // 128-byte LDS rows

// 16-byte chunk swizzle inside a 128-byte LDS row
__device__ __forceinline__ int swz(int row, int chunk) { return chunk ^ ((row ^ (row >> 3)) & 7); }

__device__ __forceinline__ uint32_t perm_lo(uint32_t hi_src, uint32_t lo_src) {
    // {lo16(hi_src), lo16(lo_src)}
    return __builtin_amdgcn_perm(hi_src, lo_src, 0x05040100u);
}
__device__ __forceinline__ uint32_t perm_hi(uint32_t hi_src, uint32_t lo_src) {
    // {hi16(hi_src), hi16(lo_src)}
    return __builtin_amdgcn_perm(hi_src, lo_src, 0x07060302u);
}

template <int BM, int BN, int WM, int WN, bool B_NT, bool EVEN>
__global__ __launch_bounds__(WM* WN * 64) void gemm_reduce_kernel(const GemmArgs g) {
    constexpr int T = WM * WN * 64;
    constexpr int WTM = BM / WM, WTN = BN / WN;   // wave tile
    constexpr int TM = WTM / 32, TN = WTN / 32;   // 32x32 MFMA blocks per wave
    constexpr int A_STAGE = BM * kRowBytes, B_STAGE = BN * kRowBytes;
    constexpr int STAGE = A_STAGE + B_STAGE;
    constexpr int A_ITERS = BM * 8 / T;           // 16-byte chunks per thread per stage
    constexpr int B_ITERS_NT = BN * 8 / T;
    constexpr int B_BLOCKS = BN / T > 0 ? BN / T : 1;  // NN: 8x8 blocks per thread per stage
    static_assert(BM % (WM * 32) == 0 && BN % (WN * 32) == 0, "wave tile must be a multiple of 32");
    static_assert((BM * 8) % T == 0 && (BN * 8) % T == 0 && (BN % T == 0 || BN < T), "load split");
    // epilogue patch: 32 rows x WTN fp32 per wave, rows padded by 4 floats
    constexpr int EP_WAVE = 32 * (WTN + 4) * 4;
    static_assert(EP_WAVE * WM * WN <= 2 * STAGE, "epilogue patch must fit in the pipeline LDS");

    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;

    int tile_m, tile_n;
    tile_of(g, blockIdx.x, 0, tile_m, tile_n);
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const uint16_t* a_tile;   // first row of the tile's A panel (gathered matrix or local shard)
    int64_t lda;
    gathered_a_tile(g, m0, BM, a_tile, lda);
    // k range of this workgroup: all of K, or with a split K loop (g.k_splits > 1, split index
    // in blockIdx.y) the split's share of the k-steps; k_begin enters every operand offset
    const int kt_all = (g.K + BK - 1) / BK;
    const int kt_begin = g.k_splits > 1 ? (int)((int64_t)kt_all * blockIdx.y / g.k_splits) : 0;
    const int kt_total = g.k_splits > 1 ? (int)((int64_t)kt_all * (blockIdx.y + 1) / g.k_splits) - kt_begin : kt_all;
    const int k_begin = kt_begin * BK;

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    // ---- operand staging: global -> registers -> LDS, one 16-byte chunk per "unit" ------
    // Global loads are buffer loads: a wave-uniform resource descriptor (tile base), a
    // per-thread 32-bit byte offset that never changes, and a wave-uniform scalar offset that
    // advances with k.  No per-load address arithmetic is left in the main loop.
    constexpr int NB_LD = B_NT ? B_ITERS_NT : B_BLOCKS * 8;   // 128-bit global loads of B per thread per stage
    constexpr int NB_ST = B_NT ? B_ITERS_NT : B_BLOCKS * 4;   // B store units per thread per stage
    constexpr uint32_t kOob = 0x80000000u;                     // offset beyond num_records: the load returns 0
    // two register sets: set (t & 1) holds tile t+1 during iteration t and is re-filled with
    // tile t+3, so a global load has two iterations to land
    u32x4 a_reg[2][A_ITERS];
    u32x4 b_reg[2][NB_LD];
    uint32_t a_goff[A_ITERS], a_loff[A_ITERS];
    uint32_t b_goff[B_NT ? B_ITERS_NT : B_BLOCKS], b_loff[B_NT ? B_ITERS_NT : B_BLOCKS];
    const int ld_kc = tid & 7;        // 16-byte chunk inside a 128-byte k-row (T % 8 == 0)
    bool nn_active = true;            // NN: this thread owns an 8x8 block of the B stage
#pragma unroll
    for (int i = 0; i < A_ITERS; ++i) {
        const int row = (i * T + tid) >> 3;
        int m = m0 + row;
        if (!EVEN) m = min(m, g.M - 1);
        a_goff[i] = (uint32_t)(((int64_t)(m - m0) * lda + ld_kc * 8) * 2);
        a_loff[i] = row * kRowBytes + swz(row, ld_kc) * 16;
    }
    if (B_NT) {
#pragma unroll
        for (int i = 0; i < B_ITERS_NT; ++i) {
            const int row = (i * T + tid) >> 3;
            int n = n0 + row;
            if (!EVEN) n = min(n, g.N - 1);
            b_goff[i] = (uint32_t)(((int64_t)(n - n0) * g.ldb + ld_kc * 8) * 2);
            b_loff[i] = A_STAGE + row * kRowBytes + swz(row, ld_kc) * 16;
        }
    } else {
#pragma unroll
        for (int i = 0; i < B_BLOCKS; ++i) {
            const int blk = i * T + tid;
            const int nc = blk % (BN / 8), kg = blk / (BN / 8);
            if (BN < T && kg >= 8) nn_active = false;     // more threads than 8x8 blocks
            int n = n0 + nc * 8;
            if (!EVEN) n = min(n, g.N - 8);
            b_goff[i] = (uint32_t)(((int64_t)(kg & 7) * 8 * g.ldb + (n - n0)) * 2);
            b_loff[i] = (uint32_t)(nc | ((kg & 7) << 16));   // packed (nc, kg); expanded at the store
        }
    }
    // descriptors: 48-bit base, stride 0 (raw), num_records 2^31-1 bytes, 32-bit data format.
    // Rows are clamped into the matrix above, so only the K tail needs the out-of-range path.
    const __amdgpu_buffer_rsrc_t a_rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void*)a_tile, 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t bt_rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void*)(g.B + (int64_t)n0 * g.ldb), 0, 0x7fffffff, 0x00020000);

    auto load_a_unit = [&](int rs, int i, int k_rel) {
        const int k0 = k_begin + k_rel;
        uint32_t off = a_goff[i];
        if (!EVEN && k0 + ld_kc * 8 >= g.K) off = kOob;
        a_reg[rs][i] = __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, off, k0 * 2, 0);
    };
    auto load_b_unit = [&](int rs, int u, int k_rel) {
        const int k0 = k_begin + k_rel;
        if (B_NT) {
            uint32_t off = b_goff[u];
            if (!EVEN && k0 + ld_kc * 8 >= g.K) off = kOob;
            b_reg[rs][u] = __builtin_amdgcn_raw_buffer_load_b128(bt_rsrc, off, k0 * 2, 0);
        } else {
            const int i = u >> 3, j = u & 7;             // block i, k-row j of the 8x8 block
            if (!nn_active) return;
            // re-based on the k-row so that the scalar offset stays small for any matrix size
            const __amdgpu_buffer_rsrc_t brs = __builtin_amdgcn_make_buffer_rsrc(
                (void*)(g.B + (int64_t)(k0 + j) * g.ldb + n0), 0, 0x7fffffff, 0x00020000);
            uint32_t off = b_goff[i];
            if (!EVEN && k0 + (int)(b_loff[i] >> 16) * 8 + j >= g.K) off = kOob;
            b_reg[rs][u] = __builtin_amdgcn_raw_buffer_load_b128(brs, off, 0, 0);
        }
    };
    // LDS is addressed by raw byte offsets: this kernel declares no static LDS, so its dynamic
    // array starts at LDS address 0.  Offsets are relative to stage 0; `st` (0 or STAGE, a power
    // of two above every in-stage offset) selects the stage by XOR.
    typedef __attribute__((address_space(3))) u32x4* lds_u32x4;
    typedef const __attribute__((address_space(3))) bf16x8* lds_frag;
    auto store_a_unit = [&](int rs, int i, uint32_t st) { *(lds_u32x4)(size_t)(a_loff[i] ^ st) = a_reg[rs][i]; };
    auto store_b_unit = [&](int rs, int u, uint32_t st) {
        if (B_NT) {
            *(lds_u32x4)(size_t)(b_loff[u] ^ st) = b_reg[rs][u];
        } else {
            // unit u = (block i, word q): columns 2q and 2q+1 of the 8x8 block, all 8 k
            const int i = u >> 2, q = u & 3;
            if (!nn_active) return;
            const int nc = (int)(b_loff[i] & 0xffff), kg = (int)(b_loff[i] >> 16);
            u32x4 even, odd;               // [n = 2q][k 0..7], [n = 2q+1][k 0..7]
            even.x = perm_lo(b_reg[rs][i * 8 + 1][q], b_reg[rs][i * 8 + 0][q]);
            even.y = perm_lo(b_reg[rs][i * 8 + 3][q], b_reg[rs][i * 8 + 2][q]);
            even.z = perm_lo(b_reg[rs][i * 8 + 5][q], b_reg[rs][i * 8 + 4][q]);
            even.w = perm_lo(b_reg[rs][i * 8 + 7][q], b_reg[rs][i * 8 + 6][q]);
            odd.x = perm_hi(b_reg[rs][i * 8 + 1][q], b_reg[rs][i * 8 + 0][q]);
            odd.y = perm_hi(b_reg[rs][i * 8 + 3][q], b_reg[rs][i * 8 + 2][q]);
            odd.z = perm_hi(b_reg[rs][i * 8 + 5][q], b_reg[rs][i * 8 + 4][q]);
            odd.w = perm_hi(b_reg[rs][i * 8 + 7][q], b_reg[rs][i * 8 + 6][q]);
            const int r0 = nc * 8 + 2 * q, r1 = r0 + 1;
            *(lds_u32x4)(size_t)((uint32_t)(A_STAGE + r0 * kRowBytes + swz(r0, kg) * 16) ^ st) = even;
            *(lds_u32x4)(size_t)((uint32_t)(A_STAGE + r1 * kRowBytes + swz(r1, kg) * 16) ^ st) = odd;
        }
    };

    // ---- MFMA fragments ---------------------------------------------------------------
    // lane -> row (A) / column (B) of a 32x32 block and which 8-wide half of the 16-wide k step
    const int frag_row = lane & 31, frag_kc = lane >> 5;
    uint32_t fa_off[TM], fb_off[TN];   // LDS byte offset of the lane's chunk at ks = 0
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int row = wm * WTM + i * 32 + frag_row;
        fa_off[i] = row * kRowBytes + swz(row, frag_kc) * 16;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int row = wn * WTN + j * 32 + frag_row;
        fb_off[j] = A_STAGE + row * kRowBytes + swz(row, frag_kc) * 16;   // A_STAGE < STAGE: survives the XOR
    }
    bf16x8 af[2][TM], bfr[2][TN];
    // chunk (2*ks + kc) ^ f(row) == (kc ^ f(row)) ^ 2*ks: the k sub-step only flips address bits 5..6
    // fa_off / fb_off carry the stage bit of the tile being computed (toggled every iteration);
    // `other` = STAGE reads from the other stage.
    auto read_frag = [&](int q, int ks, uint32_t other, int buf) {
        if (q < TM) af[buf][q] = *(lds_frag)(size_t)(fa_off[q] ^ (uint32_t)(ks << 5) ^ other);
        else bfr[buf][q - TM] = *(lds_frag)(size_t)(fb_off[q - TM] ^ (uint32_t)(ks << 5) ^ other);
    };

    // ---- software pipeline ---------------------------------------------------------------
    // Iteration t computes tile t from LDS stage t&1 while (a) the registers holding tile
    // t+1 (loaded from global memory during iteration t-1) are written to stage (t+1)&1 and
    // (b) tile t+2 is loaded into those registers.  MFMA fragments are double-buffered in
    // registers one 16-wide k sub-step ahead.  One workgroup barrier per iteration, placed
    // before the last sub-step: by then every wave has written its part of tile t+1 and has
    // issued (and waited for) its last reads of tile t.  All side work is spread between the
    // MFMAs in a fixed order.
    constexpr int NM = TM * TN, NF = TM + TN;
    const int k_last = (kt_total - 1) * BK;

#define KR_SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)
    // Side work of one iteration, in the order it is issued: A units, then B units; a unit is
    // "write the registers of tile t+1 to LDS, then re-fill them with tile t+2" (so those
    // loads have a whole iteration to land).  Row-major B consumes the 8 registers of a block
    // in 4 store units before the block is re-loaded.  The jobs are spread evenly over the MFMA
    // slots of sub-steps 0..2; sub-step 3 follows the barrier.
    constexpr int NJ = A_ITERS + (B_NT ? NB_ST : NB_ST + NB_LD);
    constexpr int NSL = 3 * NM;
    uint32_t nxt = STAGE;   // stage (relative to stage 0) that receives tile t+1
    static_assert((STAGE & (STAGE - 1)) == 0, "stage selection by XOR needs a power-of-two stage size");
    auto staging_job = [&](int rs, int j, int k2) {
        if (j < A_ITERS) {
            store_a_unit(rs, j, nxt);
            load_a_unit(rs, j, k2);
        } else if (B_NT) {
            store_b_unit(rs, j - A_ITERS, nxt);
            load_b_unit(rs, j - A_ITERS, k2);
        } else if (j - A_ITERS < NB_ST) {
            store_b_unit(rs, j - A_ITERS, nxt);
        } else {
            load_b_unit(rs, j - A_ITERS - NB_ST, k2);
        }
    };
    // one 16-wide k sub-step: NM MFMAs on fragment buffer `buf`; after each MFMA the fragment
    // reads of the next sub-step (into the other buffer) and the staging jobs of that slot
    auto mfma_step = [&](auto ks_c, auto rs_c, int k2) {
        constexpr int ks = decltype(ks_c)::value;
        constexpr int rs = decltype(rs_c)::value;
        constexpr int buf = ks & 1;
        constexpr bool staging = ks < 3;
#pragma unroll
        for (int s = 0; s < NM; ++s) {
            const int i = s / TN, j = s % TN;
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[buf][j], af[buf][i], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int q = s * NF / NM; q < (s + 1) * NF / NM; ++q)
                read_frag(q, (ks + 1) & 3, ks == 3 ? STAGE : 0, buf ^ 1);
            if constexpr (staging) {
                const int slot = ks * NM + s;
#pragma unroll
                for (int jj = slot * NJ / NSL; jj < (slot + 1) * NJ / NSL; ++jj) staging_job(rs, jj, k2);
            }
            KR_SCHED_FENCE();
        }
    };
    auto iteration = [&](int t, auto rs_c) {
        const int k2 = min((t + 3) * BK, k_last);   // tile t+3, clamped: the tail re-loads the last tile
        // The LDS offsets flip between the two stages every iteration.  Hide their values from
        // the optimiser here, or it pre-computes every (stage, sub-step) address variant outside
        // the loop and runs out of registers; the XORs it keeps inside are free next to the MFMAs.
#pragma unroll
        for (int i = 0; i < TM; ++i) asm volatile("" : "+v"(fa_off[i]));
#pragma unroll
        for (int j = 0; j < TN; ++j) asm volatile("" : "+v"(fb_off[j]));
#pragma unroll
        for (int i = 0; i < A_ITERS; ++i) asm volatile("" : "+v"(a_loff[i]));
        if (B_NT) {
#pragma unroll
            for (int i = 0; i < B_ITERS_NT; ++i) asm volatile("" : "+v"(b_loff[i]));
        }
        asm volatile("" : "+s"(nxt));
        mfma_step(std::integral_constant<int, 0>{}, rs_c, k2);
        mfma_step(std::integral_constant<int, 1>{}, rs_c, k2);
        mfma_step(std::integral_constant<int, 2>{}, rs_c, k2);
        // every LDS access of this wave so far has completed; then all waves meet
        __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0) only: the global loads stay in flight
        __builtin_amdgcn_s_barrier();
        KR_SCHED_FENCE();
        // sub-step 3 reads the fragments of sub-step 0 of tile t+1
        mfma_step(std::integral_constant<int, 3>{}, rs_c, k2);
        // switch stages: the fragment offsets follow the tile being computed
#pragma unroll
        for (int i = 0; i < TM; ++i) fa_off[i] ^= STAGE;
#pragma unroll
        for (int j = 0; j < TN; ++j) fb_off[j] ^= STAGE;
        nxt ^= STAGE;
    };

    // prologue: tile 0 -> stage 0, tiles 1 and 2 -> the two register sets, first fragments
#pragma unroll
    for (int i = 0; i < A_ITERS; ++i) load_a_unit(0, i, 0);
#pragma unroll
    for (int u = 0; u < NB_LD; ++u) load_b_unit(0, u, 0);
#pragma unroll
    for (int i = 0; i < A_ITERS; ++i) store_a_unit(0, i, 0);
#pragma unroll
    for (int u = 0; u < NB_ST; ++u) store_b_unit(0, u, 0);
    {
        const int k1 = min(BK, k_last), k2 = min(2 * BK, k_last);
#pragma unroll
        for (int i = 0; i < A_ITERS; ++i) load_a_unit(0, i, k1);
#pragma unroll
        for (int u = 0; u < NB_LD; ++u) load_b_unit(0, u, k1);
#pragma unroll
        for (int i = 0; i < A_ITERS; ++i) load_a_unit(1, i, k2);
#pragma unroll
        for (int u = 0; u < NB_LD; ++u) load_b_unit(1, u, k2);
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_s_barrier();
    KR_SCHED_FENCE();
#pragma unroll
    for (int q = 0; q < NF; ++q) read_frag(q, 0, 0, 0);

    // branch-free body (a conditional second half would put 256 live accumulators through
    // control-flow merges); an odd last tile is peeled
    int t = 0;
    for (; t + 1 < kt_total; t += 2) {
        iteration(t, std::integral_constant<int, 0>{});
        iteration(t + 1, std::integral_constant<int, 1>{});
    }
    if (t < kt_total) iteration(t, std::integral_constant<int, 0>{});
#undef KR_SCHED_FENCE
    // the tail iterations re-load and re-store the last tile: drain everything before the
    // LDS is reused by the epilogue
    __syncthreads();

    gemm_epilogue<BM, WTM, WTN, TM, TN, EVEN, EP_WAVE>(g, g.n_peers, g.bias, acc, smem, m0, n0, wm, wn, lane, wave);
}

// Second pass of the split K loop: sums the S fp32 partial products [S][M][N] in the order
// 0..S-1 and applies the epilogue of the one-pass kernel (same order of the adds, same
// rounding: with a bf16 result and peers the product is rounded to bf16 before the peers'
// partial sums are added).  One thread per 8 consecutive columns.  Bound by the round trips to memory one behind the
// other: with the parts and peers requested together 16 x 8192 x 3584 in four parts with seven peers takes 20.9 us
// instead of 23.6 (both launches).
__global__ __launch_bounds__(256) void splitk_finish_kernel(const GemmArgs g, const float* __restrict__ parts, int S) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int nv = g.N / 8;
    if (v >= (int64_t)g.M * nv) return;
    const int m = (int)((uint64_t)v <= 0xffffffffull ? (uint32_t)v / (uint32_t)nv : v / nv), n = (int)(v - (int64_t)m * nv) * 8;
    const int64_t mn = (int64_t)g.M * g.N;
    const float* p = parts + (int64_t)m * g.N + n;
    const int mb = m - g.band_row0;
    const bool in_band = mb >= 0 && mb < g.band_rows;
    const int64_t off = (int64_t)mb * g.N + n;
    // the first peers' partial sums and the parts are requested before anything is added: with few rows the kernel is
    // one round trip to memory long
    constexpr int kPeers = 7, kParts = 4;
    u32x4 pv[kPeers];
    if (in_band) {
#pragma unroll
        for (int q = 0; q < kPeers; ++q)
            if (q < g.n_peers) pv[q] = ld_stream((const u32x4*)((const uint16_t*)g.peer.p[q] + off));
    }
    float f[8];
    zero8(f);
    for (int s0 = 0; s0 < S; s0 += kParts) {
        f32x4 x[kParts][2];
#pragma unroll
        for (int j = 0; j < kParts; ++j) {
            const float* q = p + min(s0 + j, S - 1) * mn;
            x[j][0] = __builtin_nontemporal_load((const f32x4*)q);
            x[j][1] = __builtin_nontemporal_load((const f32x4*)(q + 4));
        }
#pragma unroll
        for (int j = 0; j < kParts; ++j) {
            if (s0 + j >= S) break;
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] += x[j][e / 4][e % 4];
        }
    }
    if (!in_band) {
        if (g.c_full != nullptr) st_stream((u32x4*)(g.c_full + (int64_t)m * g.N + n), pack8(f));
        return;
    }
    if (g.out_fp8) {
        store8_e4m3((uint8_t*)g.out + off, f);
        return;
    }
    if (!g.out_is_fp32) unpack8(pack8(f), f);   // the one-pass kernel rounds the product on its way to the epilogue
#pragma unroll
    for (int q = 0; q < kPeers; ++q)
        if (q < g.n_peers) add8(pv[q], f);
    for (int q = kPeers; q < g.n_peers; ++q) add8(ld_stream((const u32x4*)((const uint16_t*)g.peer.p[q] + off)), f);
    if (g.bias != nullptr) add8(*(const u32x4*)(g.bias + n), f);
    if (g.out_is_fp32) {
        float* o = (float*)g.out + off;
        *(f32x4*)o = f32x4{f[0], f[1], f[2], f[3]};
        *(f32x4*)(o + 4) = f32x4{f[4], f[5], f[6], f[7]};
    } else {
        st_stream((u32x4*)((uint16_t*)g.out + off), pack8(f));
    }
}

static hipError_t launch_splitk_finish(const GemmArgs& g, const void* parts, int S, hipStream_t st) {
    const int64_t vecs = (int64_t)g.M * (g.N / 8);
    const unsigned threads = vecs > 65536 ? 256 : 64;   // few rows: one wavefront per workgroup, on as many compute units as there are
    hipLaunchKernelGGL(splitk_finish_kernel, dim3((unsigned)((vecs + threads - 1) / threads)), dim3(threads), 0, st, g, (const float*)parts, S);
    return hipGetLastError();
}

template <int BM, int BN, int WM, int WN>
static hipError_t launch_gemm(const GemmArgs& g, bool b_nt, bool even, hipStream_t st) {
    constexpr int T = WM * WN * 64;
    constexpr int LDS = 2 * (BM + BN) * kRowBytes;
    const dim3 grid((unsigned)(g.tiles_m * g.tiles_n), (unsigned)g.k_splits), block(T);
#define KR_LAUNCH(NT, EV)                                                                             \
    do {                                                                                              \
        auto kfn = gemm_reduce_kernel<BM, BN, WM, WN, NT, EV>;                                        \
        static std::atomic<uint64_t> opted{0};                                                        \
        if (hipError_t e = lds_opt_in((const void*)kfn, LDS, opted); e != hipSuccess) return e;       \
        hipLaunchKernelGGL(kfn, grid, block, LDS, st, g);                                             \
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

using namespace kr;

constexpr int kMaxSplits = 16;
constexpr int kMinSplitSteps = 8;
// ---- 256x256 kernel: split of the last partial round ------------------------------------------
// 256 tiles run at a time (one per CU).  When the tile count leaves a last round that is at most
// 3/8 full (half, with a longer K) and K is long enough, its tiles get S = 256 / tail workgroups each (at least kMinSplitSteps k-steps per
// part, at most kMaxTailSplits parts), which turns that round from a whole one into tail/256
// of one; the price is tail * S partial tiles of 256 KiB written and read once.
constexpr int kMaxTailSplits = 8;
static void tail_split_plan(int64_t tiles, int64_t K, int* tail_out, int* splits_out) {
    *tail_out = 0;
    *splits_out = 1;
    const int64_t force = env_switches().gemm_tailsplit;   // 0: off, n: n parts (testing)
    if (force == 0 || (tiles > 128 && tiles <= 256)) return;
    // up to 128 tiles the whole launch is one partial round
    const int64_t tail = tiles % 256;
    // (measured: 16..64 tail tiles gain 5-25 % from K = 4096 on; 128 tail tiles at K = 2048 lose
    // 12 %: half a round saved does not pay for two more launches and 64 MiB of parts)
    // 97 to 128 tiles in two parts each from K = 8192 on, us: 5632 x 4224 (374 tiles) row-major x 11264 469 / 428, x 8192 351 / 324, transposed
    // 447 / 421, 336 / 322; 6080 x 4096 (384) 462 / 439, 344 / 331, 439 / 422, 322 / 320; x 4096 188 / 197.
    // Ragged shapes the same, us, whole rounds / in parts, transposed B unless said: 5486 x 3456 x 9984 397 / 310 (308 tiles),
    // 4900 x 3648 x 4096 172 / 152, row-major 188 / 157, 2312 x 8000 x 6144 271 / 218, 4584 x 7744 x 5376 348 / 324; below K = 4096
    // transposed B gains little and less with a K of 2048: 4600 x 4096 x 3072 131 / 124, x 2048 88 / 95.
    // A K from 3072 on and up to 48 such tiles, four parts: 4104 x 4096 (272 tiles) x 3072 125 / 116, row-major 132 / 118, x 3648 146 / 130,
    // 169 / 132; 4864 x 4096 (304) x 3072 126 / 124, 129 / 125, x 3648 149 / 139, 163 / 143; 64 tiles x 3072 124 / 128.
    const bool short_k = K < 4096 && tiles > 128;
    if (tail == 0 || (tail > (K >= 8192 ? 128 : short_k ? 48 : 96) && tiles > 128) || (K < (short_k ? 3072 : 4096) && force <= 0)) return;
    int64_t s = std::min<int64_t>(256 / tail, short_k ? 4 : kMaxTailSplits);
    s = std::min<int64_t>(s, (K / 64) / kMinSplitSteps);
    if (force > 0) s = std::min<int64_t>(force, K / 64);
    if (s < 2) return;
    *tail_out = (int)tail;
    *splits_out = (int)s;
}
static int64_t gemm_dtl_tail_workspace_bytes(int tail_tiles, int splits, int cols = 256) {
    return (int64_t)tail_tiles * splits * (256 * 4) * cols;
}

// fp8 operands: which tiles share their K loop, and how many workgroups each gets.  With at most 128 tiles
// the whole launch is a partial round (half the compute units or more would idle) and every tile may be
// split; otherwise the rule of the bf16 kernel, on the same number of k-steps (one is 128 long here).
// A k-step takes 0.9 us, a part that is written and summed 0.09 us, the finishing launch 3 us; the split
// with the least sum is taken if it saves a tenth of the k loop.  Measured (one pass / split, us):
// 64 x 6656 x 8192 66 / 29 in 5 parts (34 in 8), 512 x 6656 x 8192 66 / 45 in 4, 1024 x 6656 x 16384 142 / 107
// in 2, but 1024 x 6656 x 4096 38 / 48 and 512 x 6656 x 2048 23 / 32, which stay in one pass.
static void fp8_split_plan(int64_t M, int64_t N, int64_t K, int* tail_out, int* splits_out) {
    const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256), steps = (K + 127) / 128;
    *tail_out = 0;
    *splits_out = 1;
    if (tiles > 128) return tail_split_plan(tiles, K / 2, tail_out, splits_out);
    int64_t best = 81 * steps;   // nine tenths of the one-pass k loop, in 0.01 us
    for (int64_t s = 2; s <= kMaxTailSplits && s * tiles <= 256 && s <= steps / 4; ++s) {
        const int64_t cost = 90 * steps / s + 9 * tiles * s + 300;
        if (cost >= best) continue;
        best = cost;
        *tail_out = (int)tiles;
        *splits_out = (int)s;
    }
}

// fp8 operands widened to bf16 in registers (gemm_w8.hip): the columns as `panels` panels of 256, then narrower ones of
// 32 nb2 (nb2 = 0: none), or with at most 128 tiles of 256x256 every tile's K loop in `splits` parts.
// Widths: whole rounds of 256-column tiles and the narrow ones behind them, the pair that ends first.  A round costs, in
// 0.01 us, 4 us to start and finish its tiles and per k-step of 128 and 256 columns 2.05 us with up to 160 compute units
// busy, 2.56 with all of them (the power limit), 3 % more per 32 columns less.  Measured in turn, on a card of the slower ones
// (the first call's choice takes 135 to 146 us on different cards), us, 256-column tiles / 224 / the choice: 4000 x 6656 x 4096 164 / 150.5 / 146.2 (16 panels, then 160 columns), 8000 x 3584 x 8192 308.6 / 299.3 / 299.3,
// 2400 x 4992 x 8192 143.6 / 139.3 / 139.3, 8192 x 4096 x 8192 335.8 / 413.4 / 335.8.
struct W8Plan {
    int panels, nb2, splits;
};
static W8Plan plan_w8(int64_t M, int64_t N, int64_t K, bool may_split, int64_t workspace_bytes) {
    const int64_t tm = (M + 255) / 256, tn = (N + 255) / 256, tiles = tm * tn, steps = (K + 127) / 128;
    W8Plan p{(int)tn, 0, 1};
    if (const int v = env_switches().gemm_w8; v >= 0) {   // testing and tuning
        const int64_t nb2 = v / 1000, panels = std::min<int64_t>(v % 1000, N / 256);
        if (nb2 >= 4 && nb2 <= 7) return W8Plan{(int)panels, N > panels * 256 ? (int)nb2 : 0, 1};
        if (nb2 == 0 && v > 1 && may_split && v <= steps && tiles * v * (256 * 256 * 4) <= workspace_bytes) p.splits = v;
        return p;
    }
    if (tiles <= 128) {
        int64_t best = 500 + 210 * steps;
        for (int64_t s = 2; may_split && s <= kMaxSplits && s * tiles <= 256 && 2 * s <= steps && tiles * s * (256 * 256 * 4) <= workspace_bytes; ++s) {
            const int64_t cost = 900 + 210 * ((steps + s - 1) / s) + s * M * N * 8 / 50000;
            if (cost < best) {
                best = cost;
                p.splits = (int)s;
            }
        }
        return p;
    }
    auto round_cost = [&](int64_t nb, int64_t busy) {
        return 400 + steps * (205 + (busy > 160 ? 51 * (busy - 160) / 96 : 0)) * nb * (100 + 3 * (8 - nb)) / 800;
    };
    auto rounds_cost = [&](int64_t nb, int64_t n) { return n / 256 * round_cost(nb, 256) + (n % 256 > 0 ? round_cost(nb, n % 256) : 0); };
    int64_t best = rounds_cost(8, tiles);
    for (int64_t panels = 0; panels * 256 < N; ++panels) {
        for (int64_t nb = 4; nb < 8; ++nb) {
            const int64_t wide = tm * panels, narrow = tm * ((N - panels * 256 + 32 * nb - 1) / (32 * nb));
            const int64_t early_end = wide / 256 * round_cost(8, 256), late = wide % 256;
            int64_t end = early_end;
            if (late == 0) {
                end += rounds_cost(nb, narrow);
            } else {
                // `late` compute units are free one wide tile after the others: i narrow tiles on each of the others
                const int64_t late_end = early_end + round_cost(8, 256), c = round_cost(nb, 256);
                end = late_end;
                for (int64_t i = 1, done = 0; done < narrow; ++i) {
                    end = std::max(end, early_end + i * c);
                    done = i * (256 - late) + (end - late_end) / c * late;
                }
            }
            if (end < best) {
                best = end;
                p.panels = (int)panels;
                p.nb2 = (int)nb;
            }
        }
    }
    return p;
}
// workspace of the two-pass form: S fp32 partial products of the whole [M, N] result
static int64_t split_k_workspace_bytes(int64_t M, int64_t N, int S) { return (int64_t)S * M * N * 4; }

// ---- at most 128 tiles of 256x256: which kernel, and how many workgroups share a tile -----------------
// Three candidates, by what they cost in 0.01 us (measured with operands that are in no cache, M = 128 .. 2000,
// N = 1024 .. 6656, K = 512 .. 16384; the model is within 15 % of the measurements where it matters):
//   a 128x128 kernel, S workgroups per tile: 6.5 us to start and finish, 0.56 us (row-major B 0.60) per
//     k-step of 64 and round of 256 workgroups -- a compute unit takes in about 57 GB/s of operands that other
//     units are waiting for too, whatever its pipeline; S > 1 adds a launch and S fp32 parts written and read (6 us and
//     16 ns per million elements with row-major B, which runs gemm_ks_kernel; 2 us and 20 ns and parts of at least eight
//     k-steps with transposed B, gemm_reduce_kernel: fitted to every split of 13 257 random shapes, 65 to 4096 rows, where
//     this choice takes 1.009 (no peers) and 1.033 (peers) of the time of the best one);
//     S = 1 with peers and more than 16 k-steps (transposed B 15: 384 x 1712 x 1024 23.7 / 18.4) 4 us more (fitted, the cause is not separated; one or three peers, in
//     one pass / in three parts: 112 x 9216 x 1664 27.0 / 21.7, 256 x 4096 x 1536 25.0 / 20.8, 720 x 1280 x 1464 24.6 / 21.1,
//     row-major 22.4 / 20.1; 360 x 768 x 1096 21.4 / 20.5; but 300 x 2048 x 1024 16.8 / 19.6, 128 x 4096 x 1024 16.5 / 19.1);
//     Transposed B with 257 to 512 workgroups: 0.68 us and 0.18 a round, not two whole rounds (gemm_reduce_kernel has room
//     for a second workgroup on a compute unit);
//   the 256-row kernel with every tile's K loop in parts, M and N as they come: half the operand bytes per flop, but
//     parts of whole tiles.  10.7 us, 1.03 us per k-step (row-major B 1.08, 224-column tiles 0.94) and 0.25 more with all
//     compute units busy, 0.24 us per MB of parts; at least eight k-steps a part, K from 2048 on, and only where this is
//     0.88 or less of the best 128x128 form (both models are off by a tenth; whole tiles with a long K need no margin).
//     224 columns, transposed B only, where they fill enough more compute units to be 2 % ahead.
//     Two kinds of shapes where the 128x128 forms are cheaper than that model says have to clear a second bar (calls one behind
//     the other, four sets of operands in turn, 1700 shapes in all):
//     * M and N multiples of 128: those forms have no edge tiles then, and a short K does not pay for the second launch.  The bar
//       rises with the doublings of K from 2048 on: one round of 128x128 workgroups 0.51 + 0.14 a doubling (transposed B 0.51 + 0.19),
//       more 0.67 + 0.11 (0.83 + 0.04).  1180 shapes: of the 890 below the bar 64 are slower in parts, 33 by more than 3 %, up
//       to 1.16, 0.844 in the mean; above it 222 of 290 are, up to 1.33, 1.077 in the mean.  512 x 4352 x 4096 row-major with a band
//       (32.4 us / 39.2 in parts), x 3072 transposed (29.5 / 33.9), 2816 x 2560 x 3072 row-major (52.9 / 63.5) stay on 128x128;
//     * other shapes with row-major B and one round of 128x128 workgroups: 6 % ahead by a closer fit of both: in parts 25.4 us, 0.18 us
//       per k-step and 1.24 more with all compute units busy, 0.044 us per MB of operands; on 128x128 2.9 us, 0.53 us per k-step,
//       0.101 us per MB of operands, parts 0.9 us and 0.42 per MB.  93 shapes: 4 of the 58 below the bar are slower in parts, up to
//       1.04, 25 of the 35 above it, up to 1.15 (1422 x 1088 x 7424 40.7 / 47.1, 632 x 2304 x 6208 with a band 37.7 / 42.2).
//     The rest, 427 shapes: 0.55 to 1.05, 0.797 in the mean, 4 of them slower.  540 shapes of all kinds drawn after the bars were set and
//     left in parts: 25 slower, 14 by more than 3 %, up to 1.09, 0.827 in the mean.  us,
//     128x128 / in parts: 504 x 6656 x 8192 with a band 82 / 66, 576 x 4608 x 10560 row-major 101 / 78, 998 x 6400 x 6336
//     row-major 134 / 102, 1792 x 2432 x 12912 224 / 134; 512 x 6656 with a band and seven peers, 256 columns (208
//     workgroups) / 224 (240), K = 8192 68.1 / 66.3, 16384 120 / 109.
//     Left on the forms they had, which tests/test_capi_host.py and tests/test_gemm_gpu.py name: plain products of whole tiles
//     (256 columns; 224 are level where they divide N, 512 x 5376 x 6400 50.5 / 50.2, 256 x 7168 x 12928 62.9 / 62.3, and
//     66 / 63 at 512 x 6656 x 8192); whole tiles with a K that is no multiple of 64, and a K that is no multiple of 16.  Others, by
//     the same rule:
//     a K that is no multiple of 64, which makes no difference to the parts and costs the 128x128 forms more: 18 of 64 shapes go in
//     parts, 0.52 to 0.96 of the time (3144 x 1392 x 15472 270 / 141, 3224 x 1248 x 7136 row-major with a band 142 / 75, 736 x 6416
//     x 5680 105 / 78, 1016 x 3728 x 2512 38.4 / 36.5); with transposed B and at most one peer 27 of 60 shapes of 129 to 272 tiles,
//     0.52 to 1.00 (944 x 4240 x 13360 with one peer 247 / 129, 2200 x 1856 x 13616 plain 233 / 122, 1144 x 2320 x 6784 69 / 58); of
//     54 of those with N a multiple of 128 and at most 32 rows less than one of M 30 go in parts, 0.63 to 0.92 of the time but for one
//     (1000 x 4096 x 8192 plain 71.3 / 73.0; 992 x 4352 x 13824 with one peer 186 / 117, 1000 x 4224 x 4096 plain 55.1 / 48.1).
// Which 128x128 kernel, by the time of gemm_ks_kernel over that of gemm_reduce_kernel (geometric means over 20 000 random
// shapes, 1 to 8192 rows, operands in no cache):
//   transposed B, in parts: 1.034 to 1.042 at every K: gemm_reduce_kernel.  In one pass, K a multiple of 64, no peers:
//     1.05 below K = 362, 0.96 from 724 to 1448, 0.98 to 1.00 up to 8192; with peers 1.03 to 0.98, level on the whole; K no
//     multiple of 64: 1.054.  Above 256 tiles 1000 x 6656 x 1024 27 / 23 us, x 4096 75 / 73, x 8192 136 / 132; above K = 8192 it
//     loses much where its five stages in flight ask the same memory channels for rows that lie a multiple of 4 KiB
//     (and no power of two) apart: 1000 x 3328 x 12288 144 / 119, x 24576 282 / 224, 1000 x 6656 x 12288 273 / 200.
//   row-major B, up to 256 tiles: 0.88 at K = 256, 0.72 at 1024, 0.66 from 4096 on, in parts 0.88: gemm_ks_kernel.
//     Above 256 tiles gemm_reduce_kernel has two workgroups per compute unit and one tile's epilogue runs beside
//     another's k loop.  K a multiple of 64, without / with peers: 1.02 / 1.07 from 1024 to 2048, 0.94 / 0.97 above; no
//     multiple: 1.08 / 1.08, 1.01 / 1.06.  1000 x 6656 x 1024 28.6 / 28.2 us, x 2048 45 / 47, x 4096 79 / 86, x 8192 144 / 165.
struct SmallPlan {
    int big;      // columns of the large tiles, every one split: 256 or 224; 0: a 128x128 kernel
    int ks;       // gemm_ks_kernel, else gemm_reduce_kernel
    int splits;   // workgroups per tile
};
static int64_t big_tiles_of(int64_t M, int64_t N, int cols) { return ((M + 255) / 256) * ((N + cols - 1) / cols); }
static SmallPlan plan_small(int64_t M, int64_t N, int64_t K, bool b_nt, int n_peers, bool plain, bool dtl_ok, bool may_split, bool may_big) {
    const bool peers = n_peers > 0;
    SmallPlan p{0, 0, 1};
    const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128), steps = (K + 63) / 64;
    auto choose_kernel = [&]() {
        p.ks = dtl_ok && (b_nt ? p.splits == 1 && !peers && tiles <= 256 && K % 64 == 0 && K >= 640 && K <= 8192 : tiles <= 256 || (K % 64 == 0 && K >= 2048));
        if (env_switches().gemm_ks >= 0) p.ks = dtl_ok && env_switches().gemm_ks != 0;
        return p;
    };
    if (!may_split) return choose_kernel();
    if (const int v = env_switches().gemm_splitk; v >= 1 && v <= kMaxSplits) {   // testing and tuning
        p.splits = (int)std::min<int64_t>(v, steps);
        return choose_kernel();
    }
    const int64_t step = b_nt ? 56 : 60, launch = b_nt ? 200 : 600, part = b_nt ? 20 : 16, min_steps = b_nt ? kMinSplitSteps : 2;
    const bool long_peers = peers && steps > (b_nt ? 15 : 16);
    auto cost = [&](int64_t s) {
        return 650 + (tiles * s + 255) / 256 * step * ((steps + s - 1) / s) + (s > 1 ? launch + s * M * N * part / 100000 : long_peers ? 400 : 0);
    };
    int64_t best = cost(1);
    for (int64_t s = 2; s <= kMaxSplits && min_steps * s <= steps && s * tiles <= 512; ++s)
        if (const int64_t c = cost(s); c < best) {
            best = c;
            p.splits = (int)s;
        }
    // (gemm_reduce_kernel has room for a second workgroup on a compute unit, which the model does not count: with 129 to
    // 256 tiles it pays once the K loop is long, 0.86 of the time of one pass with 144 tiles from K = 12288 on, 0.94 with 208)
    if (b_nt && p.splits == 1 && tiles > 128 && tiles <= 256 && K >= 12288) p.splits = 2;
    const EnvSwitches& env = env_switches();
    const int64_t force = env.gemm_tailsplit;   // 0: off, n: n parts (testing)
    const bool whole = M % 256 == 0 && N % 256 == 0;
    const bool as_before = K < 2048 || (K % 64 != 0 && (K % 16 != 0 || whole));   // see above
    if (may_big && dtl_ok && force != 0 && (env.gemm_mfma != 32 || (whole && K % 64 == 0)) && (!as_before || force > 0)) {
        // whole tiles, K from 4096 on, as many parts as there are compute units for: no margin
        const int64_t most = std::min<int64_t>({256 / std::max<int64_t>(1, big_tiles_of(M, N, 256)), kMaxTailSplits, steps / kMinSplitSteps});
        const bool long_whole = whole && K >= 4096 && most > 1 &&
                                1400 + 120 * ((steps + most - 1) / most) + most * big_tiles_of(M, N, 256) * 262144 * 2 / 50000 < best;
        // (the second round of gemm_reduce_kernel starts beside the first, see above)
        const int64_t wgs = tiles * p.splits, per = (steps + p.splits - 1) / p.splits;
        if (b_nt && wgs > 256 && wgs <= 512) best += (68 + 18 * wgs / 256 - 2 * step) * per;
        const int64_t small_cost = best;
        const int small_splits = p.splits;
        int64_t big_cost = 0;
        best = best * 88 / 100;
        if (long_whole || (force > 0 && env.gemm_tile == 256)) best = INT64_MAX;
        for (const int cols : {256, 224}) {
            if (cols == 224 ? !b_nt || env.gemm_n224 == 0 || env.gemm_mfma == 32 || (plain && whole && env.gemm_n224 < 0) : b_nt && env.gemm_n224 == 1) continue;
            const int64_t big_tiles = big_tiles_of(M, N, cols);
            if (p.big && force <= 0) best = best * 98 / 100;   // (224 after 256: level otherwise)
            for (int64_t s = cols == 256 && long_whole && force <= 0 ? most : 2; s <= kMaxTailSplits; ++s) {
                if (force > 0 ? s != std::min<int64_t>(force, steps) : s * big_tiles > 256 || s * kMinSplitSteps > steps) continue;
                const int64_t bytes = gemm_dtl_tail_workspace_bytes((int)big_tiles, (int)s, cols), k = (steps + s - 1) / s;
                const int64_t c = 1070 + ((cols == 224 ? 94 : b_nt ? 103 : 108) + 25 * s * big_tiles / 256) * k + bytes * 241 / 10000000;
                if (bytes > KR_STATIC_SCRATCH_BYTES || c >= best) continue;   // (the form that allocates nothing takes every split)
                best = big_cost = c;
                p.big = cols;
                p.splits = (int)s;
            }
        }
        // where that model is too kind to the parts (see above)
        bool ahead = true;
        if (p.big && M % 128 == 0 && N % 128 == 0) {
            const double doublings = std::log2((double)K / 2048);
            const double limit = b_nt ? (wgs <= 256 ? 0.51 + 0.19 * doublings : 0.83 + 0.04 * doublings)
                                      : (wgs <= 256 ? 0.51 + 0.14 * doublings : 0.67 + 0.11 * doublings);
            ahead = big_cost < limit * small_cost;
        } else if (p.big && !b_nt && wgs <= 256) {
            const int64_t operands = 2 * (M + N) * K, parts = small_splits > 1 ? 4 * small_splits * M * N : 0;
            const int64_t k = (steps + p.splits - 1) / p.splits, busy = p.splits * big_tiles_of(M, N, 256);
            const int64_t in_parts = 2540 + (18 + 124 * busy / 256) * k + operands * 44 / 10000000;
            const int64_t on_128 = 286 + 53 * per + (parts > 0 ? 89 : 0) + parts * 424 / 10000000 + operands * 101 / 10000000;
            ahead = in_parts < on_128 * 94 / 100;
        }
        if (!ahead && !long_whole && force <= 0) {
            p.big = 0;
            p.splits = small_splits;
        }
    }
    return choose_kernel();
}

// ---- at most 64 rows (gemm_skinny.hip): columns per workgroup and workgroups that share a K loop -------------
// By a model of what the forms cost, in 0.01 us, fitted to measurements with B in no cache (M = 2 .. 64, N = 1024 ..
// 8192, K = 576 .. 16384; within 15 %): 6 us to start and finish, 5 us for every further round of 256 workgroups; a
// compute unit takes in 64 GB/s of 128-byte rows, and a k-row of a row-major B costs it 2.3 / 3.0 / 3.4 ns for 32 / 64 /
// 128 bytes; HBM 6 TB/s; parts of K a second launch and their bytes.  Against the 128x128 kernel and its parts, us:
// 16 x 8192 x 3584 with seven peers 20.9 -> 14.1 (row-major B 21.9 -> 18.8), 4 x 3360 x 976 14.1 -> 6.3, 4 x 2816 x 576
// row-major 15.0 -> 6.1, 16 x 1024 x 16384 22.6 -> 15.5, fp32 2 x 1216 x 1280 17.1 -> 7.8, 16 x 4096 x 4096 28.7 -> 17.6;
// 64 x 8192 x 3584 24.4 -> 19.2, row-major level (24.4 / 24.7).  From 65 rows on the rows of A, which every workgroup
// reads, outweigh B; so they do below with wide outputs and a long K, where the model does not see it.  Time of this kernel
// over that of the 128x128 kernels, bf16, N of 2048 and more (geometric means of random shapes): 33 to 64 rows, transposed
// B 0.67 at K = 2048, 0.83 at 3500, 0.97 at 4900, 1.06 at 7000, 1.17 at 9700, 1.28 at 14000, row-major 0.86, 0.98, 1.08, 1.22,
// 1.35, 1.48; 17 to 32 rows, transposed 0.87 at 7000, 0.97 at 9700, 1.07 at 14000.  Narrower ones stay below 1.
constexpr int64_t kMaxPartsBytes = KR_STATIC_SCRATCH_BYTES;   // (the form that allocates nothing takes every split)
struct SkinnyPlan {
    int cb;       // columns of a workgroup / 16; 0: not for this call
    int splits;   // parts of K, summed by a second launch
};
static SkinnyPlan plan_skinny(int64_t M, int64_t N, int64_t K, bool b_nt, int64_t e, int64_t parts_bytes) {   // e: bytes of an element
    SkinnyPlan p{0, 1};
    const EnvSwitches& env = env_switches();
    if (M > 64 || N < 16 || env.gemm_tile > 0 || env.gemm_ks >= 0 || env.gemm_splitk >= 1 || env.gemm_skinny == 0) return p;
    const bool f32 = e == 4;
    const int64_t units = (K * e + 127) / 128, rows = M <= 16 ? 16 : M <= 32 ? 32 : 64;
    parts_bytes = std::min(parts_bytes, kMaxPartsBytes);
    if (const int cb = env.gemm_skinny / 100, s = env.gemm_skinny % 100; cb > 0) {   // testing and tuning
        if (cb != 1 && cb != 2 && (cb != 4 || f32)) return p;
        p.cb = cb;
        if (s >= 1 && s <= units && s * M * N * 4 <= parts_bytes) p.splits = s;
        return p;
    }
    if (e == 2 && M > 16 && N >= 2048 && K > (M > 32 ? (b_nt ? 4096 : 3584) : b_nt ? 11264 : INT64_MAX)) return p;
    int64_t best = 0;
    for (int cb = 1; cb <= (f32 || M > 32 ? 2 : 4); cb *= 2) {
        for (int64_t s = 1; s <= kMaxSplits && (s == 1 || (4 * s <= units && s * M * N * 4 <= parts_bytes)); s *= 2) {
            const int64_t rounds = ((N + 16 * cb - 1) / (16 * cb) * s + 255) / 256, k = (K + s - 1) / s, line = 16 * cb * e;
            const int64_t b_time = b_nt ? line * k / 640 : (line <= 32 ? 23 : line <= 64 ? 30 : 34) * k / 100;
            const int64_t c = 600 + 500 * (rounds - 1) + std::max(rounds * (rows * e * k / 640 + b_time), N * K * e / 60000) +
                              (s > 1 ? 400 + 50 * s + s * M * N * 8 / 50000 : 0);
            if (p.cb != 0 && c >= best) continue;
            best = c;
            p.cb = cb;
            p.splits = (int)s;
        }
    }
    return p;
}

// ---- the workspace form for callers that cannot allocate ------------------------------------------
// The split-K workspace lives in a device array of the library instead of caller memory.  Host code
// never uses the array's name as an address: each device's copy is looked up once, with that device
// current, and the pointer kept is what the kernels get, exactly as they get the caller's workspace.
static __device__ __align__(256) unsigned char scratch[KR_STATIC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
static int static_scratch(void** out) {
    static std::mutex mu;
    static void* ptr_of_device[kMaxDevices] = {};
    int dev = -1;
    if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= kMaxDevices) return (int)hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(mu);
    if (ptr_of_device[dev] == nullptr) {
        void* ptr = nullptr;
        if (hipError_t e = hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)); e != hipSuccess) return (int)e;
        if (ptr == nullptr) return (int)hipErrorInvalidSymbol;
        ptr_of_device[dev] = ptr;
    }
    *out = ptr_of_device[dev];
    return KR_OK;
}

// ---- which kernel a call gets ----------------------------------------------------------------
// One place decides it, for the launch and for kr_gemm_plan (which reports the decision).
struct GemmPlan {
    int tile;            // 256: LDS-DMA kernel (gemm_dtl.hip); 128: register-staged kernel (this file)
    int mi16;            // 256x256 kernel: k loop on 16x16x32 blocks (else 32x32x16)
    int peers_on_mfma;   // 256x256 kernel, 32x32x16 form: whole-band tiles add their peers on the matrix cores
    int group_n;         // column panels per scheduling group
    int tail_tiles;      // 256x256 kernel: tiles of the last partial round that are split ...
    int tail_splits;     // ... into this many parts each
    int splits;          // 128x128 kernel: workgroups per tile (split K loop), 1 = one pass
    int ks;              // 128x128 tiles: k divided among the waves (gemm_ks.hip), else among 64-wide fragments of each wave
    int skinny;          // at most 64 rows: columns of a workgroup / 16 (gemm_skinny.hip), 0: another kernel
    int n224;            // 256x224 tiles instead of 256x256 (whole rounds of compute units where those leave a partial one)
};
static GemmPlan plan_of_skinny(const SkinnyPlan& sk) {
    GemmPlan p{};
    p.tile = 128;   // (the tile order of the 128x128 kernels; not used)
    p.mi16 = 1;
    p.group_n = 1;
    p.tail_splits = 1;
    p.splits = sk.splits;
    p.skinny = sk.cb;
    return p;
}
// Whether a shape has enough tiles of 256 x 256 for one-pass workgroups (see plan_gemm).  Not with transposed B, a short K
// that is no multiple of the k-step and a last round that leaves the launch less than 5/8 full: by the time of the
// 256x256 kernel over that of the 128x128 kernel (geometric means of random shapes) 1.08 below K = 448 and 0.99 from there
// to 1024, with fuller rounds 0.99 and 0.92 or less (4096 x 4672 x 416, 304 tiles, 37.5 / 30.7 us); row-major B 0.93, 0.87.
static bool many_big_tiles(int64_t M, int64_t N, int64_t K, bool b_nt) {
    const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256);
    if (b_nt && K % 64 != 0 && K < 640 && (tiles + 255) / 256 * 256 * 5 >= tiles * 8) return false;
    return tiles > 128 && K >= 256;
}
static GemmPlan plan_gemm(int64_t M, int64_t N, int64_t K, bool b_nt, int n_peers, int64_t band_rows, bool plain,
                          bool plain_bf16_all_rows, bool has_workspace, int64_t workspace_bytes, bool has_gather, bool has_progress, bool flagged,
                          bool dtl_ok, bool skinny_ok) {
    GemmPlan p{};
    if (skinny_ok && !flagged) {
        const SkinnyPlan sk = plan_skinny(M, N, K, b_nt, 2, has_workspace ? workspace_bytes : 0);
        if (sk.cb != 0) return plan_of_skinny(sk);
    }
    // Tile choice: the 256x256 tile of the LDS-DMA kernel (4 waves x 128x128) has the highest
    // MFMA work per LDS/HBM byte; it needs a K loop long enough to amortise its epilogue.
    // Otherwise 128x128 tiles; they also win while all of them fit on the
    // 256 CUs at once (512 tiles = 128 of the large ones): measured, the large tile is 15-30 %
    // faster from 144 tiles on and 5-10 % slower at 128, for K from 1024 to 8192.
    bool big = many_big_tiles(M, N, K, b_nt);
    // (few tiles: the large tile again with every tile's K loop split, where that is cheaper)
    SmallPlan small{0, 0, 1};
    if (!big || !dtl_ok || env_switches().gemm_tile == 128) {
        small = plan_small(M, N, K, b_nt, n_peers, plain, dtl_ok, has_workspace, has_workspace && !has_gather && env_switches().gemm_tile != 128);
        if (small.big && gemm_dtl_tail_workspace_bytes((int)big_tiles_of(M, N, small.big), small.splits, small.big) > workspace_bytes)
            small = plan_small(M, N, K, b_nt, n_peers, plain, dtl_ok, has_workspace, false);
        big = small.big != 0;
    }
    // KRAKEN_AMD_GEMM_TILE=128|256 overrides the choice (testing and tuning)
    if (env_switches().gemm_tile == 128) big = false;
    if (env_switches().gemm_tile == 256) big = true;
    const bool dtl = big && dtl_ok;
    p.tile = dtl ? 256 : 128;
    // KRAKEN_AMD_GEMM_PEERS=epilogue keeps the peers' partial sums out of the matrix cores
    // (they are then added in the epilogue, where a non-finite value stays in its element)
    // K no multiple of the k-step: always in the epilogue, which is where every kernel that takes such shapes
    // adds them (the matrix cores would turn the 16 columns around an Inf into NaN)
    p.peers_on_mfma = K % 64 == 0;
    if (env_switches().gemm_peers >= 0 && K % 64 == 0) p.peers_on_mfma = env_switches().gemm_peers;
    // MFMA block shape of the 256x256 kernel: 16x16x32 draws less power per flop than 32x32x16 and
    // the chip is power-limited (k loop 5-10 % faster with warm operands; results agree to fp32
    // rounding), and its peer phase takes two peers per MFMA.  KRAKEN_AMD_GEMM_MFMA=16|32 overrides.
    p.mi16 = 1;
    if (env_switches().gemm_mfma > 0) p.mi16 = env_switches().gemm_mfma == 16;
    const int bm = p.tile;
    const int64_t tiles_m = (M + bm - 1) / bm, tiles_n = (N + bm - 1) / bm;
    // Column panels per scheduling group: the tiles an XCD runs at a time form a block that is
    // group_n panels wide.  8 measured best for the compute-bound shapes; where most tiles also
    // stream the peers' partial sums (HBM-bound), 16 lets neighbouring CUs read longer runs of
    // the same rows at about the same time.
    // (transposed-contiguous B: 4 measured 1-3 % ahead of 8 on 8192x3584x8192 and on the K = 16384
    // shapes with N = 6656, level elsewhere; row-major B: 8 and 4 level)
    p.group_n = (n_peers > 0 && band_rows * 2 >= M) ? 16 : (b_nt ? 4 : 8);
    // Rows that arrive while the kernel runs: narrow groups, so that the range of tiles each XCD
    // walks spans all row blocks in the order of their arrival (every XCD then starts on the
    // local shard and waits little); with wide groups the XCDs that own the last blocks idle
    // until those have arrived.
    // The same for row bands that are flagged as they complete: every XCD then moves from band to
    // band in the order of the destinations, and a band is complete once all eight have passed it
    // (with wide groups every band would only be complete when the last group is).
    if (flagged) p.group_n = (int)((tiles_n + kXcds - 1) / kXcds);
    if (const int v = env_switches().gemm_group; v >= 1 && v <= 64) p.group_n = v;
    // 256x256 kernel: the last partial round of tiles, split over the idle CUs (workspace given)
    p.tail_tiles = 0;
    p.tail_splits = 1;
    if (dtl && small.big) {
        p.n224 = small.big == 224;
        p.tail_tiles = (int)big_tiles_of(M, N, small.big);
        p.tail_splits = small.splits;
    } else if (dtl && has_workspace && !has_progress && (p.mi16 || (M % 256 == 0 && N % 256 == 0 && K % 64 == 0))) {
        int tail, ts;
        tail_split_plan(tiles_m * tiles_n, K, &tail, &ts);
        if (tail > 0 && gemm_dtl_tail_workspace_bytes(tail, ts) <= workspace_bytes) {
            p.tail_tiles = tail;
            p.tail_splits = ts;
        }
    }
    // 256x224 tiles: a plain product (no peers, bias, band or second output; bf16 result, which the
    // caller vouches for) with transposed-contiguous B whose columns 224 divides, when that tiling
    // needs fewer column-units of work than 256-column tiles rounded up to whole rounds of the
    // 256 compute units (8192 x 3584: 448 tiles = 2 rounds of 256 columns against 512 tiles = 2
    // rounds of 224: measured 340 -> 320 us at K = 8192); a 224-column tile costs about 3 % more
    // per flop (A is read from LDS and L2 for fewer columns).  KRAKEN_AMD_GEMM_N224=0|1 overrides.
    // (An A that arrives while the kernel runs is fine: the tile waits for its rows' flags before its
    // first load, whatever its width.)
    // (Not where few tiles share their K loops: one round of whole ones leaves most of the chip idle, 256 x 7168 x 12928
    // 213 us, 77 on 128x128 tiles in parts.)
    if (dtl && !small.big && p.mi16 && b_nt && plain && plain_bf16_all_rows && M % 256 == 0 && N % 224 == 0 && K % 64 == 0) {
        const int64_t t8 = tiles_m * tiles_n, t7 = (M / 256) * (N / 224);
        const double cost8 = (double)((t8 + 255) / 256) * 256.0, cost7 = (double)((t7 + 255) / 256) * 224.0 * 1.03;
        bool use = cost7 < cost8;
        if (env_switches().gemm_n224 >= 0) use = env_switches().gemm_n224 != 0;
        if (use) {
            p.n224 = 1;
            p.tail_tiles = 0;
            p.tail_splits = 1;
        }
    }
    // Split K loop (128x128 kernels, workspace given): S workgroups share a tile's K loop and meet in the workspace.
    p.splits = 1;
    if (!dtl) {
        p.ks = small.ks;
        p.splits = small.splits;
        if (p.splits > 1 && split_k_workspace_bytes(M, N, p.splits) > workspace_bytes) p.splits = 1;
    }
    return p;
}

// fp32 operands split in registers (gemm_f32.hip): 128x128 tiles, S workgroups per tile by the same kind of model
// as plan_small: 7 us to start and finish, 0.9 us per step of 64 k and round of 256 workgroups.  These choose the parts, they
// do not give the time: 256 workgroups in one pass measure 1.6 us per step and 13.5 us outside the k loop with row-major B, 1.45
// and 12 with transposed B, three peers 1 to 2 us more than one (1000 x 4096, K = 512 .. 4096: 26.9, 38.5, 64.2, 118.5 us).
static int split_f32(int64_t M, int64_t N, int64_t K) {
    const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128), steps = (K + 63) / 64;
    if (const int v = env_switches().gemm_splitk; v >= 1 && v <= kMaxSplits) return (int)std::min<int64_t>(v, steps);   // testing and tuning
    auto cost = [&](int64_t s) {
        return 700 + (tiles * s + 255) / 256 * 90 * ((steps + s - 1) / s) + (s > 1 ? 600 + s * M * N * 16 / 100000 : 0);
    };
    int best = 1;
    for (int s = 2; s <= kMaxSplits && 2 * s <= steps && s * tiles <= 512; ++s)
        if (cost(s) < cost(best)) best = s;
    return best;
}
static GemmPlan plan_gemm_f32(int64_t M, int64_t N, int64_t K, bool b_nt, int n_peers, int64_t band_rows, int64_t workspace_bytes,
                              bool skinny_ok) {
    GemmPlan p{};
    if (skinny_ok) {
        const SkinnyPlan sk = plan_skinny(M, N, K, b_nt, 4, workspace_bytes);
        if (sk.cb != 0) return plan_of_skinny(sk);
    }
    p.tile = 128;
    p.group_n = (n_peers > 0 && band_rows * 2 >= M) ? 16 : (b_nt ? 4 : 8);
    if (const int v = env_switches().gemm_group; v >= 1 && v <= 64) p.group_n = v;
    p.tail_splits = 1;
    p.splits = split_f32(M, N, K);
    if (p.splits > 1 && split_k_workspace_bytes(M, N, p.splits) > workspace_bytes) p.splits = 1;
    return p;
}

// Everything kr_gemm_reduce_noalloc_bf16 would otherwise do on its first call on a device: loads
// the library's code for the current device (a lazily loaded code object is what allocates the
// device memory of the scratch array) and looks the array up.
extern "C" int kr_init(void) {
    if (hipError_t e = load_gemm_dtl(); e != hipSuccess) return (int)e;
    if (hipError_t e = load_gemm_ks(); e != hipSuccess) return (int)e;
    if (hipError_t e = load_gemm_skinny(); e != hipSuccess) return (int)e;
    void* p = nullptr;
    return static_scratch(&p);
}

// What the kernel exchanges with other streams while it runs (null pointer to gemm_reduce:
// nothing): the arrival flags of the all-gather matmul (progress == nullptr: A is complete) and
// the per-band counters of the producer GEMM (band_counter == nullptr: none).
struct GatherSpec {
    const void* a_local;
    int64_t lda_local;
    int64_t local_row0, local_rows;
    const uint32_t* progress;
    int64_t comm_rows;
    int64_t wait_limit_us;
    int* status;
    uint32_t* band_counter;
    uint32_t* band_signal;
    int64_t count_rows;
    const void* const* shards;   // gather inside the product: the W shards (comm_rows rows each) and the gathered matrix
    int n_shards;
    void* gather_out;
};

// Everything of the entry points except the peers: argument checks in the documented
// order, then tile choice and launch.  `peers_given` is the stacked base or the table.
static int gemm_reduce(const void* A, int64_t lda_m, int64_t lda_k, const void* B, int64_t ldb_k, int64_t ldb_n,
                       int64_t M, int64_t N, int64_t K, const void* peers_given, int n_peers,
                       const void* const* peer_ptrs, int64_t peers_stride, const void* bias,
                       int64_t band_row0, int64_t band_rows, void* c_full, void* out, int out_is_fp32,
                       int64_t tile_pivot, void* stream, const GatherSpec* gather = nullptr,
                       void* workspace = nullptr, int64_t workspace_bytes = 0, bool static_ws = false, bool f32 = false) {
    if (M < 0 || N < 0 || K < 0 || M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x7fffffffLL)
        return KR_ERR_BAD_DIM;
    if (n_peers < 0 || n_peers >= KR_MAX_WORLD) return KR_ERR_WORLD_SIZE;
    if (band_row0 < 0 || band_rows < 0 || band_row0 + band_rows > M) return KR_ERR_BAND;
    if (K % 8 != 0 || N % 8 != 0) return KR_ERR_NUMEL_MOD8;
    if (M == 0 || N == 0) return KR_OK;
    if (K == 0) return KR_ERR_BAD_DIM;
    if (A == nullptr || B == nullptr) return KR_ERR_NULL_POINTER;
    if (band_rows > 0 && out == nullptr) return KR_ERR_NULL_POINTER;
    if (n_peers > 0 && peers_given == nullptr) return KR_ERR_NULL_POINTER;
    if (lda_k != 1) return KR_ERR_LAYOUT;
    const bool b_nt = (ldb_k == 1 && (ldb_n != 1 || N == 1));
    if (!b_nt && ldb_n != 1) return KR_ERR_LAYOUT;
    const int64_t ldb = b_nt ? ldb_n : ldb_k;
    if (lda_m < K || (b_nt ? ldb < K : ldb < N)) return KR_ERR_LAYOUT;
    if (lda_m % (f32 ? 4 : 8) != 0 || ldb % (f32 ? 4 : 8) != 0) return KR_ERR_ALIGNMENT;
    if (!aligned16(A) || !aligned16(B) || !aligned16(bias) || !aligned16(c_full) || !aligned16(out))
        return KR_ERR_ALIGNMENT;
    // (arguments are checked; a shape that is split now gets the library's own workspace)
    if (static_ws && kr_gemm_workspace_bytes(M, N, K) > KR_STATIC_SCRATCH_BYTES) return KR_ERR_SCRATCH;
    if (static_ws && kr_gemm_workspace_bytes(M, N, K) > 0) {
        const int rc = static_scratch(&workspace);
        if (rc != KR_OK) return rc;
        workspace_bytes = KR_STATIC_SCRATCH_BYTES;
    }

    GemmArgs g;
    if (peer_ptrs != nullptr) {
        // separate allocations: a table of n_peers device pointers
        const int rc = n_peers > 0 ? peer_tab_from_ptrs(g.peer, peer_ptrs, n_peers) : KR_OK;
        if (rc != KR_OK) return rc;
        if (n_peers == 0) peer_tab_stacked(g.peer, A, 0, 0);
    } else {
        if (peers_stride % 8 != 0 || !aligned16(peers_given)) return KR_ERR_ALIGNMENT;
        if (n_peers > 0 && peers_stride < band_rows * N) return KR_ERR_BAD_DIM;
        peer_tab_stacked(g.peer, n_peers > 0 ? peers_given : A, n_peers, peers_stride);
    }
    g.A = (const uint16_t*)A;
    g.B = (const uint16_t*)B;
    g.lda = lda_m;
    g.ldb = ldb;
    g.M = (int)M; g.N = (int)N; g.K = (int)K;
    g.n_peers = n_peers;
    g.progress = nullptr;
    g.comm_rows = 1;
    g.a_local = nullptr;
    g.lda_local = 0;
    g.local_row0 = g.local_rows = 0;
    g.wait_ticks = 0;
    g.status = nullptr;
    if (gather != nullptr && gather->progress != nullptr) {
        g.progress = gather->progress;
        g.comm_rows = (int)gather->comm_rows;
        g.a_local = (const uint16_t*)gather->a_local;
        g.lda_local = gather->lda_local;
        g.local_row0 = (int)gather->local_row0;
        g.local_rows = (int)gather->local_rows;
        g.wait_ticks = (uint64_t)gather->wait_limit_us * 100u;   // 100 MHz constant clock
        g.status = gather->status;
    }
    g.band_counter = nullptr;
    g.band_signal = nullptr;
    g.count_rows = 1;
    if (gather != nullptr && gather->band_counter != nullptr) {
        g.band_counter = gather->band_counter;
        g.band_signal = gather->band_signal;
        g.count_rows = (int)gather->count_rows;
    }
    g.gather_out = nullptr;
    if (gather != nullptr && gather->shards != nullptr) {
        if (const int rc = peer_tab_from_ptrs(g.peer, gather->shards, gather->n_shards); rc != KR_OK) return rc;
        g.gather_out = (uint16_t*)gather->gather_out;
        g.comm_rows = (int)gather->comm_rows;
    }
    g.bias = (const uint16_t*)bias;
    g.band_row0 = (int)band_row0;
    g.band_rows = (int)band_rows;
    g.c_full = (uint16_t*)c_full;
    g.out = out;
    g.out_is_fp32 = out_is_fp32;
    g.out_fp8 = 0;

    // gemm_skinny_kernel addresses both operands and the band with 32-bit byte offsets
    const int64_t esize = f32 ? 4 : 2;
    const bool skinny_ok = M <= 64 && (M * lda_m + K + 64) * esize < 0x7fffffffLL && M * N * 2 < 0x7fffffffLL &&
                           (b_nt ? 64 * ldb + K + 64 : (K + 64) * ldb + N) * esize < 0x7fffffffLL;
    const GemmPlan plan = f32 ? plan_gemm_f32(M, N, K, b_nt, n_peers, band_rows, workspace != nullptr ? workspace_bytes : 0, skinny_ok)
                              : plan_gemm(M, N, K, b_nt, n_peers, band_rows, n_peers == 0 && c_full == nullptr && bias == nullptr,
                                    !out_is_fp32 && band_row0 == 0 && band_rows == M, workspace != nullptr, workspace_bytes, gather != nullptr, g.progress != nullptr,
                                    g.progress != nullptr || g.band_counter != nullptr,
                                    gemm_dtl_supported(g) && (g.a_local == nullptr || (int64_t)256 * g.lda_local * 2 < 0x7fffffffLL), skinny_ok);
    const bool dtl = plan.tile == 256;
    if (g.gather_out != nullptr && !dtl) return KR_ERR_BAD_DIM;   // (kr_gather_matmul_direct says which shapes)
    // The 128x128 kernels address a tile's operand panels with 32-bit byte offsets from the
    // panel's first row (through a 2 GiB buffer descriptor): row strides beyond that reach are
    // refused rather than read as zeros.  (gemm_skinny_kernel, which has fewer rows, would reach
    // further; the rule does not depend on the number of rows.)
    if (!dtl) {
        const int64_t reach = std::max<int64_t>(std::max(lda_m, ldb), g.a_local != nullptr ? g.lda_local : 0);
        if ((128 * reach + std::max(K, N)) * (f32 ? 4 : 2) >= 0x7fffffffLL) return KR_ERR_LAYOUT;
    }
    g.peers_on_mfma = plan.peers_on_mfma;
    g.mi16 = plan.mi16 || g.gather_out != nullptr;
    g.n224 = plan.n224;
    const int bm = plan.tile, bn = plan.n224 ? 224 : bm;
    g.tiles_m = (int)((M + bm - 1) / bm);
    g.tiles_n = (int)((N + bn - 1) / bn);
    if ((int64_t)g.tiles_m * g.tiles_n > 0x7fffffffLL) return KR_ERR_BAD_DIM;
    g.group_n = plan.group_n;
    g.k_splits = 1;
    g.split_out_stride = 0;
    g.tail_tiles = 0;
    if (plan.tail_tiles > 0) {
        if (!aligned16(workspace)) return KR_ERR_ALIGNMENT;
        g.tail_tiles = plan.tail_tiles;
        g.k_splits = plan.tail_splits;
    }
    const int splits = plan.splits;
    if (splits > 1 && !aligned16(workspace)) return KR_ERR_ALIGNMENT;
    int64_t pt = tile_pivot / bm;
    g.pivot_tiles = (int)(((pt % g.tiles_m) + g.tiles_m) % g.tiles_m);
    // 256-row tiles with a band: the band's tiles as a region of their own at the head of the order, dealt to all XCDs, the others behind
    // them.  In one order the band lies with one to four of the XCDs, whose compute units are then the last to get to the tiles beyond the
    // first round: us, one order / two regions, 6144 x 3072 x 2048 (288 tiles, one peer) 102.5 / 86.0, 3000 x 3000 x 600 37.6 / 34.9,
    // 7392 x 5056 x 896 (580 tiles, seven peers) 96.0 / 78.6, 8192 x 4096 x 1024 with one peer 72.7 / 63.6.  An XCD then works on two sets of
    // panels at first, which a long K does not win back: 8192 x 8192 x 3584 343 / 352, 5000 x 5000 x 5000 234 / 242, 4600 x 6000 x 4096
    // 192 / 186, 7360 x 3328 x 3072 155 / 134.
    g.band_tile0 = g.band_tile_rows = 0;
    if (dtl && n_peers > 0 && band_rows > 0 && band_rows < M && K <= 3328) {
        const int64_t r0 = band_row0 / bm, rows = (band_row0 + band_rows + bm - 1) / bm - r0;
        if (rows < g.tiles_m && rows * g.tiles_n + g.tail_tiles <= (int64_t)g.tiles_m * g.tiles_n) {
            g.band_tile0 = (int)r0;
            g.band_tile_rows = (int)rows;
        }
    }
    const bool even = (M % bm == 0 && N % bn == 0 && K % BK == 0);
    if (splits > 1) {
        // pass 1: S partial products, fp32, no epilogue work; pass 2: sum + epilogue
        GemmArgs g1 = g;
        g1.k_splits = splits;
        g1.split_out_stride = M * N;
        g1.out = workspace;
        g1.out_is_fp32 = 1;
        g1.n_peers = 0;
        g1.bias = nullptr;
        g1.band_row0 = 0;
        g1.band_rows = (int)M;
        g1.c_full = nullptr;
        hipError_t e = plan.skinny ? launch_gemm_skinny(g1, b_nt, f32 ? 4 : 2, plan.skinny, (hipStream_t)stream)
                       : f32 ? launch_gemm_f32(g1, b_nt, (hipStream_t)stream)
                       : plan.ks ? launch_gemm_ks(g1, b_nt, (hipStream_t)stream) : launch_gemm<128, 128, 2, 2>(g1, b_nt, even, (hipStream_t)stream);
        if (e != hipSuccess) return (int)e;
        return (int)launch_splitk_finish(g, workspace, splits, (hipStream_t)stream);
    }
    hipError_t e = plan.skinny ? launch_gemm_skinny(g, b_nt, f32 ? 4 : 2, plan.skinny, (hipStream_t)stream)
                       : f32 ? launch_gemm_f32(g, b_nt, (hipStream_t)stream)
                       : dtl ? launch_gemm_dtl(g, b_nt, (hipStream_t)stream, workspace)
                       : plan.ks ? launch_gemm_ks(g, b_nt, (hipStream_t)stream)
                       : launch_gemm<128, 128, 2, 2>(g, b_nt, even, (hipStream_t)stream);
    return (int)e;
}

extern "C" int kr_gemm_reduce_bf16(const void* A, int64_t lda_m, int64_t lda_k, const void* B, int64_t ldb_k,
                                   int64_t ldb_n, int64_t M, int64_t N, int64_t K, const void* peers,
                                   int n_peers, int64_t peers_stride, const void* bias, int64_t band_row0,
                                   int64_t band_rows, void* c_full, void* out, int out_is_fp32,
                                   int64_t tile_pivot, void* stream) {
    return gemm_reduce(A, lda_m, lda_k, B, ldb_k, ldb_n, M, N, K, peers, n_peers, nullptr, peers_stride, bias,
                       band_row0, band_rows, c_full, out, out_is_fp32, tile_pivot, stream);
}

extern "C" int kr_gemm_reduce_ptrs_bf16(const void* A, int64_t lda_m, int64_t lda_k, const void* B,
                                        int64_t ldb_k, int64_t ldb_n, int64_t M, int64_t N, int64_t K,
                                        const void* const* peers, int n_peers, const void* bias,
                                        int64_t band_row0, int64_t band_rows, void* c_full, void* out,
                                        int out_is_fp32, int64_t tile_pivot, void* stream) {
    // an empty table with n_peers == 0 is a plain GEMM; the flag below still selects the table path
    static const void* const kNoPeers[1] = {nullptr};
    return gemm_reduce(A, lda_m, lda_k, B, ldb_k, ldb_n, M, N, K, peers, n_peers,
                       peers != nullptr ? peers : kNoPeers, 0, bias, band_row0, band_rows, c_full, out,
                       out_is_fp32, tile_pivot, stream);
}

extern "C" int kr_all_gather_matmul_bf16(const void* A, int64_t lda_m, const void* A_local, int64_t lda_local,
                                         const void* B, int64_t ldb_k, int64_t ldb_n, int64_t M, int64_t N,
                                         int64_t K, int W, int rank, int splits_per_rank,
                                         const uint32_t* progress, int64_t wait_limit_us, int32_t* status,
                                         void* C, void* stream) {
    if (W < 1 || W > KR_MAX_WORLD) return KR_ERR_WORLD_SIZE;
    if (rank < 0 || rank >= W || splits_per_rank < 1) return KR_ERR_STRIPE;
    if (M < 0 || M % ((int64_t)W * splits_per_rank) != 0) return KR_ERR_BAND;
    if (A_local != nullptr && (!aligned16(A_local) || lda_local % 8 != 0)) return KR_ERR_ALIGNMENT;
    if (A_local != nullptr && lda_local < K) return KR_ERR_LAYOUT;
    if ((reinterpret_cast<uintptr_t>(progress) & 3u) != 0 || (reinterpret_cast<uintptr_t>(status) & 3u) != 0)
        return KR_ERR_ALIGNMENT;
    GatherSpec gs{};
    gs.a_local = A_local;
    gs.lda_local = lda_local;
    gs.local_rows = M / W;
    gs.local_row0 = gs.local_rows * rank;
    gs.progress = progress;
    gs.comm_rows = M > 0 ? M / ((int64_t)W * splits_per_rank) : 1;
    gs.wait_limit_us = wait_limit_us > 0 ? wait_limit_us : 5000000;   // 5 s
    gs.status = status;
    // no reduce: the band is every row, no peers, no bias; tile order rotated to the local shard
    return gemm_reduce(A, lda_m, 1, B, ldb_k, ldb_n, M, N, K, nullptr, 0, nullptr, 0, nullptr, 0, M, nullptr, C, 0,
                       gs.local_row0, stream, &gs);
}

// Rows gathered by the product itself: shapes with enough tiles for one-pass workgroups of 256 rows, each inside one shard.
// us, copies on a side stream with tiles that wait for their flags / a gather launch in front of the product / this form,
// W = 2, 4 and 8, 136 to 448 tiles, K = 1024 to 16384 (72 shapes): this form 0.31 to 0.99 of the first.  Of the second 0.82 to 0.95
// at K = 1024 and 0.84 to 0.98 at K = 4096 and 8192 (8 x 512 x 4096, N = 4096 155 / 115 / 101; 8 x 1024 x 8192, N = 3584
// 404 / 369 / 345), but for 257 to 352 tiles from K = 4096 on, 0.95 to 1.38: a product with a workspace splits its last round
// (8 x 512, N = 4352: K = 4096 220 / 142 / 170, 8192 366 / 243 / 320, 16384 682 / 465 / 639); at K = 16384 and other counts
// 0.97 to 1.16 (8 x 1024, N = 1280 481 / 390 / 454).
extern "C" int kr_gather_matmul_direct(int W, int64_t rows_per_shard, int64_t N, int64_t K) {
    if (W < 1 || W > KR_MAX_WORLD || rows_per_shard <= 0 || rows_per_shard % 256 != 0 || rows_per_shard > 0x7fffffffLL / W) return 0;
    if (N <= 0 || N > 0x7fffffffLL || K > 0x7fffffffLL || K % 8 != 0 || N % 8 != 0) return 0;
    GemmArgs g{};
    g.K = (int)K;
    g.lda = g.ldb = K;
    if (!gemm_dtl_supported(g) || env_switches().gemm_tile == 128) return 0;
    return many_big_tiles(W * rows_per_shard, N, K, true) ? 1 : 0;
}

extern "C" int kr_gather_matmul_bf16(const void* const* shards, int W, int rank, int64_t rows_per_shard, void* A_out, const void* B,
                                     int64_t ldb, int64_t N, int64_t K, void* C, void* stream) {
    if (W < 1 || W > KR_MAX_WORLD) return KR_ERR_WORLD_SIZE;
    if (rank < 0 || rank >= W) return KR_ERR_STRIPE;
    if (shards == nullptr || A_out == nullptr) return KR_ERR_NULL_POINTER;
    if (!aligned16(A_out)) return KR_ERR_ALIGNMENT;
    if (!kr_gather_matmul_direct(W, rows_per_shard, N, K)) return KR_ERR_BAD_DIM;
    GatherSpec gs{};
    gs.comm_rows = rows_per_shard;
    gs.shards = shards;
    gs.n_shards = W;
    gs.gather_out = A_out;
    const int64_t M = W * rows_per_shard;
    return gemm_reduce(shards[0], K, 1, B, 1, ldb, M, N, K, nullptr, 0, nullptr, 0, nullptr, 0, M, nullptr, C, 0,
                       rank * rows_per_shard, stream, &gs);
}

extern "C" int kr_gemm_producer_bf16(const void* A, int64_t lda_m, int64_t lda_k, const void* B, int64_t ldb_k,
                                     int64_t ldb_n, int64_t M, int64_t N, int64_t K, void* C, int W, int rank,
                                     uint32_t* progress, uint32_t* signal_pad, void* stream) {
    if (W < 1 || W > KR_MAX_WORLD) return KR_ERR_WORLD_SIZE;
    if (rank < 0 || rank >= W) return KR_ERR_BAND;
    if (M < 0 || M % W != 0) return KR_ERR_BAD_DIM;
    if (progress == nullptr || signal_pad == nullptr || (M > 0 && N > 0 && C == nullptr)) return KR_ERR_NULL_POINTER;
    if ((reinterpret_cast<uintptr_t>(progress) & 3u) != 0 || (reinterpret_cast<uintptr_t>(signal_pad) & 3u) != 0)
        return KR_ERR_ALIGNMENT;
    GatherSpec ps{};
    ps.band_counter = progress;
    ps.band_signal = signal_pad;
    ps.count_rows = M > 0 ? M / W : 1;
    // no reduce band: every row of C goes to `C`; tile order rotated to the band of rank + 1
    return gemm_reduce(A, lda_m, lda_k, B, ldb_k, ldb_n, M, N, K, nullptr, 0, nullptr, 0, nullptr, 0, 0, C, nullptr,
                       0, ((int64_t)(rank + 1) % W) * (M / W), stream, &ps);
}

// Product of fp8 (e4m3fn) operands on the fp8 matrix-core instruction (all_gather_matmul.py:53,121,213: fp8 shards and
// weight, fp8 result).  The kernel is the 256x256 LDS-DMA kernel with its k-step on 16x16x128 blocks; it reads the operands
// as matrices of two-byte units, hence the halved K and row strides below.  `gather`: rows of A that arrive while the
// kernel runs (flags, local shard), as for the bf16 all-gather matmul.  whole_tiles: the entry points
// that take whole tiles only.
static int gemm_fp8(const void* A, int64_t lda, const void* Bt, int64_t ldb, int64_t M, int64_t N, int64_t K,
                    void* out, int out_kind, void* stream, const GatherSpec* gather, bool whole_tiles,
                    void* workspace = nullptr, int64_t workspace_bytes = 0) {
    if (M < 0 || N < 0 || K < 0 || M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x7fffffffLL) return KR_ERR_BAD_DIM;
    if (out_kind < 0 || out_kind > 2) return KR_ERR_BAD_DIM;
    if (whole_tiles ? (M % 256 != 0 || N % 256 != 0 || K % 128 != 0) : (N % 16 != 0 || K % 16 != 0 || (K > 0 && K < 128)))
        return KR_ERR_BAD_DIM;
    if (M == 0 || N == 0) return KR_OK;
    if (K == 0) return KR_ERR_BAD_DIM;
    if (A == nullptr || Bt == nullptr || out == nullptr) return KR_ERR_NULL_POINTER;
    if (lda < K || ldb < K) return KR_ERR_LAYOUT;
    if (lda % 16 != 0 || ldb % 16 != 0 || !aligned16(A) || !aligned16(Bt) || !aligned16(out)) return KR_ERR_ALIGNMENT;
    GemmArgs g{};
    peer_tab_stacked(g.peer, A, 0, 0);
    g.A = (const uint16_t*)A;
    g.B = (const uint16_t*)Bt;
    g.lda = lda / 2;
    g.ldb = ldb / 2;
    g.M = (int)M; g.N = (int)N; g.K = (int)(K / 2);
    g.comm_rows = 1;
    g.count_rows = 1;
    int64_t pivot_row = 0;
    if (gather != nullptr && gather->progress != nullptr) {
        g.progress = gather->progress;
        g.comm_rows = (int)gather->comm_rows;
        g.a_local = (const uint16_t*)gather->a_local;
        g.lda_local = gather->lda_local / 2;
        g.local_row0 = (int)gather->local_row0;
        g.local_rows = (int)gather->local_rows;
        g.wait_ticks = (uint64_t)gather->wait_limit_us * 100u;   // 100 MHz constant clock
        g.status = gather->status;
    }
    if (gather != nullptr) pivot_row = gather->local_row0;
    if (!gemm_dtl_supported(g) || (g.a_local != nullptr && (int64_t)256 * g.lda_local * 2 >= 0x7fffffffLL)) return KR_ERR_LAYOUT;
    g.band_row0 = 0;
    g.band_rows = (int)M;
    g.out = out;
    g.out_is_fp32 = out_kind == 1;
    g.out_fp8 = out_kind == 2;
    g.tiles_m = (int)((M + 255) / 256);
    g.tiles_n = (int)((N + 255) / 256);
    g.pivot_tiles = (int)((pivot_row / 256) % g.tiles_m);
    g.group_n = env_switches().gemm_group > 0 ? env_switches().gemm_group : 4;
    g.k_splits = 1;
    g.mi16 = 1;
    if (workspace != nullptr && g.progress == nullptr) {
        if (!aligned16(workspace)) return KR_ERR_ALIGNMENT;
        int tail, ts;
        fp8_split_plan(M, N, K, &tail, &ts);
        if (tail > 0 && gemm_dtl_tail_workspace_bytes(tail, ts) <= workspace_bytes) {
            g.tail_tiles = tail;
            g.k_splits = ts;
        }
    }
    return (int)launch_gemm_dtl8(g, (hipStream_t)stream, workspace);
}

extern "C" int kr_gemm_fp8(const void* A, int64_t lda, const void* Bt, int64_t ldb, int64_t M, int64_t N, int64_t K,
                           void* out, int out_kind, void* stream) {
    return gemm_fp8(A, lda, Bt, ldb, M, N, K, out, out_kind, stream, nullptr, true);
}

extern "C" int64_t kr_gemm_fp8_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K < 128) return 0;
    int tail, ts;
    fp8_split_plan(M, N, K, &tail, &ts);
    return tail > 0 ? gemm_dtl_tail_workspace_bytes(tail, ts) : 0;
}

extern "C" int kr_gemm_fp8_ws(const void* A, int64_t lda, const void* Bt, int64_t ldb, int64_t M, int64_t N, int64_t K,
                              void* out, int out_kind, void* workspace, int64_t workspace_bytes, void* stream) {
    return gemm_fp8(A, lda, Bt, ldb, M, N, K, out, out_kind, stream, nullptr, false, workspace, workspace_bytes);
}

// At most 64 rows: gemm_skinny_kernel, which reads B once, where 256-row tiles work for rows that are not there: 0.25 to 0.9 of
// their time over 4 to 64 rows, N = 1152 to 7488, K = 1088 to 13248, and the form plan_skinny picks the best of them or level with it.
static SkinnyPlan plan_skinny_fp8(int64_t M, int64_t N, int64_t K, int64_t parts_bytes) {
    if (env_switches().gemm_w8 >= 0) return SkinnyPlan{0, 1};   // (testing and tuning of the other)
    return plan_skinny(M, N, K, true, 1, parts_bytes);
}

// The same product with sums of 24 bits: the operands are widened to bf16 on their way to the matrix cores (gemm_w8.hip).
static int gemm_fp8_wide(const void* A, int64_t lda, const void* Bt, int64_t ldb, int64_t M, int64_t N, int64_t K, void* out,
                         int64_t tile_pivot, void* workspace, int64_t workspace_bytes, void* stream) {
    if (M < 0 || N < 0 || K < 0 || M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x7fffffffLL) return KR_ERR_BAD_DIM;
    if (N % 16 != 0 || K % 16 != 0) return KR_ERR_BAD_DIM;
    // (an operand with elements has to be aligned whether or not there is a product)
    if (K > 0 && ((M > 0 && !aligned16(A)) || (N > 0 && !aligned16(Bt)))) return KR_ERR_ALIGNMENT;
    if (M == 0 || N == 0) return KR_OK;
    if (K == 0) return KR_ERR_BAD_DIM;
    if (A == nullptr || Bt == nullptr || out == nullptr) return KR_ERR_NULL_POINTER;
    if (lda < K || ldb < K) return KR_ERR_LAYOUT;
    if (lda % 16 != 0 || ldb % 16 != 0 || !aligned16(A) || !aligned16(Bt) || !aligned16(out) || !aligned16(workspace)) return KR_ERR_ALIGNMENT;
    // (a tile's panels are addressed with 32-bit byte offsets from their first row)
    if (256 * std::max(lda, ldb) >= 0x7fffffffLL) return KR_ERR_LAYOUT;
    GemmArgs g{};
    peer_tab_stacked(g.peer, A, 0, 0);
    g.A = (const uint16_t*)A;
    g.B = (const uint16_t*)Bt;
    g.lda = lda / 2;
    g.ldb = ldb / 2;
    g.M = (int)M; g.N = (int)N; g.K = (int)(K / 2);
    g.comm_rows = 1;
    g.count_rows = 1;
    g.band_rows = (int)M;
    g.out = out;
    g.out_fp8 = 1;
    g.mi16 = 1;
    if (M * lda + K + 128 < 0x7fffffffLL && 64 * ldb + K + 128 < 0x7fffffffLL && M * N * 2 < 0x7fffffffLL) {
        if (const SkinnyPlan sk = plan_skinny_fp8(M, N, K, workspace != nullptr ? workspace_bytes : 0); sk.cb != 0) {
            g.lda = lda;
            g.ldb = ldb;
            g.K = (int)K;
            g.k_splits = sk.splits;
            if (sk.splits == 1) return (int)launch_gemm_skinny(g, true, 1, sk.cb, (hipStream_t)stream);
            GemmArgs parts = g;
            parts.out = workspace;
            parts.out_fp8 = 0;
            parts.out_is_fp32 = 1;
            parts.split_out_stride = M * N;
            if (hipError_t e = launch_gemm_skinny(parts, true, 1, sk.cb, (hipStream_t)stream); e != hipSuccess) return (int)e;
            return (int)launch_splitk_finish(g, workspace, sk.splits, (hipStream_t)stream);
        }
    }
    const W8Plan p = plan_w8(M, N, K, workspace != nullptr, workspace_bytes);
    g.tiles_m = (int)((M + 255) / 256);
    g.wide_panels = p.panels;
    g.tiles_n = p.panels + (p.nb2 > 0 ? (int)((N - 256 * (int64_t)p.panels + 32 * p.nb2 - 1) / (32 * p.nb2)) : 0);
    if ((int64_t)g.tiles_m * g.tiles_n > 0x7fffffffLL) return KR_ERR_BAD_DIM;
    g.pivot_tiles = (int)(((tile_pivot / 256) % g.tiles_m + g.tiles_m) % g.tiles_m);
    g.group_n = env_switches().gemm_group > 0 ? env_switches().gemm_group : 4;
    g.k_splits = p.splits;
    if (p.splits > 1) g.tail_tiles = g.tiles_m * g.tiles_n;
    return (int)launch_gemm_w8(g, p.nb2, (hipStream_t)stream, workspace);
}

extern "C" int64_t kr_gemm_fp8_wide_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const SkinnyPlan sk = plan_skinny_fp8(M, N, K, kMaxPartsBytes);
    const W8Plan p = plan_w8(M, N, K, true, kMaxPartsBytes);
    // (strides beyond the reach of gemm_skinny_kernel, which are not known here, take the other)
    return std::max<int64_t>(sk.cb != 0 && sk.splits > 1 ? split_k_workspace_bytes(M, N, sk.splits) : 0, p.splits > 1 ? ((M + 255) / 256) * ((N + 255) / 256) * p.splits * (256 * 256 * 4) : 0);
}

extern "C" int kr_gemm_fp8_wide_ws(const void* A, int64_t lda, const void* Bt, int64_t ldb, int64_t M, int64_t N, int64_t K,
                                   void* out, int64_t tile_pivot, void* workspace, int64_t workspace_bytes, void* stream) {
    return gemm_fp8_wide(A, lda, Bt, ldb, M, N, K, out, tile_pivot, workspace, workspace_bytes, stream);
}

static int all_gather_matmul_fp8(const void* A, int64_t lda, const void* A_local, int64_t lda_local, const void* Bt,
                                 int64_t ldb, int64_t M, int64_t N, int64_t K, int W, int rank, int splits_per_rank,
                                 const uint32_t* progress, int64_t wait_limit_us, int32_t* status, void* out,
                                 int out_kind, void* stream, bool whole_tiles) {
    if (W < 1 || W > KR_MAX_WORLD) return KR_ERR_WORLD_SIZE;
    if (rank < 0 || rank >= W || splits_per_rank < 1) return KR_ERR_STRIPE;
    if (M < 0 || M % ((int64_t)W * splits_per_rank) != 0) return KR_ERR_BAND;
    if (A_local != nullptr && (!aligned16(A_local) || lda_local % 16 != 0)) return KR_ERR_ALIGNMENT;
    if (A_local != nullptr && lda_local < K) return KR_ERR_LAYOUT;
    if ((reinterpret_cast<uintptr_t>(progress) & 3u) != 0 || (reinterpret_cast<uintptr_t>(status) & 3u) != 0)
        return KR_ERR_ALIGNMENT;
    GatherSpec gs{};
    gs.a_local = A_local;
    gs.lda_local = lda_local;
    gs.local_rows = M / W;
    gs.local_row0 = gs.local_rows * rank;
    gs.progress = progress;
    gs.comm_rows = M > 0 ? M / ((int64_t)W * splits_per_rank) : 1;
    gs.wait_limit_us = wait_limit_us > 0 ? wait_limit_us : 5000000;   // 5 s
    gs.status = status;
    return gemm_fp8(A, lda, Bt, ldb, M, N, K, out, out_kind, stream, &gs, whole_tiles);
}

extern "C" int kr_all_gather_matmul_fp8(const void* A, int64_t lda, const void* A_local, int64_t lda_local, const void* Bt,
                                        int64_t ldb, int64_t M, int64_t N, int64_t K, int W, int rank, int splits_per_rank,
                                        const uint32_t* progress, int64_t wait_limit_us, int32_t* status, void* out,
                                        int out_kind, void* stream) {
    return all_gather_matmul_fp8(A, lda, A_local, lda_local, Bt, ldb, M, N, K, W, rank, splits_per_rank, progress,
                                 wait_limit_us, status, out, out_kind, stream, true);
}

extern "C" int kr_all_gather_matmul_fp8_ragged(const void* A, int64_t lda, const void* A_local, int64_t lda_local, const void* Bt,
                                        int64_t ldb, int64_t M, int64_t N, int64_t K, int W, int rank, int splits_per_rank,
                                        const uint32_t* progress, int64_t wait_limit_us, int32_t* status, void* out,
                                        int out_kind, void* stream) {
    return all_gather_matmul_fp8(A, lda, A_local, lda_local, Bt, ldb, M, N, K, W, rank, splits_per_rank, progress,
                                 wait_limit_us, status, out, out_kind, stream, false);
}

extern "C" int kr_gemm_plan(int64_t M, int64_t N, int64_t K, int b_transposed, int n_peers, int64_t band_rows,
                            int has_bias, int has_c_full, int64_t workspace_bytes, int32_t plan[8]) {
    if (plan == nullptr) return KR_ERR_NULL_POINTER;
    if (M <= 0 || N <= 0 || K <= 0 || M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x7fffffffLL) return KR_ERR_BAD_DIM;
    if (n_peers < 0 || n_peers >= KR_MAX_WORLD) return KR_ERR_WORLD_SIZE;
    if (band_rows < 0 || band_rows > M) return KR_ERR_BAND;
    // contiguous operands: the only other input of the choice is whether the 256-row panels stay
    // within the 2 GiB reach of a buffer descriptor
    GemmArgs g{};
    g.K = (int)K;
    g.lda = K;
    g.ldb = b_transposed ? K : N;
    const GemmPlan p = plan_gemm(M, N, K, b_transposed != 0, n_peers, band_rows, n_peers == 0 && !has_c_full && !has_bias,
                                 band_rows == M, workspace_bytes > 0, workspace_bytes, false, false, false, gemm_dtl_supported(g), true);
    const bool whole_band_peers = p.tile == 256 && n_peers > 0 && p.peers_on_mfma != 0;
    plan[0] = p.tile;
    plan[1] = (p.tile == 256 ? p.mi16 : p.ks || p.skinny) ? 16 : 32;   // MFMA block rows: 16x16x32 or 32x32x16
    plan[2] = p.splits;
    plan[3] = p.tail_tiles;
    plan[4] = p.tail_splits;
    plan[5] = p.group_n;
    plan[6] = whole_band_peers ? 1 : 0;
    plan[7] = (M % p.tile != 0 || N % (p.n224 ? 224 : p.tile) != 0 || K % 64 != 0) ? 1 : 0;
    if (p.n224) plan[7] |= 2;   // bit 1: 256 x 224 tiles
    if (p.skinny) plan[7] |= 4;   // bit 2: gemm_skinny_kernel
    if (p.ks) plan[7] |= 8;   // bit 3: gemm_ks_kernel
    return KR_OK;
}

extern "C" int64_t kr_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    // the large-tile kernel (same rule as the launch; strides are not known here)
    const int force_tile = env_switches().gemm_tile;
    bool big = ((M + 255) / 256) * ((N + 255) / 256) > 128 && K >= 256;
    if (force_tile == 128) big = false;
    if (force_tile == 256) big = true;
    const bool parts_forced = force_tile == 256 && env_switches().gemm_tailsplit > 0 && env_switches().gemm_mfma != 32 && big_tiles_of(M, N, 256) <= 128;
    if (big && K >= 64 && !parts_forced) {
        int tail, ts;
        tail_split_plan(((M + 255) / 256) * ((N + 255) / 256), K, &tail, &ts);
        return tail > 0 ? gemm_dtl_tail_workspace_bytes(tail, ts) : 0;
    }
    // the layout of B and the number of peers are not known here: enough for any
    int64_t bytes = 0;
    for (int form = 0; form < 8; ++form) {
        const bool b_nt = form & 1, plain = (form >> 1) == 0;
        const int n_peers = (form >> 1) == 2 ? 1 : (form >> 1) == 3 ? 2 : 0;
        if (const SkinnyPlan sk = plan_skinny(M, N, K, b_nt, 2, kMaxPartsBytes); sk.cb != 0) {
            if (sk.splits > 1) bytes = std::max(bytes, split_k_workspace_bytes(M, N, sk.splits));
            continue;
        }
        const SmallPlan p = plan_small(M, N, K, b_nt, n_peers, plain, K % 8 == 0 && K >= 64, true, force_tile != 128);
        if (p.big) {
            bytes = std::max(bytes, gemm_dtl_tail_workspace_bytes((int)big_tiles_of(M, N, p.big), p.splits, p.big));
        } else if (p.splits > 1) {
            bytes = std::max(bytes, split_k_workspace_bytes(M, N, p.splits));
        }
    }
    return bytes;
}

extern "C" int kr_gemm_reduce_ws_bf16(const void* A, int64_t lda_m, int64_t lda_k, const void* B, int64_t ldb_k,
                                      int64_t ldb_n, int64_t M, int64_t N, int64_t K, const void* peers,
                                      int n_peers, int64_t peers_stride, const void* bias, int64_t band_row0,
                                      int64_t band_rows, void* c_full, void* out, int out_is_fp32,
                                      int64_t tile_pivot, void* workspace, int64_t workspace_bytes,
                                      void* stream) {
    return gemm_reduce(A, lda_m, lda_k, B, ldb_k, ldb_n, M, N, K, peers, n_peers, nullptr, peers_stride, bias,
                       band_row0, band_rows, c_full, out, out_is_fp32, tile_pivot, stream, nullptr, workspace,
                       workspace_bytes);
}

extern "C" int kr_gemm_reduce_ptrs_ws_bf16(const void* A, int64_t lda_m, int64_t lda_k, const void* B,
                                           int64_t ldb_k, int64_t ldb_n, int64_t M, int64_t N, int64_t K,
                                           const void* const* peers, int n_peers, const void* bias,
                                           int64_t band_row0, int64_t band_rows, void* c_full, void* out,
                                           int out_is_fp32, int64_t tile_pivot, void* workspace,
                                           int64_t workspace_bytes, void* stream) {
    static const void* const kNoPeers[1] = {nullptr};
    return gemm_reduce(A, lda_m, lda_k, B, ldb_k, ldb_n, M, N, K, peers, n_peers,
                       peers != nullptr ? peers : kNoPeers, 0, bias, band_row0, band_rows, c_full, out,
                       out_is_fp32, tile_pivot, stream, nullptr, workspace, workspace_bytes);
}

extern "C" int64_t kr_gemm_f32_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    int64_t skinny_bytes = 0;
    bool skinny = false;
    for (const bool b_nt : {false, true}) {
        const SkinnyPlan sk = plan_skinny(M, N, K, b_nt, 4, kMaxPartsBytes);
        skinny = sk.cb != 0;
        if (skinny && sk.splits > 1) skinny_bytes = std::max(skinny_bytes, split_k_workspace_bytes(M, N, sk.splits));
    }
    if (skinny) return skinny_bytes;
    const int S = split_f32(M, N, K);
    return S > 1 ? split_k_workspace_bytes(M, N, S) : 0;
}

extern "C" int kr_gemm_reduce_f32_ws(const void* A, int64_t lda_m, int64_t lda_k, const void* B, int64_t ldb_k,
                                     int64_t ldb_n, int64_t M, int64_t N, int64_t K, const void* const* peers,
                                     int n_peers, const void* bias, int64_t band_row0, int64_t band_rows,
                                     void* c_full, void* out, int out_is_fp32, int64_t tile_pivot, void* workspace,
                                     int64_t workspace_bytes, void* stream) {
    static const void* const kNoPeers[1] = {nullptr};
    return gemm_reduce(A, lda_m, lda_k, B, ldb_k, ldb_n, M, N, K, peers, n_peers,
                       peers != nullptr ? peers : kNoPeers, 0, bias, band_row0, band_rows, c_full, out,
                       out_is_fp32, tile_pivot, stream, nullptr, workspace, workspace_bytes, false, /*f32=*/true);
}

// fp32 operands as pairs (kPairs in gemm_dtl.hip): which tiles share their K loop.  A k-step of 32 takes 1.66 us with 192
// compute units busy and 1.9 with 256 (1.69 PFLOP/s), 64 MiB of parts 19 us to write, read and sum.
static void pairs_split_plan(int64_t M, int64_t N, int64_t K, int* tail_out, int* splits_out) {
    const int64_t tiles = big_tiles_of(M, N, 256), steps = (K + 31) / 32;
    *tail_out = 0;
    *splits_out = 1;
    const int64_t force = env_switches().gemm_tailsplit;   // 0: off, n: n parts (testing)
    if (force == 0) return;
    const int64_t tail = tiles <= 128 ? tiles : tiles % 256;
    if (tail == 0 || (tail > 128 && force <= 0)) return;
    int64_t best = 165 * steps;
    for (int64_t s = 2; s <= kMaxTailSplits && s * tail <= 256 && s * 4 <= steps; ++s) {
        if (force > 0 && s != force) continue;
        const int64_t c = 500 + 165 * ((steps + s - 1) / s) + gemm_dtl_tail_workspace_bytes((int)tail, (int)s) * 241 / 10000000;
        if (c >= best && force <= 0) continue;
        best = c;
        *tail_out = (int)tail;
        *splits_out = (int)s;
    }
}

// Pairs or the kernel that splits in registers (split_f32), in 0.01 us.  That one runs 256 tiles of 128x128 at a time: 17 us and
// 1.5 per round and 64 k.  Pairs take 4 us and the pass, 8 bytes per element of both operands at 5.2 TB/s, then 8 us
// (one pass 18, which also stores) and the k-steps, and the parts.  us, in registers / pairs, transposed and row-major B:
// 1316 x 3136 x 9280 431 / 260, 460 / 254 (275 tiles), x 3000 155 / 113, 162 / 109; 1000 x 4096 x 8192 224 / 218, 230 / 207,
// x 2048 64 / 85, 66 / 82; 2000 x 4096 x 2048 123 / 124, 128 / 122; 512 x 4096 x 8192 128 / 151, 129 / 145; 128 x 8192 x 8192
// 81 / 197.  Above 512 tiles, as a bf16 product of three times the K / pairs, three peers, transposed B: 4096 x 4096 x 2048 202 /
// 176, x 1024 113 / 104, 6000 x 6000 x 1024 281 / 246, 3000 x 8000 x 1536 255 / 233, 8192 x 2048 x 512 76 / 69.
extern "C" int kr_gemm_f32_pairs(int64_t M, int64_t N, int64_t K) {
    if (M <= 64 || N <= 0 || K <= 0 || M > 0x7fffffffLL || N > 0x7fffffffLL || K >= 1 << 20) return 0;   // (few rows: gemm_skinny_kernel)
    if (const int v = env_switches().gemm_pairs; v >= 0) return v;   // testing and tuning
    const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128);
    if (tiles > 512) return 1;
    const int64_t s = split_f32(M, N, K), k64 = (K + 63) / 64;
    const int64_t registers = 1700 + (tiles * s + 255) / 256 * 150 * ((k64 + s - 1) / s) + (s > 1 ? 600 + s * M * N * 16 / 100000 : 0);
    int tail, splits;
    pairs_split_plan(M, N, K, &tail, &splits);
    const int64_t big = big_tiles_of(M, N, 256), rounds = tail > 0 ? (big - tail) / 256 : (big + 255) / 256, k32 = (K + 31) / 32;
    const int64_t pairs = 400 + (M + N) * K * 8 / 52000 + (rounds > 0 ? 1800 : 800) + rounds * 190 * k32 +
                          (tail > 0 ? 300 + 190 * ((k32 + splits - 1) / splits) + gemm_dtl_tail_workspace_bytes(tail, splits) / 36000 : 0);
    return pairs < registers * 95 / 100;
}

extern "C" int64_t kr_gemm_pairs_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    int tail, splits;
    pairs_split_plan(M, N, K, &tail, &splits);
    return tail > 0 ? gemm_dtl_tail_workspace_bytes(tail, splits) : 0;
}

extern "C" int kr_gemm_reduce_pairs_ws(const void* A, const void* B, int64_t M, int64_t N, int64_t K, const void* const* peers, int n_peers,
                                       const void* bias, int64_t band_row0, int64_t band_rows, void* c_full, void* out, int out_is_fp32,
                                       int64_t tile_pivot, void* workspace, int64_t workspace_bytes, void* stream) {
    if (M < 0 || N < 0 || K < 0 || M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x3fffffffLL) return KR_ERR_BAD_DIM;
    if (n_peers < 0 || n_peers >= KR_MAX_WORLD) return KR_ERR_WORLD_SIZE;
    if (band_row0 < 0 || band_rows < 0 || band_row0 + band_rows > M) return KR_ERR_BAND;
    if (N % 8 != 0) return KR_ERR_NUMEL_MOD8;
    if (M == 0 || N == 0) return KR_OK;
    if (K == 0) return KR_ERR_BAD_DIM;
    if (A == nullptr || B == nullptr || (band_rows > 0 && out == nullptr) || (n_peers > 0 && peers == nullptr)) return KR_ERR_NULL_POINTER;
    if (!aligned16(A) || !aligned16(B) || !aligned16(bias) || !aligned16(c_full) || !aligned16(out) || !aligned16(workspace)) return KR_ERR_ALIGNMENT;
    GemmArgs g{};
    if (n_peers > 0) {
        if (const int rc = peer_tab_from_ptrs(g.peer, peers, n_peers); rc != KR_OK) return rc;
    } else {
        peer_tab_stacked(g.peer, A, 0, 0);
    }
    g.A = (const uint16_t*)A;
    g.B = (const uint16_t*)B;
    g.M = (int)M; g.N = (int)N; g.K = (int)((K + 31) / 32 * 64);
    g.lda = g.ldb = g.K;
    if (!gemm_dtl_supported(g)) return KR_ERR_LAYOUT;
    g.n_peers = n_peers;
    g.comm_rows = 1;
    g.count_rows = 1;
    g.bias = (const uint16_t*)bias;
    g.band_row0 = (int)band_row0;
    g.band_rows = (int)band_rows;
    g.c_full = (uint16_t*)c_full;
    g.out = out;
    g.out_is_fp32 = out_is_fp32;
    g.tiles_m = (int)((M + 255) / 256);
    g.tiles_n = (int)((N + 255) / 256);
    if ((int64_t)g.tiles_m * g.tiles_n > 0x7fffffffLL) return KR_ERR_BAD_DIM;
    g.pivot_tiles = (int)(((tile_pivot / 256) % g.tiles_m + g.tiles_m) % g.tiles_m);
    g.group_n = n_peers > 0 && band_rows * 2 >= M ? 16 : 8;
    if (const int v = env_switches().gemm_group; v >= 1 && v <= 64) g.group_n = v;
    g.k_splits = 1;
    g.mi16 = 1;
    // Peers on the matrix cores spread a value that is not finite over 16 columns: only where the bf16 product of three times
    // the K does so too (many_big_tiles: 3 K from 256 on).  (In the epilogue 4096 x 4096 x 1024 takes 107 us with one peer, so 101.)
    const bool many = ((M + 127) / 128) * ((N + 127) / 128) > 512 && 3 * K >= 256;
    g.peers_on_mfma = K % 64 != 0 ? 0 : env_switches().gemm_peers >= 0 ? env_switches().gemm_peers : many;
    int tail, splits;
    pairs_split_plan(M, N, K, &tail, &splits);
    if (tail > 0 && workspace != nullptr && gemm_dtl_tail_workspace_bytes(tail, splits) <= workspace_bytes) {
        g.tail_tiles = tail;
        g.k_splits = splits;
    }
    return (int)launch_gemm_pairs(g, (hipStream_t)stream, workspace);
}

extern "C" int kr_gemm_reduce_noalloc_bf16(const void* A, int64_t lda_m, int64_t lda_k, const void* B,
                                           int64_t ldb_k, int64_t ldb_n, int64_t M, int64_t N, int64_t K,
                                           const void* peers, int n_peers, int64_t peers_stride,
                                           const void* bias, int64_t band_row0, int64_t band_rows,
                                           void* c_full, void* out, int out_is_fp32, int64_t tile_pivot,
                                           void* stream) {
    return gemm_reduce(A, lda_m, lda_k, B, ldb_k, ldb_n, M, N, K, peers, n_peers, nullptr, peers_stride, bias,
                       band_row0, band_rows, c_full, out, out_is_fp32, tile_pivot, stream, nullptr, nullptr, 0,
                       /*static_ws=*/true);
}

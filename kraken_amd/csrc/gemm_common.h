// Pieces shared by the GEMM kernels: argument block, tile schedule, fused epilogue.
#pragma once

#include <atomic>
#include <type_traits>

#include "common.h"

namespace kr {

struct GemmArgs {
    const uint16_t* A;
    const uint16_t* B;
    int64_t lda;   // elements between rows of A (k is contiguous)
    int64_t ldb;   // NT: elements between n-rows of B^T; NN: elements between k-rows of B
    int M, N, K;
    PeerTab peer;        // peer.p[j]: partial sums of peer j, [band_rows, N] bf16 (j < n_peers)
    int n_peers;
    const uint16_t* bias;
    int band_row0, band_rows;
    uint16_t* c_full;
    void* out;
    int out_is_fp32;
    int out_fp8;       // fp8 kernel only: the result is fp8 (e4m3fn), [M, N] bytes
    int pivot_tiles;   // rotation of the M-tile order
    int tiles_m, tiles_n;
    // all-gather matmul with arrival flags (progress == nullptr: A is complete, nothing waits)
    const uint32_t* progress;   // progress[b] == 1 once rows [b*comm_rows, (b+1)*comm_rows) of A have arrived
    int comm_rows;
    const uint16_t* a_local;    // this rank's own shard, rows [local_row0, local_row0+local_rows) of A: never waits
    int64_t lda_local;
    int local_row0, local_rows;
    uint64_t wait_ticks;        // bound of one tile's wait, in ticks of the 100 MHz constant clock
    int* status;                // set to 1 + block index by a tile whose wait ran out (may be nullptr)
    // gather inside the product (gather_out == nullptr: off): rows [r*comm_rows, (r+1)*comm_rows) of A are peer.p[r], and
    // the tiles write what they read to gather_out, [M, K] contiguous
    uint16_t* gather_out;
    // split K loop of the 128x128 kernel (k_splits == 1: off)
    int k_splits;               // workgroups per tile, each with its share of the k-steps (grid y)
    int64_t split_out_stride;   // elements between the fp32 outputs of consecutive splits (0: one output)
    // 256x256 kernel, split of the last partial round of tiles (tail_tiles == 0: off): the main
    // launch runs the first tiles_m*tiles_n - tail_tiles tiles of the schedule, a second launch
    // the remaining ones with k_splits workgroups per tile, a third sums the parts
    int tail_tiles;
    int wide_panels;     // gemm_w8_kernel: column panels of 256, the first of the tiles_n; the others are narrower
    int group_n;         // column panels per scheduling group (tile_schedule)
    int band_tile0, band_tile_rows;   // rows of tiles that touch the reduce band, ahead of all others (tile_of; 0 rows: one order)
    int peers_on_mfma;   // 256x256 kernel: add whole-band tiles' peers through the matrix cores
    int mi16;            // 256x256 kernel: k loop and peer phase on 16x16x32 MFMA blocks
    int n224;            // 256x224 tiles (tiles_n counts them), transposed-contiguous B: a plain product in whole rounds, or every tile in parts
    // producer of the copy-engine reduce-scatter (band_counter == nullptr: off): finished tiles are
    // counted per destination rank, whose band is count_rows rows of C
    uint32_t* band_counter;   // [M / count_rows] tiles finished that touch the band
    uint32_t* band_signal;    // [M / count_rows] set to 1 by the workgroup that finishes the band's last tile
    int count_rows;
};

// Opt a kernel into more than 64 KiB of dynamic LDS, once per device: the attribute belongs to the
// current device's copy of the code.  `done`: the call site's own bit mask of devices.
inline hipError_t lds_opt_in(const void* fn, int bytes, std::atomic<uint64_t>& done) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = 1ull << (dev & 63);
    if (done.load(std::memory_order_acquire) & bit) return hipSuccess;
    e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return e;
    done.fetch_or(bit, std::memory_order_release);
    return hipSuccess;
}

// LDS-DMA kernel with 256x256 tiles (gemm_dtl.hip)
bool gemm_dtl_supported(const GemmArgs& g);
hipError_t launch_gemm_dtl(const GemmArgs& g, bool b_nt, hipStream_t st, void* workspace);
hipError_t launch_gemm_dtl8(const GemmArgs& g, hipStream_t st, void* workspace);   // fp8 operands (gemm_dtl.hip)
hipError_t launch_gemm_pairs(const GemmArgs& g, hipStream_t st, void* workspace);  // fp32 operands as pairs of bf16 parts (gemm_dtl.hip)
hipError_t launch_tail_finish(const GemmArgs& g, hipStream_t st, const void* workspace);   // sums the parts of split 256x256 tiles
hipError_t launch_gemm_w8(const GemmArgs& g, int nb2, hipStream_t st, void* workspace);   // fp8 operands widened to bf16 (gemm_w8.hip)

hipError_t launch_gemm_ks(const GemmArgs& g, bool b_nt, hipStream_t st);           // 128x128 tiles, k divided between waves (gemm_ks.hip)
hipError_t launch_gemm_f32(const GemmArgs& g, bool b_nt, hipStream_t st);          // fp32 operands (gemm_f32.hip); A, B, lda, ldb in fp32 elements
hipError_t launch_gemm_skinny(const GemmArgs& g, bool b_nt, int esize, int cb, hipStream_t st);   // at most 64 rows, 16 cb columns per workgroup (gemm_skinny.hip)
hipError_t load_gemm_dtl();
hipError_t load_gemm_ks();
hipError_t load_gemm_skinny();

typedef int i32x4 __attribute__((ext_vector_type(4)));
// raw buffer descriptor: 48-bit base, stride 0, num_records bytes, 32-bit data format
__device__ __forceinline__ i32x4 raw_rsrc(const void* base, int64_t bytes) {
    const uint64_t b = (uint64_t)base;
    return i32x4{(int)(uint32_t)b, (int)((b >> 32) & 0xffff), (int)(bytes < 0x7fffffff ? (bytes > 0 ? bytes : 0) : 0x7fffffff), 0x00020000};
}
// One wave-wide LDS-DMA load: lane l's 16 bytes at (descriptor base + voff + soff) go to lds_addr + 16 l; past the
// descriptor's end zeros are written.  Inline assembly on purpose: the compiler then does not know that LDS is written
// behind its back and leaves the ordering to explicit s_waitcnt vmcnt / s_barrier pairs.
__device__ __forceinline__ void lds_dma_b128(i32x4 rsrc, uint32_t lds_addr, uint32_t voff, int soff) {
    // (one wait state between the scalar write of M0 and the instruction that reads it)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory", "m0");
}

constexpr int kXcds = 8;

// A operand of the tile that starts at row m0 (bm rows), for the all-gather matmul: rows arrive
// in blocks of g.comm_rows while the kernel runs, each block's flag in g.progress set to 1 by a
// stream-ordered write behind its copy (kraken/fused/all_gather_matmul.py:95-110: a tile of
// the local shard reads the shard itself, any other tile waits for its block's flag).  Called by
// every wave of the workgroup: each polls the flags of the blocks the tile covers with
// device-scope loads and a short sleep, then an acquire fence orders its own loads behind the
// flag (so no workgroup barrier is needed); the wait is bounded (g.wait_ticks): a tile whose flag does not come records
// 1 + block in g.status and goes on (its result is then meaningless), and later tiles see
// the status and do not wait at all, so the grid always drains.
__device__ __forceinline__ void gathered_a_tile(const GemmArgs& g, int m0, int bm, const uint16_t*& a_tile,
                                                int64_t& lda) {
    a_tile = g.A + (int64_t)m0 * g.lda;
    lda = g.lda;
    if (g.progress == nullptr) return;
    const int m1 = min(m0 + bm, g.M);
    if (g.a_local != nullptr && m0 >= g.local_row0 && m1 <= g.local_row0 + g.local_rows) {
        a_tile = g.a_local + (int64_t)(m0 - g.local_row0) * g.lda_local;
        lda = g.lda_local;
        return;
    }
    const int b_hi = (m1 - 1) / g.comm_rows;
    const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
    bool give_up = g.status != nullptr && __hip_atomic_load(g.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    for (int b = m0 / g.comm_rows; b <= b_hi && !give_up; ++b) {
        while (__hip_atomic_load(g.progress + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 1u) {
            if (__builtin_amdgcn_s_memrealtime() - t0 > g.wait_ticks) {
                give_up = true;
                if (g.status != nullptr) __hip_atomic_store(g.status, b + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
            __builtin_amdgcn_s_sleep(16);
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
}

// a value every lane of the wave holds, moved to scalar registers
__device__ __forceinline__ int64_t wave_uniform(int64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Position in the tile order of workgroup `wg` of a launch over the first `count` tiles.
// Workgroups are dealt round-robin to the 8 XCDs (each with its own L2), so workgroup ids are
// re-numbered to give every XCD a contiguous range of the order: XCD x owns positions
// [x * ntiles/8, (x+1) * ntiles/8) and a launch over fewer tiles takes the first count/8 of each
// range (`first` skips positions an earlier launch has taken).  Where 8 does not divide the count, the
// first ntiles % 8 XCDs own one position more (launches over all tiles), or the range is that of the launch over the
// first ntiles - tail_tiles, which is a multiple of 256, and the tiles behind it follow in order.
// (the plain form: a launch over all of `ntiles`)
__device__ __forceinline__ int xcd_position(int wg, int ntiles) {
    const int x = wg % kXcds;
    return x * (ntiles / kXcds) + min(x, ntiles % kXcds) + wg / kXcds;
}
__device__ __forceinline__ int schedule_position(const GemmArgs& g, int wg, int first = 0) {
    const int ntiles = g.tiles_m * g.tiles_n;
    if (ntiles % kXcds != 0 && (g.tail_tiles == 0 || g.tail_tiles == ntiles)) return xcd_position(wg, ntiles);
    if (ntiles % kXcds != 0 && first == 0) return xcd_position(wg, ntiles - g.tail_tiles);
    if (ntiles % kXcds != 0 || first % kXcds != 0) return first + wg;
    return (wg % kXcds) * (ntiles / kXcds) + first / kXcds + wg / kXcds;
}

// Map a position in the tile order to its tile (tile_m, tile_n).
__device__ __forceinline__ void tile_in_order(int pid, int tiles_m, int tiles_n, int group_n, int pivot_tiles, int& tile_m_out, int& tile_n_out) {
    // ---- tile schedule -------------------------------------------------------------------
    // Tiles are ordered in groups of group_n column panels, M fastest in steps of group_n
    // columns: the ~32 tiles an XCD runs at a time form a (32 / group_n) x group_n block that
    // shares its A and B panels through the XCD's L2 (a dozen panels for 32 tiles), and every
    // XCD works on all row bands -- the rows of the reduce band (whose tiles also stream the
    // peers' partial sums) are spread over all XCDs instead of landing on one.  The M order is
    // rotated by the pivot, so the band's (or the local shard's) tiles are the first ones of
    // every XCD.
    const int per_group = group_n * tiles_m;
    const int group = pid / per_group;
    const int first_n = group * group_n;
    const int gsz = min(tiles_n - first_n, group_n);
    const int tile_n = first_n + (pid % per_group) % gsz;
    int tile_m = (pid % per_group) / gsz;
    tile_m += pivot_tiles;
    if (tile_m >= tiles_m) tile_m -= tiles_m;
    tile_m_out = tile_m;
    tile_n_out = tile_n;
}
__device__ __forceinline__ void tile_schedule(const GemmArgs& g, int pid, int& tile_m_out, int& tile_n_out) {
    tile_in_order(pid, g.tiles_m, g.tiles_n, g.group_n, g.pivot_tiles, tile_m_out, tile_n_out);
}

// Tile of workgroup `wg`; with `first` > 0 of a launch over the tiles from position `first` on.
__device__ __forceinline__ void tile_of(const GemmArgs& g, int wg, int first, int& tile_m, int& tile_n) {
    // (without branches around the choice: the compiler keeps the tile in scalar registers only so)
    const int tiles = g.tiles_m * g.tiles_n, band = g.band_tile_rows * g.tiles_n;
    const bool in_band = first == 0 && wg < band;
    const int row0 = in_band ? g.band_tile0 : band > 0 ? g.band_tile0 + g.band_tile_rows : g.pivot_tiles;
    const int rows = in_band ? g.band_tile_rows : g.tiles_m - g.band_tile_rows;
    const int pid = band == 0 ? schedule_position(g, wg, first)
                              : first > 0 ? first - band + wg : xcd_position(in_band ? wg : wg - band, in_band ? band : tiles - g.tail_tiles - band);
    tile_in_order(pid, rows, g.tiles_n, g.group_n, 0, tile_m, tile_n);
    tile_m += row0;
    if (tile_m >= g.tiles_m) tile_m -= g.tiles_m;
    tile_m = __builtin_amdgcn_readfirstlane(tile_m);
    tile_n = __builtin_amdgcn_readfirstlane(tile_n);
}

// Fused epilogue of one workgroup tile.  `acc` are this wave's 32x32 MFMA accumulators (TM x TN
// blocks) in the TRANSPOSED layout the kernels produce by passing the B fragment as the first
// MFMA operand: lane holds row (lane & 31) of the block, register v is column
// 8*(v/4) + 4*(lane>>5) + v%4 -- four consecutive columns per register quad, so a quad is one
// contiguous store into a row-major LDS patch.  `smem` is the workgroup's LDS (free for reuse:
// every wave has passed a barrier after its last read of the operand stages).
//
// F32 = false (bf16 result): the product is rounded to bf16 on its way into the patch, as the
// reference's reduce-scatter rounds a rank's partial product before the partials are summed
// (kraken/fused/gemm_reduce_scatter_fused.py:72, summed in fp32 at :118-145); partial sums of
// the peers and the bias are then added in fp32 in the order own, peer 0, 1, ..., bias.
// F32 = true (fp32 result: the reference's fused all-reduce keeps fp32 from the accumulator to
// the output, kraken/fused/gemm_one_shot_all_reduce_fused.py:65-99): the patch holds fp32.
//
// ACC is either f32x16[TM][TN] (32x32 MFMA blocks: lane l holds row l%32 of a block and the
// columns 8(v/4) + 4(l/32) + v%4 of register v) or f32x4[2*TM][2*TN] (16x16 blocks: lane l
// holds row l%16 and the columns 4(l/16) + v); only the copy into the patch knows which.
template <bool F32, int BM, int WTM, int WTN, int TM, int TN, bool EVEN, int EP_WAVE, class ACC>
__device__ __forceinline__ void gemm_epilogue_impl(const GemmArgs& g, const int n_peers, const uint16_t* bias,
                                                   const ACC& acc, unsigned char* smem,
                                                   int m0, int n0, int wm, int wn, int lane, int wave) {
    constexpr bool MI16 = std::is_same<ACC, f32x4[2 * TM][2 * TN]>::value;
    static_assert(MI16 || std::is_same<ACC, f32x16[TM][TN]>::value, "unknown accumulator layout");
    // After the barrier above no wave reads the pipeline stages any more, and from here on
    // every wave touches only its own LDS patch, so no further workgroup barrier is needed
    // (LDS requests of one wave are served in order).  Per 32-row slab the accumulators are
    // written to the patch and read back as row-contiguous 8-element chunks.
    //
    // Loads and stores share one in-order counter on this hardware: waiting for a load that
    // was issued after a store also waits until that store has been acknowledged by memory,
    // a round trip of thousands of cycles.  So nothing in the store path may depend on a
    // load issued behind a store: the bias is fetched once, before the first store, and the
    // partial sums of the other ranks are fetched one batch ahead (the loads of batch b+1 are
    // issued before the stores of batch b), so every wait leaves the younger stores pending.
    typedef typename std::conditional<F32, float, uint16_t>::type patch_t;
    // row pitch in elements: 16 bytes of padding keep the quad stores of 16 (bf16: 8-byte) or
    // 8 (fp32: 16-byte) lanes on distinct banks and the rows 16-byte aligned
    constexpr int LD = WTN + (F32 ? 4 : 8);
    static_assert(32 * LD * (int)sizeof(patch_t) <= EP_WAVE, "patch exceeds the wave's share of LDS");
    patch_t* patch = (patch_t*)(smem + wave * EP_WAVE);
    constexpr int CPR = WTN / 8;            // 8-element chunks per patch row
    constexpr int EP_ITERS = 32 * CPR / 64; // chunks per lane per 32-row slab
    constexpr int kChunkBatch = BM >= 256 ? 4 : 2;   // the small tile keeps its register count low (occupancy)
    constexpr int kPeerGroup = 4;           // peers fetched together by the generic path
    // a wave of an edge tile with no row or column in the matrix
    if (!EVEN && (__builtin_amdgcn_readfirstlane(m0 + wm * WTM) >= g.M || __builtin_amdgcn_readfirstlane(n0 + wn * WTN) >= g.N)) return;
    const int band_lo = g.band_row0, band_hi = g.band_row0 + g.band_rows;
    const int lane_r = lane / CPR, lane_cc = lane % CPR;   // chunk (it*64 + lane): row it*(64/CPR) + lane_r
    const int n = n0 + wn * WTN + lane_cc * 8;             // first of the lane's 8 columns, same for every chunk

    float bias_f[8];
    zero8(bias_f);
    const bool has_bias = bias != nullptr;
    if (has_bias) add8(*(const u32x4*)(bias + (EVEN ? n : min(n, g.N - 8))), bias_f);

    // Round-to-nearest-even pack of two fp32 to bf16, pinned where it is written: the
    // accumulators do not change inside the slab loop, so an ordinary conversion -- or, for
    // accumulators held in AGPRs, even just the copy to a VALU-readable register -- would be
    // hoisted out of it for all slabs at once, at the price of 128 or more live registers.
    auto pack_here = [](float lo, float hi) __attribute__((always_inline)) {
        uint32_t r;
        if constexpr (BM >= 256) {   // 256 accumulators: they live in AGPRs
            uint32_t t;
            asm volatile("v_accvgpr_read_b32 %0, %2\n\tv_accvgpr_read_b32 %1, %3\n\tv_cvt_pk_bf16_f32 %0, %0, %1"
                         : "=&v"(r), "=&v"(t)
                         : "a"(lo), "a"(hi));
        } else {
            asm volatile("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(lo), "v"(hi));
        }
        return r;
    };
    // copy of slab i's accumulators to the patch.  Accumulator registers can only be indexed
    // statically, hence the uniform if-chain inside a rolled slab loop.
    auto copy_slab = [&](int i) __attribute__((always_inline)) {
        patch_t* row = MI16 ? patch + (lane & 15) * LD + 4 * (lane >> 4) : patch + (lane & 31) * LD + 4 * (lane >> 5);
#pragma unroll
        for (int ii = 0; ii < TM; ++ii) {
            if (i == ii) {
                if constexpr (MI16) {
                    // slab = block rows 2i and 2i+1 (patch rows 0..15 and 16..31), 2*TN column blocks
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int j = 0; j < 2 * TN; ++j) {
                            const f32x4& a = acc[2 * ii + h][j];
                            if constexpr (F32) {
                                *(f32x4*)(row + h * 16 * LD + j * 16) = a;
                            } else {
                                typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                                *(u32x2*)(row + h * 16 * LD + j * 16) = u32x2{pack_here(a[0], a[1]), pack_here(a[2], a[3])};
                            }
                        }
                } else {
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const f32x16& a = acc[ii][j];
                        if constexpr (F32) {
                            *(f32x4*)(row + j * 32 + 8 * q) = f32x4{a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
                        } else {
                            typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                            *(u32x2*)(row + j * 32 + 8 * q) =
                                u32x2{pack_here(a[4 * q], a[4 * q + 1]), pack_here(a[4 * q + 2], a[4 * q + 3])};
                        }
                    }
                }
                // a distinct statement per case: identical case bodies would be merged into one
                // with a run-time accumulator index, which forces the accumulators into memory
                asm volatile("; accumulators of slab %0 copied" ::"n"(ii));
            }
        }
        // keep the scheduler from pulling the accumulator reads of later slabs (256 registers
        // in all) ahead of this point
        __builtin_amdgcn_sched_barrier(0);
    };
    // one chunk of the current slab: as stored (bf16 patch) or as fp32 values
    auto read_raw = [&](int chunk) __attribute__((always_inline)) {
        const int r = chunk * (64 / CPR) + lane_r;
        return *(const u32x4*)(patch + r * LD + lane_cc * 8);
    };
    auto read_chunk = [&](int chunk, float (&f)[8]) __attribute__((always_inline)) {
        if constexpr (F32) {
            const int r = chunk * (64 / CPR) + lane_r;
            const f32x4 lo = *(const f32x4*)(patch + r * LD + lane_cc * 8);
            const f32x4 hi = *(const f32x4*)(patch + r * LD + lane_cc * 8 + 4);
            f[0] = lo.x; f[1] = lo.y; f[2] = lo.z; f[3] = lo.w;
            f[4] = hi.x; f[5] = hi.y; f[6] = hi.z; f[7] = hi.w;
        } else {
            unpack8(read_raw(chunk), f);
        }
    };
    auto store_out = [&](int64_t off, const float (&f)[8]) __attribute__((always_inline)) {
        if constexpr (F32) {
            float* o = (float*)g.out + (int64_t)blockIdx.y * g.split_out_stride + off;
            *(f32x4*)o = f32x4{f[0], f[1], f[2], f[3]};
            *(f32x4*)(o + 4) = f32x4{f[4], f[5], f[6], f[7]};
        } else {
            st_stream((u32x4*)((uint16_t*)g.out + off), pack8(f));
        }
    };

    // the wave's first row, as a scalar: the classification below must branch uniformly
    const int wave_m0 = __builtin_amdgcn_readfirstlane(m0 + wm * WTM);

    // ---- up to seven peers, and the wave has rows of the band -----------------------------------
    // Straight-line batches of kBatch chunks, peer loads double-buffered one batch ahead across slab boundaries.  A chunk's
    // row goes to `out` or to c_full, lane by lane (edges of the matrix and of the band), and neither loads nor stores are
    // under a branch, where the waits could not count them: a lane outside the band loads a valid address, a peer that is not
    // there is one address of the first one for all lanes and is masked, and both stores go out, out of range where they are not meant.
    // (Four peers that read the last one four times: 2520 x 7232 x 1024 83.4 us, 700 x 4160 x 1024 with an fp32 result 22.7; so 80.7, 21.7.)
    // Tiles at the edges used to take the loads behind the stores, as below, also for rows outside the band, and held up the
    // others: 7392 x 5056 x 896 with a band and seven peers 128 -> 96 us, 2520 x 7232 x 1024 70.5 -> 51.6, 1448 x 2048 x 832
    // 20.5 -> 16.9, fp32 results 700 x 4160 x 1024 with one peer 20.1 -> 17.8.
    auto with_peers = [&](auto np_c) __attribute__((always_inline)) {
        constexpr int P = decltype(np_c)::value, kSure = P > 3 ? 4 : 1;   // peers that are there whatever the call
        constexpr int kBatch = (P <= 3 ? 2 : 1) * (BM >= 256 ? 2 : 1), kBatches = EP_ITERS / kBatch;
        static_assert(EP_ITERS % kBatch == 0 && kBatches % 2 == 0, "the two peer buffers alternate with a static parity");
        constexpr uint32_t kOob = 0x80000000u;
        constexpr int kEl = F32 ? 4 : 2;
        u32x4 pv[2][kBatch][P];
        const int row_out = max(wave_m0, band_lo);   // first row of the band in this wave
        const __amdgpu_buffer_rsrc_t out_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (char*)g.out + ((int64_t)blockIdx.y * g.split_out_stride + (int64_t)(row_out - band_lo) * g.N) * kEl, 0, 0x7fffffff, 0x00020000);
        const __amdgpu_buffer_rsrc_t full_rsrc =
            __builtin_amdgcn_make_buffer_rsrc(g.c_full + (int64_t)wave_m0 * g.N, 0, g.c_full != nullptr ? 0x7fffffff : 0, 0x00020000);
        const int64_t safe_off = min(n, g.N - 8);
        auto row_of = [&](int chunk_abs) __attribute__((always_inline)) { return wave_m0 + chunk_abs * (64 / CPR) + lane_r; };
        auto inside = [&](int m) __attribute__((always_inline)) { return m >= band_lo && m < band_hi && (EVEN || n < g.N); };
        auto issue = [&](auto buf_c, int chunk_abs) __attribute__((always_inline)) {
            constexpr int buf = decltype(buf_c)::value;
#pragma unroll
            for (int c = 0; c < kBatch; ++c) {
                const int m = row_of(chunk_abs + c);
                const int64_t off = inside(m) ? (int64_t)(m - band_lo) * g.N + n : safe_off;
#pragma unroll
                for (int q = 0; q < P; ++q) {
                    const bool there = q < kSure || q < n_peers;
                    pv[buf][c][q] = ld_stream((const u32x4*)((const uint16_t*)g.peer.p[there ? q : 0] + (there ? off : 0)));
                }
            }
        };
        issue(std::integral_constant<int, 0>{}, 0);
#pragma nounroll
        for (int i = 0; i < TM; ++i) {
            copy_slab(i);
            const int chunk0 = i * EP_ITERS;
#pragma unroll
            for (int b = 0; b < kBatches; ++b) {
                // (the very last batch re-fetches itself, unused)
                const int next_chunk = min(chunk0 + (b + 1) * kBatch, TM * EP_ITERS - kBatch);
                if (b & 1) issue(std::integral_constant<int, 0>{}, next_chunk);
                else issue(std::integral_constant<int, 1>{}, next_chunk);
                float f[kBatch][8];
                u32x4 product[kBatch];   // as c_full gets it
#pragma unroll
                for (int c = 0; c < kBatch; ++c) {
                    read_chunk(b * kBatch + c, f[c]);
                    product[c] = pack8(f[c]);
                }
#pragma unroll
                for (int c = 0; c < kBatch; ++c) {
#pragma unroll
                    for (int q = 0; q < P; ++q) {
                        const u32x4 v = pv[b & 1][c][q];
                        if (q < kSure) {
                            add8(v, f[c]);
                            continue;
                        }
                        const uint32_t keep = q < n_peers ? 0xffffffffu : 0u;
                        add8(u32x4{v.x & keep, v.y & keep, v.z & keep, v.w & keep}, f[c]);
                    }
#pragma unroll
                    for (int e = 0; e < 8; ++e) f[c][e] += bias_f[e];
                }
#pragma unroll
                for (int c = 0; c < kBatch; ++c) {
                    const int m = row_of(chunk0 + b * kBatch + c);
                    const bool in = inside(m), full = !in && (EVEN || (m < g.M && n < g.N));
                    const uint32_t o = in ? (uint32_t)(((m - row_out) * g.N + n) * kEl) : kOob;
                    const uint32_t q = full ? (uint32_t)(((m - wave_m0) * g.N + n) * 2) : kOob;
                    constexpr int kNt = 2;   // non-temporal
                    if constexpr (F32) {
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, f32x4{f[c][0], f[c][1], f[c][2], f[c][3]}), out_rsrc, o, 0, 0);
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, f32x4{f[c][4], f[c][5], f[c][6], f[c][7]}), out_rsrc, in ? o + 16 : kOob, 0, 0);
                    } else {
                        __builtin_amdgcn_raw_buffer_store_b128(pack8(f[c]), out_rsrc, o, 0, kNt);
                    }
                    __builtin_amdgcn_raw_buffer_store_b128(product[c], full_rsrc, q, 0, kNt);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // (the stores' offsets are 32 bits from the wave's first row)
    if (n_peers > 0 && n_peers <= 7 && wave_m0 < band_hi && wave_m0 + WTM > band_lo && (int64_t)WTM * g.N * 4 < 0x7fffffffLL) {
        if (n_peers > 3) with_peers(std::integral_constant<int, 7>{});
        else with_peers(std::integral_constant<int, 3>{});
        return;
    }

    // ---- every other case, one slab at a time ------------------------------------------------
    const bool whole = EVEN || (wave_m0 + WTM <= g.M && __builtin_amdgcn_readfirstlane(n0 + wn * WTN) + WTN <= g.N);
    // One batch of kChunkBatch chunks of the current slab.  NP == 0: every row of the slab lies
    // in the band (or below the matrix) and there are no peers; NP == -2: no row of the slab lies in the band (both
    // without loads); NP == -1: generic per-lane handling (band edge inside the slab, any peer count).
    auto slab_batch = [&](auto np_c, int slab_m0, int b0) __attribute__((always_inline)) {
        constexpr int NP = decltype(np_c)::value;
        int64_t off[kChunkBatch];
        bool in_band[kChunkBatch], valid[kChunkBatch];
#pragma unroll
        for (int c = 0; c < kChunkBatch; ++c) {
            const int m = slab_m0 + (b0 + c) * (64 / CPR) + lane_r;
            valid[c] = EVEN || (m < g.M && n < g.N);
            in_band[c] = NP == 0 ? valid[c] : NP == -2 ? false : (valid[c] && m >= band_lo && m < band_hi);
            off[c] = in_band[c] ? (int64_t)(m - band_lo) * g.N + n : (int64_t)m * g.N + n;
        }
        if constexpr (!F32 && NP != -1) {
            // nothing to add but perhaps the bias: the bf16 chunks go out as they are
            if (NP == -2 || !has_bias) {
                if (NP == 0 || g.c_full != nullptr) {
                    uint16_t* dst = NP == 0 ? (uint16_t*)g.out : g.c_full;
                    u32x4 raw[kChunkBatch];
#pragma unroll
                    for (int c = 0; c < kChunkBatch; ++c) raw[c] = read_raw(b0 + c);
                    if (whole) {
#pragma unroll
                        for (int c = 0; c < kChunkBatch; ++c) st_stream((u32x4*)(dst + off[c]), raw[c]);
                    } else {
#pragma unroll
                        for (int c = 0; c < kChunkBatch; ++c)
                            if (valid[c]) st_stream((u32x4*)(dst + off[c]), raw[c]);
                    }
                }
                return;
            }
        }
        float f[kChunkBatch][8];
#pragma unroll
        for (int c = 0; c < kChunkBatch; ++c) read_chunk(b0 + c, f[c]);
        if constexpr (NP == -1) {
            // Peers in groups of kPeerGroup, all loads of a group issued before its first add;
            // the groups are unrolled, each under one uniform test.  No load is predicated:
            // a chunk outside the band reads a valid in-band address instead, a peer index
            // past the last repeats the last peer, and such values are masked to +0.0 (loads
            // under branches would make every later load wait for the whole queue).
            const int64_t safe_off = min(n, g.N - 8);
#pragma unroll
            for (int q0 = 0; q0 < KR_MAX_WORLD - 1; q0 += kPeerGroup) {
                if (q0 < n_peers) {
                    u32x4 pv[kChunkBatch][kPeerGroup];
#pragma unroll
                    for (int c = 0; c < kChunkBatch; ++c)
#pragma unroll
                        for (int q = 0; q < kPeerGroup; ++q) {
                            const int qq = min(q0 + q, n_peers - 1);
                            pv[c][q] = ld_stream(
                                (const u32x4*)((const uint16_t*)g.peer.p[qq] + (in_band[c] ? off[c] : safe_off)));
                        }
#pragma unroll
                    for (int c = 0; c < kChunkBatch; ++c)
#pragma unroll
                        for (int q = 0; q < kPeerGroup; ++q) {
                            const uint32_t keep = (in_band[c] && q0 + q < n_peers) ? 0xffffffffu : 0u;
                            add8(u32x4{pv[c][q].x & keep, pv[c][q].y & keep, pv[c][q].z & keep, pv[c][q].w & keep}, f[c]);
                        }
                }
            }
        }
#pragma unroll
        for (int c = 0; c < kChunkBatch; ++c) {
            if (in_band[c]) {
#pragma unroll
                for (int e = 0; e < 8; ++e) f[c][e] += bias_f[e];
                store_out(off[c], f[c]);
            } else if (valid[c] && g.c_full != nullptr) {
                st_stream((u32x4*)(g.c_full + off[c]), pack8(f[c]));
            }
        }
    };

#pragma nounroll
    for (int i = 0; i < TM; ++i) {
        copy_slab(i);
        const int slab_m0 = wave_m0 + i * 32;
        const bool all_in = slab_m0 >= band_lo && (slab_m0 + 32 <= band_hi || (!EVEN && band_hi == g.M));
        const bool all_out = slab_m0 + 32 <= band_lo || slab_m0 >= band_hi;
#pragma unroll
        for (int b0 = 0; b0 < EP_ITERS; b0 += kChunkBatch) {
            if (all_out) {
                slab_batch(std::integral_constant<int, -2>{}, slab_m0, b0);
            } else if (all_in && n_peers == 0) {
                slab_batch(std::integral_constant<int, 0>{}, slab_m0, b0);
            } else {
                slab_batch(std::integral_constant<int, -1>{}, slab_m0, b0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// fp32 -> fp8 (e4m3fn) of two values into one half of a word: nearest even; magnitudes from 448 on
// (infinities included) give +-448, NaN stays NaN -- the conversion kr_cast_f32_to_fp8 defines.  The
// clamp is explicit, so the instruction's own overflow handling never comes into play.
template <bool HIGH_HALF>
__device__ __forceinline__ uint32_t pack2_e4m3(float a, float b, uint32_t old) {
    const float ca = __builtin_fminf(__builtin_fmaxf(a, -448.0f), 448.0f), cb = __builtin_fminf(__builtin_fmaxf(b, -448.0f), 448.0f);
    return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(a != a ? a : ca, b != b ? b : cb, (int)old, HIGH_HALF);
}

// eight consecutive values as fp8
__device__ __forceinline__ void store8_e4m3(uint8_t* p, const float (&f)[8]) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    *(u32x2*)p = u32x2{pack2_e4m3<true>(f[2], f[3], pack2_e4m3<false>(f[0], f[1], 0u)), pack2_e4m3<true>(f[6], f[7], pack2_e4m3<false>(f[4], f[5], 0u))};
}

// fp8 store of a wave's 128 x 16 NB part of a tile held as 8 x NB accumulator blocks of 16 x 16 (lane l:
// row l%16, columns 4(l/16) .. +3 of a block): per 16-row slab a lane's four values of a block become
// one word of a per-wave LDS patch [16][16 NB + 16] bytes (with NB = 8 the pad keeps the 64 word stores of a block on
// 64 banks), and the slab leaves as 16-byte chunks of whole rows.  `dst`: the wave's first
// row and column; ld in bytes.  MASKED: only the first `rows` rows and `cols` columns (a multiple of 16) exist.
template <int NB, bool MASKED>
__device__ __forceinline__ void store_tile_fp8_blocks(const f32x4 (&acc16)[8][NB], unsigned char* smem, uint8_t* dst, int64_t ld,
                                                      int lane, int wave, int rows, int cols) {
    constexpr int LD = NB * 16 + 16;
    static_assert(16 * LD <= 4096 && NB <= 8, "patch of a wave, two chunks per lane and slab");
    unsigned char* patch = smem + wave * 4096;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            // (pinned here: copies the compiler may hoist would keep all blocks' values alive at once)
            float x0, x1, x2, x3;
            asm volatile("v_accvgpr_read_b32 %0, %2\n\tv_accvgpr_read_b32 %1, %3" : "=&v"(x0), "=&v"(x1) : "a"(acc16[i][j][0]), "a"(acc16[i][j][1]));
            asm volatile("v_accvgpr_read_b32 %0, %2\n\tv_accvgpr_read_b32 %1, %3" : "=&v"(x2), "=&v"(x3) : "a"(acc16[i][j][2]), "a"(acc16[i][j][3]));
            const uint32_t w = pack2_e4m3<true>(x2, x3, pack2_e4m3<false>(x0, x1, 0u));
            *(uint32_t*)(patch + (lane & 15) * LD + 16 * j + 4 * (lane >> 4)) = w;
        }
        asm volatile("" ::: "memory");   // the reads below see the stores above (different types, same bytes)
#pragma unroll
        for (int it = 0; it < (16 * NB + 63) / 64; ++it) {
            const int idx = it * 64 + lane, r = idx / NB, c = idx % NB;
            if (16 * NB % 64 != 0 && idx >= 16 * NB) continue;
            const u32x4 v = *(const u32x4*)(patch + r * LD + c * 16);
            if (!MASKED || (16 * i + r < rows && c * 16 < cols)) st_stream((u32x4*)(dst + (int64_t)(16 * i + r) * ld + c * 16), v);
        }
        asm volatile("" ::: "memory");   // the next slab's stores stay behind these reads
    }
}

// Producer side of the copy-engine reduce-scatter, called by the whole workgroup once its tile
// (rows m0 .. m0+bm-1) is stored (kraken/fused/gemm_reduce_scatter_ce_persistent.py:117-132):
// the tile is counted into the counter of every destination rank whose band of g.count_rows rows
// it touches, and the workgroup whose count completes a band (all column tiles of all row tiles
// that overlap it) sets the band's flag, on which a stream-ordered wait in front of the band's
// copy is parked.  Order: every wave's stores are complete at the barrier; thread 0's release
// fence then writes them back to memory before its count becomes visible, and the workgroup that
// sees the last count acquires the others' before it publishes the flag.
__device__ __forceinline__ void count_finished_tile(const GemmArgs& g, int m0, int bm) {
    __syncthreads();
    if (threadIdx.x != 0) return;
    __atomic_thread_fence(__ATOMIC_RELEASE);   // system scope
    const int m_last = min(m0 + bm, g.M) - 1;
    for (int r = m0 / g.count_rows; r <= m_last / g.count_rows; ++r) {
        const int t_lo = (int)(((int64_t)r * g.count_rows) / bm);
        const int t_hi = (int)(((int64_t)(r + 1) * g.count_rows - 1) / bm);
        const uint32_t band_tiles = (uint32_t)(t_hi - t_lo + 1) * (uint32_t)g.tiles_n;
        const uint32_t before = __hip_atomic_fetch_add(g.band_counter + r, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (before + 1 == band_tiles) {
            __atomic_thread_fence(__ATOMIC_ACQ_REL);
            __hip_atomic_store(g.band_signal + r, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// n_peers and bias are what is still to be added here (a kernel that has already put the
// peers or the bias into the accumulators passes 0 / nullptr); g is only read, never copied,
// so the peer table stays in kernel-argument memory.
template <int BM, int WTM, int WTN, int TM, int TN, bool EVEN, int EP_WAVE, class ACC>
__device__ __forceinline__ void gemm_epilogue(const GemmArgs& g, int n_peers, const uint16_t* bias,
                                              const ACC& acc, unsigned char* smem,
                                              int m0, int n0, int wm, int wn, int lane, int wave) {
    if (g.out_is_fp32) gemm_epilogue_impl<true, BM, WTM, WTN, TM, TN, EVEN, EP_WAVE, ACC>(g, n_peers, bias, acc, smem, m0, n0, wm, wn, lane, wave);
    else gemm_epilogue_impl<false, BM, WTM, WTN, TM, TN, EVEN, EP_WAVE, ACC>(g, n_peers, bias, acc, smem, m0, n0, wm, wn, lane, wave);
    if (g.band_counter != nullptr) count_finished_tile(g, m0, BM);
}

}  // namespace kr

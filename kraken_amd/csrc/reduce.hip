// W-way elementwise reduce (+bias) over W bf16 buffers (the slices of a stacked tensor, or
// W separate allocations named by a pointer table).
//
// HBM-bound: per output vector of 8 elements the kernel reads W*16 B (+16 B of
// bias) and writes 16 B, i.e. (W+1)*2 bytes per element.  A workgroup walks the
// input in blocks of kThreads*kUnroll vectors (grid-stride, at most kMaxBlocks
// workgroups = 4 per CU: measured best on MI355X, 6.05 TB/s against 5.8 TB/s for
// one block per workgroup).  Every thread owns kUnroll 128-bit vectors that are
// kThreads vectors apart, so each wave-level load covers 1 KiB of consecutive
// addresses, and all W*kUnroll loads of a thread are issued before the first
// add (the adds keep the fixed order bias?, slice 0, 1, ... W-1, so the sum is
// reproducible bit for bit).  Loads and stores are non-temporal.
#include "common.h"

namespace kr {

constexpr int kThreads = 256;
constexpr int kMaxBlocks = 4 * 256;   // 4 workgroups per CU

enum BiasMode { kNoBias = 0, kFullBias = 1, kVectorBias = 2 };

// Adds buffers r0 .. r0+G-1 at the thread's kUnroll vectors to acc, in order; all G * kUnroll loads are issued
// before the first add.  at(r, u) loads vector u of buffer r.
template <int G, int kUnroll, class LOAD>
__device__ __forceinline__ void add_group(const LOAD& at, int r0, float (&acc)[kUnroll][8]) {
    u32x4 v[G][kUnroll];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) v[g][u] = at(r0 + g, u);
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)
#pragma unroll
        for (int g = 0; g < G; ++g) add8(v[g][u], acc[u]);
}

// The same for all W buffers of a run-time W: groups of eight, and what is left in one group of its size (the
// branches are uniform).  One buffer at a time is a chain of W round trips to memory: W = 16 on 1024 x 8192
// 48.2 -> 43.4 us, W = 3 on 4096 x 4096 24.1 -> 22.4, W = 6 on 1000 x 5120 15.3 -> 14.3.
template <int kUnroll, class LOAD>
__device__ __forceinline__ void add_all(const LOAD& at, int W, float (&acc)[kUnroll][8]) {
    int r = 0;
    for (; W - r >= 8; r += 8) add_group<8, kUnroll>(at, r, acc);
    switch (W - r) {
        case 1: add_group<1, kUnroll>(at, r, acc); break;
        case 2: add_group<2, kUnroll>(at, r, acc); break;
        case 3: add_group<3, kUnroll>(at, r, acc); break;
        case 4: add_group<4, kUnroll>(at, r, acc); break;
        case 5: add_group<5, kUnroll>(at, r, acc); break;
        case 6: add_group<6, kUnroll>(at, r, acc); break;
        case 7: add_group<7, kUnroll>(at, r, acc); break;
        default: break;
    }
}

// One block of kThreads * kUnroll vectors.  A block that is not FULL (the last one) reads the input's last vector
// wherever it runs past the end, so that its loads too are all in flight together, and stores what is inside.
template <class SRC, int WT, int BIAS, bool BIAS_FIRST, int kUnroll, bool FULL>
__device__ __forceinline__ void reduce_block(const SRC& src, int W, int64_t blk, int64_t nvec,
                                             const u32x4* __restrict__ bias, uint32_t d_vec, u32x4* __restrict__ out) {
    const int64_t base = blk * (kThreads * kUnroll) + threadIdx.x;
    int64_t idx[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
        idx[u] = base + (int64_t)u * kThreads;
        if (!FULL) idx[u] = idx[u] < nvec ? idx[u] : nvec - 1;
    }
    float acc[kUnroll][8];
    u32x4 bv[kUnroll];
    if (BIAS != kNoBias) {
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) bv[u] = BIAS == kFullBias ? ld_stream(bias + idx[u]) : bias[mod_vec(idx[u], d_vec)];
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)
        if (BIAS == kNoBias || !BIAS_FIRST) zero8(acc[u]);  // 0.0f, then += slice 0 (keeps the sign of a -0.0 sum as the reference has it)
    if constexpr (WT > 0) {
        u32x4 v[WT][kUnroll];
        if constexpr (SRC::kTable && FULL) {
            // separate buffers: each buffer's block through a descriptor (base = buffer +
            // block, in scalar registers), so all W buffers share one byte offset per (lane, u)
            constexpr uint32_t kBlockBytes = kThreads * kUnroll * 16;
#pragma unroll
            for (int r = 0; r < WT; ++r) {
                const __amdgpu_buffer_rsrc_t rs = stream_rsrc(src.at(r) + blk * (kThreads * kUnroll), kBlockBytes);
#pragma unroll
                for (int u = 0; u < kUnroll; ++u) v[r][u] = ld_stream(rs, (threadIdx.x + u * kThreads) * 16u);
            }
        } else {
#pragma unroll
            for (int r = 0; r < WT; ++r)
#pragma unroll
                for (int u = 0; u < kUnroll; ++u) v[r][u] = ld_stream(src.at(r) + idx[u]);
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            if (BIAS != kNoBias && BIAS_FIRST) unpack8(bv[u], acc[u]);
#pragma unroll
            for (int r = 0; r < WT; ++r) add8(v[r][u], acc[u]);
        }
    } else {
        if (BIAS != kNoBias && BIAS_FIRST) {
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) unpack8(bv[u], acc[u]);
        }
        add_all<kUnroll>([&](int r, int u) { return ld_stream(src.at(r) + idx[u]); }, W, acc);
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
        if (BIAS != kNoBias && !BIAS_FIRST) add8(bv[u], acc[u]);
        if (FULL || base + (int64_t)u * kThreads < nvec) st_stream(out + idx[u], pack8(acc[u]));
    }
}

// WT > 0: W known at compile time (loop fully unrolled); WT == 0: run-time W.
template <class SRC, int WT, int BIAS, bool BIAS_FIRST, int kUnroll>
__global__ __launch_bounds__(kThreads) void reduce_kernel(
    const SRC src, int w_rt, int64_t nvec,
    const u32x4* __restrict__ bias, uint32_t d_vec, u32x4* __restrict__ out) {
    const int W = WT > 0 ? WT : w_rt;
    for (int64_t blk = blockIdx.x; blk * (kThreads * kUnroll) < nvec; blk += gridDim.x) {
        if ((blk + 1) * (kThreads * kUnroll) <= nvec)
            reduce_block<SRC, WT, BIAS, BIAS_FIRST, kUnroll, true>(src, W, blk, nvec, bias, d_vec, out);
        else
            reduce_block<SRC, WT, BIAS, BIAS_FIRST, kUnroll, false>(src, W, blk, nvec, bias, d_vec, out);
    }
}

// Striped ownership: output vector j (compact) comes from input vector
//   (j / blk_v) * blk_v * W + rank * blk_v + (j % blk_v).
// One vector per thread in single-wave workgroups.  TOGETHER: all of a thread's loads are requested before the first add; one
// after the other they are a chain of W round trips to memory, which is what a share of up to some thousand
// workgroups takes (kernel time, W = 8, chain / together: 256 x 4096 6.0 / 2.35 us, 2047 x 5120 with a bias 7.6 / 5.7, 8000 x 5120 19.6 / 17.8).
// Above kChainVecs the chip is full of waves either way, and with W = 8 the chain keeps HBM a little busier (16384 x 8192 48.1 /
// 49.3; W = 4 and 2 level).  256 threads a workgroup are 1 to 3 % slower in both forms at 16384 rows.
// In between four and sixteen buffers, whose slices lie a power of two apart in many calls, are read faster by a chain in
// workgroups of 256 threads, from kTogetherVecs on: W = 4, 2^18, 2^19 and 2^20 vectors 5.5 us / 6.0 together, 8.6 / 9.9, 16.3 / 17.5,
// sizes that are no power of two 0.95 to 1.06; W = 16, half as many again (below it is slower), 2^19 and 2^20 23.9 / 25.9, 45.9 / 48.2.
// The mean over 256 k to 1 M vectors of together over chain with W = 6, 8, 9, 13: 0.97 to 1.00.
constexpr int64_t kTogetherVecs = 1 << 18, kChainVecs = 1 << 20;

template <class SRC, int WT, bool TOGETHER, int THREADS>
__global__ __launch_bounds__(THREADS) void reduce_striped_kernel(
    const SRC src, int w_rt, int64_t share_nvec,
    const u32x4* __restrict__ bias, uint32_t blk_v, int rank, u32x4* __restrict__ out) {
    const int W = WT > 0 ? WT : w_rt;
    const int64_t j = (int64_t)blockIdx.x * THREADS + threadIdx.x;
    if (j >= share_nvec) return;
    const int64_t stripe = j / blk_v;
    const int64_t i = (stripe * W + rank) * blk_v + (j - stripe * blk_v);
    float acc[1][8];
    zero8(acc[0]);
    u32x4 bv = {0, 0, 0, 0};
    if constexpr (TOGETHER) {
        if (bias != nullptr) bv = ld_stream(bias + i);
        add_all<1>([&](int r, int) { return ld_stream(src.at(r) + i); }, W, acc);
    } else if constexpr (THREADS == kWave) {
#pragma unroll 1
        for (int r = 0; r < W; ++r) add8(ld_stream(src.at(r) + i), acc[0]);
        if (bias != nullptr) bv = ld_stream(bias + i);
    } else {
        // (the first buffer in front of the loop and the loop left to the compiler: 1 to 5 % at these sizes)
        add8(ld_stream(src.at(0) + i), acc[0]);
        for (int r = 1; r < W; ++r) add8(ld_stream(src.at(r) + i), acc[0]);
        if (bias != nullptr) bv = ld_stream(bias + i);
    }
    if (bias != nullptr) add8(bv, acc[0]);
    st_stream(out + j, pack8(acc[0]));
}

// Rotated-order tile reduce of the copy-engine reduce-scatter variant:
// out[v] = sum_i band_{(i + rank + 1) % W}[v], optionally rounding
// the running sum to bf16 after every add.  Up to eight bands are requested together.  The bands are
// the slices of one tensor or buffers of their own (SRC, common.h), so what the other ranks sent is read where it is.
// W known at compile time and single-wave workgroups: no branch between the requests (kernel time, W = 8: 1 x 1600 2.6 -> 2.3 us,
// 18 x 1728 2.8 -> 2.5, 1024 x 4096 level, 1024 x 8192 28.4 -> 27.4).
// Bands of kRotatedWide to kRotatedFull vectors, W = 4 and 8, lie a power of two apart in many calls: workgroups of 256 threads (us, single
// waves / 256 threads, W = 8: 256 x 4096 5.9 / 4.8, 512 x 4096 9.15 / 8.4, 768 x 4096 11.7 / 10.9, 256 x 5120 5.5 / 5.6; W = 4 5.1 / 4.9 at
// 512 x 4096); above single waves again (W = 8, 1000 x 4096 14.2 / 14.6, 1024 x 6144 20.5 / 21.8).
constexpr int64_t kRotatedWide = 1 << 17, kRotatedFull = 15 << 15;

template <class SRC, bool ACC_BF16, int WT, int THREADS>
__global__ __launch_bounds__(THREADS) void reduce_rotated_kernel(
    const SRC src, int w_rt, int64_t band_v, int rank, u32x4* __restrict__ out) {
    const int W = WT > 0 ? WT : w_rt;
    constexpr int G = 8;
    const int64_t v = (int64_t)blockIdx.x * THREADS + threadIdx.x;
    if (v >= band_v) return;
    float acc[8];
    const int first = (rank + 1) % W;
    for (int i0 = 0; i0 < W; i0 += G) {
        u32x4 x[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            if (i0 + g < W) {
                const int cur = first + i0 + g;
                x[g] = ld_stream(src.at(cur >= W ? cur - W : cur) + v);
            }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            if (i0 + g >= W) break;
            if (i0 + g == 0) {
                unpack8(x[g], acc);
            } else {
                add8(x[g], acc);
                if (ACC_BF16) unpack8(pack8(acc), acc);
            }
        }
    }
    st_stream(out + v, pack8(acc));
}

// Vectors per thread per block: 4 for large inputs (most bytes in flight per workgroup), 1
// for inputs too small to give every CU such a block (more, smaller workgroups).  Measured with
// inputs that are not in any cache: from 256 blocks of 4 x 256 vectors on (one per CU) the
// larger block wins whenever the blocks fill whole rounds of 256 CUs (32 MiB input: 9.0 -> 7.9 us,
// 64 MiB: 16.0 -> 13.5 us), and loses 5 % at one and a half rounds.
static int pick_unroll(int64_t nvec) {
    if (const int u = env_switches().reduce_unroll; u == 1 || u == 2 || u == 4) return u;
    const int64_t blocks4 = (nvec + kThreads * 4 - 1) / (kThreads * 4);
    return (blocks4 >= 768 || (blocks4 >= 256 && blocks4 % 256 == 0)) ? 4 : 1;
}

template <class SRC, int WT, int BIAS, bool BF>
static void launch_reduce3(hipStream_t s, const SRC& tab, int W, int64_t nvec, const u32x4* bias,
                           uint32_t d_vec, u32x4* out) {
    const int unroll = pick_unroll(nvec);
    const int64_t per_block = (int64_t)kThreads * unroll;
    int64_t blocks = (nvec + per_block - 1) / per_block;
    const int64_t max_blocks = env_switches().reduce_blocks > 0 ? env_switches().reduce_blocks : kMaxBlocks;
    if (blocks > max_blocks) blocks = max_blocks;
    const dim3 grid((unsigned)blocks);
    if (unroll == 2)
        hipLaunchKernelGGL((reduce_kernel<SRC, WT, BIAS, BF, 2>), grid, dim3(kThreads), 0, s, tab, W, nvec, bias,
                           d_vec, out);
    else if (unroll == 4)
        hipLaunchKernelGGL((reduce_kernel<SRC, WT, BIAS, BF, 4>), grid, dim3(kThreads), 0, s, tab, W, nvec, bias,
                           d_vec, out);
    else
        hipLaunchKernelGGL((reduce_kernel<SRC, WT, BIAS, BF, 1>), grid, dim3(kThreads), 0, s, tab, W, nvec, bias,
                           d_vec, out);
}

template <class SRC, int WT, int BIAS>
static hipError_t launch_reduce2(bool bias_first, hipStream_t s, const SRC& tab, int W,
                                 int64_t nvec, const u32x4* bias, uint32_t d_vec, u32x4* out) {
    if (bias_first)
        launch_reduce3<SRC, WT, BIAS, true>(s, tab, W, nvec, bias, d_vec, out);
    else
        launch_reduce3<SRC, WT, BIAS, false>(s, tab, W, nvec, bias, d_vec, out);
    return hipGetLastError();
}

template <class SRC, int WT>
static hipError_t launch_reduce1(int mode, bool bias_first, hipStream_t s, const SRC& tab, int W,
                                 int64_t nvec, const u32x4* bias, uint32_t d_vec, u32x4* out) {
    switch (mode) {
        case kNoBias:
            // without a bias both orders are the same kernel
            return launch_reduce2<SRC, WT, kNoBias>(true, s, tab, W, nvec, bias, d_vec, out);
        case kFullBias:
            return launch_reduce2<SRC, WT, kFullBias>(bias_first, s, tab, W, nvec, bias, d_vec, out);
        default:
            return launch_reduce2<SRC, WT, kVectorBias>(bias_first, s, tab, W, nvec, bias, d_vec, out);
    }
}

}  // namespace kr

using namespace kr;

// Argument checks shared by the stacked and the pointer-table entry points; `first` is the
// stacked tensor, or the table itself.  Returns KR_OK also for numel == 0.
static int check_reduce_common(const void* first, int W, int64_t numel, const void* out) {
    if (W < 1 || W > KR_MAX_WORLD) return KR_ERR_WORLD_SIZE;
    if (numel < 0) return KR_ERR_BAD_DIM;
    if (numel % 8 != 0) return KR_ERR_NUMEL_MOD8;
    if (numel == 0) return KR_OK;
    if (first == nullptr || out == nullptr) return KR_ERR_NULL_POINTER;
    if (!aligned16(out)) return KR_ERR_ALIGNMENT;
    return KR_OK;
}

static int check_stack(const void* stack, int64_t slice_stride) {
    if (!aligned16(stack) || slice_stride % 8 != 0) return KR_ERR_ALIGNMENT;
    if (slice_stride < 0) return KR_ERR_BAD_DIM;
    return KR_OK;
}

// bias mode from the bias arguments, or a negative argument error
static int reduce_bias_mode(const void* bias, int64_t bias_numel, int64_t numel, int64_t D) {
    if (bias == nullptr) return kNoBias;
    if (!aligned16(bias)) return KR_ERR_ALIGNMENT;
    if (bias_numel == numel) return kFullBias;
    if (D > 0 && bias_numel == D && D % 8 == 0 && numel % D == 0) return kVectorBias;
    return KR_ERR_BIAS_SHAPE;
}

template <class SRC>
static int launch_reduce(const SRC& tab, int W, int64_t numel, const void* bias, int mode, int64_t D,
                         int bias_first, void* out, void* stream) {
    const int64_t nvec = numel / 8;
    const hipStream_t s = (hipStream_t)stream;
    const u32x4* bp = (const u32x4*)bias;
    u32x4* op = (u32x4*)out;
    const uint32_t d_vec = mode == kVectorBias ? (uint32_t)(D / 8) : 1u;
    hipError_t e;
    switch (W) {
        case 2: e = launch_reduce1<SRC, 2>(mode, bias_first != 0, s, tab, W, nvec, bp, d_vec, op); break;
        case 4: e = launch_reduce1<SRC, 4>(mode, bias_first != 0, s, tab, W, nvec, bp, d_vec, op); break;
        case 8: e = launch_reduce1<SRC, 8>(mode, bias_first != 0, s, tab, W, nvec, bp, d_vec, op); break;
        default: e = launch_reduce1<SRC, 0>(mode, bias_first != 0, s, tab, W, nvec, bp, d_vec, op); break;
    }
    return (int)e;
}

extern "C" int kr_reduce_bf16(const void* stack, int W, int64_t slice_stride, int64_t numel, const void* bias,
                              int64_t bias_numel, int64_t D, int bias_first, void* out, void* stream) {
    int rc = check_reduce_common(stack, W, numel, out);
    if (rc != KR_OK) return rc;
    if (numel > 0 && (rc = check_stack(stack, slice_stride)) != KR_OK) return rc;
    const int mode = reduce_bias_mode(bias, bias_numel, numel, D);
    if (mode < 0) return mode;
    if (numel == 0) return KR_OK;
    const StackedPeers src{(const u32x4*)stack, slice_stride / 8};
    return launch_reduce(src, W, numel, bias, mode, D, bias_first, out, stream);
}

extern "C" int kr_reduce_ptrs_bf16(const void* const* bufs, int W, int64_t numel, const void* bias,
                                   int64_t bias_numel, int64_t D, int bias_first, void* out, void* stream) {
    int rc = check_reduce_common(bufs, W, numel, out);
    if (rc != KR_OK) return rc;
    const int mode = reduce_bias_mode(bias, bias_numel, numel, D);
    if (mode < 0) return mode;
    if (numel == 0) return KR_OK;
    PeerTab tab;
    if ((rc = peer_tab_from_ptrs(tab, bufs, W)) != KR_OK) return rc;
    return launch_reduce(tab, W, numel, bias, mode, D, bias_first, out, stream);
}

extern "C" int64_t kr_striped_share_numel(int64_t numel, int W, int64_t stripe_block, int rank) {
    if (W < 1 || W > KR_MAX_WORLD) return KR_ERR_WORLD_SIZE;
    if (numel < 0) return KR_ERR_BAD_DIM;
    if (numel % 8 != 0) return KR_ERR_NUMEL_MOD8;
    if (stripe_block <= 0 || stripe_block % 8 != 0 || rank < 0 || rank >= W) return KR_ERR_STRIPE;
    const int64_t stripe = stripe_block * W;
    const int64_t full = numel / stripe;
    const int64_t rem = numel - full * stripe;
    int64_t tail = rem - (int64_t)rank * stripe_block;
    if (tail < 0) tail = 0;
    if (tail > stripe_block) tail = stripe_block;
    return full * stripe_block + tail;
}

template <class SRC>
static int launch_striped(const SRC& tab, int W, int64_t share, const void* bias, int64_t stripe_block,
                          int rank, void* out, void* stream) {
    if (bias != nullptr && !aligned16(bias)) return KR_ERR_ALIGNMENT;
    const int64_t nvec = share / 8;
    if ((nvec + kWave - 1) / kWave > 0x7fffffffLL || stripe_block / 8 > 0xffffffffLL) return KR_ERR_BAD_DIM;
#define KR_LAUNCH(WT, TOGETHER, THREADS)                                                                                         \
    hipLaunchKernelGGL((reduce_striped_kernel<SRC, WT, TOGETHER, THREADS>), dim3((unsigned)((nvec + THREADS - 1) / THREADS)), dim3(THREADS), 0, \
                       (hipStream_t)stream, tab, W, nvec, (const u32x4*)bias, (uint32_t)(stripe_block / 8), rank, (u32x4*)out)
    if (nvec > kChainVecs) KR_LAUNCH(0, false, kWave);
    else if ((W == 4 && nvec >= kTogetherVecs) || (W == 16 && 2 * nvec >= 3 * kTogetherVecs)) KR_LAUNCH(0, false, kThreads);
    else if (W == 8) KR_LAUNCH(8, true, kWave);
    else if (W == 4) KR_LAUNCH(4, true, kWave);
    else if (W == 2) KR_LAUNCH(2, true, kWave);
    else KR_LAUNCH(0, true, kWave);
#undef KR_LAUNCH
    return (int)hipGetLastError();
}

extern "C" int kr_reduce_striped_bf16(const void* stack, int W, int64_t slice_stride, int64_t numel,
                                      const void* bias, int64_t stripe_block, int rank, void* out,
                                      void* stream) {
    const int64_t share = kr_striped_share_numel(numel, W, stripe_block, rank);
    if (share < 0) return (int)share;
    if (share == 0) return KR_OK;
    int rc = check_reduce_common(stack, W, numel, out);
    if (rc != KR_OK) return rc;
    if ((rc = check_stack(stack, slice_stride)) != KR_OK) return rc;
    const StackedPeers src{(const u32x4*)stack, slice_stride / 8};
    return launch_striped(src, W, share, bias, stripe_block, rank, out, stream);
}

extern "C" int kr_reduce_striped_ptrs_bf16(const void* const* bufs, int W, int64_t numel, const void* bias,
                                           int64_t stripe_block, int rank, void* out, void* stream) {
    const int64_t share = kr_striped_share_numel(numel, W, stripe_block, rank);
    if (share < 0) return (int)share;
    if (share == 0) return KR_OK;
    int rc = check_reduce_common(bufs, W, numel, out);
    if (rc != KR_OK) return rc;
    PeerTab tab;
    if ((rc = peer_tab_from_ptrs(tab, bufs, W)) != KR_OK) return rc;
    return launch_striped(tab, W, share, bias, stripe_block, rank, out, stream);
}

template <class SRC>
static int launch_rotated(const SRC& src, int W, int64_t band_v, int rank, int acc_bf16, void* out, void* stream) {
    if ((band_v + kWave - 1) / kWave > 0x7fffffffLL) return KR_ERR_BAD_DIM;
    const bool wide = band_v >= kRotatedWide && band_v < kRotatedFull;
#define KR_LAUNCH(WT, THREADS)                                                                                                     \
    do {                                                                                                                           \
        const dim3 grid((unsigned)((band_v + THREADS - 1) / THREADS)), block(THREADS);                                             \
        if (acc_bf16)                                                                                                              \
            hipLaunchKernelGGL((reduce_rotated_kernel<SRC, true, WT, THREADS>), grid, block, 0, (hipStream_t)stream, src, W, band_v, rank, (u32x4*)out); \
        else                                                                                                                       \
            hipLaunchKernelGGL((reduce_rotated_kernel<SRC, false, WT, THREADS>), grid, block, 0, (hipStream_t)stream, src, W, band_v, rank, (u32x4*)out); \
    } while (0)
    switch (W) {
        case 2: KR_LAUNCH(2, kWave); break;
        case 4: if (wide) KR_LAUNCH(4, kThreads); else KR_LAUNCH(4, kWave); break;
        case 8: if (wide) KR_LAUNCH(8, kThreads); else KR_LAUNCH(8, kWave); break;
        default: KR_LAUNCH(0, kWave); break;
    }
#undef KR_LAUNCH
    return (int)hipGetLastError();
}

// Argument checks of the rotated reduce; `first` is the stacked tensor or the table.  Returns the vectors of a band
// (0: nothing to do), or a negative argument error.
static int64_t check_rotated(const void* first, int W, int64_t rows, int64_t N, int rank, const void* out) {
    if (W < 1 || W > KR_MAX_WORLD) return KR_ERR_WORLD_SIZE;
    if (rows < 0 || N < 0) return KR_ERR_BAD_DIM;
    if (rank < 0 || rank >= W) return KR_ERR_STRIPE;
    const int64_t band = rows * N;
    if (band % 8 != 0) return KR_ERR_NUMEL_MOD8;
    if (band == 0) return 0;
    if (first == nullptr || out == nullptr) return KR_ERR_NULL_POINTER;
    if (!aligned16(out)) return KR_ERR_ALIGNMENT;
    return band / 8;
}

extern "C" int kr_reduce_rotated_bf16(const void* in, int W, int64_t rows, int64_t N, int rank, int acc_bf16,
                                      void* out, void* stream) {
    const int64_t band_v = check_rotated(in, W, rows, N, rank, out);
    if (band_v <= 0) return (int)band_v;
    if (!aligned16(in)) return KR_ERR_ALIGNMENT;
    return launch_rotated(StackedPeers{(const u32x4*)in, band_v}, W, band_v, rank, acc_bf16, out, stream);
}

extern "C" int kr_reduce_rotated_ptrs_bf16(const void* const* bands, int W, int64_t rows, int64_t N, int rank,
                                           int acc_bf16, void* out, void* stream) {
    const int64_t band_v = check_rotated(bands, W, rows, N, rank, out);
    if (band_v <= 0) return (int)band_v;
    PeerTab tab;
    if (const int rc = peer_tab_from_ptrs(tab, bands, W); rc != KR_OK) return rc;
    return launch_rotated(tab, W, band_v, rank, acc_bf16, out, stream);
}

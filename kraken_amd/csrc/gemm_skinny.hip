// GEMM with at most 64 rows (decode): the right operand is streamed once through wave-private LDS rings.
//
// With a handful of rows the product is the time it takes to read B, and a kernel made of 128x128 tiles pays for
// barriers in its ring of stages and, to have enough workgroups, for a second launch that sums parts of K.  Here a
// workgroup owns 16, 32 or 64 columns of C and all of K: its wavefronts take 128-byte units of k in turn (so that they
// read neighbouring lines at the same time), each with an LDS ring of its own, and never meet before the end.  The
// partial sums then meet once in LDS, and the epilogue (peers' partial sums, requested before the k loop, bias,
// rounding) is part of the same launch.
//
// The operands go through LDS although nothing is shared: a fragment in the layout of the matrix cores (lane l: row
// l%16) loaded straight into registers touches 16 lines per quarter of a wavefront, and the address unit then takes
// four times as long per byte as for 128-byte rows.
//
// Measured, B in no cache, seven peers: 16 x 8192 x 3584 transposed B 14.1 us (128x128 tiles in four parts and a
// finishing pass 20.9; reading B at 6.3 TB/s 9.3), 4 x 3360 x 976 6.3 (14.1), fp32 16 x 4096 x 4096 17.6 (28.7).  What bounds
// it: HBM for wide outputs, the 64 GB/s a compute unit takes in for narrow ones, 6 us of start and end for small ones.
//
// fp32 operands are split into hi and lo parts in registers and take three products (hi hi, lo hi, hi lo); fp8 operands are
// widened to bf16 in registers.  us, 256-row tiles of gemm_w8.hip / here: 16 x 4672 x 4096 23.8 / 7.4, x 13248 37.1 / 21.4 (B at 6.3 TB/s: 9.8),
// 4 x 1152 x 1088 15.6 / 5.9, 64 x 7488 x 4096 27.2 / 13.1, x 13248 45.7 / 37.4.
#include "gemm_common.h"

namespace kr {

namespace {

constexpr uint32_t kOob = 0x80000000u;
constexpr int kEarlyPeers = 7;   // peers' partial sums requested before the k loop
constexpr int kBlock = 2048;     // bytes of a unit: 16 rows (or columns) of 128 bytes of k

// MB: blocks of 16 rows, CB: columns of the workgroup / 16
constexpr int waves_of(int MB, int CB) { return MB + CB <= 3 ? 8 : 4; }
constexpr int stages_of(int MB, int CB) { return 160 * 1024 / (waves_of(MB, CB) * (MB + CB) * kBlock); }
constexpr int ring_bytes(int MB, int CB) { return stages_of(MB, CB) * (MB + CB) * kBlock; }   // of one wavefront
constexpr int red_pitch(int CB) { return 16 * CB + 4; }

typedef const __attribute__((address_space(3))) u32x4* lds_u4;
typedef const __attribute__((address_space(3))) uint32_t* lds_u1;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4* lds_tr;
typedef __attribute__((address_space(3))) f32x4* lds_f32x4;

constexpr int vmcnt_imm(int n) { return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14); }

// hi and lo bf16 parts of eight fp32 values given as bits
__device__ __forceinline__ void split8(const u32x4 (&x)[2], bf16x8& hi, bf16x8& lo) {
    u32x4 h, l;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t xa = x[j / 2][2 * (j % 2)], xb = x[j / 2][2 * (j % 2) + 1];   // (a bit cast of a vector's element reads element 0)
        const float a = __builtin_bit_cast(float, xa), b = __builtin_bit_cast(float, xb);
        h[j] = pack_bf16(a, b);
        l[j] = pack_bf16(a - bf16_lo(h[j]), b - bf16_hi(h[j]));
    }
    hi = __builtin_bit_cast(bf16x8, h);
    lo = __builtin_bit_cast(bf16x8, l);
}

// eight fp8 (e4m3) as bf16, exactly
__device__ __forceinline__ bf16x8 widen8(uint32_t w0, uint32_t w1) {
    return __builtin_bit_cast(bf16x8, u32x4{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)w0, 1.0f, false)),
                                            __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)w0, 1.0f, true)),
                                            __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)w1, 1.0f, false)),
                                            __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)w1, 1.0f, true))});
}

// row-major B: slot of a k-row in LDS that holds piece 0; a fragment read then touches every bank once or twice
template <int E, int CB>
__device__ __forceinline__ int swizzle(int k) {
    if constexpr (E == 4) return CB > 1 ? 4 * ((k >> 2) & 1) : 0;
    return CB > 2 ? 2 * ((k >> 1) & 1) + 4 * ((k >> 3) & 1) : CB > 1 ? 2 * ((k >> 3) & 1) : 0;
}

// E: bytes of an operand's element: 4 fp32, 2 bf16, 1 fp8 (transposed-contiguous B only)
template <int E, bool B_NT, int MB, int CB>
__global__ __launch_bounds__(waves_of(MB, CB) * 64) void gemm_skinny_kernel(const GemmArgs g) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // starts at LDS address 0; one ring per wavefront
    constexpr bool F32 = E == 4, F8 = E == 1;
    static_assert(!F8 || B_NT, "fp8: transposed-contiguous B");
    constexpr int NB = 16 * CB, LD = red_pitch(CB);
    constexpr int KU = 128 / E;                                // k of a unit
    constexpr int kWaves = waves_of(MB, CB), kStages = stages_of(MB, CB), kRing = ring_bytes(MB, CB);
    constexpr int kStage = (MB + CB) * kBlock, kLoads = 2 * (MB + CB);
    static_assert(16 * MB * LD * 4 <= kRing && kStages >= 2 && 32 * MB * CB <= 64 * kWaves, "LDS of a wavefront, results of a thread");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p = lane & 15, gq = lane >> 4;
    // workgroups are dealt round-robin to the XCDs: neighbouring column blocks, which share the lines of a row-major
    // B, get ids 8 apart
    const int nblk = gridDim.x, xcd = blockIdx.x % kXcds;
    const int n0 = (xcd * (nblk / kXcds) + min(xcd, nblk % kXcds) + (int)blockIdx.x / kXcds) * NB;
    // units of this workgroup (all of them, or those of part blockIdx.y), dealt to the wavefronts in turn
    const int u_all = (g.K + KU - 1) / KU;
    const int u_begin = (int)((int64_t)u_all * blockIdx.y / g.k_splits), u_end = (int)((int64_t)u_all * (blockIdx.y + 1) / g.k_splits);
    const int u_last = max(u_end - 1, 0);

    // ---- what the epilogue adds: thread t stores 8 columns of row t / (NB/8) -----------------------------
    constexpr int CV = NB / 8;
    const int er = threadIdx.x / CV, en = n0 + (threadIdx.x % CV) * 8;
    const bool stores = er < g.M && er < 16 * MB && en < g.N;
    const int mb = er - g.band_row0;
    const bool in_band = stores && mb >= 0 && mb < g.band_rows;
    const uint32_t p_off = in_band ? (uint32_t)((mb * (int64_t)g.N + en) * 2) : kOob;
    u32x4 pv[kEarlyPeers];
#pragma unroll
    for (int q = 0; q < kEarlyPeers; ++q) pv[q] = ld_stream(stream_rsrc(g.peer.p[q], q < g.n_peers ? 0x7fffffffu : 0u), p_off);

    // ---- LDS-DMA addressing -------------------------------------------------------------------
    // A (and transposed B): a load fills 8 rows of 128 bytes: lane l -> row 8r + l/8, slot l%8 holds 16-byte piece
    // slot ^ ((row >> 1) & 7).  Rows past M and columns past N re-read the last ones (their sums are never stored).
    const i32x4 a_rs = raw_rsrc(g.A, 0x7fffffff);
    const i32x4 b_rs = raw_rsrc((const char*)g.B + (B_NT ? (int64_t)n0 * g.ldb : (int64_t)n0) * E, 0x7fffffff);
    uint32_t a_off[2 * MB], b_off[2 * CB];
    int a_k[2], b_k[2];    // k of the lane's piece in loads of even and odd r, within a unit
#pragma unroll
    for (int r = 0; r < 2 * MB; ++r) {
        const int piece = (lane & 7) ^ ((4 * (r & 1) + (lane >> 4)) & 7);
        a_k[r & 1] = piece * (16 / E);
        a_off[r] = (uint32_t)((min(8 * r + (lane >> 3), g.M - 1) * g.lda + a_k[r & 1]) * E);
    }
#pragma unroll
    for (int r = 0; r < 2 * CB; ++r) {
        if constexpr (B_NT) {
            b_k[r & 1] = a_k[r & 1];
            b_off[r] = (uint32_t)((min(8 * r + (lane >> 3), g.N - 1 - n0) * g.ldb + b_k[r & 1]) * E);
        } else {
            // row-major B: a load fills 1 KiB of k-rows of NB columns, their pieces permuted by swizzle(k)
            constexpr int PR = NB * E / 16, KR = 64 / PR;   // pieces of a k-row, k-rows of a load
            const int k = KR * r + lane / PR;
            const int piece = (lane % PR) ^ swizzle<E, CB>(k);
            b_off[r] = (uint32_t)((k * g.ldb + min(piece * (16 / E), g.N - 16 / E - n0)) * E);
        }
    }
    const uint32_t ring = (uint32_t)(wave * kRing);
    auto load_unit = [&](int u, uint32_t stage) __attribute__((always_inline)) {
        const bool live = u < u_end;
        const int k0 = min(u, u_last) * KU;   // (the scalar offset stays inside the matrix)
#pragma unroll
        for (int r = 0; r < 2 * MB; ++r)
            lds_dma_b128(a_rs, ring + stage + r * 1024, live && k0 + a_k[r & 1] < g.K ? a_off[r] : kOob, k0 * E);
#pragma unroll
        for (int r = 0; r < 2 * CB; ++r) {
            if constexpr (B_NT) {
                lds_dma_b128(b_rs, ring + stage + (2 * MB + r) * 1024, live && k0 + b_k[r & 1] < g.K ? b_off[r] : kOob, k0 * E);
            } else {
                constexpr int PR = NB * E / 16, KR = 64 / PR;
                lds_dma_b128(b_rs, ring + stage + (2 * MB + r) * 1024, live && k0 + KR * r + lane / PR < g.K ? b_off[r] : kOob,
                             (int)(k0 * g.ldb * E));
            }
        }
    };

    // ---- fragments: lane -> row p of a block, pieces gq and 4 + gq ----------------------------------------
    const uint32_t f0 = (uint32_t)(p * 128 + ((gq ^ ((p >> 1) & 7)) << 4)), f1 = (uint32_t)(p * 128 + (((4 + gq) ^ ((p >> 1) & 7)) << 4));
    f32x4 acc[MB][CB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int c = 0; c < CB; ++c) acc[i][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    u32x4 af[MB][2], bf[CB][2];   // bf16: the fragments of both 32-k halves; fp32: 8 values; fp8: 16 and 16 values
    auto read_unit = [&](uint32_t stage) __attribute__((always_inline)) {
        const uint32_t a = ring + stage, b = a + MB * kBlock;
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            af[i][0] = *(lds_u4)(size_t)(a + i * kBlock + f0);
            af[i][1] = *(lds_u4)(size_t)(a + i * kBlock + f1);
        }
#pragma unroll
        for (int c = 0; c < CB; ++c) {
            if constexpr (B_NT) {
                bf[c][0] = *(lds_u4)(size_t)(b + c * kBlock + f0);
                bf[c][1] = *(lds_u4)(size_t)(b + c * kBlock + f1);
            } else if constexpr (F32) {
                // column 16c + p of k-rows 4 gq .. +3 and 16 + 4 gq .. +3
                const uint32_t o = b + (uint32_t)(4 * gq * NB * 4 + (((4 * c + (p >> 2)) ^ swizzle<E, CB>(4 * gq)) << 4) + (p & 3) * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    bf[c][0][e] = *(lds_u1)(size_t)(o + e * NB * 4);
                    bf[c][1][e] = *(lds_u1)(size_t)(o + (16 + e) * NB * 4);
                }
            } else {
                // transposing reads: group gq reads k-rows 32 h + 8 gq + p/4 (and 4 further on), columns 16c + 4 (p%4) .. +3
                const uint32_t o = b + (uint32_t)((8 * gq + (p >> 2)) * NB * 2 + (((2 * c + ((p & 3) >> 1)) ^ swizzle<E, CB>(8 * gq + (p >> 2))) << 4) + (p & 1) * 8);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(size_t)(o + 32 * h * NB * 2));
                    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(size_t)(o + (32 * h + 4) * NB * 2));
                    bf[c][h] = __builtin_bit_cast(u32x4, (s16x8){lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w});
                }
            }
        }
    };
    auto multiply = [&]() __attribute__((always_inline)) {
        if constexpr (F32) {
            bf16x8 a_hi[MB], a_lo[MB];
#pragma unroll
            for (int i = 0; i < MB; ++i) split8(af[i], a_hi[i], a_lo[i]);
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                bf16x8 b_hi, b_lo;
                split8(bf[c], b_hi, b_lo);
#pragma unroll
                for (int i = 0; i < MB; ++i) {
                    acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b_hi, a_hi[i], acc[i][c], 0, 0, 0);
                    acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b_lo, a_hi[i], acc[i][c], 0, 0, 0);
                    acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b_hi, a_lo[i], acc[i][c], 0, 0, 0);
                }
            }
        } else if constexpr (F8) {
            // (16 k of a piece in two halves of 8: both operands take their k in this order)
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                bf16x8 a8[MB];
#pragma unroll
                for (int i = 0; i < MB; ++i) a8[i] = widen8(af[i][h / 2][2 * (h % 2)], af[i][h / 2][2 * (h % 2) + 1]);
#pragma unroll
                for (int c = 0; c < CB; ++c) {
                    const bf16x8 b8 = widen8(bf[c][h / 2][2 * (h % 2)], bf[c][h / 2][2 * (h % 2) + 1]);
#pragma unroll
                    for (int i = 0; i < MB; ++i) acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b8, a8[i], acc[i][c], 0, 0, 0);
                }
            }
        } else {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < MB; ++i)
#pragma unroll
                    for (int c = 0; c < CB; ++c)
                        acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, bf[c][h]), __builtin_bit_cast(bf16x8, af[i][h]),
                                                                            acc[i][c], 0, 0, 0);
        }
    };

    // ---- k loop: kStages units in flight per wavefront; those past the end are requested out of range (zeros in LDS,
    // no traffic), so that the count of loads behind the oldest unit never changes ---------------------------
    const int u0 = u_begin + wave;
#pragma unroll
    for (int d = 0; d < kStages; ++d) load_unit(u0 + d * kWaves, d * kStage);
    uint32_t stage = 0;
#pragma nounroll
    for (int u = u0; u < u_end; u += kWaves) {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((kStages - 1) * kLoads));   // the oldest unit has arrived
        __builtin_amdgcn_sched_barrier(0);
        read_unit(stage);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): the stage has been read and may be overwritten
        __builtin_amdgcn_sched_barrier(0);
        load_unit(u + kStages * kWaves, stage);
        __builtin_amdgcn_sched_barrier(0);
        multiply();
        stage = stage == (kStages - 1) * kStage ? 0u : stage + kStage;
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));   // nothing is written into the ring any more
    __builtin_amdgcn_sched_barrier(0);

    // ---- the partial sums meet in LDS, each wavefront's in its own ring: [row][column], rows of LD ----------
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int c = 0; c < CB; ++c) *(lds_f32x4)(size_t)(ring + ((16 * i + p) * LD + 16 * c + 4 * gq) * 4) = acc[i][c];
    __syncthreads();
    if (!stores) return;
    float f[8];
    zero8(f);
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        const uint32_t o = (uint32_t)(w * kRing + (er * LD + (en - n0)) * 4);
        const f32x4 x = *(lds_f32x4)(size_t)o, y = *(lds_f32x4)(size_t)(o + 16);
        f[0] += x.x; f[1] += x.y; f[2] += x.z; f[3] += x.w;
        f[4] += y.x; f[5] += y.y; f[6] += y.z; f[7] += y.w;
    }
    if (!in_band) {
        if (g.c_full != nullptr) st_stream((u32x4*)(g.c_full + (int64_t)er * g.N + en), pack8(f));
        return;
    }
    if constexpr (F8) {
        if (g.out_fp8) {   // (no peers, no bias)
            store8_e4m3((uint8_t*)g.out + (int64_t)mb * g.N + en, f);
            return;
        }
    }
    // (a bf16 product is rounded before the partial sums are added, as in the other kernels)
    if (!g.out_is_fp32) unpack8(pack8(f), f);
#pragma unroll
    for (int q = 0; q < kEarlyPeers; ++q)
        if (q < g.n_peers) add8(pv[q], f);
    const int64_t off = (int64_t)mb * g.N + en;
    for (int q = kEarlyPeers; q < g.n_peers; ++q) add8(ld_stream((const u32x4*)((const uint16_t*)g.peer.p[q] + off)), f);
    if (g.bias != nullptr) add8(*(const u32x4*)(g.bias + en), f);
    if (g.out_is_fp32) {
        float* o = (float*)g.out + blockIdx.y * g.split_out_stride + off;
        *(f32x4*)o = f32x4{f[0], f[1], f[2], f[3]};
        *(f32x4*)(o + 4) = f32x4{f[4], f[5], f[6], f[7]};
    } else {
        st_stream((u32x4*)((uint16_t*)g.out + off), pack8(f));
    }
}

template <int E, bool B_NT, int MB, int CB>
hipError_t launch_one(const GemmArgs& g, hipStream_t st) {
    constexpr int lds = waves_of(MB, CB) * ring_bytes(MB, CB);
    auto kfn = gemm_skinny_kernel<E, B_NT, MB, CB>;
    static std::atomic<uint64_t> opted{0};
    if (hipError_t e = lds_opt_in((const void*)kfn, lds, opted); e != hipSuccess) return e;
    hipLaunchKernelGGL(kfn, dim3((unsigned)((g.N + 16 * CB - 1) / (16 * CB)), (unsigned)g.k_splits), dim3(waves_of(MB, CB) * 64), lds, st, g);
    return hipGetLastError();
}
template <int E, bool B_NT, int CB>
hipError_t launch_rows(const GemmArgs& g, hipStream_t st) {
    if (g.M <= 16) return launch_one<E, B_NT, 1, CB>(g, st);
    if (g.M <= 32) return launch_one<E, B_NT, 2, CB>(g, st);
    return launch_one<E, B_NT, 4, CB < 4 ? CB : 2>(g, st);   // (64 x 64: more results than threads)
}

}  // namespace

// Loads the file's device code for the current device (code objects are loaded on first use, which moves
// device memory).
hipError_t load_gemm_skinny() {
    hipFuncAttributes a;
    return hipFuncGetAttributes(&a, (const void*)gemm_skinny_kernel<2, true, 1, 1>);
}

hipError_t launch_gemm_skinny(const GemmArgs& g, bool b_nt, int esize, int cb, hipStream_t st) {
    if (esize == 1) return cb == 1 ? launch_rows<1, true, 1>(g, st) : cb == 2 ? launch_rows<1, true, 2>(g, st) : launch_rows<1, true, 4>(g, st);
    if (esize == 4) {
        if (b_nt) return cb == 1 ? launch_rows<4, true, 1>(g, st) : launch_rows<4, true, 2>(g, st);
        return cb == 1 ? launch_rows<4, false, 1>(g, st) : launch_rows<4, false, 2>(g, st);
    }
    if (b_nt) return cb == 1 ? launch_rows<2, true, 1>(g, st) : cb == 2 ? launch_rows<2, true, 2>(g, st) : launch_rows<2, true, 4>(g, st);
    return cb == 1 ? launch_rows<2, false, 1>(g, st) : cb == 2 ? launch_rows<2, false, 2>(g, st) : launch_rows<2, false, 4>(g, st);
}

}  // namespace kr

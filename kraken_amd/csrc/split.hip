// fp32 GEMM operands for the bf16 matrix cores: x = hi + lo with hi = bf16(x), lo = bf16(x - hi).
// One pass over the fp32 matrix writes the three bf16 blocks the 3K-long product needs,
//   A [M, K]            -> [ a_hi | a_hi | a_lo ]   ([M, 3K], blocks side by side)
//   B [K, N] row-major  -> [ b_hi ; b_lo ; b_hi ]   ([3K, N], blocks one below the other)
//   B^T [N, K]          -> [ b_hi | b_lo | b_hi ]   ([N, 3K])
// so that  A' @ B' = a_hi b_hi + a_hi b_lo + a_lo b_hi  (everything of a @ b but a_lo b_lo).
#include "common.h"

namespace kr {

// One thread per 8 consecutive columns: two 128-bit loads, three 128-bit stores.
// SIDE: blocks side by side (block b of row r starts at out + r*ld_out + b*cols), else one below
// the other (block b of row r at out + (b*rows + r)*ld_out).  sel[b]: 0 = hi, 1 = lo.
template <bool SIDE>
__global__ __launch_bounds__(256) void split_fp32_kernel(const float* __restrict__ x, int64_t rows, int cols_v, int64_t ld_x,
                                                         uint16_t* __restrict__ out, int64_t ld_out, int sel0, int sel1, int sel2) {
    const int64_t nvec = rows * cols_v;
    for (int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x; v < nvec; v += (int64_t)gridDim.x * 256) {
        const int64_t r = v / cols_v;
        const int c = (int)(v - r * cols_v) * 8;
        const f32x4 lo4 = __builtin_nontemporal_load((const f32x4*)(x + r * ld_x + c));
        const f32x4 hi4 = __builtin_nontemporal_load((const f32x4*)(x + r * ld_x + c + 4));
        const float f[8] = {lo4.x, lo4.y, lo4.z, lo4.w, hi4.x, hi4.y, hi4.z, hi4.w};
        const u32x4 hi = pack8(f);
        float h[8], d[8];
        unpack8(hi, h);
#pragma unroll
        for (int j = 0; j < 8; ++j) d[j] = f[j] - h[j];
        const u32x4 lo = pack8(d);
        const int cols = cols_v * 8;
        const int sel[3] = {sel0, sel1, sel2};
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            uint16_t* dst = SIDE ? out + r * ld_out + (int64_t)b * cols + c : out + ((int64_t)b * rows + r) * ld_out + c;
            st_stream((u32x4*)dst, sel[b] ? lo : hi);
        }
    }
}

// ---- pairs: both operands of a product in one launch ----------------------------------------------------------------
// Every operand becomes rows along k of 32 hi parts, 32 lo parts, 32 hi parts, ... (128 bytes per 32 k, zeros past K), which is
// how the matrix-core kernel takes them (kPairs in gemm_dtl.hip).  Bound by memory: 4 bytes read and 4 written per element.
// A workgroup takes 64 k of 64 rows.  K_ROWS (the elements of a k lie together, row-major B): the tile is turned through LDS,
// whose rows of 65 floats put both the row-wise stores and the eight reads along k of a lane on different banks.
struct PairsOperand {
    const float* x;
    uint16_t* out;
    int64_t ld, ld_out;      // floats between rows (K_ROWS: between k), elements between rows of the result
    int rows, k_rows;
};

__global__ __launch_bounds__(256) void split_pairs_kernel(const PairsOperand a, const PairsOperand b, int K, int k_tiles, int a_tiles) {
    __shared__ float tile[64 * 65];
    const bool second = (int)blockIdx.x >= a_tiles;
    const PairsOperand o = second ? b : a;
    const int idx = second ? (int)blockIdx.x - a_tiles : (int)blockIdx.x;
    // the tiles that read the same lines follow each other: along k, or along the rows where these lie together
    const int row_tiles = (o.rows + 63) / 64;
    const int r0 = (o.k_rows ? idx % row_tiles : idx / k_tiles) * 64, k0 = (o.k_rows ? idx / row_tiles : idx % k_tiles) * 64;
    const int t = threadIdx.x;
    if (o.k_rows) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = i * 16 + (t >> 4), r = (t & 15) * 4;
            f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
            if (k0 + k < K && r0 + r < o.rows) v = __builtin_nontemporal_load((const f32x4*)(o.x + (int64_t)(k0 + k) * o.ld + r0 + r));
#pragma unroll
            for (int e = 0; e < 4; ++e) tile[k * 65 + r + e] = v[e];
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = i * 32 + (t >> 3), k = (t & 7) * 8;
        if (r0 + r >= o.rows || k0 + k >= (K + 31) / 32 * 32) continue;
        float f[8], h[8], d[8];
        zero8(f);
        if (o.k_rows) {
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = tile[(k + e) * 65 + r];
        } else if (k0 + k < K) {
            const float* p = o.x + (int64_t)(r0 + r) * o.ld + k0 + k;
            const f32x4 x = __builtin_nontemporal_load((const f32x4*)p), y = __builtin_nontemporal_load((const f32x4*)(p + 4));
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] = x[e], f[4 + e] = y[e];
        }
        const u32x4 hi = pack8(f);
        unpack8(hi, h);
#pragma unroll
        for (int e = 0; e < 8; ++e) d[e] = f[e] - h[e];
        uint16_t* dst = o.out + (int64_t)(r0 + r) * o.ld_out + 2 * (k0 + k / 32 * 32) + k % 32;
        *(u32x4*)dst = hi;
        *(u32x4*)(dst + 32) = pack8(d);
    }
}

}  // namespace kr

using namespace kr;

// A [M, K] with k contiguous, B [K, N] with strides (ldb_k, ldb_n), one of them 1; out: A' [M, 2 Kp], B' [N, 2 Kp], Kp = K up to
// a multiple of 32.
extern "C" int kr_split_pairs_fp32(const void* A, int64_t lda, const void* B, int64_t ldb_k, int64_t ldb_n, int64_t M, int64_t N,
                                   int64_t K, void* A_out, void* B_out, void* stream) {
    if (M < 0 || N < 0 || K < 0 || M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x3fffffffLL) return KR_ERR_BAD_DIM;
    if (K % 8 != 0 || N % 8 != 0) return KR_ERR_NUMEL_MOD8;
    if (M == 0 || N == 0 || K == 0) return KR_OK;
    if (A == nullptr || B == nullptr || A_out == nullptr || B_out == nullptr) return KR_ERR_NULL_POINTER;
    const bool k_rows = !(ldb_k == 1 && (ldb_n != 1 || N == 1));
    if (k_rows && ldb_n != 1) return KR_ERR_LAYOUT;
    const int64_t ldb = k_rows ? ldb_k : ldb_n;
    if (lda < K || ldb < (k_rows ? N : K)) return KR_ERR_LAYOUT;
    if (lda % 4 != 0 || ldb % 4 != 0 || !aligned16(A) || !aligned16(B) || !aligned16(A_out) || !aligned16(B_out)) return KR_ERR_ALIGNMENT;
    const int64_t ld_out = (K + 31) / 32 * 64, k_tiles = (K + 63) / 64, a_tiles = (M + 63) / 64 * k_tiles, b_tiles = (N + 63) / 64 * k_tiles;
    if (a_tiles + b_tiles > 0x7fffffffLL) return KR_ERR_BAD_DIM;
    const PairsOperand a{(const float*)A, (uint16_t*)A_out, lda, ld_out, (int)M, 0}, b{(const float*)B, (uint16_t*)B_out, ldb, ld_out, (int)N, k_rows};
    hipLaunchKernelGGL(split_pairs_kernel, dim3((unsigned)(a_tiles + b_tiles)), dim3(256), 0, (hipStream_t)stream, a, b, (int)K, (int)k_tiles, (int)a_tiles);
    return (int)hipGetLastError();
}

extern "C" int kr_split_fp32(const void* x, int64_t rows, int64_t cols, int64_t ld_x, int side_by_side, int pattern,
                             void* out, int64_t ld_out, void* stream) {
    if (rows < 0 || cols < 0 || rows > 0x7fffffffLL || cols > 0x7fffffffLL) return KR_ERR_BAD_DIM;
    if (cols % 8 != 0) return KR_ERR_NUMEL_MOD8;
    if (rows == 0 || cols == 0) return KR_OK;
    if (x == nullptr || out == nullptr) return KR_ERR_NULL_POINTER;
    if (ld_x < cols || ld_out < (side_by_side ? 3 * cols : cols)) return KR_ERR_LAYOUT;
    if (!aligned16(x) || !aligned16(out) || ld_x % 4 != 0 || ld_out % 8 != 0) return KR_ERR_ALIGNMENT;
    if (pattern != 0 && pattern != 1) return KR_ERR_BAD_DIM;
    // pattern 0: hi, hi, lo (the left operand); 1: hi, lo, hi (the right operand)
    const int s1 = pattern == 0 ? 0 : 1, s2 = pattern == 0 ? 1 : 0;
    const int64_t nvec = rows * (cols / 8);
    const unsigned blocks = (unsigned)std::min<int64_t>((nvec + 255) / 256, 256 * 16);
    hipStream_t st = (hipStream_t)stream;
    if (side_by_side)
        hipLaunchKernelGGL(split_fp32_kernel<true>, dim3(blocks), dim3(256), 0, st, (const float*)x, rows, (int)(cols / 8), ld_x,
                           (uint16_t*)out, ld_out, 0, s1, s2);
    else
        hipLaunchKernelGGL(split_fp32_kernel<false>, dim3(blocks), dim3(256), 0, st, (const float*)x, rows, (int)(cols / 8), ld_x,
                           (uint16_t*)out, ld_out, 0, s1, s2);
    return (int)hipGetLastError();
}

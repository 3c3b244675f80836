// Stream-ordered flag write and flag wait, and the copy-engine copy they bracket: the pieces of
// the overlap of copies with a running GEMM (all-gather matmul, copy-engine reduce-scatter).
#include <algorithm>

#include "common.h"

namespace kr {

// One store, written through to memory at system scope.  What the stream did before this
// kernel (the chunk copy) is complete and written back when this kernel starts -- the order
// of commands on a stream gives that -- so the store itself needs no cache write-back of its
// own (a release here would also flush whatever the concurrently running GEMM has written).
__global__ __launch_bounds__(kWave) void write_value32_kernel(uint32_t* addr, uint32_t value) {
    if (threadIdx.x == 0) __hip_atomic_store(addr, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Stream-ordered wait: ends once *addr == value.  One lane polls with system-scope loads and a
// short sleep; the wait is bounded by `ticks` of the 100 MHz constant clock, after which 1 is
// stored to *status (if given) and the kernel ends all the same, so the stream always drains.
// The acquire fence orders what follows on the stream behind the value seen.
__global__ __launch_bounds__(kWave) void wait_value32_kernel(const uint32_t* addr, uint32_t value, uint64_t ticks,
                                                             int* status) {
    if (threadIdx.x != 0) return;
    // a wait earlier on this stream that shares the status word has already run out: the flags are
    // not coming, and waiting for each of them in turn would only add the limit once per wait
    if (status != nullptr && __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != 0) return;
    const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
    while (__hip_atomic_load(addr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != value) {
        if (__builtin_amdgcn_s_memrealtime() - t0 > ticks) {
            if (status != nullptr) __hip_atomic_store(status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            break;
        }
        __builtin_amdgcn_s_sleep(32);
    }
    __atomic_thread_fence(__ATOMIC_ACQUIRE);
}

// All chunks of a gather in one launch, each flagged as it completes.  Workgroups walk runs of 16 KiB pieces in the
// order of the chunks; the pieces are stored through to memory (system scope), the workgroup waits for its stores,
// and one lane counts the run into the chunk's flag word: 2 per run, so that no count makes a 0 read as 1, and the
// workgroup whose count is the last one stores the 1 that readers wait for.  The lowest bit is not part of the count: a
// flag that an earlier gather has left at 1 ends at 1 again.  No cache write-back is needed for that order, where a
// release would also flush what a product running beside this kernel has written.  Nothing here waits for
// anything but its own loads and stores.  At most kGatherGroups workgroups of few registers: they fit beside a GEMM
// workgroup on its compute unit.
//
// What it replaces: a copy kernel and a flag kernel per chunk, sixteen launches for eight shards.  Bound by HBM, or
// by the counts: all flags share a line that takes one count in 12.5 ns, more while tiles poll it, hence runs of up
// to 16 pieces (8 x 16 MiB: 104 us with a count per piece, 43 us with one per 16; eight copies 51; 8 x 1 MiB: 10.8 /
// 7.4 (one per 4) / 42).
constexpr int kPieceVecs = 4;                                // 16-byte vectors per thread and piece
constexpr int kGatherThreads = 256;
constexpr uint32_t kPieceBytes = kGatherThreads * kPieceVecs * 16;
constexpr int kGatherGroups = 1024;

__global__ __launch_bounds__(kGatherThreads) void gather_chunks_kernel(const PeerTab src, int W, int splits, int rank, int64_t chunk_bytes, int run_pieces,
                                                                      uint32_t runs_per_chunk, uint32_t runs, unsigned char* dst, uint32_t* flags) {
    for (uint32_t run = blockIdx.x; run < runs; run += gridDim.x) {
        const uint32_t o = run / runs_per_chunk, in_chunk = run - o * runs_per_chunk;
        const uint32_t step = o / (uint32_t)splits, split = o - step * (uint32_t)splits;
        const uint32_t from = ((uint32_t)rank + 1u + step) % (uint32_t)W;
        const uint32_t chunk = from * (uint32_t)splits + split;
        const char* in0 = (const char*)src.at((int)from) + (int64_t)split * chunk_bytes;
        unsigned char* out0 = dst + (int64_t)chunk * chunk_bytes;
        for (int p = 0; p < run_pieces; ++p) {
            const int64_t off = ((int64_t)in_chunk * run_pieces + p) * kPieceBytes, left = chunk_bytes - off;
            if (left <= 0) break;
            const uint32_t bytes = left < (int64_t)kPieceBytes ? (uint32_t)left : kPieceBytes;
            // (accesses past the piece's end read zeros and store nothing)
            const __amdgpu_buffer_rsrc_t in = stream_rsrc(in0 + off, bytes), out = stream_rsrc(out0 + off, bytes);
            u32x4 v[kPieceVecs];
#pragma unroll
            for (int j = 0; j < kPieceVecs; ++j) v[j] = ld_stream(in, (threadIdx.x + j * kGatherThreads) * 16);
#pragma unroll
            for (int j = 0; j < kPieceVecs; ++j)
                __builtin_amdgcn_raw_buffer_store_b128(v[j], out, (int)((threadIdx.x + j * kGatherThreads) * 16), 0, 1 | 16 /* sc0 sc1: system scope */);
        }
        __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): this wavefront's stores have reached memory
        __syncthreads();
        if (threadIdx.x == 0) {
            const uint32_t before = __hip_atomic_fetch_add(flags + chunk, 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (before >> 1 == runs_per_chunk - 1u) __hip_atomic_store(flags + chunk, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// The two flag primitives the kernels of the all-gather matmul and of the producer GEMM use, in
// one launch: blocks 0 .. P-1 each set their flag (release exchange, as arrive_gmem_barrier with
// op = atomic_xchg), every other block waits for the flag of producer (block - P) / (C / P)
// (acquire load in a loop, as wait_gmem_barrier) -- bounded by `ticks`, after which the block
// stores 1 + flag index to *status and ends.
__global__ __launch_bounds__(kWave) void flag_arrive_wait_kernel(uint32_t* flags, int producers, int consumers,
                                                                uint64_t ticks, int* status) {
    const int b = blockIdx.x;
    if (b < producers) {
        if (threadIdx.x == 0) __hip_atomic_exchange(flags + b, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    const int p = (b - producers) / (consumers / producers);
    const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
    while (__hip_atomic_load(flags + p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) != 1u) {
        if (__builtin_amdgcn_s_memrealtime() - t0 > ticks) {
            if (status != nullptr && threadIdx.x == 0)
                __hip_atomic_store(status, 1 + p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
        }
        __builtin_amdgcn_s_sleep(16);
    }
}

}  // namespace kr

extern "C" int kr_flag_arrive_wait(uint32_t* flags, int producers, int consumers, int64_t wait_limit_us, int* status,
                                   void* stream) {
    if (producers < 1 || consumers < 0 || producers > 4096 || consumers > 65536) return KR_ERR_BAD_DIM;
    if (consumers % producers != 0) return KR_ERR_STRIPE;
    if (flags == nullptr) return KR_ERR_NULL_POINTER;
    if ((reinterpret_cast<uintptr_t>(flags) & 3u) != 0 || (reinterpret_cast<uintptr_t>(status) & 3u) != 0)
        return KR_ERR_ALIGNMENT;
    if (wait_limit_us < 0) return KR_ERR_BAD_DIM;
    const uint64_t ticks = (uint64_t)(wait_limit_us > 0 ? wait_limit_us : 5000000) * 100u;
    hipLaunchKernelGGL(kr::flag_arrive_wait_kernel, dim3((unsigned)(producers + consumers)), dim3(kr::kWave), 0,
                       (hipStream_t)stream, flags, producers, consumers, ticks, status);
    return (int)hipGetLastError();
}

extern "C" int kr_stream_write_value32(uint32_t* addr, uint32_t value, void* stream) {
    if (addr == nullptr) return KR_ERR_NULL_POINTER;
    if ((reinterpret_cast<uintptr_t>(addr) & 3u) != 0) return KR_ERR_ALIGNMENT;
    hipLaunchKernelGGL(kr::write_value32_kernel, dim3(1), dim3(kr::kWave), 0, (hipStream_t)stream, addr, value);
    return (int)hipGetLastError();
}

extern "C" int kr_stream_wait_value32(const uint32_t* addr, uint32_t value, int64_t wait_limit_us, int* status,
                                      void* stream) {
    if (addr == nullptr) return KR_ERR_NULL_POINTER;
    if ((reinterpret_cast<uintptr_t>(addr) & 3u) != 0 || (reinterpret_cast<uintptr_t>(status) & 3u) != 0)
        return KR_ERR_ALIGNMENT;
    if (wait_limit_us < 0) return KR_ERR_BAD_DIM;
    const uint64_t ticks = (uint64_t)(wait_limit_us > 0 ? wait_limit_us : 5000000) * 100u;   // default 5 s
    hipLaunchKernelGGL(kr::wait_value32_kernel, dim3(1), dim3(kr::kWave), 0, (hipStream_t)stream, addr, value, ticks,
                       status);
    return (int)hipGetLastError();
}

extern "C" int kr_gather_chunks(const void* const* srcs, int W, int splits_per_rank, int rank, int64_t chunk_bytes, void* dst,
                                uint32_t* progress, void* stream) {
    if (W < 1 || W > KR_MAX_WORLD) return KR_ERR_WORLD_SIZE;
    if (rank < 0 || rank >= W || splits_per_rank < 1) return KR_ERR_STRIPE;
    if (chunk_bytes < 0 || chunk_bytes % 16 != 0) return KR_ERR_BAD_DIM;
    if ((chunk_bytes > 0 && dst == nullptr) || progress == nullptr) return KR_ERR_NULL_POINTER;
    if (!kr::aligned16(dst) || (reinterpret_cast<uintptr_t>(progress) & 3u) != 0) return KR_ERR_ALIGNMENT;
    kr::PeerTab tab{};   // (of empty chunks only the flags are written: one run each that copies nothing)
    if (chunk_bytes > 0)
        if (const int rc = kr::peer_tab_from_ptrs(tab, srcs, W); rc != KR_OK) return rc;
    const int64_t chunks = (int64_t)W * splits_per_rank, per_chunk = std::max<int64_t>((chunk_bytes + kr::kPieceBytes - 1) / kr::kPieceBytes, 1);
    if (chunks > 0x7fffffff || per_chunk > 0x3fffffff / chunks) return KR_ERR_BAD_DIM;
    const int64_t run_pieces = std::min<int64_t>(std::max<int64_t>(per_chunk * chunks / 128, 1), 16);
    const int64_t runs_per_chunk = (per_chunk + run_pieces - 1) / run_pieces, runs = runs_per_chunk * chunks;
    hipLaunchKernelGGL(kr::gather_chunks_kernel, dim3((unsigned)std::min<int64_t>(runs, kr::kGatherGroups)), dim3(kr::kGatherThreads), 0,
                       (hipStream_t)stream, tab, W, splits_per_rank, rank, chunk_bytes, (int)run_pieces, (uint32_t)runs_per_chunk, (uint32_t)runs,
                       (unsigned char*)dst, progress);
    return (int)hipGetLastError();
}

extern "C" int kr_copy_engine_memcpy(void* dst, const void* src, int64_t bytes, void* stream) {
    if (bytes < 0) return KR_ERR_BAD_DIM;
    if (bytes == 0) return KR_OK;
    if (dst == nullptr || src == nullptr) return KR_ERR_NULL_POINTER;
    // a device-to-device copy that the runtime hands to the copy engines instead of a copy kernel:
    // it takes no CUs from the GEMM that runs beside it
    return (int)hipMemcpyAsync(dst, src, (size_t)bytes, hipMemcpyDeviceToDeviceNoCU, (hipStream_t)stream);
}

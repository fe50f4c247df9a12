// k_readback.hip -- device image to pinned host memory, chunk by chunk (gfx950).
//
// No reference counterpart: the reference presents its image in a window.  The caller's array is
// pageable host memory, which the device cannot write.  The runtime's copy into such memory moves
// a chunk to a pinned buffer, waits, copies it on and only then starts the next one (4 MiB: 240 us).
// Here one launch writes a segment of chunks into pinned memory in order and marks each with the
// launch's number when it is there, so that the host copies one chunk on while the next ones come
// over the link.  Bound by the link and by the host's copying, at about 50 and 32 GB/s.
#include <algorithm>

#include "kernels.hpp"

namespace spr {

namespace {

constexpr int kReadThreads = 512;
// Workgroups on the link at a time: enough for its latency (32 KiB each), few enough that chunks
// arrive one after another.
constexpr int kReadBlocks = 16;

__global__ __launch_bounds__(kReadThreads) void k_read_out(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                           int64_t bytes, uint32_t* __restrict__ arrived,
                                                           uint32_t mark) {
    const int64_t chunks = (bytes + kReadChunk - 1) / kReadChunk;
    const bool wide = (reinterpret_cast<uintptr_t>(src) & 15u) == 0u;  // dst and the chunks are aligned
    for (int64_t c = blockIdx.x; c < chunks; c += gridDim.x) {
        const int64_t o = c * kReadChunk;
        const int n = (int)min((int64_t)kReadChunk, bytes - o);  // whole pixels
        const int n16 = wide ? n >> 4 : 0;
        const uint4* s4 = reinterpret_cast<const uint4*>(src + o);
        uint4* d4 = reinterpret_cast<uint4*>(dst + o);
        for (int i = threadIdx.x; i < n16; i += kReadThreads) d4[i] = s4[i];
        const uint32_t* s1 = reinterpret_cast<const uint32_t*>(src + o);
        uint32_t* d1 = reinterpret_cast<uint32_t*>(dst + o);
        for (int i = 4 * n16 + (int)threadIdx.x; i < n >> 2; i += kReadThreads) d1[i] = s1[i];
        // every wave's stores have reached the host before the mark: a fence waits for the stores of
        // its own wave only, and the barrier for none
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");  // system scope
        __syncthreads();
        if (threadIdx.x == 0)
            __hip_atomic_store(&arrived[c], mark, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

}  // namespace

hipError_t launch_read_out(const uint8_t* src, uint8_t* dst, int64_t bytes, uint32_t* arrived, uint32_t mark,
                           hipStream_t s) {
    if (bytes <= 0) return hipSuccess;
    if (bytes & 3) return hipErrorInvalidValue;
    const int64_t chunks = (bytes + kReadChunk - 1) / kReadChunk;
    k_read_out<<<(unsigned)std::min<int64_t>(chunks, kReadBlocks), kReadThreads, 0, s>>>(src, dst, bytes, arrived, mark);
    return hipGetLastError();
}

}  // namespace spr

// Logits from the host (Session rows that a CPU executor left in pageable memory): the host copies them into pinned memory of the handle, piece
// by piece, and a kernel a piece copies them on while the host fills the next.
// What bounds it: the host's copy (130 GB/s from its caches, 47 from memory), the link (57 GB/s), and 8 us that a launch and its outcome take.
// The runtime's own copy of pageable memory stages and pins in an order of its own, us with it and so: 8 KB 14 and 8, 32 KB 24 and 8.7,
// 128 KB 15 to 61 and 11, 608 KB (a row of 151,936) 29 and 25, out of the host's caches 41 and 29, 2.4 MB 87 and 73, 118 and 86.  An upload and the
// call that samples from it: 1 row of 2,000 40 and 27, of 32,000 41 and 30, of 151,936 55 and 46, 6 of 151,936 154 and 130, 16 of 2,000 176 and 32,
// 16 of 32,000 216 and 87.
#ifndef NCNN_MOE_HIP_SAMPLER_UPLOAD_H
#define NCNN_MOE_HIP_SAMPLER_UPLOAD_H

#include "sampler_bins.h"

namespace ncnn_moe_hip {

constexpr uint32_t kUploadThreads = 256;
constexpr uint32_t kUploadLoads = 2; // vectors a thread: one is 1 us slower at 608 KB, four are the same
// Pieces: one more for each 320 KB, four at most (608 KB in one piece 26.8 us, in two 24.7, in four 29; 2.4 MB in one 95, in three or four 72, in eight 83).
constexpr size_t kUploadPiece = 320u << 10;
constexpr size_t kUploadPieces = 4;
constexpr size_t kUploadStaging = 4u << 20; // a longer upload is the runtime's (9.7 MB 284 us and 237, for as much pinned memory a handle)

// One piece.  done (null: not the last piece): set to 1 once all of it has arrived; `arrived` counts its workgroups, zero between launches.
// The stores pass by the L2 (agent scope): whoever sees `done` may have another XCD read the logits.
__global__ __launch_bounds__(kUploadThreads) void upload_kernel(const uint4* from, void* to, uint32_t vectors, uint32_t* arrived, uint32_t* done)
{
    const uint32_t first = blockIdx.x * kUploadThreads * kUploadLoads + threadIdx.x;
    uint4 v[kUploadLoads];
#pragma unroll
    for (uint32_t k = 0; k < kUploadLoads; ++k)
        v[k] = from[min(first + k * kUploadThreads, vectors - 1u)];
#pragma unroll
    for (uint32_t k = 0; k < kUploadLoads; ++k)
        hand_over_vector(false, to, vectors * 16u, first + k * kUploadThreads, v[k]); // (what lies behind the last is not written)
    if (done == nullptr)
        return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0 && __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1u)
    {
        __hip_atomic_store(arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

} // namespace ncnn_moe_hip

#endif // NCNN_MOE_HIP_SAMPLER_UPLOAD_H

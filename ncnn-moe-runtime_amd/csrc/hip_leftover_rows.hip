// fp32 rows that the window kernels and the binned sums have left: sorted and replayed by one workgroup per row.
//
// A translation unit of its own: a kernel that shares its functions with those of hip_sampler.hip changes how their LDS and scalars
// are laid out there (256 x 201,088 bf16 without a window went from 65.3 to 68.2 us when this kernel stood beside them).
#include "sampler_full_order.h"

#include <hip/hip_runtime.h>

namespace ncnn_moe_hip {

// Sort and replay in ONE kernel: hardly any row is left, and a launch that finds none costs 2.3 us all the same, most of it the gap
// between two launches (33 x 100,003, windows of 200: 52.4 us with two kernels, 51.0 us so; 8 x 151,936 without a window 119.1
// and 117.8 us).
static __global__ __launch_bounds__(kSortThreads) void sort_and_replay_kernel(SamplerArgs a)
{
    static_assert(kSortThreads == kReplayThreads, "the sort and the walk share a workgroup");
    const uint32_t row = blockIdx.x;
    if (a.row_state[row] != kRowNeedsGeneral || left_to_the_wide_select(a, row))
        return;
    sort_whole_row<NCNN_MOE_LOGITS_F32, false>(a, row, threadIdx.x);
    __syncthreads(); // (the sorted keys are in device memory, written by this workgroup)
    replay_sorted_row<NCNN_MOE_LOGITS_F32, false>(a, row, threadIdx.x);
}

void launch_sort_and_replay(const SamplerArgs& a, hipStream_t stream)
{
    hipLaunchKernelGGL(sort_and_replay_kernel, dim3(a.rows), dim3(kSortThreads), 0, stream, a);
}

} // namespace ncnn_moe_hip

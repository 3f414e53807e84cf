// Kernels of the gfx950 generation sampler.
//
//   scan_select_kernel     (sampler_select.h) the one HBM pass over the [rows, vocab] logits for greedy
//                          rows and rows with a Top-K window: streaming, bound, candidate list, exact
//                          best K, the CPU sampler's epilogue.
//   general_sort_kernel    (sampler_full_order.h) full stable order of a row that has no Top-K window
//   general_replay_kernel  and the sampler's walk over it with exactly reproduced sequential sums
//                          (sampler_exact_sum.h).
//   bin_*_kernel           (sampler_bins.h) the same sums without the order: rows with no Top-K window, or one wider
//                          than 1024.
//   window_*_kernel        (sampler_windows.h) rows with a Top-K window of 65 to 1024.
#ifndef NCNN_MOE_HIP_SAMPLER_KERNELS_H
#define NCNN_MOE_HIP_SAMPLER_KERNELS_H

#include "sampler_bins.h"
#include "sampler_full_order.h"
#include "sampler_select.h"
#include "sampler_split.h"
#include "sampler_windows.h"

namespace ncnn_moe_hip {

// hip_leftover_rows.hip: fp32 rows that the windows' and sums' kernels have left pending, sorted and replayed
void launch_sort_and_replay(const SamplerArgs& a, hipStream_t stream);

#ifdef NCNN_MOE_TESTING
// Evaluates expf_libm on n values (test hook; in the testing build of the library only).
__global__ void expf_probe_kernel(const float* in, float* out, size_t n)
{
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        out[i] = expf_libm(in[i]);
}

// Divisor (sampler_bins.h) on n pairs of values (test hook, as above).
__global__ void quotient_probe_kernel(const float* dividends, const float* divisors, float* quotients, size_t n)
{
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        quotients[i] = Divisor(divisors[i]).divide(dividends[i]);
}
#endif

} // namespace ncnn_moe_hip

#endif // NCNN_MOE_HIP_SAMPLER_KERNELS_H

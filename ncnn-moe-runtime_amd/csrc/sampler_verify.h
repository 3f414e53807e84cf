// Speculative verification (src/engine/session.cpp:776-874): the accept loop over the drafted
// tokens and the draw of the token that follows them, from the filtered distributions that the
// sampling kernels exported for the target and draft rows.  One workgroup.
#ifndef NCNN_MOE_HIP_SAMPLER_VERIFY_H
#define NCNN_MOE_HIP_SAMPLER_VERIFY_H

#include "sampler_bins.h"

namespace ncnn_moe_hip {

constexpr int kVerifyThreads = 512;
static_assert(kSumThreads <= kVerifyThreads, "the exact running sums need kSumThreads threads of the workgroup that calls them");
constexpr int kVerifyCap = kSelectTopK; // candidates of a row's filtered distribution the step can use
constexpr int kVerifySlots = kVerifyCap / kWaveSize;

struct VerifyArgs
{
    uint32_t draft_count;
    float temperature;
    const ncnn_moe_sample_result* row_results; // [2 * draft_count + 1]: target rows, then draft rows
    const int32_t* distribution_ids;           // [rows][kVerifyCap]
    const float* distribution_probabilities;
    const uint32_t* distribution_count;        // [rows]: the full kept length, which may exceed kVerifyCap
    const int32_t* proposed;                   // [draft_count]
    const float* uniforms;                     // [draft_count + 1]
    float* accepted_probabilities;             // [draft_count]
    ncnn_moe_verify_result* result;
};

struct VerifyShared
{
    int32_t target_ids[kVerifyCap];
    float target_probabilities[kVerifyCap];
    int32_t draft_ids[kVerifyCap];
    float draft_probabilities[kVerifyCap];
    float ordered_residual[kVerifyCap]; // the residual in token-id order
    int32_t ordered_token[kVerifyCap];
    float found[2];                     // candidate_probability of the proposed token: target, draft
    // the step's small operands, fetched once (proposed tokens and uniforms may lie in host memory)
    ncnn_moe_sample_result row_results[2 * NCNN_MOE_MAX_DRAFT_TOKENS + 1];
    uint32_t counts[2 * NCNN_MOE_MAX_DRAFT_TOKENS + 1];
    int32_t proposed[NCNN_MOE_MAX_DRAFT_TOKENS];
    float uniforms[NCNN_MOE_MAX_DRAFT_TOKENS + 1];
};

__device__ __forceinline__ void write_verify_result(
    const VerifyArgs& v, uint32_t accepted, int32_t token, float probability, uint32_t status, uint32_t row_status,
    uint32_t accept_draws, uint32_t final_draw, uint32_t residual)
{
    ncnn_moe_verify_result r;
    r.accepted = accepted;
    r.next_token_id = status == NCNN_MOE_VERIFY_OK ? token : -1;
    r.next_probability = status == NCNN_MOE_VERIFY_OK ? probability : 0.0f;
    r.status = status;
    r.row_status = row_status;
    r.accept_draws = accept_draws;
    r.final_draw_consumed = final_draw;
    r.next_is_residual = residual;
    *v.result = r;
}

__global__ __launch_bounds__(kVerifyThreads) void speculative_verify_kernel(VerifyArgs v)
{
    __shared__ VerifyShared shared;
    const int tid = threadIdx.x;
    const int lane = tid & (kWaveSize - 1);
    const int wave = tid >> 6;
    const uint32_t drafts = v.draft_count;
    uint32_t accepted = 0;
    uint32_t accept_draws = 0;
    if (static_cast<uint32_t>(tid) < 2u * drafts + 1u)
    {
        shared.row_results[tid] = v.row_results[tid];
        shared.counts[tid] = v.distribution_count[tid];
    }
    if (static_cast<uint32_t>(tid) < drafts)
        shared.proposed[tid] = v.proposed[tid];
    if (static_cast<uint32_t>(tid) <= drafts)
        shared.uniforms[tid] = v.uniforms[tid];
    __syncthreads();

    if (v.temperature == 0.0f)
    {
        // ---- greedy (session.cpp:778-796): a drafted token stands while it is the target's own choice
        for (; accepted < drafts; ++accepted)
        {
            const ncnn_moe_sample_result target = shared.row_results[accepted];
            if (target.status != NCNN_MOE_ROW_OK)
            {
                if (tid == 0)
                    write_verify_result(v, accepted, -1, 0.0f, NCNN_MOE_VERIFY_ROW_ERROR, target.status, 0, 0, 0);
                return;
            }
            if (target.token_id != shared.proposed[accepted])
                break;
            if (tid == 0)
                v.accepted_probabilities[accepted] = 1.0f;
        }
    }
    else
    {
        // ---- session.cpp:797-842: accept with probability min(1, target / draft)
        for (; accepted < drafts; ++accepted)
        {
            const uint32_t target_row = accepted;
            const uint32_t draft_row = drafts + 1u + accepted;
            const ncnn_moe_sample_result target = shared.row_results[target_row];
            const ncnn_moe_sample_result draft = shared.row_results[draft_row];
            if (target.status != NCNN_MOE_ROW_OK || draft.status != NCNN_MOE_ROW_OK)
            {
                const uint32_t row_status = target.status != NCNN_MOE_ROW_OK ? target.status : draft.status;
                if (tid == 0)
                    write_verify_result(v, accepted, -1, 0.0f, NCNN_MOE_VERIFY_ROW_ERROR, row_status, accept_draws, 0, 0);
                return;
            }
            const uint32_t target_count = __builtin_amdgcn_readfirstlane(shared.counts[target_row]);
            const uint32_t draft_count = __builtin_amdgcn_readfirstlane(shared.counts[draft_row]);
            if (target_count > static_cast<uint32_t>(kVerifyCap) || draft_count > static_cast<uint32_t>(kVerifyCap))
            {
                // a filtered distribution longer than the step holds: reported, never approximated
                if (tid == 0)
                    write_verify_result(v, accepted, -1, 0.0f, NCNN_MOE_VERIFY_UNSUPPORTED_WINDOW, 0, accept_draws, 0, 0);
                return;
            }
            const int32_t token = shared.proposed[accepted];
            // ---- candidate_probability (session.cpp:138-148) of the proposed token in both lists; the
            // lists go to LDS on the way, for the residual that a rejection needs
            if (tid < 2)
                shared.found[tid] = 0.0f;
            __syncthreads();
            for (uint32_t j = tid; j < target_count; j += kVerifyThreads)
            {
                const int32_t id = v.distribution_ids[static_cast<size_t>(target_row) * kVerifyCap + j];
                const float probability = v.distribution_probabilities[static_cast<size_t>(target_row) * kVerifyCap + j];
                shared.target_ids[j] = id;
                shared.target_probabilities[j] = probability;
                if (id == token)
                    shared.found[0] = probability; // ids are distinct: at most one writer
            }
            for (uint32_t j = tid; j < draft_count; j += kVerifyThreads)
            {
                const int32_t id = v.distribution_ids[static_cast<size_t>(draft_row) * kVerifyCap + j];
                const float probability = v.distribution_probabilities[static_cast<size_t>(draft_row) * kVerifyCap + j];
                shared.draft_ids[j] = id;
                shared.draft_probabilities[j] = probability;
                if (id == token)
                    shared.found[1] = probability;
            }
            __syncthreads();
            const float target_probability = shared.found[0];
            const float draft_probability = shared.found[1];
            if (draft_probability <= 0.0f)
            {
                if (tid == 0)
                    write_verify_result(v, accepted, -1, 0.0f, NCNN_MOE_VERIFY_ZERO_DRAFT_PROBABILITY, 0, accept_draws, 0, 0);
                return;
            }
            const float ratio = target_probability / draft_probability;
            const float acceptance = ratio < 1.0f ? ratio : 1.0f; // std::min(1.0f, ratio)
            const float uniform = shared.uniforms[accept_draws];
            ++accept_draws;
            if (uniform >= acceptance)
            {
                // ---- rejected: sample_residual_distribution (session.cpp:150-202) over
                // max(0, target - draft), summed and walked in token-id order
                for (uint32_t j = tid; j < target_count; j += kVerifyThreads)
                {
                    const int32_t id = shared.target_ids[j];
                    float residual = shared.target_probabilities[j];
                    int rank = 0;
                    for (uint32_t q = 0; q < draft_count; ++q)
                    {
                        if (shared.draft_ids[q] == id)
                        {
                            const float difference = residual - shared.draft_probabilities[q];
                            residual = 0.0f < difference ? difference : 0.0f; // std::max(0.0f, difference)
                        }
                    }
                    for (uint32_t q = 0; q < target_count; ++q)
                        rank += shared.target_ids[q] < id ? 1 : 0;
                    shared.ordered_residual[rank] = residual;
                    shared.ordered_token[rank] = id;
                }
                __syncthreads();
                if (wave != 0)
                    return;
                // one wave walks the ordered residual: entry i in slot i / 64 of lane i % 64, one fp32
                // addition per entry in order, as std::accumulate over the dense vector does (zeros
                // leave an fp32 sum as it is)
                const int n = static_cast<int>(target_count);
                float residual[kVerifySlots];
#pragma unroll
                for (int s = 0; s < kVerifySlots; ++s)
                {
                    const int i = s * kWaveSize + lane;
                    residual[s] = i < n ? shared.ordered_residual[i] : 0.0f;
                }
                // the sums run in trips of eight entries (a loop trip of a lone wave costs as much as a
                // dozen additions); an entry past the end holds +0.0, which leaves a sum as it is
                float normalizer = 0.0f;
#pragma unroll
                for (int s = 0; s < kVerifySlots; ++s)
                {
                    const int slot_count = min(kWaveSize, n - s * kWaveSize);
                    for (int trip = 0; trip * 8 < slot_count; ++trip)
                    {
#pragma unroll
                        for (int k = 0; k < 8; ++k)
                            normalizer += read_lane(residual[s], trip * 8 + k);
                    }
                }
                if (!is_finite_f32(normalizer) || !(normalizer > 0.0f))
                {
                    if (lane == 0)
                        write_verify_result(v, accepted, -1, 0.0f, NCNN_MOE_VERIFY_RESIDUAL_EMPTY, 0, accept_draws, 0, 1);
                    return;
                }
                // uniform_real_distribution<float>(0, normalizer): canonical draw times the range
                const float sample_value = shared.uniforms[accept_draws] * normalizer;
                float cumulative = 0.0f;
                int selected = -1;
                int last_positive = -1;
#pragma unroll
                for (int s = 0; s < kVerifySlots; ++s)
                {
                    // every lane keeps the running sum at its own entry; one ballot per trip tells
                    // whether the draw has been passed (the first entry that passes it holds mass)
                    float cumulative_here = 0.0f;
                    const int slot_count = selected >= 0 ? 0 : min(kWaveSize, n - s * kWaveSize);
                    for (int trip = 0; trip * 8 < slot_count; ++trip)
                    {
#pragma unroll
                        for (int k = 0; k < 8; ++k)
                        {
                            cumulative += read_lane(residual[s], trip * 8 + k);
                            cumulative_here = lane == trip * 8 + k ? cumulative : cumulative_here;
                        }
                        const uint64_t passed = __ballot(lane < (trip + 1) * 8 && sample_value < cumulative_here);
                        if (passed != 0)
                        {
                            selected = s * kWaveSize + __builtin_ctzll(passed);
                            break;
                        }
                    }
                    const uint64_t positive = __ballot(residual[s] > 0.0f);
                    if (selected < 0 && slot_count > 0 && positive != 0)
                        last_positive = s * kWaveSize + 63 - __builtin_clzll(positive);
                }
                if (selected < 0)
                    selected = last_positive; // session.cpp:189-198: the last token that has any residual mass
                if (selected < 0)
                {
                    if (lane == 0)
                        write_verify_result(v, accepted, -1, 0.0f, NCNN_MOE_VERIFY_RESIDUAL_FAILED, 0, accept_draws, 1, 1);
                    return;
                }
                if (lane == 0)
                    write_verify_result(v, accepted, shared.ordered_token[selected],
                                        shared.ordered_residual[selected] / normalizer, NCNN_MOE_VERIFY_OK, 0,
                                        accept_draws, 1, 1);
                return;
            }
            if (tid == 0)
                v.accepted_probabilities[accepted] = target_probability;
            __syncthreads(); // found[] is reset by the next position
        }
    }

    // ---- session.cpp:871-873: the target's own sample at the first position that was not accepted
    // (greedy mismatch) or after the last drafted token (everything accepted)
    const ncnn_moe_sample_result next = shared.row_results[accepted];
    if (tid == 0)
    {
        if (next.status != NCNN_MOE_ROW_OK)
            write_verify_result(v, accepted, -1, 0.0f, NCNN_MOE_VERIFY_ROW_ERROR, next.status, accept_draws, 0, 0);
        else
            write_verify_result(v, accepted, next.token_id, next.probability, NCNN_MOE_VERIFY_OK, 0, accept_draws,
                                next.draw_consumed, 0);
    }
}

// The same step for filtered distributions of any length (a row without a Top-K window whose Top-P
// keeps more than kVerifyCap tokens): the lists stay in global memory, `list_cap` entries per row, and
// a rejection builds the residual as the CPU does, as a dense vector over the vocabulary
// (session.cpp:150-202): the draft's probabilities are scattered into one vector, max(0, target - draft)
// into another, and the sequential fp32 sum and the walk to the draw over that vector (zeros leave an
// fp32 sum as it is) come from the exact parallel running sum.  One workgroup of kReplayThreads threads.
struct VerifyDenseArgs
{
    VerifyArgs step;       // distribution_ids / distribution_probabilities hold list_cap entries per row
    uint32_t list_cap;
    uint32_t vocab;
    float* dense_draft;    // [vocab]
    float* dense_residual; // [vocab]
};

struct VerifyDenseShared
{
    ReplayScratch replay;
    float found[2];
    int last_positive;
    ncnn_moe_sample_result row_results[2 * NCNN_MOE_MAX_DRAFT_TOKENS + 1];
    uint32_t counts[2 * NCNN_MOE_MAX_DRAFT_TOKENS + 1];
    int32_t proposed[NCNN_MOE_MAX_DRAFT_TOKENS];
    float uniforms[NCNN_MOE_MAX_DRAFT_TOKENS + 1];
};

__global__ __launch_bounds__(kReplayThreads) void speculative_verify_dense_kernel(VerifyDenseArgs d)
{
    __shared__ VerifyDenseShared shared;
    const VerifyArgs& v = d.step;
    const int tid = threadIdx.x;
    const uint32_t drafts = v.draft_count;
    uint32_t accepted = 0;
    uint32_t accept_draws = 0;
    if (static_cast<uint32_t>(tid) < 2u * drafts + 1u)
    {
        shared.row_results[tid] = v.row_results[tid];
        shared.counts[tid] = v.distribution_count[tid];
    }
    if (static_cast<uint32_t>(tid) < drafts)
        shared.proposed[tid] = v.proposed[tid];
    if (static_cast<uint32_t>(tid) <= drafts)
        shared.uniforms[tid] = v.uniforms[tid];
    __syncthreads();

    // ---- session.cpp:797-842 (a greedy step never needs the lists and is served by the kernel above)
    for (; accepted < drafts; ++accepted)
    {
        const uint32_t target_row = accepted;
        const uint32_t draft_row = drafts + 1u + accepted;
        const ncnn_moe_sample_result target = shared.row_results[target_row];
        const ncnn_moe_sample_result draft = shared.row_results[draft_row];
        if (target.status != NCNN_MOE_ROW_OK || draft.status != NCNN_MOE_ROW_OK)
        {
            const uint32_t row_status = target.status != NCNN_MOE_ROW_OK ? target.status : draft.status;
            if (tid == 0)
                write_verify_result(v, accepted, -1, 0.0f, NCNN_MOE_VERIFY_ROW_ERROR, row_status, accept_draws, 0, 0);
            return;
        }
        const uint32_t target_count = __builtin_amdgcn_readfirstlane(shared.counts[target_row]);
        const uint32_t draft_count = __builtin_amdgcn_readfirstlane(shared.counts[draft_row]);
        if (target_count > d.list_cap || draft_count > d.list_cap)
        {
            if (tid == 0)
                write_verify_result(v, accepted, -1, 0.0f, NCNN_MOE_VERIFY_UNSUPPORTED_WINDOW, 0, accept_draws, 0, 0);
            return;
        }
        const int32_t* const target_ids = v.distribution_ids + static_cast<size_t>(target_row) * d.list_cap;
        const float* const target_probabilities = v.distribution_probabilities + static_cast<size_t>(target_row) * d.list_cap;
        const int32_t* const draft_ids = v.distribution_ids + static_cast<size_t>(draft_row) * d.list_cap;
        const float* const draft_probabilities = v.distribution_probabilities + static_cast<size_t>(draft_row) * d.list_cap;
        const int32_t token = shared.proposed[accepted];
        // ---- candidate_probability (session.cpp:138-148) of the proposed token in both lists
        if (tid < 2)
            shared.found[tid] = 0.0f;
        __syncthreads();
        for (uint32_t j = tid; j < target_count; j += kReplayThreads)
        {
            if (target_ids[j] == token)
                shared.found[0] = target_probabilities[j]; // ids are distinct: at most one writer
        }
        for (uint32_t j = tid; j < draft_count; j += kReplayThreads)
        {
            if (draft_ids[j] == token)
                shared.found[1] = draft_probabilities[j];
        }
        __syncthreads();
        const float target_probability = shared.found[0];
        const float draft_probability = shared.found[1];
        if (draft_probability <= 0.0f)
        {
            if (tid == 0)
                write_verify_result(v, accepted, -1, 0.0f, NCNN_MOE_VERIFY_ZERO_DRAFT_PROBABILITY, 0, accept_draws, 0, 0);
            return;
        }
        const float ratio = target_probability / draft_probability;
        const float acceptance = ratio < 1.0f ? ratio : 1.0f; // std::min(1.0f, ratio)
        const float uniform = shared.uniforms[accept_draws];
        ++accept_draws;
        if (uniform >= acceptance)
        {
            // ---- rejected: sample_residual_distribution (session.cpp:150-202), dense over the vocabulary
            for (uint32_t i = tid; i < d.vocab; i += kReplayThreads)
            {
                d.dense_draft[i] = 0.0f;
                d.dense_residual[i] = 0.0f;
            }
            if (tid == 0)
                shared.last_positive = -1;
            __syncthreads();
            for (uint32_t j = tid; j < draft_count; j += kReplayThreads)
                d.dense_draft[draft_ids[j]] = draft_probabilities[j];
            __syncthreads();
            for (uint32_t j = tid; j < target_count; j += kReplayThreads)
            {
                const int32_t id = target_ids[j];
                const float difference = target_probabilities[j] - d.dense_draft[id];
                const float residual = 0.0f < difference ? difference : 0.0f; // std::max(0.0f, difference)
                d.dense_residual[id] = residual;
                if (residual > 0.0f)
                    atomicMax(&shared.last_positive, id);
            }
            __syncthreads();
            const float* const residual = d.dense_residual;
            const RunningSum total = exact_running_sum_of_array<false, false>(residual, 1.0f, 1.0f, d.vocab, kStopNever, 0.0f, shared.replay, tid);
            const float normalizer = total.sum;
            if (!is_finite_f32(normalizer) || !(normalizer > 0.0f))
            {
                if (tid == 0)
                    write_verify_result(v, accepted, -1, 0.0f, NCNN_MOE_VERIFY_RESIDUAL_EMPTY, 0, accept_draws, 0, 1);
                return;
            }
            // uniform_real_distribution<float>(0, normalizer): canonical draw times the range
            const float sample_value = shared.uniforms[accept_draws] * normalizer;
            __syncthreads();
            const RunningSum walk = exact_running_sum_of_array<false, false>(residual, 1.0f, 1.0f, d.vocab, kStopAbove, sample_value, shared.replay, tid);
            // session.cpp:189-198: past the end, the last token that has any residual mass
            const int selected = walk.stopped ? static_cast<int>(walk.stop_index) : shared.last_positive;
            if (selected < 0)
            {
                if (tid == 0)
                    write_verify_result(v, accepted, -1, 0.0f, NCNN_MOE_VERIFY_RESIDUAL_FAILED, 0, accept_draws, 1, 1);
                return;
            }
            if (tid == 0)
                write_verify_result(v, accepted, selected, residual[selected] / normalizer, NCNN_MOE_VERIFY_OK, 0, accept_draws, 1, 1);
            return;
        }
        if (tid == 0)
            v.accepted_probabilities[accepted] = target_probability;
        __syncthreads(); // found[] is reset by the next position
    }

    // ---- session.cpp:871-873: the target's own sample after the last drafted token
    const ncnn_moe_sample_result next = shared.row_results[accepted];
    if (tid == 0)
    {
        if (next.status != NCNN_MOE_ROW_OK)
            write_verify_result(v, accepted, -1, 0.0f, NCNN_MOE_VERIFY_ROW_ERROR, next.status, accept_draws, 0, 0);
        else
            write_verify_result(v, accepted, next.token_id, next.probability, NCNN_MOE_VERIFY_OK, 0, accept_draws,
                                next.draw_consumed, 0);
    }
}

// The same step for rows that the binned sums served (no Top-K window): each row's filtered distribution is known as its
// three sums and its last element kept, so a token's probability needs its logit alone, and nothing is listed.  A
// rejection's residual is a dense vector over the vocabulary, made, summed and walked by three launches, a workgroup per
// 4,096 entries:
//   verify_residual_kernel  the accept loop (every workgroup walks it for itself; the first writes the outcome), and on a
//                           rejection the entries of max(0, target - draft) and their plain sums per 64
//   verify_steps_kernel     what each 64 entries do to a running sum of the exponent that those plain sums foretell, and
//                           what each 4,096 do
//   verify_draw_kernel      the exact sum over the composed steps (entries are looked at only where it leaves its binade),
//                           then the draw inside the one stretch whose partial sums pass it
// What bounds it: launches and trips to memory (the step reads 1.3 MB of logits and 0.6 MB of residual).  With exported
// lists, a pair sort of every row and one workgroup for the residual a step of 5 drafts over 151,936 logits took 640 us.
constexpr uint32_t kResidualSub = kWaveSize;
constexpr uint32_t kResidualChunk = kWaveSize * kResidualSub;
constexpr int kResidualThreads = 512;
constexpr uint32_t kResidualEach = kResidualChunk / kResidualThreads;

struct VerifySumsArgs
{
    SamplerArgs a;                 // logits and options of the 2 * draft_count + 1 rows
    const BinRow* records;         // their filters
    uint32_t draft_count;
    float temperature;
    const int32_t* proposed;       // [draft_count]
    const float* uniforms;         // [draft_count + 1]
    float* accepted_probabilities; // [draft_count]
    ncnn_moe_verify_result* result;
    float* residual;               // [chunks][kResidualChunk]
    float* sub_sums;               // [chunks][kWaveSize]
    uint4* sub_steps;              // [chunks][kWaveSize]: exponent, step on an even mantissa, step on an odd one
    uint4* chunk_steps;            // [chunks]
    double* chunk_sums;            // [chunks]
    int32_t* chunk_last;           // [chunks]: the last entry that holds mass, -1 for none
    uint32_t* decision;            // [0] 1: rejected, the residual decides; [1] positions accepted; [2] uniforms used
};

// The probability of a token in a row's filtered distribution (0 for one that is not in it).
template <int DTYPE>
__device__ __forceinline__ float filtered_probability(const void* row_pointer, uint32_t token, const BinRow& filter, float temperature, const uint64_t* exp2_table)
{
    const float value = load_logit<DTYPE>(row_pointer, token);
    const uint32_t key = descending_key(value);
    if (key > filter.filter_key || (key == filter.filter_key && token > filter.filter_token))
        return 0.0f;
    const float term = expf_libm(value / temperature - filter.maximum, exp2_table);
    return term < filter.least_term ? 0.0f : (term / filter.normalizer) / filter.renormalizer;
}

struct VerifyWalkShared
{
    float found[2 * NCNN_MOE_MAX_DRAFT_TOKENS];
    ncnn_moe_sample_result row_results[2 * NCNN_MOE_MAX_DRAFT_TOKENS + 1];
    BinRow filters[2 * NCNN_MOE_MAX_DRAFT_TOKENS + 1];
    float uniforms[NCNN_MOE_MAX_DRAFT_TOKENS + 1];
    float wave_sums[kResidualThreads / kWaveSize];
    int32_t last;
    uint64_t exp2_table[32];
};

template <int DTYPE>
__global__ __launch_bounds__(kResidualThreads) void verify_residual_kernel(VerifySumsArgs v)
{
    __shared__ VerifyWalkShared shared;
    const SamplerArgs& a = v.a;
    const int tid = threadIdx.x;
    const int lane = tid & (kWaveSize - 1);
    const uint32_t drafts = v.draft_count;
    const uint32_t rows = 2u * drafts + 1u;
    const bool writes = blockIdx.x == 0u && tid == 0;
    const auto row_pointer = [&a](uint32_t row) {
        return static_cast<const void*>(static_cast<const char*>(a.logits) + static_cast<size_t>(row) * a.row_stride * LogitsVector<DTYPE>::kElementBytes);
    };
    const auto outcome = [&](uint32_t accepted, int32_t token, float probability, uint32_t status, uint32_t row_status, uint32_t accept_draws, uint32_t final_draw) {
        if (!writes)
            return;
        v.decision[0] = 0u;
        ncnn_moe_verify_result r;
        r.accepted = accepted;
        r.next_token_id = status == NCNN_MOE_VERIFY_OK ? token : -1;
        r.next_probability = status == NCNN_MOE_VERIFY_OK ? probability : 0.0f;
        r.status = status;
        r.row_status = row_status;
        r.accept_draws = accept_draws;
        r.final_draw_consumed = final_draw;
        r.next_is_residual = 0;
        *v.result = r;
    };
    if (static_cast<uint32_t>(tid) < rows)
    {
        shared.row_results[tid] = a.results[tid];
        shared.filters[tid] = v.records[tid];
    }
    if (static_cast<uint32_t>(tid) <= drafts)
        shared.uniforms[tid] = v.uniforms[tid];
    if (tid >= kWaveSize && tid < kWaveSize + 32)
        shared.exp2_table[tid - kWaveSize] = kExp2Table[tid - kWaveSize];
    if (tid == 0)
        shared.last = -1;
    __syncthreads();
    // candidate_probability (session.cpp:138-148) of every proposed token: the targets', then the drafts'
    if (static_cast<uint32_t>(tid) < 2u * drafts)
    {
        const uint32_t i = static_cast<uint32_t>(tid) % drafts;
        const uint32_t row = static_cast<uint32_t>(tid) < drafts ? i : drafts + 1u + i;
        const uint32_t token = static_cast<uint32_t>(v.proposed[i]);
        shared.found[tid] = token < a.vocab && shared.filters[row].filtered != 0u
            ? filtered_probability<DTYPE>(row_pointer(row), token, shared.filters[row], v.temperature, shared.exp2_table) : 0.0f;
    }
    __syncthreads();
    // ---- session.cpp:797-842: accept with probability min(1, target / draft)
    uint32_t accepted = 0;
    for (; accepted < drafts; ++accepted)
    {
        const ncnn_moe_sample_result target = shared.row_results[accepted];
        const ncnn_moe_sample_result draft = shared.row_results[drafts + 1u + accepted];
        if (target.status != NCNN_MOE_ROW_OK || draft.status != NCNN_MOE_ROW_OK)
            return outcome(accepted, -1, 0.0f, NCNN_MOE_VERIFY_ROW_ERROR, target.status != NCNN_MOE_ROW_OK ? target.status : draft.status, accepted, 0);
        // (a row that the sort served has no filter: the step is run again with exported lists)
        if (shared.filters[accepted].filtered == 0u || shared.filters[drafts + 1u + accepted].filtered == 0u)
            return outcome(accepted, -1, 0.0f, NCNN_MOE_VERIFY_UNSUPPORTED_WINDOW, 0, accepted, 0);
        const float target_probability = shared.found[accepted];
        const float draft_probability = shared.found[drafts + accepted];
        if (draft_probability <= 0.0f)
            return outcome(accepted, -1, 0.0f, NCNN_MOE_VERIFY_ZERO_DRAFT_PROBABILITY, 0, accepted, 0);
        const float ratio = target_probability / draft_probability;
        const float acceptance = ratio < 1.0f ? ratio : 1.0f; // std::min(1.0f, ratio)
        if (shared.uniforms[accepted] >= acceptance)
            break;
        if (writes)
            v.accepted_probabilities[accepted] = target_probability;
    }
    if (accepted == drafts)
    {
        // ---- session.cpp:871-873: the target's own sample after the last drafted token
        const ncnn_moe_sample_result next = shared.row_results[accepted];
        if (next.status != NCNN_MOE_ROW_OK)
            return outcome(accepted, -1, 0.0f, NCNN_MOE_VERIFY_ROW_ERROR, next.status, accepted, 0);
        return outcome(accepted, next.token_id, next.probability, NCNN_MOE_VERIFY_OK, 0, accepted, next.draw_consumed);
    }
    // ---- rejected: this workgroup's entries of max(0, target - draft) (session.cpp:150-202)
    if (writes)
    {
        v.decision[0] = 1u;
        v.decision[1] = accepted;
        v.decision[2] = accepted + 1u;
    }
    const void* const target_logits = row_pointer(accepted);
    const void* const draft_logits = row_pointer(drafts + 1u + accepted);
    const BinRow& target_filter = shared.filters[accepted];
    const BinRow& draft_filter = shared.filters[drafts + 1u + accepted];
    const uint32_t first = blockIdx.x * kResidualChunk + static_cast<uint32_t>(tid) * kResidualEach;
    float own[kResidualEach];
    float sum = 0.0f;
    int32_t last = -1;
#pragma unroll
    for (uint32_t j = 0; j < kResidualEach; ++j)
    {
        const uint32_t token = first + j;
        own[j] = 0.0f;
        if (token < a.vocab)
        {
            const float target = filtered_probability<DTYPE>(target_logits, token, target_filter, v.temperature, shared.exp2_table);
            if (target > 0.0f)
            {
                const float difference = target - filtered_probability<DTYPE>(draft_logits, token, draft_filter, v.temperature, shared.exp2_table);
                own[j] = 0.0f < difference ? difference : 0.0f; // std::max(0.0f, difference)
                last = own[j] > 0.0f ? static_cast<int32_t>(token) : last;
            }
        }
        sum += own[j];
    }
    float* const out = v.residual + static_cast<size_t>(blockIdx.x) * kResidualChunk + static_cast<uint32_t>(tid) * kResidualEach;
#pragma unroll
    for (uint32_t j = 0; j < kResidualEach; j += 4u)
        *reinterpret_cast<float4*>(out + j) = float4{own[j], own[j + 1], own[j + 2], own[j + 3]};
    // plain sums of 64 entries (eight threads') and of the chunk
    static_assert(kResidualSub / kResidualEach == 8, "eight threads hold the entries of a plain sum");
    sum += __shfl_xor(sum, 1, kWaveSize);
    sum += __shfl_xor(sum, 2, kWaveSize);
    sum += __shfl_xor(sum, 4, kWaveSize);
    if ((tid & 7) == 0)
        v.sub_sums[static_cast<size_t>(blockIdx.x) * kWaveSize + (tid >> 3)] = sum;
    sum += __shfl_xor(sum, 8, kWaveSize);
    sum += __shfl_xor(sum, 16, kWaveSize);
    sum += __shfl_xor(sum, 32, kWaveSize);
    if (lane == 0)
        shared.wave_sums[tid >> 6] = sum;
    if (last >= 0)
        atomicMax(&shared.last, last);
    __syncthreads();
    if (tid == 0)
    {
        double total = 0.0;
        for (int w = 0; w < kResidualThreads / kWaveSize; ++w)
            total += shared.wave_sums[w];
        v.chunk_sums[blockIdx.x] = total;
        v.chunk_last[blockIdx.x] = shared.last;
    }
}

__global__ __launch_bounds__(kResidualThreads) void verify_steps_kernel(VerifySumsArgs v)
{
    constexpr uint32_t kWaves = kResidualThreads / kWaveSize;
    __shared__ uint4 steps[kWaveSize];
    __shared__ double wave_sums[kWaves];
    if (v.decision[0] == 0u)
        return;
    const int tid = threadIdx.x;
    const int lane = tid & (kWaveSize - 1);
    const uint32_t wave = same_in_all(static_cast<uint32_t>(tid) >> 6);
    const uint32_t chunk = blockIdx.x;
    float own[kWaveSize / kWaves];
#pragma unroll
    for (uint32_t k = 0; k < kWaveSize / kWaves; ++k)
        own[k] = v.residual[static_cast<size_t>(chunk) * kResidualChunk + (k * kWaves + wave) * kResidualSub + lane];
    const float sub_sum = v.sub_sums[static_cast<size_t>(chunk) * kWaveSize + lane];
    // what the chunks in front of this one add up to, about
    double before = 0.0;
    for (uint32_t c = tid; c < chunk; c += kResidualThreads)
        before += v.chunk_sums[c];
#pragma unroll
    for (int distance = kWaveSize / 2; distance > 0; distance >>= 1)
        before += __shfl_xor(before, distance, kWaveSize);
    if (lane == 0)
        wave_sums[wave] = before;
    __syncthreads();
    before = 0.0;
    for (uint32_t w = 0; w < kWaves; ++w)
        before += wave_sums[w];
    const float front = static_cast<float>(before) + (wave_prefix_sum_f32(sub_sum) - sub_sum); // lane l: in front of the l-th 64 entries
#pragma unroll
    for (uint32_t k = 0; k < kWaveSize / kWaves; ++k)
    {
        const uint32_t sub = k * kWaves + wave;
        const uint32_t exponent = max(same_in_all(__float_as_uint(read_lane(front, static_cast<int>(sub)))) >> 23, 1u);
        const ParityStep through = wave_scan_steps(step_of_term(own[k], static_cast<int>(exponent)));
        if (lane == kWaveSize - 1)
            steps[sub] = uint4{exponent, through.even, through.odd, 0u};
    }
    __syncthreads();
    if (wave == 0u)
    {
        // the chunk's own step, where all of it lies in one binade (else an exponent that no sum has)
        const uint4 mine = steps[lane];
        v.sub_steps[static_cast<size_t>(chunk) * kWaveSize + lane] = mine;
        const ParityStep through = wave_scan_steps(ParityStep{mine.y, mine.z});
        const uint32_t first_exponent = same_in_all(mine.x);
        const bool one_binade = __builtin_amdgcn_ballot_w64(mine.x != first_exponent) == 0ull;
        if (lane == kWaveSize - 1)
            v.chunk_steps[chunk] = uint4{one_binade ? first_exponent : 0u, through.even, through.odd, 0u};
    }
}

// Adds up to 64 composed steps, lane l's `mine` (exponent, even, odd) the l-th, from `first` on, as long as each has the
// sum's exponent and leaves the mantissa below the goal.  Returns the first that does not; `behind` is every lane's sum.
__device__ __forceinline__ uint32_t add_composed_steps(const uint4& mine, uint32_t first, uint32_t count, int mode, float bound, float& sum, float& behind)
{
    const uint32_t lane = static_cast<uint32_t>(lane_id());
    int exponent;
    uint32_t mantissa;
    decode_sum(sum, exponent, mantissa);
    const uint32_t goal = min(stop_mantissa(mode, bound, exponent), kBinadeFull);
    const bool ahead = lane >= first && lane < count;
    const bool usable = ahead && mine.x == static_cast<uint32_t>(exponent);
    const ParityStep through = wave_scan_steps(ParityStep{usable ? mine.y : 0u, usable ? mine.z : 0u});
    const uint32_t after = apply_step(mantissa, through);
    behind = encode_sum(exponent, min(after, kBinadeFull - 1u));
    const uint64_t bad = __builtin_amdgcn_ballot_w64(ahead && !(usable && after < goal));
    const uint32_t first_bad = bad != 0ull ? static_cast<uint32_t>(__builtin_ctzll(bad)) : count;
    if (first_bad > first)
        sum = read_lane(behind, static_cast<int>(first_bad - 1u));
    return first_bad;
}

__global__ __launch_bounds__(kResidualThreads) void verify_draw_kernel(VerifySumsArgs v, uint32_t chunks)
{
    __shared__ __align__(16) float entries[kResidualSub];
    __shared__ __align__(16) float in_order[kWaveSize];
    if (v.decision[0] == 0u || threadIdx.x >= kWaveSize)
        return;
    const uint32_t lane = threadIdx.x;
    const uint32_t accepted = v.decision[1];
    const uint32_t accept_draws = v.decision[2];
    const float uniform = v.uniforms[accept_draws];
    // one chunk, 64 entries at a time; true where the stop condition holds at entry `index`
    const auto walk_chunk = [&](uint32_t chunk, int mode, float bound, float& sum, uint32_t& index) -> bool {
        const uint4 mine = v.sub_steps[static_cast<size_t>(chunk) * kWaveSize + lane];
        float behind;
        for (uint32_t sub = 0; sub < kWaveSize;)
        {
            sub = add_composed_steps(mine, sub, kWaveSize, mode, bound, sum, behind);
            if (sub == kWaveSize)
                break;
            const uint32_t first = chunk * kResidualChunk + sub * kResidualSub;
            entries[lane] = v.residual[first + lane];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            __builtin_amdgcn_wave_barrier();
            const WaveSum result = wave_add_in_order<0>(entries, kResidualSub, sum, mode, bound, 1.0f, 1.0f, in_order);
            __builtin_amdgcn_wave_barrier();
            sum = result.sum;
            if (result.stopped)
            {
                index = first + result.index;
                return true;
            }
            ++sub;
        }
        return false;
    };
    const auto finish = [&](int32_t token, float probability, uint32_t status, uint32_t final_draw) {
        if (lane != 0u)
            return;
        ncnn_moe_verify_result r;
        r.accepted = accepted;
        r.next_token_id = status == NCNN_MOE_VERIFY_OK ? token : -1;
        r.next_probability = status == NCNN_MOE_VERIFY_OK ? probability : 0.0f;
        r.status = status;
        r.row_status = 0;
        r.accept_draws = accept_draws;
        r.final_draw_consumed = final_draw;
        r.next_is_residual = 1;
        *v.result = r;
    };
    // ---- the sum.  Every chunk's partial sum is kept (in place of its composed step)
    float sum = 0.0f;
    int32_t last = -1;
    float* const partial = reinterpret_cast<float*>(v.chunk_sums);
    for (uint32_t base = 0; base < chunks; base += kWaveSize)
    {
        const uint32_t count = min(chunks - base, static_cast<uint32_t>(kWaveSize));
        const uint4 mine = lane < count ? v.chunk_steps[base + lane] : uint4{0u, 0u, 0u, 0u};
        last = max(last, lane < count ? v.chunk_last[base + lane] : -1);
        float own = 0.0f; // the sum behind the lane's chunk
        for (uint32_t c = 0; c < count;)
        {
            float behind;
            const uint32_t stop = add_composed_steps(mine, c, count, kStopNever, 0.0f, sum, behind);
            own = lane >= c && lane < stop ? behind : own;
            c = stop;
            if (c == count)
                break;
            uint32_t index = 0;
            walk_chunk(base + c, kStopNever, 0.0f, sum, index);
            own = lane == c ? sum : own;
            ++c;
        }
        if (lane < count)
            partial[base + lane] = own;
    }
    last = static_cast<int32_t>(wave_max_u32(static_cast<uint32_t>(last + 1))) - 1;
    const float normalizer = sum;
    if (!is_finite_f32(normalizer) || !(normalizer > 0.0f))
        return finish(-1, 0.0f, NCNN_MOE_VERIFY_RESIDUAL_EMPTY, 0);
    // ---- the draw: uniform_real_distribution<float>(0, normalizer) is the canonical draw times the range.  The first
    // partial sum above it lies in the first chunk whose last one is.
    const float sample_value = uniform * normalizer;
    int32_t selected = last; // session.cpp:189-198: past the end, the last token that has any residual mass
    float before = 0.0f;
    for (uint32_t base = 0; base < chunks; base += kWaveSize)
    {
        const uint32_t count = min(chunks - base, static_cast<uint32_t>(kWaveSize));
        const float own = lane < count ? partial[base + lane] : 0.0f;
        const uint64_t passing = __builtin_amdgcn_ballot_w64(lane < count && own > sample_value);
        if (passing != 0ull)
        {
            const int c = __builtin_ctzll(passing);
            if (c > 0)
                before = read_lane(own, c - 1);
            uint32_t index = 0;
            if (walk_chunk(base + static_cast<uint32_t>(c), kStopAbove, sample_value, before, index))
                selected = static_cast<int32_t>(index);
            break;
        }
        before = read_lane(own, static_cast<int>(count) - 1);
    }
    if (selected < 0)
        return finish(-1, 0.0f, NCNN_MOE_VERIFY_RESIDUAL_FAILED, 1);
    finish(selected, v.residual[selected] / normalizer, NCNN_MOE_VERIFY_OK, 1);
}

} // namespace ncnn_moe_hip

#endif // NCNN_MOE_HIP_SAMPLER_VERIFY_H

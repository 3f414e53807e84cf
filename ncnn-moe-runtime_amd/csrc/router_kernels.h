// Expert router kernels (src/graph/expert_dispatcher.cpp:12-157 of the runtime, on the device):
//   router_select_kernel  up to 256 tokens: scores, Top-K routes, normalised weights, and the routes to their places
//   router_batch_kernel   more tokens: scores, Top-K routes, normalised weights
//   router_group_kernel   ... and one workgroup per 256 tokens: their routes to their places in the plan
#ifndef NCNN_MOE_HIP_ROUTER_KERNELS_H
#define NCNN_MOE_HIP_ROUTER_KERNELS_H

#include "ncnn_moe_hip_router.h"
#include "sampler_device.h"

namespace ncnn_moe_hip {

constexpr int kRouterWavesPerBlock = 8;
constexpr int kRouterThreads = kRouterWavesPerBlock * kWaveSize;
constexpr int kRouterChunkTokens = 256; // tokens whose routes one workgroup of the grouping kernel places

// log1pf bit-identical to glibc 2.35's (sysdeps/ieee754/flt-32/s_log1pf.c) for finite x > 0, which is
// all stable_softplus hands it (an exponential).  Plain fp32 operations in the library's order; built
// without contraction, so every one rounds once.  Compared with libm on every positive float.
// log1pf_libm_general: for x of 2^-29 or more and finite.  The library's range cases (x < 0.41422: no reduction; x < 2^53:
// reduce 1 + x and keep the rounding error of the sum as a correction; above: reduce x itself; 1 + x next to a power of
// two: a shorter series) are selects, so that lanes in different ranges, and a lane's experts, share one instruction stream.
__device__ __forceinline__ float log1pf_libm_general(float x)
{
    const float ln2_hi = 6.9313812256e-01f, ln2_lo = 9.0580006145e-06f;
    const float Lp1 = 6.6666668653e-01f, Lp2 = 4.0000000596e-01f, Lp3 = 2.8571429849e-01f, Lp4 = 2.2222198546e-01f,
                Lp5 = 1.8183572590e-01f, Lp6 = 1.5313838422e-01f, Lp7 = 1.4798198640e-01f;
    const int32_t hx = static_cast<int32_t>(__float_as_uint(x));
    const bool direct = hx < 0x3ed413d7;
    const bool huge = hx >= 0x5a000000;
    float u = huge ? x : 1.0f + x;
    int32_t hu = static_cast<int32_t>(__float_as_uint(u));
    int32_t k = (hu >> 23) - 127;
    float c = (k > 0) ? 1.0f - (u - x) : x - (u - 1.0f); // correction term
    c = huge ? 0.0f : c / u;
    hu &= 0x007fffff;
    const bool low_half = hu < 0x3504f7;
    u = __uint_as_float(static_cast<uint32_t>(hu) | (low_half ? 0x3f800000u : 0x3f000000u)); // u, or u / 2
    k = low_half ? k : k + 1;
    hu = low_half ? hu : (0x00800000 - hu) >> 2;
    float f = u - 1.0f;
    k = direct ? 0 : k;
    f = direct ? x : f;
    hu = direct ? 1 : hu;
    const float hfsq = 0.5f * f * f;
    const float kf = static_cast<float>(k);
    const float s = f / (2.0f + f);
    const float z = s * s;
    const float R = z * (Lp1 + z * (Lp2 + z * (Lp3 + z * (Lp4 + z * (Lp5 + z * (Lp6 + z * Lp7))))));
    const float near = f - (hfsq - s * (hfsq + R));
    const float far = kf * ln2_hi - ((hfsq - (s * (hfsq + R) + (kf * ln2_lo + c))) - f);
    // |f| < 2^-20
    const float short_R = hfsq * (1.0f - 0.66666666666666666f * f);
    const float short_near = f == 0.0f ? 0.0f : f - short_R;
    const float short_far = f == 0.0f ? kf * ln2_hi + (c + kf * ln2_lo) : kf * ln2_hi - ((short_R - (kf * ln2_lo + c)) - f);
    const float of_short = k == 0 ? short_near : short_far;
    const float of_long = k == 0 ? near : far;
    return hu == 0 ? of_short : of_long;
}

__device__ __forceinline__ float log1pf_libm_positive(float x)
{
    const int32_t hx = static_cast<int32_t>(__float_as_uint(x));
    if (hx < 0x31000000) // x < 2^-29
    {
        if (hx < 0x24800000) // x < 2^-54
            return x;
        return x - x * x * 0.5f;
    }
    if (hx >= 0x7f800000)
        return x + x;
    return log1pf_libm_general(x);
}

// Wave-wide reductions through the data-parallel primitives: four exchanges inside each row of 16
// lanes (lane pairs at distance 1 and 2, then the two mirrors), then the four rows through scalar reads.
template <int CONTROL>
__device__ __forceinline__ int dpp_move(int value)
{
    return __builtin_amdgcn_mov_dpp(value, CONTROL, 0xf, 0xf, true);
}

constexpr int kDppSwapPairs = 0xB1;   // quad_perm:[1,0,3,2]
constexpr int kDppSwapHalves = 0x4E;  // quad_perm:[2,3,0,1]
constexpr int kDppHalfMirror = 0x141; // row_half_mirror
constexpr int kDppMirror = 0x140;     // row_mirror

__device__ __forceinline__ float wave_max(float value)
{
    value = fmaxf(value, __int_as_float(dpp_move<kDppSwapPairs>(__float_as_int(value))));
    value = fmaxf(value, __int_as_float(dpp_move<kDppSwapHalves>(__float_as_int(value))));
    value = fmaxf(value, __int_as_float(dpp_move<kDppHalfMirror>(__float_as_int(value))));
    value = fmaxf(value, __int_as_float(dpp_move<kDppMirror>(__float_as_int(value))));
    return fmaxf(fmaxf(read_lane(value, 0), read_lane(value, 16)), fmaxf(read_lane(value, 32), read_lane(value, 48)));
}

// expf_libm without its branches, for x finite or -inf: the function's two ends as selects, so that the exponentials of a
// lane's experts overlap (one behind the other, each waits for its table entry and its chain of double operations).
__device__ __forceinline__ float expf_selects(float x, const uint64_t* exp2_table)
{
    const float y = expf_of_small_argument(fminf(fmaxf(x, -104.0f), 89.0f), exp2_table);
    return x < -0x1.9fe368p6f ? 0.0f : x > 0x1.62e42ep6f ? __builtin_inff() : y;
}

// score_router_logit (src/graph/expert_dispatcher.cpp:24-38)
__device__ __forceinline__ float sigmoid_score(float logit, const uint64_t* exp2_table)
{
    return 1.0f / (1.0f + expf_selects(-logit, exp2_table));
}

__device__ __forceinline__ float sqrt_softplus_score(float logit, const uint64_t* exp2_table)
{
    // (the exponential of a logit in [-20, 20] is at least 2^-29 and far below 2^53: log1pf's general range)
    const float exponential = expf_selects(logit, exp2_table);
    const float general = log1pf_libm_general(logit >= -20.0f && logit <= 20.0f ? exponential : 1.0f);
    const float softplus = logit > 20.0f ? logit : logit < -20.0f ? exponential : general;
    return __builtin_sqrtf(softplus); // correctly rounded: built with -fhip-fp32-correctly-rounded-divide-sqrt
}

struct RouterArgs
{
    const float* logits;          // [tokens][experts]
    const float* selection_bias;  // [experts] or null
    const uint32_t* explicit_ids; // [tokens][top_k] or null
    uint32_t tokens;
    uint32_t experts;
    uint32_t top_k;
    uint32_t score_function;
    uint32_t renormalize;
    float scaling;
    uint32_t rank_quads;          // see ranks_quads
    uint32_t* selected_experts;   // [tokens][top_k], rank order
    float* selected_weights;      // [tokens][top_k]
    uint32_t* chunk_counts;       // [chunks][experts] assignments per chunk of 256 tokens and expert, zero at launch
    uint32_t* error_words;        // [0]: non-finite logit seen, [1]: min over failing tokens of (token << 3 | status), ~0 if none
    uint32_t* finished_chunks;    // workgroups of the grouping kernel that are done, zero at launch
    uint32_t* finished_selects;   // workgroups of the fused select kernel that are done, zero at launch
    uint32_t* expert_offsets;     // [experts + 1]
    ncnn_moe_expert_route* routes; // [tokens * top_k]
    uint32_t* status;             // the call's ncnn_moe_router_status
};

// The chunk counters of one chunk, in words: whole groups of four experts.
__host__ __device__ inline uint32_t chunk_count_stride(uint32_t experts)
{
    return (experts + 3u) / 4u * 4u;
}

constexpr uint32_t kRankedQuads = kWaveSize / 4; // see select_best

// Whether the threshold of a token's selection comes from its quads: up to three quarters as many routes as there are quads with experts.  12 routes of 64 experts
// and more find it there mostly (16,384 tokens of 128 experts, softmax, 24.1 -> 21.3 us, of 16 and 3 routes 16.9 -> 14.4); where nearly every quad has to have its
// share above it (10 routes of 20 experts, 16 of 64), most rows are searched as well (20.5 -> 21.1).
__host__ __device__ inline uint32_t ranks_quads(uint32_t experts, uint32_t top_k)
{
    const uint32_t quads = experts < 4u * kRankedQuads ? (experts + 3u) / 4u : kRankedQuads;
    return 4u * top_k <= 3u * quads ? 1u : 0u;
}

// A wave's scratch for the routes of one token.  Its members are read in vectors of 16 bytes.
struct alignas(16) RouteScratch
{
    uint64_t candidates[kWaveSize + 4]; // ordered selection score (32 bits), complement of the expert id (32)
    float scores[kWaveSize + 4];        // the candidates' scores
    float selected[kWaveSize + 4];      // the selected scores, in rank order, then zeros
    uint32_t quads[kRankedQuads];       // the largest key of each four lanes
};
static_assert(offsetof(RouteScratch, candidates) % 16 == 0 && offsetof(RouteScratch, selected) % 16 == 0 && offsetof(RouteScratch, quads) % 16 == 0 &&
                  sizeof(RouteScratch) % 16 == 0,
              "vector reads of a token's scratch");

// This wave's LDS accesses in front of it come before those behind it (a wave's LDS operations run in order: only the
// compiler has to keep it).
__device__ __forceinline__ void wave_lds_fence()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

// The sum of a row of `padded` scores (a multiple of 16), one addition at a time in expert order, as the CPU's loop; lanes
// may sum different rows.  The scores past the last expert are 0, which leaves the sum as it is.
__device__ __forceinline__ float sequential_row_sums(const float* row_of_lane, uint32_t padded)
{
    const float4* quads = reinterpret_cast<const float4*>(row_of_lane);
    float sum = 0.0f;
#pragma unroll 1
    for (uint32_t q = 0; q < padded / 4u; q += 4u)
    {
        float4 four[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            four[k] = quads[q + k];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            sum = (((sum + four[k].x) + four[k].y) + four[k].z) + four[k].w;
    }
    return sum;
}

// The same by 16 lanes: each holds four consecutive scores and adds them to the sum that its lower neighbour holds, 16 times over
// for 64 scores; after turn k the lanes up to k are final.  The wave's four rows of lanes do the same; every lane returns the sum.  256
// scores: 280 instructions and four reads of LDS, where a chain on broadcast reads takes 320 and 64, 512 cycles of the compute unit's LDS
// (300 tokens of 512 experts 17.2 -> 16.1 us, 16,384 of 256 28.7 -> 28.1).
__device__ __forceinline__ float sequential_sum_by_lanes(const float* row, uint32_t padded, int lane)
{
    const int place = lane & 15;
    float sum = 0.0f;
#pragma unroll 1
    for (uint32_t first = 0; first < padded; first += kWaveSize)
    {
        float4 own = *reinterpret_cast<const float4*>(row + first + 4u * static_cast<uint32_t>(place));
        const float carried = __uint_as_float(dpp_source<0x121, 0xf>(__float_as_uint(sum))); // row_ror:1: the first lane reads the last
        own.x = place == 0 ? carried + own.x : own.x;
        sum = 0.0f;
#pragma unroll
        for (int turn = 0; turn < 16; ++turn)
        {
            // (row_shr:1; the first lane reads 0, which leaves its sum as it is)
            sum = (((__uint_as_float(dpp_source<0x111, 0xf>(__float_as_uint(sum))) + own.x) + own.y) + own.z) + own.w;
        }
    }
    return read_lane(sum, 15);
}

// The same for calls of many tokens: a lane's row in a chain of its own beside those of other lanes, the next 16 scores on their way while these are added.
__device__ __forceinline__ float sequential_row_sums_ahead(const float* row_of_lane, uint32_t padded)
{
    const float4* quads = reinterpret_cast<const float4*>(row_of_lane);
    float4 now[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        now[k] = quads[k];
    float sum = 0.0f;
#pragma unroll 2
    for (uint32_t q = 4; q <= padded / 4u; q += 4u)
    {
        float4 next[4];
        const uint32_t ahead = min(q, padded / 4u - 4u);
#pragma unroll
        for (int k = 0; k < 4; ++k)
            next[k] = quads[ahead + k];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            sum = (((sum + now[k].x) + now[k].y) + now[k].z) + now[k].w;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            now[k] = next[k];
    }
    return sum;
}

// ---- select_topk_routes (src/graph/expert_dispatcher.cpp:61-77): the best top_k of a token's experts by (score + bias
// descending, expert id ascending).  Expert e lives in slot e / 64 of lane e % 64.
// A threshold with top_k to `most` scores at or above it: the top_k-th largest of the sixteen numbers that are the largest of four lanes
// each (a ranking of 16 words by way of LDS); some 11 of 256 scores are at or above that for 8 routes, 21 for 12, and top_k are for certain.  With more
// routes than three quarters of the quads, or too many scores above it (a few experts of one quad hold the best), it is searched over the scores'
// order-preserving bits: from the largest score down in growing steps, then by halving, where a step is one comparison per slot, and the
// counting runs on the scalar unit.  The search alone took four steps and more for most tokens (16,384 tokens of 256 experts and 8 routes,
// softmax, selection 8 us of 27.4; so 4.5 of 23.7).  The experts above the threshold are collected in id order and ranked against each
// other.  Where equal scores leave no such threshold, the lowest ids among the equals are collected.
// What bounds it: instructions, some 100 per token of 256 experts and 8 routes, where choosing one route per round by
// wave-wide maxima took some 500.
// Up to kRankedExperts experts are ranked against each other at once, by lane reads: the threshold and the trips through LDS
// cost more there (one token of 8 experts and 2 routes: 6.2 to 6.6 us so, 5.9 to 6.2 ranked; 16 experts are ranked in
// 6.4 us, 6.0 so).
// Returns the sum of the selected scores in rank order (src/graph/expert_dispatcher.cpp:137-143); the calling lane's
// route is `my_expert` with `my_rank` (none: a rank of top_k or more).
constexpr uint32_t kRankedExperts = 8;

template <int SLOTS>
__device__ __forceinline__ float select_best(const RouterArgs& r, bool rank_quads, const float (&score)[SLOTS], const float (&bias)[SLOTS],
                                             RouteScratch& scratch, int lane, uint32_t& my_expert, uint32_t& my_rank, float& my_score)
{
    const uint32_t top_k = r.top_k;
    uint32_t key[SLOTS];
    uint32_t largest = 0u;
#pragma unroll
    for (int s = 0; s < SLOTS; ++s)
    {
        const float keyed = score[s] + bias[s];
        const uint32_t bits = __float_as_uint(keyed); // (never -0: a score is not)
        const uint32_t ordered = bits ^ (static_cast<uint32_t>(static_cast<int32_t>(bits) >> 31) | 0x80000000u);
        key[s] = static_cast<uint32_t>(s * kWaveSize + lane) >= r.experts ? 0u : keyed != keyed ? 1u : ordered;
        largest = max(largest, key[s]);
    }
    if (SLOTS == 1 && r.experts <= kRankedExperts)
    {
        uint32_t rank = 0;
#pragma unroll
        for (uint32_t e = 0; e < kRankedExperts; ++e) // (past the last expert: keys of 0, in front of none)
        {
            const uint32_t other = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(key[0]), static_cast<int>(e)));
            rank += other > key[0] || (other == key[0] && e < static_cast<uint32_t>(lane)) ? 1u : 0u;
        }
        my_expert = static_cast<uint32_t>(lane);
        my_rank = my_expert < r.experts ? rank : 0xffffffffu;
        my_score = score[0];
        float selected_sum = 0.0f;
        for (uint32_t i = 0; i < top_k; ++i)
            selected_sum += read_lane(my_score, __builtin_ctzll(__builtin_amdgcn_ballot_w64(my_rank == i)));
        return selected_sum;
    }
    const auto count_from = [&](uint32_t least) {
        uint32_t count = 0;
#pragma unroll
        for (int s = 0; s < SLOTS; ++s)
            count += static_cast<uint32_t>(__popcll(__builtin_amdgcn_ballot_w64(key[s] >= least)));
        return count;
    };
    const uint32_t most = min(static_cast<uint32_t>(kWaveSize), top_k + top_k / 2u + 8u);
    uint32_t threshold;
    uint32_t equals = 0xffffffffu; // how many scores that equal the threshold are taken
    bool search = !rank_quads;
    if (!search)
    {
        uint32_t of_quad = largest;
        of_quad = max(of_quad, static_cast<uint32_t>(dpp_move<kDppSwapPairs>(static_cast<int>(of_quad))));
        of_quad = max(of_quad, static_cast<uint32_t>(dpp_move<kDppSwapHalves>(static_cast<int>(of_quad))));
        scratch.quads[lane >> 2] = of_quad; // (four lanes, the same number)
        wave_lds_fence();
        const uint4 others = *reinterpret_cast<const uint4*>(&scratch.quads[4 * (lane & 3)]);
        int above = (others.x > of_quad ? 1 : 0) + (others.y > of_quad ? 1 : 0) + (others.z > of_quad ? 1 : 0) + (others.w > of_quad ? 1 : 0);
        above += dpp_move<kDppSwapPairs>(above);
        above += dpp_move<kDppSwapHalves>(above);
        const uint64_t kth = __builtin_amdgcn_ballot_w64(above == static_cast<int>(top_k) - 1);
        search = kth == 0ull; // (two quads' largest are the same)
        if (!search)
        {
            threshold = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(of_quad), __builtin_ctzll(kth)));
            search = count_from(threshold) > most;
        }
    }
    if (search)
    {
        largest = wave_max_u32(largest);
        uint32_t low = 1u, high = largest + 1u; // as many as wanted from `low` on, too few from `high` on
        uint32_t step = 1u << 22;               // half a binade
        threshold = largest > step ? largest - step : 1u;
        for (;;)
        {
            const uint32_t count = count_from(threshold);
            if (count >= top_k && count <= most)
                break;
            if (count < top_k)
                high = threshold;
            else
            {
                low = threshold;
                step = 0u;
            }
            if (high - low <= 1u)
            {
                threshold = low;
                equals = top_k - count_from(low + 1u);
                break;
            }
            step = step < 0x40000000u ? step * 2u : step;
            const bool falls = step != 0u && largest - low > step && largest - step < high;
            threshold = falls ? largest - step : low + (high - low) / 2u;
        }
    }
    uint32_t count = 0, equals_before = 0;
#pragma unroll
    for (int s = 0; s < SLOTS; ++s)
    {
        bool taken = key[s] >= threshold;
        if (equals != 0xffffffffu)
        {
            const uint64_t equal = __builtin_amdgcn_ballot_w64(key[s] == threshold);
            taken = key[s] > threshold || (key[s] == threshold && equals_before + static_cast<uint32_t>(lanes_below(equal)) < equals);
            equals_before += static_cast<uint32_t>(__popcll(equal));
        }
        const uint64_t mask = __builtin_amdgcn_ballot_w64(taken);
        if (taken)
        {
            const uint32_t place = count + static_cast<uint32_t>(lanes_below(mask));
            scratch.candidates[place] = (static_cast<uint64_t>(key[s]) << 32) | (0xffffffffu - static_cast<uint32_t>(s * kWaveSize + lane));
            scratch.scores[place] = score[s];
        }
        count += static_cast<uint32_t>(__popcll(mask));
    }
    if (lane < 4)
    {
        scratch.candidates[count + static_cast<uint32_t>(lane)] = 0ull;
        scratch.selected[top_k + static_cast<uint32_t>(lane)] = 0.0f;
    }
    wave_lds_fence();
    const uint64_t mine = static_cast<uint32_t>(lane) < count ? scratch.candidates[lane] : 0ull;
    my_score = static_cast<uint32_t>(lane) < count ? scratch.scores[lane] : 0.0f;
    uint32_t rank = 0;
    for (uint32_t i = 0; i < count; i += 4u)
    {
        const ulonglong2 two = *reinterpret_cast<const ulonglong2*>(&scratch.candidates[i]);
        const ulonglong2 more = *reinterpret_cast<const ulonglong2*>(&scratch.candidates[i + 2u]);
        rank += (two.x > mine ? 1u : 0u) + (two.y > mine ? 1u : 0u) + (more.x > mine ? 1u : 0u) + (more.y > mine ? 1u : 0u);
    }
    my_expert = 0xffffffffu - static_cast<uint32_t>(mine);
    my_rank = static_cast<uint32_t>(lane) < count ? rank : 0xffffffffu;
    if (my_rank < top_k)
        scratch.selected[my_rank] = my_score;
    wave_lds_fence();
    float selected_sum = 0.0f;
    for (uint32_t i = 0; i < top_k; i += 4u)
    {
        const float4 four = *reinterpret_cast<const float4*>(&scratch.selected[i]);
        selected_sum = (((selected_sum + four.x) + four.y) + four.z) + four.w;
    }
    return selected_sum;
}

// The routes that the caller names (src/graph/expert_dispatcher.cpp:124-135), rank = position; `scores`: the token's
// scores, `divisor`: what they still have to be divided by.  False: an id is out of range.
__device__ __forceinline__ bool take_explicit(const RouterArgs& r, const float* scores, float divisor, uint32_t token, int lane, uint32_t& my_expert,
                                              uint32_t& my_rank, float& my_score, float& selected_sum)
{
    const int top_k = static_cast<int>(r.top_k);
    my_expert = lane < top_k ? r.explicit_ids[static_cast<size_t>(token) * r.top_k + lane] : 0u;
    if (__builtin_amdgcn_ballot_w64(my_expert >= r.experts) != 0ull)
    {
        if (lane == 0)
            atomicMin(&r.error_words[1], (token << 3) | NCNN_MOE_ROUTER_EXPERT_OUT_OF_RANGE);
        return false;
    }
    my_rank = lane < top_k ? static_cast<uint32_t>(lane) : 0xffffffffu;
    my_score = lane < top_k ? scores[my_expert] / divisor : 0.0f;
    selected_sum = 0.0f;
    for (int rank = 0; rank < top_k; ++rank)
        selected_sum += read_lane(my_score, rank);
    return true;
}

// A token's routes from its scores in LDS (not yet divided by `divisor`), by one wave.  Not FUSED: `held` has them as well, expert e in slot
// e / 64 of lane e % 64 (zeros past the last expert), and `counts` counts the routes to each expert.
template <int SLOTS, bool FUSED>
__device__ __forceinline__ void route_token(
    const RouterArgs& r, bool rank_quads, const float* scores, const float (&held)[SLOTS], float divisor, RouteScratch& scratch, uint32_t* counts, uint32_t token,
    int lane)
{
    uint32_t my_expert, my_rank;
    float my_score, selected_sum;
    if (r.explicit_ids != nullptr)
    {
        if (!take_explicit(r, scores, divisor, token, lane, my_expert, my_rank, my_score, selected_sum))
            return;
    }
    else
    {
        float score[SLOTS], bias[SLOTS];
#pragma unroll
        for (int s = 0; s < SLOTS; ++s)
        {
            const uint32_t e = static_cast<uint32_t>(s * kWaveSize + lane);
            bias[s] = (e < r.experts && r.selection_bias != nullptr) ? r.selection_bias[e] : 0.0f;
            score[s] = FUSED ? (e < r.experts ? scores[e] : 0.0f) : held[s];
        }
        if (r.score_function == NCNN_MOE_ROUTER_SOFTMAX)
        {
#pragma unroll
            for (int s = 0; s < SLOTS; ++s)
                score[s] = score[s] / divisor;
        }
        selected_sum = select_best<SLOTS>(r, rank_quads, score, bias, scratch, lane, my_expert, my_rank, my_score);
    }
    // ---- src/graph/expert_dispatcher.cpp:144-150
    if (r.renormalize != 0u && selected_sum <= 0.0f)
    {
        if (lane == 0)
            atomicMin(&r.error_words[1], (token << 3) | NCNN_MOE_ROUTER_NON_POSITIVE_SUM);
        return;
    }
    if (my_rank < r.top_k)
    {
        const float weight = (r.renormalize != 0u ? my_score / selected_sum : my_score) * r.scaling;
        uint32_t* const expert_out = &r.selected_experts[static_cast<size_t>(token) * r.top_k + my_rank];
        float* const weight_out = &r.selected_weights[static_cast<size_t>(token) * r.top_k + my_rank];
        if constexpr (FUSED)
        {
            // written through the per-XCD L2: the workgroup that groups the routes may sit on another XCD
            store_agent(expert_out, my_expert);
            store_agent(reinterpret_cast<uint32_t*>(weight_out), __float_as_uint(weight));
        }
        else
        {
            *expert_out = my_expert;
            *weight_out = weight;
            // (a call of one chunk is counted by the workgroup that groups it)
            atomicAdd(&counts[my_expert], 1u);
        }
    }
}

// Calls of more than one chunk: a wave takes a token from its logits to its routes, without waiting for another wave.  Under the softmax
// the scores pass through LDS, so that their sum, one addition at a time in expert order, is a chain of additions on few reads.
// Up to 512 experts the workgroup's routes are counted in LDS and added to the chunk's counters a line at a time: an atomic a route cost as
// much as all the rest where experts are few (8 experts and 2 routes, 2,048 tokens 18.2 -> 9.7 us, 16,384 26.8 -> 14.8; 64 and 6, 1,024 tokens
// 13.2 -> 10.5, 16,384 22.1 -> 18.9; 256 and 8, 16,384 28.7 -> 27.2).  More experts hardly share routes, and the counters' way through LDS costs
// more than it saves (1,024 experts, 257 tokens 22.7 and 22.4, 16,384 76.1 and 75.2 without).
// Two or four tokens a wave: 0 to 15 % slower from 64 experts on.
// The softmax's sums are chains of additions in expert order.  Where a compute unit has more than eight tokens (kChainsApart), those of
// a workgroup's tokens go side by side in the lanes of one wave: 256 additions and 64 reads of LDS for eight tokens, where a token's
// own wave takes 280 instructions.  With fewer there are instructions to spare, and the wave that all wait for is the slowest part (the kernel
// alone, 256 experts, a wave each and side by side: 512 tokens 5.4 and 5.7 us, 2,048 5.7 and 6.0, 4,096 7.2 and 6.8, 8,192 10.5 and 9.2,
// 16,384 17.5 and 15.8).  Up to 64 experts a token's own wave takes 80 instructions, and the choice alone costs its searched rows 1 to 2 % (16,384
// tokens of 20 experts and 10 routes 20.5, 20.8 and 21.1, of 33 and 12 21.7, 21.9 and 22.4: before the quads, a wave each, side by side).
// What bounds it: instructions, some 400 per token of 256 experts under the softmax: 110 for the exponentials, 50 for
// the divisions, 100 for the selection, 40 for its share of the sums.
//
// RANK_QUADS: ranks_quads' answer.  Decided inside the kernel it cost the calls that search up to 2 % (16,384 tokens, softmax and sigmoid: of 20 experts and
// 10 routes 20.5 and 17.3 without quads, 20.7 and 17.6 decided inside, 20.65 and 17.5 so; of 12 and 9 20.4 and 18.2, 20.7 and 18.4, 20.5 and 18.3; of 16 and 8
// 19.1 and 16.0, 19.4 and 16.3, 19.25 and 16.15).
//
// Waves of a workgroup: eight, which add their counts up together (16,384 tokens of 8 experts 14.8 us, with four 16.4).  But four
// from 257 experts on where that gives every compute unit one at most (1,024 tokens): a token is then so much work that waves two to a SIMD
// wait for each other (512 experts, sqrt softplus, 257 tokens 16.6 and 16.0, 1,024 17.3 and 16.4; 1,536 17.5 and 17.7), and from 513 on always
// (1,024 experts, softmax, 257 tokens 22.8 and 21.3, 16,384 64.8 and 63.6).
constexpr int kBatchWaves = 8;
constexpr int kFewBatchWaves = 4;
constexpr uint32_t kFewBatchTokens = 256u * kFewBatchWaves;
constexpr uint32_t kChainsApart = 256u * kBatchWaves; // tokens

template <int SLOTS, int WAVES, bool RANK_QUADS>
__global__ __launch_bounds__(WAVES * kWaveSize) void router_batch_kernel(RouterArgs r)
{
    constexpr int kThreads = WAVES * kWaveSize;
    constexpr bool kCountsInLds = SLOTS <= 8;
    static_assert(kRouterChunkTokens % WAVES == 0, "a workgroup's tokens are of one chunk");
    __shared__ __align__(16) float rows[WAVES][SLOTS * kWaveSize + 4]; // (four more: the rows' chains read other banks)
    __shared__ float sums[WAVES];
    __shared__ __align__(16) RouteScratch scratch[WAVES];
    __shared__ uint32_t workgroup_counts[kCountsInLds ? SLOTS * kWaveSize : 1]; // the workgroup's routes to each expert
    __shared__ uint64_t exp2_table[32];
    const int lane = threadIdx.x & (kWaveSize - 1);
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const uint32_t token = blockIdx.x * WAVES + static_cast<uint32_t>(wave);
    uint32_t* const chunk_counts = r.chunk_counts + static_cast<size_t>(blockIdx.x * WAVES / kRouterChunkTokens) * chunk_count_stride(r.experts);
    const float* const logits = r.logits + static_cast<size_t>(min(token, r.tokens - 1u)) * r.experts;
    float score[SLOTS];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s)
    {
        const uint32_t e = static_cast<uint32_t>(s * kWaveSize + lane);
        score[s] = e < r.experts ? logits[e] : -__builtin_inff();
    }
    if (threadIdx.x < 32)
        exp2_table[threadIdx.x] = kExp2Table[threadIdx.x];
    if constexpr (kCountsInLds)
    {
        for (uint32_t e = threadIdx.x; e < SLOTS * kWaveSize; e += kThreads)
            workgroup_counts[e] = 0u;
    }
    __syncthreads();
    bool finite = true;
    float maximum = -__builtin_inff();
#pragma unroll
    for (int s = 0; s < SLOTS; ++s)
    {
        finite = finite && (static_cast<uint32_t>(s * kWaveSize + lane) >= r.experts || is_finite_f32(score[s]));
        maximum = fmaxf(maximum, score[s]);
    }
    const bool routed = token < r.tokens && __builtin_amdgcn_ballot_w64(!finite) == 0ull; // (the same in all lanes)
    // src/graph/expert_dispatcher.cpp:98-102: any non-finite logit of the call fails it
    if (token < r.tokens && !routed && lane == 0)
        atomicOr(&r.error_words[0], 1u);
    // ---- router_scores (src/graph/expert_dispatcher.cpp:40-59)
    float sum = 1.0f;
    // (past the last expert: 0)
    const auto each_score = [&](auto score_of) {
#pragma unroll
        for (int s = 0; s < SLOTS; ++s)
        {
            const float of_expert = score_of(score[s]);
            score[s] = static_cast<uint32_t>(s * kWaveSize + lane) < r.experts ? of_expert : 0.0f;
            rows[wave][s * kWaveSize + lane] = score[s];
        }
    };
    if (r.score_function == NCNN_MOE_ROUTER_SOFTMAX)
    {
        if (routed)
        {
            maximum = wave_max(maximum);
            each_score([&](float x) { return expf_selects(x - maximum, exp2_table); });
        }
        if (SLOTS > 1 && r.tokens > kChainsApart)
        {
            __syncthreads();
            // (the waves take turns, so that the SIMDs share the chains; a row without routes sums what lies there)
            if (wave == static_cast<int>((blockIdx.x ^ (blockIdx.x >> 3) ^ (blockIdx.x >> 8)) % WAVES) && lane < WAVES)
                sums[lane] = sequential_row_sums_ahead(rows[lane], (r.experts + 15u) / 16u * 16u);
            __syncthreads();
            sum = sums[wave];
        }
        else if (routed)
        {
            wave_lds_fence();
            sum = sequential_sum_by_lanes(rows[wave], (r.experts + kWaveSize - 1u) / kWaveSize * kWaveSize, lane);
        }
    }
    else if (routed)
    {
        if (r.score_function == NCNN_MOE_ROUTER_SIGMOID)
            each_score([&](float x) { return sigmoid_score(x, exp2_table); });
        else
            each_score([&](float x) { return sqrt_softplus_score(x, exp2_table); });
        wave_lds_fence();
    }
    if (routed)
        route_token<SLOTS, false>(r, RANK_QUADS, rows[wave], score, sum, scratch[wave], kCountsInLds ? workgroup_counts : chunk_counts, token, lane);
    if constexpr (kCountsInLds)
    {
        __syncthreads();
        for (uint32_t e = threadIdx.x; e < r.experts; e += kThreads)
        {
            const uint32_t count = workgroup_counts[e];
            if (count != 0u)
                atomicAdd(&chunk_counts[e], count);
        }
    }
}

// Calls of one chunk of tokens (decode-sized): a workgroup takes kStagedTokensPerBlock tokens and all its threads compute
// the scores, one or a few experts each, into LDS; a wave per token then selects from there.  (A token's scores are two
// fifths of a lone wave's time for it; spread over four waves they take a quarter as long.)
constexpr int kStagedTokensPerBlock = 2;
constexpr int kStagedThreadsPerToken = kRouterThreads / kStagedTokensPerBlock;

struct RouterShared
{
    float scores[kStagedTokensPerBlock][NCNN_MOE_ROUTER_MAX_EXPERTS];
    uint32_t non_finite[kStagedTokensPerBlock];    // the token holds a non-finite logit
    float maximum[kRouterWavesPerBlock];           // softmax: the waves' maxima
    RouteScratch scratch[kStagedTokensPerBlock];
    uint64_t exp2_table[32];
};
static_assert(offsetof(RouterShared, scores) % 16 == 0 && offsetof(RouterShared, scratch) % 16 == 0, "vector reads of the tokens' scores and scratch");

__device__ __forceinline__ void stage_token_scores(const RouterArgs& r, RouterShared& shared, uint32_t first_token)
{
    const int slot = threadIdx.x / kStagedThreadsPerToken;
    const int member = threadIdx.x % kStagedThreadsPerToken;
    const uint32_t token = first_token + static_cast<uint32_t>(slot);
    if (threadIdx.x < kStagedTokensPerBlock)
        shared.non_finite[threadIdx.x] = 0u;
    constexpr int kPerThread = NCNN_MOE_ROUTER_MAX_EXPERTS / kStagedThreadsPerToken;
    float logit[kPerThread];
    bool finite = true;
    float maximum = -__builtin_inff();
    const float* logits = r.logits + static_cast<size_t>(token < r.tokens ? token : 0u) * r.experts;
#pragma unroll
    for (int k = 0; k < kPerThread; ++k)
    {
        const uint32_t e = static_cast<uint32_t>(k * kStagedThreadsPerToken + member);
        logit[k] = (token < r.tokens && e < r.experts) ? logits[e] : -__builtin_inff();
        finite = finite && (e >= r.experts || is_finite_f32(logit[k]));
        maximum = fmaxf(maximum, logit[k]);
    }
    if (threadIdx.x < 32)
        shared.exp2_table[threadIdx.x] = kExp2Table[threadIdx.x];
    if (r.score_function == NCNN_MOE_ROUTER_SOFTMAX)
    {
        // the row maximum first (src/graph/expert_dispatcher.cpp:44-46); the sum stays with the selecting wave
        maximum = wave_max(maximum);
        if ((threadIdx.x & (kWaveSize - 1)) == 0)
            shared.maximum[threadIdx.x >> 6] = maximum;
    }
    __syncthreads();
    if (token < r.tokens && !finite)
        shared.non_finite[slot] = 1u;
    if (r.score_function == NCNN_MOE_ROUTER_SOFTMAX)
    {
        constexpr int kWavesPerToken = kStagedThreadsPerToken / kWaveSize;
        maximum = shared.maximum[slot * kWavesPerToken];
#pragma unroll
        for (int w = 1; w < kWavesPerToken; ++w)
            maximum = fmaxf(maximum, shared.maximum[slot * kWavesPerToken + w]);
    }
    // (the row is filled up to a multiple of 64 with zeros; its sum takes it up to a multiple of 16)
    const uint32_t padded = (r.experts + kWaveSize - 1u) / kWaveSize * kWaveSize;
    const auto each_score = [&](auto score_of) {
#pragma unroll
        for (int k = 0; k < kPerThread; ++k)
        {
            const uint32_t e = static_cast<uint32_t>(k * kStagedThreadsPerToken + member);
            if (e < padded)
                shared.scores[slot][e] = e >= r.experts ? 0.0f : score_of(logit[k]);
        }
    };
    if (r.score_function == NCNN_MOE_ROUTER_SOFTMAX)
        each_score([&](float x) { return expf_selects(x - maximum, shared.exp2_table); });
    else if (r.score_function == NCNN_MOE_ROUTER_SIGMOID)
        each_score([&](float x) { return sigmoid_score(x, shared.exp2_table); });
    else
        each_score([&](float x) { return sqrt_softplus_score(x, shared.exp2_table); });
    __syncthreads();
}

// Grouping is a stable counting sort of the flat assignment array (token-major, so already in
// (token, rank) order) by expert id.  The select kernel counts assignments per (chunk of 256 tokens,
// expert); one workgroup per chunk then places its chunk's routes:
//   position = routes of lower experts (all chunks) + this expert's routes in earlier chunks
//              + this expert's routes earlier in the chunk.
// The last workgroup to have read the scratch counters, perhaps while others place their routes, returns them to zero for the next call.
struct GroupShared
{
    uint32_t wave_base[kRouterWavesPerBlock][NCNN_MOE_ROUTER_MAX_EXPERTS];
    uint32_t wave_totals[kRouterWavesPerBlock];
    uint32_t is_last;
    uint32_t routed[NCNN_MOE_ROUTER_MAX_EXPERTS];        // several chunks: routes of all of them
    uint32_t routed_before[NCNN_MOE_ROUTER_MAX_EXPERTS]; // ... and of those in front of this one
};

// What another workgroup of the same launch wrote is read around the L2, what the launch before wrote is not.
template <bool FUSED>
__device__ __forceinline__ uint32_t load_route_word(const uint32_t* address)
{
    return FUSED ? load_agent(address) : *address;
}

constexpr int kGroupExpertsPerThread = NCNN_MOE_ROUTER_MAX_EXPERTS / kRouterThreads; // experts one thread owns, at most
constexpr int kGroupBatch = 8;                                                       // loads in flight per lane

template <bool FUSED>
__device__ __forceinline__ void place_chunk_routes(const RouterArgs& r, GroupShared& shared, uint32_t chunk, uint32_t chunks)
{
    const int tid = threadIdx.x;
    const int lane = tid & (kWaveSize - 1);
    const int wave = tid >> 6;
    const uint32_t experts = r.experts;

    // this wave's tokens of the chunk: consecutive ones, an equal share of the chunk's (a short chunk is
    // spread over all waves: placing is sequential inside a wave); the first loads go out before anything waits
    const uint32_t chunk_first = chunk * kRouterChunkTokens;
    const uint32_t chunk_tokens = min(static_cast<uint32_t>(kRouterChunkTokens), r.tokens - chunk_first);
    const uint32_t share = (chunk_tokens + kRouterWavesPerBlock - 1) / kRouterWavesPerBlock;
    const uint32_t wave_first = static_cast<uint32_t>(wave) * share;
    const uint32_t first_token = chunk_first + wave_first;
    const uint32_t wave_tokens = wave_first < chunk_tokens ? min(share, chunk_tokens - wave_first) : 0u;
    const uint32_t first_assignment = first_token * r.top_k;
    const uint32_t count = wave_tokens * r.top_k;
    uint32_t first_named[kGroupBatch];
    float first_weight[kGroupBatch];
#pragma unroll
    for (int k = 0; k < kGroupBatch; ++k)
    {
        const uint32_t i = static_cast<uint32_t>(k * kWaveSize + lane);
        first_named[k] = i < count ? load_route_word<FUSED>(&r.selected_experts[first_assignment + i]) : 0xffffffffu;
        first_weight[k] = i < count ? __uint_as_float(load_route_word<FUSED>(reinterpret_cast<const uint32_t*>(&r.selected_weights[first_assignment + i]))) : 0.0f;
    }
    const uint32_t non_finite = load_route_word<FUSED>(&r.error_words[0]);
    const uint32_t first_bad = load_route_word<FUSED>(&r.error_words[1]);
    uint32_t status = NCNN_MOE_ROUTER_OK;
    if (non_finite != 0u)
        status = NCNN_MOE_ROUTER_NON_FINITE_LOGIT;
    else if (first_bad != 0xffffffffu)
        status = first_bad & 7u;
    if (chunk == 0 && tid == 0)
        *r.status = status;

    // Several chunks: a workgroup that has read the counters and the error words counts itself, and places its routes while that is under way.
    uint32_t finished = 0u;
    const auto arrive = [&]() {
        if (tid == 0)
            finished = __hip_atomic_fetch_add(r.finished_chunks, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    if (status != NCNN_MOE_ROUTER_OK)
    {
        if constexpr (!FUSED)
        {
            __syncthreads();
            arrive();
        }
        if (chunk == 0)
        {
            for (uint32_t e = tid; e <= experts; e += kRouterThreads)
                r.expert_offsets[e] = 0u;
        }
    }
    else
    {
        // ---- a histogram of the experts of this wave's tokens
        const auto build_histogram = [&]() {
            for (uint32_t e = lane; e < experts; e += kWaveSize)
                shared.wave_base[wave][e] = 0u;
            lds_barrier();
            for (uint32_t first = 0; first < count; first += kGroupBatch * kWaveSize)
            {
                uint32_t named[kGroupBatch];
#pragma unroll
                for (int k = 0; k < kGroupBatch; ++k)
                {
                    const uint32_t i = first + static_cast<uint32_t>(k * kWaveSize + lane);
                    named[k] = first_named[k];
                    if (first != 0u)
                        named[k] = i < count ? load_route_word<FUSED>(&r.selected_experts[first_assignment + i]) : 0xffffffffu;
                }
#pragma unroll
                for (int k = 0; k < kGroupBatch; ++k)
                {
                    if (named[k] != 0xffffffffu)
                        atomicAdd(&shared.wave_base[wave][named[k]], 1u);
                }
            }
            __syncthreads();
        };
        // ---- this thread's experts: their routes in all chunks, and in the chunks before this one.
        // A call of one chunk has no chunk counters: the totals are the sums of the waves' histograms.
        const uint32_t per_thread = (experts + kRouterThreads - 1) / kRouterThreads;
        uint32_t total[kGroupExpertsPerThread];
        uint32_t before[kGroupExpertsPerThread];
#pragma unroll
        for (int j = 0; j < kGroupExpertsPerThread; ++j)
        {
            total[j] = 0u;
            before[j] = 0u;
        }
        if constexpr (FUSED)
        {
            build_histogram();
#pragma unroll
            for (int j = 0; j < kGroupExpertsPerThread; ++j)
            {
                const uint32_t e = tid * per_thread + j;
                if (static_cast<uint32_t>(j) < per_thread && e < experts)
                {
#pragma unroll
                    for (int w = 0; w < kRouterWavesPerBlock; ++w)
                        total[j] += shared.wave_base[w][e];
                }
            }
        }
        else
        {
            // a wave adds every eighth chunk's counters, four experts a lane, the loads of eight chunks in flight together (a
            // load per expert and chunk, a few at a time, was half of the kernel)
            for (uint32_t e = tid; e < experts; e += kRouterThreads)
                shared.routed[e] = shared.routed_before[e] = 0u;
            lds_barrier();
            const uint32_t quads = chunk_count_stride(experts) / 4u;
            for (uint32_t first_quad = 0; first_quad < quads; first_quad += kWaveSize)
            {
                const uint32_t quad = first_quad + static_cast<uint32_t>(lane);
                const uint4* counts = reinterpret_cast<const uint4*>(r.chunk_counts) + min(quad, quads - 1u);
                uint4 of_all{0u, 0u, 0u, 0u}, of_earlier{0u, 0u, 0u, 0u};
                for (uint32_t first = static_cast<uint32_t>(wave); first < chunks; first += kRouterWavesPerBlock * kGroupBatch)
                {
                    uint4 routed[kGroupBatch];
#pragma unroll
                    for (int k = 0; k < kGroupBatch; ++k)
                        routed[k] = counts[static_cast<size_t>(min(first + k * kRouterWavesPerBlock, chunks - 1u)) * quads];
#pragma unroll
                    for (int k = 0; k < kGroupBatch; ++k)
                    {
                        const uint32_t c = first + k * kRouterWavesPerBlock;
                        const uint32_t all = c < chunks ? 0xffffffffu : 0u, earlier = c < chunk ? 0xffffffffu : 0u;
                        of_all.x += routed[k].x & all, of_all.y += routed[k].y & all, of_all.z += routed[k].z & all, of_all.w += routed[k].w & all;
                        of_earlier.x += routed[k].x & earlier, of_earlier.y += routed[k].y & earlier;
                        of_earlier.z += routed[k].z & earlier, of_earlier.w += routed[k].w & earlier;
                    }
                }
                const uint32_t add[8] = {of_all.x, of_all.y, of_all.z, of_all.w, of_earlier.x, of_earlier.y, of_earlier.z, of_earlier.w};
#pragma unroll
                for (uint32_t j = 0; j < 4u; ++j)
                {
                    if (4u * quad + j < experts)
                    {
                        atomicAdd(&shared.routed[4u * quad + j], add[j]);
                        atomicAdd(&shared.routed_before[4u * quad + j], add[4u + j]);
                    }
                }
            }
            lds_barrier();
            arrive();
#pragma unroll
            for (int j = 0; j < kGroupExpertsPerThread; ++j)
            {
                const uint32_t e = tid * per_thread + j;
                if (static_cast<uint32_t>(j) < per_thread && e < experts)
                {
                    total[j] = shared.routed[e];
                    before[j] = shared.routed_before[e];
                }
            }
        }
        uint32_t thread_sum = 0u;
#pragma unroll
        for (int j = 0; j < kGroupExpertsPerThread; ++j)
            thread_sum += total[j];
        uint32_t inclusive = thread_sum;
#pragma unroll
        for (int step = 1; step < kWaveSize; step <<= 1)
        {
            const uint32_t other = __shfl_up(inclusive, step, kWaveSize);
            inclusive += lane >= step ? other : 0u;
        }
        if (lane == kWaveSize - 1)
            shared.wave_totals[wave] = inclusive;
        if constexpr (FUSED)
            __syncthreads();
        else
            build_histogram();
        uint32_t exclusive = inclusive - thread_sum;
        for (int w = 0; w < wave; ++w)
            exclusive += shared.wave_totals[w];
        // ---- first position of each of this thread's experts for each wave of this chunk
#pragma unroll
        for (int j = 0; j < kGroupExpertsPerThread; ++j)
        {
            const uint32_t e = tid * per_thread + j;
            if (static_cast<uint32_t>(j) < per_thread && e < experts)
            {
                if (chunk == 0)
                    r.expert_offsets[e] = exclusive;
                uint32_t running = exclusive + before[j];
#pragma unroll
                for (int w = 0; w < kRouterWavesPerBlock; ++w)
                {
                    const uint32_t here = shared.wave_base[w][e];
                    shared.wave_base[w][e] = running;
                    running += here;
                }
            }
            exclusive += total[j];
        }
        if (chunk == 0 && tid == 0)
            r.expert_offsets[experts] = r.tokens * r.top_k;
        __syncthreads();

        // ---- place the wave's routes, 64 at a time in assignment order
        const int bits = 32 - __clz(static_cast<int>(experts - 1u) | 1);
        for (uint32_t first = 0; first < count; first += kGroupBatch * kWaveSize)
        {
            uint32_t named[kGroupBatch];
            float weight[kGroupBatch];
#pragma unroll
            for (int k = 0; k < kGroupBatch; ++k)
            {
                const uint32_t i = first + static_cast<uint32_t>(k * kWaveSize + lane);
                named[k] = first_named[k];
                weight[k] = first_weight[k];
                if (first != 0u)
                {
                    named[k] = i < count ? load_route_word<FUSED>(&r.selected_experts[first_assignment + i]) : 0xffffffffu;
                    weight[k] = i < count ? __uint_as_float(load_route_word<FUSED>(reinterpret_cast<const uint32_t*>(&r.selected_weights[first_assignment + i]))) : 0.0f;
                }
            }
#pragma unroll
            for (int k = 0; k < kGroupBatch; ++k)
            {
                if (first + static_cast<uint32_t>(k * kWaveSize) >= count)
                    break;
                const bool valid = named[k] != 0xffffffffu;
                uint64_t same = __ballot(valid);
                for (int b = 0; b < bits; ++b)
                {
                    const bool set = ((named[k] >> b) & 1u) != 0u;
                    const uint64_t vote = __ballot(set);
                    same &= set ? vote : ~vote;
                }
                if (valid)
                {
                    const uint32_t earlier = static_cast<uint32_t>(lanes_below(same));
                    const uint32_t position = shared.wave_base[wave][named[k]] + earlier;
                    if (earlier == 0u)
                        shared.wave_base[wave][named[k]] = position + static_cast<uint32_t>(__popcll(same));
                    const uint32_t i = first_assignment + first + static_cast<uint32_t>(k * kWaveSize + lane);
                    ncnn_moe_expert_route route;
                    route.token_index = i / r.top_k;
                    route.rank = i - route.token_index * r.top_k;
                    route.weight = weight[k];
                    r.routes[position] = route;
                }
                // the group leaders' updates, before this wave's next 64 read them (waves run different
                // numbers of rounds: nothing here may wait for another wave)
                __builtin_amdgcn_s_waitcnt(0xc07f);
                __builtin_amdgcn_wave_barrier();
            }
        }
    }

    // ---- the last workgroup to have read the counters and the error words clears them for the next call
    if (tid == 0)
        shared.is_last = FUSED || finished == chunks - 1u ? 1u : 0u;
    __syncthreads();
    if (shared.is_last != 0u)
    {
        for (uint32_t i = tid; !FUSED && i < chunks * (chunk_count_stride(experts) / 4u); i += kRouterThreads)
            reinterpret_cast<uint4*>(r.chunk_counts)[i] = uint4{0u, 0u, 0u, 0u};
        if (tid == 0)
        {
            r.error_words[0] = 0u;
            r.error_words[1] = 0xffffffffu;
            *r.finished_chunks = 0u;
        }
    }
}

__global__ __launch_bounds__(kRouterThreads) void router_group_kernel(RouterArgs r)
{
    __shared__ GroupShared shared;
    place_chunk_routes<false>(r, shared, blockIdx.x, gridDim.x);
}

// Calls of at most one chunk of tokens: the workgroup that finishes last also places the routes, so the whole dispatch is
// one launch.
template <int SLOTS>
__global__ __launch_bounds__(kRouterThreads) void router_select_kernel(RouterArgs r)
{
    __shared__ RouterShared shared;
    __shared__ GroupShared group_shared;
    const int lane = threadIdx.x & (kWaveSize - 1);
    const int wave = threadIdx.x >> 6;
    const uint32_t token = blockIdx.x * kStagedTokensPerBlock + wave;
    stage_token_scores(r, shared, blockIdx.x * kStagedTokensPerBlock);
    if (wave < kStagedTokensPerBlock && token < r.tokens)
    {
        if (shared.non_finite[wave] != 0u)
        {
            // src/graph/expert_dispatcher.cpp:98-102: any non-finite logit of the call fails it
            if (lane == 0)
                atomicOr(&r.error_words[0], 1u);
        }
        else
        {
            const float sum = r.score_function == NCNN_MOE_ROUTER_SOFTMAX ? sequential_row_sums(shared.scores[wave], (r.experts + 15u) / 16u * 16u) : 1.0f;
            const float none[SLOTS] = {};
            route_token<SLOTS, true>(r, r.rank_quads != 0u, shared.scores[wave], none, sum, shared.scratch[wave], nullptr, token, lane);
        }
    }
    // this workgroup's routes (written through), counts and error words (atomics) have landed once
    // its waves have waited for them; then the workgroup is counted, and whoever counts last reads
    // every other workgroup's around its own L2: no cache write-back or invalidate is needed
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0)
    {
        const uint32_t finished = __hip_atomic_fetch_add(r.finished_selects, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        group_shared.is_last = finished == gridDim.x - 1u ? 1u : 0u;
    }
    __syncthreads();
    if (group_shared.is_last == 0u)
        return;
    if (threadIdx.x == 0)
        *r.finished_selects = 0u;
    place_chunk_routes<true>(r, group_shared, 0u, 1u);
}

__global__ void log1pf_probe_kernel(const float* in, float* out, size_t n)
{
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        out[i] = log1pf_libm_positive(in[i]);
}

} // namespace ncnn_moe_hip

#endif // NCNN_MOE_HIP_ROUTER_KERNELS_H

// Rows with a Top-K window of 65 to 1024 (and narrower ones that the first select hands on): candidates, then the walk.
//
//   window_candidates   a row's logits are streamed once, by several workgroups, each of which keeps the logits of its part
//                       that reach a bound and hands them over.  The bound comes from a sample of the whole row (one to
//                       four 16-byte vectors a thread, evenly spaced): with r = row length / sample size, the sample's m-th
//                       largest value is reached by about m r logits of the row, give or take r sqrt(m), and m solves
//                       m r - 5.5 r sqrt(m) = K.  Every workgroup of the row works the bound out for itself.
//   window_finish       one workgroup per row puts the candidates in order (value descending, index ascending) and walks
//                       the window's first K: the three sums with sum_head of sampler_bins.h.
//   window_chain        both in one launch, for calls of no more rows than compute units.
// A row of fewer finite logits than its window has all of them as candidates and ends there.  A row whose candidates are fewer
// than its window because the sample misled, or more than a list holds (thousands of ties), stays pending for the
// full-order kernels.
//
// Bound: the stream at many rows (the row is read once and a part in 24 a second time), the chain sample - stream - order - sums
// at few.  The one-workgroup-per-row select it stands in for took 65 to 115 us at any number of rows.
#ifndef NCNN_MOE_HIP_SAMPLER_WINDOWS_H
#define NCNN_MOE_HIP_SAMPLER_WINDOWS_H

#include "sampler_bins.h"

namespace ncnn_moe_hip {

constexpr uint32_t kWindowListCap = 4096;        // candidates of a row
constexpr uint32_t kWindowSampleRatio = 24;      // logits of the row per logit of the sample aimed at ...
constexpr uint32_t kWindowSampleVectors = 4;     // ... within so many vectors a thread
constexpr uint32_t kWindowMaxVocab = 1u << 19;   // beyond it a window of 1024 may not fit the list
constexpr uint32_t kWindowRankedTies = 256;      // neighbours in value that are ranked against each other; more are sorted
constexpr uint32_t kWindowSawNan = 1u;
constexpr uint32_t kWindowHasAll = 2u;           // every finite logit is a candidate
constexpr uint32_t kWindowBins = 4096;           // of the sample's histogram: the upper twelve bits of a key
constexpr uint32_t kWindowFineBins = 256;

struct WindowArgs
{
    SamplerArgs a;
    uint32_t* list;         // the rows served: [0] their number, then the rows
    uint32_t* counts;       // [rows] candidates; zero when a launch begins (window_finish returns them to zero)
    uint32_t* flags;        // [rows] kWindowSawNan, kWindowHasAll; the same
    uint32_t* keys;         // [rows][kWindowListCap]
    uint32_t* tokens;       // [rows][kWindowListCap]
    uint32_t windows_are_selects; // as in BinArgs
    uint32_t listing;
    uint32_t* other_list;   // where the sums' rows are listed as well (null: nowhere)
    uint32_t turn;          // WindowTurn
    const uint32_t* sums_list; // of the two turns: the sums' rows, listed by an earlier launch
    unsigned long long* arrivals; // as in BinArgs: of a row the word behind those two (see window_chain)
};

// Beside the binned sums the candidates are collected by one of two launches, and the other leaves at once: the number of rows
// of each kind is known to the device only.
enum WindowTurn : uint32_t
{
    kWindowsOnce = 0,
    kWindowsAhead = 1,  // behind the launch that writes the sums' terms: where the windows are the longer piece of work
    kWindowsBehind = 2  // behind the last launch that reads the sums' rows as a stream: everywhere else
};

// Are the windows so much more than the sums that what streams them should not wait for the sums' passes?  The passes over a few
// dozen rows are chains that leave the memory idle, some 45 us, and the walks behind them hide no more than the stream of some 500
// rows of 129,280.  Rows with windows and rows without one, us ahead / behind (Top-K 300, normal logits of spread 2 and 3): 900 and 32
// of 1,024 of 129,280 306 / 352 and 286 / 347, 640 and 32 298 / 306 and 274 / 303, 1,900 and 64 of 2,048 462 / 562 and 446 / 557,
// 2,200 and 64 of 4,096 of 32,000 358 / 401 and 348 / 397, 500 and 64 of 600 of 262,144 390 / 389 and 343 / 380.  With more rows to
// sum behind is faster (640 and 100 of 1,024 335 / 313 and 301 / 301, 1,024 and 500 of 2,048 730 / 676 and 638 / 634), and with fewer
// windows it depends on how long the walks are (400 and 32 of 512, spread 1.5 270 / 247, 2 232 / 250, 3 211 / 241; 230 and 32 of 256 of
// 151,936 198 / 170; 92 and 92 of 512 252 / 226).
constexpr uint32_t kWindowsAheadRatio = 7;
constexpr uint64_t kWindowsAheadLogits = 1ull << 26;

__device__ __forceinline__ bool windows_go_ahead(uint32_t windows, uint32_t sums, uint32_t vocab)
{
    return windows >= kWindowsAheadRatio * sums && static_cast<uint64_t>(windows) * vocab >= kWindowsAheadLogits;
}

struct WindowCandidatesShared
{
    alignas(16) uint32_t counts[kWindowBins];
    uint32_t fine_counts[kWindowFineBins]; // ... of the samples in one of them: the next eight bits
    uint32_t wave_totals[kBinWaves];
    uint32_t keys[kWindowListCap];
    uint32_t tokens[kWindowListCap];
    uint32_t found, above; // see find_from_top
    uint32_t count, base, saw_nan;
};

// The bin of `counts` (from the top) in which the count from the top reaches `wanted` (1 at least, and no more than there are):
// shared.found, and in shared.above what is counted above it.  Every thread calls it.
template <uint32_t BINS, int THREADS>
__device__ __forceinline__ void find_from_top(const uint32_t (&counts)[BINS], WindowCandidatesShared& shared, uint32_t wanted, int tid)
{
    constexpr uint32_t kEach = BINS / THREADS == 0 ? 1 : BINS / THREADS;
    const int wave = tid >> 6;
    const uint32_t first = static_cast<uint32_t>(tid) * kEach; // counted from the top
    uint32_t own[kEach];
    uint32_t total = 0;
#pragma unroll
    for (uint32_t k = 0; k < kEach; ++k)
    {
        own[k] = first + k < BINS ? counts[BINS - 1u - (first + k)] : 0u;
        total += own[k];
    }
    const uint32_t through = wave_prefix_sum_u32(total);
    if ((tid & (kWaveSize - 1)) == kWaveSize - 1)
        shared.wave_totals[wave] = through;
    __syncthreads();
    uint32_t before = through - total;
#pragma unroll
    for (int w = 0; w < THREADS / kWaveSize; ++w)
        before += w < wave ? shared.wave_totals[w] : 0u;
#pragma unroll
    for (uint32_t k = 0; k < kEach; ++k)
    {
        if (before < wanted && before + own[k] >= wanted)
        {
            shared.found = BINS - 1u - (first + k);
            shared.above = before;
        }
        before += own[k];
    }
    __syncthreads();
}

// Everything that bound_of_sample counts in is returned to zero; a barrier has to follow.
template <int THREADS>
__device__ __forceinline__ void clear_sample_counts(WindowCandidatesShared& shared, int tid)
{
    for (uint32_t i = tid; i < kWindowBins / 4u; i += THREADS)
        reinterpret_cast<uint4*>(shared.counts)[i] = uint4{0u, 0u, 0u, 0u};
    if (tid < static_cast<int>(kWindowFineBins))
        shared.fine_counts[tid] = 0u;
}

// How many vectors of a row its sample has, out of `whole`.
__device__ __forceinline__ uint32_t sampled_vectors(uint32_t whole)
{
    return min(whole, min(kWindowSampleVectors, max(1u, whole / (kWindowSampleRatio * kBinThreads))) * kBinThreads);
}

// The key that a row's candidates reach (0: all of them do), from its sample of `sampled` vectors out of `whole`: sample_vector(k, x) gives
// the thread's k-th, k below MOST (UNROLLED: MOST where those are in registers, else 1).  The counts hold zeros (clear_sample_counts); every thread calls it.
template <int DTYPE, int THREADS, uint32_t MOST, uint32_t UNROLLED, typename SampleVector>
__device__ __forceinline__ uint32_t bound_of_sample(
    WindowCandidatesShared& shared, uint32_t vocab, uint32_t window, uint32_t whole, uint32_t sampled, SampleVector sample_vector, int tid)
{
    constexpr uint32_t kWidth = LogitsVector<DTYPE>::kWidth;
#pragma unroll UNROLLED
    for (uint32_t k = 0; k < MOST; ++k)
    {
        float x[kWidth];
        if (k * THREADS < sampled && sample_vector(k, x))
        {
#pragma unroll
            for (uint32_t c = 0; c < kWidth; ++c)
            {
                // (only what can be among the largest matters: a NaN counts as nothing)
                if (x[c] == x[c])
                    atomicAdd(&shared.counts[ascending_key(x[c]) >> 20], 1u);
            }
        }
    }
    __syncthreads();
    const float ratio = static_cast<float>(vocab) / static_cast<float>(max(1u, sampled * kWidth));
    const float root = 0.5f * (5.5f + sqrtf(30.25f + 4.0f * static_cast<float>(window) / ratio));
    const uint32_t wanted = sampled == whole ? min(window, sampled * kWidth) : min(static_cast<uint32_t>(root * root) + 1u, sampled * kWidth);
    if (sampled * kWidth < window + 2u * kWidth) // a short row: its few logits are all candidates
        return 0u;
    // (a row of NaNs only has no sample, and nothing is found)
    if (tid == 0)
        shared.found = 0u, shared.above = 0u;
    find_from_top<kWindowBins, THREADS>(shared.counts, shared, wanted, tid);
    const uint32_t coarse = same_in_all(shared.found);
    const uint32_t still = wanted - same_in_all(shared.above);
    // the next eight bits of the samples in that bin
#pragma unroll UNROLLED
    for (uint32_t k = 0; k < MOST; ++k)
    {
        float x[kWidth];
        if (k * THREADS < sampled && sample_vector(k, x))
        {
#pragma unroll
            for (uint32_t c = 0; c < kWidth; ++c)
            {
                const uint32_t key = ascending_key(x[c]);
                if (x[c] == x[c] && key >> 20 == coarse)
                    atomicAdd(&shared.fine_counts[(key >> 12) & (kWindowFineBins - 1u)], 1u);
            }
        }
    }
    __syncthreads();
    if (tid == 0)
        shared.found = 0u;
    find_from_top<kWindowFineBins, THREADS>(shared.fine_counts, shared, still, tid);
    return (coarse << 20) | (same_in_all(shared.found) << 12);
}

template <int DTYPE>
__device__ __forceinline__ void window_candidates(const WindowArgs& g, const BinGrid& grid, const RowList& listed_rows, WindowCandidatesShared& shared, int tid)
{
    using Vector = LogitsVector<DTYPE>;
    constexpr uint32_t kWidth = Vector::kWidth;
    constexpr int kLoads = DTYPE == NCNN_MOE_LOGITS_F32 ? 4 : 2;
    const SamplerArgs& a = g.a;
    const int lane = tid & (kWaveSize - 1);
    for (uint32_t slot = grid.first_slot; slot < grid.rows; slot += grid.slot_step)
    {
        const uint32_t row = same_in_all(row_of_slot(g.listing, g.list, listed_rows, slot));
        const uint32_t top_k = same_in_all(a.params[row].top_k);
        const uint32_t window = top_k == 0u || top_k >= a.vocab ? a.vocab : top_k;
        const BinStretch s = bin_stretch<Vector::kElementBytes>(a, row, grid.part, grid.parts);
        const char* base = static_cast<const char*>(a.logits) + static_cast<size_t>(row) * a.row_stride * Vector::kElementBytes -
            static_cast<size_t>(s.misalignment) * Vector::kElementBytes;
        // ---- the sample: vectors that lie inside the row as a whole
        const uint32_t first_whole = (s.misalignment + kWidth - 1u) / kWidth;
        const uint32_t whole = s.end / kWidth - min(first_whole, s.end / kWidth);
        const uint32_t sampled = sampled_vectors(whole);
        if (tid == 0)
        {
            shared.count = 0u;
            shared.saw_nan = 0u;
            // (pending until window_finish has finished it: a first select that comes later leaves these rows alone)
            if (grid.part == 0u)
                a.row_state[row] = kRowNeedsGeneral;
        }
        clear_sample_counts<kBinThreads>(shared, tid);
        __syncthreads();
        const auto sample_vector = [&](uint32_t k, float (&x)[kWidth]) -> bool {
            const uint32_t i = k * kBinThreads + tid;
            if (i >= sampled)
                return false;
            const uint32_t v = first_whole + static_cast<uint32_t>(static_cast<uint64_t>(i) * whole / sampled);
            Vector::unpack(*reinterpret_cast<const uint4*>(base + static_cast<size_t>(v) * 16u), x);
            return true;
        };
        const uint32_t reached = bound_of_sample<DTYPE, kBinThreads, kWindowSampleVectors, 1>(shared, a.vocab, window, whole, sampled, sample_vector, tid);
        // (an infinite logit below everything is no candidate: the window counts finite logits)
        const uint32_t lowest = ascending_key(-3.402823466e38f);
        const bool has_all = reached <= lowest;
        const float bound = value_from_ascending_key(max(reached, lowest));
        // ---- the part's logits at or above it
        const uint32_t first = s.first * 8u / kWidth, last = min(s.last * 8u / kWidth, (s.end + kWidth - 1u) / kWidth);
        bool saw_nan = false;
        for (uint32_t at = first + tid; at < last + kBinThreads; at += kLoads * kBinThreads)
        {
            // (whole waves stay in the loop: its appends are theirs)
            if (at - lane >= last)
                break;
            uint4 raw[kLoads];
#pragma unroll
            for (int k = 0; k < kLoads; ++k)
                raw[k] = *reinterpret_cast<const uint4*>(base + static_cast<size_t>(min(at + k * kBinThreads, last - 1u)) * 16u);
#pragma unroll
            for (int k = 0; k < kLoads; ++k)
            {
                const uint32_t v = at + k * kBinThreads;
                float x[kWidth];
                Vector::unpack(raw[k], x);
                const uint32_t position = v * kWidth;
                uint32_t hits = 0;
#pragma unroll
                for (uint32_t c = 0; c < kWidth; ++c)
                {
                    const bool inside = v < last && position + c - s.misalignment < a.vocab;
                    hits |= inside && x[c] >= bound ? 1u << c : 0u;
                    saw_nan = saw_nan || (inside && x[c] != x[c]);
                }
                if (__builtin_amdgcn_ballot_w64(hits != 0u) != 0ull)
                {
                    const uint32_t own = static_cast<uint32_t>(__popc(hits));
                    const uint32_t through = wave_prefix_sum_u32(own);
                    uint32_t place = 0;
                    if (lane == kWaveSize - 1)
                        place = atomicAdd(&shared.count, through);
                    place = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(place), kWaveSize - 1)) + through - own;
#pragma unroll
                    for (uint32_t c = 0; c < kWidth; ++c)
                    {
                        if ((hits >> c & 1u) != 0u)
                        {
                            if (place < kWindowListCap)
                            {
                                shared.keys[place] = ascending_key(x[c]);
                                shared.tokens[place] = position + c - s.misalignment;
                            }
                            ++place;
                        }
                    }
                }
            }
        }
        if (__builtin_amdgcn_ballot_w64(saw_nan) != 0ull && lane == 0)
            shared.saw_nan = 1u;
        __syncthreads();
        // ---- handed over: one counter per row
        const uint32_t count = shared.count;
        if (tid == 0)
        {
            shared.base = count != 0u ? atomicAdd(&g.counts[row], count) : 0u;
            const uint32_t seen = (shared.saw_nan != 0u ? kWindowSawNan : 0u) | (has_all && grid.part == 0u ? kWindowHasAll : 0u);
            if (seen != 0u)
                atomicOr(&g.flags[row], seen);
        }
        __syncthreads();
        const uint32_t place = shared.base;
        for (uint32_t i = tid; i < min(count, kWindowListCap); i += kBinThreads)
        {
            if (place + i < kWindowListCap)
            {
                g.keys[static_cast<size_t>(row) * kWindowListCap + place + i] = shared.keys[i];
                g.tokens[static_cast<size_t>(row) * kWindowListCap + place + i] = shared.tokens[i];
            }
        }
        __syncthreads();
    }
}

struct WindowFinishShared
{
    alignas(16) uint32_t keys[kWindowListCap]; // (keys and tokens together: the pairs that sort_candidates sorts)
    alignas(16) uint32_t tokens[kWindowListCap];
    uint32_t counters[kWindowListCap];
    alignas(16) float terms[kSelectTopK];
    HeadScratch head;
    BinScanScratch scan;
    uint32_t least, most, neighbours;
    uint64_t exp2_table[32];
};

// Puts `count` pairs (key in the upper 32 bits, complement of the token below) in descending order: bitonic, in LDS.  Rows of few
// distinct values, or with one value far above the others, have thousands of candidates next to each other, and ranking those
// against each other takes as the square of their number (33 x 100,003 logits in halves, a window of 200: 143 us so, 73 us
// sorted; where they are few the ranks are faster, 52 against some 90 us).
template <int WAVES>
__device__ __forceinline__ void sort_candidates(uint64_t* pairs, uint32_t count, int tid)
{
    constexpr uint32_t kThreads = WAVES * kWaveSize;
    uint32_t size = 1u;
    while (size < count)
        size *= 2u;
    for (uint32_t i = count + tid; i < size; i += kThreads)
        pairs[i] = 0u;
    __syncthreads();
    for (uint32_t length = 2u; length <= size; length *= 2u)
    {
        for (uint32_t distance = length / 2u; distance > 0u; distance /= 2u)
        {
            for (uint32_t i = tid; i < size / 2u; i += kThreads)
            {
                const uint32_t first = 2u * i - (i & (distance - 1u));
                const uint32_t second = first + distance;
                const uint64_t a = pairs[first], b = pairs[second];
                if ((a < b) == ((first & length) == 0u) && a != b)
                {
                    pairs[first] = b;
                    pairs[second] = a;
                }
            }
            __syncthreads();
        }
    }
}

// One row's `count` candidates to its result: candidate(i, key, token) gives the i-th, `seen` what the row's parts saw (kWindowSawNan,
// kWindowHasAll).  WAVES waves call it.
template <int DTYPE, int WAVES, typename Candidate>
__device__ __forceinline__ void window_finish(
    const WindowArgs& g, uint32_t row, const ncnn_moe_sample_params& p, float uniform, uint32_t count, uint32_t seen, Candidate candidate, WindowFinishShared& shared, int tid)
{
    constexpr uint32_t kThreads = WAVES * kWaveSize;
    constexpr uint32_t kPerThread = kWindowListCap / kThreads;
    const SamplerArgs& a = g.a;
    const uint32_t wanted = p.top_k == 0u || p.top_k >= a.vocab ? a.vocab : p.top_k;
    if (tid < 32)
        shared.exp2_table[tid] = kExp2Table[tid];
    if (tid == 0)
    {
        shared.least = 0xffffffffu;
        shared.most = 0u;
        shared.neighbours = 0u;
    }
    __syncthreads();
    // (fewer candidates than the window, and logits below the bound: the sample misled)
    if (count > kWindowListCap || (count < wanted && (seen & kWindowHasAll) == 0u))
        return;
    uint8_t flags = counts_as_select(g.windows_are_selects, a.vocab, p) ? 0 : NCNN_MOE_ROW_FLAG_GENERAL_PATH;
    if ((seen & kWindowSawNan) != 0u)
        flags |= NCNN_MOE_ROW_FLAG_HAS_NAN;
    const auto reject = [&]() {
        if (tid == 0)
        {
            write_error(a, row, NCNN_MOE_ROW_NO_FINITE_LOGIT, flags);
            a.row_state[row] = kRowDoneLater;
        }
    };
    if (count == 0u)
        return reject();
    const uint32_t window = min(wanted, count);
    // False: finished, or left.  The threads hold kEach candidates each at most (a window of 200 has some 1,100, one of 1,000 2,300).
    constexpr uint32_t kFewEach = kPerThread / 2u;
    const auto put_in_order = [&](auto each) -> bool {
        constexpr uint32_t kEach = decltype(each)::value;
        uint32_t keys[kEach], tokens[kEach];
        uint32_t least = 0xffffffffu, most = 0u;
#pragma unroll
        for (uint32_t k = 0; k < kEach; ++k)
        {
            const uint32_t i = k * kThreads + tid;
            keys[k] = tokens[k] = 0u;
            if (i < count)
                candidate(i, keys[k], tokens[k]);
            least = i < count ? min(least, keys[k]) : least;
            most = max(most, keys[k]);
            if (i < count)
                shared.counters[i] = 0u;
        }
        most = wave_max_u32(most);
        least = ~wave_max_u32(~least);
        if ((tid & (kWaveSize - 1)) == 0)
        {
            atomicMax(&shared.most, most);
            atomicMin(&shared.least, least);
        }
        __syncthreads();
        most = same_in_all(shared.most);
        least = same_in_all(shared.least);
        const float largest = value_from_ascending_key(most);
        const float maximum = largest / p.temperature;
        if (!is_finite_f32(largest))
            return reject(), false;
        if (!is_finite_f32(maximum))
            return false;
        // ---- in order: about where a candidate belongs by its value, then against those that belong in the same place
        const float smallest = value_from_ascending_key(least);
        const float scale = largest > smallest ? static_cast<float>(count) / (largest - smallest) : 0.0f;
        uint32_t fine[kEach], turn[kEach];
#pragma unroll
        for (uint32_t k = 0; k < kEach; ++k)
        {
            fine[k] = turn[k] = 0u;
            if (k * kThreads + tid < count)
            {
                fine[k] = min(count - 1u, static_cast<uint32_t>((largest - value_from_ascending_key(keys[k])) * scale));
                turn[k] = atomicAdd(&shared.counters[fine[k]], 1u);
            }
        }
        uint32_t neighbours = 0;
#pragma unroll
        for (uint32_t k = 0; k < kEach; ++k)
            neighbours = max(neighbours, turn[k]);
        neighbours = wave_max_u32(neighbours);
        if ((tid & (kWaveSize - 1)) == 0 && neighbours >= kWindowRankedTies)
            atomicMax(&shared.neighbours, neighbours);
        __syncthreads();
        constexpr uint32_t kWindowEach = kSelectTopK / kThreads;
        static_assert(kWindowEach * kThreads == kSelectTopK, "the threads hold the widest window");
        const auto term_of = [&](uint32_t key) { return expf_libm(value_from_ascending_key(key) / p.temperature - maximum, shared.exp2_table); };
        if (same_in_all(shared.neighbours) != 0u)
        {
            static_assert(offsetof(WindowFinishShared, tokens) == kWindowListCap * sizeof(uint32_t), "keys and tokens lie one behind the other");
            uint64_t* const pairs = reinterpret_cast<uint64_t*>(shared.keys);
            for (uint32_t k = 0; k < kPerThread; ++k)
            {
                const uint32_t i = k * kThreads + tid;
                uint32_t key, token;
                if (i < count)
                {
                    candidate(i, key, token);
                    pairs[i] = (static_cast<uint64_t>(key) << 32) | (0xffffffffu - token);
                }
            }
            sort_candidates<WAVES>(pairs, count, tid);
            uint64_t own[kWindowEach];
#pragma unroll
            for (uint32_t k = 0; k < kWindowEach; ++k)
                own[k] = pairs[k * kThreads + tid];
            __syncthreads();
#pragma unroll
            for (uint32_t k = 0; k < kWindowEach; ++k)
            {
                const uint32_t i = k * kThreads + tid;
                if (i < window)
                {
                    shared.tokens[i] = 0xffffffffu - static_cast<uint32_t>(own[k]);
                    shared.terms[i] = term_of(static_cast<uint32_t>(own[k] >> 32));
                }
            }
            __syncthreads();
            return true;
        }
        uint32_t held[kEach];
        uint32_t total[1] = {0u};
        const uint32_t first = tid * kEach;
#pragma unroll
        for (uint32_t k = 0; k < kEach; ++k)
        {
            held[k] = first + k < count ? shared.counters[first + k] : 0u;
            total[0] += held[k];
        }
        uint32_t totals[1];
        bin_scan<WAVES>(total, totals, shared.scan, tid);
        uint32_t front = total[0];
#pragma unroll
        for (uint32_t k = 0; k < kEach; ++k)
        {
            if (first + k < count)
                shared.counters[first + k] = front;
            front += held[k];
        }
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < kEach; ++k)
        {
            if (k * kThreads + tid < count)
            {
                const uint32_t at = shared.counters[fine[k]] + turn[k];
                shared.keys[at] = keys[k];
                shared.tokens[at] = tokens[k];
            }
        }
        __syncthreads();
        uint32_t rank[kEach];
#pragma unroll
        for (uint32_t k = 0; k < kEach; ++k)
        {
            rank[k] = 0u;
            if (k * kThreads + tid < count)
            {
                const uint32_t low = shared.counters[fine[k]];
                const uint32_t high = fine[k] + 1u < count ? shared.counters[fine[k] + 1u] : count;
                rank[k] = low;
                if (low < window) // (what lies behind the window need not be in order)
                {
                    for (uint32_t j = low; j < high; ++j)
                    {
                        const uint32_t other = shared.keys[j];
                        rank[k] += other > keys[k] || (other == keys[k] && shared.tokens[j] < tokens[k]) ? 1u : 0u;
                    }
                }
                else
                    rank[k] = window;
            }
        }
        __syncthreads();
        // ---- the window: its tokens, and its terms, a thread for each
#pragma unroll
        for (uint32_t k = 0; k < kEach; ++k)
        {
            if (k * kThreads + tid < count && rank[k] < window)
            {
                shared.keys[rank[k]] = keys[k];
                shared.tokens[rank[k]] = tokens[k];
            }
        }
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < kWindowEach; ++k)
        {
            const uint32_t i = k * kThreads + tid;
            if (i < window)
                shared.terms[i] = term_of(shared.keys[i]);
        }
        __syncthreads();
        return true;
    };
    if (!(count <= kFewEach * kThreads ? put_in_order(std::integral_constant<uint32_t, kFewEach>{}) : put_in_order(std::integral_constant<uint32_t, kPerThread>{})))
        return;
    sum_chunks<WAVES>(shared.head, shared.terms, window, tid);
    sum_head<WAVES, 0>(shared.head, shared.terms, window, kStopNever, 0.0f, 1.0f, 1.0f, tid);
    const float normalizer = same_in_all(shared.head.sum);
    uint32_t candidates = window;
    if (p.min_p > 0.0f)
    {
        const float threshold = (1.0f / normalizer) * p.min_p;
        const float* terms = shared.terms;
        candidates = wave_partition_point(window, [terms, normalizer, threshold](uint32_t i) { return terms[i] / normalizer >= threshold; });
    }
    sum_head<WAVES, 1>(shared.head, shared.terms, candidates, kStopAtOrAbove, p.top_p, normalizer, 1.0f, tid);
    const float renormalizer = same_in_all(shared.head.sum);
    const uint32_t top_p_stop = same_in_all(shared.head.stop);
    const uint32_t kept = top_p_stop != 0xffffffffu ? top_p_stop + 1u : candidates;
    uint32_t selected = 0;
    if (kept > 1u)
    {
        sum_head<WAVES, 2>(shared.head, shared.terms, kept, kStopAbove, uniform, normalizer, renormalizer, tid);
        const uint32_t stop = same_in_all(shared.head.stop);
        selected = stop != 0xffffffffu ? stop : kept - 1u;
    }
    if (tid == 0)
    {
        const float probability = kept == 1u ? 1.0f : (shared.terms[selected] / normalizer) / renormalizer;
        write_token(a, row, p, static_cast<int32_t>(shared.tokens[selected]), probability, kept, kept == 1u ? 0 : 1, flags);
        a.row_state[row] = kRowDoneLater;
    }
}

// (bound to 64 registers, so that two workgroups share a compute unit: 33 rows of 100,003 take 18 us instead of 25)
template <int DTYPE>
__global__ __launch_bounds__(kBinThreads, 8) void window_candidates_kernel(WindowArgs g)
{
    __shared__ WindowCandidatesShared shared;
    __shared__ RowList listed_rows;
    const uint32_t rows = list_rows_in_place(g.a, g.listing, true, true, g.list, g.other_list, listed_rows, threadIdx.x);
    if (g.turn != kWindowsOnce && windows_go_ahead(rows, g.sums_list[0], g.a.vocab) != (g.turn == kWindowsAhead))
        return;
    window_candidates<DTYPE>(g, bin_grid(rows, g.a.vocab), listed_rows, shared, threadIdx.x);
}

template <int DTYPE>
__global__ __launch_bounds__(kWalkThreads) void window_finish_kernel(WindowArgs g)
{
    __shared__ WindowFinishShared shared;
    const int tid = threadIdx.x;
    const uint32_t rows = same_in_all(g.list[0]);
    for (uint32_t slot = blockIdx.x; slot < rows; slot += gridDim.x)
    {
        const uint32_t row = same_in_all(g.list[1u + slot]);
        const uint32_t count = same_in_all(g.counts[row]);
        const uint32_t seen = same_in_all(g.flags[row]);
        const ncnn_moe_sample_params p = g.a.params[row];
        const float uniform = same_in_all(g.a.uniforms[row]);
        __syncthreads(); // (every thread has read the counters)
        if (tid == 0)
        {
            g.counts[row] = 0u;
            g.flags[row] = 0u;
        }
        const auto candidate = [&](uint32_t i, uint32_t& key, uint32_t& token) {
            key = g.keys[static_cast<size_t>(row) * kWindowListCap + i];
            token = g.tokens[static_cast<size_t>(row) * kWindowListCap + i];
        };
        window_finish<DTYPE, kWalkWaves>(g, row, p, uniform, count, seen, candidate, shared, tid);
        __syncthreads();
    }
}

// Both in one launch, for calls of no more rows than compute units: the part that is the last to hand its candidates over finishes the
// row, so nothing waits.  A workgroup has a compute unit to itself, and with it the registers (256) to ask for the sample and the first
// kWindowAhead vectors a thread of its part together, in front of the bound.
//
// What bounds it: a chain.  33 rows of 100,003 logits, a window of 200, us: rows listed 1.6, sample and part loaded 1.8, bound 2.9, logits
// compared and listed 1.7, handed over 1.5, taken over 1.5, put in order 2.8, the three sums 1.2, 2.1 and 1.1; 256 rows of 151,936
// the stream, 30 of 47.  us a call, by two launches and by this one: 33 x 100,003, windows of 200 36.4 and 29.1, of 1,000 41.6 and 34.2;
// 1 x 50,257 25.9 and 23.9, 1 x 151,936 30.8 and 28.5, 8 x 151,936 34.2 and 30.1, 64 x 151,936 44.2 and 36.8, 4 x 5,000 30.6 and 29.9, 100 x
// 32,000 35.6 and 28.3, 100 x 129,280 49.5 and 43.5, 200 x 151,936 82.8 and 75.2, 256 x 16,384 36.6 and 28.2, x 151,936 72.5 and 67.1; bf16
// 33 x 100,003 36.6 and 28.7, 256 x 201,088 68.8 and 60.1.  With the hits' keys and tokens stored vector by vector, as window_candidates
// does, the part took 4.2 instead of 1.7 (33 x 100,003 31.6 a call, 256 x 151,936 80.8): eight waves have no others to hide behind.
//
// arrivals[2] of a row: candidates that the parts have handed over (kWindowCountBits), how many saw a NaN (above), and how many have
// handed theirs over (from kWindowPartShift on); the last one returns it to zero.
constexpr uint32_t kWindowAhead = 16;
constexpr uint32_t kWindowCountBits = 24, kWindowPartShift = 32;
constexpr uint32_t kWindowMostSample = kWindowSampleVectors * kBinThreads / kWalkThreads;
static_assert(kWindowMaxVocab < 1u << kWindowCountBits && kMaxBinParts < 1u << (kWindowPartShift - kWindowCountBits), "the counts of a row's parts fit their bits");

template <int DTYPE>
__global__ __launch_bounds__(kWalkThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void window_chain_kernel(WindowArgs g)
{
    using Vector = LogitsVector<DTYPE>;
    constexpr uint32_t kWidth = Vector::kWidth;
    __shared__ WindowCandidatesShared shared;
    __shared__ WindowFinishShared finish;
    __shared__ RowList listed_rows;
    __shared__ uint32_t options[kRowOptionWords];
    __shared__ uint32_t row_count, row_seen, is_last;
    const SamplerArgs& a = g.a;
    const int tid = threadIdx.x;
    const int lane = tid & (kWaveSize - 1);
    clear_sample_counts<kWalkThreads>(shared, tid);
    const uint32_t rows = list_rows_in_place<kWalkWaves>(a, g.listing, true, true, g.list, g.other_list, listed_rows, tid);
    const BinGrid grid = bin_grid(rows, a.vocab, kMaxBinParts, kChainGrid);
    for (uint32_t slot = grid.first_slot; slot < grid.rows; slot += grid.slot_step)
    {
        const uint32_t row = same_in_all(row_of_slot(g.listing, g.list, listed_rows, slot));
        const BinStretch s = bin_stretch<Vector::kElementBytes>(a, row, grid.part, grid.parts);
        const char* base = static_cast<const char*>(a.logits) + static_cast<size_t>(row) * a.row_stride * Vector::kElementBytes -
            static_cast<size_t>(s.misalignment) * Vector::kElementBytes;
        const auto vector_at = [&](uint32_t v) { return *reinterpret_cast<const uint4*>(base + static_cast<size_t>(v) * 16u); };
        // ---- all that the row's first steps read is asked for at once
        const uint32_t option = read_option(a, row, tid);
        const uint32_t first_whole = (s.misalignment + kWidth - 1u) / kWidth;
        const uint32_t whole = s.end / kWidth - min(first_whole, s.end / kWidth);
        const uint32_t sampled = sampled_vectors(whole);
        uint4 sample[kWindowMostSample];
#pragma unroll
        for (uint32_t k = 0; k < kWindowMostSample; ++k)
        {
            const uint32_t i = k * kWalkThreads + tid;
            if (i < sampled)
                sample[k] = vector_at(first_whole + static_cast<uint32_t>(static_cast<uint64_t>(i) * whole / sampled));
        }
        const uint32_t first = s.first * 8u / kWidth, last = min(s.last * 8u / kWidth, (s.end + kWidth - 1u) / kWidth);
        uint4 raw[kWindowAhead];
        const auto ask = [&](uint32_t from) {
#pragma unroll
            for (uint32_t k = 0; k < kWindowAhead; ++k)
            {
                const uint32_t v = from + k * kWalkThreads + tid;
                if (v < last)
                    raw[k] = vector_at(v);
            }
        };
        ask(first);
        if (tid == 0)
        {
            shared.count = 0u;
            shared.saw_nan = 0u;
        }
        if (tid < static_cast<int>(kRowOptionWords))
            options[tid] = option;
        __syncthreads();
        const ncnn_moe_sample_params p = params_of(options);
        const uint32_t window = p.top_k == 0u || p.top_k >= a.vocab ? a.vocab : p.top_k;
        const auto sample_vector = [&](uint32_t k, float (&x)[kWidth]) -> bool {
            if (k * kWalkThreads + tid >= sampled)
                return false;
            Vector::unpack(sample[k], x);
            return true;
        };
        const uint32_t reached = bound_of_sample<DTYPE, kWalkThreads, kWindowMostSample, kWindowMostSample>(shared, a.vocab, window, whole, sampled, sample_vector, tid);
        // (an infinite logit below everything is no candidate: the window counts finite logits)
        const uint32_t lowest = ascending_key(-3.402823466e38f);
        const bool has_all = reached <= lowest;
        const float bound = value_from_ascending_key(max(reached, lowest));
        // ---- the part's logits at or above it: counted, placed by one addition a wave, their tokens listed
        constexpr uint32_t kHitWords = kWindowAhead * kWidth / 32u;
        bool saw_nan = false;
        for (uint32_t from = first; from < last;)
        {
            // (bit k * kWidth + c of the mask: component c of the thread's k-th vector)
            uint32_t hits[kHitWords];
            uint32_t own = 0;
#pragma unroll
            for (uint32_t w = 0; w < kHitWords; ++w)
                hits[w] = 0u;
#pragma unroll
            for (uint32_t k = 0; k < kWindowAhead; ++k)
            {
                const uint32_t v = from + k * kWalkThreads + tid;
                if (v < last)
                {
                    float x[kWidth];
                    Vector::unpack(raw[k], x);
                    uint32_t reaching = 0;
                    bool nan = false;
#pragma unroll
                    for (uint32_t c = 0; c < kWidth; ++c)
                        reaching |= x[c] >= bound ? 1u << c : 0u;
#pragma unroll
                    for (uint32_t c = 0; c < kWidth; c += 2u)
                        nan = nan || __builtin_isunordered(x[c], x[c + 1u]);
                    if (v < first_whole || v >= first_whole + whole)
                    {
                        // (the vectors at the row's ends hold what is not of the row)
                        nan = false;
                        uint32_t inside = 0;
#pragma unroll
                        for (uint32_t c = 0; c < kWidth; ++c)
                        {
                            const bool of_row = v * kWidth + c - s.misalignment < a.vocab;
                            inside |= of_row ? 1u << c : 0u;
                            nan = nan || (of_row && x[c] != x[c]);
                        }
                        reaching &= inside;
                    }
                    saw_nan = saw_nan || nan;
                    hits[k * kWidth / 32u] |= reaching << (k * kWidth % 32u);
                }
            }
#pragma unroll
            for (uint32_t w = 0; w < kHitWords; ++w)
                own += static_cast<uint32_t>(__popc(hits[w]));
            const uint32_t through = wave_prefix_sum_u32(own);
            uint32_t place = 0;
            if (lane == kWaveSize - 1 && through != 0u)
                place = atomicAdd(&shared.count, through);
            place = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(place), kWaveSize - 1)) + through - own;
#pragma unroll
            for (uint32_t w = 0; w < kHitWords; ++w)
            {
                while (hits[w] != 0u)
                {
                    const uint32_t bit = w * 32u + static_cast<uint32_t>(__builtin_ctz(hits[w]));
                    if (place < kWindowListCap)
                        shared.tokens[place] = (from + bit / kWidth * kWalkThreads + tid) * kWidth + bit % kWidth - s.misalignment;
                    ++place;
                    hits[w] &= hits[w] - 1u;
                }
            }
            from += kWindowAhead * kWalkThreads;
            if (from < last)
                ask(from);
        }
        if (__builtin_amdgcn_ballot_w64(saw_nan) != 0ull && lane == 0)
            shared.saw_nan = 1u;
        __syncthreads();
        // ---- their keys, which are read once more: few of them, at a place in registers that only the thread knows
        const uint32_t count = shared.count;
        const auto key_of = [&](uint32_t token) {
            const char* const logits = base + static_cast<size_t>(token + s.misalignment) * Vector::kElementBytes;
            if (DTYPE == NCNN_MOE_LOGITS_F32)
                return ascending_key(*reinterpret_cast<const float*>(logits));
            return ascending_key(__uint_as_float(static_cast<uint32_t>(*reinterpret_cast<const uint16_t*>(logits)) << 16));
        };
        // ---- handed over.  A part that is the row's only one finishes it from LDS
        uint32_t* const row_keys = g.keys + static_cast<size_t>(row) * kWindowListCap;
        uint32_t* const row_tokens = g.tokens + static_cast<size_t>(row) * kWindowListCap;
        constexpr uint32_t kListBytes = kWindowListCap * sizeof(uint32_t);
        const uint32_t saw_all = has_all ? kWindowHasAll : 0u; // (the same in all parts)
        if (grid.parts == 1u)
        {
            for (uint32_t i = tid; i < min(count, kWindowListCap); i += kWalkThreads)
                shared.keys[i] = key_of(shared.tokens[i]);
            if (tid == 0)
            {
                row_count = count;
                row_seen = saw_all | (shared.saw_nan != 0u ? kWindowSawNan : 0u);
                is_last = 1u;
            }
        }
        else
        {
            unsigned long long* const arrivals = g.arrivals + static_cast<size_t>(row) * kArrivalWords + 2u;
            if (tid == 0)
            {
                const unsigned long long own = count | (shared.saw_nan != 0u ? 1ull << kWindowCountBits : 0ull);
                row_count = static_cast<uint32_t>(__hip_atomic_fetch_add(arrivals, own, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) & ((1u << kWindowCountBits) - 1u);
            }
            uint32_t key = 0, token = 0;
            if (tid < min(count, kWindowListCap))
            {
                token = shared.tokens[tid];
                key = key_of(token);
            }
            __syncthreads();
            const uint32_t place = row_count;
            for (uint32_t i = tid; i < min(count, kWindowListCap); i += kWalkThreads)
            {
                if (i >= kWalkThreads)
                {
                    token = shared.tokens[i];
                    key = key_of(token);
                }
                if (place + i < kWindowListCap)
                {
                    hand_over(false, row_keys, kListBytes, place + i, key);
                    hand_over(false, row_tokens, kListBytes, place + i, token);
                }
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // (stored before the part is counted)
            __syncthreads();
            if (tid == 0)
            {
                const unsigned long long seen = __hip_atomic_fetch_add(arrivals, 1ull << kWindowPartShift, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                is_last = static_cast<uint32_t>(seen >> kWindowPartShift) + 1u == grid.parts ? 1u : 0u;
                row_count = static_cast<uint32_t>(seen) & ((1u << kWindowCountBits) - 1u);
                row_seen = saw_all | ((static_cast<uint32_t>(seen) >> kWindowCountBits) != 0u ? kWindowSawNan : 0u);
                if (is_last != 0u)
                    __hip_atomic_store(arrivals, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        __syncthreads();
        if (same_in_all(is_last) != 0u)
        {
            const auto candidate = [&](uint32_t i, uint32_t& key, uint32_t& token) {
                if (grid.parts == 1u)
                {
                    key = shared.keys[i];
                    token = shared.tokens[i];
                }
                else
                {
                    key = taken_over<true>(row_keys, kListBytes, i);
                    token = taken_over<true>(row_tokens, kListBytes, i);
                }
            };
            window_finish<DTYPE, kWalkWaves>(g, row, p, same_in_all(__uint_as_float(options[kParamsWords])), same_in_all(row_count), same_in_all(row_seen), candidate, finish, tid);
        }
        __syncthreads();
        clear_sample_counts<kWalkThreads>(shared, tid);
    }
}

} // namespace ncnn_moe_hip

#endif // NCNN_MOE_HIP_SAMPLER_WINDOWS_H

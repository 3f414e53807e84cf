// Binned sums: the sampler's walk over a row whose order is never worked out.
//
// The CPU sampler adds the row's terms exp(logit/T - max) one by one in descending order, three times over (the
// normaliser, the Top-P walk, the draw), and every partial sum is rounded to fp32.  While such a sum stays inside one
// binade its mantissa grows by round(term / ulp) per term, which depends on the sum in one case only: a term that ends
// exactly half an ulp above a multiple of it.  So the terms of a stretch of the sorted row in which the sum neither
// leaves its binade nor meets such a term may be added in any order, as integers.  The rows served here (no Top-K
// window, or one wider than the first select's) are therefore not sorted:
//   * the terms fall into kBins bins by their bit pattern (0.4 to 0.8 % of a term wide; bins follow the sorted order);
//   * the head of the row (the bins of its first 1,920 elements at most) is sorted in LDS and added exactly as the
//     CPU does, which takes the sum through most of its binades;
//   * every other bin is one integer: the sum of its terms' steps at the exponent that the running sum will have there;
//   * the few bins in which the order matters - the sum leaves its binade, a stop condition is met, the window or the
//     Min-P cut ends - are fetched element by element and sorted: those that can be foreseen from the bins' masses by the
//     pass that adds the others, the rest on demand by a pass over the row's terms;
//   * a term that lies half way between two sums is rounded by the parity of the sum in front of it, which follows from
//     the parities of the steps in front of it: between two such values every term of a bin has the same step, so one
//     bit per step value and bin (the parity of the odd steps of that value) tells.
// A term of 2^-25 or less never moves any of the three sums (the first term is 1, so half an ulp of the normaliser is
// at least 2^-24; the other two sums start at the first term divided by the same numbers as every other): such terms
// are in no bin.  A foreseen exponent is checked against the exact sum before a bin's integer is used.
//
// Each workgroup takes a part of one row: (1) maximum and counts, (2) terms and bin counts, (3) head fetched, steps of the
// normaliser's sum, (4) normaliser walked, steps of the Top-P sum, Top-P walked, steps of the draw's sum, draw walked.  Calls of few
// elements do all of it in one launch (bin_chain_kernel), larger ones (1) to (3) in a launch each and the walks in a fourth
// (bin_walks_kernel).  Inside a launch a row's parts meet where they hand something to each other (parts_meet): 1 us and the loads of what was
// handed over, where another launch costs a gap of 2 to 3, 1.5 before it knows its row and loads that find nothing in the L2.
// One launch for the three walks: 8 rows of 151,936 without a window 105.3 -> 99.2 us, 512 of 129,280 with mixed options 222.1 -> 218.2;
// one for all: 8 rows 99.2 -> 93.4, 33 x 100,003 with windows of 200, for which the launches find no row, 47.1 -> 39.4, a verification
// step of 5 drafts without a window 163.1 -> 146.
//
// What bounds it: instructions, of which each SIMD has those of two wavefronts to issue, and trips to LDS and memory one behind the
// other (8 rows of 151,936: 6, 6, 13 and 55 to 60 for the walks; of a walk some 5 us add the next sum's steps); at a hundred rows and
// more the reads of the rows and their terms, and the slowest row's walk.
#ifndef NCNN_MOE_HIP_SAMPLER_BINS_H
#define NCNN_MOE_HIP_SAMPLER_BINS_H

#include "sampler_full_order.h"

namespace ncnn_moe_hip {

constexpr int kBinThreads = 1024;
constexpr int kBinWaves = kBinThreads / kWaveSize;
constexpr int kWalkThreads = 512;                // the walk: half the waves cost half of what every wave of it does
constexpr int kWalkWaves = kWalkThreads / kWaveSize;
constexpr uint32_t kBinsPerBinade = 64;
constexpr uint32_t kBinBinades = 25;
constexpr uint32_t kBins = kBinBinades * kBinsPerBinade;
constexpr uint32_t kBinWords = kBins / 32;
constexpr uint32_t kBinQuads = kBins / 4;        // a thread of the row's scan holds four consecutive bins
constexpr uint32_t kOneBits = 0x3f800000u;       // the largest term
constexpr uint32_t kTailDistance = kBinBinades << 23; // in bits below it: terms of 2^-25 or less move no sum
constexpr float kTailArgument = -17.4f;          // exp of anything less is below 2^-25 (2^-25 = exp(-17.33))
constexpr uint32_t kOffsetBits = 12;             // where in its bin a term lies, summed per bin
constexpr uint32_t kBinHead = 1920;              // elements of the sorted head at most, 30 chunks of sum_head: behind so many a term half
                                                 // way seldom has to be fetched, 9 us and more each
constexpr uint32_t kBinWholeRow = 2048;          // ... unless these are all that the sums run over
constexpr uint32_t kBinListCap = 4096;           // head and foreseen bins, elements
constexpr uint32_t kBinExtraCap = 1536;          // elements fetched on demand at a time
constexpr uint32_t kBinStops = 512;
// Steps are added modulo 2^32, and a sum of them counts while it is below 2^24.  A bin whose terms may take 2^25 steps and
// more is therefore not added but fetched, and a row whose bins together may take 2^32 is left to the full-order kernels.
constexpr float kBinMostSteps = 33554432.0f;
constexpr uint32_t kBinStepUnit = 16;            // log2 of the unit in which a row's steps are added up once more
constexpr uint32_t kBinStopBits = 11;            // ... above the row's number of stops, in one word
static_assert(kBins < 1u << kBinStopBits && (kBins << (26 - kBinStepUnit)) < 1u << (32 - kBinStopBits), "the steps of 2^25 and a little a bin fit beside the stops");
constexpr int kMaskedDifference = 14;            // so many binades below the sum a bin's terms (within a 64th of each other) take 18 different steps at most
// ... and so many below it 66: the first bins of that distance have masks of four times the width.  A term half way that no mask
// tells costs its row a fetch, and nearly all of those were 12 or 13 binades below the sum (of 94 rows in a batch of mixed options
// some 13 % had one in each sum, and the batch waits for its slowest row).
constexpr int kWideDifference = 12;
constexpr float kNearlyTopP = 0.85f;                // of the Top-P, in the longest head: see the head of bin_sum_kernel
constexpr uint32_t kWideBins = 128;
constexpr uint32_t kWideParities = 2, kWideHalves = 4; // words a bin
constexpr uint32_t kWideWords = kWideParities + kWideHalves;
constexpr uint32_t kMaskWords = 2u * kBins + kWideBins * kWideWords; // of a part: two words a bin, then the wide ones
static_assert(kMaskWords % 4u == 0u && kBins % 4u == 0u, "masks are moved in vectors of four words");
constexpr uint32_t kBinRequests = 64;            // ... and how often per walk
constexpr uint32_t kBinComparedTies = 256;       // equal terms of a list that are told apart by comparing each with each
constexpr uint32_t kMaxBinParts = 16;
constexpr uint32_t kPartsAtATime = 4;            // loads of the parts' numbers in flight together
constexpr uint32_t kBinPartElements = 2048;      // a part is not made smaller
constexpr uint32_t kArrivalWords = 16;           // of a row (see parts_meet): a cache line
constexpr uint32_t kBinGrid = 512;               // workgroups of each launch: two per compute unit
// (1) to (4) are one launch, bin_chain_kernel, where a part holds so few elements that what a launch costs by itself outweighs what it is
// good for: kernels (1) to (3) of 1,024 threads, two workgroups to a compute unit, get through many elements faster.  us a call without a
// window, by one launch and by four, with the elements of a part of the chain: 17 rows of 151,936 (15,200) 107 and 122, 40 of 32,000 (5,300) 82 and
// 103, of 100,003 (16,700) 116 and 125, of 129,280 (21,500) 131 and 130; 64 of 2,000 35 and 44, of 64,000 (16,000) 111 and 117, of 100,003
// (25,000) 135 and 132; 100 of 16,384 (8,200) 82 and 93, of 50,257 (25,100) 128 and 123; 256 of 16,384 101 and 109; 4 of 1,000,000 (62,500)
// 242 and 228, 16 of 400,000 (25,000) 147 and 144.  Where rows have windows as well, most of the call's rows are not these, and the launches that find
// none cost 2 us each: mixed options, 40 rows of 129,280 132 and 139, 100 143 and 155; windows of 300, 33 of 100,003 38 and 44, 100 of 129,280
// (64,600) 50 and 57, 256 of 50,257 46 and 52.  A chain has a compute unit to itself: its walks want 220 registers, and at 128, which two
// workgroups to a compute unit leave, some of them and 200 scalars pass through scratch and lane moves (17 rows of 151,936 131 us so).  Few rows too
// long for it lose nothing by that: 1 to 16 rows of 330,000 to 4,000,000 in four launches take 0.81 to 1.01 of the time that three walks with 220
// registers each took (16 x 330,000 176 and 151, 4 x 600,000 231 and 197, 1 x 600,000 175.5 and 176.7).  More rows
// than compute units would take turns (300 of 16,384 168 and 124).
constexpr uint32_t kChainGrid = kBinGrid / 2u;
constexpr uint32_t kChainRows = kChainGrid;
constexpr uint32_t kChainPartElements = 20000;
constexpr uint32_t kChainPartElementsWithWindows = 80000;
constexpr uint32_t kBinMaxVocab = (1u << 22) - 16u; // a rank fits 22 bits
// Foreseen sums decide what is prepared, never what a sum is: a walk that finds its exact sum elsewhere fetches what it needs.
// They are off by a few 1e-5 on most rows and by 4e-4 (normal logits) to 2e-3 (logits rounded to eighths) on some: a bin
// that was listed or fetched enters the next forecast with a guess of its terms, and the next sum's terms round differently.
// The margin for listing stays at 1e-4 all the same: where a sum grows by single ulps it lists 1,700 elements at most on
// both sides of a power of two, so that they always fit, and a miss costs the one row a fetch.
constexpr float kForeseenFirst = 1e-4f;          // relative error allowed for the sums foreseen from the bins' masses
constexpr float kForeseenLater = 1e-4f;          // ... and from the steps of the sum before
constexpr float kForeseenEnd = 4e-3f;            // ... before a bin is taken to lie behind the end of the sum and gets no steps
static_assert(kBinQuads <= kWalkThreads && kBinListCap % kWalkThreads == 0 && kBinListCap <= 64 * kWaveSize, "the walk's thread and lane counts");

// A bin as the walk sees it: kind (2 bits), biased exponent assumed for the running sum (8), elements in front of it (22).
constexpr uint32_t kBinAdded = 0u;  // its elements' steps are added as one integer
constexpr uint32_t kBinListed = 1u; // its elements are in the list
constexpr uint32_t kBinBeyond = 2u; // behind the end of the sum, as far as that can be foreseen
constexpr uint32_t kBinWanted = 3u; // its elements are needed and not in the list: fetched on demand

__device__ __forceinline__ uint32_t packed_kind(uint32_t packed) { return packed >> 30; }
__device__ __forceinline__ uint32_t packed_exponent(uint32_t packed) { return (packed >> 22) & 0xffu; }
__device__ __forceinline__ uint32_t packed_front(uint32_t packed) { return packed & 0x3fffffu; }

enum BinRowState : uint32_t
{
    kBinRowLeft = 0,  // not (or no longer) served here: finished, or left to the full-order kernels
    kBinRowGoesOn = 1, // the next launch goes on with it
    kBinRowRejected = 2 // no finite logit, or +inf among them: the first walk reports it
};

// What the launches of a call keep of a row.  A launch reads what earlier ones wrote and writes other words (its own
// workgroups read the row's record at different times).
struct BinRow
{
    uint32_t state[2];      // after launches (2), (3)
    uint32_t shift;         // a term's bin: (kOneBits - bits) >> shift
    uint32_t window;        // elements of the Top-K window (finite logits at most)
    uint32_t binned;        // elements in bins
    uint32_t saw_nan;
    uint32_t head_bins;     // bins [0, head_bins) are the head, head_count elements
    uint32_t head_count;
    uint32_t wide_first;    // of the normaliser's sum: the first of the kWideBins bins with wide masks
    uint32_t listed;        // elements in the first list, the head among them
    uint32_t served;        // the row was finished here
    // the filtered distribution, where BinArgs::want_filters asks for it: probability((exp(logit/T - maximum) / normalizer)
    // / renormalizer) of the elements kept, which are those up to filter_key, filter_token in the row's order whose term is
    // least_term or more
    uint32_t filtered;
    float normalizer, renormalizer;
    uint32_t kept;
    float maximum;
    uint32_t filter_key;    // descending key
    uint32_t filter_token;
    float least_term;
};

struct BinArgs
{
    SamplerArgs a;
    uint32_t* list;        // the rows served: [0] their number, then the rows
    uint4* stats;          // [pairs] (row, part): largest and smallest finite logit, finite logits, flags
    uint32_t* counts;      // [pairs][2][kBins]: terms in each bin, and the sum of their places in it (kOffsetBits)
    uint32_t* before;      // [pairs][kBins]: elements of each bin in the parts in front
    uint32_t* steps[2];    // [pairs][kBins], of alternate launches
    uint32_t* ties[2];     // [pairs][3][kBinWords]: bins with terms half way, with two of one value, and with some that their masks cannot hold
    uint32_t* masks[2];    // [pairs][kMaskWords]: parities of the odd steps, and the values half way, by step (see add_bin_steps)
    uint32_t* packed;      // [rows][kBins]
    float* list_terms[2];  // [rows][kBinListCap]
    uint32_t* list_tokens[2];
    uint32_t* head_tokens; // [rows][kBinListCap], sorted
    BinRow* records;       // [rows]
    unsigned long long* arrivals; // [rows][kArrivalWords], zero between launches: see parts_meet
    uint32_t most_looks;   // ... at the first meeting, see most_looks_of
    uint32_t most_parts;   // of a row: see most_parts_of
    uint32_t want_filters;
    uint32_t windows_are_selects; // rows with a window of the wide select's widths do not count as full-order rows
    uint32_t listing;      // RowListing: how the first launch finds its rows
    uint32_t* window_list; // where it lists those with a window as well (null: nowhere; see list_rows_in_place)
};

__device__ __forceinline__ uint32_t same_in_all(uint32_t value)
{
    return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(value)));
}

__device__ __forceinline__ float same_in_all(float value)
{
    return __uint_as_float(same_in_all(__float_as_uint(value)));
}

// A row's options, and its uniform behind them: the first threads read a word each, once a launch (they may lie in host memory).
constexpr uint32_t kParamsWords = sizeof(ncnn_moe_sample_params) / 4u;
constexpr uint32_t kRowOptionWords = kParamsWords + 1u;
static_assert(sizeof(ncnn_moe_sample_params) % 4u == 0u, "the options are whole words");

__device__ __forceinline__ uint32_t read_option(const SamplerArgs& a, uint32_t row, int tid)
{
    uint32_t word = 0;
    if (tid < static_cast<int>(kParamsWords))
        word = reinterpret_cast<const uint32_t*>(a.params + row)[tid];
    else if (tid == static_cast<int>(kParamsWords))
        word = __float_as_uint(a.uniforms[row]);
    return word;
}

__device__ __forceinline__ ncnn_moe_sample_params params_of(const uint32_t (&options)[kRowOptionWords])
{
    ncnn_moe_sample_params p;
    __builtin_memcpy(&p, options, sizeof(p));
    return p;
}

// The rows that the first select left when it ended, those with a window of the window kernels' widths apart from the others.
enum RowListing : uint32_t
{
    kRowsListed = 0,    // a launch of its own has listed them
    kRowsByState = 1,   // the first select has run: the rows that it left pending
    kRowsByOptions = 2  // ... runs beside: the rows whose options say so
};

// (Those that this launch has finished since are still among them: a launch that lists its rows in place may finish some before its
// last workgroups start, where other launches hold their places, and these have to come to the same list.)
__device__ __forceinline__ bool row_is_left(const SamplerArgs& a, uint32_t row, bool by_options, bool windows_apart, bool& window)
{
    uint32_t effective_k = 0;
    int status = NCNN_MOE_ROW_OK;
    // (all of it is asked for at once)
    uint32_t words[kParamsWords];
#pragma unroll
    for (uint32_t i = 0; i < kParamsWords; ++i)
        words[i] = reinterpret_cast<const uint32_t*>(a.params + row)[i];
    uint32_t state = by_options ? 0u : a.row_state[row];
#pragma unroll
    for (uint32_t i = 0; i < kParamsWords; ++i)
        asm volatile("" : "+v"(words[i]));
    asm volatile("" : "+v"(state));
    ncnn_moe_sample_params p;
    __builtin_memcpy(&p, words, sizeof(p));
    const int mode = resolve_row_mode(p, a.vocab, static_cast<uint32_t>(kFastTopK), a.force_general, effective_k, status);
    window = windows_apart && effective_k <= static_cast<uint32_t>(kSelectTopK);
    return by_options ? mode == kModeGeneral : (mode == kModeGeneral || mode == kModeTopK) && state != kRowDone;
}

// A call of no more rows than a workgroup has threads needs no launch that lists them: every workgroup of the first launch that
// wants the list works it out for itself (1.6 us more than reading it, where the launch took 3.0 us with the gap in front of it),
// and one writes it down for the launches behind.
constexpr uint32_t kRowsListedInPlace = kBinThreads;

struct RowList
{
    uint32_t wave_totals[kBinWaves];
    uint16_t rows[kRowsListedInPlace];
};

// (For a workgroup of WAVES waves, and calls of no more rows than it has threads.)
// How many rows there are; they are list[1 ..] where listing is kRowsListed, else shared.rows.  `others` (null: nowhere): the rows of
// the other kind are listed there for a later launch.
template <int WAVES = kBinWaves>
__device__ __forceinline__ uint32_t list_rows_in_place(
    const SamplerArgs& a, uint32_t listing, bool windows_apart, bool want_windows, uint32_t* list, uint32_t* others, RowList& shared, int tid)
{
    if (listing == kRowsListed)
        return same_in_all(list[0]);
    const int wave = tid >> 6;
    const uint32_t row = static_cast<uint32_t>(tid);
    bool left = false, window = false;
    if (row < a.rows)
        left = row_is_left(a, row, listing == kRowsByOptions, windows_apart, window);
    // where a row stands among those for which `mine` holds, and their number
    const auto place_of = [&](bool mine, uint32_t& total) {
        const uint64_t mask = __builtin_amdgcn_ballot_w64(mine);
        if ((tid & (kWaveSize - 1)) == 0)
            shared.wave_totals[wave] = static_cast<uint32_t>(__popcll(mask));
        __syncthreads();
        uint32_t before = 0;
        total = 0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w)
        {
            before += w < wave ? shared.wave_totals[w] : 0u;
            total += shared.wave_totals[w];
        }
        return before + static_cast<uint32_t>(lanes_below(mask));
    };
    uint32_t rows = 0;
    const bool mine = left && window == want_windows;
    const uint32_t place = place_of(mine, rows);
    if (mine)
        shared.rows[place] = static_cast<uint16_t>(row);
    if (blockIdx.x == 0u)
    {
        if (mine)
            list[1u + place] = row;
        if (tid == 0)
            list[0] = rows;
        if (others != nullptr)
        {
            __syncthreads();
            uint32_t other_rows = 0;
            const bool other = left && window != want_windows;
            const uint32_t other_place = place_of(other, other_rows);
            if (other)
                others[1u + other_place] = row;
            if (tid == 0)
                others[0] = other_rows;
        }
    }
    __syncthreads();
    return same_in_all(rows);
}

__device__ __forceinline__ uint32_t row_of_slot(uint32_t listing, const uint32_t* list, const RowList& shared, uint32_t slot)
{
    return listing == kRowsListed ? list[1u + slot] : shared.rows[slot];
}

// How a launch's workgroups cover the listed rows: all parts of a row on one XCD (workgroups are dealt out to the XCDs
// in turn), so that what one launch leaves of a row is found in that XCD's L2 by the next.
struct BinGrid
{
    uint32_t rows, parts, first_slot, slot_step, part;
};

__device__ __forceinline__ BinGrid bin_grid(uint32_t rows, uint32_t vocab, uint32_t most_parts = kMaxBinParts, uint32_t workgroups = kBinGrid)
{
    BinGrid r;
    r.rows = rows;
    const uint32_t per_xcd = workgroups / 8u;
    const uint32_t slots_per_xcd = max(1u, (r.rows + 7u) / 8u);
    const uint32_t most = min(most_parts, (vocab + kBinPartElements - 1u) / kBinPartElements);
    r.parts = max(1u, min(most, per_xcd / slots_per_xcd));
    const uint32_t lanes = per_xcd / r.parts; // slots in flight on an XCD
    const uint32_t within = blockIdx.x >> 3;
    r.part = within % r.parts;
    r.first_slot = within / r.parts < lanes ? (within / r.parts) * 8u + (blockIdx.x & 7u) : 0xffffffffu;
    r.slot_step = lanes * 8u;
    return r;
}

// The stretch of a row that a part covers, in groups of eight positions; positions count from the 16-byte boundary
// below the row, and [misalignment, end) hold its logits.
struct BinStretch
{
    uint32_t misalignment, end, first, last;
};

template <int ELEMENT_BYTES>
__device__ __forceinline__ BinStretch bin_stretch(const SamplerArgs& a, uint32_t row, uint32_t part, uint32_t parts)
{
    const char* pointer = static_cast<const char*>(a.logits) + static_cast<size_t>(row) * a.row_stride * ELEMENT_BYTES;
    BinStretch s;
    s.misalignment = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(pointer) & 15u) / ELEMENT_BYTES;
    s.end = s.misalignment + a.vocab;
    const uint32_t groups = (s.end + 7u) / 8u;
    const uint32_t each = (groups + parts - 1u) / parts;
    s.first = min(groups, part * each);
    s.last = min(groups, s.first + each);
    return s;
}

__device__ __forceinline__ bool counts_as_select(uint32_t windows_are_selects, uint32_t vocab, const ncnn_moe_sample_params& p)
{
    const uint32_t window = p.top_k == 0u || p.top_k >= vocab ? vocab : p.top_k;
    return windows_are_selects != 0u && window <= static_cast<uint32_t>(kSelectTopK);
}

__device__ __forceinline__ float* bin_terms(const SamplerArgs& a, uint32_t row)
{
    return reinterpret_cast<float*>(a.sort_indices[0] + row * a.sort_stride);
}

// What the parts of a row hand to each other inside one launch (ACROSS).  Loads pass around the compute units' L1 caches (agent scope), and
// so do stores where the parts are not all on one XCD (`near`, see parts_meet).  Where they are, and bin_grid sees to it, they meet in
// that XCD's L2: a store of agent scope goes to memory and leaves no line there, and every load behind it is a trip to
// memory (16 vectors a thread, 102 KB a row: 3.4 us instead of 1.5; 8 rows of 151,936 without a window, which hand over four
// times, 93 us instead of 85).  As buffer instructions, not as atomics: the compiler orders those, and waits for each before it issues the
// next.  `base`, `bytes`: the same in all lanes of a wave; what lies behind them is not written, and reads as zero.
typedef uint32_t BinVector __attribute__((ext_vector_type(4)));
constexpr int kAgentScope = 16; // SC1 of a buffer instruction

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* base, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00027000);
}

__device__ __forceinline__ void hand_over(bool near, void* base, uint32_t bytes, uint32_t index, uint32_t value)
{
    if (near)
        __builtin_amdgcn_raw_buffer_store_b32(value, buffer_of(base, bytes), static_cast<int>(index * 4u), 0, 0);
    else
        __builtin_amdgcn_raw_buffer_store_b32(value, buffer_of(base, bytes), static_cast<int>(index * 4u), 0, kAgentScope);
}

template <bool ACROSS>
__device__ __forceinline__ uint32_t taken_over(const void* base, uint32_t bytes, uint32_t index)
{
    return __builtin_amdgcn_raw_buffer_load_b32(buffer_of(base, bytes), static_cast<int>(index * 4u), 0, ACROSS ? kAgentScope : 0);
}

// ... vectors of four words, `index` of them behind `base`
__device__ __forceinline__ void hand_over_vector(bool near, void* base, uint32_t bytes, uint32_t index, const uint4& value)
{
    const BinVector v{value.x, value.y, value.z, value.w};
    if (near)
        __builtin_amdgcn_raw_buffer_store_b128(v, buffer_of(base, bytes), static_cast<int>(index * 16u), 0, 0);
    else
        __builtin_amdgcn_raw_buffer_store_b128(v, buffer_of(base, bytes), static_cast<int>(index * 16u), 0, kAgentScope);
}

template <bool ACROSS>
__device__ __forceinline__ uint4 taken_over_vector(const void* base, uint32_t bytes, uint32_t index)
{
    const BinVector v = __builtin_bit_cast(BinVector, __builtin_amdgcn_raw_buffer_load_b128(buffer_of(base, bytes), static_cast<int>(index * 16u), 0, ACROSS ? kAgentScope : 0));
    return uint4{v.x, v.y, v.z, v.w};
}

// (of numbers; the compiler's own make sure first that none of them is a signalling NaN, an instruction each)
__device__ __forceinline__ float largest_of_three(float a, float b, float c)
{
    float result;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(result) : "v"(a), "v"(b), "v"(c));
    return result;
}

__device__ __forceinline__ float smallest_of_three(float a, float b, float c)
{
    float result;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(result) : "v"(a), "v"(b), "v"(c));
    return result;
}

// Kernels (1) to (3) are bound to 64 registers: two workgroups of 1,024 threads share a compute unit then, and the 512
// workgroups of a launch that many rows fill run at once, not in two rounds (512 rows of 129,280 of mixed options: 17, 26
// and 32 us before, 14, 22 and 25 us with the bound).
//
// ---- (1) largest and smallest finite logit, number of finite logits, NaN and +inf seen
// `wave_stats`: one for each of the workgroup's waves.  The first wave returns those of the part.
template <int DTYPE, int THREADS>
__device__ __forceinline__ uint4 stats_of_part(const SamplerArgs& a, const BinGrid& grid, uint32_t row, uint4* wave_stats, int tid)
{
    using Vector = LogitsVector<DTYPE>;
    constexpr uint32_t kWidth = Vector::kWidth;
    constexpr int kLoads = 4 * kBinThreads / THREADS;
    {
        const BinStretch s = bin_stretch<Vector::kElementBytes>(a, row, grid.part, grid.parts);
        const char* base = static_cast<const char*>(a.logits) + static_cast<size_t>(row) * a.row_stride * Vector::kElementBytes -
            static_cast<size_t>(s.misalignment) * Vector::kElementBytes;
        const uint32_t first = s.first * 8u / kWidth, last = min(s.last * 8u / kWidth, (s.end + kWidth - 1u) / kWidth);
        float largest = -INFINITY, smallest = INFINITY;
        uint32_t finite = 0, flags = 0;
        const auto take = [&](float x) {
            const uint32_t magnitude = __float_as_uint(x) & 0x7fffffffu;
            const bool counts = magnitude < 0x7f800000u;
            largest = fmaxf(largest, counts ? x : -INFINITY);
            smallest = fminf(smallest, counts ? x : INFINITY);
            finite += counts ? 1u : 0u;
            flags |= magnitude > 0x7f800000u ? static_cast<uint32_t>(kScanSawNan) : 0u;
            flags |= __float_as_uint(x) == 0x7f800000u ? static_cast<uint32_t>(kScanSawPositiveInfinity) : 0u;
        };
        // (a vector that holds other elements too: the row's first and last)
        const auto take_inside = [&](uint32_t v) {
            float x[kWidth];
            Vector::unpack(*reinterpret_cast<const uint4*>(base + static_cast<size_t>(v) * 16u), x);
#pragma unroll
            for (uint32_t c = 0; c < kWidth; ++c)
            {
                if (v * kWidth + c - s.misalignment < a.vocab)
                    take(x[c]);
            }
        };
        const uint32_t first_whole = max(first, (s.misalignment + kWidth - 1u) / kWidth);
        const uint32_t last_whole = min(last, s.end / kWidth);
        if (tid == 0 && first < min(first_whole, last))
            take_inside(first);
        if (tid == kWaveSize && first_whole <= last_whole && last_whole < last)
            take_inside(last_whole);
        for (uint32_t at = first_whole + tid; at < last_whole; at += kLoads * THREADS)
        {
            uint4 raw[kLoads];
#pragma unroll
            for (int k = 0; k < kLoads; ++k)
                raw[k] = *reinterpret_cast<const uint4*>(base + min(at + k * THREADS, last_whole - 1u) * 16u); // (rows below 2^32 bytes)
            // (as if all were finite, a quarter of the instructions: 512 rows of mixed options 17.4 -> 16.3 us, then the stream of their
            // 49 MB; a vector behind the last is that one again)
            float largest_here = largest, smallest_here = smallest;
            uint32_t twice = 0; // the largest of the bits without their signs, times two
#pragma unroll
            for (int k = 0; k < kLoads; ++k)
            {
                float x[kWidth];
                Vector::unpack(raw[k], x);
#pragma unroll
                for (uint32_t c = 0; c < kWidth; c += 2u)
                {
                    largest_here = largest_of_three(largest_here, x[c], x[c + 1]);
                    smallest_here = smallest_of_three(smallest_here, x[c], x[c + 1]);
                    twice = max(max(twice, __float_as_uint(x[c]) << 1), __float_as_uint(x[c + 1]) << 1);
                }
            }
            if (twice < 0xff000000u)
            {
                largest = largest_here;
                smallest = smallest_here;
                finite += kWidth * min(static_cast<uint32_t>(kLoads), (last_whole - at + THREADS - 1u) / THREADS);
            }
            else
            {
#pragma unroll
                for (int k = 0; k < kLoads; ++k)
                {
                    if (at + k * THREADS < last_whole)
                    {
                        float x[kWidth];
                        Vector::unpack(raw[k], x);
#pragma unroll
                        for (uint32_t c = 0; c < kWidth; ++c)
                            take(x[c]);
                    }
                }
            }
        }
        const auto reduce = [&](int lanes) {
            for (int distance = lanes / 2; distance > 0; distance >>= 1)
            {
                largest = fmaxf(largest, __shfl_xor(largest, distance, kWaveSize));
                smallest = fminf(smallest, __shfl_xor(smallest, distance, kWaveSize));
                finite += __shfl_xor(finite, distance, kWaveSize);
                flags |= __shfl_xor(flags, distance, kWaveSize);
            }
        };
        reduce(kWaveSize);
        if ((tid & (kWaveSize - 1)) == 0)
            wave_stats[tid >> 6] = uint4{__float_as_uint(largest), __float_as_uint(smallest), finite, flags};
        __syncthreads();
        if (tid < kWaveSize)
        {
            constexpr int kWaves = THREADS / kWaveSize;
            const uint4 of_wave = wave_stats[tid & (kWaves - 1)];
            largest = __uint_as_float(of_wave.x), smallest = __uint_as_float(of_wave.y), finite = of_wave.z, flags = of_wave.w;
            reduce(kWaves);
        }
        return uint4{__float_as_uint(largest), __float_as_uint(smallest), finite, flags};
    }
}

template <int DTYPE>
__global__ __launch_bounds__(kBinThreads, 8) void bin_stats_kernel(BinArgs g)
{
    __shared__ uint4 wave_stats[kBinWaves];
    __shared__ RowList listed_rows;
    const SamplerArgs& a = g.a;
    const int tid = threadIdx.x;
    const uint32_t rows = list_rows_in_place(a, g.listing, g.windows_are_selects != 0u, false, g.list, g.window_list, listed_rows, tid);
    const BinGrid grid = bin_grid(rows, a.vocab, g.most_parts);
    for (uint32_t slot = grid.first_slot; slot < grid.rows; slot += grid.slot_step)
    {
        const uint32_t row = same_in_all(row_of_slot(g.listing, g.list, listed_rows, slot));
        const uint4 of_part = stats_of_part<DTYPE, kBinThreads>(a, grid, row, wave_stats, tid);
        if (tid == 0)
            g.stats[slot * grid.parts + grid.part] = of_part;
        __syncthreads();
    }
}

// Correctly rounded quotients by one divisor: two corrections of dividend x reciprocal, each with its exact remainder (P. Markstein,
// Computation of elementary functions on the IBM RISC System/6000 processor, 1990: a quotient less than an ulp off, corrected with
// the remainder times the correctly rounded reciprocal, is the correctly rounded one).  Five instructions instead of the ten and a
// reciprocal of a division; for numbers whose quotient and remainder are far from the denormal ones, as the bins' terms are: they are
// 2^-25 to 1, a normaliser is 1 to 2^22, the divisor behind it no less than the first term over the normaliser, 2^-22.
struct Divisor
{
    float value, reciprocal;
    __device__ __forceinline__ explicit Divisor(float divisor) : value(divisor), reciprocal(1.0f / divisor) {}
    __device__ __forceinline__ float divide(float dividend) const
    {
        const float about = dividend * reciprocal;
        const float near = __builtin_fmaf(__builtin_fmaf(-about, value, dividend), reciprocal, about);
        return __builtin_fmaf(__builtin_fmaf(-near, value, dividend), reciprocal, near);
    }
};

// ---- (2) the terms, in the row's order, and how many fall into each bin
// What is known of a row before its sums: the same in each of its parts.
struct BinRowStart
{
    uint32_t state, shift, window, saw_nan;
};

// `bins`: 2 x kBins words of LDS.  ACROSS: the launch itself has written the parts' statistics, and the counts are for itself.
template <int DTYPE, int THREADS, bool ACROSS>
__device__ __forceinline__ BinRowStart terms_of_part(
    const BinArgs& g, const BinGrid& grid, uint32_t slot, uint32_t row, const ncnn_moe_sample_params& p, bool near, uint32_t* bins, uint4* part_stats,
    const uint64_t* exp2_table, int tid)
{
    using Vector = LogitsVector<DTYPE>;
    constexpr uint32_t kWidth = Vector::kWidth;
    constexpr int kLoads = (DTYPE == NCNN_MOE_LOGITS_F32 ? 4 : 2) * kBinThreads / THREADS;
    const SamplerArgs& a = g.a;
    {
        if (tid < static_cast<int>(grid.parts))
            part_stats[tid] = taken_over_vector<ACROSS>(g.stats + slot * grid.parts, grid.parts * 16u, static_cast<uint32_t>(tid));
        for (uint32_t i = tid; i < 2u * kBinQuads; i += THREADS)
            reinterpret_cast<uint4*>(bins)[i] = uint4{0u, 0u, 0u, 0u};
        __syncthreads();
        float largest = -INFINITY, smallest = INFINITY;
        uint32_t finite = 0, flags = 0;
        for (uint32_t q = 0; q < grid.parts; ++q)
        {
            const uint4 other = part_stats[q];
            largest = fmaxf(largest, __uint_as_float(other.x));
            smallest = fminf(smallest, __uint_as_float(other.y));
            finite += other.z;
            flags |= other.w;
        }
        const float maximum = largest / p.temperature;
        const bool rejected = finite == 0u || (flags & kScanSawPositiveInfinity) != 0u;
        const bool served = !rejected && is_finite_f32(maximum);
        // (the bins cover the row's range of terms, or the 25 binades that matter)
        const float least = fmaxf(smallest / p.temperature - maximum, kTailArgument);
        uint32_t distance = served ? kOneBits - __float_as_uint(expf_libm(least, exp2_table)) : 0u;
        distance = min(distance, kTailDistance - 1u);
        uint32_t shift = 0;
        while ((distance >> shift) >= kBins)
            ++shift;
        const uint32_t place_mask = (1u << shift) - 1u;
        const uint32_t place_shift = shift > kOffsetBits ? shift - kOffsetBits : 0u;
        const BinRowStart start{served ? kBinRowGoesOn : rejected ? kBinRowRejected : kBinRowLeft, shift,
                                (p.top_k > 0u && p.top_k < a.vocab && finite > p.top_k) ? p.top_k : finite, (flags & kScanSawNan) != 0u ? 1u : 0u};
        if (grid.part == 0u && tid == 0)
        {
            BinRow& record = g.records[row];
            // (pending until a walk has finished it: a first select that runs beside leaves these rows alone)
            a.row_state[row] = kRowNeedsGeneral;
            record.state[0] = start.state;
            record.shift = shift;
            record.window = start.window;
            record.served = 0u;
            record.filtered = 0u;
            record.maximum = maximum;
            record.saw_nan = start.saw_nan;
        }
        if (served)
        {
            const BinStretch s = bin_stretch<Vector::kElementBytes>(a, row, grid.part, grid.parts);
            const char* base = static_cast<const char*>(a.logits) + static_cast<size_t>(row) * a.row_stride * Vector::kElementBytes -
                static_cast<size_t>(s.misalignment) * Vector::kElementBytes;
            float* terms = bin_terms(a, row);
            const uint32_t terms_bytes = (s.end + 7u) / 8u * 32u;
            const uint32_t first = s.first * 8u / kWidth, last = min(s.last * 8u / kWidth, (s.end + kWidth - 1u) / kWidth);
            // Divided by the temperature with corrections (see Divisor) where that is exact: a quotient neither overflows nor, unless it is so small that
            // the maximum swallows it, comes near the denormal numbers.  (A logit of -inf becomes a NaN on the way: zero as well.)  What bounds the terms is
            // instructions, 42 an element with divisions and a look at each element's place in the row, 35 so: 12.2 million logits 26.0 -> 23.4 us.
            const Divisor by(p.temperature);
            const float outermost = fmaxf(fabsf(largest), fabsf(smallest));
            const bool corrected = p.temperature >= 0x1p-20f && p.temperature <= 0x1p20f && outermost <= 0x1p60f && fabsf(maximum) >= 0x1p-20f;
            const auto terms_of = [&](auto quotient) {
                for (uint32_t at = first + tid; at < last; at += kLoads * THREADS)
                {
                    uint4 raw[kLoads];
#pragma unroll
                    for (int k = 0; k < kLoads; ++k)
                    {
                        const uint32_t v = min(at + k * THREADS, last - 1u);
                        raw[k] = *reinterpret_cast<const uint4*>(base + v * 16u); // (rows below 2^32 bytes)
                    }
#pragma unroll
                    for (int k = 0; k < kLoads; ++k)
                    {
                        const uint32_t v = at + k * THREADS;
                        if (v >= last)
                            break;
                        float x[kWidth], t[kWidth];
                        Vector::unpack(raw[k], x);
                        const uint32_t position = v * kWidth;
                        if (position < s.misalignment || position + kWidth > s.end) // (the row's first vector or its last)
                        {
#pragma unroll
                            for (uint32_t c = 0; c < kWidth; ++c)
                                x[c] = position + c >= s.misalignment && position + c < s.end ? x[c] : -INFINITY;
                        }
#pragma unroll
                        for (uint32_t c = 0; c < kWidth; ++c)
                        {
                            const float argument = quotient(x[c]) - maximum;
                            // (a comparison that NaN fails as well)
                            t[c] = argument >= kTailArgument ? expf_of_small_argument(argument, exp2_table) : 0.0f;
                            const uint32_t below = kOneBits - __float_as_uint(t[c]);
                            if (below < kTailDistance)
                            {
                                atomicAdd(&bins[below >> shift], 1u);
                                atomicAdd(&bins[kBins + (below >> shift)], (below & place_mask) >> place_shift);
                            }
                        }
#pragma unroll
                        for (uint32_t c = 0; c < kWidth; c += 4u)
                            hand_over_vector(near, terms, terms_bytes, (position + c) / 4u,
                                             uint4{__float_as_uint(t[c]), __float_as_uint(t[c + 1]), __float_as_uint(t[c + 2]), __float_as_uint(t[c + 3])});
                    }
                }
            };
            if (corrected)
                terms_of([&](float x) { return by.divide(x); });
            else
                terms_of([&](float x) { return x / p.temperature; });
            // (the last group of eight positions of the row may reach a vector further than the row does)
            if (kWidth == 4u && tid == 0 && s.last * 2u > last && last > first)
                hand_over_vector(near, terms, terms_bytes, last, uint4{0u, 0u, 0u, 0u});
            __syncthreads();
            for (uint32_t i = tid; i < 2u * kBinQuads; i += THREADS)
                hand_over_vector(near, g.counts + static_cast<size_t>(slot * grid.parts + grid.part) * 2u * kBins, 2u * kBins * 4u, i, reinterpret_cast<uint4*>(bins)[i]);
        }
        return start;
    }
}

template <int DTYPE>
__global__ __launch_bounds__(kBinThreads, 8) void bin_terms_kernel(BinArgs g)
{
    __shared__ __align__(16) uint32_t bins[2 * kBins];
    __shared__ uint4 part_stats[kMaxBinParts];
    __shared__ uint64_t exp2_table[32];
    const BinGrid grid = bin_grid(g.list[0], g.a.vocab, g.most_parts);
    const int tid = threadIdx.x;
    if (tid < 32)
        exp2_table[tid] = kExp2Table[tid];
    for (uint32_t slot = grid.first_slot; slot < grid.rows; slot += grid.slot_step)
    {
        const uint32_t row = g.list[1u + slot];
        terms_of_part<DTYPE, kBinThreads, false>(g, grid, slot, row, g.a.params[row], true, bins, part_stats, exp2_table, tid);
        __syncthreads();
    }
}

// Exclusive prefix sums over the workgroup's threads (and the totals) of some integers and a float.
struct BinScanScratch
{
    uint32_t u[4][kBinWaves];
    float f[kBinWaves];
};

// The inclusive sums over each row of 16 lanes, and over the wave.
__device__ __forceinline__ uint32_t row16_prefix_sum_u32(uint32_t value)
{
    value += dpp_source<0x111, 0xf>(value); // row_shr:1
    value += dpp_source<0x112, 0xf>(value); // row_shr:2
    value += dpp_source<0x114, 0xf>(value); // row_shr:4
    value += dpp_source<0x118, 0xf>(value); // row_shr:8
    return value;
}

__device__ __forceinline__ float row16_prefix_sum_f32(float value)
{
    value += __uint_as_float(dpp_source<0x111, 0xf>(__float_as_uint(value)));
    value += __uint_as_float(dpp_source<0x112, 0xf>(__float_as_uint(value)));
    value += __uint_as_float(dpp_source<0x114, 0xf>(__float_as_uint(value)));
    value += __uint_as_float(dpp_source<0x118, 0xf>(__float_as_uint(value)));
    return value;
}

__device__ __forceinline__ float wave_prefix_sum_f32(float value)
{
    value = row16_prefix_sum_f32(value);
    value += __uint_as_float(dpp_source<0x142, 0xa>(__float_as_uint(value)));
    value += __uint_as_float(dpp_source<0x143, 0xc>(__float_as_uint(value)));
    return value;
}

template <int WAVES, bool WITH_FLOAT, int COUNT>
__device__ __forceinline__ void bin_scan_of(uint32_t (&u)[COUNT], uint32_t (&totals)[COUNT], float& f, BinScanScratch& scratch, int tid)
{
    const int lane = tid & (kWaveSize - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint32_t own[COUNT];
    uint32_t inclusive[COUNT];
#pragma unroll
    for (int i = 0; i < COUNT; ++i)
    {
        own[i] = u[i];
        inclusive[i] = wave_prefix_sum_u32(u[i]);
        if (lane == kWaveSize - 1)
            scratch.u[i][wave] = inclusive[i];
    }
    const float inclusive_f = WITH_FLOAT ? wave_prefix_sum_f32(f) : 0.0f;
    if (WITH_FLOAT && lane == kWaveSize - 1)
        scratch.f[wave] = inclusive_f;
    __syncthreads();
    static_assert(WAVES <= 16, "the waves' sums lie in one row of lanes");
#pragma unroll
    for (int i = 0; i < COUNT; ++i)
    {
        const uint32_t through = row16_prefix_sum_u32(lane < WAVES ? scratch.u[i][lane] : 0u);
        totals[i] = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(through), WAVES - 1));
        const uint32_t before = wave > 0 ? static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(through), wave - 1)) : 0u;
        u[i] = before + inclusive[i] - own[i];
    }
    if (WITH_FLOAT)
    {
        const float through = row16_prefix_sum_f32(lane < WAVES ? scratch.f[lane] : 0.0f);
        const float before = wave > 0 ? read_lane(through, wave - 1) : 0.0f;
        f = before + (inclusive_f - f);
    }
    __syncthreads();
}

template <int WAVES, int COUNT>
__device__ __forceinline__ void bin_scan(uint32_t (&u)[COUNT], uint32_t (&totals)[COUNT], float& f, BinScanScratch& scratch, int tid)
{
    bin_scan_of<WAVES, true>(u, totals, f, scratch, tid);
}

template <int WAVES, int COUNT>
__device__ __forceinline__ void bin_scan(uint32_t (&u)[COUNT], uint32_t (&totals)[COUNT], BinScanScratch& scratch, int tid)
{
    float none = 0.0f;
    bin_scan_of<WAVES, false>(u, totals, none, scratch, tid);
}

// The largest term that a bin can hold (the lower end of a bin is the upper end of the next).
__device__ __forceinline__ float bin_top(uint32_t bin, uint32_t shift)
{
    return __uint_as_float(kOneBits - (bin << shift));
}

// Plans a sum over the bins behind the head: what becomes of each of the calling thread's four bins (from `bin` on).
//   front          elements in front of each bin; front[4] behind the last
//   mass           about what the sum holds in front of each bin
//   limit          elements that the sum runs over; cut_bin: no bin behind it takes part, and the sum may end inside it
//   bound          the sum may end once it reaches this; error: relative error of the masses that lists bins
struct BinPlan
{
    uint32_t kind[4];
    uint32_t exponent[4];
    uint32_t fetched; // bit j: bin j is fetched where it does not fit the list: the sum ends inside it, or its steps are too many to add
    uint32_t listed; // elements of the four bins that should be in the list
};

__device__ __forceinline__ BinPlan plan_bins(
    uint32_t bin, const uint32_t (&front)[5], const float (&mass)[5], uint32_t head_bins, uint32_t limit, uint32_t cut_bin, float bound, float error,
    uint32_t shift, float scale)
{
    BinPlan plan;
    plan.listed = 0;
    plan.fetched = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        const uint32_t b = bin + j;
        const uint32_t count = front[j + 1] - front[j];
        const float low = mass[j] * (1.0f - error);
        const float high = mass[j + 1] * (1.0f + error);
        plan.exponent[j] = (__float_as_uint(mass[j]) >> 23) & 0xffu;
        uint32_t kind = kBinAdded;
        if (b < head_bins || front[j] >= limit || b > cut_bin || mass[j] * (1.0f - kForeseenEnd) > bound)
            kind = kBinBeyond;
        else if (count > 0u)
        {
            const bool ends = front[j + 1] > limit || b == cut_bin;
            // (terms below half an ulp of the lower of the two sums move neither)
            const bool moves = bin_top(b, shift) * scale * 1.0001f >= __uint_as_float((max(__float_as_uint(low) >> 23, 25u) - 24u) << 23);
            const bool leaves = moves && ((__float_as_uint(low) ^ __float_as_uint(high)) >> 23) != 0u;
            // (a step is a term in ulps of the sum, rounded; the quotient below is a few roundings off)
            const float ulps_per_one = __uint_as_float((277u - min(max(plan.exponent[j], 24u), 250u)) << 23);
            const float most_steps = static_cast<float>(count) * (bin_top(b, shift) * scale * 1.0001f * ulps_per_one + 1.0f);
            const bool too_many = most_steps >= kBinMostSteps;
            plan.fetched |= ends || too_many ? 1u << j : 0u;
            if (ends || leaves || (high >= bound && low <= bound))
            {
                kind = kBinListed;
                plan.listed += count;
            }
            else if (too_many)
                kind = kBinWanted;
        }
        plan.kind[j] = kind;
    }
    return plan;
}

// Whether the calling lane is the first of its wave (of those that call) for which `holds`: the one of them that speaks for the wave.
__device__ __forceinline__ bool leads_wave(bool holds)
{
    const uint64_t mask = __builtin_amdgcn_ballot_w64(holds);
    return mask != 0ull && lane_id() == __builtin_ctzll(mask);
}

// The first of the thread's bins whose terms are kWideDifference binades and more below the sum (kBins: none).
__device__ __forceinline__ uint32_t first_wide_bin(const BinPlan& plan, uint32_t bin, uint32_t shift, float scale)
{
    uint32_t first = kBins;
#pragma unroll
    for (int j = 3; j >= 0; --j)
    {
        const uint32_t top_exponent = __float_as_uint(bin_top(bin + j, shift) * scale) >> 23;
        if (plan.kind[j] == kBinAdded && plan.exponent[j] >= top_exponent + kWideDifference)
            first = bin + j;
    }
    return first;
}

// Where the thread's listed bins lie in the list (base: the position of the first); a bin that does not fit is not listed.
__device__ __forceinline__ uint32_t fit_plan(BinPlan& plan, const uint32_t (&front)[5], uint32_t base, uint32_t (&place)[4])
{
    uint32_t position = base;
    uint32_t end_of_list = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        place[j] = position;
        if (plan.kind[j] == kBinListed)
        {
            position += front[j + 1] - front[j];
            if (position > kBinListCap)
                plan.kind[j] = (plan.fetched >> j & 1u) != 0u ? kBinWanted : kBinAdded;
            else
                end_of_list = position;
        }
    }
    return end_of_list;
}

// Adds the steps of a part's terms to the bins' integers, and puts the terms of listed bins into the list.
//   entries   per bin: bit 31 the bin is listed and the rest is the next place of this part in the list; bit 30 it takes
//             no part in the sum; else the exponent assumed for the sum
//   ties      bins with a term half way between two sums (its step is counted rounded up), with a second one of the same
//             value, and with one that the masks cannot tell (the bin's terms take more than 32 steps)
//   masks     per bin, for terms kMaskedDifference binades and more below the sum: bit (step / 2) % 32 the parity of the
//             odd steps of that value; then bit step % 32 for a term half way between `step` and the next.  The kWideBins bins
//             from wide_first on have the same with 64 and 128 bits
// What bounds it: instructions, and with two waves a SIMD the trips to LDS for the bins' entries: there (kFewWaves) four terms look theirs up
// together, and their steps are made without a branch (a part of 9,500 terms by 512 threads, warm 4.95 -> 4.45 us, where the
// instructions are new 5.55 -> 5.05; of the 4.95, 0.1 were the additions to the bins and 1.5 the parities).  With eight waves a SIMD branches cost less than what
// they pass by (512 workgroups of 1,024 threads, 30,400 terms each, 17.0 with a branch, 18.0 without).  Steps are made from the terms scaled to ulps of the
// sum, with shifts of their mantissas both took 0.3 to 0.8 us more.
template <int PHASE, int THREADS, bool ACROSS>
__device__ __forceinline__ void add_bin_steps(
    const float* terms, const BinStretch& s, uint32_t shift, uint32_t first_bin, uint32_t bin_count, float divisor, float second_divisor,
    uint32_t* entries, uint32_t* steps, uint32_t* ties, uint32_t* masks, uint32_t wide_first, float* list_terms, uint32_t* list_tokens, bool near, int tid)
{
    constexpr bool kFewWaves = THREADS < kBinThreads;
    // (five, where there are registers, gain where they save a trip only: by 512 threads parts of 8,193 to 10,240 terms 5.1 -> 4.85 us, of 2,000 1.39 -> 1.43,
    // of 6,250 3.64 -> 3.69, of 12,500 6.26 -> 6.31)
    constexpr int kLoads = 4;
    const uint32_t bytes = (s.end + 7u) / 8u * 32u;
    const uint32_t first = s.first * 2u, last = s.last * 2u;
    const Divisor by(divisor), by_second(second_divisor);
    // whether the term takes part at all, and its bin's entry
    const auto entry_of = [&](float t, uint32_t& bin) {
        const uint32_t below = kOneBits - __float_as_uint(t);
        bin = below >> shift;
        const bool in = below < kTailDistance && bin - first_bin < bin_count;
        return in ? entries[min(bin, kBins - 1u)] : 0x40000000u;
    };
    // the term in ulps of the sum: exact, but for what is far below half of one
    const auto in_ulps = [&](float term, int exponent) {
        if (PHASE >= 1)
            term = by.divide(term);
        if (PHASE >= 2)
            term = by_second.divide(term);
        return __builtin_amdgcn_ldexpf(term, 150 - exponent);
    };
    // a term half way between two sums, or no smaller than the sum
    const auto is_special = [](float ulps, float rest) { return rest == 0.5f || ulps >= 8388608.0f; };
    const auto note_special = [&](uint32_t bin, uint32_t half_way, bool wide, bool told) {
        uint32_t* const wide_masks = masks + 2u * kBins + (bin - wide_first) * kWideWords;
        const uint32_t bit = 1u << (bin & 31u);
        atomicOr(&ties[bin >> 5], bit);
        if (!told)
            atomicOr(&ties[2u * kBinWords + (bin >> 5)], bit);
        else if ((atomicOr(wide ? &wide_masks[kWideParities + (half_way >> 5) % kWideHalves] : &masks[kBins + bin], 1u << (half_way & 31u)) >> (half_way & 31u) & 1u) != 0u)
            atomicOr(&ties[kBinWords + (bin >> 5)], bit);
    };
    const auto note_odd = [&](uint32_t bin, uint32_t step, bool wide) {
        atomicXor(&masks[wide ? 2u * kBins + (bin - wide_first) * kWideWords + (step >> 6) % kWideParities : bin], 1u << ((step >> 1) & 31u));
    };
    const auto list = [&](uint32_t bin, float t, uint32_t position) {
        const uint32_t place = atomicAdd(&entries[bin], 1u) & 0x7fffffffu;
        hand_over(near, list_terms, kBinListCap * 4u, place, __float_as_uint(t));
        hand_over(near, list_tokens, kBinListCap * 4u, place, position - s.misalignment);
    };
    constexpr float kTold = static_cast<float>(1 << (24 - kMaskedDifference)); // (masks of nearer terms are not looked at)
    for (uint32_t at = first + tid; at < last; at += kLoads * THREADS)
    {
        uint4 raw[kLoads];
#pragma unroll
        for (int k = 0; k < kLoads; ++k)
            raw[k] = taken_over_vector<ACROSS>(terms, bytes, min(at + k * THREADS, last - 1u));
#pragma unroll
        for (int k = 0; k < kLoads; ++k)
        {
            const uint32_t v = at + k * THREADS;
            if (v >= last)
                break;
            const float t[4] = {__uint_as_float(raw[k].x), __uint_as_float(raw[k].y), __uint_as_float(raw[k].z), __uint_as_float(raw[k].w)};
            if constexpr (kFewWaves)
            {
                uint32_t bin[4], entry[4];
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    entry[c] = entry_of(t[c], bin[c]);
#pragma unroll
                for (int c = 0; c < 4; ++c)
                {
                    const bool added = (entry[c] & 0xc0000000u) == 0u;
                    const float ulps = in_ulps(t[c], added ? static_cast<int>(entry[c]) : 350); // (none at all where it is not added)
                    const float rest = __builtin_amdgcn_fractf(ulps);
                    const uint32_t step = static_cast<uint32_t>(ulps) + (rest >= 0.5f ? 1u : 0u);
                    const bool wide = bin[c] - wide_first < kWideBins;
                    const bool told = wide || ulps < kTold;
                    const bool special = is_special(ulps, rest) || (entry[c] & 0x80000000u) != 0u;
                    if (step != 0u)
                        atomicAdd(&steps[bin[c]], step);
                    if ((step & 1u) != 0u && told && !special)
                        note_odd(bin[c], step, wide);
                    if (special)
                    {
                        if (added)
                            note_special(bin[c], step - 1u, wide, told);
                        else
                            list(bin[c], t[c], v * 4u + c);
                    }
                }
            }
            else
            {
#pragma unroll
                for (int c = 0; c < 4; ++c)
                {
                    uint32_t bin;
                    const uint32_t entry = entry_of(t[c], bin);
                    if ((entry & 0xc0000000u) == 0u)
                    {
                        const float ulps = in_ulps(t[c], static_cast<int>(entry));
                        const float rest = __builtin_amdgcn_fractf(ulps);
                        const uint32_t step = static_cast<uint32_t>(ulps) + (rest >= 0.5f ? 1u : 0u);
                        atomicAdd(&steps[bin], step);
                        const bool wide = bin - wide_first < kWideBins;
                        const bool told = wide || ulps < kTold;
                        if (is_special(ulps, rest))
                            note_special(bin, step - 1u, wide, told);
                        else if ((step & 1u) != 0u && told)
                            note_odd(bin, step, wide);
                    }
                    else if ((entry & 0x80000000u) != 0u)
                        list(bin, t[c], v * 4u + c);
                }
            }
        }
    }
}

// What a row's sums hand to each other, in LDS: the same in each of its parts, which all do the same.
struct BinWalkRow
{
    uint32_t shift;         // a term's bin: (kOneBits - bits) >> shift
    uint32_t window;        // elements of the Top-K window (finite logits at most)
    uint32_t saw_nan;
    uint32_t options[kRowOptionWords]; // ncnn_moe_sample_params, then the uniform
    uint32_t binned;        // elements in bins
    uint32_t head_bins;     // bins [0, head_bins) are the head, head_count elements
    uint32_t head_count;
    float normalizer, renormalizer;
    float head_sum;         // the next walk's sum behind the head
    uint32_t limit;         // elements that it runs over at most
    uint32_t kept;
    uint32_t cut_bin;       // Min-P: the bin that holds the smallest term kept (kBins: no cut inside the bins), and that term
    float cut_term;
    uint32_t cut_in_tail;   // ... or it lies in no bin
    uint32_t listed;        // elements in the list of the next walk (the first walk's holds the head, the others' places behind it)
    uint32_t wide_first;    // of its sum: the first of the kWideBins bins with wide masks
};

// ---- (3) the head and the bins whose order is foreseen to matter go to the list; the others' steps of the normaliser
struct BinSumShared
{
    uint32_t bins_behind_heads[2], heads_hold[2], end_of_list, wide_first_of_row;
    float longest_holds, row_holds;
};

// `entries`, `steps`: kBins words of LDS, `masks`: kMaskWords, `ties`: 3 x kBinWords.  ACROSS: the launch itself has written the parts'
// counts, and the steps are for itself.  Fills in `carried` for the first walk, and returns the calling thread's four bins.
template <int THREADS, bool ACROSS>
__device__ __forceinline__ uint4 sum_of_part(
    const BinArgs& g, const BinGrid& grid, uint32_t slot, uint32_t row, float top_p, float min_p, bool near, const BinStretch& s, uint32_t* entries, uint32_t* steps, uint32_t* masks, uint32_t* ties,
    BinScanScratch& scan, BinSumShared& shared, BinWalkRow& carried, int tid)
{
    constexpr int kWaves = THREADS / kWaveSize;
    constexpr bool kPlacesApart = THREADS / 2 >= static_cast<int>(kBinQuads); // other threads load where in their bins the terms lie
    uint32_t (&bins_behind_heads)[2] = shared.bins_behind_heads;
    uint32_t (&heads_hold)[2] = shared.heads_hold;
    uint32_t &end_of_list = shared.end_of_list, &wide_first_of_row = shared.wide_first_of_row;
    float &longest_holds = shared.longest_holds, &row_holds = shared.row_holds;
    const SamplerArgs& a = g.a;
    const uint32_t bin = 4u * static_cast<uint32_t>(tid);
    const bool holds_bins = tid < static_cast<int>(kBinQuads);
    {
        const uint32_t shift = same_in_all(carried.shift);
        const uint32_t window = same_in_all(carried.window);
        uint4 words{0u, 0u, 0u, 0u};
        // counts of the thread's bins, of the whole row and of the parts in front of this one, and where in their bins the terms lie
        uint32_t count[4] = {0u, 0u, 0u, 0u}, before[4] = {0u, 0u, 0u, 0u};
        // (counted in vectors of four bins, `first_vector` of each part's; `before`: of the parts in front)
        const auto collect = [&](uint32_t first_vector, uint32_t (&all)[4], uint32_t (&in_front)[4]) {
            uint32_t* const counts = g.counts + static_cast<size_t>(slot * grid.parts) * 2u * kBins;
            const uint32_t bytes = grid.parts * 2u * kBins * 4u;
            // (four parts' at a time: all sixteen's, in fours where a row has fewer parts, gave long rows nothing, and the code made every short one wait: 3 rows
            // of 600 28.2 us so and 29.0, 5 of 5,000 37.5 and 38.4, 60 of 4,000 37.9 and 38.8, 8 of 151,936 86.9 and 87.4)
            for (uint32_t first = 0; first < grid.parts; first += kPartsAtATime)
            {
                uint4 of_part[kPartsAtATime];
#pragma unroll
                for (uint32_t k = 0; k < kPartsAtATime; ++k)
                    of_part[k] = taken_over_vector<ACROSS>(counts, bytes, min(first + k, grid.parts - 1u) * 2u * kBinQuads + first_vector);
#pragma unroll
                for (uint32_t k = 0; k < kPartsAtATime; ++k)
                {
                    const uint32_t some = first + k < grid.parts ? 0xffffffffu : 0u;
                    const uint32_t some_before = first + k < grid.part ? 0xffffffffu : 0u;
                    const uint32_t c[4] = {of_part[k].x, of_part[k].y, of_part[k].z, of_part[k].w};
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                    {
                        all[j] += c[j] & some; // (places: below 2^22 x 2^12; only a bin of a million terms wraps, a wrong guess)
                        in_front[j] += c[j] & some_before;
                    }
                }
            }
        };
        uint32_t places[4] = {0u, 0u, 0u, 0u};
        if constexpr (kPlacesApart)
        {
            const bool holds_places = tid >= THREADS / 2 && tid < THREADS / 2 + static_cast<int>(kBinQuads);
            if (holds_bins || holds_places)
                collect(holds_bins ? static_cast<uint32_t>(tid) : kBinQuads + static_cast<uint32_t>(tid) - THREADS / 2, count, before);
            if (holds_places)
                reinterpret_cast<uint4*>(steps)[tid - THREADS / 2] = uint4{count[0], count[1], count[2], count[3]};
            __syncthreads();
            if (holds_bins)
            {
                const uint4 words = reinterpret_cast<const uint4*>(steps)[tid];
                places[0] = words.x, places[1] = words.y, places[2] = words.z, places[3] = words.w;
            }
            else
            {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    count[j] = before[j] = 0u;
            }
        }
        else if (holds_bins)
        {
            uint32_t none[4] = {0u, 0u, 0u, 0u};
            collect(static_cast<uint32_t>(tid), count, before);
            collect(kBinQuads + static_cast<uint32_t>(tid), places, none);
        }
        if (tid == 0)
        {
            bins_behind_heads[0] = bins_behind_heads[1] = heads_hold[0] = heads_hold[1] = end_of_list = 0u;
            wide_first_of_row = kBins;
        }
        if (holds_bins)
            reinterpret_cast<uint4*>(steps)[tid] = uint4{0u, 0u, 0u, 0u};
        for (uint32_t i = tid; i < kMaskWords / 4u; i += THREADS)
            reinterpret_cast<uint4*>(masks)[i] = uint4{0u, 0u, 0u, 0u};
        if (tid < static_cast<int>(3u * kBinWords))
            ties[tid] = 0u;
        // elements and mass in front of the thread's bins: first the plain masses, then what the sum makes of them (a term
        // of few ulps of the sum is rounded, the same way all over a bin: up to half an ulp a term, thousands of them)
        uint32_t front[5];
        float mass[5];
        uint32_t binned;
        {
            uint32_t total[1] = {count[0] + count[1] + count[2] + count[3]};
            uint32_t totals[1];
            float own[4];
            float masses = 0.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                const float top = bin_top(bin + j, shift);
                const float width = top - bin_top(bin + j + 1u, shift);
                own[j] = count[j] == 0u ? 0.0f
                    : static_cast<float>(count[j]) * top - width * static_cast<float>(places[j]) * (shift > kOffsetBits ? 1.0f / (1u << kOffsetBits) : 1.0f / static_cast<float>(1u << shift));
                masses += own[j];
            }
            bin_scan<kWaves>(total, totals, masses, scan, tid);
            binned = totals[0];
            front[0] = total[0];
            mass[0] = masses;
            float rounded = 0.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                front[j + 1] = front[j] + count[j];
                mass[j + 1] = mass[j] + own[j];
                if (count[j] != 0u && mass[j] > 0.0f)
                {
                    const uint32_t exponent = __float_as_uint(mass[j]) >> 23; // (the sum is 1 or more: no denormal ulps)
                    const float ulp = __uint_as_float((max(exponent, 24u) - 23u) << 23);
                    const float steps_per_ulp = __uint_as_float((277u - min(max(exponent, 24u), 250u)) << 23); // 1 / ulp
                    const float lowest = bin_top(bin + j + 1u, shift) * steps_per_ulp;
                    const float span = bin_top(bin + j, shift) * steps_per_ulp - lowest;
                    if (span < 1.0f)
                    {
                        const float whole = floorf(lowest + 0.5f);
                        const float above = fminf(fmaxf((lowest + span - (whole + 0.5f)) / span, 0.0f), 1.0f);
                        own[j] = static_cast<float>(count[j]) * (whole + above) * ulp;
                    }
                }
                rounded += own[j];
            }
            uint32_t none[1] = {0u};
            bin_scan<kWaves>(none, totals, rounded, scan, tid);
            mass[0] = rounded;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                mass[j + 1] = mass[j] + own[j];
        }
        // The head: as many bins as hold kBinHead elements at most, or those that hold the whole of a narrow window.  Where a
        // bin's terms are kWideDifference binades below the sum, its masks tell how those half way are rounded, and a sorted head
        // would save the walk nothing: it ends there (two binades further: verification without a window 168 us instead of 163)
        // unless the longest head holds the row's Top-P as well, and with it the ends of the second and third walk (64 x 4,096,
        // Top-P 0.95: 81.8 us with the head that ends early, 58.8 us so), or nearly: most draws end in it then (100 x 8,192, Top-P
        // 0.9: 114.1 us where it has to hold all of it, 104.4 us so; 32 x 32,000 and 8 x 151,936, whose heads hold less, as before).
        // What counts as nearly matters little: over 100 x 4,096, 8,192 and 16,384, 32 x 16,384 and 32,000 and 8 x 151,936, Top-P 0.8 to
        // 0.99 and spreads of 2 to 3, the mean of 72 such calls is 96.0 us at 0.5, 95.9 at 0.7 to 0.85, 96.2 at 0.9 and 97.9 at 1.
        // A row or a window of kBinWholeRow elements at most is all head, and its first walk its last: 300 x 2,000, Top-P 1, 158 us with
        // heads of 1,920 at most, 75 us so.  The longest head is kept as well where the Min-P cut lies in it and not in the early one: the
        // other sums end at the cut (100 x 32,000, Top-P 0.9 and Min-P 0.02: 107.0 us without, 92.5 us so; 4 x 50,257 72.9 and 59.8;
        // 300 x 16,384, Top-P 1 and Min-P 0.02: 132.6 and 100.4).
        const bool window_in_head = window <= kBinWholeRow;
        const uint32_t most_in_head = binned <= kBinWholeRow ? kBinWholeRow : kBinHead;
        {
            // (the bins of a head are the first ones: one that is not of it ends it)
            uint32_t first_not[2] = {kBins, kBins};
#pragma unroll
            for (int j = 3; j >= 0; --j)
            {
                const bool in_longest = window_in_head ? front[j] < window : front[j + 1] <= most_in_head;
                const bool told_by_masks = !window_in_head && bin_top(bin + j, shift) * static_cast<float>(1 << kWideDifference) < mass[j];
                if (!in_longest && bin + j != 0u)
                    first_not[0] = bin + j;
                if ((!in_longest || told_by_masks) && bin + j != 0u)
                    first_not[1] = bin + j;
            }
#pragma unroll
            for (int head = 0; head < 2; ++head)
            {
                // smallest over the workgroup, through the largest of the complement
                const uint32_t most = wave_max_u32(holds_bins ? kBins - first_not[head] : 0u);
                if ((tid & (kWaveSize - 1)) == 0 && most != 0u)
                    atomicMax(&bins_behind_heads[head], most);
            }
            if (tid == static_cast<int>(kBinQuads) - 1)
                row_holds = mass[4];
        }
        __syncthreads();
        const uint32_t longest_bins = kBins - bins_behind_heads[0], early_bins = kBins - bins_behind_heads[1];
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            if (holds_bins && bin + j + 1u == longest_bins)
            {
                heads_hold[0] = front[j + 1];
                longest_holds = mass[j + 1];
            }
            if (holds_bins && bin + j + 1u == early_bins)
                heads_hold[1] = front[j + 1];
        }
        __syncthreads();
        const bool nearly_holds_top_p = longest_holds >= kNearlyTopP * top_p * row_holds;
        const bool holds_cut = bin_top(longest_bins, shift) < min_p && !(bin_top(early_bins, shift) < min_p); // (a term survives from about min_p on)
        const uint32_t taken = nearly_holds_top_p || holds_cut ? 0u : 1u;
        uint32_t head_bins = taken == 0u ? longest_bins : early_bins;
        uint32_t head_count = heads_hold[taken];
        if (head_count > kBinListCap)
            head_bins = head_count = 0u; // (thousands of equal terms at the row's top: no head, the walks begin by fetching them)
        const bool beyond = window > head_count && binned > head_count; // the sum goes on behind the head
        BinPlan plan = plan_bins(bin, front, mass, head_bins, beyond ? window : 0u, kBins, INFINITY, kForeseenFirst, shift, 1.0f);
        uint32_t listed[1] = {holds_bins ? plan.listed : 0u};
        {
            uint32_t totals[1];
            bin_scan<kWaves>(listed, totals, scan, tid);
        }
        uint32_t place[4];
        const uint32_t own_end = fit_plan(plan, front, head_count + listed[0], place);
        if (holds_bins)
        {
            const uint32_t wide_first = first_wide_bin(plan, bin, shift, 1.0f);
            if (leads_wave(wide_first < kBins))
                atomicMin(&wide_first_of_row, wide_first);
            uint32_t packed[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                const bool in_head = bin + j < head_bins;
                packed[j] = (plan.kind[j] << 30) | (plan.exponent[j] << 22) | front[j];
                entries[bin + j] = in_head ? (0x80000000u | (front[j] + before[j]))
                    : plan.kind[j] == kBinListed ? (0x80000000u | (place[j] + before[j]))
                    : plan.kind[j] == kBinAdded ? plan.exponent[j] : 0x40000000u;
            }
            words = uint4{packed[0], packed[1], packed[2], packed[3]};
            reinterpret_cast<uint4*>(g.before + static_cast<size_t>(slot * grid.parts + grid.part) * kBins)[tid] = uint4{before[0], before[1], before[2], before[3]};
            if (own_end != 0u)
                atomicMax(&end_of_list, own_end);
        }
        __syncthreads();
        if (tid == 0)
        {
            carried.binned = binned;
            carried.head_bins = head_bins;
            carried.head_count = head_count;
            carried.listed = max(end_of_list, head_count);
            carried.wide_first = wide_first_of_row;
        }
        add_bin_steps<0, THREADS, ACROSS>(bin_terms(a, row), s, shift, 0u, beyond ? kBins : head_bins, 1.0f, 1.0f, entries, steps, ties, masks, wide_first_of_row,
                                      g.list_terms[0] + static_cast<size_t>(row) * kBinListCap, g.list_tokens[0] + static_cast<size_t>(row) * kBinListCap, near, tid);
        __syncthreads();
        if (beyond)
        {
            const size_t pair = slot * grid.parts + grid.part;
            if (holds_bins)
                hand_over_vector(near, g.steps[0] + pair * kBins, kBins * 4u, static_cast<uint32_t>(tid), reinterpret_cast<uint4*>(steps)[tid]);
            for (uint32_t i = tid; i < kMaskWords / 4u; i += THREADS)
                hand_over_vector(near, g.masks[0] + pair * kMaskWords, kMaskWords * 4u, i, reinterpret_cast<uint4*>(masks)[i]);
            if (tid < static_cast<int>(3u * kBinWords))
                hand_over(near, g.ties[0] + pair * 3u * kBinWords, 3u * kBinWords * 4u, static_cast<uint32_t>(tid), ties[tid]);
        }
        return words;
    }
}

__global__ __launch_bounds__(kBinThreads, 8) void bin_sum_kernel(BinArgs g, uint32_t element_bytes)
{
    __shared__ __align__(16) uint32_t entries[kBins];
    __shared__ __align__(16) uint32_t steps[kBins];
    __shared__ __align__(16) uint32_t masks[kMaskWords];
    __shared__ uint32_t ties[3 * kBinWords];
    __shared__ BinScanScratch scan;
    __shared__ BinSumShared shared;
    __shared__ BinWalkRow carried;
    const SamplerArgs& a = g.a;
    const BinGrid grid = bin_grid(g.list[0], a.vocab, g.most_parts);
    const int tid = threadIdx.x;
    for (uint32_t slot = grid.first_slot; slot < grid.rows; slot += grid.slot_step)
    {
        const uint32_t row = g.list[1u + slot];
        BinRow& record = g.records[row];
        if (record.state[0] != kBinRowGoesOn)
        {
            if (grid.part == 0u && tid == 0)
                record.state[1] = record.state[0];
            continue;
        }
        if (tid == 0)
        {
            carried.shift = record.shift;
            carried.window = record.window;
        }
        __syncthreads();
        const BinStretch s = element_bytes == 4u ? bin_stretch<4>(a, row, grid.part, grid.parts) : bin_stretch<2>(a, row, grid.part, grid.parts);
        const uint4 words = sum_of_part<kBinThreads, false>(g, grid, slot, row, same_in_all(a.params[row].top_p), same_in_all(a.params[row].min_p), true, s, entries, steps, masks, ties, scan, shared, carried, tid);
        if (grid.part == 0u && tid < static_cast<int>(kBinQuads))
            reinterpret_cast<uint4*>(g.packed + static_cast<size_t>(row) * kBins)[tid] = words;
        if (grid.part == 0u && tid == 0)
        {
            record.state[1] = kBinRowGoesOn;
            record.binned = carried.binned;
            record.head_bins = carried.head_bins;
            record.head_count = carried.head_count;
            record.listed = carried.listed;
            record.wide_first = carried.wide_first;
        }
        __syncthreads();
    }
}

struct WaveSum
{
    float sum;
    uint32_t index; // of the term at which the stop condition first held
    bool stopped;
};

// The terms at terms[0 .. count) (LDS, in descending order) added to `sum` by one wave, one addition behind the other, 64 of them in some
// 530 cycles (`scratch`: see wave_sequential_total).  Scans of the terms' steps, two terms a lane and one scan more for each
// binade that the sum leaves, took 2,000 to 2,300 cycles for up to 128 terms.
template <int PHASE>
__device__ __forceinline__ WaveSum wave_add_in_order(
    const float* terms, uint32_t count, float sum, int mode, float bound, float divisor, float second_divisor, float* scratch)
{
    const uint32_t lane = static_cast<uint32_t>(lane_id());
    for (uint32_t first = 0; first < count; first += kWaveSize)
    {
        const uint32_t here = min(count - first, static_cast<uint32_t>(kWaveSize));
        float own = lane < here ? terms[first + lane] : 0.0f;
        if (PHASE >= 1)
            own = own / divisor;
        if (PHASE >= 2)
            own = own / second_divisor;
        scratch[lane] = own;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (uint32_t part = 0; part < here; part += kTotalled)
        {
            const float behind = wave_sequential_total(scratch, static_cast<int>(part), sum);
            if ((mode == kStopAtOrAbove && behind >= bound) || (mode == kStopAbove && behind > bound))
            {
                // (the sums never fall: one of these is the first)
                own = lane < kTotalled ? scratch[part + lane] : 0.0f;
                own = lane == 0u ? sum + own : own;
                const float sums = wave_sequential_sums_of_first<16>(own, kTotalled);
                const bool stops = (mode == kStopAtOrAbove && sums >= bound) || (mode == kStopAbove && sums > bound);
                const int at = __builtin_ctzll(__builtin_amdgcn_ballot_w64(lane < kTotalled && stops));
                return WaveSum{read_lane(sums, at), first + part + static_cast<uint32_t>(at), true};
            }
            sum = behind;
        }
        __builtin_amdgcn_wave_barrier();
    }
    return WaveSum{sum, 0u, false};
}

// `count` additions of one term.
template <int PHASE>
__device__ __forceinline__ WaveSum wave_add_repeated(
    float term, uint32_t count, float sum, int mode, float bound, float divisor, float second_divisor)
{
    if (PHASE >= 1)
        term = term / divisor;
    if (PHASE >= 2)
        term = term / second_divisor;
    uint32_t done = 0;
    while (done < count)
    {
        int exponent;
        uint32_t mantissa;
        decode_sum(sum, exponent, mantissa);
        const uint32_t stop_at = stop_mantissa(mode, bound, exponent);
        const uint32_t limit = min(stop_at, kBinadeFull);
        const ParityStep single = step_of_term(term, exponent);
        const bool odd = (mantissa & 1u) != 0u;
        const uint32_t left = count - done;
        if (mantissa + repeated_step(odd, single, left) < limit)
            return WaveSum{encode_sum(exponent, mantissa + repeated_step(odd, single, left)), 0u, false};
        uint32_t none = 0, some = left; // `none` additions stay below the limit, `some` reach it
        while (some - none > 1u)
        {
            const uint32_t middle = none + ((some - none) >> 1);
            if (mantissa + repeated_step(odd, single, middle) >= limit)
                some = middle;
            else
                none = middle;
        }
        const uint32_t before = mantissa + repeated_step(odd, single, none);
        const uint32_t after = apply_step(before, single);
        if (after < kBinadeFull)
            return WaveSum{encode_sum(exponent, after), done + none, true};
        sum = encode_sum(exponent, before) + term;
        if ((mode == kStopAtOrAbove && sum >= bound) || (mode == kStopAbove && sum > bound))
            return WaveSum{sum, done + none, true};
        done += none + 1u;
    }
    return WaveSum{sum, 0u, false};
}

// Of the sums over a sorted stretch of terms in LDS (sum_chunks, sum_head): per 64 terms their plain sum,
// and what they do to a sum of that exponent.
struct HeadScratch
{
    alignas(16) float in_order[kWaveSize]; // (see wave_sequential_total)
    float chunk_sum[kWaveSize];
    uint32_t chunk_exponent[kWaveSize], chunk_even[kWaveSize], chunk_odd[kWaveSize];
    float sum;
    uint32_t stop; // 0xffffffff: no element met the stop condition
};

constexpr uint32_t kBinMasks = 128;      // bins with terms half way whose masks the walk keeps
constexpr uint32_t kHasMasks = 0x8000u;
constexpr uint32_t kStopExponent = 0x80000000u; // a stop: nothing but a new exponent from this bin on
constexpr uint32_t kStopRun = 0x40000000u;      // ... the next bins are listed as well
constexpr uint32_t kStopBin = 0x3fffffffu;

struct BinWalkShared
{
    alignas(16) uint32_t packed[kBins + 4]; // [kBins]: the elements in bins
    alignas(16) uint32_t prefix[kBins + 4]; // steps added in front of each bin (modulo 2^32)
    alignas(16) float terms[kBinListCap + kBinExtraCap];
    alignas(16) uint32_t tokens[kBinListCap + kBinExtraCap];
    uint16_t places[kBins + 2];             // where a listed bin's elements begin (as many are listed in front of the others); kHasMasks + i: the bin's masks are the i-th
    uint32_t bin_masks[kWideWords * kBinMasks]; // of bins with terms half way: parities, then the values half way (one word each unless the bin is a wide one)
    uint16_t mask_bin[kBinMasks];
    uint32_t mask_count, any_ties;
    uint32_t stop_bin[kBinStops];           // bins at which the walk looks closer, in order (kStopBin, kStopExponent, kStopRun)
    uint32_t ties[2 * kBinWords];           // bins with terms half way; those of them that the masks do not tell
    BinScanScratch scan;
    HeadScratch head;
    // the walk's state between two fetches
    uint32_t status; // 0: elements of bins [low, high] are wanted; 1: ended; 2: given up
    uint32_t low, high;
    uint32_t extra_count, extra_least, extra_most;
    float sum;
    uint32_t stopped;
    uint32_t stop_rank;  // rank in the sorted row, and place in terms[], of the element the sum stopped at
    uint32_t stop_at;
    uint32_t taken;      // elements added when the sum ran to its end
    uint32_t listed_end, wide_first;
    int32_t token;
    uint32_t least_key, most_key, matches; // see token_of_equal
    uint32_t many;                          // see order_elements
    uint32_t met, near;                     // see parts_meet
    BinWalkRow row;
};

constexpr uint32_t kBinExtraPlace = kBinListCap;

// How many places for each of `count` elements order_elements tells apart: two where the counters fit.
__device__ __forceinline__ uint32_t fineness_of(uint32_t place, uint32_t count)
{
    return count <= 4u * kWalkThreads && (place & ~3u) + 2u * count + 8u <= kBinListCap + kBinExtraCap ? 2u : 1u;
}

// Puts `count` elements (thread i % kWalkThreads holds element i, its term and token in registers) in descending order of
// their terms at terms[place ..], tokens[place ..].  `fine` is about where each belongs (0 .. fineness * count - 1, falling with the
// term): elements of one `fine` are neighbours, few of them unless they are equal, and are ranked against each other.
// The place where the tokens go (and some behind it) counts the elements of each `fine` first.  Every thread calls it.
// What bounds it: trips to LDS one behind the other (zero, count, front, place, rank, write).  A thread's elements make them
// together, four at a time, and are told apart twice as finely as there are elements: one element behind the other, with as many
// places as elements, 1,910 of them took 10,400 cycles, 5,200 in the ranking; so 6,300 and 2,400.
template <uint32_t PER_THREAD>
__device__ __forceinline__ void order_elements(
    BinWalkShared& shared, uint32_t place, uint32_t count, uint32_t fineness, const float (&own)[PER_THREAD], const uint32_t (&token)[PER_THREAD],
    const uint32_t (&fine)[PER_THREAD], int tid)
{
    constexpr uint32_t kMixed = 0x80000000u; // the elements of this `fine` are not all equal
    constexpr uint32_t kMany = 16;           // ... which is looked at where so many have one `fine`
    constexpr uint32_t kTogether = PER_THREAD < 4u ? PER_THREAD : 4u;
    static_assert(PER_THREAD % kTogether == 0u, "a thread's elements are whole groups");
    uint32_t* const counters = shared.tokens + (place & ~3u); // (16-byte aligned)
    uint32_t* const tokens = shared.tokens + place;
    float* const terms = shared.terms + place;
    const uint32_t places = fineness * count;
    uint32_t at[PER_THREAD], turn[PER_THREAD];
    // calls f(k, whether the thread has a k-th element) for each k, those of four k behind each other without a branch between
    const auto each_element = [&](auto f) {
#pragma unroll
        for (uint32_t first = 0; first < PER_THREAD; first += kTogether)
        {
            if (first * kWalkThreads < count)
            {
#pragma unroll
                for (uint32_t k = first; k < first + kTogether; ++k)
                    f(k, k * kWalkThreads + tid < count);
            }
        }
    };
    for (uint32_t i = 4u * static_cast<uint32_t>(tid); i < places; i += 4u * kWalkThreads)
        *reinterpret_cast<uint4*>(counters + i) = uint4{0u, 0u, 0u, 0u};
    if (tid == 0)
        shared.many = 0u;
    __syncthreads();
    each_element([&](uint32_t k, bool mine) {
        turn[k] = 0u;
        if (mine)
            turn[k] = atomicAdd(&counters[fine[k]], 1u);
    });
    {
        uint32_t most = 0;
        each_element([&](uint32_t k, bool) { most = max(most, turn[k]); });
        if (most + 1u >= kMany)
            shared.many = 1u;
    }
    __syncthreads();
    const bool many = same_in_all(shared.many) != 0u;
    {
        // (four counters a thread, eight where that is not enough)
        const uint32_t groups = places <= 4u * kWalkThreads ? 1u : 2u;
        static_assert(PER_THREAD <= 8u, "two groups of four counters a thread");
        const uint32_t first = 4u * groups * static_cast<uint32_t>(tid);
        uint4 held[2] = {uint4{0u, 0u, 0u, 0u}, uint4{0u, 0u, 0u, 0u}};
        if (first < places)
            held[0] = *reinterpret_cast<const uint4*>(counters + first);
        if (groups == 2u && first + 4u < places)
            held[1] = *reinterpret_cast<const uint4*>(counters + first + 4u);
        const uint32_t of_first = held[0].x + held[0].y + held[0].z + held[0].w;
        uint32_t total[1] = {of_first + held[1].x + held[1].y + held[1].z + held[1].w};
        uint32_t totals[1];
        bin_scan<kWalkWaves>(total, totals, shared.scan, tid);
        const auto fronts_of = [](uint32_t front, const uint4& v) { return uint4{front, front + v.x, front + v.x + v.y, front + v.x + v.y + v.z}; };
        if (first < places)
            *reinterpret_cast<uint4*>(counters + first) = fronts_of(total[0], held[0]);
        if (groups == 2u && first + 4u < places)
            *reinterpret_cast<uint4*>(counters + first + 4u) = fronts_of(total[0] + of_first, held[1]);
    }
    __syncthreads();
    uint32_t low[PER_THREAD], length[PER_THREAD];
    each_element([&](uint32_t k, bool) {
        low[k] = counters[fine[k]];
        length[k] = counters[min(fine[k] + 1u, places - 1u)];
    });
    each_element([&](uint32_t k, bool mine) {
        length[k] = mine ? (fine[k] + 1u < places ? length[k] : count) - low[k] : 0u;
        at[k] = low[k] + turn[k];
        if (mine)
            terms[at[k]] = own[k];
    });
    __syncthreads();
    if (many)
    {
        // (thousands of equal elements are not ranked against each other)
        each_element([&](uint32_t k, bool mine) {
            if (mine && terms[low[k]] != own[k])
                atomicOr(&counters[fine[k]], kMixed);
        });
        __syncthreads();
        each_element([&](uint32_t k, bool mine) { length[k] = mine && (counters[fine[k]] & kMixed) != 0u ? length[k] : 0u; });
    }
#pragma unroll
    for (uint32_t first = 0; first < PER_THREAD; first += kTogether)
    {
        if (first * kWalkThreads >= count)
            break;
        uint32_t longest = 0;
#pragma unroll
        for (uint32_t k = first; k < first + kTogether; ++k)
        {
            length[k] = length[k] > 1u ? length[k] : 0u;
            at[k] = length[k] != 0u ? low[k] : at[k];
            longest = max(longest, length[k]);
        }
        for (uint32_t t = 0; __builtin_amdgcn_ballot_w64(t < longest) != 0ull; t += 2u)
        {
            float other[2][kTogether];
#pragma unroll
            for (uint32_t i = 0; i < kTogether; ++i)
            {
                // (behind the group's last element: any, which is left out below)
                other[0][i] = terms[t < length[first + i] ? low[first + i] + t : 0u];
                other[1][i] = terms[t + 1u < length[first + i] ? low[first + i] + t + 1u : 0u];
            }
#pragma unroll
            for (uint32_t i = 0; i < kTogether; ++i)
            {
                const uint32_t k = first + i;
                // (as numbers the terms are ordered like their bits, and an equal one counts where its turn is the earlier)
                at[k] += t < length[k] && __float_as_uint(other[0][i]) >= __float_as_uint(own[k]) + (t < turn[k] ? 0u : 1u) ? 1u : 0u;
                at[k] += t + 1u < length[k] && __float_as_uint(other[1][i]) >= __float_as_uint(own[k]) + (t + 1u < turn[k] ? 0u : 1u) ? 1u : 0u;
            }
        }
    }
    __syncthreads();
    each_element([&](uint32_t k, bool mine) {
        if (mine)
        {
            terms[at[k]] = own[k];
            tokens[at[k]] = token[k];
        }
    });
    __syncthreads();
}

// About where in a bin of `count` elements a term lies.
__device__ __forceinline__ uint32_t fine_place(float term, uint32_t shift, uint32_t count)
{
    const uint32_t within = (kOneBits - __float_as_uint(term)) & ((1u << shift) - 1u);
    return static_cast<uint32_t>((static_cast<uint64_t>(within) * count) >> shift);
}

// Fetches the elements of bins [shared.low, shared.high] (at most kBinExtraCap of them; shared.extra_count: how many there
// are), in order, to shared.terms[kBinExtraPlace ..].
// What bounds it: the row's terms through one compute unit with two wavefronts per SIMD in flight (8 to 9 us for 151,936),
// then the elements found (1,500 of them some 20 us more: a place each, then order).  Every load waited for in turn and five
// instructions per element took 20 us before any was found, and with many rows the call waits for the one that fetches most
// often; with the next loads under way and one comparison per element a call of 512 mixed rows of 129,280 took 352 us
// instead of 366.
template <bool CHAINED>
__device__ __forceinline__ void fetch_bins(const float* terms, uint32_t positions, uint32_t misalignment, uint32_t shift, BinWalkShared& shared, int tid)
{
    constexpr uint32_t kLoads = CHAINED ? 8 : 4; // (twice: those under way and those looked at)
    constexpr uint32_t kStride = kLoads * kWalkThreads;
    if (tid == 0)
    {
        shared.extra_count = 0u;
        shared.extra_least = 0xffffffffu;
        shared.extra_most = 0u;
    }
    __syncthreads();
    const uint32_t top = kOneBits - (shared.low << shift);        // bits of the largest term wanted
    const uint32_t width = (shared.high + 1u - shared.low) << shift;
    // (the bins end kTailDistance below one: neither a term below them nor a zero lies within `width` of `top`)
    static_assert((kBins << 17) == kTailDistance && ((kTailDistance - 1u) >> 17) < kBins, "a bin is at most 2^17 wide");
    const uint32_t vectors = positions / 4u;
    const auto load = [&](uint4 (&raw)[kLoads], uint32_t at) {
#pragma unroll
        for (uint32_t k = 0; k < kLoads; ++k)
            raw[k] = taken_over_vector<CHAINED>(terms, positions * 4u, min(at + k * kWalkThreads, vectors - 1u));
    };
    // (a wave makes room for its elements with one addition: one addition, minimum and maximum an element, all of them to
    // the same three words, took 40 ns each, 60 us where the bins hold 1,500)
    uint32_t least = 0xffffffffu, most = 0u;
    const auto take = [&](const uint4 (&raw)[kLoads], uint32_t at) {
#pragma unroll
        for (uint32_t k = 0; k < kLoads; ++k)
        {
            const uint32_t bits[4] = {raw[k].x, raw[k].y, raw[k].z, raw[k].w};
            const uint32_t nearest = min(min(top - bits[0], top - bits[1]), min(top - bits[2], top - bits[3]));
            const uint32_t v = at + k * kWalkThreads;
            const bool some = nearest < width && v < vectors;
            if (__builtin_amdgcn_ballot_w64(some) == 0ull)
                continue;
            uint32_t own = 0;
#pragma unroll
            for (uint32_t c = 0; c < 4u; ++c)
                own += some && top - bits[c] < width ? 1u : 0u;
            const uint32_t through = wave_prefix_sum_u32(own);
            uint32_t place = 0;
            if (lane_id() == kWaveSize - 1)
                place = atomicAdd(&shared.extra_count, through);
            place = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(place), kWaveSize - 1)) + through - own;
#pragma unroll
            for (uint32_t c = 0; c < 4u; ++c)
            {
                if (some && top - bits[c] < width)
                {
                    least = min(least, bits[c]);
                    most = max(most, bits[c]);
                    if (place < kBinExtraCap)
                    {
                        shared.terms[kBinExtraPlace + place] = __uint_as_float(bits[c]);
                        shared.tokens[kBinExtraPlace + place] = v * 4u + c - misalignment;
                    }
                    ++place;
                }
            }
        }
    };
    {
        uint4 raw[kLoads], more[kLoads];
        load(raw, tid);
        for (uint32_t at = tid; same_in_all(at) < vectors; at += 2u * kStride) // (whole waves stay in the loop)
        {
            load(more, at + kStride);
            take(raw, at);
            load(raw, at + 2u * kStride);
            take(more, at + kStride);
        }
    }
    least = ~wave_max_u32(~least);
    most = wave_max_u32(most);
    if (lane_id() == 0 && most != 0u)
    {
        atomicMin(&shared.extra_least, least);
        atomicMax(&shared.extra_most, most);
    }
    __syncthreads();
    const uint32_t count = shared.extra_count;
    if (count <= kBinExtraCap)
    {
        constexpr uint32_t kPerThread = (kBinExtraCap + kWalkThreads - 1) / kWalkThreads;
        const uint32_t fineness = fineness_of(kBinExtraPlace, count);
        const float places_per_bit = static_cast<float>(fineness * count) / static_cast<float>(width);
        float own[kPerThread];
        uint32_t token[kPerThread], fine[kPerThread];
#pragma unroll
        for (uint32_t k = 0; k < kPerThread; ++k)
        {
            const uint32_t i = k * kWalkThreads + tid;
            own[k] = 1.0f;
            token[k] = fine[k] = 0u;
            if (i < count)
            {
                own[k] = shared.terms[kBinExtraPlace + i];
                token[k] = shared.tokens[kBinExtraPlace + i];
                // (rounded, but never falling where the term falls)
                fine[k] = min(static_cast<uint32_t>(static_cast<float>(top - __float_as_uint(own[k])) * places_per_bit), fineness * count - 1u);
            }
        }
        __syncthreads();
        order_elements<kPerThread>(shared, kBinExtraPlace, count, fineness, own, token, fine, tid);
    }
}

// The plain sum of each 64 of `count` terms (4096 at most): a row of 16 lanes holds 64 terms, a lane four of them.
template <int WAVES>
__device__ __forceinline__ void sum_chunks(HeadScratch& scratch, const float* terms, uint32_t count, int tid)
{
    for (uint32_t i = 4u * static_cast<uint32_t>(tid); same_in_all(i) < count; i += 4u * WAVES * kWaveSize)
    {
        const float4 own = *reinterpret_cast<const float4*>(terms + i);
        const float sum = row16_prefix_sum_f32(((i < count ? own.x : 0.0f) + (i + 1u < count ? own.y : 0.0f)) + ((i + 2u < count ? own.z : 0.0f) + (i + 3u < count ? own.w : 0.0f)));
        if ((tid & 15) == 15)
            scratch.chunk_sum[i / kWaveSize] = sum;
    }
    __syncthreads();
}

// What four terms a lane, 64 a row of 16 lanes, do to a sum of that exponent: the row's last lane has the whole of it.
__device__ __forceinline__ ParityStep row16_steps(const float (&terms)[4], int exponent)
{
    uint32_t sum = 0;
    bool differ = false; // a term half way between two sums
#pragma unroll
    for (int c = 0; c < 4; ++c)
    {
        // (as step_of_term, for zero and normal numbers: zero comes out as a step of zero)
        const uint32_t bits = __float_as_uint(terms[c]);
        const uint32_t mantissa = (bits & 0x7fffffu) | 0x800000u;
        const int difference = exponent - static_cast<int>(bits >> 23);
        const uint32_t shift = static_cast<uint32_t>(min(max(difference, 1), 25));
        const uint32_t half = 1u << (shift - 1u);
        differ = differ || ((mantissa & (2u * half - 1u)) == half && difference > 0);
        sum += difference > 0 ? (mantissa + half) >> shift : kBinadeFull;
    }
    if (__builtin_amdgcn_ballot_w64(differ) == 0ull)
    {
        // (64 steps of 2^24 at most)
        const uint32_t through = min(row16_prefix_sum_u32(sum), kStepCap);
        return ParityStep{through, through};
    }
    ParityStep steps[4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
        steps[c] = step_of_term(terms[c], exponent);
    ParityStep through = compose_steps(compose_steps(steps[0], steps[1]), compose_steps(steps[2], steps[3]));
#define NCNN_MOE_SCAN_STAGE(CONTROL) through = compose_steps(ParityStep{dpp_source<CONTROL, 0xf>(through.even), dpp_source<CONTROL, 0xf>(through.odd)}, through);
    NCNN_MOE_SCAN_STAGE(0x111)
    NCNN_MOE_SCAN_STAGE(0x112)
    NCNN_MOE_SCAN_STAGE(0x114)
    NCNN_MOE_SCAN_STAGE(0x118)
#undef NCNN_MOE_SCAN_STAGE
    return through;
}

// The sum of `count` terms in descending order (scratch.sum, scratch.stop), exactly as a sequential loop makes it; every thread calls it.  The waves work
// out what each 64 terms do to a sum of the exponent that it should have there (from sum_chunks), while the first wave adds the first
// terms in order; it then takes the chunks whose exponent was right in one scan and adds the terms of the others in order.
// What bounds it: dependent instructions of the first wave, some 530 cycles for 64 terms in order, 300 for each scan.  2,044 terms on 8
// waves, sums that leave one to three binades behind the first 64 terms: the normaliser's 2,500 to 5,300 cycles, the Top-P sum's 3,200 to
// 5,800, the draw's 3,500 to 5,200; with the first 256 terms in order at 12 cycles each, a chunk at a time a wave and scans of the terms'
// steps for a chunk in which the sum leaves its binade 7,000 to 10,400, 5,200 to 11,800 and 4,800 to 8,400.
template <int WAVES, int PHASE>
__device__ __forceinline__ void sum_head(HeadScratch& scratch, const float* terms, uint32_t count, int mode, float bound, float divisor, float second_divisor, int tid)
{
    constexpr uint32_t kInOrder = 2; // chunks added in order (four of them where there are no more: 3,000 to 3,800 cycles instead of 2,300 to 3,400)
    const int lane = tid & (kWaveSize - 1);
    const uint32_t wave = same_in_all(static_cast<uint32_t>(tid) >> 6);
    const uint32_t chunks = (count + kWaveSize - 1u) / kWaveSize;
    const auto scaled = [&](float t) {
        if (PHASE >= 1)
            t = t / divisor;
        if (PHASE >= 2)
            t = t / second_divisor;
        return t;
    };
    float sum = 0.0f;
    uint32_t stop = 0xffffffffu;
    if (wave == 0u)
    {
        // (its share would be the terms among which those half way are frequent)
        const WaveSum result = wave_add_in_order<PHASE>(terms, min(count, kInOrder * kWaveSize), sum, mode, bound, divisor, second_divisor, scratch.in_order);
        sum = result.sum;
        if (result.stopped)
            stop = result.index;
    }
    else
    {
        const float scale = PHASE == 0 ? 1.0f : PHASE == 1 ? 1.0f / divisor : 1.0f / (divisor * second_divisor);
        const float chunk_sum = static_cast<uint32_t>(lane) < chunks ? scratch.chunk_sum[lane] : 0.0f;
        const float chunk_front = wave_prefix_sum_f32(chunk_sum) - chunk_sum;
        for (uint32_t i = kInOrder * kWaveSize + 4u * static_cast<uint32_t>(tid - kWaveSize); same_in_all(i) < count; i += 4u * (WAVES - 1) * kWaveSize)
        {
            // (the last wave's lanes may lie behind the last chunk: those have no terms, and no place in the scratch)
            const float4 raw = *reinterpret_cast<const float4*>(terms + (i < count ? i : 0u));
            const float own[4] = {i < count ? scaled(raw.x) : 0.0f, i + 1u < count ? scaled(raw.y) : 0.0f, i + 2u < count ? scaled(raw.z) : 0.0f,
                                  i + 3u < count ? scaled(raw.w) : 0.0f};
            const uint32_t exponent = __float_as_uint(__shfl(chunk_front, static_cast<int>(i / kWaveSize), kWaveSize) * scale) >> 23;
            const ParityStep through = row16_steps(own, static_cast<int>(exponent));
            if ((tid & 15) == 15 && i / kWaveSize < chunks)
            {
                scratch.chunk_exponent[i / kWaveSize] = exponent;
                scratch.chunk_even[i / kWaveSize] = through.even;
                scratch.chunk_odd[i / kWaveSize] = through.odd;
            }
        }
    }
    __syncthreads();
    if (wave == 0u)
    {
        uint32_t c = kInOrder;
        uint32_t own_exponent = 0, own_even = 0, own_odd = 0;
        if (stop == 0xffffffffu && static_cast<uint32_t>(lane) < chunks && static_cast<uint32_t>(lane) >= kInOrder)
        {
            own_exponent = scratch.chunk_exponent[lane];
            own_even = scratch.chunk_even[lane];
            own_odd = scratch.chunk_odd[lane];
        }
        // (the chunks from c on that the sum runs through are consecutive: the steps up to each are one difference.  64 numbers of
        // 2^25 at most: what is past the binade is only compared against it)
        const uint32_t through = wave_prefix_sum_u32(min(own_even, 2u * kBinadeFull));
        while (c < chunks && stop == 0xffffffffu)
        {
            int exponent;
            uint32_t mantissa;
            decode_sum(sum, exponent, mantissa);
            const uint32_t goal = min(stop_mantissa(mode, bound, exponent), kBinadeFull);
            const uint32_t in_front = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(through), static_cast<int>(c - 1u)));
            const bool ahead = static_cast<uint32_t>(lane) >= c && static_cast<uint32_t>(lane) < chunks;
            const uint32_t behind = mantissa + (through - in_front);
            const uint64_t special = __builtin_amdgcn_ballot_w64(ahead && (own_exponent != static_cast<uint32_t>(exponent) || own_even != own_odd || behind >= goal));
            const uint32_t first_special = special != 0ull ? static_cast<uint32_t>(__builtin_ctzll(special)) : chunks;
            if (first_special > c)
                mantissa = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(behind), static_cast<int>(first_special - 1u)));
            c = first_special;
            sum = encode_sum(exponent, mantissa);
            if (c >= chunks)
                break;
            const uint32_t of_chunk = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>((mantissa & 1u) != 0u ? own_odd : own_even), static_cast<int>(c)));
            if (static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(own_exponent), static_cast<int>(c))) == static_cast<uint32_t>(exponent) &&
                mantissa + of_chunk < goal)
                sum = encode_sum(exponent, mantissa + of_chunk); // (a term half way between two sums among its terms)
            else
            {
                const uint32_t first = c * kWaveSize;
                const WaveSum result = wave_add_in_order<PHASE>(terms + first, min(count - first, static_cast<uint32_t>(kWaveSize)), sum, mode, bound, divisor, second_divisor, scratch.in_order);
                sum = result.sum;
                if (result.stopped)
                    stop = first + result.index;
            }
            ++c;
        }
        if (lane == 0)
        {
            scratch.sum = sum;
            scratch.stop = stop;
        }
    }
    __syncthreads();
}

// The walk over the bins behind the head, from `sum` on: every thread calls it; the first wave walks, the workgroup
// fetches what it asks for.  Ends with shared.status 1 (ended: sum, stopped, ...) or 2 (given up).
//   limit     elements that the sum runs over at most; cut_bin, cut_term: it ends at the first term below cut_term,
//             which lies in that bin (kBins: nowhere)
template <int PHASE, bool CHAINED>
__device__ __forceinline__ void walk_bins(
    BinWalkShared& shared, uint32_t stops, const float* row_terms, uint32_t positions, uint32_t misalignment, uint32_t shift, uint32_t head_bins, uint32_t wide_first,
    uint32_t limit, uint32_t cut_bin, float cut_term, float start_sum, int mode, float bound, float divisor, float second_divisor, int tid)
{
    uint32_t cur = head_bins;
    uint32_t stop = 0;
    float sum = start_sum;
    bool fetched = false;
    bool unforeseen = false; // the sum goes on behind the end that was foreseen: every bin from here on is fetched
    const auto front_of = [&shared](uint32_t bin) { return packed_front(shared.packed[bin]); };
    for (uint32_t requests = 0;; ++requests)
    {
        if (tid < kWaveSize)
        {
            uint32_t status = 3u;
            const auto finish = [&](uint32_t outcome) {
                status = outcome;
                shared.status = outcome;
                shared.sum = sum;
            };
            // of `count` elements from `place` on, of bins [bin, last_bin]: how many the sum takes
            const auto share_of_sum = [&](uint32_t bin, uint32_t last_bin, uint32_t place, uint32_t count) {
                uint32_t take = min(count, limit - min(limit, front_of(bin)));
                if (cut_bin >= bin && cut_bin <= last_bin)
                {
                    const float* elements = shared.terms + place;
                    take = min(take, wave_partition_point(count, [elements, cut_term](uint32_t i) { return elements[i] >= cut_term; }));
                }
                return take;
            };
            const auto end_at = [&](uint32_t taken) {
                shared.stopped = 0u;
                shared.taken = taken;
                finish(1u);
            };
            const auto stopped_at = [&](uint32_t rank, uint32_t place) {
                shared.stopped = 1u;
                shared.stop_rank = rank;
                shared.stop_at = place;
                finish(1u);
            };
            // every term of the bin, and of those behind it, is below half an ulp of the sum: none moves it
            const auto moves_nothing = [&](uint32_t bin) {
                float top = bin_top(bin, shift);
                if (PHASE >= 1)
                    top = top / divisor;
                if (PHASE >= 2)
                    top = top / second_divisor;
                return top < __uint_as_float((max(__float_as_uint(sum) >> 23, 25u) - 24u) << 23);
            };
            const auto ask_for = [&](uint32_t low, uint32_t high) {
                shared.low = low;
                shared.high = high;
                finish(requests < kBinRequests ? 0u : 2u);
            };
            // as many bins in front of `end` as can be fetched at a time
            const auto ask_for_most = [&](uint32_t low, uint32_t end) {
                const uint32_t front = front_of(low);
                const uint32_t more = wave_partition_point(end - low, [&shared, low, front](uint32_t i) {
                    return packed_front(shared.packed[low + i + 1u]) - front <= kBinExtraCap;
                });
                ask_for(low, low + max(more, 1u) - 1u);
            };
            if (fetched)
            {
                const uint32_t low = shared.low, high = shared.high, count = shared.extra_count;
                const uint32_t front = front_of(low);
                fetched = false;
                if (count > kBinExtraCap && shared.extra_least != shared.extra_most)
                    finish(2u);
                else
                {
                    uint32_t take;
                    WaveSum result;
                    if (count > kBinExtraCap)
                    {
                        // thousands of equal terms
                        const float term = __uint_as_float(shared.extra_least);
                        take = min(count, limit - min(limit, front));
                        take = cut_bin >= low && cut_bin <= high && term < cut_term ? 0u : take;
                        result = wave_add_repeated<PHASE>(term, take, sum, mode, bound, divisor, second_divisor);
                    }
                    else
                    {
                        take = share_of_sum(low, high, kBinExtraPlace, count);
                        result = wave_add_in_order<PHASE>(shared.terms + kBinExtraPlace, take, sum, mode, bound, divisor, second_divisor, shared.head.in_order);
                    }
                    sum = result.sum;
                    if (result.stopped)
                        stopped_at(front + result.index, count > kBinExtraCap ? 0xffffffffu : kBinExtraPlace + result.index);
                    else if (take < count)
                        end_at(front + take);
                    cur = high + 1u;
                    while ((shared.stop_bin[stop] & kStopBin) <= high)
                        ++stop;
                }
            }
            while (status == 3u)
            {
                // (the end, unless there is more to run over and the exact sum has not met its stop condition)
                unforeseen = unforeseen || packed_kind(shared.packed[cur]) == kBinBeyond;
                if (unforeseen)
                {
                    const uint32_t front = front_of(cur);
                    if (cur > cut_bin || front >= limit || front == front_of(kBins))
                        end_at(min(limit, front));
                    else if (!moves_nothing(cur))
                        ask_for_most(cur, min(cut_bin + 1u, kBins));
                    else if (cut_bin < kBins && front_of(cut_bin) < limit)
                        ask_for(cut_bin, cut_bin); // (the elements behind this one move nothing, but are counted up to the cut)
                    else
                        end_at(min(limit, front_of(kBins)));
                    continue;
                }
                const uint32_t stop_word = shared.stop_bin[stop];
                const uint32_t stop_here = stop_word & kStopBin;
                if (cur < stop_here)
                {
                    // bins that are one integer each
                    const uint32_t front = front_of(cur);
                    const uint32_t front_prefix = shared.prefix[cur];
                    if (front_of(stop_here) == front)
                    {
                        cur = stop_here;
                        continue;
                    }
                    int exponent;
                    uint32_t mantissa;
                    decode_sum(sum, exponent, mantissa);
                    const uint32_t goal = min(stop_mantissa(mode, bound, exponent), kBinadeFull);
                    if (packed_exponent(shared.packed[cur]) == static_cast<uint32_t>(exponent))
                    {
                        const uint32_t total = shared.prefix[stop_here] - front_prefix;
                        if (mantissa + total < goal && total < kBinadeFull)
                        {
                            sum = encode_sum(exponent, mantissa + total);
                            cur = stop_here;
                            continue;
                        }
                        const uint32_t first = cur;
                        const uint32_t* prefix = shared.prefix;
                        const uint32_t good = wave_partition_point(stop_here - cur, [prefix, first, front_prefix, mantissa, goal](uint32_t i) {
                            const uint32_t through = prefix[first + i + 1u] - front_prefix;
                            return through < kBinadeFull && mantissa + through < goal;
                        });
                        if (good > 0u)
                            sum = encode_sum(exponent, mantissa + (shared.prefix[cur + good] - front_prefix));
                        cur += good;
                        ask_for(cur, cur);
                    }
                    else if (moves_nothing(cur))
                        cur = stop_here;
                    else
                    {
                        // the sum has another exponent than was foreseen
                        ask_for_most(cur, stop_here);
                    }
                }
                else if ((stop_word & kStopExponent) != 0u)
                    ++stop; // (a new exponent from this bin on)
                else if (packed_kind(shared.packed[stop_here]) != kBinListed)
                {
                    // terms half way: their roundings follow from the masks, unless the sum has another exponent than was
                    // foreseen or leaves its binade (or stops) in this bin
                    const uint32_t place = shared.places[stop_here];
                    int exponent;
                    uint32_t mantissa;
                    decode_sum(sum, exponent, mantissa);
                    const uint32_t goal = min(stop_mantissa(mode, bound, exponent), kBinadeFull);
                    bool known = (place & kHasMasks) != 0u && packed_exponent(shared.packed[stop_here]) == static_cast<uint32_t>(exponent);
                    if (known)
                    {
                        const uint32_t total = shared.prefix[stop_here + 1u] - shared.prefix[stop_here];
                        const uint32_t* const masks = shared.bin_masks + kWideWords * (place & ~kHasMasks);
                        const bool wide = stop_here - wide_first < kWideBins;
                        float top = bin_top(stop_here, shift);
                        if (PHASE >= 1)
                            top = top / divisor;
                        if (PHASE >= 2)
                            top = top / second_divisor;
                        known = exponent - static_cast<int>(__float_as_uint(top) >> 23) >= (wide ? kWideDifference : kMaskedDifference);
                        const uint32_t highest = step_of_term(top, exponent).odd + 1u;
                        uint32_t parity = mantissa, less = 0, odd_in_front = 0;
                        // lane l: the terms of step highest - l, and the value half way between that step and the one below
                        // (a wide bin's: 64 steps, then those behind them)
                        constexpr uint32_t kSteps = 24, kWideSteps = 80;
                        for (uint32_t first = 0; first < (wide ? kWideSteps : kSteps); first += kWaveSize)
                        {
                            const uint32_t number = first + static_cast<uint32_t>(lane_id());
                            const uint32_t step = highest - number, half = step - 1u;
                            const bool in_range = number < (wide ? kWideSteps : kSteps);
                            const uint32_t parities = masks[wide ? (step >> 6) % kWideParities : 0u];
                            const uint32_t halves = masks[kWideParities + (wide ? (half >> 5) % kWideHalves : 0u)];
                            const uint64_t odd_steps = __builtin_amdgcn_ballot_w64(in_range && (step & 1u) != 0u && (parities >> ((step >> 1) & 31u) & 1u) != 0u);
                            uint64_t half_way = __builtin_amdgcn_ballot_w64(in_range && (halves >> (half & 31u) & 1u) != 0u);
                            while (half_way != 0ull)
                            {
                                const uint32_t l = static_cast<uint32_t>(__builtin_ctzll(half_way));
                                half_way &= half_way - 1ull;
                                const uint32_t below = highest - first - l - 1u; // the value lies half way between this step and the next
                                const uint32_t in_front = odd_in_front + static_cast<uint32_t>(__popcll(odd_steps & ((2ull << l) - 1ull)));
                                const uint32_t up = (parity + in_front + below) & 1u; // to the even neighbour
                                parity += below + up;
                                less += 1u - up;
                            }
                            odd_in_front += static_cast<uint32_t>(__popcll(odd_steps));
                        }
                        known = known && total < kBinadeFull && mantissa + total < goal;
                        if (known)
                        {
                            sum = encode_sum(exponent, mantissa + total - less);
                            cur = stop_here + 1u;
                            ++stop;
                        }
                    }
                    if (!known)
                        ask_for(stop_here, stop_here);
                }
                else
                {
                    const uint32_t place = shared.places[stop_here];
                    const uint32_t front = front_of(stop_here);
                    // Listed bins one behind the other lie side by side in the list and are added together: in the last binades
                    // of a sum, and in short rows, 100 bins and more of a few elements each are listed, at 1 us a bin (64 rows
                    // of 4,096 without a window: 261 us so, 72 us together).  They end where elements are not in the list.
                    uint32_t behind = stop_here + 1u;
                    if ((stop_word & kStopRun) != 0u)
                    {
                        const uint32_t first = behind + 1u;
                        behind += wave_partition_point(kBins - behind, [&shared, first, place, front](uint32_t i) {
                            return shared.places[first + i] - place == packed_front(shared.packed[first + i]) - front;
                        });
                    }
                    const uint32_t count = front_of(behind) - front;
                    const uint32_t take = share_of_sum(stop_here, behind - 1u, place, count);
                    const WaveSum result = wave_add_in_order<PHASE>(shared.terms + place, take, sum, mode, bound, divisor, second_divisor, shared.head.in_order);
                    sum = result.sum;
                    if (result.stopped)
                        stopped_at(front + result.index, place + result.index);
                    else if (take < count)
                        end_at(front + take);
                    cur = behind;
                    ++stop;
                    if ((stop_word & kStopRun) != 0u)
                        stop += wave_partition_point(stops - stop, [&shared, stop, behind](uint32_t i) { return (shared.stop_bin[stop + i] & kStopBin) < behind; });
                }
            }
        }
        __syncthreads();
        if (shared.status != 0u)
            return;
        fetch_bins<CHAINED>(row_terms, positions, misalignment, shift, shared, tid);
        fetched = true;
    }
}

// The token of the rank-th (from 0) of the row's elements whose term is `term`, in the row's order: for a stretch of thousands
// of equal terms, which no list holds.  Their logits are equal too, or a few neighbouring values: the logit is found by
// bisection of the keys, then its rank-th index, each by a pass over the row's terms (8 us of one compute unit for 151,936).
template <int DTYPE>
__device__ __noinline__ int32_t token_of_equal(
    const SamplerArgs& a, uint32_t row, BinWalkShared& shared, const float* terms, uint32_t positions, uint32_t misalignment, float term, uint32_t rank, int tid)
{
    const char* pointer = static_cast<const char*>(a.logits) + static_cast<size_t>(row) * a.row_stride * LogitsVector<DTYPE>::kElementBytes;
    const uint32_t wanted = __float_as_uint(term);
    const uint32_t vectors = positions / 4u;
    const int lane = tid & (kWaveSize - 1);
    const uint32_t wave = same_in_all(static_cast<uint32_t>(tid) >> 6);
    const auto key_of = [&](uint32_t v, uint32_t c) { return descending_key(load_logit<DTYPE>(pointer, v * 4u + c - misalignment)); };
    // which of a vector's four elements match: the term, and the key where [least, most] is given
    const auto matching = [&](uint32_t v, bool by_key, uint32_t least, uint32_t most) {
        const uint4 raw = taken_over_vector<true>(terms, positions * 4u, v);
        uint32_t hits = (raw.x == wanted ? 1u : 0u) | (raw.y == wanted ? 2u : 0u) | (raw.z == wanted ? 4u : 0u) | (raw.w == wanted ? 8u : 0u);
        if (by_key)
        {
            for (uint32_t c = 0; c < 4u; ++c)
            {
                if ((hits >> c & 1u) != 0u)
                {
                    const uint32_t key = key_of(v, c);
                    hits &= ~(key < least || key > most ? 1u << c : 0u);
                }
            }
        }
        return hits;
    };
    __syncthreads();
    if (tid == 0)
    {
        shared.least_key = 0xffffffffu;
        shared.most_key = 0u;
    }
    __syncthreads();
    {
        uint32_t least = 0xffffffffu, most = 0u;
        for (uint32_t v = tid; v < vectors; v += kWalkThreads)
        {
            const uint32_t hits = matching(v, false, 0u, 0u);
            for (uint32_t c = 0; c < 4u; ++c)
            {
                if ((hits >> c & 1u) != 0u)
                {
                    const uint32_t key = key_of(v, c);
                    least = min(least, key);
                    most = max(most, key);
                }
            }
        }
        least = ~wave_max_u32(~least);
        most = wave_max_u32(most);
        if (lane == 0)
        {
            atomicMin(&shared.least_key, least);
            atomicMax(&shared.most_key, most);
        }
    }
    __syncthreads();
    uint32_t low = same_in_all(shared.least_key), high = same_in_all(shared.most_key);
    const uint32_t first_key = low;
    const bool by_key = low != high;
    while (low < high)
    {
        const uint32_t middle = low + (high - low) / 2u;
        __syncthreads();
        if (tid == 0)
            shared.matches = 0u;
        __syncthreads();
        uint32_t own = 0;
        for (uint32_t v = tid; v < vectors; v += kWalkThreads)
            own += static_cast<uint32_t>(__popc(matching(v, true, first_key, middle)));
        const uint32_t of_wave = wave_prefix_sum_u32(own);
        if (lane == kWaveSize - 1)
            atomicAdd(&shared.matches, of_wave);
        __syncthreads();
        const uint32_t through = same_in_all(shared.matches);
        if (through > rank)
            high = middle;
        else
            low = middle + 1u;
    }
    // ---- the elements of that key by index: those of smaller keys are counted off with them
    const uint32_t of_wave = ((vectors + kWalkWaves - 1u) / kWalkWaves + kWaveSize - 1u) / kWaveSize * kWaveSize;
    const uint32_t first = min(vectors, wave * of_wave), last = min(vectors, first + of_wave);
    uint32_t smaller = 0, own = 0;
    for (uint32_t v = first + lane; v < last; v += kWaveSize)
    {
        own += static_cast<uint32_t>(__popc(matching(v, by_key, low, low)));
        if (low != first_key)
            smaller += static_cast<uint32_t>(__popc(matching(v, true, first_key, low - 1u)));
    }
    const uint32_t own_of_wave = wave_prefix_sum_u32(own), smaller_of_wave = wave_prefix_sum_u32(smaller);
    __syncthreads();
    if (lane == kWaveSize - 1)
    {
        shared.scan.u[0][wave] = own_of_wave;
        shared.scan.u[1][wave] = smaller_of_wave;
    }
    __syncthreads();
    uint32_t before = 0, below = 0;
    for (uint32_t w = 0; w < static_cast<uint32_t>(kWalkWaves); ++w)
    {
        before += w < wave ? shared.scan.u[0][w] : 0u;
        below += shared.scan.u[1][w];
    }
    const uint32_t index = rank - below;
    const uint32_t in_wave = shared.scan.u[0][wave];
    if (index >= before && index - before < in_wave)
    {
        uint32_t count = before;
        for (uint32_t base = first; base < last; base += kWaveSize)
        {
            const uint32_t v = base + lane;
            const uint32_t hits = v < last ? matching(v, by_key, low, low) : 0u;
            const uint32_t held = static_cast<uint32_t>(__popc(hits));
            const uint32_t through = wave_prefix_sum_u32(held);
            uint32_t at = count + through - held;
            for (uint32_t c = 0; c < 4u; ++c)
            {
                if ((hits >> c & 1u) != 0u)
                {
                    if (at == index)
                        shared.token = static_cast<int32_t>(v * 4u + c - misalignment);
                    ++at;
                }
            }
            count += static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(through), kWaveSize - 1));
            if (count > index)
                break;
        }
    }
    __syncthreads();
    const int32_t token = same_in_all(static_cast<uint32_t>(shared.token));
    __syncthreads();
    return token;
}

// The token of the element at terms[at] of a list [list_first, list_end) in order, which holds all elements of its term: those
// are in no particular order, and are told apart by their logits and indices, each against each while they are few (2,000
// of them took 500 us so).
template <int DTYPE>
__device__ __forceinline__ int32_t token_of_listed(
    const SamplerArgs& a, uint32_t row, BinWalkShared& shared, const float* row_terms, uint32_t positions, uint32_t misalignment, const uint32_t* tokens,
    uint32_t at, uint32_t list_first, uint32_t list_end, int tid)
{
    const float term = shared.terms[at];
    const float* terms = shared.terms;
    const uint32_t low = list_first + wave_partition_point(at - list_first, [terms, list_first, term](uint32_t i) { return terms[list_first + i] > term; });
    const uint32_t high = at + 1u + wave_partition_point(list_end - at - 1u, [terms, at, term](uint32_t i) { return terms[at + 1u + i] >= term; });
    if (high - low == 1u)
        return static_cast<int32_t>(tokens[at]);
    if (high - low > kBinComparedTies)
        return token_of_equal<DTYPE>(a, row, shared, row_terms, positions, misalignment, same_in_all(term), same_in_all(at - low), tid);
    const char* pointer = static_cast<const char*>(a.logits) + static_cast<size_t>(row) * a.row_stride * LogitsVector<DTYPE>::kElementBytes;
    uint32_t* const keys = shared.packed; // (where the bins' words were)
    static_assert(kBinComparedTies <= kBins, "the keys fit");
    __syncthreads();
    for (uint32_t i = low + tid; i < high; i += kWalkThreads)
        keys[i - low] = descending_key(load_logit<DTYPE>(pointer, tokens[i]));
    __syncthreads();
    for (uint32_t i = low + tid; i < high; i += kWalkThreads)
    {
        const uint32_t token = tokens[i];
        const uint32_t key = keys[i - low];
        uint32_t rank = 0;
        for (uint32_t j = low; j < high; ++j)
        {
            const uint32_t other = keys[j - low];
            rank += other < key || (other == key && tokens[j] < token) ? 1u : 0u;
        }
        if (rank == at - low)
            shared.token = static_cast<int32_t>(token);
    }
    __syncthreads();
    const int32_t token = shared.token;
    __syncthreads();
    return token;
}

// ---- (4): walk 0 walks the normaliser and, inside the head, the Top-P sum and the draw, walk 1 the Top-P sum
// behind the head (and the draw inside it), walk 2 the draw behind the head.  Walks 0 and 1 then have the bins' steps of the next
// sum added for the calling part of the row, unless the row is finished.  Every part of a row walks for itself.
// CHAINED: a walk of bin_chain_kernel, which has written what the first one reads and has a compute unit to itself.

__device__ __forceinline__ uint8_t flags_of_row(const BinArgs& g, const ncnn_moe_sample_params& p, uint32_t saw_nan)
{
    return static_cast<uint8_t>((counts_as_select(g.windows_are_selects, g.a.vocab, p) ? 0u : static_cast<uint32_t>(NCNN_MOE_ROW_FLAG_GENERAL_PATH)) |
                                (saw_nan != 0u ? static_cast<uint32_t>(NCNN_MOE_ROW_FLAG_HAS_NAN) : 0u));
}

// A row that is finished, or not served, before its first walk.
__device__ __forceinline__ void end_early(const BinArgs& g, uint32_t part, uint32_t row, const ncnn_moe_sample_params& p, uint32_t state, uint32_t saw_nan, int tid)
{
    if (state == kBinRowRejected && part == 0u && tid == 0)
    {
        write_error(g.a, row, NCNN_MOE_ROW_NO_FINITE_LOGIT, flags_of_row(g, p, saw_nan));
        g.a.row_state[row] = kRowDoneLater;
    }
}

enum BinWalkOutcome : uint32_t
{
    kBinWalkEnds = 0,  // the row is finished, or left to the full-order kernels
    kBinWalkGoesOn = 1 // the next walk goes on with it
};

template <int DTYPE, int WALK, bool CHAINED>
__device__ __forceinline__ BinWalkOutcome bin_walk(const BinArgs& g, const BinGrid& grid, uint32_t slot, uint32_t row, bool near, BinWalkShared& shared, uint4& words_of_thread, int tid)
{
    constexpr int kFrom = WALK & 1;      // which of the alternating buffers this walk reads
    constexpr int kTo = kFrom ^ 1;
    constexpr bool kAcross = WALK > 0 || CHAINED; // ... and whether this launch has written it
    const SamplerArgs& a = g.a;
    const uint32_t bin = 4u * static_cast<uint32_t>(tid);
    const bool holds_bins = tid < static_cast<int>(kBinQuads);
    BinRow& record = g.records[row];
    BinWalkRow& carried = shared.row;
    const auto result_flags = [&](const ncnn_moe_sample_params& p) { return flags_of_row(g, p, carried.saw_nan); };
    {
        __syncthreads(); // (a row before this one: its last readers of shared are done)
        if (tid < static_cast<int>(2u * kBinWords))
            shared.ties[tid] = 0u;
        if (tid == 0)
            shared.any_ties = 0u;
        __syncthreads();
        const float top_p = same_in_all(params_of(carried.options).top_p);
        const float min_p = same_in_all(params_of(carried.options).min_p);
        const float uniform = __uint_as_float(same_in_all(carried.options[kParamsWords]));
        const uint32_t shift = same_in_all(carried.shift);
        const uint32_t window = same_in_all(carried.window);
        const uint32_t binned = same_in_all(carried.binned);
        const uint32_t head_bins = same_in_all(carried.head_bins);
        const uint32_t head_count = same_in_all(carried.head_count);
        const uint32_t listed = same_in_all(carried.listed);
        const uint32_t wide_first = same_in_all(carried.wide_first);
        const uint32_t limit = WALK == 0 ? window : same_in_all(carried.limit);
        const uint32_t cut_bin = WALK == 1 ? same_in_all(carried.cut_bin) : kBins;
        const float cut_term = WALK == 1 ? same_in_all(carried.cut_term) : 0.0f;
        uint32_t cut_in_tail = WALK == 1 ? same_in_all(carried.cut_in_tail) : 0u;
        const bool behind_head = limit > head_count && binned > head_count; // this launch's own sum goes on behind the head
        float normalizer = WALK == 0 ? 1.0f : same_in_all(carried.normalizer);
        float renormalizer = WALK == 2 ? same_in_all(carried.renormalizer) : 1.0f;
        const float sum_so_far = WALK == 0 ? 0.0f : same_in_all(carried.head_sum);
        uint32_t kept = WALK == 2 ? same_in_all(carried.kept) : 0u;
        const BinStretch s = bin_stretch<LogitsVector<DTYPE>::kElementBytes>(a, row, grid.part, grid.parts);
        const uint32_t positions = (s.end + 7u) / 8u * 8u;
        const float* row_terms = bin_terms(a, row);
        // (the sorted head's terms stay in LDS; its tokens make room there for the steps of the next sum, and the first part alone
        // looks at them again)
        uint32_t* const sorted_tokens_out = g.head_tokens + static_cast<size_t>(row) * kBinListCap;

        // ---- the list, the bins and their steps.  The head is ordered by walk 0, and no longer needed by walk 2.
        constexpr uint32_t kPerThread = kBinListCap / kWalkThreads;
        const uint32_t list_first = WALK == 0 ? 0u : head_count;
        float own_terms[kPerThread];
        uint32_t own_tokens[kPerThread];
        {
            const float* from_terms = g.list_terms[kFrom] + static_cast<size_t>(row) * kBinListCap;
            const uint32_t* from_tokens = g.list_tokens[kFrom] + static_cast<size_t>(row) * kBinListCap;
#pragma unroll
            for (uint32_t k = 0; k < kPerThread; ++k)
            {
                const uint32_t i = list_first + k * kWalkThreads + tid;
                own_terms[k] = 0.0f;
                own_tokens[k] = 0u;
                if (list_first + k * kWalkThreads < listed)
                {
                    own_terms[k] = __uint_as_float(taken_over<kAcross>(from_terms, listed * 4u, i));
                    own_tokens[k] = taken_over<kAcross>(from_tokens, listed * 4u, i);
                }
            }
        }
        const uint4 words = words_of_thread;
        uint32_t own_steps[4] = {0u, 0u, 0u, 0u};
        uint32_t tie_word = 0, untold_word = 0;
        const uint32_t tie_lane = static_cast<uint32_t>(tid) & (kWaveSize - 1);
        if (behind_head)
        {
            const size_t first_pair = slot * grid.parts;
            // (every wave collects the words of some parts' bins with terms half way: by one wave, a part behind the other, they
            // arrived 2 us after everything else.  Asked for in front of the steps, whose loads are waited for one by one)
            constexpr uint32_t kEach = kMaxBinParts / kWalkWaves;
            static_assert(kMaxBinParts % kWalkWaves == 0, "as many parts for each wave");
            uint32_t words_of_part[kEach][3];
#pragma unroll
            for (uint32_t k = 0; k < kEach; ++k)
            {
                const uint32_t q = same_in_all(static_cast<uint32_t>(tid) / kWaveSize) + k * kWalkWaves;
#pragma unroll
                for (uint32_t w = 0; w < 3u; ++w)
                    words_of_part[k][w] = taken_over<kAcross>(g.ties[kFrom] + first_pair * 3u * kBinWords, grid.parts * 3u * kBinWords * 4u, (q * 3u + w) * kBinWords + tie_lane);
            }
            if (holds_bins && bin + 3u >= head_bins)
            {
                uint32_t* const from = g.steps[kFrom] + first_pair * kBins;
                const uint32_t bytes = grid.parts * kBins * 4u;
                constexpr uint32_t kTogether = CHAINED ? kMaxBinParts : kPartsAtATime;
                for (uint32_t first = 0; first < grid.parts; first += kTogether)
                {
                    uint4 of_part[kTogether];
#pragma unroll
                    for (uint32_t k = 0; k < kTogether; ++k)
                        of_part[k] = taken_over_vector<kAcross>(from, bytes, min(first + k, grid.parts - 1u) * kBinQuads + static_cast<uint32_t>(tid));
#pragma unroll
                    for (uint32_t k = 0; k < kTogether; ++k)
                    {
                        const uint32_t some = first + k < grid.parts ? 0xffffffffu : 0u;
                        own_steps[0] += of_part[k].x & some, own_steps[1] += of_part[k].y & some;
                        own_steps[2] += of_part[k].z & some, own_steps[3] += of_part[k].w & some;
                    }
                }
            }
            if (tie_lane < kBinWords)
            {
#pragma unroll
                for (uint32_t k = 0; k < kEach; ++k)
                {
                    tie_word |= words_of_part[k][0];
                    untold_word |= words_of_part[k][1] | words_of_part[k][2];
                }
            }
        }
        static_assert(kBinWords <= kWaveSize, "a word a lane");
        if (holds_bins)
            *reinterpret_cast<uint4*>(shared.packed + bin) = words;
        if (tie_word != 0u)
        {
            atomicOr(&shared.ties[tie_lane], tie_word);
            shared.any_ties = 1u;
        }
        if (untold_word != 0u)
            atomicOr(&shared.ties[kBinWords + tie_lane], untold_word);
        if (tid == 0)
            shared.mask_count = 0u;
        if (tid < 4)
            shared.packed[kBins + tid] = (kBinBeyond << 30) | binned;
        __syncthreads();
        // ---- stops: bins that the walk looks into, and bins from which on another exponent was assumed
        uint32_t front[5];
        float mass[5]; // about what the sum holds in front of each bin, behind the head (in the sum's own units)
        uint32_t stops;
        {
            const uint32_t packed[4] = {words.x, words.y, words.z, words.w};
            uint32_t kind[4];
            float own_mass[4];
            uint32_t stop_word[4];
            uint32_t sums[3] = {0u, 0u, 0u}; // steps added, elements listed, stops and (above them) steps in coarse units
            float masses = 0.0f;
            const float scale = 1.0f / (normalizer * renormalizer);
            const uint32_t tie_bits = holds_bins ? shared.ties[bin >> 5] >> (bin & 31u) : 0u;
            const uint32_t untold_bits = holds_bins ? shared.ties[kBinWords + (bin >> 5)] >> (bin & 31u) : 0u;
            // The bins whose terms half way the masks tell: their masks, from every part.  They lie anywhere among the bins, so
            // they are listed first and 16 lanes take the parts of each (a thread that went through its bins' parts one after
            // the other took 3 us a bin; 8 x 151,936 without a window: 148 us then, 135 us so).
            if (behind_head && same_in_all(shared.any_ties) != 0u)
            {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    if (holds_bins && bin + j >= head_bins && packed_kind(packed[j]) == kBinAdded && (tie_bits >> j & 1u) != 0u && (untold_bits >> j & 1u) == 0u)
                    {
                        const uint32_t i = atomicAdd(&shared.mask_count, 1u);
                        if (i < kBinMasks)
                        {
                            shared.mask_bin[i] = static_cast<uint16_t>(bin + j);
                            shared.places[bin + j] = static_cast<uint16_t>(i);
                        }
                        else
                            shared.places[bin + j] = static_cast<uint16_t>(kBinMasks);
                    }
                }
                __syncthreads();
                const uint32_t part = static_cast<uint32_t>(tid) & (kMaxBinParts - 1u);
                const uint32_t mask_count = min(shared.mask_count, kBinMasks);
                for (uint32_t i = static_cast<uint32_t>(tid) / kMaxBinParts; i < mask_count; i += kWalkThreads / kMaxBinParts)
                {
                    const uint32_t* const of_parts = g.masks[kFrom] + static_cast<size_t>(slot * grid.parts) * kMaskWords;
                    const uint32_t bytes = grid.parts * kMaskWords * 4u; // (a part that there is not, and a word that there is not: zero)
                    const uint32_t mask_bin = shared.mask_bin[i];
                    const bool wide = mask_bin - wide_first < kWideBins;
                    uint32_t words_of_bin[kWideWords];
#pragma unroll
                    for (uint32_t w = 0; w < kWideWords; ++w)
                    {
                        const uint32_t narrow = w == 0u ? mask_bin : w == kWideParities ? kBins + mask_bin : bytes;
                        words_of_bin[w] = taken_over<kAcross>(of_parts, bytes, part * kMaskWords + (wide ? 2u * kBins + (mask_bin - wide_first) * kWideWords + w : narrow));
                    }
                    uint32_t twice = 0u;
#pragma unroll
                    for (int distance = 1; distance < static_cast<int>(kMaxBinParts); distance *= 2)
                    {
                        twice |= __shfl_xor(twice, distance, kMaxBinParts);
#pragma unroll
                        for (uint32_t w = 0; w < kWideWords; ++w)
                        {
                            const uint32_t others = __shfl_xor(words_of_bin[w], distance, kMaxBinParts);
                            if (w >= kWideParities)
                                twice |= words_of_bin[w] & others;
                            words_of_bin[w] = w < kWideParities ? words_of_bin[w] ^ others : words_of_bin[w] | others;
                        }
                    }
                    if (part == 0u)
                    {
                        // (a value half way that two parts have seen is there twice, which a mask cannot tell)
                        if (twice != 0u)
                            shared.mask_bin[i] = static_cast<uint16_t>(kBins);
#pragma unroll
                        for (uint32_t w = 0; w < kWideWords; ++w)
                            shared.bin_masks[kWideWords * i + w] = words_of_bin[w];
                    }
                }
                __syncthreads();
            }
            const auto masks_of = [&](int j, uint32_t b, uint32_t kind_here, uint32_t packed_here, bool behind) {
                if (!(behind && kind_here == kBinWanted && packed_kind(packed_here) == kBinAdded && (untold_bits >> j & 1u) == 0u))
                    return 0u;
                const uint32_t i = shared.places[b];
                return i < kBinMasks && shared.mask_bin[i] == b ? kHasMasks | i : 0u;
            };
            uint32_t masked[4];
            uint32_t previous = holds_bins && bin > head_bins ? shared.packed[bin - 1u] : packed[0];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                front[j] = packed_front(packed[j]);
            uint4 next{0u, 0u, 0u, 0u};
            if (holds_bins)
                next = *reinterpret_cast<const uint4*>(shared.packed + bin + 4u);
            front[4] = packed_front(next.x);
            // (which of this thread's bins and the three behind them are listed)
            const uint32_t kinds[7] = {packed_kind(words.x), packed_kind(words.y), packed_kind(words.z), packed_kind(words.w),
                                       packed_kind(next.x), packed_kind(next.y), packed_kind(next.z)};
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                const uint32_t b = bin + j;
                const uint32_t count = front[j + 1] - front[j];
                const bool behind = holds_bins && b >= head_bins;
                if (b <= head_bins)
                    previous = packed[j];
                kind[j] = packed_kind(packed[j]);
                if (kind[j] == kBinAdded && (tie_bits >> j & 1u) != 0u)
                    kind[j] = kBinWanted;
                const bool ends = behind && kind[j] == kBinBeyond && (b == head_bins || packed_kind(previous) != kBinBeyond);
                const bool looks = behind && (kind[j] == kBinListed || kind[j] == kBinWanted);
                const bool changes = behind && kind[j] != kBinBeyond && packed_exponent(previous) != packed_exponent(packed[j]);
                const bool run = kinds[j] == kBinListed && kinds[j + 1] == kBinListed && kinds[j + 2] == kBinListed && kinds[j + 3] == kBinListed;
                stop_word[j] = ends || looks ? (run ? b | kStopRun : b) : changes ? (b | kStopExponent) : 0xffffffffu;
                masked[j] = masks_of(j, b, kind[j], packed[j], behind);
                const bool adds = behind && (kind[j] == kBinAdded || masked[j] != 0u);
                own_steps[j] = adds ? own_steps[j] : 0u;
                own_mass[j] = adds ? static_cast<float>(own_steps[j]) * __uint_as_float((max(packed_exponent(packed[j]), 24u) - 23u) << 23)
                    : looks ? static_cast<float>(count) * bin_top(b, shift) * (1.0f - 0.4f / kBinsPerBinade) * scale : 0.0f;
                sums[0] += own_steps[j];
                sums[1] += behind && kind[j] == kBinListed ? count : 0u;
                sums[2] += (stop_word[j] != 0xffffffffu ? 1u : 0u) + (own_steps[j] >> kBinStepUnit << kBinStopBits);
                masses += own_mass[j];
                previous = packed[j];
            }
            uint32_t totals[3];
            bin_scan<kWalkWaves>(sums, totals, masses, shared.scan, tid);
            const uint32_t all_stops = totals[2] & ((1u << kBinStopBits) - 1u);
            const bool overflows = kBinStops <= all_stops || (totals[2] >> kBinStopBits) + kBins >= 1u << (32 - kBinStepUnit);
            stops = min(all_stops, kBinStops - 1u);
            uint32_t prefix = sums[0], place = head_count + sums[1], stop = sums[2] & ((1u << kBinStopBits) - 1u);
            mass[0] = masses;
            if (holds_bins)
            {
                uint32_t new_packed[4];
                uint32_t prefixes[4];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    const uint32_t b = bin + j;
                    const uint32_t count = front[j + 1] - front[j];
                    const bool behind = b >= head_bins;
                    mass[j + 1] = mass[j] + own_mass[j];
                    prefixes[j] = prefix;
                    prefix += own_steps[j];
                    if (stop_word[j] != 0xffffffffu && stop + 1u < kBinStops)
                        shared.stop_bin[stop] = stop_word[j];
                    stop += stop_word[j] != 0xffffffffu ? 1u : 0u;
                    uint32_t where = behind ? place : front[j];
                    if (behind && kind[j] == kBinListed)
                        place += count;
                    if (masked[j] != 0u)
                        where = masked[j];
                    shared.places[b] = static_cast<uint16_t>(where);
                    new_packed[j] = (packed[j] & 0x3fffffffu) | (kind[j] << 30);
                }
                *reinterpret_cast<uint4*>(shared.packed + bin) = uint4{new_packed[0], new_packed[1], new_packed[2], new_packed[3]};
                *reinterpret_cast<uint4*>(shared.prefix + bin) = uint4{prefixes[0], prefixes[1], prefixes[2], prefixes[3]};
            }
            else
            {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    mass[j + 1] = mass[j];
            }
            if (tid == static_cast<int>(kBinQuads) - 1)
            {
                shared.prefix[kBins] = prefix;
                shared.places[kBins] = static_cast<uint16_t>(place);
            }
            if (tid == 0)
            {
                shared.stop_bin[stops] = kBins;
                shared.status = overflows ? 2u : 1u;
            }
            // ---- the listed elements in order: a bin's elements lie side by side in the list
            __syncthreads();
            const uint32_t fineness = fineness_of(list_first, listed - list_first);
            uint32_t fine[kPerThread];
#pragma unroll
            for (uint32_t k = 0; k < kPerThread; ++k)
            {
                fine[k] = 0u;
                if (list_first + k * kWalkThreads + tid < listed)
                {
                    const uint32_t b = (kOneBits - __float_as_uint(own_terms[k])) >> shift;
                    fine[k] = fineness * (shared.places[b] - list_first) +
                        fine_place(own_terms[k], shift, fineness * (packed_front(shared.packed[b + 1u]) - packed_front(shared.packed[b])));
                }
            }
            if (WALK > 0 && listed - list_first <= kWalkThreads)
            {
                const float first_term[1] = {own_terms[0]};
                const uint32_t first_token[1] = {own_tokens[0]}, first_fine[1] = {fine[0]};
                order_elements<1>(shared, list_first, listed - list_first, fineness, first_term, first_token, first_fine, tid);
            }
            else
                order_elements<kPerThread>(shared, list_first, listed - list_first, fineness, own_terms, own_tokens, fine, tid);
        }
        if (shared.status == 2u)
        {
            return kBinWalkEnds; // (more places to look at, or more steps, than the walk holds: left to the full-order kernels)
        }
        // ---- the sums.  `head_sum`: of the sum that the next launch goes on with; `next_*`: what it runs over
        float head_sum = 0.0f;
        uint32_t next_limit = 0, next_cut_bin = kBins;
        float next_cut_term = 0.0f;
        bool top_p_done = WALK == 2;
        bool given_up = false;
        if constexpr (WALK == 0)
        {
            const uint32_t head = min(window, head_count);
            sum_chunks<kWalkWaves>(shared.head, shared.terms, head_count, tid);
            sum_head<kWalkWaves, 0>(shared.head, shared.terms, head, kStopNever, 0.0f, 1.0f, 1.0f, tid);
            float sum = same_in_all(shared.head.sum);
#pragma unroll
            for (int j = 0; j < 5; ++j)
                mass[j] += sum;
            if (behind_head)
            {
                walk_bins<0, CHAINED>(shared, stops, row_terms, positions, s.misalignment, shift, head_bins, wide_first, window, kBins, 0.0f, sum, kStopNever, 0.0f, 1.0f, 1.0f, tid);
                given_up = shared.status == 2u;
                sum = same_in_all(shared.sum);
            }
            if (given_up)
            {
                return kBinWalkEnds;
            }
            normalizer = sum;
            // Min-P: the survivors are a prefix; where it ends inside the head it is known at once, else the smallest
            // term that survives is (fp32 division is monotone, and the term is within a few ulps of threshold x normaliser)
            uint32_t candidates = window;
            bool candidates_known = window <= head_count;
            if (min_p > 0.0f)
            {
                const float threshold = (1.0f / normalizer) * min_p;
                const float* terms = shared.terms;
                const uint32_t first = wave_partition_point(head, [terms, normalizer, threshold](uint32_t i) { return terms[i] / normalizer >= threshold; });
                if (first < head)
                {
                    candidates = first;
                    candidates_known = true;
                }
                else if (window > head_count)
                {
                    const float about = threshold * normalizer;
                    if (!(about > 3.1e-8f)) // (2^-25 and some ulps: below every bin)
                        cut_in_tail = 1u;
                    else
                    {
                        const uint32_t probe = __float_as_uint(about) + static_cast<uint32_t>(tid & (kWaveSize - 1)) - 32u;
                        const uint64_t survives = __builtin_amdgcn_ballot_w64(__uint_as_float(probe) / normalizer >= threshold);
                        const uint32_t cut_bits = __float_as_uint(about) - 32u + static_cast<uint32_t>(__builtin_ctzll(survives | 0x8000000000000000ull));
                        next_cut_term = __uint_as_float(cut_bits);
                        const uint32_t below = kOneBits - cut_bits;
                        if (below < kTailDistance)
                            next_cut_bin = min(below >> shift, kBins);
                    }
                }
            }
            if (!candidates_known && head_count == binned)
            {
                // every term that is in a bin is in the head, and what lies behind moves no sum: the sum runs to the
                // window's end, or, with a Min-P cut, over what is in the bins
                given_up = cut_in_tail != 0u;
                candidates = min_p > 0.0f ? binned : window;
                candidates_known = true;
            }
            sum_head<kWalkWaves, 1>(shared.head, shared.terms, min(candidates, head_count), kStopAtOrAbove, top_p, normalizer, 1.0f, tid);
            head_sum = same_in_all(shared.head.sum);
            const uint32_t stop = same_in_all(shared.head.stop);
            if (given_up && stop == 0xffffffffu)
            {
                return kBinWalkEnds;
            }
            if (stop != 0xffffffffu || candidates_known)
            {
                kept = stop != 0xffffffffu ? stop + 1u : candidates;
                renormalizer = head_sum;
                top_p_done = true;
            }
            else
                next_limit = window;
        }
        if constexpr (WALK == 1)
        {
            walk_bins<1, CHAINED>(shared, stops, row_terms, positions, s.misalignment, shift, head_bins, wide_first, limit, cut_bin, cut_term, sum_so_far, kStopAtOrAbove, top_p,
                         normalizer, 1.0f, tid);
            const bool stopped = shared.stopped != 0u;
            // (a sum that no stop condition ends runs to the window's end, or to the Min-P cut, which no bin may hold)
            given_up = shared.status == 2u || (!stopped && limit > binned && cut_in_tail != 0u);
            if (given_up)
            {
                return kBinWalkEnds;
            }
            // (behind the bins nothing moves the sum: it runs to its limit unless the cut ends it)
            kept = stopped ? shared.stop_rank + 1u : (cut_bin < kBins ? shared.taken : (limit > binned ? limit : shared.taken));
            kept = same_in_all(kept);
            renormalizer = same_in_all(shared.sum);
            top_p_done = true;
#pragma unroll
            for (int j = 0; j < 5; ++j)
                mass[j] += sum_so_far;
            __syncthreads();
        }
        if (WALK < 2 && g.want_filters != 0u && top_p_done && grid.part == 0u)
        {
            // the last element kept: in the head, where the Top-P sum stopped, or (no stop, no window) the last finite one, or
            // the last whose term the Min-P cut keeps; a row whose last element lies elsewhere gets no filter
            const bool in_head = kept <= head_count;
            const bool stopped_behind = !in_head && WALK == 1 && shared.stopped != 0u;
            const uint32_t last = in_head ? kept - 1u : stopped_behind ? same_in_all(shared.stop_at) : 0xffffffffu;
            const bool in_equal = stopped_behind && last == 0xffffffffu; // ... among thousands of equal terms
            const uint32_t top_k = same_in_all(params_of(carried.options).top_k);
            const bool unlimited = top_k == 0u || top_k >= a.vocab;
            const bool runs_on = !in_head && !stopped_behind;
            const bool by_cut = runs_on && WALK == 1 && cut_bin < kBins && (unlimited || kept < limit);
            const bool everything = by_cut || (runs_on && kept == window && min_p == 0.0f && unlimited);
            uint32_t filter_key = kLastFiniteKey, filter_token = a.vocab;
            if (last != 0xffffffffu || in_equal)
            {
                const bool extra = WALK == 1 && last >= kBinExtraPlace;
                const uint32_t first_of_list = extra ? kBinExtraPlace : WALK == 1 && !in_head ? head_count : 0u;
                const uint32_t end_of_list = extra ? kBinExtraPlace + same_in_all(shared.extra_count) : WALK == 1 && !in_head ? listed : head_count;
                int32_t token;
                if (WALK == 1 && in_equal)
                    token = token_of_equal<DTYPE>(a, row, shared, row_terms, positions, s.misalignment, __uint_as_float(same_in_all(shared.extra_least)),
                                                  kept - 1u - packed_front(same_in_all(shared.packed[shared.low])), tid);
                else
                    token = token_of_listed<DTYPE>(a, row, shared, row_terms, positions, s.misalignment, WALK == 1 && in_head ? sorted_tokens_out : shared.tokens, last, first_of_list, end_of_list, tid);
                filter_token = static_cast<uint32_t>(token);
                filter_key = descending_key(load_logit<DTYPE>(static_cast<const char*>(a.logits) + static_cast<size_t>(row) * a.row_stride * LogitsVector<DTYPE>::kElementBytes, filter_token));
            }
            if (tid == 0 && (last != 0xffffffffu || in_equal || everything))
            {
                record.normalizer = normalizer;
                record.renormalizer = renormalizer;
                record.kept = kept;
                record.filter_key = filter_key;
                record.filter_token = filter_token;
                record.least_term = by_cut ? cut_term : 0.0f;
                record.filtered = 1u;
            }
            __syncthreads();
        }
        // ---- the draw, inside the head or behind it
        if (top_p_done)
        {
            uint32_t at = 0, first_of_list = 0, end_of_list = head_count;
            const uint32_t* tokens = WALK == 1 ? sorted_tokens_out : shared.tokens;
            bool found = kept == 1u && head_count != 0u;
            if (WALK < 2 && !found)
            {
                if (WALK == 1)
                    sum_chunks<kWalkWaves>(shared.head, shared.terms, head_count, tid);
                sum_head<kWalkWaves, 2>(shared.head, shared.terms, min(kept, head_count), kStopAbove, uniform, normalizer, renormalizer, tid);
                head_sum = same_in_all(shared.head.sum);
                const uint32_t stop = same_in_all(shared.head.stop);
                found = stop != 0xffffffffu || kept <= head_count;
                at = stop != 0xffffffffu ? stop : kept - 1u;
                next_limit = kept;
            }
            if constexpr (WALK == 2)
            {
                walk_bins<2, CHAINED>(shared, stops, row_terms, positions, s.misalignment, shift, head_bins, wide_first, limit, kBins, 0.0f, sum_so_far, kStopAbove, uniform,
                             normalizer, renormalizer, tid);
                // (no partial sum exceeds the draw: the last element kept, which may lie anywhere: left to the full-order kernels)
                at = same_in_all(shared.stop_at);
                if (shared.status != 1u || shared.stopped == 0u)
                    return kBinWalkEnds;
                found = true;
                first_of_list = at >= kBinExtraPlace ? kBinExtraPlace : head_count;
                end_of_list = at >= kBinExtraPlace ? kBinExtraPlace + same_in_all(shared.extra_count) : listed;
            }
            if (found)
            {
                if (grid.part == 0u)
                {
                    int32_t token;
                    float term;
                    if (WALK == 2 && at == 0xffffffffu) // (among thousands of equal terms)
                    {
                        term = __uint_as_float(same_in_all(shared.extra_least));
                        token = token_of_equal<DTYPE>(a, row, shared, row_terms, positions, s.misalignment, term,
                                                      same_in_all(shared.stop_rank) - packed_front(same_in_all(shared.packed[shared.low])), tid);
                    }
                    else
                    {
                        token = token_of_listed<DTYPE>(a, row, shared, row_terms, positions, s.misalignment, tokens, at, first_of_list, end_of_list, tid);
                        term = shared.terms[at];
                    }
                    if (tid == 0)
                    {
                        const ncnn_moe_sample_params p = params_of(carried.options);
                        write_token(a, row, p, token, kept == 1u ? 1.0f : (term / normalizer) / renormalizer, kept, kept == 1u ? 0 : 1, result_flags(p));
                        a.row_state[row] = kRowDoneLater;
                        record.served = 1u;
                    }
                }
                return kBinWalkEnds;
            }
            if (WALK == 0 || head_count == binned)
            {
                // (the draw passes every term in a bin: the last element kept lies in no list)
                return kBinWalkEnds;
            }
        }
        if constexpr (WALK < 2)
        {
            // ---- the bins' steps of the next sum: the Top-P sum's behind WALK 0, the draw's behind WALK 1
            const float scale = 1.0f / (WALK == 0 ? normalizer : renormalizer);
#pragma unroll
            for (int j = 0; j < 5; ++j)
                mass[j] *= scale;
            uint4 before{0u, 0u, 0u, 0u}; // elements of the thread's bins in the parts in front (where the next list takes this part's)
            if (holds_bins)
                before = reinterpret_cast<const uint4*>(g.before + static_cast<size_t>(slot * grid.parts + grid.part) * kBins)[tid];
            BinPlan plan = plan_bins(bin, front, mass, head_bins, next_limit, next_cut_bin, WALK == 0 ? top_p : uniform, kForeseenLater, shift,
                                     1.0f / (WALK == 0 ? normalizer : normalizer * renormalizer));
            uint32_t to_list[1] = {holds_bins ? plan.listed : 0u};
            {
                uint32_t totals[1];
                bin_scan<kWalkWaves>(to_list, totals, shared.scan, tid);
            }
            uint32_t place[4];
            const uint32_t own_end = fit_plan(plan, front, head_count + to_list[0], place);
            uint32_t* const entries = shared.prefix;
            uint32_t* const steps = shared.packed;
            uint32_t* const masks = shared.tokens;                      // (the list has been used)
            uint32_t* const ties = shared.tokens + kMaskWords;
            static_assert(kMaskWords + 3u * kBinWords <= kBinListCap + kBinExtraCap, "masks and words fit where the list was");
            // the sorted head's tokens are kept for the next walk
            if (WALK == 0 && grid.part == 0u)
            {
                for (uint32_t i = tid; i < head_count; i += kWalkThreads)
                    sorted_tokens_out[i] = shared.tokens[i];
            }
            if (tid == 0)
            {
                shared.listed_end = 0u;
                shared.wide_first = kBins;
            }
            __syncthreads();
            if (tid < static_cast<int>(3u * kBinWords))
                ties[tid] = 0u;
            for (uint32_t i = tid; i < kMaskWords / 4u; i += kWalkThreads)
                reinterpret_cast<uint4*>(masks)[i] = uint4{0u, 0u, 0u, 0u};
            if (holds_bins)
            {
                const uint32_t next_wide = first_wide_bin(plan, bin, shift, 1.0f / (WALK == 0 ? normalizer : normalizer * renormalizer));
                if (leads_wave(next_wide < kBins))
                    atomicMin(&shared.wide_first, next_wide);
                uint32_t next_packed[4];
                const uint32_t in_front[4] = {before.x, before.y, before.z, before.w};
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    next_packed[j] = (plan.kind[j] << 30) | (plan.exponent[j] << 22) | front[j];
                    uint32_t entry = plan.kind[j] == kBinAdded ? plan.exponent[j] : 0x40000000u;
                    if (plan.kind[j] == kBinListed)
                        entry = 0x80000000u | (place[j] + in_front[j]);
                    entries[bin + j] = entry;
                }
                *reinterpret_cast<uint4*>(steps + bin) = uint4{0u, 0u, 0u, 0u};
                words_of_thread = uint4{next_packed[0], next_packed[1], next_packed[2], next_packed[3]};
            }
            __syncthreads();
            if (own_end != 0u && holds_bins)
                atomicMax(&shared.listed_end, own_end);
            add_bin_steps<WALK + 1, kWalkThreads, CHAINED>(row_terms, s, shift, head_bins, kBins - head_bins, normalizer, renormalizer, entries, steps, ties, masks, shared.wide_first,
                                                  g.list_terms[kTo] + static_cast<size_t>(row) * kBinListCap, g.list_tokens[kTo] + static_cast<size_t>(row) * kBinListCap, near, tid);
            __syncthreads();
            const size_t pair = slot * grid.parts + grid.part;
            if (holds_bins)
                hand_over_vector(near, g.steps[kTo] + pair * kBins, kBins * 4u, static_cast<uint32_t>(tid), *reinterpret_cast<uint4*>(steps + bin));
            for (uint32_t i = tid; i < kMaskWords / 4u; i += kWalkThreads)
                hand_over_vector(near, g.masks[kTo] + pair * kMaskWords, kMaskWords * 4u, i, reinterpret_cast<uint4*>(masks)[i]);
            if (tid < static_cast<int>(3u * kBinWords))
                hand_over(near, g.ties[kTo] + pair * 3u * kBinWords, 3u * kBinWords * 4u, static_cast<uint32_t>(tid), ties[tid]);
            if (tid == 0)
            {
                carried.normalizer = normalizer;
                carried.renormalizer = renormalizer;
                carried.kept = kept;
                carried.head_sum = head_sum;
                carried.limit = next_limit;
                carried.listed = max(shared.listed_end, head_count);
                carried.wide_first = shared.wide_first;
                if (WALK == 0)
                {
                    carried.cut_bin = next_cut_bin;
                    carried.cut_term = next_cut_term;
                    carried.cut_in_tail = cut_in_tail;
                }
            }
        }
    }
    return WALK < 2 ? kBinWalkGoesOn : kBinWalkEnds;
}

// The parts of a row meet: what each has handed over before is there for all behind it.  False: given up, because a part did not come.
// Every thread calls it; `meeting` counts from 1, `wait`: whether the caller takes anything over.
//
// A row's P parts are every eighth of 8 P workgroups that follow each other (bin_grid), and a workgroup has parts of one row only where rows
// have several.  Workgroups start in order, and a part comes before it waits, so the wait ends on a device that holds 8 P workgroups at a time:
// most_parts_of sees to that.  Workgroups of other launches may hold the places, for a while, or, where they wait for parts of their own rows
// that find no place either, for good: three calls of 8 rows that share a device can each hold 10 of a row's 16 places.  So a part that has
// looked most_looks times at the first meeting gives the row up, which is then left to the full-order kernels.  Behind the first meeting all
// parts have started, and are waited for kLaterLooks times as long.
//
// arrivals[0] counts the parts that have come to the row's meetings and, above, how many came to the first from each XCD: from then on
// shared.near tells whether all are on one.  arrivals[1] counts those that are done with the row: the last of them returns both to zero.
constexpr uint32_t kLaterLooks = 16;
constexpr uint32_t kPartsApart = 1u << 31; // in most_looks: the parts hand over as if they were on several XCDs (tests)
constexpr unsigned long long kArrivalsOnly = 0xffffull;
constexpr unsigned long long kRowGivenUp = 1ull << 63;
constexpr uint32_t kXcdShift = 16, kXcdBits = 5;
static_assert(kMaxBinParts < 1u << kXcdBits, "the parts that come from one XCD are counted in kXcdBits");

// How often a part looks at the first meeting, half a microsecond a look: about as long as sorting the row takes instead (8 rows of 310,000
// without a bin that serves them 0.5 ms, 1 of 1,000,000 5.5 ms, of 4,000,000 21 ms), so that waiting in vain costs no more than giving up too
// early.  Side by side the call's own select and window kernels hold places while they stream: a look for each MB, 2 TB/s.
constexpr uint32_t kFewestLooks = 1000;
constexpr uint32_t kLogitsALook = 100;

inline uint32_t most_looks_of(uint32_t rows, uint32_t vocab, uint32_t element_bytes, bool side_by_side)
{
    const uint64_t beside = side_by_side ? static_cast<uint64_t>(rows) * vocab * element_bytes >> 20 : 0u;
    const uint64_t looks = (vocab / kLogitsALook > kFewestLooks ? vocab / kLogitsALook : kFewestLooks) + beside;
    return static_cast<uint32_t>(looks < 0xffffffffu / kLaterLooks ? looks : 0xffffffffu / kLaterLooks);
}

// The parts of a row whose 8 P workgroups a device of `compute_units` holds at a time, one to a compute unit at least: 16 from half a
// card on, 8 and 4 on partitions of two XCDs and of one, where a row of 16 parts would wait for workgroups that cannot start.
inline uint32_t most_parts_of(uint32_t compute_units)
{
    const uint32_t parts = compute_units / 8u;
    return parts < 1u ? 1u : parts < kMaxBinParts ? parts : kMaxBinParts;
}

__device__ __forceinline__ uint32_t own_xcd()
{
    return __builtin_amdgcn_s_getreg(20 | (3 << 11)) & 7u; // HW_REG_XCC_ID
}

__device__ __forceinline__ bool parts_meet(unsigned long long* arrivals, uint32_t parts, uint32_t meeting, bool wait, uint32_t most_looks, BinWalkShared& shared, int tid)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // (stores have arrived in the L2, or in memory, when they are counted)
    if (parts == 1u)
    {
        if (tid == 0)
            shared.near = 1u;
        __syncthreads();
        return true;
    }
    __syncthreads();
    if (tid == 0)
    {
        const unsigned long long own_place = 1ull << (kXcdShift + kXcdBits * own_xcd());
        const unsigned long long one = meeting == 1u ? 1ull + own_place : 1ull;
        unsigned long long seen = __hip_atomic_fetch_add(arrivals, one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + one;
        const uint32_t goal = meeting * parts;
        const uint32_t first_looks = most_looks & ~kPartsApart;
        const uint32_t most = meeting == 1u ? first_looks : first_looks * kLaterLooks;
        const auto come = [&]() { return static_cast<uint32_t>(seen & kArrivalsOnly) >= goal; };
        for (uint32_t looks = 0; wait && !come() && (seen & kRowGivenUp) == 0ull; ++looks)
        {
            if (looks == most)
            {
                __hip_atomic_fetch_or(arrivals, kRowGivenUp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
            __builtin_amdgcn_s_sleep(1);
            seen = __hip_atomic_load(arrivals, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        shared.met = wait && come() ? 1u : 0u;
        if (meeting == 1u)
            shared.near = (seen & ~kRowGivenUp) >> kXcdShift == parts * (own_place >> kXcdShift) && (most_looks & kPartsApart) == 0u ? 1u : 0u;
    }
    __syncthreads();
    return same_in_all(shared.met) != 0u;
}

__device__ __forceinline__ void part_leaves(unsigned long long* arrivals, uint32_t parts, int tid)
{
    if (parts > 1u && tid == 0 && __hip_atomic_fetch_add(arrivals + 1, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1ull == parts)
    {
        __hip_atomic_store(arrivals, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(arrivals + 1, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// The launch's arguments (its only ones, BinArgs) read once more: what is read at a kernel's start is kept to its end otherwise, here in
// some hundred scalar registers that there are not.
__device__ __forceinline__ const BinArgs& arguments_read_anew()
{
    using ConstantBytes = const __attribute__((address_space(4))) uint8_t;
    ConstantBytes* p = (ConstantBytes*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const BinArgs*)p;
}

// The walks of a row, from where its parts have met `met` times (not at all: whether they are on one XCD is not known before the first
// walk has handed over).
template <int DTYPE, bool CHAINED>
__device__ __forceinline__ void walk_row(
    const BinGrid& grid, uint32_t slot, uint32_t row, unsigned long long* arrivals, uint32_t met, uint32_t most_looks, BinWalkShared& shared, uint4 words, int tid)
{
    const auto near = [&]() { return same_in_all(shared.near) != 0u; };
    // (behind the second meeting the first part goes on alone)
    if (bin_walk<DTYPE, 0, CHAINED>(arguments_read_anew(), grid, slot, row, CHAINED ? near() : grid.parts == 1u, shared, words, tid) == kBinWalkGoesOn &&
        parts_meet(arrivals, grid.parts, met + 1u, true, most_looks, shared, tid) &&
        bin_walk<DTYPE, 1, CHAINED>(arguments_read_anew(), grid, slot, row, near(), shared, words, tid) == kBinWalkGoesOn &&
        parts_meet(arrivals, grid.parts, met + 2u, grid.part == 0u, most_looks, shared, tid) && grid.part == 0u)
        bin_walk<DTYPE, 2, CHAINED>(arguments_read_anew(), grid, slot, row, true, shared, words, tid);
}

template <int DTYPE>
__global__ __launch_bounds__(kWalkThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void bin_walks_kernel(BinArgs g)
{
    __shared__ BinWalkShared shared;
    const BinGrid grid = bin_grid(g.list[0], g.a.vocab, g.most_parts);
    const int tid = threadIdx.x;
    for (uint32_t slot = grid.first_slot; slot < grid.rows; slot += grid.slot_step)
    {
        const uint32_t row = same_in_all(g.list[1u + slot]);
        unsigned long long* const arrivals = g.arrivals + static_cast<size_t>(row) * kArrivalWords;
        const BinRow& record = g.records[row];
        const uint32_t state = same_in_all(record.state[1]);
        if (tid == 0)
        {
            shared.row.shift = record.shift;
            shared.row.window = record.window;
            shared.row.saw_nan = record.saw_nan;
            shared.row.binned = record.binned;
            shared.row.head_bins = record.head_bins;
            shared.row.head_count = record.head_count;
            shared.row.listed = record.listed;
            shared.row.wide_first = record.wide_first;
        }
        const uint32_t option = read_option(g.a, row, tid);
        uint4 words{0u, 0u, 0u, 0u};
        if (tid < static_cast<int>(kBinQuads))
            words = reinterpret_cast<const uint4*>(g.packed + static_cast<size_t>(row) * kBins)[tid];
        if (tid < static_cast<int>(kRowOptionWords))
            shared.row.options[tid] = option;
        __syncthreads();
        if (state == kBinRowGoesOn)
            walk_row<DTYPE, false>(grid, slot, row, arrivals, 0u, g.most_looks, shared, words, tid);
        else
            end_early(g, grid.part, row, params_of(shared.row.options), state, record.saw_nan, tid);
        part_leaves(arrivals, grid.parts, tid);
        __syncthreads();
    }
}

// (1) to (4) in one launch.
template <int DTYPE>
__global__ __launch_bounds__(kWalkThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void bin_chain_kernel(BinArgs g)
{
    __shared__ BinWalkShared shared;
    __shared__ BinSumShared of_sum;
    __shared__ RowList listed_rows;
    __shared__ uint4 stats[kMaxBinParts];
    __shared__ uint64_t exp2_table[32];
    static_assert(kWalkWaves <= static_cast<int>(kMaxBinParts), "the waves' statistics and the parts' take turns");
    const int tid = threadIdx.x;
    if (tid < 32)
        exp2_table[tid] = kExp2Table[tid];
    const uint32_t rows = list_rows_in_place<kWalkWaves>(g.a, g.listing, g.windows_are_selects != 0u, false, g.list, g.window_list, listed_rows, tid);
    const BinGrid grid = bin_grid(rows, g.a.vocab, g.most_parts, kChainGrid);
    for (uint32_t slot = grid.first_slot; slot < grid.rows; slot += grid.slot_step)
    {
        const uint32_t row = same_in_all(row_of_slot(g.listing, g.list, listed_rows, slot));
        unsigned long long* const arrivals = g.arrivals + static_cast<size_t>(row) * kArrivalWords;
        const BinStretch s = bin_stretch<LogitsVector<DTYPE>::kElementBytes>(g.a, row, grid.part, grid.parts);
        const uint32_t option = read_option(g.a, row, tid);
        if (grid.part == 0u && tid == 0)
        {
            // (whatever becomes of the row: an earlier call's do not count)
            g.records[row].served = 0u;
            g.records[row].filtered = 0u;
        }
        const uint4 of_part = stats_of_part<DTYPE, kWalkThreads>(g.a, grid, row, stats, tid);
        if (tid < static_cast<int>(kRowOptionWords))
            shared.row.options[tid] = option;
        if (tid == 0)
            hand_over_vector(grid.parts == 1u, g.stats + slot * grid.parts, grid.parts * 16u, grid.part, of_part);
        if (parts_meet(arrivals, grid.parts, 1u, true, g.most_looks, shared, tid))
        {
            const bool near = same_in_all(shared.near) != 0u;
            const BinRowStart start = terms_of_part<DTYPE, kWalkThreads, true>(arguments_read_anew(), grid, slot, row, params_of(shared.row.options), near, shared.tokens, stats, exp2_table, tid);
            if (tid == 0)
            {
                shared.row.shift = start.shift;
                shared.row.window = start.window;
                shared.row.saw_nan = start.saw_nan;
            }
            if (same_in_all(start.state) != kBinRowGoesOn)
                end_early(g, grid.part, row, params_of(shared.row.options), start.state, start.saw_nan, tid);
            else if (parts_meet(arrivals, grid.parts, 2u, true, g.most_looks, shared, tid))
            {
                const uint4 words = sum_of_part<kWalkThreads, true>(arguments_read_anew(), grid, slot, row, same_in_all(params_of(shared.row.options).top_p),
                    same_in_all(params_of(shared.row.options).min_p), near, s, shared.prefix, shared.packed, shared.tokens, shared.tokens + kMaskWords, shared.scan, of_sum, shared.row, tid);
                if (parts_meet(arrivals, grid.parts, 3u, true, g.most_looks, shared, tid))
                    walk_row<DTYPE, true>(grid, slot, row, arrivals, 3u, g.most_looks, shared, words, tid);
            }
        }
        part_leaves(arrivals, grid.parts, tid);
        __syncthreads();
    }
}

// Lists the rows that the first select leaves, those with a window (null: nowhere) and the others, for a call of more rows than
// kRowsListedInPlace.  One workgroup.
__global__ __launch_bounds__(kBinThreads) void later_rows_list_kernel(SamplerArgs a, uint32_t by_options, uint32_t* windows, uint32_t* others)
{
    __shared__ uint32_t wave_totals[2][kBinWaves];
    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    uint32_t listed[2] = {0u, 0u};
    for (uint32_t first = 0; first < a.rows; first += kBinThreads)
    {
        const uint32_t row = first + static_cast<uint32_t>(tid);
        bool mine[2] = {false, false};
        if (row < a.rows)
        {
            bool window = false;
            const bool left = row_is_left(a, row, by_options != 0u, windows != nullptr, window);
            mine[0] = left && window;
            mine[1] = left && !window;
        }
        uint64_t mask[2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
        {
            mask[i] = __builtin_amdgcn_ballot_w64(mine[i]);
            if ((tid & (kWaveSize - 1)) == 0)
                wave_totals[i][wave] = static_cast<uint32_t>(__popcll(mask[i]));
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i)
        {
            uint32_t before = 0, total = 0;
#pragma unroll
            for (int w = 0; w < kBinWaves; ++w)
            {
                before += w < wave ? wave_totals[i][w] : 0u;
                total += wave_totals[i][w];
            }
            uint32_t* const list = i == 0 ? windows : others;
            if (mine[i] && list != nullptr)
                list[1u + listed[i] + before + static_cast<uint32_t>(lanes_below(mask[i]))] = row;
            listed[i] += total;
        }
        __syncthreads();
    }
    if (tid == 0)
    {
        if (windows != nullptr)
            windows[0] = listed[0];
        if (others != nullptr)
            others[0] = listed[1];
    }
}

} // namespace ncnn_moe_hip

#endif // NCNN_MOE_HIP_SAMPLER_BINS_H

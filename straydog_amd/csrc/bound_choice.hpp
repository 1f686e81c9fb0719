// The k highest of many by a workgroup of 1024 threads, in order of their names: the k-th highest of the values that each are the highest of their own share of all
// is a bound that k values reach and little more; a histogram of those finds the bin that the k-th highest lies in, and a bit a name lets the chosen leave in
// order.
//
// One workgroup's pass over a row is bound by its instructions, by the steps that wait for each other and, as every line of code runs once, by
// fetching them: 256 workgroups at once, a compute unit each, took up to 23 us over code that one alone ran in 10.  So nothing here is
// ordered before the end, and few loops are unrolled.
#pragma once
#include "wave_ops.hpp"

namespace sd {

constexpr int CHOICE_THREADS = 1024, CHOICE_WAVES = CHOICE_THREADS / 64, CHOICE_NAMES = 65536, CHOICE_LIST = RANGE_BINS / 2, CHOICE_FEW = 64;

// What a choice keeps between its steps, in LDS.
struct ChoiceShared {
    union {
        uint32_t bound_bins[RANGE_BINS];
        uint2 list[CHOICE_LIST];                // (value, name), for what has the bound by then
    };
    union {
        uint32_t bins[RANGE_BINS];
        uint2 members[CHOICE_FEW];              // of one bin, when the histogram is done with
        uint32_t equal[CHOICE_NAMES / 32];      // ... or a bit for each
    };
    uint32_t chosen[CHOICE_NAMES / 32];         // a bit a name
    uint32_t wave_sums[CHOICE_WAVES], ends[CHOICE_WAVES][2], threshold, remaining, held, named, listed, in_bin;
};

// A workgroup's first step: the counts, the bins and the bits to zero (a barrier follows, group_range's for one).
__device__ __forceinline__ void choice_begin(ChoiceShared& sh) {
    const unsigned t = threadIdx.x;
    sh.bound_bins[t] = 0u; sh.bound_bins[t + CHOICE_THREADS] = 0u;
    sh.bins[t] = 0u; sh.bins[t + CHOICE_THREADS] = 0u;
    sh.chosen[t] = 0u; sh.chosen[t + CHOICE_THREADS] = 0u;
    if (t == 0) { sh.remaining = 0u; sh.named = 0u; sh.listed = 0u; sh.in_bin = 0u; }
}

// The lowest and the highest of the threads' (lowest, highest).
__device__ __forceinline__ void group_range(uint32_t& lowest, uint32_t& highest, uint32_t (*ends)[2]) {
    lowest = wave_least(lowest); highest = wave_most(highest);
    if (threadIdx.x % 64 == 0) { ends[threadIdx.x / 64][0] = lowest; ends[threadIdx.x / 64][1] = highest; }
    __syncthreads();
    const unsigned lane = threadIdx.x % 64;
    lowest = wave_least(ends[lane % CHOICE_WAVES][0]); highest = wave_most(ends[lane % CHOICE_WAVES][1]);
}

// The sum of `mine` over the threads before this one (a barrier).
__device__ __forceinline__ uint32_t group_before(uint32_t mine, uint32_t* wave_sums) {
    const unsigned lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t upto = wave_prefix(mine);
    if (lane == 63) wave_sums[wave] = upto;
    __syncthreads();
    const uint32_t waves = wave_prefix(lane < unsigned(CHOICE_WAVES) ? wave_sums[lane] : 0u);
    return upto - mine + (wave ? uint32_t(__builtin_amdgcn_readlane(int(waves), int(wave) - 1)) : 0u);
}

// The bin in which the wanted-th highest value lies, its rank in it and how many values the bin holds: sh.threshold, sh.remaining, sh.held (as they were
// where there are fewer values).
__device__ __forceinline__ void range_pick(ChoiceShared& sh, const uint32_t* bins, uint32_t wanted) {
    const unsigned t = threadIdx.x;
    const uint32_t high = bins[RANGE_BINS - 1 - 2 * t], low = bins[RANGE_BINS - 2 - 2 * t], above = group_before(high + low, sh.wave_sums);
    if (above < wanted && above + high + low >= wanted) {
        const bool second = above + high < wanted;
        sh.threshold = RANGE_BINS - 1 - 2 * t - second;
        sh.remaining = wanted - above - (second ? high : 0u);
        sh.held = second ? low : high;
    }
    __syncthreads();
}

// The values from .. last over the bins; those far above the others share the highest.
struct Range {
    uint32_t from, last;
    int shift;
    __device__ __forceinline__ Range(uint32_t from, uint32_t most, uint32_t last) : from(from), last(last), shift(range_shift(max(most, from) - from)) {}
    __device__ __forceinline__ bool holds(uint32_t value) const { return value >= from && value <= last; }
    __device__ __forceinline__ uint32_t bin(uint32_t value) const { return min((value - from) >> shift, RANGE_BINS - 1); }
    __device__ __forceinline__ void narrow(uint32_t bin) {
        from += bin << shift;
        if (bin != RANGE_BINS - 1) last = from + min(last - from, (1u << shift) - 1);
    }
};

// A bin that holds too many (range is narrowed to it): its own values' range over all the bins.  False: they are all equal.  values(use) gives use() each value
// and its name.
template<class Values>
__device__ __forceinline__ bool range_refine(ChoiceShared& sh, uint32_t* bins, Range& range, Values values) {
    uint32_t lowest = 0xffffffffu, highest = 0u;
    values([&](uint32_t value, uint32_t) { if (range.holds(value)) { lowest = min(lowest, value); highest = max(highest, value); } });
    const uint32_t wanted = sh.remaining;
    group_range(lowest, highest, sh.ends);
    range = Range(lowest, highest, highest);
    if (lowest == highest) return false;
    bins[threadIdx.x] = 0u; bins[threadIdx.x + CHOICE_THREADS] = 0u;
    __syncthreads();
    values([&](uint32_t value, uint32_t) { if (range.holds(value)) atomicAdd(&bins[range.bin(value)], 1u); });
    __syncthreads();
    range_pick(sh, bins, wanted);
    range.narrow(sh.threshold);
    return true;
}

// A bound by values that each are the highest of their own share of all: thread t's count of them (those that are not `none`).  The k-th highest of them, to
// a bin of their range, rounded down, that no more than `most` of them reach; high: where the values that reach it are to be spread to.  0: there are fewer than k (high: 0), or
// too many are equal (high: to what).  The range ends at four times as far up as the highest that four neighbouring waves all reach: an infinity, or a few scores far above the others, would leave
// those in a handful of bins, whose additions wait for each other (a row of 4096 with an infinity 13.9 us, without 5.8; the passes alone 8.1).
template<int COUNT>
__device__ __forceinline__ uint32_t bound_by_maxima(ChoiceShared& sh, const uint32_t (&top)[COUNT], uint32_t none, uint32_t k, uint32_t most, uint32_t& high) {
    uint32_t lowest = 0xffffffffu, highest = 0u;
    const auto values = [&](auto use) {
        #pragma unroll
        for (int i = 0; i < COUNT; ++i)
            if (top[i] != none) use(top[i], 0u);
    };
    values([&](uint32_t value, uint32_t) { lowest = min(lowest, value); highest = max(highest, value); });
    choice_begin(sh);
    group_range(lowest, highest, sh.ends);
    high = highest <= lowest ? highest : 0u;
    if (highest <= lowest || k > most) return 0u;           // (none, or all equal)
    high = sh.ends[threadIdx.x % CHOICE_WAVES][1];
    high = min(high, from_lane<LANE_XOR_1>(0u, high));
    high = min(high, from_lane<LANE_XOR_2>(0u, high));
    high = wave_most(high);
    high = high > lowest && high - lowest < (highest - lowest) / 4 ? high + 3 * (high - lowest) : highest;       // (0: waves without a value)
    Range range(lowest, high, highest);
    values([&](uint32_t value, uint32_t) { atomicAdd(&sh.bound_bins[range.bin(value)], 1u); });
    __syncthreads();
    range_pick(sh, sh.bound_bins, k);
    if (!sh.remaining) { high = 0u; return 0u; }
    range.narrow(sh.threshold);
    while (k - sh.remaining + sh.held > most)
        if (!range_refine(sh, sh.bound_bins, range, values)) { high = range.from; return 0u; }
    return range.from;
}

// The choice of the k highest of the values that reach `bound` (`values` gives them with their names: k at least, few above `high`), of equal ones those of the lowest names: a histogram
// over their range finds the bin of the k-th highest (one more over that bin's, where it holds more than CHOICE_FEW), and each of the few values in that bin counts those
// before it; a bin of many equal ones has a bit for each.  emit(slot, name) for each in order of the names.
template<class Values, class Emit>
__device__ __forceinline__ void choose(ChoiceShared& sh, uint32_t k, uint32_t bound, uint32_t high, Values values, Emit emit) {
    const unsigned t = threadIdx.x, lane = t % 64;
    Range range(bound, high, 0xffffffffu);
    values([&](uint32_t value, uint32_t) { atomicAdd(&sh.bins[range.bin(value)], 1u); });
    __syncthreads();
    range_pick(sh, sh.bins, k);
    range.narrow(sh.threshold);
    bool equal = false;
    while (!equal && sh.held > unsigned(CHOICE_FEW)) equal = !range_refine(sh, sh.bins, range, values);
    const uint32_t need = sh.remaining, held = sh.held;
    if (equal) {
        sh.equal[t] = 0u; sh.equal[t + CHOICE_THREADS] = 0u;
        __syncthreads();
    }
    const auto mark = [](uint32_t* bits, uint32_t name) { atomicOr(&bits[name / 32], 1u << (name % 32)); };
    values([&](uint32_t value, uint32_t name) {
        if (value < range.from) return;
        if (value > range.last) mark(sh.chosen, name);
        else if (equal) mark(sh.equal, name);
        else sh.members[atomicAdd(&sh.in_bin, 1u)] = make_uint2(value, name);
    });
    __syncthreads();
    if (!equal) {
        // (sixteen threads a member)
        constexpr unsigned EACH = CHOICE_THREADS / CHOICE_FEW;
        const uint2 own = sh.members[min(t / EACH, held - 1)];
        uint32_t before = 0;
        for (uint32_t j = 0; j < held; j += EACH) {
            const uint2 other = sh.members[min(j + t % EACH, held - 1)];
            const bool is = j + t % EACH < held && (other.x > own.x || (other.x == own.x && other.y < own.y));
            before += uint32_t(__popcll((__ballot(is) >> (lane / EACH * EACH)) & ((1u << EACH) - 1)));
        }
        if (t % EACH == 0 && t / EACH < held && before < need) mark(sh.chosen, own.y);
        __syncthreads();
    }
    uint32_t words[2] = {sh.chosen[2 * t], sh.chosen[2 * t + 1]};
    if (equal) {
        uint32_t ties[2] = {sh.equal[2 * t], sh.equal[2 * t + 1]};
        const uint32_t before = group_before(uint32_t(__popc(ties[0]) + __popc(ties[1])), sh.wave_sums);
        uint32_t left = need > before ? need - before : 0u;
        #pragma unroll
        for (int w = 0; w < 2; ++w)
            for (; left && ties[w]; --left, ties[w] &= ties[w] - 1) words[w] |= ties[w] & (0u - ties[w]);
        __syncthreads();
    }
    size_t slot = group_before(uint32_t(__popc(words[0]) + __popc(words[1])), sh.wave_sums);
    #pragma unroll 1
    for (int w = 0; w < 2; ++w) {
        uint32_t bits = w ? words[1] : words[0];
        while (bits) {
            emit(slot++, 64 * t + 32 * w + uint32_t(__ffs(bits)) - 1);
            bits &= bits - 1;
        }
    }
}

}  // namespace sd

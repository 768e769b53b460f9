// The chunk-length rule of the work planners: what the host planner (tv_plan.cpp) and the device
// planner (tv_plan_device.hip) must agree on, once, for both.
//
// A plan cuts every request's prefix into chunks whose cost is at most a chunk target; costs are
// in quarter key-steps of a one-head item (about 185 a microsecond of a workgroup's streaming).
#pragma once

#include <math.h>
#include <stdint.h>

#include <algorithm>

namespace tv {

constexpr int kMinChunkKeys = 64;
constexpr int64_t kFillRounds = 4;   // item rounds the chunk target is chosen for

// Cost of one key of a work item.  A two-head item stages both heads' K/V but every wave still
// runs one head's 16 MFMAs per tile, so a tile costs it ~1.25x a one-head tile, not 2x
// (per-workgroup timestamps: 1.30 vs 1.03 us per tile on 64 requests of mixed lengths).
// Weighting by the head count left two-head chunks at half the length of one-head chunks of
// the same cost.
__host__ __device__ __forceinline__ constexpr int64_t cost_weight(int hpw) { return hpw == 2 ? 5 : 4; }

// A tree tile takes the general loop (ancestor masks, per-key slot addresses) and costs
// about two prefix tiles (per-workgroup timestamps on 8 requests of 64-node trees: 16.3 us for
// the last-chunk items, 11 prefix tiles + 2 tree tiles, against 13.2 us for 12 prefix
// tiles).  The chunk lengths of a split prefix are set so that the last chunk, which also
// walks the tree, ends level with the others: the prefix is cut as if it held this many
// keys per tree node more, within the same number of chunks.
constexpr int64_t kTreeKeyWeight = 2;

__host__ __device__ __forceinline__ constexpr int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

// a / b.  A generic 32-bit division is ~35 dependent instructions on the device, and the device
// planner is one wave's chain of them: below 2^22 a reciprocal's estimate is off by at most one.
__host__ __device__ __forceinline__ uint32_t divide(uint32_t a, uint32_t b) {
#ifdef __HIP_DEVICE_COMPILE__
    if (a < (1u << 22)) {
        const uint32_t q = static_cast<uint32_t>(static_cast<float>(a) * __builtin_amdgcn_rcpf(static_cast<float>(b)));
        const int32_t r = static_cast<int32_t>(a - q * b);
        return r < 0 ? q - 1 : static_cast<uint32_t>(r) >= b ? q + 1 : q;
    }
#endif
    return a / b;
}

__host__ __device__ __forceinline__ float reciprocal(float x) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_rcpf(x);
#else
    return 1.f / x;
#endif
}

// Longest chunk of a request whose items may cost `tau` (two heads an item or one): it gives the
// chunk count, ceil(prefix / it); the chunks then share the prefix evenly.
__host__ __device__ __forceinline__ uint32_t chunk_limit(int64_t tau, int hpw, int64_t max_chunk) {
    const uint32_t t = tau < 0xffffffffll ? static_cast<uint32_t>(tau) : 0xffffffffu;
    const uint32_t quota = hpw == 2 ? t / 5 : t / 4, cap = static_cast<uint32_t>(max_chunk);
    static_assert(cost_weight(1) == 4 && cost_weight(2) == 5, "the divisors");
    const uint32_t c = quota < cap ? quota : cap;
    const uint32_t r = ((c > kMinChunkKeys ? c : kMinChunkKeys) + 31u) / 32u * 32u;
    return r < cap ? r : cap;
}
__host__ __device__ __forceinline__ uint32_t chunk_count(uint32_t prefix, uint32_t limit) {
    return prefix > 0 ? divide(prefix + limit - 1, limit) : 1u;
}

// Keys of a chunk of a prefix of p keys before a tree of n nodes, cut into `chunks`: the prefix and
// the tree's weight shared evenly, in multiples of 32 keys, as far as that keeps the count (the
// chunks before the last stay below the prefix) and the cap.
__host__ __device__ __forceinline__ uint32_t chunk_keys_of(uint32_t p, uint32_t n, uint32_t chunks, int64_t max_chunk) {
    uint32_t chunk = (divide(p + chunks - 1, chunks) + 31) / 32 * 32;
    if (chunks > 1) {
        const uint32_t even = (divide(p + static_cast<uint32_t>(kTreeKeyWeight) * n + chunks - 1, chunks) + 31) / 32 * 32;
        const uint32_t keep = divide(p - 1, chunks - 1) / 32 * 32, cap = static_cast<uint32_t>(max_chunk);
        const uint32_t level = even < keep ? even : keep;
        const uint32_t most = level < cap ? level : cap;
        chunk = chunk > most ? chunk : most;
    }
    return chunk < 32 ? 32 : chunk;
}

// Choice of the chunk target, from `target`, the even share of a compute unit, and `now`, its
// item count.
//   More than kFillRounds rounds of items keep it: their last round weighs little.
//   Above one, items are made to fill whole rounds, those of the even share or fewer, whichever
//   span is estimated shorter: a round costs its longest item and kRoundCost (the item's
//   lookups, first loads and stores), an item kSlotCost (what of its merge the launch does not
//   hide).  8 requests of 1354-4060 keys and 18-54 nodes, 8 KV heads: 496 items in two rounds
//   56 us, 256 in one 38; a one-head shard of 32 requests of 1.1k-8.1k keys: 499 items 66 us,
//   249 items 50.
//   Within one round, fewer items stream longer but write and merge fewer partial rows.  The count
//   that balances the two, sqrt(cost / kItemCost), is taken if the plan's span estimate
//   (span_estimate, over the actual items) is kGainPercent shorter: 2 requests of 2000 keys and
//   8 nodes at head size 256, 256 items 40.6 us, 104 items 25.5; but 10 requests of 66-456 keys on
//   one head, 69 items 19.1 us, 48 items 21.3, which the estimate calls level.
// The three over 600 drawn batches, against the even share refilled only where its rounds were
// part-empty: 0.933 of its time, 29 of them more than 2 % slower and 7 more than 5 %.  Taking the
// balance without the estimate: 0.934, 50 and 18; never taking it: 0.947, 3 and 2, but half as
// long again on some that it gains.  The planner does not know the head size, whose partial rows
// cost from half (64) to four times (256) as much: that is what is left.
// `search(lo, hi, guess, sure, step, cap)`: the smallest i in [lo, hi] whose items at target
// i * step number at most cap, 0 if hi's do not (`sure`: they do); `guess` is a likely upper bound
// of it.  `shorter(tau, base)`: gains() of their spans.  Item counts fall as the target grows
// (chunk_count(p, chunk_limit(q)) does, and the even sharing keeps it), so any search finds the
// same target.
constexpr int64_t kRoundCost = 1000;
constexpr int64_t kSlotCost = 2;
constexpr int64_t kTauStep = 128;      // 32 keys of a one-head item
constexpr int64_t kItemCost = 5;       // of an item more, against its share of the streaming
constexpr int64_t kPartialCost = 8;    // of 256 live partial rows, written and merged
constexpr int64_t kPartCost = 60;      // of a chunk more in the longest merge
constexpr int64_t kLaunchCost = 1500;  // of the launches themselves
constexpr int64_t kGainPercent = 4;

// What a plan's span is estimated from: its longest item, the live rows of its partial results,
// the chunks of its longest merge.
struct PlanSpan {
    int64_t longest, partial_rows, parts;
};
__host__ __device__ __forceinline__ int64_t span_estimate(const PlanSpan& s) {
    return kLaunchCost + s.longest + kPartialCost * s.partial_rows / 256 + kPartCost * s.parts;
}
__host__ __device__ __forceinline__ bool gains(const PlanSpan& s, const PlanSpan& base) {
    return span_estimate(s) * (100 + kGainPercent) < span_estimate(base) * 100;
}
// A request's share of it: p keys, n nodes, `rows` score rows (over all heads).
__host__ __device__ __forceinline__ PlanSpan request_span(uint32_t p, uint32_t n, int64_t rows, int64_t weight,
                                                          uint32_t limit, int64_t max_chunk) {
    const uint32_t chunks = chunk_count(p, limit);
    const uint32_t chunk = chunk_keys_of(p, n, chunks, max_chunk);
    const uint32_t before = static_cast<uint64_t>(chunks - 1) * chunk < p ? (chunks - 1) * chunk : p;
    const int64_t last = weight * (static_cast<int64_t>(p - before) + n), full = chunks > 1 ? weight * chunk : 0;
    return {last > full ? last : full, chunks > 1 ? rows * chunks : 0, static_cast<int64_t>(chunks)};
}

struct PlanTotals {
    int64_t cost;          // of all items
    int64_t prefix_cost;   // ... without the trees
    int64_t units;         // items of an uncut batch
    int64_t target, now;
    int64_t compute_units;
};

template <class Search, class Shorter>
__host__ __device__ __forceinline__ int64_t plan_target(const PlanTotals& t, Search search, Shorter shorter) {
    if (t.now > kFillRounds * t.compute_units) return t.target;
    const bool one_round = t.now <= t.compute_units;
    int64_t balance = 0;
    if (one_round) {
        // An integer square root, as far as it matters.
        if (t.cost >= kItemCost * t.now * t.now || t.units >= t.now || t.cost > INT32_MAX) return t.target;
        const int32_t x = static_cast<int32_t>(t.cost) / static_cast<int32_t>(kItemCost);
        int32_t n = static_cast<int32_t>(sqrtf(static_cast<float>(x)));
        while (n * n > x) --n;
        while ((n + 1) * (n + 1) <= x) ++n;
        balance = n < t.units ? t.units : n;
    }
    const float prefix_cost = static_cast<float>(t.prefix_cost);
    const int64_t most = t.cost / kTauStep + 1;   // uncut
    const int64_t rounds = (t.now + t.compute_units - 1) / t.compute_units;
    int64_t best = t.target, span = 0;
    for (int64_t k = rounds; k >= 1; --k) {
        const int64_t cap = one_round ? balance : k * t.compute_units;
        const bool refill = !one_round && k == rounds;   // at most the even share; else above it
        int64_t tau = t.target;
        if (!refill || t.now < cap) {
            if (t.units > cap) break;
            // A limit is at most quota + 63 keys, and 5 is the largest weight: fewer than `cap` items take
            // a target above prefix_cost / cap - 315, and prefix_cost / (cap - units) + 5 is enough unless
            // a limit is capped.  Floats, with a margin: bounds only shorten the search.
            const int64_t step = refill ? 1 : kTauStep;
            const float above = prefix_cost * reciprocal(static_cast<float>(static_cast<int32_t>(cap))) * 0.99999f;
            int64_t lo = (static_cast<int32_t>(above < 1e9f ? above : 1e9f) - 316) / step, hi = refill ? t.target : most;
            const int64_t least = refill ? 1 : t.target / kTauStep + 1;
            if (lo < least) lo = least;
            if (hi < lo) {
                if (refill) lo = hi; else hi = lo;
            }
            int64_t guess = hi;
            if (t.units < cap) {
                const float enough = prefix_cost * reciprocal(static_cast<float>(static_cast<int32_t>(cap - t.units))) * 1.00001f;
                guess = (static_cast<int32_t>(enough < 1e9f ? enough : 1e9f) + 6) / step + 1;
            }
            if (guess < lo) guess = lo;
            if (guess > hi) guess = hi;
            const int64_t found = search(lo, hi, guess, refill, step, cap);
            if (found == 0) break;   // capped limits: no target holds it
            tau = found * step;
        }
        if (one_round) return shorter(tau, t.target) ? tau : t.target;
        const int64_t s = k * (tau + kRoundCost) + kSlotCost * cap;
        if (k == rounds || s < span) {
            span = s;
            best = tau;
        }
    }
    return best;
}

}  // namespace tv

// Which XCD takes which levels of which points (grid_levels.hip), and how many points one launch may have.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace tnn {

constexpr uint32_t kXcds = 8;

// Workgroup b is the (b / 8)-th of XCD b % 8 (workgroups go to the XCDs in turn; were they not, nothing but locality would be lost);
// XCD k takes the items [first[k], first[k + 1]) of the list of all (level, chunk of points) of the levels up to `n_own`, level by level, and then
// an eighth of the chunks of each further level, `each` at most.
struct LevelPlan {
    uint32_t first[kXcds + 1];
    uint32_t n_chunks;
    uint32_t n_own, each;
};

// Shares of equal cost (of a level: cost[l]). Returns the most items an XCD has: the launch is 8 times as many workgroups.
inline uint32_t plan_levels(const double *cost, uint32_t n_levels, LevelPlan *plan) {
    double total = 0.0, before = 0.0;
    for (uint32_t l = 0; l < n_levels; ++l) total += cost[l];
    uint32_t most = 0;
    for (uint32_t k = 0, l = 0; k <= kXcds; ++k) {
        const double until = total * k / kXcds;
        while (l + 1 < n_levels && before + cost[l] < until) before += cost[l++];
        const double part = std::min(1.0, std::max(0.0, (until - before) / cost[l]));
        plan->first[k] = k == kXcds ? n_levels * plan->n_chunks : l * plan->n_chunks + (uint32_t)(part * plan->n_chunks + 0.5);
        if (k > 0) most = std::max(most, plan->first[k] - plan->first[k - 1]);
    }
    return most;
}

// The levels from n_own on are shared, those in front dealt out by cost. Returns the most items an XCD has.
inline uint32_t plan_shared_levels(const double *cost, uint32_t n_own, uint32_t n_levels, LevelPlan *plan) {
    plan->n_own = n_own;
    plan->each = (plan->n_chunks + kXcds - 1) / kXcds;
    for (uint32_t k = 0; k <= kXcds; ++k) plan->first[k] = 0;
    return (n_own ? plan_levels(cost, n_own, plan) : 0) + plan->each * (n_levels - n_own);
}

// The turn-th item of an XCD; false where there is none.
#ifdef __HIPCC__
__host__ __device__
#endif
inline bool plan_item(const LevelPlan &plan, uint32_t n_levels, uint32_t xcd, uint32_t turn, uint32_t *level, uint32_t *chunk) {
    // (one division for both kinds: it is what a workgroup of a small batch waits for)
    const uint32_t first = plan.first[xcd], end = plan.first[xcd + 1], item = first + turn;
    const bool own = item < end;
    const uint32_t number = own ? item : item - end, chunks = own ? plan.n_chunks : plan.each, l = number / chunks;
    *level = l + (own ? 0u : plan.n_own);
    *chunk = number - l * chunks + (own ? 0u : (xcd + *level) % kXcds * plan.each); // (another eighth in every level: a batch of few chunks is not one XCD's)
    return *level < n_levels && *chunk < plan.n_chunks;
}

// The most chunks of a launch, whatever the levels cost: a launch has fewer than 2^32 threads, and one XCD may have nearly all items
// (16 levels, 256 threads: 2^17 chunks, 2^25 points and more; a level's tables are long in L2 by then).
inline size_t level_part_chunks(uint32_t n_levels, uint32_t threads) {
    const size_t items = ((size_t(1) << 32) - 1) / (kXcds * threads);
    return std::max<size_t>(1, items / n_levels);
}

} // namespace tnn

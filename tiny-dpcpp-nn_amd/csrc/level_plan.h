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

// Whether all XCDs take a level at a time, an eighth of the points each, instead of one or two of them the whole level. In cell order an eighth is a part of
// space. Two or three large levels are in use at once then and not eight: 32 MB a level is what the 256 MB in front of the memory hold, and there is nothing to balance by
// a guess of what levels cost, which is wrong where points share more lines than scattered ones (a picture's rows). But eight XCDs fetch the level,
// which scattered points have to make up for: as many rows of corners for each of its lines. Field, 3-D, 16 levels, us, by XCDs / shared, scattered and a picture's rows (in
// cell order from 5 * 2^17 points): 4 MB a level, 2^18 points 96 / 114 and 50 / 45, 2^19 180 / 198 and 81 / 69, 700 000 207 / 213 and 147 / 101, 10^6 289 / 292 and 204 / 133, 2^20 341 / 339 and 238 / 159 (8 levels 122 / 132 and 63 / 56, 170 / 180 and 88 / 78); 2 MB, 2^19 162 / 162 and 76 / 66; 256 KB and
// 1 MB, 2^19 152 / 157 and 164 / 168, rows 77 / 70 and 79 / 71, 2^20 281 / 267 and 297 / 282, 210 / 152 and 219 / 153; 8 MB, 2^18 158 / 168 and 64 / 51, 2^19 303 / 307 and 101 / 79, 2^20 512 / 491 and 304 / 175; 16 MB, 2^17 104 / 113, 2^18 198 / 204 and 83 / 58, 2^20 636 / 597 and 362 / 186;
// 32 MB, 20 000 points 35 / 30 and 21 / 16, 2^17 121 / 122 and 62 / 40, 2^21 1286 / 1177 and 774 / 339. 8 levels, 2^20 4 MB 157 / 154 and 111 / 73, 32 MB 281 / 253 and 181 / 81. 2-D, 4 MB, 2^19 93 / 99, 2^20 173 / 177; 8 MB, 2^19 123 / 128, 2^20 199 / 196; 16 MB,
// 2^19 152 / 149; 32 MB, 2^16 32 / 30, 2^20 252 / 219;
// 256 KB and 2 MB, 8 levels, 2^20 86 / 86 and 89 / 89, rows 60 / 54 and 61 / 53, 16 levels 122 / 121 and 120 / 125, rows 103 / 98 and 102 / 101. So scattered points lose 1 to 5 % at the sizes from which a rule
// begins (8 MB, 2^19; 16 MB, 2^18; 2-D, 2 MB, 2^20), for the up to 30 % that rows gain there. Levels of up to 4 MB an XCD's own L2 holds, and they are shared from 3 * 2^18 points on only:
// a level of 8 MB is shared by fewer points than one of 2 MB. (Two shared levels at a time, a coarse one's chunks between a fine one's: 32 MB 1170 -> 1145, 4 MB 328 -> 438.)
inline bool shared_level(uint32_t entries, size_t entry_bytes, uint32_t n_dims, size_t M) {
    const size_t MB = size_t(1) << 20, bytes = entries * entry_bytes, rows = M << (n_dims - 1), lines = bytes / 128;
    if (bytes > 16 * MB) return true;
    if (bytes > 4 * MB) return rows >= (bytes > 8 * MB ? 8 : 32) * lines;
    return M >= (size_t(3) << 18) && rows >= 128 * lines;
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

// The binned route of the grid's backward pass (grid_binned.hip): which levels take it and where its scratch lies.
#pragma once

#include "grid_device.h"

namespace tnn {

constexpr uint32_t kMaxBinned = 32;         // levels one launch bins
constexpr size_t kBinBatch = size_t(1) << 19; // points binned at a time, at most
constexpr uint32_t kBinMaxBins = 1024;      // bins of a level
constexpr uint32_t kBinSliceBytes = 128 * 1024; // most of a bin's slice of the table (LDS of a workgroup)

// All that the kernels need of a level, side by side: a workgroup has it after one scalar load.
struct BinLevel {
    uint32_t level;
    uint32_t offset, size, resolution, flags; // as in GridLevels
    float scale;
    uint32_t bins_log2, run_log2; // the level's runs of 2^run_log2 entries go to its 2^bins_log2 bins in turn
    uint32_t places;              // entries a bin has room for
    uint32_t copies_log2;         // copies of its sums that a crowded bin has
    uint32_t first_bin;           // bins of the levels in front of this one
    uint32_t first_quad;          // the same in fours of bins
};

struct BinPlan {
    uint32_t n_levels;
    uint32_t n_bins;                    // of all levels
    uint32_t n_quads;                   // the same in fours of bins
    uint32_t room_bins;                 // bins that the workspace has room for: those that the levels have in a short batch
    uint32_t slice_lds;                 // LDS bytes of the largest slice
    uint32_t sums_lds;                  // the same with copies of short slices
    uint32_t batch;                     // points binned at a time
    uint32_t later_bin[kMaxBinned - 1]; // first bin of the second level and those behind it, ~0 where there is none
    BinLevel at[kMaxBinned];
};

// Adds level l to the plan if it can take the route.
bool bin_plan_add(BinPlan *p, uint32_t l, const GridLevels &lv, const GridParams &gp, uint32_t n_dims, uint32_t n_features, size_t M);
size_t bin_scratch_bytes(const BinPlan &p, uint32_t n_dims, uint32_t n_features);
// What the plan's levels need for its batch and for any smaller one.
size_t bin_scratch_bytes_up_to(BinPlan p, uint32_t n_dims, uint32_t n_features);
// Whether the binning's launch can take the reduction with it, and then it is the first launch of a scatter (kBinning alone), before any that adds to the table.
bool bins_take_reduction(const BinPlan &p, uint32_t n_features, int dy_dtype, size_t M, const TrainReduce &r);
enum BinStage { kBinning = 1, kSums = 2, kBinningAndSums = 3 };
// Nothing in the scratch has to be cleared. With `overwrite` every entry of the plan's levels
// is written, whatever it held.
int launch_grid_binned(const BinPlan &p, const GridParams &gp, const GradLayout &dl, uint32_t n_dims, uint32_t n_features, const float *x,
                       const float4 *order, const void *dLdy, int dy_dtype, float *grad, bool overwrite, size_t M, void *scratch, hipStream_t s,
                       BinStage stage = kBinningAndSums, const TrainReduce *reduce = nullptr);

} // namespace tnn

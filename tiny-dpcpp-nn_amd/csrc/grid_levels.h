// The grid encoding level by level (grid_levels.hip): where its values lie, and what other translation units need of it.
#pragma once

#include "grid_device.h"

namespace tnn {

// An encoded batch by levels: feature f of level l and point i is element (l * pitch + i) * F + f, points in the order they were
// visited in. 64 points start on a line of their own for every F and type.
inline size_t level_pitch(size_t M) { return (M + 63) & ~(size_t)63; }

// Whether a batch is small enough for the kernel to write rows itself, pieces of a line from several XCDs. us, three dimensions and 2^14, 2^19, 2^22
// entries, direct / one thread a point (grid_forward_kernel): 16 000 points 8 / 22, 16 / 41, 22 / 41; 65 000 points 23 / 26, 46 / 49, 74 / 64. (2-D 7.7 / 13,
// 8.8 / 19, 11.5 / 19; 23 / 16, 33 / 24, 43 / 27.)
bool grid_rows_direct(size_t M);
// out: by levels (padded_width 0), or rows of padded_width values.
int launch_grid_levels(const tnn_grid_desc *desc, const GridLevels &lv, const GridParams &gp, const float *x, const float4 *order, const void *table, void *out,
                       int out_dtype, uint32_t padded_width, size_t M, hipStream_t s);

} // namespace tnn

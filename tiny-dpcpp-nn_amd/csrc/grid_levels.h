// The grid encoding level by level (grid_levels.hip): where its values lie, and what other translation units need of it.
#pragma once

#include "grid_device.h"

namespace tnn {

// An encoded batch by levels: feature f of level l and point i is element (l * pitch + i) * F + f, points in the order they were
// visited in; the points from M up to the pitch hold the last one's values. There are whole groups of 16 features: the levels beyond the
// last hold zeros.
__host__ __device__ inline size_t level_pitch(size_t M) { return (M + 63) & ~(size_t)63; }
__host__ __device__ inline uint32_t padded_levels(uint32_t n_levels, uint32_t F) { return ((n_levels * F + 15) & ~15u) / F; }
inline size_t levels_elements(const tnn_grid_desc *desc, size_t M) {
    return level_pitch(M) * padded_levels(desc->n_levels, desc->n_features_per_level) * desc->n_features_per_level;
}

// A lane's pieces of a point's encoded row as the first product of a network takes them (mlp_tile.h): features 16 kb + 8 h + [0, 8) of it. Point `first` + j, `first` the same for the whole wave; neighbouring points lie side by side in every level.
template <typename T, int W, int F>
__device__ __forceinline__ void load_level_pieces(typename Storage<T>::vec8 (&r)[W / 16], const T *levels, size_t pitch, uint32_t n_levels, size_t first, int j, int h) {
    typedef T part_t __attribute__((ext_vector_type(F)));
    typedef const __attribute__((address_space(1))) part_t *global_t;
    const size_t lane = ((size_t)(h * (8 / F)) * pitch + j) * F;
#pragma unroll
    for (int kb = 0; kb < W / 16; ++kb) {
        r[kb] = typename Storage<T>::vec8{};
        if ((uint32_t)(16 * kb) >= n_levels * F) continue;
#pragma unroll
        for (int g = 0; g < 8 / F; ++g) {
            const T *const level = levels + ((size_t)(16 * kb / F + g) * pitch + first) * F;
            const part_t v = *(global_t)(unsigned long long)(level + lane);
#pragma unroll
            for (int f = 0; f < F; ++f) r[kb][g * F + f] = v[f]; // (nothing else: a caller may want the loads under way)
        }
    }
}

// Whether a batch is small enough for the kernel to write rows itself, pieces of a line from several XCDs. us, three dimensions and 2^14, 2^19, 2^22
// entries, direct / one thread a point (grid_forward_kernel): 16 000 points 8 / 22, 16 / 41, 22 / 41; 65 000 points 23 / 26, 46 / 49, 74 / 64. (2-D 7.7 / 13,
// 8.8 / 19, 11.5 / 19; 23 / 16, 33 / 24, 43 / 27.)
bool grid_rows_direct(size_t M);
size_t level_bytes(const tnn_grid_desc *desc, uint32_t l);
size_t largest_level_bytes(const tnn_grid_desc *desc);
// out: by levels (padded_width 0), or rows of padded_width values.
int launch_grid_levels(const tnn_grid_desc *desc, const GridLevels &lv, const GridParams &gp, const float *x, const float4 *order, const void *table, void *out,
                       int out_dtype, uint32_t padded_width, size_t M, hipStream_t s);

} // namespace tnn

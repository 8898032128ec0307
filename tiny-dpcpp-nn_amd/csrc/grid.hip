// Multi-resolution hash-grid encoding for gfx950: forward gather + N-linear interpolation,
// backward scatter-add into an fp32 gradient table.
//
// Reference behaviour being reproduced: include/encodings/grid.h:37-135 (kernel_grid),
// :137-245 (kernel_grid_backward), :588-659 (offset table), :682-694 (zero padding of the output),
// include/common/common_device.h:700-775 (hashes, grid_index, grid_scale, grid_resolution).
//
// One thread owns one point and walks all levels: the coordinates are read once, every corner of a
// level is gathered before the blend (2^D independent loads in flight), and the whole encoded row is
// written as contiguous 16-byte pieces. Per-level constants (scale, resolution, table offset, size,
// how many dimensions enter the dense index, whether the level is hashed) are evaluated once on the
// host and reach the kernel as scalar kernel arguments; no thread evaluates exp2.
#include "grid_binned.h"
#include "adam_update.h"
#include "grid_levels.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>

namespace tnn {

// include/common/common_device.h:745-765 evaluated for the loop bounds only: the stride sequence
// depends on (resolution, size, n_dims) and not on the position.
static void fill_levels(const tnn_grid_desc *d, GridLevels *lv) {
    for (uint32_t l = 0; l < d->n_levels; ++l) {
        const uint32_t size = d->offsets[l + 1] - d->offsets[l];
        lv->offset[l] = d->offsets[l];
        lv->size[l] = size;
        lv->scale[l] = d->scales[l];
        lv->resolution[l] = d->resolutions[l];
        uint32_t stride = 1, dims_used = 0;
        for (uint32_t dim = 0; dim < d->n_dims && stride <= size; ++dim) {
            ++dims_used;
            stride *= d->resolutions[l];
        }
        const bool hashed = (d->grid_type == TNN_GRID_HASH) && (size < stride);
        const bool pow2 = (size & (size - 1)) == 0;
        lv->flags[l] = dims_used | (hashed ? 16u : 0u) | (pow2 ? 32u : 0u);
    }
}

constexpr int kGridThreads = 256;


// Levels are processed in groups whose outputs fill one 16-byte piece of the encoded row: all gathers of a
// group (GL * 2^D independent loads) are issued before the first blend, and the row is written in whole
// 16-byte pieces (a per-level 4-byte store turns into a 32-byte masked write at the memory controller).
template <int D, int F, typename P, typename O>
__global__ void __launch_bounds__(kGridThreads)
    grid_forward_kernel(const GridLevels lv, const GridParams gp, const float *__restrict__ xin, const float4 *__restrict__ order,
                        const P *__restrict__ table, O *__restrict__ out, long long M) {
    constexpr int PER16 = 16 / (int)sizeof(O);            // outputs per 16-byte piece
    constexpr int GL = (PER16 / F) > 0 ? (PER16 / F) : 1; // levels per group (F = 8 with fp32 output: 1 level, 2 pieces)
    constexpr int NOUT = GL * F;
    typedef O ovec __attribute__((ext_vector_type(NOUT)));
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= M) return;
    // In cell order (grid_order.hip) thread i takes the i-th record, coordinates and row number, instead of row i.
    float x[D];
    long long row = i;
    if (order) {
        const float4 r = order[i];
        x[0] = r.x;
        x[1] = r.y;
        if (D > 2) x[D - 1] = r.z;
        row = (long long)__float_as_uint(r.w);
    } else {
#pragma unroll
        for (int d = 0; d < D; ++d) x[d] = xin[i * D + d];
    }
    O *orow = out + row * gp.padded_width;
    const bool row_aligned = ((gp.padded_width * sizeof(O)) % 16 == 0) && ((reinterpret_cast<uintptr_t>(out) & 15) == 0);

    // The first kHeld pieces of a row (128 bytes with 16-byte pieces) are kept in registers and stored together when the
    // last of them is done, so that a row's pieces reach L2 back to back and leave it as one write; pieces computed
    // thousands of cycles apart would each sit in L2 as a partly written line among the table's lines.
    constexpr int kHeld = (NOUT * sizeof(O) == 16) ? 8 : 0;
    ovec held[kHeld > 0 ? kHeld : 1];
    auto do_group = [&](const uint32_t l0, ovec &o) __attribute__((always_inline)) {
        LevelConst lc[GL];
#pragma unroll
        for (int gl = 0; gl < GL; ++gl) lc[gl] = level_const(lv, (l0 + gl < gp.n_levels) ? l0 + gl : l0);
        const int n_valid = (int)((gp.n_levels - l0 < (uint32_t)GL) ? gp.n_levels - l0 : (uint32_t)GL);
        float r[NOUT];
        encode_levels<D, F, P, GL>(lc, n_valid, gp, x, table, r);
#pragma unroll
        for (int e = 0; e < NOUT; ++e) o[e] = to_out<O>(r[e]);
    };
    auto store_group = [&](const uint32_t l0, const ovec &o) __attribute__((always_inline)) {
        const uint32_t col0 = l0 * F;
        if (row_aligned && l0 + GL <= gp.n_levels) {
            if constexpr (NOUT * sizeof(O) == 16) {
                *reinterpret_cast<ovec *>(orow + col0) = o;
            } else { // F = 8 with fp32 output: two 16-byte pieces
#pragma unroll
                for (int e = 0; e < NOUT; ++e) orow[col0 + e] = o[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < NOUT; ++e)
                if (l0 + e / F < gp.n_levels) orow[col0 + e] = o[e];
        }
    };
#pragma unroll
    for (int p = 0; p < kHeld; ++p)
        if ((uint32_t)(p * GL) < gp.n_levels) do_group((uint32_t)(p * GL), held[p]);
#pragma unroll
    for (int p = 0; p < kHeld; ++p)
        if ((uint32_t)(p * GL) < gp.n_levels) store_group((uint32_t)(p * GL), held[p]);
    for (uint32_t l0 = kHeld * GL; l0 < gp.n_levels; l0 += GL) {
        ovec o;
        do_group(l0, o);
        store_group(l0, o);
    }
    // zero padding of the row (include/encodings/grid.h:682-694), in 16-byte pieces where the row allows it
    uint32_t c = gp.n_levels * F;
    if (row_aligned) {
        typedef O zvec __attribute__((ext_vector_type(PER16)));
        for (; c < gp.padded_width && (c % PER16) != 0; ++c) orow[c] = to_out<O>(0.0f);
        for (; c + PER16 <= gp.padded_width; c += PER16) *reinterpret_cast<zvec *>(orow + c) = zvec{};
    }
    for (; c < gp.padded_width; ++c) orow[c] = to_out<O>(0.0f);
}

template <int D>
__global__ void __launch_bounds__(kGridThreads)
    grid_indices_kernel(const GridLevels lv, const GridParams gp, const float *__restrict__ xin, uint32_t *__restrict__ out,
                        long long M) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= M) return;
    float x[D];
#pragma unroll
    for (int d = 0; d < D; ++d) x[d] = xin[i * D + d];
    for (uint32_t l = 0; l < gp.n_levels; ++l) {
        uint32_t cell[D];
        float frac[D];
        cell_of<D>(x, lv.scale[l], gp.interpolation, cell, frac);
#pragma unroll
        for (int c = 0; c < (1 << D); ++c) {
            uint32_t loc[D];
#pragma unroll
            for (int d = 0; d < D; ++d) loc[d] = (c & (1 << d)) ? cell[d] + 1 : cell[d];
            out[(i * gp.n_levels + l) * (1 << D) + c] = level_index<D>(loc, lv.size[l], lv.resolution[l], lv.flags[l], gp.hash_type);
        }
    }
}

// Which levels the backward pass accumulates in LDS first, and how the 1-D grid is split between the two routes.
struct BackwardPlan {
    uint32_t n_small;          // levels, or single features of levels, of which a copy fits the LDS budget
    uint32_t small_blocks;     // workgroups per such part, each takes `chunk` consecutive points
    uint32_t chunk;
    uint32_t big_blocks;       // workgroups per other level, a group of lanes per point
    uint8_t small_level[TNN_GRID_MAX_LEVELS];
    uint8_t small_feature[TNN_GRID_MAX_LEVELS];
    uint8_t big_level[TNN_GRID_MAX_LEVELS];
    // Points in cell order only: levels too large for a private copy of the whole level, where a stretch of consecutive
    // points still lands on few enough cells for a private copy of the box around them (kMaxTiled such levels).
    uint32_t n_tiled;
    uint32_t budget;           // LDS bytes a workgroup may use
    uint32_t tiled_start[17]; // first workgroup of each such level among the tiled workgroups, and their total
    uint8_t tiled_level[16];
    uint8_t tiled_chunk_log2[16]; // a stretch of the level is 2^n consecutive points
    uint8_t tiled_pieces[16];     // workgroups per row of the order's coarse cells; they take the row's stretches in turn
    uint32_t bins_per_row;        // coarse cells in a row (64 in 2-D, 16 in 3-D), n_rows rows
    uint32_t n_rows;
    size_t more_up_to;            // points up to which a batch in the caller's order bins more levels, 0: none does
};
constexpr uint32_t kMaxTiled = 16;
constexpr uint8_t kAllFeatures = 255;
// Points of the batch per cell of a level, at least, for the boxed route: against the direct route, and against the binned one,
// whose levels cost the same whatever their cells (2-D, 2^18 points: a level of 0.31 points a cell takes 6.6 us boxed and 3.0
// binned; one of 0.7, 4.8 and 7.7; 1.6: 3.8 and 6.4; 3.5: 3.1 and 7.5; 7.9: 2.6 and 6.3).
constexpr double kBoxedMinPerCell = 0.3, kBoxedMinPerCellBinned = 0.5;

constexpr size_t kMoreBinnedBelow = size_t(1) << 17; // points of a batch in the caller's order that may bin more levels (plan_backward)

constexpr int kGridWave = 64;                    // lanes of a wave
constexpr int kBwdThreads = 512;                 // the backward kernel's workgroups
constexpr int kDirectPasses = 8;                 // groups of kBwdThreads / lanes-per-point points a direct-route workgroup takes
constexpr uint32_t kPrivateLdsBytes = 64 * 1024; // LDS budget of a workgroup; two such workgroups fit a CU
// In cell order more levels take an LDS route, and the launch's LDS size holds for every workgroup, also for those of the
// direct route, which need none: four workgroups of 40 KiB fill a CU's wave slots.
constexpr uint32_t kPrivateLdsBytesOrdered = 40 * 1024;
constexpr uint32_t kCopiedBytesOrdered = 16 * 1024; // and of a level that is copied whole
constexpr uint32_t kPrivateChunk = 4096;         // points per workgroup on the LDS route

// Coordinates and row number of the i-th point: row i of x, or the i-th record of the cell order (grid_order.hip).
template <int D>
__device__ __forceinline__ long long load_point(const float *__restrict__ xin, const float4 *__restrict__ order, long long i, float (&x)[D]) {
    if (order) {
        const float4 r = order[i];
        x[0] = r.x;
        x[1] = r.y;
        if (D > 2) x[D - 1] = r.z;
        return (long long)__float_as_uint(r.w);
    }
#pragma unroll
    for (int d = 0; d < D; ++d) x[d] = xin[i * D + d];
    return i;
}

// Gradient contributions of one point to one level: visits (entry index, weight) of every corner. Bit d of `turn` has the corners
// of dimension d visited far side first: lanes whose points share a cell then add to different entries in one instruction.
template <int D, typename Fn>
__device__ __forceinline__ void for_each_corner(const float (&x)[D], float scale, uint32_t size, uint32_t res, uint32_t flags,
                                                uint32_t hash_type, uint32_t interpolation, uint32_t turn, Fn &&fn) {
    uint32_t cell[D];
    float frac[D];
    cell_of<D>(x, scale, interpolation, cell, frac);
    if (interpolation == TNN_INTERP_NEAREST) {
        fn(level_index<D>(cell, size, res, flags, hash_type), 1.0f);
        return;
    }
    float side_weight[D][2];
    uint32_t side[D][2];
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const uint32_t far = (turn >> d) & 1;
        side_weight[d][0] = far ? frac[d] : 1 - frac[d];
        side_weight[d][1] = far ? 1 - frac[d] : frac[d];
        side[d][0] = cell[d] + far;
        side[d][1] = cell[d] + 1 - far;
    }
#pragma unroll
    for (int c = 0; c < (1 << D); ++c) {
        float weight = 1.0f;
        uint32_t loc[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            weight *= side_weight[d][(c >> d) & 1];
            loc[d] = side[d][(c >> d) & 1];
        }
        fn(level_index<D>(loc, size, res, flags, hash_type), weight);
    }
}

typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

// Adds the F gradient values of one table entry. fp32 tables: one atomic per value (the reference's grad_t). fp16 tables:
// one packed atomic (global_atomic_pk_add_f16) per pair of features, half as many atomic operations.
template <int F> __device__ __forceinline__ void add_entry(float *entry, const float (&v)[F]) {
#pragma unroll
    for (int f = 0; f < F; ++f) unsafeAtomicAdd(entry + f, v[f]);
}
template <int F> __device__ __forceinline__ void add_entry(fp16_t *entry, const float (&v)[F]) {
    static_assert(F % 2 == 0, "packed fp16 gradients need an even number of features per level");
#pragma unroll
    for (int f = 0; f < F; f += 2) {
        const f16x2_t pair = {(fp16_t)v[f], (fp16_t)v[f + 1]};
        (void)__builtin_amdgcn_flat_atomic_fadd_v2f16(reinterpret_cast<f16x2_t *>(entry + f), pair);
    }
}

// Lanes over the features of one entry on the direct route: one per value for an fp32 table, one per packed pair for fp16.
template <int F, typename GT> struct BackwardLanes { static constexpr int FL = F; };
template <int F> struct BackwardLanes<F, fp16_t> { static constexpr int FL = F / 2; };

// Lane i of a row of 16 lanes reads lane i - N (row_shr) or i + N (row_shl) of the same row; lanes without such a
// neighbour keep their own value.
template <int N> __device__ __forceinline__ int row_shr(int v) {
    if constexpr (N >= 16) return v;
    else return __builtin_amdgcn_update_dpp(v, v, 0x110 + N, 0xf, 0xf, false);
}
template <int N> __device__ __forceinline__ int row_shl(int v) {
    if constexpr (N >= 16) return v;
    else return __builtin_amdgcn_update_dpp(v, v, 0x100 + N, 0xf, 0xf, false);
}
// One step of a segmented inclusive sum inside rows of 16 lanes: lanes whose run is still open take the sum STEP lanes up.
template <int STEP, int FV> __device__ __forceinline__ void segmented_step(float (&v)[FV], bool &open, int rl) {
    const bool open_up = row_shr<STEP>((int)open) != 0;
    const bool reach = rl >= STEP;
#pragma unroll
    for (int f = 0; f < FV; ++f) {
        const float up = __int_as_float(row_shr<STEP>(__float_as_int(v[f])));
        v[f] += (reach && open) ? up : 0.0f;
    }
    open = reach ? (open && open_up) : open;
}

// Scatter-add of dL/dy into the gradient table (include/encodings/grid.h:137-245 of the reference: float atomics,
// order not defined). Two routes inside one launch:
//   * small levels (the coarse ones, where every point of the batch lands on a few hundred entries and global
//     atomics queue up on the same addresses): a workgroup adds the contributions of a chunk of points into a
//     private copy of the level in LDS and then issues one global atomic per touched entry;
//   * the other levels: a group of lanes per (point, level), atomics straight to the table; workgroups of one level
//     are dispatched together, so its slice of the table is the hot one in L2.
template <int D, int F, typename G, typename GT>
__global__ void __launch_bounds__(kBwdThreads)
    grid_backward_kernel(const GridLevels lv, const GridParams gp, const BackwardPlan bp, const GradLayout dl, const float *__restrict__ xin,
                         const float4 *__restrict__ order, const uint32_t *__restrict__ bin_start, const G *__restrict__ dLdy,
                         GT *__restrict__ grad, long long M) {
    extern __shared__ double priv[];
    const uint32_t n_small_blocks = bp.n_small * bp.small_blocks;
    // Workgroups start in the order of their numbers. Those of the LDS routes and those of the direct route are bound by
    // different things (LDS atomics; atomic requests to memory), so their numbers are interleaved in proportion: both kinds
    // are resident on every CU from the start, instead of one kind queueing behind the other.
    const uint32_t n_lds_blocks = n_small_blocks + bp.tiled_start[bp.n_tiled];
    // (Cell order only. In the caller's order the few long workgroups of the LDS route come first, as measured faster.)
    const uint32_t n_direct_before =
        order ? (uint32_t)(((unsigned long long)blockIdx.x * (gridDim.x - n_lds_blocks)) / gridDim.x) : (blockIdx.x < n_lds_blocks ? 0u : blockIdx.x - n_lds_blocks);
    const bool is_direct = order ? (uint32_t)(((unsigned long long)(blockIdx.x + 1) * (gridDim.x - n_lds_blocks)) / gridDim.x) != n_direct_before
                                 : blockIdx.x >= n_lds_blocks;
    const uint32_t lds_block = blockIdx.x - n_direct_before; // this workgroup's number among those of its kind
    if (!is_direct && lds_block < n_small_blocks) {
        // the features of the level this workgroup adds: all, or one where a copy of all of them does not fit
        const uint32_t part = lds_block / bp.small_blocks, l = bp.small_level[part];
        const uint32_t f_first = bp.small_feature[part] == kAllFeatures ? 0 : bp.small_feature[part];
        const uint32_t n_f = bp.small_feature[part] == kAllFeatures ? F : 1;
        const uint32_t size = lv.size[l], res = lv.resolution[l], flags = lv.flags[l];
        const float scale = lv.scale[l];
        for (uint32_t e = threadIdx.x; e < size * n_f; e += kBwdThreads) priv[e] = 0.0;
        __syncthreads();
        const long long first = (long long)(lds_block % bp.small_blocks) * bp.chunk;
        const long long last = first + bp.chunk < M ? first + bp.chunk : M;
        // In cell order the lanes of a wave take points a stripe apart: neighbours would queue up on one LDS address.
        const uint32_t wave_no = threadIdx.x / kGridWave, lane = threadIdx.x % kGridWave;
        const uint32_t start = order ? lane * (bp.chunk / kGridWave) + wave_no : threadIdx.x;
        const uint32_t step = order ? kBwdThreads / kGridWave : kBwdThreads, turns = bp.chunk / kBwdThreads;
        for (uint32_t t = 0; t < turns; ++t) {
            const long long i = first + start + (long long)t * step;
            if (i >= last) continue;
            float x[D];
            const long long row = load_point<D>(xin, order, i, x);
            const G *dy = dLdy + (dl.by_position ? i : row) * dl.row_stride + l * dl.level_stride + f_first;
            float gy[F];
#pragma unroll
            for (int f = 0; f < F; ++f)
                if (f < (int)n_f) gy[f] = (float)dy[f] * dl.scale;
            for_each_corner<D>(x, scale, size, res, flags, gp.hash_type, gp.interpolation, lane, [&](uint32_t idx, float w) {
#pragma unroll
                for (int f = 0; f < F; ++f)
                    if (f < (int)n_f) lds_add(&priv[f * size + idx], w * gy[f]);
            });
        }
        __syncthreads();
        GT *g = grad + (size_t)lv.offset[l] * F + f_first;
        if constexpr (std::is_same<GT, float>::value) {
            // neighbouring lanes take neighbouring values, so that the values of a 32-byte sector leave in one request
            for (uint32_t e = threadIdx.x; e < size * n_f; e += kBwdThreads) {
                const float v = (float)priv[n_f == F ? e % F * size + e / F : e];
                if (v != 0.0f) unsafeAtomicAdd(g + (n_f == F ? e : (size_t)e * F), v);
            }
        } else {
            for (uint32_t e = threadIdx.x; e < size; e += kBwdThreads) {
                float v[F];
                bool any = false;
#pragma unroll
                for (int f = 0; f < F; ++f) {
                    v[f] = (float)priv[f * size + e];
                    any |= v[f] != 0.0f;
                }
                if (any) add_entry<F>(g + (size_t)e * F, v);
            }
        }
        return;
    }
    if (!is_direct) {
        // Cell order, a level whose workgroups each take stretches of consecutive points of one row of the order's coarse
        // cells (grid_order.hip walks the coarse cells row by row, x fastest, and leaves the first position of every
        // coarse cell behind the records): such a stretch lies in a few neighbouring cells, so the corners it touches fill
        // a small box of the level's cells. The workgroup accumulates in a private copy of it in LDS (double),
        // and adds every touched entry to the table once. A stretch whose box does not fit (points far apart: the bins of
        // the points outside the unit cube, a sparse region) adds to the table directly.
        const uint32_t tb = lds_block - n_small_blocks;
        uint32_t ti = 0;
        while (ti + 1 < bp.n_tiled && tb >= bp.tiled_start[ti + 1]) ++ti;
        const uint32_t l = bp.tiled_level[ti];
        const uint32_t chunk = 1u << bp.tiled_chunk_log2[ti], pieces = bp.tiled_pieces[ti];
        const uint32_t rowno = (tb - bp.tiled_start[ti]) / pieces, piece = (tb - bp.tiled_start[ti]) % pieces;
        const uint32_t size = lv.size[l], res = lv.resolution[l], flags = lv.flags[l];
        const float scale = lv.scale[l];
        const long long row_first = bin_start[rowno * bp.bins_per_row];
        const long long row_end = rowno + 1 < bp.n_rows ? (long long)bin_start[(rowno + 1) * bp.bins_per_row] : M;
        // Eight neighbouring lanes take eight consecutive points, which share lines of the records and of dL/dy and lie in few cells, so that they
        // take the cell's corners each in another order; the next eight lanes are an eighth of the stretch further, in other cells
        // (2-D, 2^18 points: eight 35.3 us, one 36.4, 64 39.4; corners in the same order and one lane 40.7; 3-D, 2^20 points 151, 151, 149 and 165).
        constexpr uint32_t n_waves = kBwdThreads / kGridWave;
        const uint32_t stripe = chunk / kGridWave, wv = threadIdx.x / kGridWave, ln = threadIdx.x % kGridWave;
        GT *g = grad + (size_t)lv.offset[l] * F;
        for (long long first = row_first + (long long)piece * chunk; first < row_end; first += (long long)pieces * chunk) {
            const uint32_t count = (uint32_t)((first + chunk < row_end ? first + chunk : row_end) - first);
            // The cells the points of the coarse cells between the stretch's first and last can be in. Points outside the unit
            // cube are in an end cell of the order; what lies outside the box adds to the table directly.
            int lo[D];
            uint32_t ext[D];
            long long n_local = 1;
            {
                constexpr int bits = OrderBits<D>::coarse;
                const uint32_t c0 = quantise(order[first].x, bits), c1 = quantise(order[first + count - 1].x, bits);
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    const uint32_t from = d == 0 ? c0 : (rowno >> (bits * (d - 1))) & ((1u << bits) - 1), to = d == 0 ? c1 : from;
                    lo[d] = (int)floorf(__builtin_fmaf(scale, (float)from / (float)(1 << bits), 0.5f));
                    const int hi = (int)floorf(__builtin_fmaf(scale, (float)(to + 1) / (float)(1 << bits), 0.5f));
                    ext[d] = (uint32_t)(hi - lo[d] + 2); // the far corners are one cell further
                    n_local *= ext[d];
                }
            }
            const bool fits = n_local * F * (long long)sizeof(double) <= (long long)bp.budget;
            if (fits) {
                __syncthreads(); // the private copy of the stretch before is done with
                for (uint32_t e = threadIdx.x; e < (uint32_t)n_local * F; e += kBwdThreads) priv[e] = 0.0;
                __syncthreads();
            }
            for (uint32_t k = wv; k < stripe; k += n_waves) {
                const uint32_t pl = (ln / 8) * (stripe * 8) + k * 8 + ln % 8;
                if (pl >= count) continue;
                float x[D];
                const long long row = load_point<D>(xin, order, first + pl, x);
                const G *dy = dLdy + (dl.by_position ? first + pl : row) * dl.row_stride + l * dl.level_stride;
                float gy[F];
#pragma unroll
                for (int f = 0; f < F; ++f) gy[f] = (float)dy[f] * dl.scale;
                uint32_t cell[D];
                float frac[D];
                cell_of<D>(x, scale, gp.interpolation, cell, frac);
                bool inside = fits;
#pragma unroll
                for (int d = 0; d < D; ++d) inside &= (uint32_t)((int)cell[d] - lo[d]) < ext[d] - 1;
                float side_weight[D][2];
                uint32_t side[D][2], place[D][2], stride = 1;
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    const uint32_t far = (ln >> d) & 1; // (as for_each_corner)
                    side_weight[d][0] = far ? frac[d] : 1 - frac[d];
                    side_weight[d][1] = far ? 1 - frac[d] : frac[d];
                    side[d][0] = cell[d] + far;
                    side[d][1] = cell[d] + 1 - far;
                    place[d][0] = (uint32_t)((int)side[d][0] - lo[d]) * stride;
                    place[d][1] = (uint32_t)((int)side[d][1] - lo[d]) * stride;
                    stride *= ext[d];
                }
#pragma unroll
                for (int c = 0; c < (1 << D); ++c) {
                    float weight = 1.0f;
                    uint32_t loc[D], local = 0;
#pragma unroll
                    for (int d = 0; d < D; ++d) {
                        weight *= side_weight[d][(c >> d) & 1];
                        loc[d] = side[d][(c >> d) & 1];
                        local += place[d][(c >> d) & 1];
                    }
                    if (inside) {
#pragma unroll
                        for (int f = 0; f < F; ++f) lds_add(&priv[f * (uint32_t)n_local + local], weight * gy[f]);
                    } else {
                        float v[F];
#pragma unroll
                        for (int f = 0; f < F; ++f) v[f] = weight * gy[f];
                        add_entry<F>(g + (size_t)level_index<D>(loc, size, res, flags, gp.hash_type) * F, v);
                    }
                }
            }
            if (!fits) continue;
            __syncthreads();
            constexpr uint32_t VL = std::is_same<GT, float>::value ? F : 1; // lanes per entry (fp16 tables take features in pairs)
            for (uint32_t n = threadIdx.x; n < (uint32_t)n_local * VL; n += kBwdThreads) {
                const uint32_t e = n / VL;
                float v[F / VL];
                bool any = false;
#pragma unroll
                for (uint32_t f = 0; f < F / VL; ++f) {
                    v[f] = (float)priv[(n % VL + f) * (uint32_t)n_local + e];
                    any |= v[f] != 0.0f;
                }
                if (!any) continue;
                uint32_t loc[D], rest = e;
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    loc[d] = (uint32_t)(lo[d] + (int)(rest % ext[d]));
                    rest /= ext[d];
                }
                add_entry<F / VL>(g + (size_t)level_index<D>(loc, size, res, flags, gp.hash_type) * F + n % VL, v);
            }
        }
        return;
    }
    // A group of 2 * FL neighbouring lanes owns one (point, level): lane (dx, fl) adds feature fl (fp16 table: the pair of
    // features fl) of the corners on side dx of the cell along the first dimension. The memory side retires atomic
    // requests per 32-byte sector, about 20 * 10^9 a second, however many lanes of one instruction fall into the sector:
    // the features of an entry always do, and the two corners along the first dimension are neighbouring entries
    // wherever that dimension enters the index unhashed or the hash leaves it in the low bits.
    constexpr int FL = BackwardLanes<F, GT>::FL, LPI = 2 * FL;
    const uint32_t b = n_direct_before;
    const uint32_t l = bp.big_level[b / bp.big_blocks];
    // kDirectPasses groups of points per workgroup, one after the other: a workgroup that ended after two atomics per lane
    // left the launch bound by the rate at which workgroups are dispatched
    GT *const g = grad + (size_t)lv.offset[l] * F + (threadIdx.x % FL) * (F / FL);
    const uint32_t size = lv.size[l], res = lv.resolution[l], flags = lv.flags[l];
    for (int pass = 0; pass < kDirectPasses; ++pass) {
    const long long i_raw = ((long long)(b % bp.big_blocks) * kDirectPasses + pass) * (kBwdThreads / LPI) + threadIdx.x / LPI;
    const bool live = i_raw < M;
    if (i_raw - threadIdx.x / LPI >= M) break; // the whole workgroup is past the end
    if (!live && !order) continue;
    const long long i = live ? i_raw : M - 1; // in cell order every lane stays for the exchange between lanes below
    const int dx = (threadIdx.x % LPI) / FL, fl = threadIdx.x % FL;
    float x[D];
    const long long row = load_point<D>(xin, order, i, x);
    constexpr int FV = F / FL; // values per lane: 1 (fp32 table) or 2 (fp16 table)
    const G *dy = dLdy + (dl.by_position ? i : row) * dl.row_stride + l * dl.level_stride + fl * FV;
    float gy[FV];
#pragma unroll
    for (int f = 0; f < FV; ++f) gy[f] = live ? (float)dy[f] * dl.scale : 0.0f;
    uint32_t cell[D];
    float frac[D];
    cell_of<D>(x, lv.scale[l], gp.interpolation, cell, frac);
    if (gp.interpolation == TNN_INTERP_NEAREST) {
        if (dx == 0 && live) add_entry<FV>(g + (size_t)level_index<D>(cell, size, res, flags, gp.hash_type) * F, gy);
        continue;
    }
#pragma unroll
    for (int rest = 0; rest < (1 << (D - 1)); ++rest) {
        const int c = 2 * rest + dx; // same corner numbering and weight product as for_each_corner
        float weight = 1.0f;
        uint32_t loc[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if ((c & (1 << d)) == 0) {
                weight *= 1 - frac[d];
                loc[d] = cell[d];
            } else {
                weight *= frac[d];
                loc[d] = cell[d] + 1;
            }
        }
        float v[FV];
#pragma unroll
        for (int f = 0; f < FV; ++f) v[f] = weight * gy[f];
        const uint32_t idx = level_index<D>(loc, size, res, flags, gp.hash_type);
        if (order) {
            // Points in cell order: neighbouring groups of lanes often hold the same entry. Runs of equal entries inside a row
            // of 16 lanes are summed first (a segmented sum over the lanes LPI apart, which hold the same side and feature
            // of the next points) and the last lane of a run adds the total: one atomic per run instead of one per point.
            // Lanes exchange through DPP row shifts, not through the LDS crossbar, which the workgroups of the LDS routes
            // on the same CU keep busy with their atomics. The order of the additions is not defined in the reference
            // either (grid.h:215-243).
            const int rl = (int)(threadIdx.x % 16);
            const uint32_t idx_prev = (uint32_t)row_shr<LPI>((int)idx);
            bool open = rl >= LPI && idx_prev == idx; // this lane's run starts further up than the steps so far have reached
            if constexpr (LPI < 16) {
                segmented_step<LPI, FV>(v, open, rl);
                if constexpr (2 * LPI < 16) segmented_step<2 * LPI, FV>(v, open, rl);
                if constexpr (4 * LPI < 16) segmented_step<4 * LPI, FV>(v, open, rl);
                if constexpr (8 * LPI < 16) segmented_step<8 * LPI, FV>(v, open, rl);
            }
            const uint32_t idx_next = (uint32_t)row_shl<LPI>((int)idx);
            const bool last = rl + LPI >= 16 || idx_next != idx;
            if (last) add_entry<FV>(g + (size_t)idx * F, v);
        } else {
            add_entry<FV>(g + (size_t)idx * F, v);
        }
    }
    }
}

__global__ void __launch_bounds__(256) fill_zero_kernel(const ClearRange clear) { clear_range(clear, blockIdx.x, gridDim.x); }

int check_grid_desc(const tnn_grid_desc *d) {
    if (!d) return fail(TNN_ERR_INVALID_ARGUMENT, "desc is NULL");
    if (d->n_dims != 2 && d->n_dims != 3) return fail(TNN_ERR_UNSUPPORTED, "GridEncoding: n_dims_to_encode %u (2 or 3 are built)", d->n_dims);
    if (d->n_levels == 0 || d->n_levels > TNN_GRID_MAX_LEVELS)
        return fail(TNN_ERR_INVALID_ARGUMENT, "GridEncoding: n_levels %u must be at most MAX_N_LEVELS %d", d->n_levels, TNN_GRID_MAX_LEVELS);
    const uint32_t F = d->n_features_per_level;
    if (F != 1 && F != 2 && F != 4 && F != 8) return fail(TNN_ERR_INVALID_ARGUMENT, "GridEncoding: n_features_per_level must be 1, 2, 4, or 8.");
    if (d->param_dtype != TNN_FP32 && d->param_dtype != TNN_FP16) return fail(TNN_ERR_UNSUPPORTED, "table dtype %u", d->param_dtype);
    if (d->grid_type > TNN_GRID_TILED || d->hash_type > TNN_HASH_RNG || d->interpolation > TNN_INTERP_SMOOTHSTEP)
        return fail(TNN_ERR_INVALID_ARGUMENT, "invalid grid / hash / interpolation type");
    return TNN_OK;
}

template <int D, int F, typename P>
static int launch_grid_forward_o(const GridLevels &lv, const GridParams &gp, const float *x, const float4 *order, const void *table,
                                 void *out, int out_dtype, size_t M, hipStream_t s) {
    const unsigned blocks = (unsigned)((M + kGridThreads - 1) / kGridThreads);
    switch (out_dtype) {
    case TNN_FP32:
        TNN_LAUNCH((grid_forward_kernel<D, F, P, float>), dim3(blocks), dim3(kGridThreads), 0, s, lv, gp, x, order, (const P *)table,
                           (float *)out, (long long)M);
        break;
    case TNN_BF16:
        TNN_LAUNCH((grid_forward_kernel<D, F, P, bf16_t>), dim3(blocks), dim3(kGridThreads), 0, s, lv, gp, x, order, (const P *)table,
                           (bf16_t *)out, (long long)M);
        break;
    case TNN_FP16:
        TNN_LAUNCH((grid_forward_kernel<D, F, P, fp16_t>), dim3(blocks), dim3(kGridThreads), 0, s, lv, gp, x, order, (const P *)table,
                           (fp16_t *)out, (long long)M);
        break;
    default: return fail(TNN_ERR_UNSUPPORTED, "out_dtype %d", out_dtype);
    }
    return check_launch("grid_forward_kernel");
}

template <int D, int F>
static int launch_grid_forward_p(const tnn_grid_desc *d, const GridLevels &lv, const GridParams &gp, const float *x, const float4 *order,
                                 const void *table, void *out, int out_dtype, size_t M, hipStream_t s) {
    if (d->param_dtype == TNN_FP32) return launch_grid_forward_o<D, F, float>(lv, gp, x, order, table, out, out_dtype, M, s);
    return launch_grid_forward_o<D, F, fp16_t>(lv, gp, x, order, table, out, out_dtype, M, s);
}

// Coarse cells of the order along a dimension (grid_order.hip), and rows of them.
static uint32_t coarse_cells(uint32_t n_dims) { return n_dims == 2 ? 64 : 16; }

// Cell order: log2 of the points of a stretch whose box of the level's cells fits the LDS budget, -1 where none does or the level has too few points a
// cell for it (beyond that a box holds hardly more than one contribution per entry and saves no atomics). The order walks a lattice of 64^2 (16^3)
// coarse cells row by row, x fastest: with the points spread evenly a row holds M / 64 (M / 256) of them, and a stretch of C of these spans that share of the
// level's width plus a coarse cell, and one coarse cell in the other dimensions. A stretch that breaks the estimate is caught in the kernel.
// (Short stretches: many workgroups of some ten microseconds each spread over the CUs far more evenly than few long ones.) A level that has boxes has them in every larger batch.
static int boxed_chunk_log2(uint32_t resolution, uint32_t n_dims, uint32_t F, double min_per_cell, size_t M) {
    const double R = (double)resolution, coarse = (double)coarse_cells(n_dims), per_row = (double)M * coarse / 4096.0;
    if ((double)M / (n_dims == 2 ? R * R : R * R * R) < min_per_cell) return -1;
    for (int c = 10; c >= 9; --c) {
        const double share = std::min(1.0, (double)(1u << c) / std::max(per_row, 1.0));
        double cells = (share * R + R / coarse + 2.0) * (R / coarse + 2.0);
        if (n_dims == 3) cells *= R / coarse + 2.0;
        if (cells * F * sizeof(double) <= 0.9 * (double)kPrivateLdsBytesOrdered) return c;
    }
    return -1;
}

// From and up to how many points boxes do not pay beside bins. Where no level is copied whole either, as in three dimensions, and the bins take all, batches without boxes have no launch
// for them: optimisation step with the ordering, 3-D, us, with boxes / all levels binned: 16 levels of 2^15 entries, 2^12 points 59 / 49, 2^13 63 / 52, 2^15 85 / 71, 114 688 160 / 144; of
// 2^19 2^13 142 / 129, 2^15 165 / 150, 114 688 234 / 217; 8 levels of 2^17 entries 64 / 52, 77 / 65, 124 / 112; of 2^19 72 / 60, 89 / 73, 133 / 121, 2^18 184 / 190. (Where the bins refuse
// levels of too few points the launch stays: 16 levels of 2^19, 2^12 points 136 / 144. 2-D, where the coarsest levels are copied, 2^13 55 / 56, 2^16 77 / 82.)
// Points that crowd a part of the volume queue up on the few entries of coarse levels, which boxes hold as well as even ones, the more of them a cell has on the mean of the levels and the more of the levels are
// such. The scatter alone, all levels binned over boxes, 815 drawn grids of one and two features and batches of 2^12 to 122 000 points, on average, and how many are more than a tenth slower: up to
// two points a cell even ones 0.68 (none), a picture's rows 0.79 (1 %), normally distributed 0.77 (1 %), in a cube of half the side 0.76 (none), of a fifth 0.83 (6 %), of a twentieth 0.81 (9 %); two
// to six, 8 levels and more from 16 cells a side on, 0.75 (none), 0.94, 0.81, 0.87, 0.95, 1.13 (56 %: what lies in one of 8000 parts of the volume); fewer or coarser levels two to
// four 0.72, 0.98, 0.98, 0.92, 1.14, 0.94, beyond 0.85, 1.16, 1.21, 1.17, 1.41, 1.23, and these have boxes there. Records of four and eight features lose at either end: 8 levels of 2^19 entries, 2^13 even points
// 32 / 36 and 40 / 56, 2^15 in a cube of a twentieth 212 / 327 and 397 / 640; eight features, 6 small levels (base 8, scale 1.25), 2^16 points 65 / 95 and 294 / 1190.
// And up to as many points as take no more memory for it than 2^17 in the caller's order, which copy some levels (122 880 for 16 levels, one of them copied); smaller batches may take more
// than in the caller's order (8 levels of 2^19 entries, 2^13 points 9 MB and none; 8 small levels, base 11, scale 1.25, 10 828 points 12 MB and none).
struct NoBoxes {
    size_t from = 1, to = 0;
    bool operator()(size_t M) const { return M >= from && M <= to; }
};
// (`M`: for batches of that size and up alone; where there are none at all up to it, no plan is made.)
static NoBoxes no_boxes_for(const GridLevels &lv, const GridParams &gp, uint32_t n_dims, uint32_t F, size_t M = 0) {
    NoBoxes r;
    if (n_dims != 3 || F > 2 || gp.n_levels > kMaxBinned || M >= kMoreBinnedBelow) return r;
    uint32_t copied = 0, largest = 0, coarsest = ~0u;
    double per_cell = 0.0; // of one point, on all levels
    for (uint32_t l = 0; l < gp.n_levels; ++l) {
        const size_t feature_bytes = (size_t)lv.size[l] * sizeof(double);
        if (feature_bytes * F <= kCopiedBytesOrdered) return r;
        copied += feature_bytes <= kPrivateLdsBytes;
        largest = std::max(largest, lv.size[l]);
        coarsest = std::min(coarsest, lv.resolution[l]);
        const double R = (double)lv.resolution[l];
        per_cell += 1.0 / (R * R * R);
    }
    const double a_cell = gp.n_levels >= 8 && coarsest >= 16 ? 6.0 : 2.0;
    const size_t crowded = (size_t)std::min(a_cell * gp.n_levels / per_cell, (double)kMoreBinnedBelow);
    const size_t to = std::min({kMoreBinnedBelow * (gp.n_levels - copied) / gp.n_levels, kMoreBinnedBelow - 1, crowded});
    if (M > to) return r;
    BinPlan bins{};
    for (uint32_t l = 0; l < gp.n_levels; ++l)
        if (!bin_plan_add(&bins, l, lv, gp, n_dims, F, to)) return r;
    while (r.from < to && (r.from << (n_dims - 1)) < largest / 16) r.from *= 2; // (as bin_plan_add refuses them, to a power of two)
    r.to = to;
    return r;
}

// Binned from where the atomics it saves (one request per pair of corners, 20e9 a second) take longer than its two launches:
// 2^18 requests. (2-D, 11 such levels, 12 000 points: 20 us either way; 2^16 points: 42 against 95.)
static bool enough_to_bin(size_t M, uint32_t n_levels, uint32_t n_dims) { return ((unsigned long long)M * n_levels << (n_dims - 1)) >= (1ull << 18); }

// Which route every level takes: n_big levels are left for the direct one (bp->big_level), those of `bins` for the binned one
// (grid_binned.hip), which needs scratch memory and is planned for only when `bins` is given.
static BackwardPlan plan_backward(const GridLevels &lv, const GridParams &gp, uint32_t n_dims, uint32_t F, bool ordered, bool fp32_table, size_t M, BinPlan *bins,
                                  uint32_t *n_big_levels, uint32_t *lds, const NoBoxes *without = nullptr) { // (`without`: what no_boxes_for says of any batch)
    const int D = (int)n_dims;
    // A level goes the LDS route when its slice fits the budget and a chunk of points makes clearly more atomics
    // than the flush of the private copy does (chunk * 2^D contributions against `size` entries).
    BackwardPlan bp{};
    bp.chunk = kPrivateChunk;
    bp.budget = ordered ? kPrivateLdsBytesOrdered : kPrivateLdsBytes;
    const bool nearest = gp.interpolation == TNN_INTERP_NEAREST;
    const size_t per_chunk = (M < bp.chunk ? M : (size_t)bp.chunk) << (nearest ? 0 : D);
    uint32_t n_big = 0, lds_bytes = 0;
    const auto divide = [&](size_t contributions, size_t an_entry) {
        bp.n_small = n_big = lds_bytes = 0;
        for (uint32_t l = 0; l < gp.n_levels; ++l) {
            const size_t feature_bytes = (size_t)lv.size[l] * sizeof(double), bytes = feature_bytes * F;
            // (in cell order only the coarsest levels: the box of a stretch is far smaller than a level from 8 KiB on)
            const bool worth_it = per_chunk >= 2 * (size_t)lv.size[l] && contributions >= an_entry * (size_t)lv.size[l];
            if (worth_it && bytes <= (ordered ? kCopiedBytesOrdered : bp.budget)) {
                bp.small_feature[bp.n_small] = kAllFeatures;
                bp.small_level[bp.n_small++] = (uint8_t)l;
                if (bytes > lds_bytes) lds_bytes = (uint32_t)bytes;
            } else if (worth_it && !ordered && fp32_table && F == 2 && feature_bytes <= bp.budget && bp.n_small + 2 <= TNN_GRID_MAX_LEVELS) {
                for (uint32_t f = 0; f < F; ++f) {
                    bp.small_feature[bp.n_small] = (uint8_t)f;
                    bp.small_level[bp.n_small++] = (uint8_t)l;
                }
                if (feature_bytes > lds_bytes) lds_bytes = (uint32_t)feature_bytes;
            } else {
                bp.big_level[n_big++] = (uint8_t)l;
            }
        }
    };
    const auto bin_others = [&] { return bins && enough_to_bin(M, n_big, n_dims); };
    divide(0, 0);
    // Beside binned levels a copy of the whole level has to be worth its additions to the table, for the chunks of 1024 points that a batch is cut into
    // in the end: a level of more entries than a chunk has contributions is binned, too (whole scatter, 2-D, 2^16 points, 2^15 entries 37.8 -> 32.9 us;
    // 2^15 points, 2^19 entries 39.3 either way), and in three dimensions, where that leaves none as a rule and so a launch less, one of more than
    // a quarter as many (20 000 points 52 -> 42.5; 2^16 63.5 -> 54.5; 2^17 93 -> 94; with that rule in two
    // dimensions 2^16 points 35.9; points in a square or cube of 5 % of the side, which meet few of such a level's entries, 2^16 points 2-D 84 -> 72,
    // 3-D 312 -> 218, since crowded bins have copies of their sums, 120 and 393 without). The records of such levels take memory: batches that need more of it for them than 2^17 points do
    // without (16 levels in 3-D: 122 880 points), and that many and more, for which 2^18 points would gain 4 of 81, do not have them.
    if (!ordered && !nearest && bin_others() && gp.n_levels <= kMaxBinned) {
        const size_t without = n_big;
        divide(std::min<size_t>(M, 1024) << D, D == 2 ? 1 : 4);
        if (n_big > without) bp.more_up_to = std::min(kMoreBinnedBelow / 1024 * without / n_big * 1024, kMoreBinnedBelow - 1);
        if (M > bp.more_up_to) divide(0, 0);
    }
    // Cell order: of the other levels, those with boxes take the boxed route.
    if (ordered && gp.n_levels > 0 && !nearest && !(bin_others() && (without ? *without : no_boxes_for(lv, gp, n_dims, F, M))(M))) {
        bp.bins_per_row = coarse_cells(n_dims);
        bp.n_rows = 4096 / bp.bins_per_row;
        const double per_row = (double)M / bp.n_rows;
        uint32_t kept = 0;
        for (uint32_t i = 0; i < n_big; ++i) {
            const uint32_t l = bp.big_level[i];
            const int chunk_log2 = bp.n_tiled < kMaxTiled ? boxed_chunk_log2(lv.resolution[l], n_dims, F, bins ? kBoxedMinPerCellBinned : kBoxedMinPerCell, M) : -1;
            if (chunk_log2 >= 0) {
                const uint32_t pieces = (uint32_t)std::min(64.0, std::ceil(per_row / (double)(1u << chunk_log2)) + 1.0);
                bp.tiled_level[bp.n_tiled] = (uint8_t)l;
                bp.tiled_chunk_log2[bp.n_tiled] = (uint8_t)chunk_log2;
                bp.tiled_pieces[bp.n_tiled] = (uint8_t)pieces;
                bp.tiled_start[bp.n_tiled + 1] = bp.tiled_start[bp.n_tiled] + bp.n_rows * pieces;
                ++bp.n_tiled;
                if (bp.budget > lds_bytes) lds_bytes = bp.budget;
            } else {
                bp.big_level[kept++] = (uint8_t)l;
            }
        }
        n_big = kept;
    }
    // (few workgroups of the LDS route leave most of the chip idle: shorter ones then)
    while (bp.chunk > 1024 && (M / bp.chunk) * bp.n_small < 256) bp.chunk /= 2;
    bp.small_blocks = (uint32_t)((M + bp.chunk - 1) / bp.chunk);
    if (bins) *bins = BinPlan{};
    if (bin_others()) {
        uint32_t kept = 0;
        for (uint32_t i = 0; i < n_big; ++i)
            if (!bin_plan_add(bins, bp.big_level[i], lv, gp, n_dims, F, M)) bp.big_level[kept++] = bp.big_level[i];
        n_big = kept;
    }
    *n_big_levels = n_big;
    *lds = lds_bytes;
    return bp;
}

template <int D, int F, typename TAB>
static int launch_grid_backward_g(const GridLevels &lv, const GridParams &gp, BackwardPlan bp, const GradLayout &dl, uint32_t n_big, uint32_t lds_bytes, const float *x,
                                  const float4 *order, const void *dLdy, int dy_dtype, TAB *grad, size_t M, hipStream_t s) {
    constexpr int per_block = kDirectPasses * kBwdThreads / (2 * BackwardLanes<F, TAB>::FL); // (point, level) pairs per workgroup on the direct route
    bp.big_blocks = (uint32_t)((M + per_block - 1) / per_block);
    const uint32_t *bin_start =
        order ? reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(order) + order_record_bytes(M)) : nullptr;
    const unsigned long long blocks = (unsigned long long)bp.n_small * bp.small_blocks + bp.tiled_start[bp.n_tiled] + (unsigned long long)n_big * bp.big_blocks;
    if (blocks > 0x7fffffffull) return fail(TNN_ERR_UNSUPPORTED, "grid backward: batch too large for one launch");
    if (blocks == 0) return TNN_OK;
    const dim3 grid((unsigned)blocks);
#define TNN_BWD(GT)                                                                                                    \
    do {                                                                                                               \
        auto k = grid_backward_kernel<D, F, GT, TAB>;                                                                  \
        if (lds_bytes > 48 * 1024 &&                                                                                   \
            !reserve_lds(reinterpret_cast<const void *>(k), lds_bytes)) \
            return fail(TNN_ERR_HIP, "cannot reserve %u bytes of LDS", lds_bytes);                                     \
        TNN_LAUNCH(k, grid, dim3(kBwdThreads), lds_bytes, s, lv, gp, bp, dl, x, order, bin_start, (const GT *)dLdy, grad, (long long)M);    \
    } while (0)
    switch (dy_dtype) {
    case TNN_FP32: TNN_BWD(float); break;
    case TNN_BF16: TNN_BWD(bf16_t); break;
    case TNN_FP16: TNN_BWD(fp16_t); break;
    default: return fail(TNN_ERR_UNSUPPORTED, "dy_dtype %d", dy_dtype);
    }
#undef TNN_BWD
    return check_launch("grid_backward_kernel");
}

#define TNN_DISPATCH_DF(desc, CALL)                                                              \
    do {                                                                                         \
        const uint32_t F__ = (desc)->n_features_per_level;                                       \
        if ((desc)->n_dims == 2) {                                                               \
            constexpr int D_ = 2;                                                                \
            if (F__ == 1) { constexpr int F_ = 1; CALL; }                                        \
            else if (F__ == 2) { constexpr int F_ = 2; CALL; }                                   \
            else if (F__ == 4) { constexpr int F_ = 4; CALL; }                                   \
            else { constexpr int F_ = 8; CALL; }                                                 \
        } else {                                                                                 \
            constexpr int D_ = 3;                                                                \
            if (F__ == 1) { constexpr int F_ = 1; CALL; }                                        \
            else if (F__ == 2) { constexpr int F_ = 2; CALL; }                                   \
            else if (F__ == 4) { constexpr int F_ = 4; CALL; }                                   \
            else { constexpr int F_ = 8; CALL; }                                                 \
        }                                                                                        \
    } while (0)

} // namespace tnn

using namespace tnn;

TNN_API int tnn_grid_desc_init(tnn_grid_desc *desc, uint32_t n_dims, uint32_t n_levels, uint32_t n_features_per_level,
                               uint32_t log2_hashmap_size, uint32_t base_resolution, float per_level_scale,
                               uint32_t grid_type, uint32_t hash_type, uint32_t interpolation, uint32_t param_dtype) {
    if (!desc) return fail(TNN_ERR_INVALID_ARGUMENT, "desc is NULL");
    memset(desc, 0, sizeof(*desc));
    desc->n_dims = n_dims;
    desc->n_levels = n_levels;
    desc->n_features_per_level = n_features_per_level;
    desc->log2_hashmap_size = log2_hashmap_size;
    desc->base_resolution = base_resolution;
    desc->per_level_scale = per_level_scale;
    desc->grid_type = grid_type;
    desc->hash_type = hash_type;
    desc->interpolation = interpolation;
    desc->param_dtype = param_dtype;
    int rc = check_grid_desc(desc);
    if (rc) return rc;
    if (log2_hashmap_size > 31) return fail(TNN_ERR_INVALID_ARGUMENT, "log2_hashmap_size %u", log2_hashmap_size);
    if (base_resolution == 0 || !(per_level_scale > 0.0f)) return fail(TNN_ERR_INVALID_ARGUMENT, "base_resolution / per_level_scale");

    // include/encodings/grid.h:604-644 with grid_scale / grid_resolution (common_device.h:767-775)
    const float log2_pls = std::log2(per_level_scale);
    uint64_t offset = 0;
    for (uint32_t i = 0; i < n_levels; ++i) {
        const float scale = std::exp2((float)i * log2_pls) * (float)base_resolution - 1.0f;
        const uint32_t resolution = (uint32_t)std::ceil(scale) + 1u;
        const uint32_t max_params = UINT32_MAX / 2;
        uint32_t params_in_level;
        if (std::pow((float)resolution, (float)n_dims) > (float)max_params) {
            params_in_level = max_params;
        } else {
            params_in_level = 1;
            for (uint32_t k = 0; k < n_dims; ++k) params_in_level *= resolution;
        }
        params_in_level = (params_in_level + 7u) / 8u * 8u;
        if (grid_type == TNN_GRID_TILED) {
            uint32_t t = 1;
            for (uint32_t k = 0; k < n_dims; ++k) t *= base_resolution;
            if (t < params_in_level) params_in_level = t;
        } else if (grid_type == TNN_GRID_HASH) {
            const uint32_t t = 1u << log2_hashmap_size;
            if (t < params_in_level) params_in_level = t;
        }
        desc->offsets[i] = (uint32_t)offset;
        desc->scales[i] = scale;
        desc->resolutions[i] = resolution;
        offset += params_in_level;
        if (offset > UINT32_MAX) return fail(TNN_ERR_INVALID_ARGUMENT, "grid table exceeds 2^32 entries");
    }
    desc->offsets[n_levels] = (uint32_t)offset;
    return TNN_OK;
}

TNN_API size_t tnn_grid_n_params(const tnn_grid_desc *desc) {
    if (check_grid_desc(desc)) return 0;
    return (size_t)desc->offsets[desc->n_levels] * desc->n_features_per_level;
}

namespace tnn {
int grid_common(const tnn_grid_desc *desc, uint32_t padded_width, size_t M, GridLevels *lv, GridParams *gp) {
    int rc = check_grid_desc(desc);
    if (rc) return rc;
    // include/encodings/grid.h:665-677
    if (padded_width == 0) return fail(TNN_ERR_INVALID_ARGUMENT, "Can't have width == 0");
    if (padded_width < desc->n_levels * desc->n_features_per_level)
        return fail(TNN_ERR_INVALID_ARGUMENT, "Dimension mismatch grid encoding output: padded width %u < %u features", padded_width,
                    desc->n_levels * desc->n_features_per_level);
    if (M == 0) return fail(TNN_ERR_INVALID_ARGUMENT, "batch_size == 0");
    if (M > 0x7fffffffull * kGridThreads) return fail(TNN_ERR_INVALID_ARGUMENT, "batch too large");
    fill_levels(desc, lv);
    gp->n_levels = desc->n_levels;
    gp->hash_type = desc->hash_type;
    gp->interpolation = desc->interpolation;
    gp->padded_width = padded_width;
    return TNN_OK;
}
} // namespace tnn

TNN_API int tnn_grid_forward(const tnn_grid_desc *desc, const float *d_x, const void *d_table, void *d_out, int out_dtype,
                             uint32_t padded_width, size_t M, tnn_stream_t stream) {
    GridLevels lv;
    GridParams gp;
    int rc = grid_common(desc, padded_width, M, &lv, &gp);
    if (rc) return rc;
    if (!d_x || !d_table || !d_out) return fail(TNN_ERR_INVALID_ARGUMENT, "NULL pointer argument");
    if (grid_rows_direct(M)) return launch_grid_levels(desc, lv, gp, d_x, nullptr, d_table, d_out, out_dtype, padded_width, M, as_stream(stream));
    TNN_DISPATCH_DF(desc, rc = (launch_grid_forward_p<D_, F_>(desc, lv, gp, d_x, nullptr, d_table, d_out, out_dtype, M, as_stream(stream))));
    return rc;
}

TNN_API int tnn_grid_forward_ordered(const tnn_grid_desc *desc, const void *d_order, const void *d_table, void *d_out, int out_dtype,
                                     uint32_t padded_width, size_t M, tnn_stream_t stream) {
    GridLevels lv;
    GridParams gp;
    int rc = grid_common(desc, padded_width, M, &lv, &gp);
    if (rc) return rc;
    if (!d_order || !d_table || !d_out) return fail(TNN_ERR_INVALID_ARGUMENT, "NULL pointer argument");
    if (reinterpret_cast<uintptr_t>(d_order) & 15) return fail(TNN_ERR_INVALID_ARGUMENT, "d_order must be 16-byte aligned");
    if (grid_rows_direct(M))
        return launch_grid_levels(desc, lv, gp, nullptr, static_cast<const float4 *>(d_order), d_table, d_out, out_dtype, padded_width, M, as_stream(stream));
    TNN_DISPATCH_DF(desc, rc = (launch_grid_forward_p<D_, F_>(desc, lv, gp, nullptr, static_cast<const float4 *>(d_order), d_table, d_out,
                                                              out_dtype, M, as_stream(stream))));
    return rc;
}

namespace tnn {
// The binned levels are written whole: where they are the last ones, as the finest are, only what lies in front of them is cleared.
static ClearRange range_to_clear(const tnn_grid_desc *desc, const BinPlan &bins, void *d_grad_table, int grad_dtype) {
    size_t entries = desc->offsets[desc->n_levels];
    if (bins.n_levels && bins.at[0].level + bins.n_levels == desc->n_levels) entries = std::min<size_t>(entries, bins.at[0].offset);
    const size_t bytes = entries * desc->n_features_per_level * (grad_dtype == TNN_FP32 ? sizeof(float) : sizeof(fp16_t));
    ClearRange c;
    c.p = static_cast<float4 *>(d_grad_table);
    c.n4 = bytes / 16;
    c.n_tail = (uint32_t)((bytes - c.n4 * 16) / sizeof(float)); // level sizes are multiples of 8 entries: fp16 tables leave no tail
    return c;
}

int grid_backward_clear(const tnn_grid_desc *desc, bool ordered, bool with_workspace, void *d_grad_table, int grad_dtype, size_t M, ClearRange *clear) {
    GridLevels lv;
    GridParams gp;
    const int rc = grid_common(desc, desc->n_levels * desc->n_features_per_level, M, &lv, &gp);
    if (rc) return rc;
    if (reinterpret_cast<uintptr_t>(d_grad_table) & 15) return fail(TNN_ERR_INVALID_ARGUMENT, "d_grad_table must be 16-byte aligned");
    BinPlan bins{};
    uint32_t n_big, lds;
    const bool fp32 = grad_dtype == TNN_FP32;
    (void)plan_backward(lv, gp, desc->n_dims, desc->n_features_per_level, ordered, fp32, M, with_workspace && fp32 ? &bins : nullptr, &n_big, &lds);
    *clear = range_to_clear(desc, bins, d_grad_table, grad_dtype);
    return TNN_OK;
}

// d_x may be given beside d_order, for the routes that read the rows of a row-major dL/dy better in the caller's order.
int grid_backward_impl(const tnn_grid_desc *desc, const float *d_x, const float4 *d_order, const void *d_dLdy, int dy_dtype, uint32_t padded_width,
                       const GradLayout &dl, void *d_grad_table, int grad_dtype, int overwrite, size_t M, void *d_workspace, size_t workspace_bytes,
                       hipStream_t s, bool cleared, const ReduceInFront *front) {
    GridLevels lv;
    GridParams gp;
    int rc = grid_common(desc, padded_width, M, &lv, &gp);
    if (rc) return rc;
    if ((!d_x && !d_order) || !d_dLdy || !d_grad_table) return fail(TNN_ERR_INVALID_ARGUMENT, "NULL pointer argument");
    if (d_order && (reinterpret_cast<uintptr_t>(d_order) & 15)) return fail(TNN_ERR_INVALID_ARGUMENT, "d_order must be 16-byte aligned");
    if (grad_dtype != TNN_FP32 && grad_dtype != TNN_FP16) return fail(TNN_ERR_UNSUPPORTED, "gradient table dtype %d", grad_dtype);
    if (grad_dtype == TNN_FP16 && desc->n_features_per_level % 2 != 0)
        return fail(TNN_ERR_UNSUPPORTED, "fp16 gradient tables need an even number of features per level (features are added in pairs)");
    const uint32_t n_features = desc->n_features_per_level;
    // With scratch memory the levels of the direct route are binned instead; without, and in fp16 tables, they are not.
    BinPlan bins{};
    uint32_t n_big = 0, lds_bytes = 0;
    uintptr_t scratch = (reinterpret_cast<uintptr_t>(d_workspace) + 255) & ~(uintptr_t)255;
    const bool binned = d_workspace && grad_dtype == TNN_FP32;
    BackwardPlan bp = plan_backward(lv, gp, desc->n_dims, n_features, d_order != nullptr, grad_dtype == TNN_FP32, M, binned ? &bins : nullptr, &n_big, &lds_bytes);
    if (bins.n_levels && workspace_bytes < bin_scratch_bytes(bins, desc->n_dims, n_features) + (scratch - reinterpret_cast<uintptr_t>(d_workspace)))
        return fail(TNN_ERR_WORKSPACE, "grid backward: workspace of %zu bytes given, %zu needed", workspace_bytes, bin_scratch_bytes(bins, desc->n_dims, n_features) + 256);
    if (overwrite && (reinterpret_cast<uintptr_t>(d_grad_table) & 15)) return fail(TNN_ERR_INVALID_ARGUMENT, "d_grad_table must be 16-byte aligned");
    const auto launch_bins = [&](BinStage stage, const TrainReduce *reduce) {
        return launch_grid_binned(bins, gp, dl, desc->n_dims, n_features, d_x, d_x && !dl.by_position ? nullptr : d_order, d_dLdy, dy_dtype, (float *)d_grad_table, overwrite != 0, M,
                                  reinterpret_cast<void *>(scratch), s, stage, reduce);
    };
    const bool together = front && bins.n_levels && bins_take_reduction(bins, n_features, dy_dtype, M, *front->reduce);
    if (front && (rc = together ? launch_bins(kBinning, front->reduce) : front->launch(*front->reduce, s))) return rc;
    if (overwrite && !cleared) {
        // a fill kernel rather than a memset node, so the call can be captured into a HIP graph
        const ClearRange clear = range_to_clear(desc, bins, d_grad_table, grad_dtype);
        if (clear.n4 || clear.n_tail) {
            const size_t blocks = std::min<size_t>(4096, std::max<size_t>(4, (clear.n4 + 255) / 256));
            TNN_LAUNCH(fill_zero_kernel, dim3((unsigned)blocks), dim3(256), 0, s, clear);
            if ((rc = check_launch("fill_zero_kernel"))) return rc;
        }
    }
    if (grad_dtype == TNN_FP32) {
        TNN_DISPATCH_DF(desc, rc = (launch_grid_backward_g<D_, F_, float>(lv, gp, bp, dl, n_big, lds_bytes, d_x, d_order, d_dLdy, dy_dtype,
                                                                          (float *)d_grad_table, M, s)));
        if (rc == TNN_OK && bins.n_levels) rc = launch_bins(together ? kSums : kBinningAndSums, nullptr);
    } else {
        const uint32_t F = desc->n_features_per_level;
#define TNN_PACKED(D_, F_) \
    rc = launch_grid_backward_g<D_, F_, fp16_t>(lv, gp, bp, dl, n_big, lds_bytes, d_x, d_order, d_dLdy, dy_dtype, (fp16_t *)d_grad_table, M, s)
        if (desc->n_dims == 2) {
            if (F == 2) TNN_PACKED(2, 2); else if (F == 4) TNN_PACKED(2, 4); else TNN_PACKED(2, 8);
        } else {
            if (F == 2) TNN_PACKED(3, 2); else if (F == 4) TNN_PACKED(3, 4); else TNN_PACKED(3, 8);
        }
#undef TNN_PACKED
    }
    return rc;
}
} // namespace tnn

// A caller's row-major dL/dy.
static GradLayout rows_of(const tnn_grid_desc *desc, uint32_t padded_width) { return GradLayout{padded_width, desc ? desc->n_features_per_level : 0, 0, 1.0f}; }

TNN_API int tnn_grid_backward(const tnn_grid_desc *desc, const float *d_x, const void *d_dLdy, int dy_dtype,
                              uint32_t padded_width, float *d_grad_table, int overwrite, size_t M, tnn_stream_t stream) {
    return grid_backward_impl(desc, d_x, nullptr, d_dLdy, dy_dtype, padded_width, rows_of(desc, padded_width), d_grad_table, TNN_FP32, overwrite, M, nullptr, 0, as_stream(stream));
}

TNN_API int tnn_grid_backward_ordered(const tnn_grid_desc *desc, const void *d_order, const void *d_dLdy, int dy_dtype,
                                      uint32_t padded_width, float *d_grad_table, int overwrite, size_t M, tnn_stream_t stream) {
    if (!d_order) return tnn::fail(TNN_ERR_INVALID_ARGUMENT, "d_order is NULL");
    return grid_backward_impl(desc, nullptr, static_cast<const float4 *>(d_order), d_dLdy, dy_dtype, padded_width, rows_of(desc, padded_width), d_grad_table, TNN_FP32,
                              overwrite, M, nullptr, 0, as_stream(stream));
}

TNN_API size_t tnn_grid_backward_workspace_bytes(const tnn_grid_desc *desc, size_t M) {
    GridLevels lv;
    GridParams gp;
    if (check_grid_desc(desc) || grid_common(desc, desc->n_levels * desc->n_features_per_level, M, &lv, &gp)) return 0;
    // What holds a batch holds a smaller one: the most that any batch of up to M points needs, in either order.
    const uint32_t D = desc->n_dims, F = desc->n_features_per_level;
    size_t most = 0, most_points = 0; // (points times levels)
    uint32_t n_big, lds;
    BinPlan bins{};
    const bool followed = gp.n_levels <= kMaxBinned; // (of more levels than are ever binned as many as are are taken to be, at every size)
    if (followed) {
        // The caller's order: as many levels at every size, but more up to one size (plan_backward).
        const size_t more = plan_backward(lv, gp, D, F, false, true, M, &bins, &n_big, &lds).more_up_to;
        most = bin_scratch_bytes_up_to(bins, D, F);
        most_points = (size_t)bins.batch * bins.n_levels;
        if (more && M > more) {
            (void)plan_backward(lv, gp, D, F, false, true, more, &bins, &n_big, &lds);
            most = std::max(most, bin_scratch_bytes_up_to(bins, D, F));
        }
    }
    const NoBoxes without = no_boxes_for(lv, gp, D, F);
    const size_t no_boxes = M >= without.from ? without.to : 0; // (below `from` a batch has boxes and needs less)
    // Cell order: levels that are not copied leave the bins for boxes one by one as the batch grows, each at a size of its own.
    uint32_t n = 0, level[TNN_GRID_MAX_LEVELS], most_bins = 0;
    size_t boxed_from[TNN_GRID_MAX_LEVELS];
    for (uint32_t l = 0; l < gp.n_levels; ++l) {
        if ((size_t)lv.size[l] * F * sizeof(double) <= kCopiedBytesOrdered) continue;
        const double R = (double)lv.resolution[l], enough = std::ceil(kBoxedMinPerCellBinned * (D == 2 ? R * R : R * R * R));
        const auto boxed = [&](size_t points) {
            return boxed_chunk_log2(lv.resolution[l], D, F, kBoxedMinPerCellBinned, points) >= 0 && points > no_boxes;
        };
        level[n] = l;
        boxed_from[n] = ~(size_t)0;
        if (followed && enough <= (double)M) {
            size_t no = (size_t)enough - 1, yes = (size_t)enough;
            if (!boxed(yes)) { // (its boxes do not fit yet)
                no = yes;
                yes = boxed(M) ? M : boxed_from[n];
            }
            while (yes - no > 1 && yes <= M) (boxed((no + yes) / 2) ? yes : no) = (no + yes) / 2;
            boxed_from[n] = yes;
        }
        ++n;
    }
    bool is_binned[TNN_GRID_MAX_LEVELS];
    size_t asked = 0;
    const auto in_order = [&](size_t points) {
        if (points == asked) return; // (levels that have boxes from the same size on, as all do that batches without boxes hold back)
        asked = points;
        if (followed && points <= no_boxes) { // (the levels of one plan)
            (void)plan_backward(lv, gp, D, F, true, true, points, &bins, &n_big, &lds, &without);
            most = std::max(most, bin_scratch_bytes_up_to(bins, D, F));
            return;
        }
        const size_t batch = std::min(points, kBinBatch);
        uint32_t in_boxes = 0, others = 0, binned = 0;
        for (uint32_t i = 0; i < n; ++i) others += boxed_from[i] > points || in_boxes++ >= kMaxTiled;
        // (by a quarter fewer points and levels need less, whatever their workgroups and tables)
        if (!enough_to_bin(points, others, D) || (batch + 1024) * others * 4 <= most_points * 3) return;
        if (most_bins == 0) {
            for (uint32_t i = 0; i < n; ++i) {
                bins = BinPlan{};
                is_binned[i] = bin_plan_add(&bins, level[i], lv, gp, D, F, M);
                most_bins = std::max(most_bins, bins.room_bins);
            }
        }
        in_boxes = 0;
        for (uint32_t i = 0; i < n; ++i) binned += (boxed_from[i] > points || in_boxes++ >= kMaxTiled) && is_binned[i];
        bins.n_levels = std::min(binned, kMaxBinned);
        bins.room_bins = bins.n_levels * most_bins;
        bins.n_quads = (bins.room_bins + 3) / 4;
        bins.batch = (uint32_t)batch;
        most = std::max(most, bin_scratch_bytes_up_to(bins, D, F));
    };
    in_order(M);
    for (uint32_t i = 0; i < n; ++i)
        if (boxed_from[i] <= M && boxed_from[i] > 1) in_order(boxed_from[i] - 1);
    return most + 256;
}

TNN_API int tnn_grid_backward_wants_order(const tnn_grid_desc *desc, size_t M) {
    GridLevels lv;
    GridParams gp;
    if (check_grid_desc(desc) || grid_common(desc, desc->n_levels * desc->n_features_per_level, M, &lv, &gp)) return 0;
    // Where the bins take all levels they are as fast as the boxes of cell order, without the ordering. Where they refuse the finest
    // (tables beyond 2^21 entries of eight features, 2^23 of two), with x alone and with both, us, evenly spread points:
    // eight features, 2^22 entries, 2^17 points 990 and 960, 2^18 1512 and 1377, 2^20 4800 and 4054; two features, 2^24
    // entries 777 and 808, 1081 and 1091, 3059 and 2810. Nearest sends a point to one entry a level, and the caller's order is the
    // faster one at every size (3-D, 2^19 entries, 2^18 points 227 and 232, 2^20 862 and 859; 2-D 193 and 212, 775 and 945).
    if (gp.interpolation == TNN_INTERP_NEAREST || M < (size_t(1) << 18)) return 0;
    BinPlan bins{};
    uint32_t n_big, lds;
    (void)plan_backward(lv, gp, desc->n_dims, desc->n_features_per_level, false, true, M, &bins, &n_big, &lds);
    return n_big != 0;
}

TNN_API int tnn_grid_backward_binned(const tnn_grid_desc *desc, const float *d_x, const void *d_order, const void *d_dLdy, int dy_dtype,
                                     uint32_t padded_width, float *d_grad_table, int overwrite, size_t M, void *d_workspace, size_t workspace_bytes,
                                     tnn_stream_t stream) {
    if (!d_workspace) return tnn::fail(TNN_ERR_WORKSPACE, "grid backward: no workspace");
    return grid_backward_impl(desc, d_x, static_cast<const float4 *>(d_order), d_dLdy, dy_dtype, padded_width, rows_of(desc, padded_width), d_grad_table, TNN_FP32, overwrite,
                              M, d_workspace, workspace_bytes, as_stream(stream));
}

TNN_API int tnn_grid_backward_packed(const tnn_grid_desc *desc, const float *d_x, const void *d_dLdy, int dy_dtype,
                                     uint32_t padded_width, void *d_grad_table_f16, int overwrite, size_t M, tnn_stream_t stream) {
    return grid_backward_impl(desc, d_x, nullptr, d_dLdy, dy_dtype, padded_width, rows_of(desc, padded_width), d_grad_table_f16, TNN_FP16, overwrite, M, nullptr, 0, as_stream(stream));
}

TNN_API int tnn_grid_indices(const tnn_grid_desc *desc, const float *d_x, uint32_t *d_indices, size_t M, tnn_stream_t stream) {
    GridLevels lv;
    GridParams gp;
    int rc = grid_common(desc, desc ? desc->n_levels * desc->n_features_per_level : 0, M, &lv, &gp);
    if (rc) return rc;
    if (!d_x || !d_indices) return fail(TNN_ERR_INVALID_ARGUMENT, "NULL pointer argument");
    const unsigned blocks = (unsigned)((M + kGridThreads - 1) / kGridThreads);
    if (desc->n_dims == 2)
        TNN_LAUNCH((grid_indices_kernel<2>), dim3(blocks), dim3(kGridThreads), 0, as_stream(stream), lv, gp, d_x, d_indices, (long long)M);
    else
        TNN_LAUNCH((grid_indices_kernel<3>), dim3(blocks), dim3(kGridThreads), 0, as_stream(stream), lv, gp, d_x, d_indices, (long long)M);
    return check_launch("grid_indices_kernel");
}

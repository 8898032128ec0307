// Grid encoding level by level (gfx950).
//
// Reference behaviour being reproduced: include/encodings/grid.h:37-135 (kernel_grid; the same sums, bit for bit, as
// grid_forward_kernel). The reference, too, takes the levels as the slow dimension of its launch (:696-731).
//
// What bounds a gather is where its line comes from: lines of 128 bytes at random arrive 66 * 10^9 times a second from the memory
// side and 265 * 10^9 times from an XCD's own 4 MB of L2 (64 bytes a cycle and CU), whether 4, 8 or 16 bytes of a line are wanted.
// A kernel whose waves walk all levels of their points (grid_forward_kernel) has the whole table in use at once, in every XCD. Here
// an XCD takes a level at a time, for all points: its L2 holds that level, and a level is fetched by one or two XCDs instead of eight. Levels that L2 does
// not hold, and those of which a batch takes every line many times, all XCDs take one after the other, an eighth of the points each (shared_level).
// The corners of a cell along the first dimension lie in one line nearly always. Two loads of a lane fetch it twice, because
// the lines that a CU's waves have under way are many times what its vector cache holds; here two neighbouring lanes load the two
// corners of a row, of one's point and then of the other's, and exchange what they loaded.
// Measured, fp32 table and rows: 3-D, 16 levels, 2^19 entries, 2^20 points 253 us in cell order and 332 in the caller's (one load a lane: 547 and
// 534; all levels of a point in one thread: 519 and 754), of which the levels beyond L2's reach of a thread a point 455 -> 170 for eight of them;
// 2-D, 2^18 points 25.6 and 39 (42 and 76). 5001 points 3-D: 6 us (38).
// A batch that is small then has a wave for every level, too, and not one wave that walks through all of them.
#include "grid_levels.h"
#include "level_plan.h"

#include <algorithm>
#include <cmath>

namespace tnn {

constexpr int kLevelThreads = 256;

// Points of a thread. Few, so that a batch is many workgroups (us with 1, 2, 4 and 8 points a thread, 2-D: 20 000 points 5.0, 5.6, 6.3, 7.8; 2^16 10.8, 10.7,
// 11.5, 14.1; 2^18 29.4, 29.8, 32.0, 33.7, before two corners were one load), but two in three dimensions where the batch is large (2^20 points, one and two: 265, 254).
template <int D, int F, bool LARGE> struct LevelShape {
    static constexpr int kPoints = F > 4 ? 1 : D == 2 ? (F <= 2 ? 2 : 1) : LARGE ? 2 : 1;
    static constexpr int kChunk = kLevelThreads * kPoints; // points of a workgroup
};
constexpr size_t kLargeBatch = size_t(1) << 19;

// The neighbouring lane's value: lanes 2 k and 2 k + 1 exchange (DPP quad_perm).
__device__ __forceinline__ uint32_t swap_pair(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0xB1, 0xf, 0xf, false); }
__device__ __forceinline__ float swap_pair(float v) { return __uint_as_float(swap_pair(__float_as_uint(v))); }

// Entries of a cell's corners on one side of it along the first dimension (side 1: the far one): bit d - 1 of a row's number says which
// side of dimension d it lies on. The values of level_index.
template <int D>
__device__ __forceinline__ void row_entries(const uint32_t (&cell)[D], uint32_t side, uint32_t size, uint32_t res, uint32_t flags, uint32_t hash_type,
                                            uint32_t (&entry)[1 << (D - 1)]) {
    constexpr int R = 1 << (D - 1);
    const uint32_t x = cell[0] + side;
    if ((flags & 48u) == 48u && hash_type == TNN_HASH_COHERENT_PRIME) {
        const uint32_t y0 = cell[1] * 2654435761u, y1 = y0 + 2654435761u;
        const uint32_t z0 = D > 2 ? cell[D - 1] * 805459861u : 0u, z1 = z0 + 805459861u;
#pragma unroll
        for (int r = 0; r < R; ++r) entry[r] = (x ^ ((r & 1) ? y1 : y0) ^ (D > 2 ? ((r & 2) ? z1 : z0) : 0u)) & (size - 1);
    } else if ((flags & 31u) == (uint32_t)D) {
        const uint32_t first = D > 2 ? x + res * (cell[1] + res * cell[D - 1]) : x + res * cell[1];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            entry[r] = first + ((r & 1) ? res : 0u) + ((r & 2) ? res * res : 0u);
            if (flags & 32u) entry[r] &= size - 1;
            else if (entry[r] >= size) entry[r] %= size;
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            uint32_t loc[D];
            loc[0] = x;
#pragma unroll
            for (int d = 1; d < D; ++d) loc[d] = cell[d] + ((r >> (d - 1)) & 1);
            entry[r] = level_index<D>(loc, size, res, flags, hash_type);
        }
    }
}

// Whether the two corners of a row are neighbouring entries that one load takes: a level that is not hashed. In two dimensions, where most levels are not
// (2^18 points in cell order 27.8 -> 25.6 us; three dimensions, 2^20 points 242 -> 240, and 2^22 entries, 2^21 points 1116 -> 1125).
__host__ __device__ constexpr bool side_by_side(uint32_t n_dims, uint32_t flags, size_t entry_bytes) {
    return n_dims == 2 && entry_bytes >= 4 && entry_bytes <= 8 && (flags & 31u) == n_dims;
}
// Two neighbouring entries in one load (of an entry's alignment, which is at least 4 bytes).
template <typename P, int F> __device__ __forceinline__ void load_pair(const P *__restrict__ p, float (&near)[F], float (&far)[F]) {
    typedef P pair_t __attribute__((ext_vector_type(2 * F), aligned(F * sizeof(P))));
    const pair_t t = *reinterpret_cast<const pair_t *>(p);
#pragma unroll
    for (int f = 0; f < F; ++f) {
        near[f] = (float)t[f];
        far[f] = (float)t[F + f];
    }
}

// From what a lane loaded for the even and the odd lane's point to the near and the far corner of its own.
template <int F> __device__ __forceinline__ void exchange_corners(uint32_t side, float (&even)[F], float (&odd)[F]) {
#pragma unroll
    for (int f = 0; f < F; ++f) {
        const float mine = side ? odd[f] : even[f], other = swap_pair(side ? even[f] : odd[f]);
        even[f] = side ? other : mine;
        odd[f] = side ? mine : other;
    }
}

// The columns of the rows behind the encoding's (zeros, include/encodings/grid.h:682-694): 2^padding_shift lanes a row, in workgroups of their own. (With the
// last level's threads writing a row's padding each, 1000 rows of 128 columns with one to eight levels took 35 us in two dimensions; 4 this way, 5.5 to 8.5 in grid_forward_kernel.)
__host__ __device__ constexpr uint32_t padding_shift(uint32_t columns) {
    uint32_t shift = 0;
    while (shift < 6 && (1u << shift) < columns) ++shift;
    return shift;
}
template <typename O> __device__ __forceinline__ void clear_padding(O *__restrict__ out, uint32_t first, uint32_t padded_width, long long M, uint32_t block) {
    const uint32_t shift = padding_shift(padded_width - first), thread = block * kLevelThreads + threadIdx.x;
    const long long i = thread >> shift;
    if (i >= M) return;
    for (uint32_t c = first + (thread & ((1u << shift) - 1)); c < padded_width; c += 1u << shift) out[i * padded_width + c] = to_out<O>(0.0f);
}

template <int D, int F, typename P, typename O, bool ROWS, bool LARGE>
__global__ void __launch_bounds__(kLevelThreads)
    grid_levels_kernel(const GridLevels lv, const GridParams gp, const LevelPlan plan, const float *__restrict__ xin, const float4 *__restrict__ order,
                       const P *__restrict__ table, O *__restrict__ out, long long M, size_t pitch, uint32_t pad_from) {
    typedef LevelShape<D, F, LARGE> S;
    constexpr int U = S::kPoints, R = 1 << (D - 1); // R: rows of two corners along the first dimension
    typedef O ovec __attribute__((ext_vector_type(F)));
    if constexpr (ROWS) {
        if (blockIdx.x >= pad_from) {
            clear_padding<O>(out, gp.n_levels * F, gp.padded_width, M, blockIdx.x - pad_from);
            return;
        }
    }
    const uint32_t xcd = blockIdx.x % kXcds, turn = blockIdx.x / kXcds;
    uint32_t l, chunk;
    if (!plan_item(plan, gp.n_levels, xcd, turn, &l, &chunk)) return;
    const long long i0 = (long long)chunk * S::kChunk + threadIdx.x;
    const uint32_t size = lv.size[l], res = lv.resolution[l], flags = lv.flags[l];
    const float scale = lv.scale[l];
    const P *const level = table + (size_t)lv.offset[l] * F;
    const bool nearest = gp.interpolation == TNN_INTERP_NEAREST;
    const uint32_t side = threadIdx.x & 1;

    // (lanes past the end stay, as the last point's: their neighbours exchange with them)
    float x[U][D];
    uint32_t row[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const long long i = i0 + u * kLevelThreads < M ? i0 + u * kLevelThreads : M - 1;
        if (order) {
            const float4 r = order[i];
            x[u][0] = r.x;
            x[u][1] = r.y;
            if (D > 2) x[u][D - 1] = r.z;
            row[u] = __float_as_uint(r.w);
        } else {
#pragma unroll
            for (int d = 0; d < D; ++d) x[u][d] = xin[i * D + d];
        }
    }
    // of a row of corners: what this lane loads for the even and the odd lane's point, and then the near and the far corner of its own
    float even[U][R][F], odd[U][R][F], frac[U][D];
    // A level that is not hashed has the two corners side by side: one load for both, unless the index of any of the wave's wraps.
    bool together = side_by_side(D, flags, F * sizeof(P)) && !nearest;
    if (together) {
        uint32_t near[U][R];
        bool wraps = false;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            uint32_t cell[D];
            cell_of<D>(x[u], scale, gp.interpolation, cell, frac[u]);
            const uint32_t first = cell[0] + res * cell[1];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                near[u][r] = first + ((r & 1) ? res : 0u); // (two dimensions)
                wraps |= near[u][r] >= size - 1; // (a level has 8 entries and more)
            }
        }
        together = !__any(wraps);
        if (together) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int r = 0; r < R; ++r) load_pair<P, F>(level + (size_t)near[u][r] * F, even[u][r], odd[u][r]);
        }
    }
    if (!together) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            uint32_t cell[D], of_even[D], of_odd[D], a[R], b[R];
            cell_of<D>(x[u], scale, gp.interpolation, cell, frac[u]);
            if (nearest) {
                load_entry<P, F>(level + (size_t)level_index<D>(cell, size, res, flags, gp.hash_type) * F, even[u][0]);
                continue;
            }
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const uint32_t other = swap_pair(cell[d]);
                of_even[d] = side ? other : cell[d];
                of_odd[d] = side ? cell[d] : other;
            }
            row_entries<D>(of_even, side, size, res, flags, gp.hash_type, a);
            row_entries<D>(of_odd, side, size, res, flags, gp.hash_type, b);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                load_entry<P, F>(level + (size_t)a[r] * F, even[u][r]);
                load_entry<P, F>(level + (size_t)b[r] * F, odd[u][r]);
            }
        }
        if (D == 2 && !nearest) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int r = 0; r < R; ++r) exchange_corners<F>(side, even[u][r], odd[u][r]);
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const long long i = i0 + u * kLevelThreads;
        if (D == 3 && !nearest) { // (where they are first used)
#pragma unroll
            for (int r = 0; r < R; ++r) exchange_corners<F>(side, even[u][r], odd[u][r]);
        }
        ovec o;
#pragma unroll
        for (int f = 0; f < F; ++f) {
            float v = 0.0f;
            if (nearest) {
                v = even[u][0][f];
            } else {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    // the products and the order of encode_levels
                    float near_weight = 1 - frac[u][0], far_weight = frac[u][0];
#pragma unroll
                    for (int d = 1; d < D; ++d) {
                        const float w = (r & (1 << (d - 1))) ? frac[u][d] : 1 - frac[u][d];
                        near_weight *= w;
                        far_weight *= w;
                    }
                    v = __builtin_fmaf(near_weight, even[u][r][f], v);
                    v = __builtin_fmaf(far_weight, odd[u][r][f], v);
                }
            }
            o[f] = to_out<O>(as_fp32(v)); // (pinned as encode_levels pins it)
        }
        if (i >= (ROWS ? M : (long long)level_pitch(M))) continue;
        if constexpr (ROWS) {
            O *const to = out + (order ? (size_t)row[u] : (size_t)i) * gp.padded_width;
#pragma unroll
            for (int f = 0; f < F; ++f) to[l * F + f] = o[f];
        } else {
            __builtin_nontemporal_store(o, reinterpret_cast<ovec *>(out + ((size_t)l * pitch + i) * F));
            if (l + 1 == gp.n_levels)
                for (uint32_t p = l + 1; p < padded_levels(gp.n_levels, F); ++p) *reinterpret_cast<ovec *>(out + ((size_t)p * pitch + i) * F) = ovec{};
        }
    }
}

// Rows of the encoded matrix from the levels: a thread a piece of PER values, so that a wave writes whole lines. Bound by the bytes (3-D,
// 16 levels of two features, fp32, 2^20 points: 268 MB in 40 us in the caller's order; 61 in cell order, where a row's line is written apart from its neighbours').
template <int F, typename O>
__global__ void __launch_bounds__(256) grid_rows_kernel(const O *__restrict__ levels, const float4 *__restrict__ order, O *__restrict__ out, long long M, size_t pitch,
                                                        uint32_t n_levels, uint32_t padded_width) {
    constexpr uint32_t PER = 16 / sizeof(O), TOGETHER = F < (int)PER ? F : PER; // values of a piece; of those that lie side by side in `levels`
    typedef O piece_t __attribute__((ext_vector_type(PER)));
    typedef O part_t __attribute__((ext_vector_type(TOGETHER)));
    const uint32_t pieces = (padded_width + PER - 1) / PER;
    const bool whole = padded_width % PER == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    const long long n = M * pieces;
    for (long long t = (long long)blockIdx.x * 256 + threadIdx.x; t < n; t += (long long)gridDim.x * 256) {
        const long long i = t / pieces;
        const uint32_t c0 = (uint32_t)(t % pieces) * PER;
        piece_t v = {};
#pragma unroll
        for (uint32_t e = 0; e < PER; e += TOGETHER) {
            const uint32_t l = (c0 + e) / F, f = (c0 + e) % F;
            if (l >= n_levels) continue; // zero padding (include/encodings/grid.h:682-694)
            const part_t part = *reinterpret_cast<const part_t *>(levels + ((size_t)l * pitch + i) * F + f);
#pragma unroll
            for (uint32_t k = 0; k < TOGETHER; ++k) v[e + k] = part[k];
        }
        O *const to = out + (order ? (size_t)__float_as_uint(order[i].w) : (size_t)i) * padded_width + c0;
        if (whole) {
            *reinterpret_cast<piece_t *>(to) = v;
        } else {
#pragma unroll
            for (uint32_t e = 0; e < PER; ++e)
                if (c0 + e < padded_width) to[e] = v[e];
        }
    }
}

// What 2^23 points cost in a level, us: the loads, and the lines they miss in a CU's cache. `misses` in units of lines that come from L2, by the level's
// bytes: measured (3-D, 2^20 points) 32 KB 61 us, 95 KB 106, 281 KB 137, 2.7 MB 143, 4 MB 168, 8 MB 280, 24 MB 514, 32 MB 554, a few lines 49.
// In cell order the lanes of a wave share lines: 0.34 points a cell leave 0.13 of them (of 4 MB; 0.04 of 24 MB), 0.036 0.83 (0.49).
static double level_cost(const GridLevels &lv, uint32_t l, uint32_t n_dims, size_t entry_bytes, bool ordered, size_t M) {
    constexpr double at[][2] = {{14.0, 0.0}, {15.0, 0.13}, {16.6, 0.6}, {18.1, 0.93}, {21.4, 1.0}, {22.0, 1.26}, {23.0, 2.4}, {24.6, 4.9}, {25.0, 5.3}};
    constexpr int n = sizeof(at) / sizeof(at[0]);
    const double size = std::min(at[n - 1][0], std::max(at[0][0], std::log2((double)lv.size[l] * (double)entry_bytes)));
    int i = 1;
    while (i + 1 < n && size > at[i][0]) ++i;
    double misses = at[i - 1][1] + (at[i][1] - at[i - 1][1]) * (size - at[i - 1][0]) / (at[i][0] - at[i - 1][0]);
    if (ordered) {
        const double per_cell = (double)M / std::pow((double)lv.resolution[l], (double)n_dims);
        misses /= 1.0 + std::pow(per_cell / (0.1 * std::pow(1.26 / std::max(misses, 1.26), 0.73)), 1.5);
    }
    // (one load for two corners is worth most where lanes share lines: of a batch in the caller's order the lines are what a level costs)
    const bool pairs = ordered && side_by_side(n_dims, lv.flags[l], entry_bytes);
    return n_dims == 2 ? (pairs ? 18.0 : 29.0) + 43.0 * misses : 49.0 + 95.0 * misses;
}

// us a batch takes by levels (3-D, 2^19 entries, 2^20 points: 332 measured, 253 in cell order).
static double levels_us(const GridLevels &lv, uint32_t n_levels, uint32_t n_dims, size_t entry_bytes, bool ordered, size_t M) {
    double cost = 0.0;
    for (uint32_t l = 0; l < n_levels; ++l) cost += level_cost(lv, l, n_dims, entry_bytes, ordered, M);
    return cost * (double)M / (double)(1 << 23);
}

// One launch: the points [begin, begin + M) of a batch.
template <int D, int F, typename P, typename O>
static int launch_levels_part(const GridLevels &lv, const GridParams &gp, const float *x, const float4 *order, const void *table, O *out, bool rows, bool large,
                              size_t begin, size_t M, size_t batch, hipStream_t s) {
    LevelPlan plan;
    const size_t chunk = large ? LevelShape<D, F, D == 3>::kChunk : LevelShape<D, F, false>::kChunk;
    plan.n_chunks = (uint32_t)((M + chunk - 1) / chunk);
    double cost[TNN_GRID_MAX_LEVELS];
    for (uint32_t l = 0; l < gp.n_levels; ++l) cost[l] = level_cost(lv, l, D, F * sizeof(P), order != nullptr, batch);
    uint32_t n_own = gp.n_levels;
    while (n_own > 0 && shared_level(lv.size[n_own - 1], F * sizeof(P), D, batch)) --n_own;
    const uint32_t most = plan_shared_levels(cost, n_own, gp.n_levels, &plan);
    auto k = grid_levels_kernel<D, F, P, O, false, false>;
    if (rows) k = grid_levels_kernel<D, F, P, O, true, false>;
    if (large) k = grid_levels_kernel<D, F, P, O, false, D == 3>;
    const uint32_t padding = rows ? gp.padded_width - gp.n_levels * F : 0;
    const size_t pad_blocks = padding ? ((M << padding_shift(padding)) + kLevelThreads - 1) / kLevelThreads : 0;
    TNN_LAUNCH(k, dim3(most * kXcds + (unsigned)pad_blocks), dim3(kLevelThreads), 0, s, lv, gp, plan, x ? x + begin * D : nullptr, order ? order + begin : nullptr, (const P *)table,
               out + (rows ? 0 : begin * F), (long long)M, level_pitch(batch), most * kXcds);
    return check_launch("grid_levels_kernel");
}

template <int D, int F, typename P, typename O>
static int launch_levels(const GridLevels &lv, const GridParams &gp, const float *x, const float4 *order, const void *table, void *out, bool rows, size_t M,
                         hipStream_t s) {
    const bool large = D == 3 && M >= kLargeBatch && !rows;
    const size_t chunk = large ? LevelShape<D, F, D == 3>::kChunk : LevelShape<D, F, false>::kChunk;
    const size_t part = level_part_chunks(gp.n_levels, kLevelThreads) * chunk;
    if (rows && M > part) return fail(TNN_ERR_UNSUPPORTED, "grid encoding by levels: rows of small batches only");
    for (size_t begin = 0; begin < M; begin += part)
        if (const int rc = launch_levels_part<D, F, P, O>(lv, gp, x, order, table, (O *)out, rows, large, begin, std::min(part, M - begin), M, s))
            return rc;
    return TNN_OK;
}

int launch_grid_levels(const tnn_grid_desc *desc, const GridLevels &lv, const GridParams &gp, const float *x, const float4 *order, const void *table, void *out,
                       int out_dtype, uint32_t padded_width, size_t M, hipStream_t s) {
    GridParams p = gp;
    p.padded_width = padded_width;
#define TNN_LEVELS_O(D, F, P)                                                                                                                \
    switch (out_dtype) {                                                                                                                     \
    case TNN_FP32: return launch_levels<D, F, P, float>(lv, p, x, order, table, out, padded_width != 0, M, s);                               \
    case TNN_BF16: return launch_levels<D, F, P, bf16_t>(lv, p, x, order, table, out, padded_width != 0, M, s);                              \
    case TNN_FP16: return launch_levels<D, F, P, fp16_t>(lv, p, x, order, table, out, padded_width != 0, M, s);                              \
    default: return fail(TNN_ERR_UNSUPPORTED, "out_dtype %d", out_dtype);                                                                    \
    }
#define TNN_LEVELS_P(D, F)                                                                                                                   \
    if (desc->param_dtype == TNN_FP32) TNN_LEVELS_O(D, F, float)                                                                              \
    TNN_LEVELS_O(D, F, fp16_t)
#define TNN_LEVELS_F(D)                                                                                                                      \
    switch (desc->n_features_per_level) {                                                                                                    \
    case 1: TNN_LEVELS_P(D, 1)                                                                                                               \
    case 2: TNN_LEVELS_P(D, 2)                                                                                                               \
    case 4: TNN_LEVELS_P(D, 4)                                                                                                               \
    default: TNN_LEVELS_P(D, 8)                                                                                                              \
    }
    if (desc->n_dims == 2) { TNN_LEVELS_F(2) }
    TNN_LEVELS_F(3)
#undef TNN_LEVELS_F
#undef TNN_LEVELS_P
#undef TNN_LEVELS_O
}

bool grid_rows_direct(size_t M) { return M <= (size_t(1) << 14); }

template <typename O>
static int launch_rows(uint32_t F, const void *levels, const float4 *order, void *out, uint32_t n_levels, uint32_t padded_width, size_t M, hipStream_t s) {
    auto k = F == 1 ? grid_rows_kernel<1, O> : F == 2 ? grid_rows_kernel<2, O> : F == 4 ? grid_rows_kernel<4, O> : grid_rows_kernel<8, O>;
    const size_t pieces = M * ((padded_width * sizeof(O) + 15) / 16);
    TNN_LAUNCH(k, dim3((unsigned)std::min<size_t>((pieces + 255) / 256, size_t(1) << 20)), dim3(256), 0, s, (const O *)levels, order, (O *)out, (long long)M, level_pitch(M), n_levels,
               padded_width);
    return check_launch("grid_rows_kernel");
}

} // namespace tnn

using namespace tnn;

static size_t dtype_bytes(int dtype) { return dtype == TNN_FP32 ? 4 : 2; }
static size_t entry_bytes(const tnn_grid_desc *desc) { return desc->n_features_per_level * dtype_bytes(desc->param_dtype); }

size_t tnn::level_bytes(const tnn_grid_desc *desc, uint32_t l) { return (size_t)(desc->offsets[l + 1] - desc->offsets[l]) * entry_bytes(desc); }

size_t tnn::largest_level_bytes(const tnn_grid_desc *desc) {
    size_t bytes = 0;
    for (uint32_t l = 0; l < desc->n_levels; ++l) bytes = std::max(bytes, tnn::level_bytes(desc, l));
    return bytes;
}

// Whether M points (more than rows are written directly for) are faster by levels and a pass for the rows than by the kernel that walks all levels of a point.
// Two launches and a scratch allocation are 11 us through the module however little there is to do, the one kernel 7; beyond that it takes a level's gathers
// after another's, 0.7 us each in two dimensions and 1.4 in three where lines come from L2, up to 2.6 where they do not, as long as a CU's waves hold the batch
// (2^16 points), and puts points in cell order from 2^18 on. Points of a picture's rows share lines as they walk nearly as well as by levels (16 levels of 2^19 entries,
// us, walking / by levels: 2-D, 2^15 points 15 / 15, 2^17 25 / 30, 2^18 55 / 45; 3-D, 2^15 31 / 17, 2^17 38 / 37, 2^20 192 / 275, scattered 569 / 353); which they are is not
// known here, and an encoding on its own stands in front of a model whose points are scattered. Drawn for such points (16028 configurations: 0.83 of the walking kernel's time on average,
// 1 % more than a tenth longer; rows 0.96, 18 %) (fp32, two features unless said otherwise):
static bool levels_pay(const tnn_grid_desc *desc, size_t M) {
    const uint32_t L = desc->n_levels, F = desc->n_features_per_level;
    const size_t largest = tnn::largest_level_bytes(desc);
    uint32_t n_large = 0, n_fine = 0; // levels of 1 MB and more; levels with no more than a point a cell
    for (uint32_t l = 0; l < L; ++l) {
        n_large += (desc->offsets[l + 1] - desc->offsets[l]) * entry_bytes(desc) >= (size_t(1) << 20);
        const double side = desc->resolutions[l];
        n_fine += side * side * (desc->n_dims == 3 ? side : 1.0) >= (double)M;
    }
    if (desc->n_dims == 2) {
        // Lines of eight features: 8 levels 15 / 20 (2^16 points), 52 / 62 (2^18); 16 levels 28 / 21 (2^15), 66 / 84 (100 000), 110 / 180 (2^18).
        if (F == 8 && L > 4) return L > 12 && M <= (size_t(1) << 15);
        // 32 MB a level, 16 levels: 20 / 15 (24 000 points), 27 / 31 (2^16), 74 / 98 (2^18).
        if (largest > (size_t(8) << 20)) return L > 8 && M < (size_t(1) << 15);
        // 8 levels of up to 600 KB: 7 / 11 (2^14 points), 12 / 15 (2^17), 20 / 19 (200 000), 35 / 24 (2^18, ordered); three of 4 MB: 33 / 24 (200 000).
        // 12 levels of up to 128 KB: 10 / 11, 19 / 23, 32 / 32, 41 / 40; of up to 4 MB 12 / 11, 25 / 25, 48 / 34, 42 / 42. 16 levels: 13 / 11 to 46 / 36 and 20 / 13 to 80 / 45.
        if (M < (size_t(1) << 18)) return L > 12 || (n_large >= 3 && (L > 8 || M > (size_t(1) << 16)));
        // Ordered points of levels with many of them a cell share lines as they walk: 2^19 points, finest level 820 a side 70 / 79, 1956 66 / 77, 7006 96 / 94, 524288 106 / 87;
        // 12 levels of up to 1384 61 / 71. 8 levels 51 / 41. From 2^19 on 169 / 190 (2^20 points).
        return M < (size_t(3) << 17) || (M < (size_t(1) << 19) && (L <= 8 || 8 * n_fine >= 3 * L));
    }
    // 32 MB a level, 16 levels: 42 / 30 (24 000 points), 64 / 63 (2^16), 111 / 93 (100 000), 224 / 237 (2^18); 8 levels 21 / 20, 25 / 26, 39 / 37, 61 / 69.
    if (largest > (size_t(16) << 20)) return L > 4 && M < (size_t(1) << (L > 12 ? 17 : 16));
    // 4 levels: 7 / 11 (2^14 points), 11 / 13 (100 000), 16 / 16 (150 000), 37 / 22 (2^18, ordered), 49 / 39.
    if (L <= 4) return M >= (size_t(1) << 18) && M < (size_t(7) << 16);
    // Eight features, 16 levels of up to 16 MB: 59 / 51 (2^15 points), 79 / 89 (2^16), 139 / 130 (100 000), 313 / 449 (2^18); of 512 KB 47 / 27, 45 / 46, 92 / 63, 176 / 152;
    // 8 levels of up to 16 MB 70 / 75 (2^17), 100 / 126.
    const size_t widest = M >= (size_t(1) << 18) ? 2 : L > 8 ? 16 : 8; // MB
    if (F == 8 && M > (size_t(1) << 15) && (M <= (size_t(1) << 16) || largest > widest << 20)) return false;
    // 8 levels of up to 128 KB: 11 / 11 (2^14 points), 13 / 15 (2^16), 24 / 21 (2^17), 50 / 38 (2^18); of up to 1 MB 17 / 11, 19 / 15, 32 / 25, 54 / 44. 16 levels: 22 / 11 to 100 / 71,
    // 41 / 16 to 173 / 100.
    if (M <= (size_t(1) << 16)) return L > 8 || largest >= (size_t(1) << 19);
    // 16 MB a level: 116 / 90 (200 000 points), 161 / 157 (2^18), 270 / 303 (2^19).
    // As in two dimensions: 2^19 points, 8 levels, finest 212 a side 80 / 89, 2048 144 / 94; 16 levels, 4058 303 / 196; 2^20 points 569 / 353, 8 levels 140 / 146.
    return M < (size_t(7) << 16) || (largest <= (size_t(8) << 20) && 2 * n_fine >= L);
}

TNN_API size_t tnn_grid_forward_workspace_bytes(const tnn_grid_desc *desc, int out_dtype, size_t M) {
    if (check_grid_desc(desc) || M == 0 || grid_rows_direct(M) || !levels_pay(desc, M)) return 0;
    return levels_elements(desc, M) * dtype_bytes(out_dtype) + 256;
}

TNN_API int tnn_grid_levels_want_order(const tnn_grid_desc *desc, size_t M) {
    GridLevels lv;
    GridParams gp;
    if (check_grid_desc(desc) || grid_common(desc, desc->n_levels * desc->n_features_per_level, M, &lv, &gp)) return 0;
    if (M < (size_t(1) << 18)) return 0;
    const double ordering = 17.0 + 25.0 * (double)M / (double)(1 << 20); // us (2^18 points 21, 2^20 46, 2^21 65)
    return levels_us(lv, gp.n_levels, desc->n_dims, entry_bytes(desc), false, M) - levels_us(lv, gp.n_levels, desc->n_dims, entry_bytes(desc), true, M) > ordering;
}

TNN_API int tnn_grid_forward_by_level(const tnn_grid_desc *desc, const float *d_x, const void *d_order, const void *d_table, void *d_out, int out_dtype, uint32_t padded_width,
                                      size_t M, void *d_workspace, size_t workspace_bytes, tnn_stream_t stream) {
    GridLevels lv;
    GridParams gp;
    int rc = grid_common(desc, padded_width, M, &lv, &gp);
    if (rc) return rc;
    if ((!d_x && !d_order) || !d_table || !d_out) return fail(TNN_ERR_INVALID_ARGUMENT, "NULL pointer argument");
    if (reinterpret_cast<uintptr_t>(d_order) & 15) return fail(TNN_ERR_INVALID_ARGUMENT, "d_order must be 16-byte aligned");
    if (out_dtype != TNN_FP32 && out_dtype != TNN_BF16 && out_dtype != TNN_FP16) return fail(TNN_ERR_UNSUPPORTED, "out_dtype %d", out_dtype);
    const uintptr_t base = (reinterpret_cast<uintptr_t>(d_workspace) + 255) & ~(uintptr_t)255;
    const size_t need = levels_elements(desc, M) * dtype_bytes(out_dtype) + (base - reinterpret_cast<uintptr_t>(d_workspace));
    if (!d_workspace || workspace_bytes < need) return fail(TNN_ERR_WORKSPACE, "workspace of %zu bytes given, %zu needed", workspace_bytes, need);
    const float4 *order = static_cast<const float4 *>(d_order);
    void *levels = reinterpret_cast<void *>(base);
    hipStream_t s = as_stream(stream);
    if ((rc = launch_grid_levels(desc, lv, gp, d_x, order, d_table, levels, out_dtype, 0, M, s))) return rc;
    const uint32_t F = desc->n_features_per_level;
    if (out_dtype == TNN_FP32) return launch_rows<float>(F, levels, order, d_out, desc->n_levels, padded_width, M, s);
    if (out_dtype == TNN_BF16) return launch_rows<bf16_t>(F, levels, order, d_out, desc->n_levels, padded_width, M, s);
    return launch_rows<fp16_t>(F, levels, order, d_out, desc->n_levels, padded_width, M, s);
}

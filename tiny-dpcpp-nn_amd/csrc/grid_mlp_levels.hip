// Forward pass of a network behind a grid encoding, by levels: the encoding level by level (grid_levels.hip), then a kernel of the network that reads
// the levels. C entry points of that pass and of the backward pass on the levels it leaves.
//
// Reference behaviour being reproduced: dpcpp_bindings/tiny_dpcpp_nn/modules.py:357-421, as grid_mlp.inc does in one kernel; the values are
// the same, bit for bit. The one kernel moves fewer bytes, but its gathers are as the encoding of all levels of a point has them: lines from the memory
// side, two waves a SIMD to wait for them. (2-D, 16 levels, 2^19 entries, fp32 table, 2^18 points in cell order, two hidden layers of 64: 45.5 us; 27 and 15
// this way. 3-D, 3000 points: 37 and 6 + 6.)
#include "grid_levels.h"
#include "mlp_tile.h"

#include <algorithm>

namespace tnn {
int make_weight_push(const tnn_mlp_desc *desc, const void *src, int unpadded_input_width, int unpadded_output_width, int use_bias, void *packed, void *packed_t,
                     void *fwd, void *bwd, WeightPush *p); // mlp.hip

constexpr int kLevelsMlpThreads = 512;

// A wave owns a tile of 32 points; it asks for the next one's levels while it computes. Weights in LDS. Bound by the bytes and, in a small batch, by
// the latency of one tile after the weights.
template <typename T, int W, int F>
__global__ void __launch_bounds__(kLevelsMlpThreads, W == 128 ? 2 : 4)
    levels_mlp_kernel(const T *__restrict__ levels, size_t pitch, uint32_t n_levels, const float4 *__restrict__ order, const typename Storage<T>::vec8 *__restrict__ wprep,
                      T *__restrict__ out, int n_mats, int act, int out_act, long long M, int y_cols, const WeightPush push) {
    typedef Tile<T, W> TL;
    typedef typename Storage<T>::vec8 vec8;
    constexpr int NK = TL::NK, NI = TL::NI;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    vec8 *lds_w = reinterpret_cast<vec8 *>(smem_raw);
    if ((int)blockIdx.x >= push.blocks) { // (only with a push: a workgroup beside those that compute)
        push_copies<T, W>(push, n_mats);
        return;
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 31, h = lane >> 5;
    const long long n_tiles = (M + 31) / 32, stride = (long long)push.blocks * (blockDim.x >> 6);
    long long tile = (long long)blockIdx.x * (blockDim.x >> 6) + wave;
    vec8 nxt[NK];
    uint32_t next_row = 0;
    auto request = [&](const long long t) __attribute__((always_inline)) {
        const long long i = t * 32 + j < M ? t * 32 + j : M - 1;
        load_level_pieces<T, W, F>(nxt, levels, pitch, n_levels, (size_t)t * 32, j, h);
        next_row = order ? __float_as_uint(order[i].w) : (uint32_t)i;
    };
    if (tile < n_tiles) request(tile);
    stage_weights<T, W>(lds_w, wprep, n_mats, push);
    if (push.master) push_copies<T, W>(push, n_mats);
    while (tile < n_tiles) {
        const bool valid = tile * 32 + j < M;
        const long long row = order ? (long long)next_row : tile * 32 + j;
        vec8 cur[NK];
#pragma unroll
        for (int kb = 0; kb < NK; ++kb) {
            cur[kb] = nxt[kb];
            asm volatile("" : "+v"(cur[kb])); // (waited for here, before the next tile's are asked for)
        }
        tile += stride;
        if (tile < n_tiles) request(tile);
        f32x16 acc[NI];
        for (int l = 0; l < n_mats - 1; ++l) {
            TL::template matmul<true>(acc, cur, lds_w, wprep, l, lane);
            TL::repack_rt(cur, acc, act);
        }
        TL::template matmul<true>(acc, cur, lds_w, wprep, n_mats - 1, lane);
        TL::repack_rt(cur, acc, out_act);
        if (y_cols < W)
            TL::store_columns(cur, out, y_cols, row, h, valid);
        else
            TL::store(cur, out, row, h, valid);
    }
}

template <typename T, int W, int F>
static int launch_levels_mlp(const tnn_mlp_desc *mlp, const void *levels, uint32_t n_levels, const float4 *order, const void *wprep, void *y, int y_cols, size_t M,
                             WeightPush push, hipStream_t s) {
    typedef typename Storage<T>::vec8 vec8;
    const int n_mats = mlp->n_hidden_layers + 1;
    const size_t lds = prepared_elems(mlp) * sizeof(T); // checked against the device by the caller
    auto k = levels_mlp_kernel<T, W, F>;
    if (!reserve_lds(reinterpret_cast<const void *>(k), lds)) return fail(TNN_ERR_HIP, "cannot reserve %zu bytes of LDS", lds);
    const int per_cu = resident_per_cu(reinterpret_cast<const void *>(k), kLevelsMlpThreads, lds);
    const long long tiles = ((long long)M + 31) / 32, per_block = kLevelsMlpThreads / 64;
    const long long blocks = std::min((tiles + per_block - 1) / per_block, (long long)device_info().n_cu * per_cu);
    const int grid = push_grid(&push, (int)blocks, kLevelsMlpThreads, prepared_elems(mlp));
    TNN_LAUNCH(k, dim3((unsigned)grid), dim3(kLevelsMlpThreads), lds, s, (const T *)levels, level_pitch(M), n_levels, order, (const vec8 *)wprep, (T *)y, n_mats,
               mlp->activation, mlp->output_activation, (long long)M, y_cols, push);
    return check_launch("levels_mlp_kernel");
}

template <typename T>
static int launch_levels_mlp_w(const tnn_grid_desc *grid, const tnn_mlp_desc *mlp, const void *levels, const float4 *order, const void *wprep, void *y, int y_cols,
                               size_t M, const WeightPush &push, hipStream_t s) {
#define TNN_LM(W, F) return launch_levels_mlp<T, W, F>(mlp, levels, grid->n_levels, order, wprep, y, y_cols, M, push, s)
#define TNN_LM_F(W)                                 \
    switch (grid->n_features_per_level) {           \
    case 1: TNN_LM(W, 1);                           \
    case 2: TNN_LM(W, 2);                           \
    case 4: TNN_LM(W, 4);                           \
    default: TNN_LM(W, 8);                          \
    }
    switch (mlp->width) {
    case 16: TNN_LM_F(16)
    case 32: TNN_LM_F(32)
    case 64: TNN_LM_F(64)
    default: TNN_LM_F(128)
    }
#undef TNN_LM_F
#undef TNN_LM
}

} // namespace tnn

using namespace tnn;

TNN_API size_t tnn_grid_levels_bytes(const tnn_grid_desc *grid, size_t M) {
    return check_grid_desc(grid) || M == 0 ? 0 : levels_elements(grid, M) * 2;
}

// Whether M points are faster by levels. That is two launches and a scratch allocation, 11.7 us through the module however few the points are; one kernel is 8 us, and takes
// a tile's gathers in a row: more with each level and corner, least at small widths, whose registers leave a SIMD more waves. From 2^18 points on it has them in cell order first. Points of a
// picture's rows share their lines of the table in one kernel as well as by levels or better, scattered ones do not, and which they are is not known here: by levels where
// neither is slower. Drawn over 11898 configurations (dimensions, levels, features, width, table, resolutions, points; one kernel / levels, us, scattered points and a picture's rows). With this
// rule 1.0 % of them are more than 10 % slower than one kernel for one or the other; on average they take 0.76 of its time, rows 0.78 (the faster one each time 0.72 and 0.77; a rule
// that looked at dimensions, points and levels only 0.81 and 0.85, and 6.8 % were slower).
static bool levels_pay(const tnn_grid_desc *grid, int width, size_t M) {
    const uint32_t D = grid->n_dims, L = grid->n_levels, F = grid->n_features_per_level;
    const size_t largest = largest_level_bytes(grid), MB = size_t(1) << 20;
    // The constants of so many levels do not fit one kernel's scalar registers: 3-D, width 128, two features 25 000 of its 100 000 instructions read and write lanes for them, and by levels
    // takes 0.05 to 0.23 of its time; width 64, one feature 5 000 of 33 000, 0.3.
    if (width == 128 && F <= (D == 3 ? 2u : 1u)) return true;
    if (width == 64 && F == 1 && D == 3) return true;
    if (D == 2) {
        // Width 64, two features. 8 levels of up to 1 MB: 2^18 points 40 / 21, 2^20 0.75 of the time and 0.63; 12 levels 2^20 1.10 and 0.79; 16 levels 2^18 0.78 and 0.69, beyond 2^19 1.16 and 1.12;
        // of up to 8 MB 0.89 and 0.71, beyond 2^19 1.18 and 1.09; beyond 8 MB 1.1 to 1.3. 8 levels of eight features 1.1 to 1.3.
        if (M >= (size_t(1) << 18)) return L * F <= 36 && (largest <= MB ? M * L <= (size_t(1) << 23) : largest <= 8 * MB && M < (size_t(1) << 19));
        if (width == 128) return F > 1 && L > 10; // 0.6 and 0.7
        // 16 levels of more than 1 MB: 2^13 points 0.60 and 0.84, 2^14 0.72 and 1.05; of less 1.1 and 1.2, and so are fewer levels.
        return width == 64 && F == 2 && L > 12 && largest > MB && M >= (size_t(1) << 13) && M < 24000;
    }
    // 12 and 16 levels: 0.3 to 0.7 and 0.5 to 0.9; of more than 8 MB, 2^15 points 0.65 and 0.97, 2^16 0.89 and 1.34. 8 levels 0.8 and 1.0 to 1.1.
    if (L > 10 && M < (size_t(1) << 15)) return width >= 32 && (M < 24000 || (F <= 2 && largest <= 8 * MB));
    // Twice an XCD's L2 and more, which all XCDs share (shared_level). Drawn with 1 to 24 levels, one and two features, widths 16 to 64 and 2^20 to 2^22 points (4906 configurations, half of them of one to
    // five levels; one kernel's time = 1, scattered points and a picture's rows): two features and width 32 and more 0.91 and 0.62; of the others, whose waves are more, those with three levels as large as
    // the largest (whose tables are full: the levels that cost lines) 0.89 and 0.79; in all 4 % more than a tenth slower for one or the other. With fewer such levels 1.09 (up to 1.57) and 0.81, 50 %. 16 levels of
    // 32 MB, width 64, 2^21 points 1304 / 1170 us and 430 / 328; three, two of them of more than 8 MB 248 / 199 and 222 / 152; two of 32 MB, width 16 243 / 270 and 119 / 102. Four features, 8 levels,
    // 2^19 points 209 / 215 and 76 / 99.
    // The points are in cell order from 5 * 2^17 on, and without it 2^19 take 1.0 to 1.3 of one kernel's time for 12 levels and fewer, 0.92 to 1.0 for 16 of two features. Between, such fields would be as much faster as
    // beyond (16 levels of 32 MB, 3 * 2^18 points 0.88 and 0.91, 2^20 0.87 and 1.0). They are one kernel up to 2^20 points not because that were faster, but because callers and tests
    // count on its taking no scratch memory there.
    if (largest > 8 * MB) {
        uint32_t n_largest = 0;
        for (uint32_t l = 0; l < L; ++l) n_largest += level_bytes(grid, l) == largest;
        return F <= 2 && M > (size_t(1) << 20) && ((F == 2 && width >= 32) || n_largest > 2);
    }
    if (largest > MB && width == 16) return false;
    // Two features: 0.3 to 0.8 and 0.2 to 0.9. Four and eight: 6 levels 2^18 points 0.8 to 1.0 and 0.6, 8 levels 1.0 and 0.9, 2^19 1.1 and 1.4.
    if (M >= (size_t(1) << 18)) return F <= 2 || (L <= 6 && M < (size_t(1) << 19)) || (L * F <= 16 && largest <= MB);
    // Between: 16 levels 0.5 and 0.9 (2^15 to 2^16 points 0.6 and 1.0). 8 levels, width 64: 2^15 points 0.7 and 1.1, 2^16 0.6 and 0.9; 4 levels 0.84 and 0.76, 2 levels 2^17 0.65. Four features
    // 0.55 and 1.1 to 1.8; width 32, 4 levels 2^16 points 1.15, width 16, 8 levels 0.7 and 1.3.
    if (F > 2 || width < 32) return false;
    return L > 10 || (width == 64 && M >= (size_t(1) << (L > 2 ? 16 : 17)));
}

TNN_API int tnn_grid_mlp_width_wants_levels(const tnn_grid_desc *grid, int width, size_t M) { return !check_grid_desc(grid) && M != 0 && levels_pay(grid, width, M); }

TNN_API int tnn_grid_mlp_wants_levels(const tnn_grid_desc *grid, size_t M) { return tnn_grid_mlp_width_wants_levels(grid, 64, M); }

TNN_API int tnn_grid_mlp_forward_levels(const tnn_grid_desc *grid, const tnn_mlp_desc *mlp, const float *d_src_packed, int unpadded_input_width,
                                        int unpadded_output_width, int use_bias, void *d_packed_T, void *d_packed_transposed_T, void *d_prepared_fwd,
                                        void *d_prepared_bwd, const float *d_x, const void *d_order, const void *d_table, void *d_levels, void *d_y, int y_cols,
                                        size_t M, tnn_stream_t stream) {
    GridLevels lv;
    GridParams gp;
    int rc = tnn_grid_mlp_supported(grid, mlp);
    if (rc) return rc;
    if ((rc = grid_common(grid, (uint32_t)mlp->width, M, &lv, &gp))) return rc;
    if (y_cols < 1 || y_cols > mlp->width) return fail(TNN_ERR_INVALID_ARGUMENT, "%d output columns for a network of width %d", y_cols, mlp->width);
    if ((!d_x && !d_order) || !d_table || !d_prepared_fwd || !d_levels || !d_y) return fail(TNN_ERR_INVALID_ARGUMENT, "NULL pointer argument");
    if ((reinterpret_cast<uintptr_t>(d_order) & 15) || (reinterpret_cast<uintptr_t>(d_levels) & 15))
        return fail(TNN_ERR_INVALID_ARGUMENT, "d_order and d_levels must be 16-byte aligned");
    WeightPush push;
    if (d_src_packed) {
        if ((rc = make_weight_push(mlp, d_src_packed, unpadded_input_width, unpadded_output_width, use_bias, d_packed_T, d_packed_transposed_T, d_prepared_fwd,
                                   d_prepared_bwd, &push)))
            return rc;
        if (reinterpret_cast<uintptr_t>(d_src_packed) & 7) { // (read in pairs)
            if ((rc = tnn_mlp_set_packed_weights(mlp, d_src_packed, TNN_FP32, unpadded_input_width, unpadded_output_width, use_bias, d_packed_T,
                                                 d_packed_transposed_T, d_prepared_fwd, d_prepared_bwd, stream)))
                return rc;
            push = WeightPush{};
        }
    }
    const float4 *order = static_cast<const float4 *>(d_order);
    hipStream_t s = as_stream(stream);
    if ((rc = launch_grid_levels(grid, lv, gp, d_x, order, d_table, d_levels, mlp->dtype, 0, M, s))) return rc;
    if (mlp->dtype == TNN_BF16) return launch_levels_mlp_w<bf16_t>(grid, mlp, d_levels, order, d_prepared_fwd, d_y, y_cols, M, push, s);
    return launch_levels_mlp_w<fp16_t>(grid, mlp, d_levels, order, d_prepared_fwd, d_y, y_cols, M, push, s);
}

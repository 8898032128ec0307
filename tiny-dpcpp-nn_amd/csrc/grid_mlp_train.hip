// C entry points of the training step on an encoded input: hash-grid encoding by levels (grid_levels.hip), network
// forward, L2 loss, backward pass and Adam on the network's weights (kernels: grid_mlp_train.inc, built once per network
// type), then the scatter of dL/d(encoding) into the table's gradient (grid.hip).
#include "adam_update.h"
#include "grid_levels.h"
#include "mlp_train_shape.h"
#include "train_reduce.h"

#include <algorithm>

namespace tnn {
#define TNN_DECLARE(T)                                                                                                                                 \
    int grid_mlp_train_launch_##T(const tnn_mlp_desc *d, const FusedPlan &p, const void *levels, uint32_t n_levels, const float4 *order, const void *wf, \
                                  const void *wb, const float *targets, float loss_scale, void *y, float *loss_sum, void *d_enc, size_t M,               \
                                  float *partials, float *loss_partials, const TrainTail &tail, hipStream_t s);                                        \
    int grid_mlp_given_launch_##T(const tnn_mlp_desc *d, const FusedPlan &p, const void *levels, uint32_t n_levels, const float4 *order, const void *wf, \
                                  const void *wb, const void *dLdy, void *d_enc, size_t M, float *partials, float *loss_partials, const TrainTail &tail, \
                                  hipStream_t s);                                                                                                       \
    int grid_mlp_reduce_launch_##T(const TrainReduce &r, hipStream_t s);
TNN_DECLARE(bf16)
TNN_DECLARE(fp16)
#undef TNN_DECLARE
} // namespace tnn

using namespace tnn;

static size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// The shapes the one-kernel step is built for: the width-64 network with ReLU and at most four hidden layers (the kernel
// of the plain training step that keeps a workgroup's tiles in LDS), two features per level.
static int train_shape_check(const tnn_grid_desc *grid, const tnn_mlp_desc *mlp, size_t M, GridLevels *lv, GridParams *gp, FusedPlan *plan) {
    int rc = check_mlp_desc(mlp);
    if (rc) return rc;
    if ((rc = grid_common(grid, (uint32_t)mlp->width, M, lv, gp))) return rc;
    if (mlp->width != 64 || mlp->activation != TNN_ACT_RELU || grid->n_features_per_level != 2)
        return fail(TNN_ERR_UNSUPPORTED, "fused encoding + training step: built for width 64, ReLU and 2 features per level; run the three calls");
    *plan = fused_plan(mlp, M);
    if (!plan->supported) return fail(TNN_ERR_UNSUPPORTED, "fused encoding + training step: no fused training kernel for this depth; run the three calls");
    return TNN_OK;
}

TNN_API int tnn_grid_mlp_train_supported(const tnn_grid_desc *grid, const tnn_mlp_desc *mlp) {
    GridLevels lv;
    GridParams gp;
    FusedPlan plan;
    return train_shape_check(grid, mlp, 8, &lv, &gp, &plan);
}

// Where a pass keeps what: dL/d(encoding) by levels for the scatter, the partial weight gradients and losses of the workgroups, and a
// part that first holds the encoded levels and then, when the network is through with them, what the scatter sorts the contributions into.
struct GridTrainMemory {
    size_t levels_bytes, bytes;
    void *enc_grad = nullptr, *levels = nullptr;
    float *loss_partials = nullptr, *partials = nullptr;
    void *scatter = nullptr;
    size_t scatter_bytes = 0;

    GridTrainMemory(const tnn_grid_desc *grid, const FusedPlan &plan, size_t M)
        : levels_bytes(align256(levels_elements(grid, M) * 2)),
          bytes(levels_bytes + align256(plan.loss_bytes) + align256(plan.partial_bytes) + 512 + std::max(levels_bytes, tnn_grid_backward_workspace_bytes(grid, M))) {}
    void place(const FusedPlan &plan, void *workspace, size_t workspace_bytes) {
        uintptr_t base = align256(reinterpret_cast<uintptr_t>(workspace));
        enc_grad = reinterpret_cast<void *>(base);
        base += levels_bytes;
        loss_partials = reinterpret_cast<float *>(base);
        base += align256(plan.loss_bytes);
        partials = reinterpret_cast<float *>(base);
        base += align256(plan.partial_bytes);
        levels = scatter = reinterpret_cast<void *>(base);
        scatter_bytes = workspace_bytes - (base - reinterpret_cast<uintptr_t>(workspace));
    }
};

// (The reduction behind the network's kernel clears the table's gradient where that is overwritten. It is launched with the scatter.)
// dL/d(encoding), in the network's type, by levels and in the order the kernel took the points, into the table's gradient
static int scatter_levels(const tnn_grid_desc *grid, const tnn_mlp_desc *mlp, const float *d_x, const float4 *order, const GridTrainMemory &m, float scale,
                          float *d_grad_table, int overwrite, size_t M, const TrainReduce &reduce, hipStream_t s) {
    ReduceInFront front{&reduce, mlp->dtype == TNN_BF16 ? grid_mlp_reduce_launch_bf16 : grid_mlp_reduce_launch_fp16};
    const GradLayout dl{grid->n_features_per_level, level_pitch(M) * grid->n_features_per_level, 1, scale};
    return grid_backward_impl(grid, order ? nullptr : d_x, order, m.enc_grad, mlp->dtype, (uint32_t)mlp->width, dl, d_grad_table, TNN_FP32, overwrite, M, m.scatter,
                              m.scatter_bytes, s, overwrite != 0, &front);
}

TNN_API size_t tnn_grid_mlp_train_step_workspace_bytes(const tnn_grid_desc *grid, const tnn_mlp_desc *mlp, size_t M) {
    GridLevels lv;
    GridParams gp;
    FusedPlan plan;
    if (train_shape_check(grid, mlp, M ? M : 8, &lv, &gp, &plan)) return 0;
    return GridTrainMemory(grid, plan, M ? M : 8).bytes;
}

TNN_API int tnn_grid_mlp_train_step_l2_adam(const tnn_grid_desc *grid, const tnn_mlp_desc *mlp, const float *d_x, const void *d_order,
                                            const void *d_table, void *d_prepared_fwd, void *d_prepared_bwd, const float *d_targets,
                                            float loss_scale, void *d_y, float *d_loss_sum, float *d_master_packed, float *d_m, float *d_v,
                                            int step, float lr, float beta1, float beta2, float eps, void *d_packed_T, float *d_grad_table,
                                            int overwrite, size_t M, void *d_workspace, size_t workspace_bytes, tnn_stream_t stream) {
    GridLevels lv;
    GridParams gp;
    FusedPlan plan;
    int rc = train_shape_check(grid, mlp, M ? M : 8, &lv, &gp, &plan);
    if (rc) return rc;
    if (M == 0 || (M % 8) != 0) return fail(TNN_ERR_INVALID_ARGUMENT, "batch size %zu is not a positive multiple of 8", M);
    if ((!d_x && !d_order) || !d_table || !d_prepared_fwd || !d_prepared_bwd || !d_targets || !d_master_packed || !d_m || !d_v || !d_grad_table)
        return fail(TNN_ERR_INVALID_ARGUMENT, "NULL pointer argument");
    if (reinterpret_cast<uintptr_t>(d_order) & 15) return fail(TNN_ERR_INVALID_ARGUMENT, "d_order must be 16-byte aligned");
    if (loss_scale == 0.0f) return fail(TNN_ERR_INVALID_ARGUMENT, "loss_scale must not be 0");
    if (step < 1) return fail(TNN_ERR_INVALID_ARGUMENT, "step counts from 1");
    GridTrainMemory m(grid, plan, M);
    if (!d_workspace || workspace_bytes < m.bytes) return fail(TNN_ERR_WORKSPACE, "workspace of %zu bytes given, %zu needed", workspace_bytes, m.bytes);
    m.place(plan, d_workspace, workspace_bytes);
    hipStream_t s = as_stream(stream);

    TrainTail tail;
    TrainReduce reduce;
    tail.later = &reduce;
    tail.use_adam = true;
    tail.adam = make_adam_args(d_master_packed, d_m, d_v, 1.0f / loss_scale, step, lr, beta1, beta2, eps, d_packed_T, d_prepared_fwd, d_prepared_bwd,
                               mlp->width);
    const float4 *order = static_cast<const float4 *>(d_order);
    if (overwrite && (rc = grid_backward_clear(grid, order != nullptr, true, d_grad_table, TNN_FP32, M, &tail.clear))) return rc;
    if ((rc = launch_grid_levels(grid, lv, gp, d_x, order, d_table, m.levels, mlp->dtype, 0, M, s))) return rc;
    const auto launch = mlp->dtype == TNN_BF16 ? grid_mlp_train_launch_bf16 : grid_mlp_train_launch_fp16;
    if ((rc = launch(mlp, plan, m.levels, grid->n_levels, order, d_prepared_fwd, d_prepared_bwd, d_targets, loss_scale, d_y, d_loss_sum, m.enc_grad, M, m.partials,
                     m.loss_partials, tail, s)))
        return rc;
    return scatter_levels(grid, mlp, d_x, order, m, 1.0f, d_grad_table, overwrite, M, reduce, s);
}

// d_levels: the encoded batch as a forward pass left it, or null, and it is formed from d_table.
static int grid_mlp_backward(const tnn_grid_desc *grid, const tnn_mlp_desc *mlp, const float *d_x, const void *d_order, const void *d_table,
                             const void *d_levels, const void *d_prepared_fwd, const void *d_prepared_bwd, const void *d_dLdy, float *d_grad_table, int overwrite, size_t M,
                             void *d_workspace, size_t workspace_bytes, TrainTail tail, hipStream_t s) {
    GridLevels lv;
    GridParams gp;
    FusedPlan plan;
    int rc = train_shape_check(grid, mlp, M, &lv, &gp, &plan);
    if (rc) return rc;
    if ((!d_x && !d_order) || (!d_table && !d_levels) || !d_prepared_fwd || !d_prepared_bwd || !d_dLdy || (!tail.dW && !tail.packed.p))
        return fail(TNN_ERR_INVALID_ARGUMENT, "NULL pointer argument");
    if ((reinterpret_cast<uintptr_t>(d_order) & 15) || (reinterpret_cast<uintptr_t>(d_levels) & 15))
        return fail(TNN_ERR_INVALID_ARGUMENT, "d_order and d_levels must be 16-byte aligned");
    GridTrainMemory m(grid, plan, M);
    if (!d_workspace || workspace_bytes < m.bytes) return fail(TNN_ERR_WORKSPACE, "workspace of %zu bytes given, %zu needed", workspace_bytes, m.bytes);
    m.place(plan, d_workspace, workspace_bytes);
    const float4 *order = static_cast<const float4 *>(d_order);
    if (d_grad_table && overwrite && (rc = grid_backward_clear(grid, order != nullptr, true, d_grad_table, TNN_FP32, M, &tail.clear))) return rc;
    if (!d_levels) {
        if ((rc = launch_grid_levels(grid, lv, gp, d_x, order, d_table, m.levels, mlp->dtype, 0, M, s))) return rc;
        d_levels = m.levels;
    }
    TrainReduce reduce;
    if (d_grad_table) tail.later = &reduce;
    // without a gradient table the network's gradients are all that is asked for: no dL/d(encoding) leaves the kernel
    const auto launch = mlp->dtype == TNN_BF16 ? grid_mlp_given_launch_bf16 : grid_mlp_given_launch_fp16;
    rc = launch(mlp, plan, d_levels, grid->n_levels, order, d_prepared_fwd, d_prepared_bwd, d_dLdy, d_grad_table ? m.enc_grad : nullptr, M, m.partials, m.loss_partials,
                tail, s);
    if (rc || !d_grad_table) return rc;
    return scatter_levels(grid, mlp, d_x, order, m, tail.result_scale, d_grad_table, overwrite, M, reduce, s);
}

TNN_API int tnn_grid_mlp_backward(const tnn_grid_desc *grid, const tnn_mlp_desc *mlp, const float *d_x, const void *d_order, const void *d_table,
                                  const void *d_prepared_fwd, const void *d_prepared_bwd, const void *d_dLdy, void *d_dW, int dW_is_fp32,
                                  float *d_grad_table, int overwrite, size_t M, void *d_workspace, size_t workspace_bytes, tnn_stream_t stream) {
    int rc = tnn_grid_mlp_train_supported(grid, mlp);
    if (rc) return rc;
    if (M == 0 || (M % 8) != 0) return fail(TNN_ERR_INVALID_ARGUMENT, "batch size %zu is not a positive multiple of 8", M);
    if (!d_dW) return fail(TNN_ERR_INVALID_ARGUMENT, "NULL pointer argument");
    TrainTail tail;
    tail.dW = d_dW;
    tail.dW_is_fp32 = dW_is_fp32;
    return grid_mlp_backward(grid, mlp, d_x, d_order, d_table, nullptr, d_prepared_fwd, d_prepared_bwd, d_dLdy, d_grad_table, overwrite, M, d_workspace,
                             workspace_bytes, tail, as_stream(stream));
}

TNN_API int tnn_grid_mlp_backward_rows(const tnn_grid_desc *grid, const tnn_mlp_desc *mlp, const float *d_x, const void *d_order, const void *d_table,
                                       const void *d_prepared_fwd, const void *d_prepared_bwd, const void *d_dLdy, int dy_cols, float dy_scale,
                                       float result_scale, void *d_dW_packed, int dW_dtype, float *d_grad_table, int overwrite, size_t M,
                                       void *d_workspace, size_t workspace_bytes, tnn_stream_t stream) {
    int rc = check_mlp_desc(mlp);
    if (rc) return rc;
    TrainTail tail;
    if ((rc = rows_tail(mlp, dy_cols, dy_scale, result_scale, d_dW_packed, dW_dtype, M, &tail))) return rc;
    return grid_mlp_backward(grid, mlp, d_x, d_order, d_table, nullptr, d_prepared_fwd, d_prepared_bwd, d_dLdy, d_grad_table, overwrite, M, d_workspace,
                             workspace_bytes, tail, as_stream(stream));
}

TNN_API int tnn_grid_mlp_backward_levels_rows(const tnn_grid_desc *grid, const tnn_mlp_desc *mlp, const float *d_x, const void *d_order, const void *d_levels,
                                              const void *d_prepared_fwd, const void *d_prepared_bwd, const void *d_dLdy, int dy_cols, float dy_scale,
                                              float result_scale, void *d_dW_packed, int dW_dtype, float *d_grad_table, int overwrite, size_t M,
                                              void *d_workspace, size_t workspace_bytes, tnn_stream_t stream) {
    int rc = check_mlp_desc(mlp);
    if (rc) return rc;
    if (!d_levels) return fail(TNN_ERR_INVALID_ARGUMENT, "NULL pointer argument");
    TrainTail tail;
    if ((rc = rows_tail(mlp, dy_cols, dy_scale, result_scale, d_dW_packed, dW_dtype, M, &tail))) return rc;
    return grid_mlp_backward(grid, mlp, d_x, d_order, nullptr, d_levels, d_prepared_fwd, d_prepared_bwd, d_dLdy, d_grad_table, overwrite, M, d_workspace,
                             workspace_bytes, tail, as_stream(stream));
}

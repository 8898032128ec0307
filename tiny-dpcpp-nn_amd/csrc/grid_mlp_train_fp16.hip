// Training step kernels of a network behind a grid encoding, fp16 network.
#include "grid_mlp_train.inc"

namespace tnn {
int grid_mlp_train_launch_fp16(const tnn_mlp_desc *d, const FusedPlan &p, const void *levels, uint32_t n_levels, const float4 *order, const void *wf,
                               const void *wb, const float *targets, float loss_scale, void *y, float *loss_sum, void *d_enc, size_t M, float *partials,
                               float *loss_partials, const TrainTail &tail, hipStream_t s) {
    return launch_levels_train_n<fp16_t>(d, p, levels, n_levels, order, wf, wb, targets, loss_scale, y, loss_sum, d_enc, M, partials, loss_partials, tail, s);
}
int grid_mlp_reduce_launch_fp16(const TrainReduce &r, hipStream_t s) { return launch_train_reduce<fp16_t>(r, s); }
} // namespace tnn

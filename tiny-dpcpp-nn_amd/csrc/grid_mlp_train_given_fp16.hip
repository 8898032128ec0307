// Backward pass of a network behind a grid encoding for a loss gradient given by the caller, fp16 network.
#define TNN_TRAIN_GIVEN 1
#include "grid_mlp_train.inc"

namespace tnn {
int grid_mlp_given_launch_fp16(const tnn_mlp_desc *d, const FusedPlan &p, const void *levels, uint32_t n_levels, const float4 *order, const void *wf,
                               const void *wb, const void *dLdy, void *d_enc, size_t M, float *partials, float *loss_partials, const TrainTail &tail,
                               hipStream_t s) {
    return launch_levels_train_n<fp16_t>(d, p, levels, n_levels, order, wf, wb, static_cast<const float *>(dLdy), 1.0f, nullptr, nullptr, d_enc, M, partials,
                                         loss_partials, tail, s);
}
} // namespace tnn

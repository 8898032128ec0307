// The reduction behind a training kernel: the sums of the workgroups' partial weight gradients, what becomes of them (a gradient, Adam), the loss, and memory that
// is cleared on the side. A launch of its own (mlp_train.inc), or the first workgroups of a launch that follows anyway (grid_binned.hip).
#pragma once

#include "adam_update.h"

#include <algorithm>

namespace tnn {

struct TrainReduce {
    const float *partials = nullptr, *loss_partials = nullptr;
    int n_partials = 0, n_elems = 0;
    void *dW_T = nullptr; // gradients of the network's type, or
    float *dW_f32 = nullptr;
    float *loss_sum = nullptr;
    bool use_adam = false;
    AdamArgs adam{};
    PackedGradient packed{};
    ClearRange clear{};
    unsigned clear_blocks() const { return clear.p ? (unsigned)std::min<size_t>(1024, clear.n4 / 1024 + 1) : 0u; } // (two stores a thread while they are few)
    unsigned blocks() const { return clear.reduce_blocks + clear_blocks(); }
};

// Sums the per-workgroup partials in a fixed order. A workgroup owns 64 consecutive dW
// elements: each of 32 groups of 16 lanes (one float4 per lane, a 256-byte row piece; with 256 threads every group of lanes is two of them, one after the
// other) adds up every 32nd
// partial with all of its loads in flight at once; 64 lanes then add up the 32 group sums of one element each, again
// in a fixed order. With ADAM the same lane takes the sum straight into the optimizer: it updates the fp32 master
// copy and re-stages the rounded weight for the next step's kernels (dW is then written only if asked for).
// ONE: there are at most 256 partials; half of the registers.
template <typename T, bool ADAM, int THREADS, bool ONE>
__device__ __forceinline__ void train_reduce_block(const float *__restrict__ partials, const float *__restrict__ loss_partials, int n_partials, int n_elems,
                                                   T *__restrict__ dW_T, float *__restrict__ dW_f32, float *__restrict__ loss_sum, const AdamArgs &adam,
                                                   const PackedGradient &packed, uint32_t block, float4 (*red)[16]) {
    const int c = threadIdx.x & 15;
    const int idx = block * 64 + c * 4; // n_elems is a multiple of 256
    // the optimizer state of the weight this lane will update is requested with the partials, not behind their sum
    AdamElement state{};
    if (ADAM && threadIdx.x < 64) state = adam_fetch_element(adam, block * 64 + threadIdx.x);
#pragma unroll 1
    for (int g = threadIdx.x >> 4; g < 32; g += THREADS / 16) {
        float4 s[8];
        if constexpr (ONE) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                s[u] = float4{0.f, 0.f, 0.f, 0.f};
                if (g + 32 * u < n_partials) s[u] = *reinterpret_cast<const float4 *>(partials + (size_t)(g + 32 * u) * n_elems + idx);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) { s[u].x += 0.f; s[u].y += 0.f; s[u].z += 0.f; s[u].w += 0.f; } // (the bits of a sum that starts at zero)
        } else {
#pragma unroll
            for (int u = 0; u < 8; ++u) s[u] = float4{0.f, 0.f, 0.f, 0.f};
            for (int p0 = g; p0 < n_partials; p0 += 256) {
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int p = p0 + 32 * u;
                    if (p < n_partials) {
                        const float4 v = *reinterpret_cast<const float4 *>(partials + (size_t)p * n_elems + idx);
                        s[u].x += v.x; s[u].y += v.y; s[u].z += v.z; s[u].w += v.w;
                    }
                }
            }
        }
        float4 t;
        t.x = ((s[0].x + s[1].x) + (s[2].x + s[3].x)) + ((s[4].x + s[5].x) + (s[6].x + s[7].x));
        t.y = ((s[0].y + s[1].y) + (s[2].y + s[3].y)) + ((s[4].y + s[5].y) + (s[6].y + s[7].y));
        t.z = ((s[0].z + s[1].z) + (s[2].z + s[3].z)) + ((s[4].z + s[5].z) + (s[6].z + s[7].z));
        t.w = ((s[0].w + s[1].w) + (s[2].w + s[3].w)) + ((s[4].w + s[5].w) + (s[6].w + s[7].w));
        red[g][c] = t;
        if (THREADS == 512) break;
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        // lane e adds up element e of the 32 group sums: four running sums of eight, then a fixed tree
        const float *sums = reinterpret_cast<const float *>(&red[0][0]) + threadIdx.x;
        float q[4] = {sums[0], sums[64], sums[128], sums[192]};
#pragma unroll
        for (int w = 4; w < 32; ++w) q[w & 3] += sums[64 * w];
        const float grad = (q[0] + q[1]) + (q[2] + q[3]);
        const int e = block * 64 + threadIdx.x;
        if (dW_f32) {
            dW_f32[e] = grad;
        } else if (dW_T) {
            dW_T[e] = (T)grad;
        }
        if (packed.p) store_packed_gradient<T>(packed, e, grad);
        if (ADAM) adam_apply_element<T>(adam, e, state, grad);
    }
    // the loss: one wave, lane-strided loads (all in flight together), then a fixed-order butterfly
    if (loss_sum && block == 0 && threadIdx.x >= THREADS - 64) {
        const int lane = threadIdx.x & 63;
        float sum = 0.0f;
        for (int i = lane; i < n_partials; i += 64) sum += loss_partials[i];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
        if (lane == 0) *loss_sum = sum;
    }
}

} // namespace tnn

// Scatter-add of dL/dy into the levels of a hash-grid's gradient table that are too large for a private copy in LDS
// (include/encodings/grid.h:137-245 of the reference: float atomics, order not defined), without atomics to memory.
//
// The memory side retires an atomic request per 32-byte sector, about 20 * 10^9 a second, and a point of a hashed level
// needs 2^(D-1) or more of them: 2.1 ms for 2^20 points of a 3-D grid of 16 levels (2^19 entries). Here the contributions
// are sorted by destination first:
//   1. grid_bin_kernel cuts a level into bins of consecutive entries and writes every contribution as a record into its
//      bin. The two corners along the first dimension are neighbouring entries in a dense level and differ in the low bits
//      of the index in a coherently hashed one, so they share a bin and travel as one record of two entries.
//   2. grid_bin_sum_kernel takes a bin at a time, sums its records into a copy of the bin's entries in LDS and writes the
//      entries to the table as whole lines.
// A record of two features is 16 bytes written once and read once, where the two atomic requests it replaces occupy the
// memory side for 64.
#include "grid_binned.h"

#include <algorithm>
#include <cmath>

namespace tnn {

constexpr int kBinThreads = 512;
constexpr int kBinPoints = 2; // points of a thread
constexpr int kBinSumThreads = 512;

// Two neighbouring entries of a bin, the position between them, and the gradient times the weights of the other dimensions.
template <int F> struct alignas(F == 1 ? 4 : F == 2 ? 16 : 8) BinRecord {
    uint32_t where; // entry of the near side (15 bits), of the far side (15 bits), whether either is meant (bits 30, 31)
    float frac;
    float g[F];
};

template <int F> static size_t record_bytes_of() { return sizeof(BinRecord<F>); }
static size_t record_bytes(uint32_t F) { return F == 1 ? record_bytes_of<1>() : F == 2 ? record_bytes_of<2>() : F == 4 ? record_bytes_of<4>() : record_bytes_of<8>(); }

template <int D>
__device__ __forceinline__ long long bin_point(const float *__restrict__ xin, const float4 *__restrict__ order, long long i, float (&x)[D]) {
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

// Entries of the 2^(D-1) pairs of corners along the first dimension: bit d-1 of the pair's number says which side of
// dimension d it lies on.
template <int D>
__device__ __forceinline__ void pair_entries(const uint32_t (&cell)[D], uint32_t size, uint32_t res, uint32_t flags, uint32_t hash_type,
                                             uint32_t (&near)[1 << (D - 1)], uint32_t (&far)[1 << (D - 1)]) {
    if ((flags & 48u) == 48u && hash_type == TNN_HASH_COHERENT_PRIME) {
        // the hashed levels of the default configuration: the first dimension enters unmultiplied, the others' terms are shared
        const uint32_t mask = size - 1, y0 = cell[1] * 2654435761u, y1 = y0 + 2654435761u;
        const uint32_t z0 = D > 2 ? cell[D - 1] * 805459861u : 0u, z1 = z0 + 805459861u;
#pragma unroll
        for (int c = 0; c < (1 << (D - 1)); ++c) {
            const uint32_t rest = ((c & 1) ? y1 : y0) ^ (D > 2 ? ((c & 2) ? z1 : z0) : 0u);
            near[c] = (cell[0] ^ rest) & mask;
            far[c] = ((cell[0] + 1) ^ rest) & mask;
        }
        return;
    }
#pragma unroll
    for (int c = 0; c < (1 << (D - 1)); ++c) {
        uint32_t lo[D], hi[D];
        lo[0] = cell[0];
        hi[0] = cell[0] + 1;
#pragma unroll
        for (int d = 1; d < D; ++d) lo[d] = hi[d] = cell[d] + ((c >> (d - 1)) & 1);
        near[c] = level_index<D>(lo, size, res, flags, hash_type);
        far[c] = level_index<D>(hi, size, res, flags, hash_type);
    }
}

// One workgroup bins up to kBinPoints x kBinThreads consecutive points of one level: it counts its records per bin, which
// gives every record its place among them, reserves that much of every bin with one atomic, and writes the records there, so
// that a bin receives them in runs. The levels of the same points are consecutive workgroups of one XCD, which shares the
// rows of dL/dy between them in its L2.
// A record beyond a bin's capacity (points that cluster on few cells) goes to the table as atomics.
template <int D, int F, typename G>
__global__ void __launch_bounds__(kBinThreads)
    grid_bin_kernel(const GridLevels lv, const GridParams gp, const BinPlan bp, const GradLayout dl, const float *__restrict__ xin,
                    const float4 *__restrict__ order, const G *__restrict__ dLdy, uint32_t *__restrict__ cursors, BinRecord<F> *__restrict__ records,
                    float *__restrict__ grad, long long first, long long last, uint32_t per_wg) {
    constexpr int NP = 1 << (D - 1); // pairs of a point
    static_assert(kBinThreads * kBinPoints * NP <= 4096 && kBinMaxBins <= 1024, "a record's place is packed into 12 + 10 + 10 bits");
    __shared__ uint32_t base[kBinMaxBins];  // records per bin, then the first place of them
    __shared__ uint32_t split[kBinMaxBins]; // the same for far sides that lie in another bin than the near side
    const uint32_t turn = blockIdx.x / 8, k = turn % bp.n_levels;
    const long long begin = first + (long long)((turn / bp.n_levels) * 8 + blockIdx.x % 8) * per_wg;
    if (begin >= last) return;
    const long long end = begin + per_wg < last ? begin + per_wg : last;
    const uint32_t l = bp.level[k], slice = bp.slice_log2[k], n_bins = bp.first_bin[k + 1] - bp.first_bin[k];
    const uint32_t size = lv.size[l], res = lv.resolution[l], flags = lv.flags[l], capacity = bp.capacity[k];
    const float scale = lv.scale[l];
    uint32_t *const cursor = cursors + bp.first_bin[k];
    BinRecord<F> *const bins = records + bp.first_record[k];

    for (uint32_t b = threadIdx.x; b < n_bins; b += kBinThreads) base[b] = split[b] = 0;
    __syncthreads();
    const uint32_t mask = (1u << slice) - 1;
    float frac[kBinPoints][D], gy[kBinPoints][F];
    uint32_t where[kBinPoints][NP], place[kBinPoints][NP]; // place: rank in the bin (12 bits), bin, bin of the far side
#pragma unroll
    for (int u = 0; u < kBinPoints; ++u) {
        const long long i = begin + threadIdx.x + u * kBinThreads;
        if (i >= end) continue;
        float x[D];
        const long long row = bin_point<D>(xin, order, i, x);
        const G *dy = dLdy + (dl.by_position ? i : row) * dl.row_stride + l * dl.level_stride;
#pragma unroll
        for (int f = 0; f < F; ++f) gy[u][f] = (float)dy[f];
        uint32_t cell[D], near[NP], far[NP];
        cell_of<D>(x, scale, gp.interpolation, cell, frac[u]);
        pair_entries<D>(cell, size, res, flags, gp.hash_type, near, far);
#pragma unroll
        for (int c = 0; c < NP; ++c) {
            const uint32_t bin = near[c] >> slice, far_bin = far[c] >> slice;
            place[u][c] = atomicAdd(&base[bin], 1u) | (bin << 12) | (far_bin << 22);
            where[u][c] = (near[c] & mask) | ((far[c] & mask) << 15);
            if (far_bin != bin) atomicAdd(&split[far_bin], 1u);
        }
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < n_bins; b += kBinThreads) {
        const uint32_t n = base[b], n_split = split[b];
        const uint32_t at = n + n_split ? atomicAdd(&cursor[b], n + n_split) : 0u;
        base[b] = at;
        split[b] = at + n;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kBinPoints; ++u) {
        if (begin + threadIdx.x + u * kBinThreads >= end) continue;
#pragma unroll
        for (int c = 0; c < NP; ++c) {
            float weight = 1.0f;
#pragma unroll
            for (int d = 1; d < D; ++d) weight *= (c >> (d - 1)) & 1 ? frac[u][d] : 1 - frac[u][d];
            BinRecord<F> r;
            r.frac = frac[u][0];
#pragma unroll
            for (int f = 0; f < F; ++f) r.g[f] = weight * gy[u][f];
            const uint32_t bin = (place[u][c] >> 12) & 1023u, far_bin = place[u][c] >> 22;
            const auto put = [&](uint32_t to, uint32_t at, uint32_t sides) {
                r.where = where[u][c] | (sides << 30);
                if (at < capacity) {
                    bins[(size_t)to * capacity + at] = r;
                    return;
                }
                float *const g = grad + ((size_t)lv.offset[l] + ((size_t)to << slice)) * F;
#pragma unroll
                for (int f = 0; f < F; ++f) {
                    if (sides & 1) unsafeAtomicAdd(g + (size_t)(r.where & 0x7fff) * F + f, (1 - r.frac) * r.g[f]);
                    if (sides & 2) unsafeAtomicAdd(g + (size_t)((r.where >> 15) & 0x7fff) * F + f, r.frac * r.g[f]);
                }
            };
            put(bin, base[bin] + (place[u][c] & 4095u), far_bin == bin ? 3u : 1u);
            if (far_bin != bin) put(far_bin, atomicAdd(&split[far_bin], 1u), 2u);
        }
    }
}

// One workgroup sums one bin. Bound by the LDS atomics (two values of two features per record) and the records' bytes.
template <int F>
__global__ void __launch_bounds__(kBinSumThreads)
    grid_bin_sum_kernel(const GridLevels lv, const BinPlan bp, uint32_t *__restrict__ cursors, const BinRecord<F> *__restrict__ records,
                        float *__restrict__ grad, int store) {
    extern __shared__ double sums[];
    uint32_t k = 0;
    while (k + 1 < bp.n_levels && blockIdx.x >= bp.first_bin[k + 1]) ++k;
    const uint32_t l = bp.level[k], bin = blockIdx.x - bp.first_bin[k];
    const uint32_t first = bin << bp.slice_log2[k], size = lv.size[l];
    const uint32_t n = min(1u << bp.slice_log2[k], size - first);
    for (uint32_t e = threadIdx.x; e < n * F; e += kBinSumThreads) sums[e] = 0.0;
    const uint32_t written = cursors[blockIdx.x];
    const uint32_t n_records = min(written, bp.capacity[k]);
    const BinRecord<F> *const rec = records + bp.first_record[k] + (size_t)bin * bp.capacity[k];
    __syncthreads();
    if (threadIdx.x == 0) cursors[blockIdx.x] = 0; // for the next part of the batch
    constexpr int kAhead = 4; // records of a lane in flight
    for (uint32_t i = threadIdx.x; i < n_records; i += kAhead * kBinSumThreads) {
        BinRecord<F> r[kAhead];
#pragma unroll
        for (int a = 0; a < kAhead; ++a) {
            const uint32_t at = i + a * kBinSumThreads;
            r[a] = rec[at < n_records ? at : i];
            if (at >= n_records) r[a].where = 0;
        }
#pragma unroll
        for (int a = 0; a < kAhead; ++a) {
            const uint32_t near = r[a].where & 0x7fff, far = (r[a].where >> 15) & 0x7fff;
            if (r[a].where & (1u << 30)) {
#pragma unroll
                for (int f = 0; f < F; ++f) lds_add(&sums[near * F + f], (1 - r[a].frac) * r[a].g[f]);
            }
            if (r[a].where & (1u << 31)) {
#pragma unroll
                for (int f = 0; f < F; ++f) lds_add(&sums[far * F + f], r[a].frac * r[a].g[f]);
            }
        }
    }
    __syncthreads();
    float *const g = grad + ((size_t)lv.offset[l] + first) * F;
    if (store && written <= bp.capacity[k]) { // the bin's entries have no other contributions
        for (uint32_t e = threadIdx.x; e < n * F; e += kBinSumThreads) g[e] = (float)sums[e];
    } else {
        for (uint32_t e = threadIdx.x; e < n * F; e += kBinSumThreads) g[e] += (float)sums[e];
    }
}

bool bin_plan_add(BinPlan *p, uint32_t l, const GridLevels &lv, const GridParams &gp, uint32_t n_dims, uint32_t n_features, size_t M) {
    if (p->n_levels >= kMaxBinned || gp.interpolation == TNN_INTERP_NEAREST) return false;
    const size_t size = lv.size[l], entry = n_features * sizeof(double);
    // About 128 bins a level: a workgroup's share of a bin is then a run of several lines, and the bins of all levels are
    // enough workgroups for the sums. Larger levels have bins as large as LDS allows.
    uint32_t slice = 4;
    while (slice < 15 && (size >> slice) > 128 && ((size_t)2 << slice) * entry <= kBinSliceBytes) ++slice;
    const size_t bins = (size + ((size_t)1 << slice) - 1) >> slice;
    if (bins > kBinMaxBins) return false;
    p->batch = (uint32_t)std::min<size_t>(M, size_t(1) << 19);
    // (other hashes than the coherent one send the two corners along the first dimension to different bins)
    const bool apart = (lv.flags[l] & 16u) && gp.hash_type != TNN_HASH_COHERENT_PRIME;
    const double mean = (double)p->batch * (double)(1u << (n_dims - 1)) * (apart ? 2.0 : 1.0) / ((double)size / (double)(1u << slice));
    const double room = std::ceil((1.25 * mean + 8.0 * std::sqrt(mean) + 64.0) / 32.0) * 32.0;
    if (room * (double)bins + p->n_records > 4.0e9) return false;
    const uint32_t k = p->n_levels++;
    p->level[k] = (uint8_t)l;
    p->slice_log2[k] = (uint8_t)slice;
    p->capacity[k] = (uint32_t)room;
    p->first_record[k] = p->n_records;
    p->n_records += (uint32_t)room * (uint32_t)bins;
    p->first_bin[k] = p->n_bins;
    p->n_bins += (uint32_t)bins;
    p->first_bin[k + 1] = p->n_bins;
    p->slice_lds = std::max<uint32_t>(p->slice_lds, (uint32_t)(entry << slice));
    return true;
}

static size_t cursor_bytes(const BinPlan &p) { return ((size_t)p.n_bins * sizeof(uint32_t) + 255) & ~(size_t)255; }

size_t bin_scratch_bytes(const BinPlan &p, uint32_t n_features) {
    return p.n_levels ? cursor_bytes(p) + (size_t)p.n_records * record_bytes(n_features) : 0;
}

template <int D, int F, typename G>
static int launch_binned(const BinPlan &p, const GridLevels &lv, const GridParams &gp, const GradLayout &dl, const float *x, const float4 *order, const void *dLdy,
                         float *grad, bool overwrite, size_t M, void *scratch, hipStream_t s) {
    uint32_t *const cursors = static_cast<uint32_t *>(scratch);
    BinRecord<F> *const records = reinterpret_cast<BinRecord<F> *>(static_cast<char *>(scratch) + cursor_bytes(p));
    const auto sum = grid_bin_sum_kernel<F>;
    if (p.slice_lds > 48 * 1024 &&
        hipFuncSetAttribute(reinterpret_cast<const void *>(sum), hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.slice_lds) != hipSuccess)
        return fail(TNN_ERR_HIP, "cannot reserve %u bytes of LDS", p.slice_lds);
    for (size_t first = 0; first < M; first += p.batch) {
        const size_t last = std::min(M, first + p.batch), n = last - first;
        const uint32_t per_wg = n * p.n_levels < size_t(512) * kBinThreads * kBinPoints ? kBinThreads : kBinThreads * kBinPoints;
        const size_t stretches = (n + per_wg - 1) / per_wg;
        TNN_LAUNCH((grid_bin_kernel<D, F, G>), dim3((unsigned)((stretches + 7) / 8 * 8 * p.n_levels)), dim3(kBinThreads), 0, s, lv, gp, p, dl, x, order,
                   (const G *)dLdy, cursors, records, grad, (long long)first, (long long)last, per_wg);
        int rc = check_launch("grid_bin_kernel");
        if (rc) return rc;
        TNN_LAUNCH(sum, dim3(p.n_bins), dim3(kBinSumThreads), p.slice_lds, s, lv, p, cursors, (const BinRecord<F> *)records, grad,
                   (int)(overwrite && first == 0));
        if ((rc = check_launch("grid_bin_sum_kernel"))) return rc;
    }
    return TNN_OK;
}

int launch_grid_binned(const BinPlan &p, const GridLevels &lv, const GridParams &gp, const GradLayout &dl, uint32_t n_dims, uint32_t n_features, const float *x,
                       const float4 *order, const void *dLdy, int dy_dtype, float *grad, bool overwrite, size_t M, void *scratch, hipStream_t s) {
#define TNN_BIN_G(D, F)                                                                                                                    \
    switch (dy_dtype) {                                                                                                                    \
    case TNN_FP32: return launch_binned<D, F, float>(p, lv, gp, dl, x, order, dLdy, grad, overwrite, M, scratch, s);                            \
    case TNN_BF16: return launch_binned<D, F, bf16_t>(p, lv, gp, dl, x, order, dLdy, grad, overwrite, M, scratch, s);                           \
    case TNN_FP16: return launch_binned<D, F, fp16_t>(p, lv, gp, dl, x, order, dLdy, grad, overwrite, M, scratch, s);                           \
    default: return fail(TNN_ERR_UNSUPPORTED, "dy_dtype %d", dy_dtype);                                                                     \
    }
#define TNN_BIN_F(D)                                                                                                                       \
    switch (n_features) {                                                                                                                  \
    case 1: TNN_BIN_G(D, 1)                                                                                                                \
    case 2: TNN_BIN_G(D, 2)                                                                                                                \
    case 4: TNN_BIN_G(D, 4)                                                                                                                \
    default: TNN_BIN_G(D, 8)                                                                                                               \
    }
    if (n_dims == 2) { TNN_BIN_F(2) }
    TNN_BIN_F(3)
#undef TNN_BIN_F
#undef TNN_BIN_G
}

} // namespace tnn

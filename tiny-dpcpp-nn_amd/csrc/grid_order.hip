// Cell order for the points of a batch (gfx950): a permutation of the rows that puts points of the same part of space
// next to each other, so that the lanes of a wave and the waves of a workgroup gather from the same 128-byte lines of
// the grid's table at the same time. A random batch misses L2 on almost every gather of a level beyond 4 MiB and pays
// a whole line per 4-byte entry; in cell order the dense and the coarser hashed levels share their lines. Every row's
// result is computed exactly as before, in another lane, and written to its own row: results do not change.
//
// The reference has no such pass: its kernel_grid (include/encodings/grid.h:37-135) takes the points as they come, one
// work-item per (point, level), levels as the slow grid dimension (:696-731).
//
// Two steps, neither needs a stable order:
//   1. counting sort by a 12-bit key, the leading bits of every coordinate with the first dimension fastest (x runs along
//      a table line): per-workgroup histograms in LDS, one small scan kernel, scatter with LDS counters;
//   2. inside every one of the 4096 bins, a counting sort by the next bits of every coordinate.
// A record is 16 bytes: up to three coordinates and the row number.
#include "grid_device.h"

namespace tnn {

constexpr int kOrderThreads = 1024;
constexpr int kOrderBins = 4096;      // 12-bit key
constexpr int kOrderMaxWg = 256;      // histogram workgroups (the scan keeps a bin's counts of sixteen of them in each of sixteen lanes)
constexpr int kOrderAhead = 4;        // points of a thread under way at once (the whole ordering, 2^18 points: 24.8 us one by one, 21.1 with this and the refinement)
constexpr int kRefineEach = 8;        // records of a thread in a piece of a bin
constexpr int kRefineBins = 64;       // 6 further bits
constexpr size_t kSmallOrder = 8192; // points that one workgroup puts into their bins (order_small_kernel)

struct OrderPlan {
    int n_wg;
    long long chunk; // points per histogram workgroup, a multiple of kOrderThreads
    size_t record_bytes, hist_bytes, total_bytes;
};

static OrderPlan order_plan(size_t M) {
    OrderPlan p;
    long long wg = ((long long)M + 4 * kOrderThreads - 1) / (4 * kOrderThreads); // at least four rounds per workgroup
    if (wg > kOrderMaxWg) wg = kOrderMaxWg;
    if (wg < 1) wg = 1;
    p.n_wg = (int)wg;
    long long chunk = ((long long)M + wg - 1) / wg;
    p.chunk = (chunk + kOrderThreads - 1) / kOrderThreads * kOrderThreads;
    p.record_bytes = order_record_bytes(M);
    // (one workgroup's points need the starts of the bins alone)
    p.hist_bytes = (M <= kSmallOrder ? 1 : (size_t)p.n_wg) * kOrderBins * sizeof(uint32_t);
    p.total_bytes = M <= kSmallOrder ? 0 : kOrderBins * sizeof(uint32_t);
    return p;
}

template <int D> __device__ __forceinline__ uint32_t coarse_key(const float (&x)[D]) {
    constexpr int b = OrderBits<D>::coarse;
    uint32_t k = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) k |= quantise(x[d], b) << (b * d);
    return k;
}
template <int D> __device__ __forceinline__ uint32_t fine_key(const float (&x)[D]) {
    constexpr int b = OrderBits<D>::coarse, f = OrderBits<D>::fine;
    uint32_t k = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) k |= (quantise(x[d], b + f) & ((1u << f) - 1)) << (f * d);
    return k;
}

template <int D> __device__ __forceinline__ void load_point(const float *__restrict__ xin, long long i, float (&x)[D]) {
#pragma unroll
    for (int d = 0; d < D; ++d) x[d] = xin[i * D + d];
}

// Step 1a: histogram of the workgroup's chunk of points over the 4096 bins.
template <int D>
__global__ void __launch_bounds__(kOrderThreads)
    order_hist_kernel(const float *__restrict__ xin, long long M, long long chunk, uint32_t *__restrict__ hist) {
    __shared__ uint32_t h[kOrderBins];
    for (int b = threadIdx.x; b < kOrderBins; b += kOrderThreads) h[b] = 0;
    __syncthreads();
    const long long begin = (long long)blockIdx.x * chunk;
    long long end = begin + chunk;
    if (end > M) end = M;
    for (long long i0 = begin + threadIdx.x; i0 < end; i0 += kOrderAhead * kOrderThreads) {
        float x[kOrderAhead][D];
#pragma unroll
        for (int u = 0; u < kOrderAhead; ++u) load_point<D>(xin, i0 + u * kOrderThreads < end ? i0 + u * kOrderThreads : end - 1, x[u]);
#pragma unroll
        for (int u = 0; u < kOrderAhead; ++u)
            if (i0 + u * kOrderThreads < end) atomicAdd(&h[coarse_key<D>(x[u])], 1u);
    }
    __syncthreads();
    uint32_t *mine = hist + (size_t)blockIdx.x * kOrderBins;
    for (int b = threadIdx.x; b < kOrderBins; b += kOrderThreads) mine[b] = h[b];
}

// The sum of what the threads of a workgroup in front of this one have.
__device__ __forceinline__ uint32_t order_sum_in_front(uint32_t mine, uint32_t *__restrict__ wave_sum) {
    uint32_t incl = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t v = __shfl_up(incl, off, 64);
        if ((int)(threadIdx.x & 63) >= off) incl += v;
    }
    if ((threadIdx.x & 63) == 63) wave_sum[threadIdx.x >> 6] = incl;
    __syncthreads();
    uint32_t at = incl - mine;
#pragma unroll
    for (uint32_t w = 0; w < kOrderThreads / 64; ++w) at += w < threadIdx.x >> 6 ? wave_sum[w] : 0u;
    return at;
}
// Where four neighbouring bins start, from how many points each has and how many there are in front of all four.
__device__ __forceinline__ uint4 bin_starts(const uint4 c, uint32_t at) { return uint4{at, at + c.x, at + c.x + c.y, at + c.x + c.y + c.z}; }

// Step 1b: what the workgroups in front of a workgroup have in each bin, in place, and every bin's total; where the bins start follows from the totals, which
// every workgroup of the next step adds up by itself. A workgroup takes sixteen bins, a lane of it every sixteenth histogram's count of one, all under way at once; in a bin the histograms lie
// in that order, the first one first. (With the bins' starts formed here, 64 workgroups read all totals of runs of bins, and a bin's counts one after the other in LDS: 256 histograms
// 14.1 -> 6.1 us, 64 histograms 5.5 -> 4.1. Optimisation step, 2-D, 16 levels of 2^17 entries, 2^18 points 171.0 -> 166.4 us; encoding, 3-D, 2^20 points, forward and backward 887 -> 873; a field of a picture's rows 167 -> 158.)
constexpr int kScanThreads = 256;
constexpr int kScanBins = 16;
__global__ void __launch_bounds__(kScanThreads)
    order_scan_kernel(uint32_t *__restrict__ hist, uint32_t *__restrict__ totals, int n_wg) {
    constexpr int LANES = kScanThreads / kScanBins, EACH = kOrderMaxWg / LANES;
    __shared__ uint32_t part[LANES][kScanBins];
    const int bin = threadIdx.x % kScanBins, r = threadIdx.x / kScanBins;
    uint32_t *const column = hist + kScanBins * blockIdx.x + bin;
    uint32_t count[EACH], sum = 0;
#pragma unroll
    for (int k = 0; k < EACH; ++k) count[k] = r + LANES * k < n_wg ? column[(size_t)(r + LANES * k) * kOrderBins] : 0u;
#pragma unroll
    for (int k = 0; k < EACH; ++k) sum += count[k];
    part[r][bin] = sum;
    __syncthreads();
    uint32_t at = 0;
#pragma unroll
    for (int q = 0; q < LANES; ++q) at += q < r ? part[q][bin] : 0u;
    if (r == LANES - 1) totals[kScanBins * blockIdx.x + bin] = at + sum;
#pragma unroll
    for (int k = 0; k < EACH; ++k) {
        if (r + LANES * k < n_wg) column[(size_t)(r + LANES * k) * kOrderBins] = at;
        at += count[k];
    }
}

// Step 1c: every point goes to the next free position of its bin (the workgroup's own counters, in LDS).
template <int D>
__global__ void __launch_bounds__(kOrderThreads)
    order_scatter_kernel(const float *__restrict__ xin, long long M, long long chunk, uint32_t *__restrict__ hist, const uint32_t *__restrict__ totals,
                         float4 *__restrict__ records) {
    static_assert(kOrderBins == 4 * kOrderThreads, "four bins a thread");
    __shared__ uint4 next4[kOrderBins / 4];
    __shared__ uint32_t wave_sum[kOrderThreads / 64];
    uint32_t *const next = reinterpret_cast<uint32_t *>(next4);
    uint4 *const mine = reinterpret_cast<uint4 *>(hist + (size_t)blockIdx.x * kOrderBins) + threadIdx.x;
    const uint4 before = *mine, c = reinterpret_cast<const uint4 *>(totals)[threadIdx.x];
    const uint4 start = bin_starts(c, order_sum_in_front(c.x + c.y + c.z + c.w, wave_sum));
    next4[threadIdx.x] = uint4{start.x + before.x, start.y + before.y, start.z + before.z, start.w + before.w};
    if (blockIdx.x == 0) *mine = start; // (which the refinement and the scatter of gradients read; nobody else reads the first workgroup's counts)
    __syncthreads();
    const long long begin = (long long)blockIdx.x * chunk;
    long long end = begin + chunk;
    if (end > M) end = M;
    for (long long i0 = begin + threadIdx.x; i0 < end; i0 += kOrderAhead * kOrderThreads) {
        float x[kOrderAhead][D];
#pragma unroll
        for (int u = 0; u < kOrderAhead; ++u) load_point<D>(xin, i0 + u * kOrderThreads < end ? i0 + u * kOrderThreads : end - 1, x[u]);
#pragma unroll
        for (int u = 0; u < kOrderAhead; ++u) {
            const long long i = i0 + u * kOrderThreads;
            if (i >= end) continue;
            const uint32_t pos = atomicAdd(&next[coarse_key<D>(x[u])], 1u);
            float4 r;
            r.x = x[u][0];
            r.y = x[u][1];
            r.z = (D > 2) ? x[u][D - 1] : 0.0f;
            r.w = __uint_as_float((uint32_t)i);
            records[pos] = r;
        }
    }
}

// Step 1 of a batch that one workgroup holds in its registers: histogram, starting positions and places in one launch instead of three, each of which was some 3 us
// for nothing but its latency. What bounds it are the records that one CU writes to places of their own (optimisation step with the ordering, 16 levels of 2^15 entries, 2-D, us, three launches / one: 1024 points
// 49.4 / 43.3, 2048 50.8 / 44.0, 4096 52.2 / 45.5, 8192 54.7 / 50.7, with sixteen points a thread 12 288 58.9 / 58.7, 16 384 57.1 / 59.3; 3-D, 4096 48.6 / 42.2, 8192 51.9 / 48.2).
template <int D, int EACH>
__global__ void __launch_bounds__(kOrderThreads)
    order_small_kernel(const float *__restrict__ xin, uint32_t M, uint32_t *__restrict__ starts, float4 *__restrict__ records) {
    __shared__ uint4 h4[kOrderBins / 4];
    __shared__ uint32_t wave_sum[kOrderThreads / 64];
    static_assert(kOrderBins == 4 * kOrderThreads, "four bins a thread");
    uint32_t *const h = reinterpret_cast<uint32_t *>(h4);
    const uint32_t tid = threadIdx.x;
    float x[EACH][D];
#pragma unroll
    for (int u = 0; u < EACH; ++u) load_point<D>(xin, tid + u * kOrderThreads < M ? tid + u * kOrderThreads : M - 1, x[u]);
    h4[tid] = uint4{0u, 0u, 0u, 0u};
    __syncthreads();
    uint32_t key[EACH], rank[EACH];
#pragma unroll
    for (int u = 0; u < EACH; ++u) {
        key[u] = coarse_key<D>(x[u]);
        rank[u] = tid + u * kOrderThreads < M ? atomicAdd(&h[key[u]], 1u) : 0u;
    }
    __syncthreads();
    const uint4 c = h4[tid], start = bin_starts(c, order_sum_in_front(c.x + c.y + c.z + c.w, wave_sum));
    h4[tid] = start;
    reinterpret_cast<uint4 *>(starts)[tid] = start;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < EACH; ++u) {
        const uint32_t i = tid + u * kOrderThreads;
        if (i < M) records[h[key[u]] + rank[u]] = float4{x[u][0], x[u][1], D > 2 ? x[u][D - 1] : 0.0f, __uint_as_float(i)};
    }
}

// Step 2: the records of a bin by the next bits of their coordinates, in pieces of at most kRefinePiece that a workgroup sorts in its registers. The first
// kOrderBins / PER workgroups take the first pieces of PER bins each. Where points crowd a bin is many pieces, and the further workgroups take the others, side
// by side: workgroup e the piece that starts in [e, e + 1) * kRefinePiece, which is one at most, since the piece in front of it is full and of the same bin.
// PER 4, up to 256 points a bin on average: bins of few records are a wave's each, so that no wave of the workgroup is idle, unless one of the four is
// larger (they lie far apart: of a picture's rows one is). PER 1: more workgroups where bins fill them.
// The whole ordering, us, against pieces that wait in LDS and follow each other in one workgroup of 64 threads (of 256): 2-D, 2^18 points 21.7, 21.8 (25.5),
// 2^20 45.5, - (47.4), 2^21 63.4, - (64.2); 2^18 points in a square of a twentieth of the side 22.5, 172 (68), of a hundredth 23.5, 615 (194); 3-D, 2^20 points in a cube
// of a twentieth 41.5, - (831), near a sphere 43.2, - (44.8), the rows of a picture 40.4, - (41.5). Pieces of 1024 (128 threads) are as fast to sort, but gathers
// behind them share fewer lines (3-D, 2^21 points near a sphere, all levels 831 us for 793).
constexpr int kRefineThreads = 256;
constexpr int kRefinePiece = kRefineEach * kRefineThreads;

// Sorts n <= kRefineEach * GROUP records with GROUP threads. Every thread of the workgroup has to come (the groups share its barriers).
template <int D, int GROUP> __device__ __forceinline__ void refine_piece(float4 *__restrict__ records, int n, int tid, uint32_t *next) {
    if (tid < kRefineBins) next[tid] = 0;
    float4 rec[kRefineEach];
    uint32_t key[kRefineEach];
#pragma unroll
    for (int u = 0; u < kRefineEach; ++u) {
        rec[u] = float4{0.0f, 0.0f, 0.0f, 0.0f};
        if (tid + u * GROUP < n) rec[u] = records[tid + u * GROUP];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kRefineEach; ++u) {
        key[u] = 0;
        if (tid + u * GROUP < n) {
            float x[D];
            x[0] = rec[u].x;
            x[1] = rec[u].y;
            if (D > 2) x[D - 1] = rec[u].z;
            key[u] = fine_key<D>(x);
            atomicAdd(&next[key[u]], 1u);
        }
    }
    __syncthreads(); // (and all records of the piece are in registers)
    if (tid < kRefineBins) {
        const uint32_t c = next[tid];
        uint32_t incl = c;
#pragma unroll
        for (int off = 1; off < kRefineBins; off <<= 1) {
            const uint32_t v = __shfl_up(incl, off, 64);
            if (tid >= off) incl += v;
        }
        next[tid] = incl - c;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kRefineEach; ++u)
        if (tid + u * GROUP < n) records[atomicAdd(&next[key[u]], 1u)] = rec[u];
    __syncthreads();
}

template <int D, int PER>
__global__ void __launch_bounds__(kRefineThreads)
    order_refine_kernel(const uint32_t *__restrict__ starts, float4 *__restrict__ records, long long M) {
    static_assert(kOrderBins == 64 * 64 && kRefineBins == 64, "the search below is two steps of a wave; a wave scans the counts");
    constexpr int kGroups = kOrderBins / PER;
    __shared__ uint32_t next[PER][kRefineBins];
    const int tid = threadIdx.x, lane = tid & 63, block = blockIdx.x;
    auto begin_of = [&](int bin) { return bin < kOrderBins ? (long long)starts[bin] : M; }; // (workgroup 0's start of a bin is the start of the bin)
    if (block >= kGroups) {
        const long long before = (long long)(block - kGroups + 1) * kRefinePiece - 1; // a record of the piece in front, if there is one of this bin
        int bin = 64 * (__popcll(__ballot((long long)starts[64 * lane] <= before)) - 1);
        bin += __popcll(__ballot((long long)starts[bin + lane] <= before)) - 1;
        const long long begin = starts[bin], p0 = begin + ((before - begin) / kRefinePiece + 1) * kRefinePiece, left = begin_of(bin + 1) - p0;
        if (left > 0) refine_piece<D, kRefineThreads>(records + p0, (int)(left < kRefinePiece ? left : kRefinePiece), tid, next[0]);
        return;
    }
    if constexpr (PER > 1) {
        static_assert(PER == kRefineThreads / 64, "a wave for each bin");
        long long begin = 0, most = 0;
        int n = 0;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const long long first = starts[block + k * kGroups], size = begin_of(block + k * kGroups + 1) - first;
            most = most > size ? most : size;
            if (tid / 64 == k) {
                begin = first;
                n = (int)size;
            }
        }
        if (most <= kRefineEach * 64) {
            refine_piece<D, 64>(records + begin, n, lane, next[tid / 64]);
            return;
        }
    }
#pragma unroll 1
    for (int k = 0; k < PER; ++k) {
        const long long first = starts[block + k * kGroups], size = begin_of(block + k * kGroups + 1) - first;
        if (size > 1) refine_piece<D, kRefineThreads>(records + first, (int)(size < kRefinePiece ? size : kRefinePiece), tid, next[0]);
    }
}

} // namespace tnn

using namespace tnn;

TNN_API size_t tnn_grid_order_bytes(const tnn_grid_desc *desc, size_t M) {
    if (check_grid_desc(desc) || M == 0) return 0;
    const OrderPlan p = order_plan(M);
    return p.record_bytes + p.hist_bytes + p.total_bytes + 256;
}

TNN_API int tnn_grid_order_points(const tnn_grid_desc *desc, const float *d_x, size_t M, void *d_order, size_t order_bytes,
                                  tnn_stream_t stream) {
    int rc = check_grid_desc(desc);
    if (rc) return rc;
    if (!d_x || !d_order) return fail(TNN_ERR_INVALID_ARGUMENT, "NULL pointer argument");
    if (M == 0) return fail(TNN_ERR_INVALID_ARGUMENT, "batch_size == 0");
    if (M > 0xffffffffull) return fail(TNN_ERR_INVALID_ARGUMENT, "row numbers are 32 bits: at most 2^32 - 1 points");
    if (reinterpret_cast<uintptr_t>(d_order) & 255) return fail(TNN_ERR_INVALID_ARGUMENT, "d_order must be 256-byte aligned");
    const size_t need = tnn_grid_order_bytes(desc, M);
    if (order_bytes < need) return fail(TNN_ERR_WORKSPACE, "order buffer of %zu bytes given, %zu needed", order_bytes, need);
    const OrderPlan p = order_plan(M);
    float4 *records = static_cast<float4 *>(d_order);
    uint32_t *hist = reinterpret_cast<uint32_t *>(static_cast<char *>(d_order) + p.record_bytes);
    uint32_t *totals = reinterpret_cast<uint32_t *>(static_cast<char *>(d_order) + p.record_bytes + p.hist_bytes);
    hipStream_t s = as_stream(stream);
#define TNN_ORDER(D_)                                                                                                                  \
    do {                                                                                                                               \
        if (M <= kSmallOrder) {                                                                                                        \
            auto small = order_small_kernel<D_, kSmallOrder / kOrderThreads>;                                                          \
            if (M <= 4 * kOrderThreads) small = order_small_kernel<D_, 4>;                                                             \
            if (M <= 2 * kOrderThreads) small = order_small_kernel<D_, 2>;                                                             \
            TNN_LAUNCH(small, dim3(1), dim3(kOrderThreads), 0, s, d_x, (uint32_t)M, hist, records);                                    \
            if ((rc = check_launch("order_small_kernel"))) return rc;                                                                  \
        } else {                                                                                                                       \
            TNN_LAUNCH((order_hist_kernel<D_>), dim3(p.n_wg), dim3(kOrderThreads), 0, s, d_x, (long long)M, p.chunk, hist);             \
            if ((rc = check_launch("order_hist_kernel"))) return rc;                                                                   \
            TNN_LAUNCH(order_scan_kernel, dim3(kOrderBins / kScanBins), dim3(kScanThreads), 0, s, hist, totals, p.n_wg);               \
            if ((rc = check_launch("order_scan_kernel"))) return rc;                                                                   \
            TNN_LAUNCH((order_scatter_kernel<D_>), dim3(p.n_wg), dim3(kOrderThreads), 0, s, d_x, (long long)M, p.chunk, hist, (const uint32_t *)totals, records); \
            if ((rc = check_launch("order_scatter_kernel"))) return rc;                                                                \
        }                                                                                                                              \
        if (M <= (size_t)kOrderBins * 256)                                                                                             \
            TNN_LAUNCH((order_refine_kernel<D_, 4>), dim3(kOrderBins / 4 + (unsigned)(M / kRefinePiece)), dim3(kRefineThreads), 0, s, (const uint32_t *)hist, records, (long long)M); \
        else                                                                                                                           \
            TNN_LAUNCH((order_refine_kernel<D_, 1>), dim3(kOrderBins + (unsigned)(M / kRefinePiece)), dim3(kRefineThreads), 0, s, (const uint32_t *)hist, records, (long long)M); \
        return check_launch("order_refine_kernel");                                                                                    \
    } while (0)
    if (desc->n_dims == 2) TNN_ORDER(2);
    TNN_ORDER(3);
#undef TNN_ORDER
}

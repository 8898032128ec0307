// Scatter-add of dL/dy into the levels of a hash-grid's gradient table that are too large for a private copy in LDS
// (include/encodings/grid.h:137-245 of the reference: float atomics, order not defined), without atomics to memory.
//
// The memory side retires an atomic request per 32-byte sector, about 20 * 10^9 a second, and a point of a hashed level
// needs 2^(D-1) or more of them: 2.1 ms for 2^20 points of a 3-D grid of 16 levels (2^19 entries). Here the contributions
// are sorted by destination first:
//   1. grid_bin_kernel deals runs of a level's entries out to bins and writes every contribution as a record into its
//      bin. The two corners along the first dimension are neighbouring entries in a dense level and differ in the low bits
//      of the index in a coherently hashed one, so nearly always they share a bin and travel as one record of two entries.
//      (Long runs make long stores; but a hashed level's runs longer than its x range are dealt out by the other
//      dimensions alone, and in 2-D the few hundred values of y fill the bins very unevenly: bin_plan_add.)
//   2. grid_bin_sum_kernel takes a bin at a time, sums its records into a copy of the bin's entries in LDS and writes the
//      entries to the table as whole lines.
// A record of two features is 16 bytes written once and read once, where the two atomic requests it replaces occupy the
// memory side for 64.
// Measured, 2^20 points, 3-D, 2^19 entries, 15 levels this way: 2 x (164 + 172) us, 3 TB/s of records both ways; before, the
// atomics of the ten finest of these levels alone took 1.5 ms.
#include "grid_binned.h"

#include <algorithm>
#include <cmath>

namespace tnn {

constexpr int kBinSumThreads = 1024; // at most

// A binning workgroup: its threads (at most), the points of a thread, and the most records it sorts in LDS. 2048 records of 16
// bytes let four workgroups of 8 waves share a CU, whose phases (loads, LDS, stores) then overlap; wider records take half as many.
// (3-D, 2^19 points, 15 levels of two features: 164 us; 4096 records 177, 1024 184.)
template <int D, int F> struct BinShape {
    static constexpr int kThreads = F <= 2 ? 512 : 256;
    static constexpr int kPoints = D == 2 && F <= 2 ? 2 : 1;
    static constexpr int kPairs = 1 << (D - 1);
    static constexpr int kRecords = kThreads * kPoints * kPairs;
};

// Entry e of a level: its bin and its place there.
struct Bins {
    uint32_t n_log2, run_log2;
    __device__ __forceinline__ uint32_t bin(uint32_t e) const { return (e >> run_log2) & ((1u << n_log2) - 1); }
    __device__ __forceinline__ uint32_t place(uint32_t e) const { return ((e >> (run_log2 + n_log2)) << run_log2) | (e & ((1u << run_log2) - 1)); }
    __device__ __forceinline__ uint32_t entry(uint32_t bin, uint32_t place) const {
        return ((((place >> run_log2) << n_log2) | bin) << run_log2) | (place & ((1u << run_log2) - 1));
    }
};

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

// One workgroup bins kPoints points a thread of one level: it counts its records per bin, which gives every record its place among
// them, reserves that much of every bin with one atomic, sorts the records by bin in LDS and writes them from there, so that a
// wave stores whole runs: neighbouring lanes, neighbouring records. Bound by the records' bytes on their way to memory, 3.0 TB/s
// at 12, 16, 24 and 40 bytes a record. (Every lane storing its own records, as many L2 requests as records times pieces of 16
// bytes: four features 166 -> 133 us, eight 138 -> 119, one 36 -> 27, two as fast either way, 3-D or 2-D, 2^18 points.) The levels of the same points are consecutive workgroups of one
// XCD, which shares the rows of dL/dy between them in its L2.
// Records beyond a bin's capacity are counted and dropped.
template <int D, int F, typename G>
__global__ void __launch_bounds__((BinShape<D, F>::kThreads))
    grid_bin_kernel(const GridLevels lv, const GridParams gp, const BinPlan bp, const GradLayout dl, const float *__restrict__ xin,
                    const float4 *__restrict__ order, const G *__restrict__ dLdy, uint32_t *__restrict__ cursors, BinRecord<F> *__restrict__ records,
                    long long first, long long last) {
    typedef BinShape<D, F> S;
    constexpr int NP = S::kPairs, P = S::kPoints;
    static_assert(S::kRecords <= 4096 && kBinMaxBins <= 1024, "a record's place is packed into 12 + 10 + 10 bits");
    const int T = blockDim.x;
    extern __shared__ __align__(16) unsigned char bin_smem[];
    BinRecord<F> *const sorted = reinterpret_cast<BinRecord<F> *>(bin_smem);
    uint16_t *const bin_of = reinterpret_cast<uint16_t *>(sorted + T * P * NP); // of a sorted record
    uint32_t *const base = reinterpret_cast<uint32_t *>(bin_of + T * P * NP);    // records per bin, then the first sorted one of them
    const uint32_t turn = blockIdx.x / 8, k = turn % bp.n_levels, per_wg = T * P;
    const long long begin = first + (long long)((turn / bp.n_levels) * 8 + blockIdx.x % 8) * per_wg;
    if (begin >= last) return;
    const long long end = begin + per_wg < last ? begin + per_wg : last;
    const Bins dealt{bp.bins_log2[k], bp.run_log2[k]};
    const uint32_t l = bp.level[k], n_bins = 1u << dealt.n_log2;
    uint32_t *const split = base + n_bins; // records per bin of far sides that lie in another bin than the near side, then the next place of one
    uint32_t *const shift = split + n_bins; // place in the bin less place among the sorted records
    uint32_t *const wave_sum = shift + n_bins;
    const uint32_t size = lv.size[l], res = lv.resolution[l], flags = lv.flags[l], capacity = bp.capacity[k];
    const float scale = lv.scale[l];
    uint32_t *const cursor = cursors + bp.first_bin[k];
    BinRecord<F> *const bins = records + bp.first_record[k];

    for (uint32_t b = threadIdx.x; b < n_bins; b += T) base[b] = split[b] = 0;
    __syncthreads();
    float frac[P][D], gy[P][F];
    uint32_t where[P][NP], place[P][NP]; // place: rank in the bin (12 bits), bin, bin of the far side
#pragma unroll
    for (int u = 0; u < P; ++u) {
        const long long i = begin + threadIdx.x + u * T;
        if (i >= end) continue;
        float x[D];
        const long long row = bin_point<D>(xin, order, i, x);
        const G *dy = dLdy + (dl.by_position ? i : row) * dl.row_stride + l * dl.level_stride;
#pragma unroll
        for (int f = 0; f < F; ++f) gy[u][f] = (float)dy[f] * dl.scale;
        uint32_t cell[D], near[NP], far[NP];
        cell_of<D>(x, scale, gp.interpolation, cell, frac[u]);
        pair_entries<D>(cell, size, res, flags, gp.hash_type, near, far);
#pragma unroll
        for (int c = 0; c < NP; ++c) {
            const uint32_t bin = dealt.bin(near[c]), far_bin = dealt.bin(far[c]);
            place[u][c] = atomicAdd(&base[bin], 1u) | (bin << 12) | (far_bin << 22);
            where[u][c] = dealt.place(near[c]) | (dealt.place(far[c]) << 15);
            if (far_bin != bin) atomicAdd(&split[far_bin], 1u);
        }
    }
    __syncthreads();
    // A running sum over the bins' counts, `each` neighbouring bins a thread (at most 1024 bins over at least 128 threads).
    constexpr int kEach = 8;
    const uint32_t each = (n_bins + T - 1) / T, b0 = threadIdx.x * each;
    uint32_t count[kEach], mine = 0;
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
        count[e] = (uint32_t)e < each && b0 + e < n_bins ? base[b0 + e] : 0u;
        mine += count[e];
    }
    uint32_t upto = mine; // of the wave's lanes up to this one
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t below = __shfl_up(upto, off, 64);
        if ((int)(threadIdx.x & 63) >= off) upto += below;
    }
    if ((threadIdx.x & 63) == 63) wave_sum[threadIdx.x >> 6] = upto;
    __syncthreads();
    uint32_t at = upto - mine, total = 0;
    for (int w = 0; w < T / 64; ++w) {
        const uint32_t sum = wave_sum[w];
        if (w < (int)(threadIdx.x >> 6)) at += sum;
        total += sum;
    }
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
        const uint32_t b = b0 + e;
        if ((uint32_t)e < each && b < n_bins) {
            const uint32_t n_split = split[b];
            const uint32_t reserved = count[e] + n_split ? atomicAdd(&cursor[b], count[e] + n_split) : 0u;
            base[b] = at;
            shift[b] = reserved - at;
            split[b] = reserved + count[e];
            at += count[e];
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < P; ++u) {
        if (begin + threadIdx.x + u * T >= end) continue;
#pragma unroll
        for (int c = 0; c < NP; ++c) {
            float weight = 1.0f;
#pragma unroll
            for (int d = 1; d < D; ++d) weight *= (c >> (d - 1)) & 1 ? frac[u][d] : 1 - frac[u][d];
            BinRecord<F> r;
            r.frac = frac[u][0];
#pragma unroll
            for (int f = 0; f < F; ++f) r.g[f] = weight * gy[u][f];
            const uint32_t bin = (place[u][c] >> 12) & 1023u, far_bin = place[u][c] >> 22, slot = base[bin] + (place[u][c] & 4095u);
            r.where = where[u][c] | ((far_bin == bin ? 3u : 1u) << 30);
            sorted[slot] = r;
            bin_of[slot] = (uint16_t)bin;
            if (far_bin != bin) {
                r.where = where[u][c] | (2u << 30);
                const uint32_t to = atomicAdd(&split[far_bin], 1u);
                if (to < capacity) bins[(size_t)far_bin * capacity + to] = r;
            }
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < total; i += T) {
        const uint32_t bin = bin_of[i], to = shift[bin] + i;
        if (to < capacity) bins[(size_t)bin * capacity + to] = sorted[i];
    }
}

// LDS of it with T threads.
template <int D, int F> static size_t bin_lds(const BinPlan &p, unsigned T) {
    uint32_t n_bins = 0;
    for (uint32_t k = 0; k < p.n_levels; ++k) n_bins = std::max(n_bins, 1u << p.bins_log2[k]);
    return (size_t)T * BinShape<D, F>::kPoints * BinShape<D, F>::kPairs * (sizeof(BinRecord<F>) + sizeof(uint16_t)) + (3 * n_bins + 16) * sizeof(uint32_t);
}

// One workgroup sums one bin and stores (or adds) its entries. Bound by the records' bytes and the LDS atomics (two values of two
// features per record). A bin that more records were meant for than it has room for is summed from the points instead, all of them
// passing its workgroup by. The bin's cursor is left at zero for the next part of the batch.
template <int D, int F, typename G>
__global__ void __launch_bounds__(kBinSumThreads)
    grid_bin_sum_kernel(const GridLevels lv, const GridParams gp, const BinPlan bp, const GradLayout dl, const float *__restrict__ xin,
                        const float4 *__restrict__ order, const G *__restrict__ dLdy, uint32_t *__restrict__ cursors,
                        const BinRecord<F> *__restrict__ records, float *__restrict__ grad, long long first, long long last, int store) {
    extern __shared__ double sums[];
    uint32_t k = 0;
    while (k + 1 < bp.n_levels && blockIdx.x >= bp.first_bin[k + 1]) ++k;
    const uint32_t l = bp.level[k], bin = blockIdx.x - bp.first_bin[k];
    const Bins dealt{bp.bins_log2[k], bp.run_log2[k]};
    const uint32_t size = lv.size[l];
    const uint32_t n = bp.places[k]; // the last ones may be beyond the level
    for (uint32_t e = threadIdx.x; e < n * F; e += blockDim.x) sums[e] = 0.0;
    const uint32_t written = cursors[blockIdx.x];
    const BinRecord<F> *const rec = records + bp.first_record[k] + (size_t)bin * bp.capacity[k];
    __syncthreads();
    if (threadIdx.x == 0) cursors[blockIdx.x] = 0;
    if (written <= bp.capacity[k]) {
        constexpr int kAhead = 4; // records of a lane in flight
        for (uint32_t i = threadIdx.x; i < written; i += kAhead * blockDim.x) {
            BinRecord<F> r[kAhead];
#pragma unroll
            for (int a = 0; a < kAhead; ++a) {
                const uint32_t at = i + a * blockDim.x;
                r[a] = rec[at < written ? at : i];
                if (at >= written) r[a].where = 0;
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
    } else {
        for (long long i = first + threadIdx.x; i < last; i += blockDim.x) {
            float x[D], frac[D];
            const long long row = bin_point<D>(xin, order, i, x);
            uint32_t cell[D], near[1 << (D - 1)], far[1 << (D - 1)];
            cell_of<D>(x, lv.scale[l], gp.interpolation, cell, frac);
            pair_entries<D>(cell, size, lv.resolution[l], lv.flags[l], gp.hash_type, near, far);
            const G *dy = dLdy + (dl.by_position ? i : row) * dl.row_stride + l * dl.level_stride;
#pragma unroll
            for (int c = 0; c < (1 << (D - 1)); ++c) {
                const bool near_mine = dealt.bin(near[c]) == bin, far_mine = dealt.bin(far[c]) == bin;
                if (!near_mine && !far_mine) continue;
                float weight = 1.0f;
#pragma unroll
                for (int d = 1; d < D; ++d) weight *= (c >> (d - 1)) & 1 ? frac[d] : 1 - frac[d];
#pragma unroll
                for (int f = 0; f < F; ++f) {
                    const float v = weight * ((float)dy[f] * dl.scale);
                    if (near_mine) lds_add(&sums[dealt.place(near[c]) * F + f], (1 - frac[0]) * v);
                    if (far_mine) lds_add(&sums[dealt.place(far[c]) * F + f], frac[0] * v);
                }
            }
        }
    }
    __syncthreads();
    float *const g = grad + (size_t)lv.offset[l] * F;
    for (uint32_t v = threadIdx.x; v < n * F; v += blockDim.x) {
        const uint32_t e = dealt.entry(bin, v / F);
        if (e >= size) continue;
        float *const to = g + (size_t)e * F + v % F;
        *to = store ? (float)sums[v] : *to + (float)sums[v]; // (store: the bin's entries have no other contributions)
    }
}

bool bin_plan_add(BinPlan *p, uint32_t l, const GridLevels &lv, const GridParams &gp, uint32_t n_dims, uint32_t n_features, size_t M) {
    if (p->n_levels >= kMaxBinned || gp.interpolation == TNN_INTERP_NEAREST) return false;
    const size_t size = lv.size[l], entry = n_features * sizeof(double);
    // A bin stores all of its entries; atomics touch only those that have contributions, and cost as much when there is one for
    // every 16 entries (3-D, 2^22 entries a level: 2^16 points).
    if ((M << (n_dims - 1)) < size / 16) return false;
    // 128 bins a level: a workgroup's share of a bin is then a run of several lines, and the bins of all levels are enough
    // workgroups for the sums (64 or 256: the one pass gains what the other loses). Small levels have fewer, large ones as
    // many as it takes for a bin to fit LDS.
    uint32_t n_log2 = 7;
    while (n_log2 > 0 && (size >> (n_log2 + 4)) == 0) --n_log2;
    while (n_log2 < 31 && ((size >> n_log2) * entry > kBinSliceBytes || (size >> n_log2) > 0x7fff)) ++n_log2;
    const size_t bins = (size_t)1 << n_log2;
    if (bins > kBinMaxBins) return false;
    p->batch = (uint32_t)std::min<size_t>(M, size_t(1) << 19);
    // A hashed level deals out groups of cells that share a run of x and all of the other coordinates, at random: runs as long as
    // leaves a bin 64 groups, down to 16 entries (a line of two features). Dense levels are dealt out in order: consecutive
    // entries to a bin. (Other hashes than the coherent one send every corner by itself.)
    const bool hashed = (lv.flags[l] & 16u) != 0, apart = hashed && gp.hash_type != TNN_HASH_COHERENT_PRIME;
    const double R = (double)lv.resolution[l];
    const auto groups = [&](uint32_t run) { return std::max(R / (double)((size_t)1 << run), 1.0) * std::pow(R, (double)n_dims - 1.0) / (double)bins; };
    uint32_t run_log2 = 4;
    while (((size_t)1 << (run_log2 + n_log2)) < size && (!hashed || apart || groups(run_log2 + 1) >= 64.0)) ++run_log2;
    const size_t places = ((size + ((size_t)1 << (run_log2 + n_log2)) - 1) >> (run_log2 + n_log2)) << run_log2;
    if (places > 0x7fff || places * entry > kBinSliceBytes) return false;
    // What points spread evenly send a bin, and how far above it the fullest bin may be.
    const double split = apart ? 2.0 : 1.0 + 1.0 / (double)((size_t)1 << run_log2);
    const double mean = (double)p->batch * (double)(1u << (n_dims - 1)) * split * (double)places / (double)size;
    const double uneven = hashed && !apart ? std::min(4.0 / std::sqrt(std::max(groups(run_log2), 1.0)), 3.0) : 0.0;
    const double room = std::ceil(((1.2 + uneven) * mean + 8.0 * std::sqrt(mean) + 64.0) / 32.0) * 32.0;
    if (room * (double)bins + p->n_records > 4.0e9) return false;
    const uint32_t k = p->n_levels++;
    p->level[k] = (uint8_t)l;
    p->bins_log2[k] = (uint8_t)n_log2;
    p->run_log2[k] = (uint8_t)run_log2;
    p->places[k] = (uint16_t)places;
    p->capacity[k] = (uint32_t)room;
    p->first_record[k] = p->n_records;
    p->n_records += (uint32_t)room * (uint32_t)bins;
    p->first_bin[k] = p->n_bins;
    p->n_bins += (uint32_t)bins;
    p->first_bin[k + 1] = p->n_bins;
    p->slice_lds = std::max<uint32_t>(p->slice_lds, (uint32_t)(entry * places));
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
    const auto sum = grid_bin_sum_kernel<D, F, G>;
    if (!reserve_lds(reinterpret_cast<const void *>(sum), p.slice_lds))
        return fail(TNN_ERR_HIP, "cannot reserve %u bytes of LDS", p.slice_lds);
    typedef BinShape<D, F> S;
    const auto bin = grid_bin_kernel<D, F, G>;
    if (!reserve_lds(reinterpret_cast<const void *>(bin), bin_lds<D, F>(p, S::kThreads)))
        return fail(TNN_ERR_HIP, "cannot reserve %zu bytes of LDS", bin_lds<D, F>(p, S::kThreads));
    // (as many waves on a CU as it takes whatever LDS the bins need; small bins are over before 16 waves are under way)
    const unsigned sum_threads = p.slice_lds > 32 * 1024 ? kBinSumThreads : kBinSumThreads / 2;
    for (size_t first = 0; first < M; first += p.batch) {
        const size_t last = std::min(M, first + p.batch), n = last - first;
        // (a small batch: half as many threads, twice as many workgroups, while there are fewer than two for every CU)
        const unsigned T = n * p.n_levels < size_t(512) * S::kThreads * S::kPoints ? S::kThreads / 2 : S::kThreads;
        const size_t stretches = (n + T * S::kPoints - 1) / (T * S::kPoints);
        TNN_LAUNCH(bin, dim3((unsigned)((stretches + 7) / 8 * 8 * p.n_levels)), dim3(T), (bin_lds<D, F>(p, T)), s, lv, gp, p, dl, x, order,
                   (const G *)dLdy, cursors, records, (long long)first, (long long)last);
        int rc = check_launch("grid_bin_kernel");
        if (rc) return rc;
        TNN_LAUNCH(sum, dim3(p.n_bins), dim3(sum_threads), p.slice_lds, s, lv, gp, p, dl, x, order, (const G *)dLdy, cursors,
                   (const BinRecord<F> *)records, grad, (long long)first, (long long)last, (int)(overwrite && first == 0));
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

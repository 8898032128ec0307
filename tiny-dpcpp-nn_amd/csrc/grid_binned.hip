// Scatter-add of dL/dy into the levels of a hash-grid's gradient table that are too large for a private copy in LDS
// (include/encodings/grid.h:137-245 of the reference: float atomics, order not defined), without atomics to memory.
//
// The memory side retires an atomic request per 32-byte sector, about 20 * 10^9 a second, and a point of a hashed level
// needs 2^(D-1) or more of them: 2.1 ms for 2^20 points of a 3-D grid of 16 levels (2^19 entries). Here the contributions
// are sorted by destination first:
//   1. grid_bin_kernel deals runs of a level's entries out to bins. A workgroup sorts the contributions of a stretch of points by
//      bin in LDS and writes them as one piece of consecutive records, with a table of where each bin's begin. The two corners
//      along the first dimension are neighbouring entries in a dense level and differ in the low bits of the index in a
//      coherently hashed one, so nearly always they share a bin and travel as one record of two entries.
//      (Long runs of entries share more; but a hashed level's runs longer than its x range are dealt out by the other
//      dimensions alone, and in 2-D the few hundred values of y fill the bins very unevenly: bin_plan_add.)
//   2. grid_bin_sum_kernel takes a bin at a time, sums its records of all pieces into a copy of the bin's entries in LDS and
//      writes the entries to the table as whole lines.
// A record of two features is 16 bytes written once and read once, where the two atomic requests it replaces occupy the
// memory side for 64. A piece has room for whatever its points need, so no bin can be too full: points that crowd a few cells
// make some bins longer than others, and that is all. (Bins of a fixed size, filled by all workgroups through shared cursors, are
// as fast for points spread evenly, but what finds no room has to go elsewhere. 2^20 points, 3-D, 2^19 entries, whole scatter, from
// points in the inner 90 % of the cube / in a cube of 5 % of the side: the overfull bins summed from the points 4.0 / 5.8 ms, the surplus
// added with atomics 0.76 / 36 ms, pieces 0.75 / 3.9 ms; evenly spread 0.74, 0.76 and 0.75 ms. Pieces now: 0.54 / 3.1 ms, evenly spread 0.54.)
// Measured, 2^20 points, 3-D, 2^19 entries, the ten finest levels: 2 x (99 + 97) us; as atomics 1.5 ms.
#include "grid_binned.h"
#include "mlp_tile.h"
#include "train_reduce.h"

#include <algorithm>
#include <cmath>
#include <iterator>

namespace tnn {

constexpr int kBinSumThreads = 1024; // at most
constexpr uint32_t kBinSumGroup = 8;    // lanes that walk through a share of a bin's records together
constexpr int kBinPiecesEach = 4;        // pieces a thread of the sums looks up, at most
// Copies of the sums of a crowded bin (grid_bin_sum_kernel): at most sixteen, in 8 KB and what keeps an entry's copies in different banks. Bins of more than 4 KB have one.
constexpr uint32_t kBinCopiesLog2 = 4, kBinCopySkew = 2; // (doubles between two copies)
constexpr size_t kBinCopiesBytes = 8 * 1024 + (sizeof(double) * kBinCopySkew << kBinCopiesLog2);
constexpr uint32_t kBinNeighbours = 16;  // consecutive bins on an XCD
constexpr uint32_t kBinPiecePad = 144; // records between two pieces, at most (bin_launch), so that workgroups in step do not all write to the same channels

// A binning workgroup: its threads (at most), the points of a thread, and the pairs of corners it sorts in LDS. 2048 records of 16
// bytes let four workgroups of 8 waves share a CU, whose phases (loads, LDS, stores) then overlap; wider records take half as many.
template <int D, int F> struct BinShape {
    static constexpr int kThreads = F <= 2 ? 512 : 256;
    static constexpr int kPoints = D == 2 && F <= 2 ? 2 : 1;
    static constexpr int kPairs = 1 << (D - 1);
    static constexpr int kRecords = kThreads * kPoints * kPairs;
};

// Entry e of a level: its bin and its place there. Runs of 2^run_log2 entries go to the bins in turn, every round of them starting
// at another bin: a region of a dense level then meets all bins about equally, also where a row of the level is a multiple of a round.
struct Bins {
    uint32_t n_log2, run_log2;
    __device__ __forceinline__ uint32_t turn(uint32_t round) const { return (round * 2654435769u) >> 22; }
    __device__ __forceinline__ uint32_t bin(uint32_t e) const { return ((e >> run_log2) + turn(e >> (run_log2 + n_log2))) & ((1u << n_log2) - 1); }
    __device__ __forceinline__ uint32_t place(uint32_t e) const { return ((e >> (run_log2 + n_log2)) << run_log2) | (e & ((1u << run_log2) - 1)); }
    __device__ __forceinline__ uint32_t entry(uint32_t bin, uint32_t place) const {
        const uint32_t round = place >> run_log2, run = (bin - turn(round)) & ((1u << n_log2) - 1);
        return (((round << n_log2) | run) << run_log2) | (place & ((1u << run_log2) - 1));
    }
};

// Two neighbouring entries of a bin, the position between them, and the gradient times the weights of the other dimensions.
template <int F> struct alignas(F == 1 ? 4 : F == 2 ? 16 : 8) BinRecord {
    uint32_t where; // entry of the near side (15 bits), of the far side (15 bits), whether either is meant (bits 30, 31)
    float frac;
    float g[F];
};

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

// The sum up to each lane of a row of 16 (DPP row_shr).
__device__ __forceinline__ uint32_t row_sums(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true);
    return v;
}

// The sum of the values of the waves in front of this one, and of all: a wave's value a lane.
__device__ __forceinline__ uint32_t sums_in_front(const uint32_t *__restrict__ of_wave, uint32_t &total) {
    static_assert(kBinSumThreads / 64 <= 16, "a row of 16 lanes holds the waves' values");
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t upto = row_sums(lane < blockDim.x / 64 ? of_wave[lane] : 0u);
    total = (uint32_t)__builtin_amdgcn_readlane((int)upto, 15);
    return wave > 0 ? (uint32_t)__builtin_amdgcn_readlane((int)upto, (int)wave - 1) : 0u;
}

// What the threads of a workgroup in front of this one have, and what all have.
__device__ __forceinline__ uint32_t running_sum(uint32_t mine, uint32_t *__restrict__ wave_sum, uint32_t &total) {
    // of the wave's lanes up to this one: rows of 16 lanes first (DPP row_shr), then the last lane of a row to the rows above
    uint32_t upto = row_sums(mine);
    upto += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)upto, 0x142, 0xa, 0xf, false); // row_bcast:15 into rows 1 and 3
    upto += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)upto, 0x143, 0xc, 0xf, false); // row_bcast:31 into rows 2 and 3
    if ((threadIdx.x & 63) == 63) wave_sum[threadIdx.x >> 6] = upto;
    __syncthreads();
    return upto - mine + sums_in_front(wave_sum, total);
}

// Where a bin's records in a piece begin and end (two 16-bit numbers, side by side in a word): by four bins, then by pieces. A workgroup of the sums reads its bin's
// of all pieces, eight pieces to a line that it shares with three neighbouring bins; with all bins of a piece side by side it read a
// line for each (3-D, 2^19 points, 10 levels: 123.5 us, now 119; 2^18 in the caller's order 95, 89).
__device__ __forceinline__ size_t run_slot(uint32_t first_quad, uint32_t bin, uint32_t n_stretches, uint32_t stretch) {
    return ((size_t)(first_quad + bin / 4) * n_stretches + stretch) * 4 + bin % 4;
}

// One workgroup bins kPoints points a thread of one level: it counts its records per bin, which gives every record its place among
// them, sorts the records in LDS and writes them to its piece of the scratch, so that a wave stores whole lines. A far side that
// lies in another bin than the near side is a record of its own; LDS has room for one in eight, those beyond go to the
// piece directly. The levels of the same points are consecutive workgroups of one XCD, which shares the rows of dL/dy between
// them in its L2.
// No one unit bounds it (3-D, 2^19 points, 10 levels, 99 us): 346 MB written, the records all in whole 64-byte requests, at 3.5 TB/s where a
// fill reaches 6.9; the vector units are at work 45 % of the time, LDS a sixth, and a wave waits for 41 % of its.
// TAKEN: the reduction of the training kernel that left dL/dy (and what it clears) is the first workgroups of this launch: both wait for that kernel only, and what adds to the table
// waits for both. It was a launch of its own of 4 to 7 us, a chain of loads and one sum, and makes this one longer (2-D, 2^18 points, with Adam: 6.9 us gone, 15.3 -> 18.1 here). Optimisation step with the
// ordering, 16 levels, us, before / now: 2-D, 2^17 entries a level, 20 000 points 68.4 / 64.6, 2^15, 2^16 points 82.0 / 77.4, 2^19, 2^18 210 / 203; 3-D, 2^19, 2^17 257 / 253; a module's forward and backward pass,
// 2-D, 2^19, 2^18 177 / 171. Registers for eight waves a SIMD, as without.
template <int D, int F, typename G, typename TAKEN = std::false_type>
__global__ void __launch_bounds__((BinShape<D, F>::kThreads), (std::is_same<TAKEN, TrainReduce>::value ? 8 : 1))
    grid_bin_kernel(const GridParams gp, const BinPlan bp, const GradLayout dl, const float *__restrict__ xin,
                    const float4 *__restrict__ order, const G *__restrict__ dLdy, uint32_t *__restrict__ runs, BinRecord<F> *__restrict__ records,
                    long long first, long long last, uint32_t n_stretches, uint32_t pitch, uint32_t room, const TAKEN taken, uint32_t taken_blocks) {
    typedef BinShape<D, F> S;
    constexpr int NP = S::kPairs, P = S::kPoints;
    static_assert(S::kRecords <= 4096 && kBinMaxBins <= 1024, "a record's place is packed into 12 + 10 + 10 bits");
    const uint32_t T = blockDim.x;
    extern __shared__ __align__(16) unsigned char bin_smem[];
    if constexpr (std::is_same<TAKEN, TrainReduce>::value) {
        if (blockIdx.x < taken_blocks) { // (a multiple of 8: the others' numbers say which XCD they are on)
            const uint32_t n = taken.clear.reduce_blocks;
            if (blockIdx.x >= n) {
                clear_range(taken.clear, blockIdx.x - n, taken_blocks - n);
                return;
            }
            float4(*const red)[16] = reinterpret_cast<float4(*)[16]>(bin_smem);
            const auto reduce = [&](auto adam, auto threads) __attribute__((always_inline)) {
                train_reduce_block<G, decltype(adam)::value, decltype(threads)::value, true>(taken.partials, taken.loss_partials, taken.n_partials, taken.n_elems,
                                                                                            static_cast<G *>(taken.dW_T), taken.dW_f32, taken.loss_sum, taken.adam,
                                                                                            taken.packed, blockIdx.x, red);
            };
            if (T == 512) {
                if (taken.use_adam) reduce(std::true_type{}, std::integral_constant<int, 512>{});
                else reduce(std::false_type{}, std::integral_constant<int, 512>{});
            } else {
                if (taken.use_adam) reduce(std::true_type{}, std::integral_constant<int, 256>{});
                else reduce(std::false_type{}, std::integral_constant<int, 256>{});
            }
            return;
        }
    }
    const uint32_t block = blockIdx.x - (std::is_same<TAKEN, TrainReduce>::value ? taken_blocks : 0u);
    BinRecord<F> *const sorted = reinterpret_cast<BinRecord<F> *>(bin_smem);
    uint32_t *const base = reinterpret_cast<uint32_t *>(sorted + room); // records per bin, then the place of the bin's first one
    const uint32_t turn = block / 8, k = turn % bp.n_levels, stretch = (turn / bp.n_levels) * 8 + block % 8;
    if (stretch >= n_stretches) return;
    const long long begin = first + (long long)stretch * (T * P);
    const long long end = begin + T * P < last ? begin + T * P : last;
    const BinLevel at_level = bp.at[k];
    const Bins dealt{at_level.bins_log2, at_level.run_log2};
    const uint32_t l = at_level.level, n_bins = 1u << dealt.n_log2;
    uint32_t *const split = base + n_bins; // the same for far sides in another bin, then the place of the next of them
    uint32_t *const wave_sum = split + n_bins;
    const uint32_t size = at_level.size, res = at_level.resolution, flags = at_level.flags;
    const float scale = at_level.scale;
    BinRecord<F> *const piece = records + ((size_t)k * n_stretches + stretch) * pitch;

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
    constexpr int kEach = 8; // neighbouring bins of a thread, at most (1024 bins, 128 threads)
    const uint32_t each = (n_bins + T - 1) / T, b0 = threadIdx.x * each;
    uint32_t count[kEach], apart[kEach], mine = 0, total;
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
        count[e] = apart[e] = 0;
        if ((uint32_t)e >= each) continue; // (the same for all threads)
        const bool any = b0 + e < n_bins;
        count[e] = any ? base[b0 + e] : 0u;
        apart[e] = any ? split[b0 + e] : 0u;
        mine += count[e] + apart[e];
    }
    uint32_t at = running_sum(mine, wave_sum, total);
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
        if ((uint32_t)e >= each) break;
        const uint32_t b = b0 + e;
        if (b < n_bins) {
            base[b] = at;
            split[b] = at + count[e];
            const uint32_t next = at + count[e] + apart[e];
            runs[run_slot(at_level.first_quad, b, n_stretches, stretch)] = at | (next << 16);
            at = next;
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
            const uint32_t bin = (place[u][c] >> 12) & 1023u, far_bin = place[u][c] >> 22;
            const auto put = [&](uint32_t to, uint32_t sides) {
                r.where = where[u][c] | (sides << 30);
                if (to < room) sorted[to] = r;
                else piece[to] = r;
            };
            put(base[bin] + (place[u][c] & 4095u), far_bin == bin ? 3u : 1u);
            if (far_bin != bin) put(atomicAdd(&split[far_bin], 1u), 2u);
        }
    }
    __syncthreads();
    const uint32_t staged = total < room ? total : room;
    // The records leave with the streaming hint, in words that lie side by side whatever a record's size: they are read by whichever XCD takes their bins, and
    // written plainly they drove rows of dL/dy and lines of points out of this one's L2 (3-D, 2^18 points in the caller's order, binning and sums 157 -> 142 us;
    // 2^20 in cell order 412 -> 396; eight features, 2^17 points 337 -> 330 the whole scatter; 2-D, 2^18: binning 17.5 -> 15.7, sums 22.3 -> 23.4).
    typedef uint32_t word_t __attribute__((ext_vector_type(F == 1 ? 1 : F == 2 ? 4 : 2)));
    constexpr uint32_t kWords = sizeof(BinRecord<F>) / sizeof(word_t);
    const word_t *const from = reinterpret_cast<const word_t *>(sorted);
    word_t *const to = reinterpret_cast<word_t *>(piece);
    for (uint32_t i = threadIdx.x; i < staged * kWords; i += T) __builtin_nontemporal_store(from[i], to + i);
}

// A workgroup sums a bin and stores (or adds) its entries, a plane of sums a feature (lds_add; interleaved 25.0 -> 22.3 us, 2-D,
// 2^18 points), then the bin that lies a grid further on. The bin's runs of records in the pieces follow each other here (`first`: records in front of a
// piece's run); eight lanes take an equal share of them all, whatever the runs' lengths, and walk from run to run. Neighbouring bins, whose
// runs share lines, are workgroups of one XCD, sixteen at a time. kAhead: records of a lane in flight.
// Long bins are bound by the LDS atomics, two entries of F values a record (3-D, 2^19 points, 10 levels, 97 us: LDS at work 66 % of the time, 490 MB read). Short ones were bound by what comes before the first record: a workgroup a
// bin, 3-D, 2^15 points, took 30 us, 18 of them without a record read or an entry written. So a workgroup stays for several of the shortest (launch_binned): where the next bin's
// runs lie is loaded while this one's records are summed, and sums are cleared as they are read. What was left of it were instructions, eight and more waves a bin of them:
// the prefix sums over the waves are a value a lane, a wave without pieces leaves the look-up out, and two entries leave together (3-D, 2^15 points 30 -> 20.3 us,
// 100 003 46 -> 37.5, 2^19 101 -> 96; 2-D, 20 011 points 11.3 -> 8.2, 2^16 12.3 -> 9.7, 2^18 23.4 -> 20.8).
// Points that crowd a part of the volume meet a few of a coarse level's entries only: lanes queue up on them, and the longest bin is the kernel's time. A small bin
// has room for copies of its sums, and short bins take one as if they had not (whole scatter, 2^16 points, even / in a square or cube of 5 % of the side, before the
// coarsest levels were binned, then, with copies: 2-D, 2^19 entries 51 / 77, 40 / 124, 40 / 72 us; 3-D 66 / 313, 48 / 394, 48 / 231; 2-D, 2^15 entries 43 / 84, 35 / 120, 35 / 72).
template <int F, int kAhead>
__global__ void __launch_bounds__(kBinSumThreads, F <= 2 ? 8 : 4)
    grid_bin_sum_kernel(const BinPlan bp, const uint32_t *__restrict__ runs_of, const BinRecord<F> *__restrict__ records,
                        float *__restrict__ grad, uint32_t n_stretches, uint32_t pitch, int store) {
    constexpr uint32_t kWaves = kBinSumThreads / 64, kGroup = kBinSumGroup;
    constexpr int kEach = kBinPiecesEach;
    extern __shared__ __align__(16) double sums[];
    uint32_t *const wave_sum = reinterpret_cast<uint32_t *>(sums + bp.sums_lds / sizeof(double));
    uint32_t *const wave_runs = wave_sum + kWaves;
    uint32_t *const group_run = wave_runs + kWaves;       // run that a group's first record is in
    uint32_t *const first = group_run + kBinSumThreads / kGroup; // records in front of a run
    uint32_t *const start = first + n_stretches + 1;       // place of the run's first record in the pieces, less `first`
    const uint32_t threads_log2 = 31 - __builtin_clz(blockDim.x); // (a power of two)
    const uint32_t each = (n_stretches + blockDim.x - 1) >> threads_log2;
    const bool has_pieces = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63u) * each < n_stretches; // (a wave without any has nothing to look up and nothing to add up)
    const auto first_piece = [&]() __attribute__((always_inline)) {
        uint32_t s0 = threadIdx.x * each;
        asm volatile("" : "+v"(s0)); // (what follows from it is formed where it is used: kept over the bins it spills)
        return s0;
    };
    // (the grid is a multiple of 8 kBinNeighbours: a workgroup's bins grow, and are one XCD's)
    const auto bin_of = [&](uint32_t block) { return (block / (8 * kBinNeighbours) * 8 + block % 8) * kBinNeighbours + block / 8 % kBinNeighbours; };
    // (the list of the levels' first bins over the lanes and the level's numbers side by side: two loads, where an entry and a number at a time were
    // waited for one after the other: 3-D, 100 003 points 46.3 -> 44.0 us)
    const uint32_t lane = threadIdx.x & 63, later_bin = lane < kMaxBinned - 1 ? bp.later_bin[lane] : ~0u;
    const auto level_of = [&](uint32_t number) { return (uint32_t)__popcll(__ballot(number >= later_bin)); };
    uint32_t ends[kEach]; // where the bin's records begin in the piece, and where the next bin's do
    const auto look_up = [&](uint32_t number) __attribute__((always_inline)) {
        const BinLevel &at_level = bp.at[level_of(number)];
        const uint32_t *const runs_here = runs_of + run_slot(at_level.first_quad, number - at_level.first_bin, n_stretches, 0);
        const uint32_t s0 = first_piece();
#pragma unroll
        for (int e = 0; e < kEach; ++e) {
            if ((uint32_t)e >= each) break;
            ends[e] = s0 + e < n_stretches ? runs_here[(size_t)(s0 + e) * 4] : 0u;
        }
    };
    uint32_t number = bin_of(blockIdx.x);
    if (number >= bp.n_bins) return;
    look_up(number);
    for (uint32_t e = threadIdx.x; e < bp.slice_lds / sizeof(double); e += blockDim.x) sums[e] = 0.0;
    for (uint32_t block = blockIdx.x + gridDim.x;; block += gridDim.x) {
        const uint32_t k = level_of(number);
        const BinLevel at_level = bp.at[k];
        const uint32_t n = at_level.places; // the last ones may be beyond the level
        uint32_t count[kEach], begin[kEach], mine = 0, run = 0, runs = 0; // runs that hold any records: in front of this thread's, in its wave
        if (has_pieces) {
#pragma unroll
            for (int e = 0; e < kEach; ++e) {
                if ((uint32_t)e >= each) break; // (the same for all threads)
                begin[e] = ends[e] & 0xffffu;
                count[e] = (ends[e] >> 16) - begin[e];
                mine += count[e];
                const unsigned long long any = __ballot(count[e] != 0);
                run += __popcll(any & ((1ull << lane) - 1));
                runs += __popcll(any);
            }
        }
        if (lane == 0) wave_runs[threadIdx.x >> 6] = runs;
        uint32_t total, n_runs, at = running_sum(mine, wave_sum, total);
        run += sums_in_front(wave_runs, n_runs);
        // (whole rounds of a group: all but the last groups then have all of their lanes at work)
        const uint32_t share = ((total + blockDim.x - 1) >> threads_log2) * kGroup, s0 = first_piece();
        if (has_pieces) {
#pragma unroll
            for (int e = 0; e < kEach; ++e) {
                if ((uint32_t)e >= each) break;
                if (count[e] == 0) continue;
                for (uint32_t g = (at + share - 1) / share; g * share < at + count[e]; ++g) group_run[g] = run;
                first[run] = at;
                start[run++] = (s0 + e) * pitch + begin[e] - at;
                at += count[e];
            }
        }
        if (threadIdx.x == 0) first[n_runs] = total;
        // Of a bin with more than eight records a lane, whose points are crowded where even ones leave it a fraction of that, neighbouring lanes add to copies of their own.
        const uint32_t copies = total > 8 * blockDim.x ? 1u << at_level.copies_log2 : 1u, copy = n * F + kBinCopySkew;
        if (copies > 1)
            for (uint32_t e = n * F + threadIdx.x; e < copies * copy; e += blockDim.x) sums[e] = 0.0;
        const uint32_t next = bin_of(block);
        if (next < bp.n_bins) look_up(next);
        __syncthreads();
        const BinRecord<F> *const rec = records + (size_t)k * n_stretches * pitch;
        const uint32_t group = threadIdx.x / kGroup, end = (group + 1) * share < total ? (group + 1) * share : total;
        double *const own = sums + (threadIdx.x & (copies - 1)) * copy;
        uint32_t i = group * share + threadIdx.x % kGroup, s = i < end ? group_run[group] : 0u;
        for (; i < end; i += kAhead * kGroup) {
            uint32_t at_a[kAhead];
#pragma unroll
            for (int a = 0; a < kAhead; ++a) {
                // (lanes past the end walk to the last run and read its last record)
                const uint32_t wanted = i + a * kGroup < total ? i + a * kGroup : total - 1;
                while (wanted >= first[s + 1]) ++s; // (first[n_runs] is beyond every record)
                at_a[a] = start[s] + wanted;
            }
            BinRecord<F> r[kAhead];
#pragma unroll
            for (int a = 0; a < kAhead; ++a) r[a] = rec[at_a[a]];
#pragma unroll
            for (int a = 0; a < kAhead; ++a) {
                const uint32_t where = i + a * kGroup < end ? r[a].where : 0u, near = where & 0x7fff, far = (where >> 15) & 0x7fff;
                if (where & (1u << 30)) {
#pragma unroll
                    for (int f = 0; f < F; ++f) lds_add(&own[f * n + near], (1 - r[a].frac) * r[a].g[f]);
                }
                if (where & (1u << 31)) {
#pragma unroll
                    for (int f = 0; f < F; ++f) lds_add(&own[f * n + far], r[a].frac * r[a].g[f]);
                }
            }
        }
        __syncthreads();
        const Bins dealt{at_level.bins_log2, at_level.run_log2};
        const uint32_t bin = number - at_level.first_bin, size = at_level.size;
        float *const g = grad + (size_t)at_level.offset * F;
        if (store && ((size | at_level.offset) & 1) == 0) { // the bin's entries have no other contributions
            // Two neighbouring entries a thread: a run has an even number, and the table is 16-byte aligned.
            constexpr int kStore = 2 * F < 4 ? 2 * F : 4;
            typedef float store_t __attribute__((ext_vector_type(kStore)));
            typedef double pair_t __attribute__((ext_vector_type(2)));
            for (uint32_t v = 2 * threadIdx.x; v < n; v += 2 * blockDim.x) {
                const uint32_t e = dealt.entry(bin, v);
                float sum[2 * F];
#pragma unroll
                for (int f = 0; f < F; ++f) {
                    pair_t *const both = reinterpret_cast<pair_t *>(sums + f * n + v);
                    pair_t d = *both;
                    *both = pair_t{0.0, 0.0};
                    for (uint32_t c = 1; c < copies; ++c) {
                        pair_t *const other = reinterpret_cast<pair_t *>(sums + c * copy + f * n + v);
                        d += *other;
                        *other = pair_t{0.0, 0.0};
                    }
                    sum[f] = (float)d[0];
                    sum[F + f] = (float)d[1];
                }
                if (e >= size) continue;
                store_t *const to = reinterpret_cast<store_t *>(g + (size_t)e * F);
#pragma unroll
                for (int q = 0; q < 2 * F / kStore; ++q) {
                    store_t w;
#pragma unroll
                    for (int j = 0; j < kStore; ++j) w[j] = sum[q * kStore + j];
                    to[q] = w;
                }
            }
        } else { // (a tiled level may have any number of entries, and begin anywhere)
            for (uint32_t v = threadIdx.x; v < n * F; v += blockDim.x) {
                const uint32_t e = dealt.entry(bin, v / F), from = v % F * n + v / F;
                double sum = 0.0;
                for (uint32_t c = 0; c < copies; ++c) {
                    sum += sums[c * copy + from];
                    sums[c * copy + from] = 0.0;
                }
                if (e >= size) continue;
                float *const to = g + (size_t)e * F + v % F;
                *to = store ? (float)sum : *to + (float)sum;
            }
        }
        if (next >= bp.n_bins) return;
        number = next;
    }
}

bool bin_plan_add(BinPlan *p, uint32_t l, const GridLevels &lv, const GridParams &gp, uint32_t n_dims, uint32_t n_features, size_t M) {
    if (p->n_levels >= kMaxBinned || gp.interpolation == TNN_INTERP_NEAREST) return false;
    const size_t size = lv.size[l], entry = n_features * sizeof(double);
    // A bin stores all of its entries; atomics touch only those that have contributions, and cost as much when there is one for
    // every 16 entries (3-D, 2^22 entries a level: 2^16 points).
    if ((M << (n_dims - 1)) < size / 16) return false;
    // 128 bins a level: a workgroup's share of a bin is then a run of several lines, and the bins of all levels are enough
    // workgroups for the sums. 256 where 128 would take more than 32 KB of LDS each, so that four workgroups share a CU while some wait
    // for their first records (2-D, 2^18 points: 29 -> 27 us; 3-D, 2^16: 48 -> 40; four features, 2^19 262 -> 236); but up to 64 KB, two workgroups of
    // 1024 threads, where a bin of 256 would still hold 8192 records, whose runs then share half as many lines with other bins' (256 and 128
    // bins: 3-D, 2^19 points 119, 108; 2^18 89, 88; 2^17 51, 57; 2-D, 2^19 66, 67; 2^18 22, 27). Small
    // levels have fewer, large ones as many as it takes for a bin to fit LDS.
    const bool long_bins = (std::min<size_t>(M, kBinBatch) << (n_dims - 1)) >> 8 >= 8192;
    const auto bins_log2 = [&](size_t slice) {
        uint32_t n = (size >> 7) * entry > slice ? 8 : 7;
        while (n > 0 && (size >> (n + 4)) == 0) --n;
        while (n < 31 && ((size >> n) * entry > kBinSliceBytes || (size >> n) > 0x7fff)) ++n;
        return n;
    };
    const uint32_t short_log2 = bins_log2(32 * 1024), n_log2 = long_bins ? bins_log2(64 * 1024) : short_log2;
    const size_t bins = (size_t)1 << n_log2;
    if (bins > kBinMaxBins) return false;
    p->batch = (uint32_t)std::min<size_t>(M, kBinBatch);
    // A hashed level deals out groups of cells that share a run of x and all of the other coordinates, at random: runs as long as
    // leaves a bin 64 groups, down to 16 entries (a line of two features). A dense level deals out runs of that length: points that
    // crowd a region of it then still meet all of its bins. (Other hashes than the coherent one send every corner by itself,
    // at random: consecutive entries to a bin.)
    const bool hashed = (lv.flags[l] & 16u) != 0, apart = hashed && gp.hash_type != TNN_HASH_COHERENT_PRIME;
    const double R = (double)lv.resolution[l];
    const double rows = n_dims == 2 ? R : R * R; // (a product: std::pow was half of a plan's time, three of which a pass makes)
    const auto groups = [&](uint32_t run) { return std::max(R / (double)((size_t)1 << run), 1.0) * rows / (double)bins; };
    uint32_t run_log2 = 4;
    while (((size_t)1 << (run_log2 + n_log2)) < size && (apart || (hashed && groups(run_log2 + 1) >= 64.0))) ++run_log2;
    const size_t places = ((size + ((size_t)1 << (run_log2 + n_log2)) - 1) >> (run_log2 + n_log2)) << run_log2;
    if (places > 0x7fff || places * entry > kBinSliceBytes) return false;
    const auto sums_bytes = [&](uint32_t copies) { return copies ? (entry * places + sizeof(double) * kBinCopySkew) << copies : entry * places; };
    uint32_t copies_log2 = 0;
    while (copies_log2 < kBinCopiesLog2 && sums_bytes(copies_log2 + 1) <= kBinCopiesBytes) ++copies_log2;
    if (p->n_levels == 0) std::fill(std::begin(p->later_bin), std::end(p->later_bin), ~0u);
    else p->later_bin[p->n_levels - 1] = p->n_bins;
    p->at[p->n_levels++] = BinLevel{l, lv.offset[l], lv.size[l], lv.resolution[l], lv.flags[l], lv.scale[l], n_log2, run_log2, (uint32_t)places, copies_log2, p->n_bins, p->n_quads};
    p->n_bins += (uint32_t)bins;
    p->room_bins += 1u << short_log2;
    p->n_quads += (uint32_t)((bins + 3) / 4);
    p->slice_lds = std::max<uint32_t>(p->slice_lds, (uint32_t)sums_bytes(0));
    p->sums_lds = std::max<uint32_t>(p->sums_lds, (uint32_t)sums_bytes(copies_log2));
    return true;
}

// The launches of a part of the batch.
struct BinLaunch {
    uint32_t threads, stretch, n_stretches; // of a binning workgroup, its points, and how many there are
    uint32_t room, pitch;                   // records that fit its LDS; from one piece to the next
    size_t offset_bytes, scratch_bytes;
};
// A batch of fewer points times levels has binning workgroups of half as many threads, and twice as many of them: fewer than two for every CU otherwise.
template <int D, int F> constexpr size_t kSmallBatch = size_t(512) * BinShape<D, F>::kThreads * BinShape<D, F>::kPoints;

template <int D, int F> static BinLaunch bin_launch(const BinPlan &p) {
    typedef BinShape<D, F> S;
    BinLaunch b;
    b.threads = (size_t)p.batch * p.n_levels < kSmallBatch<D, F> ? S::kThreads / 2 : S::kThreads;
    b.stretch = b.threads * S::kPoints;
    b.n_stretches = (p.batch + b.stretch - 1) / b.stretch;
    b.room = b.stretch * S::kPairs / 8 * 9;
    // Room for two records a pair of corners (were every far side a record of its own), and for kBinPiecePad records a piece and two bytes a bin and piece, which hold the table of
    // runs, four bytes each, and leave the rest between the pieces (3-D, 2^19 entries: 112 records of 144 a piece).
    const size_t pieces = (size_t)p.n_levels * b.n_stretches, least = 2 * b.stretch * S::kPairs;
    const size_t room = (((size_t)b.n_stretches * p.room_bins * 2 + 255) & ~(size_t)255) + pieces * (least + kBinPiecePad) * sizeof(BinRecord<F>);
    b.offset_bytes = ((size_t)b.n_stretches * p.n_quads * 4 * sizeof(uint32_t) + 255) & ~(size_t)255;
    b.pitch = (uint32_t)least;
    if (room > b.offset_bytes) b.pitch = (uint32_t)std::max(least, (room - b.offset_bytes) / (pieces * sizeof(BinRecord<F>)) / 8 * 8);
    b.scratch_bytes = std::max(room, b.offset_bytes + pieces * b.pitch * sizeof(BinRecord<F>));
    return b;
}

size_t bin_scratch_bytes(const BinPlan &p, uint32_t n_dims, uint32_t n_features) {
    if (!p.n_levels) return 0;
#define TNN_BIN_BYTES(F) (n_dims == 2 ? bin_launch<2, F>(p) : bin_launch<3, F>(p)).scratch_bytes
    switch (n_features) {
    case 1: return TNN_BIN_BYTES(1);
    case 2: return TNN_BIN_BYTES(2);
    case 4: return TNN_BIN_BYTES(4);
    default: return TNN_BIN_BYTES(8);
    }
#undef TNN_BIN_BYTES
}

size_t bin_scratch_bytes_up_to(BinPlan p, uint32_t n_dims, uint32_t n_features) {
    if (!p.n_levels) return 0;
    // (the largest batch of small workgroups has twice the pads and tables of a slightly larger one)
#define TNN_BIN_SMALL(F) (n_dims == 2 ? kSmallBatch<2, F> : kSmallBatch<3, F>)
    const size_t small = n_features == 1 ? TNN_BIN_SMALL(1) : n_features == 2 ? TNN_BIN_SMALL(2) : n_features == 4 ? TNN_BIN_SMALL(4) : TNN_BIN_SMALL(8);
#undef TNN_BIN_SMALL
    const size_t bytes = bin_scratch_bytes(p, n_dims, n_features);
    if ((size_t)p.batch * p.n_levels < small) return bytes;
    p.batch = (uint32_t)((small - 1) / p.n_levels);
    return std::max(bytes, bin_scratch_bytes(p, n_dims, n_features));
}

template <int D, int F, typename G>
static int launch_binned(const BinPlan &p, const GridParams &gp, const GradLayout &dl, const float *x, const float4 *order, const void *dLdy,
                         float *grad, bool overwrite, size_t M, void *scratch, hipStream_t s, BinStage stage, const TrainReduce *reduce) {
    typedef BinShape<D, F> S;
    const BinLaunch b = bin_launch<D, F>(p);
    uint32_t *const runs = static_cast<uint32_t *>(scratch);
    BinRecord<F> *const records = reinterpret_cast<BinRecord<F> *>(static_cast<char *>(scratch) + b.offset_bytes);
    uint32_t most_bins = 0;
    for (uint32_t k = 0; k < p.n_levels; ++k) most_bins = std::max(most_bins, 1u << p.at[k].bins_log2);
    const auto bin = grid_bin_kernel<D, F, G>;
    const size_t bin_lds = (size_t)b.room * sizeof(BinRecord<F>) + (2 * most_bins + 16) * sizeof(uint32_t);
    const size_t sum_lds = p.sums_lds + (2 * kBinSumThreads / 64 + kBinSumThreads / kBinSumGroup + 2 * b.n_stretches + 1) * sizeof(uint32_t);
    // (about as many waves on a CU as it holds, whatever LDS the bins need: small bins are over before many are under way)
    unsigned sum_threads = p.slice_lds > 48 * 1024 ? kBinSumThreads : p.slice_lds > 20 * 1024 ? kBinSumThreads / 2 : kBinSumThreads / 4;
    while (sum_threads * kBinPiecesEach < b.n_stretches) sum_threads *= 2;
    // Records a lane has of an even spread, and those that are split (one in sixteen of a level with runs of 16 entries): five in flight where four and the
    // split ones make five (2-D, 2^18 points 27.3 -> 24.9 us; where five make a round less of more records, the whole scatter is within 1 % with four and with five, from nine a lane
    // to fifteen, and one feature 2 to 3 % faster with five), two where that is all there are, and
    // the rest would be instructions for nothing (3-D, 2^15 points, with the stores of two entries: 25.4 -> 20.3).
    const size_t a_lane = ((size_t)p.batch * S::kPairs / 16 * 17 / most_bins + sum_threads - 1) / sum_threads;
    const auto sum = a_lane <= 2 ? grid_bin_sum_kernel<F, 2> : a_lane == 5 ? grid_bin_sum_kernel<F, 5> : grid_bin_sum_kernel<F, 4>;
    if (!reserve_lds(reinterpret_cast<const void *>(bin), bin_lds) || !reserve_lds(reinterpret_cast<const void *>(sum), sum_lds))
        return fail(TNN_ERR_HIP, "cannot reserve %zu and %zu bytes of LDS", bin_lds, sum_lds);
    // A workgroup stays for several bins (as many workgroups as threads and LDS of the CUs allow, in whole rounds of bins; the registers of eight features let three in of four,
    // and the fourth starts where one is through: 3-D, 2^17 entries, 2^13 points 26.3 us, with three 25.8, but of twenty points 59 and 67) where what comes before a bin's first record is most of its
    // time: bins of 256 records, of 128 with eight features. Longer ones have a workgroup each, which starts wherever one is through: a workgroup that met several bins
    // of crowded points was the kernel's time. Twenty points only, whole scatter, us, before workgroups stayed for bins, for all of them, now: 2-D, 2^19 entries, 2^16 points
    // 113, 137, 106; 2^18 358, 631, 321; 3-D, 2^17 points 317, 411, 294; eight features 766, 1087, 686. Even points, for all of them, now: 2-D, 2^16 points 39.9, 41.7; 2^18
    // 75.6, 78.3; 3-D, 2^15 points 35.4, 38.7; 2^16 48.1, 48.4; 2^18 151, 146; 2^19 268, 255. Bins of 256 records, a workgroup each, now: 3-D, 2^14 points 32.5, 30.1.
    constexpr size_t kRound = 8 * kBinNeighbours;
    size_t sum_blocks = (p.n_bins + kRound - 1) / kRound * kRound;
    if ((size_t)p.batch * S::kPairs / most_bins <= (F == 8 ? 128 : 256)) {
        const size_t held = device_info().n_cu * std::min<size_t>(2048 / sum_threads, 160 * 1024 / sum_lds) / kRound * kRound;
        if (held > 0 && sum_blocks > held) sum_blocks = held;
    }
    for (size_t first = 0; first < M; first += p.batch) {
        const size_t last = std::min(M, first + p.batch);
        const uint32_t n_stretches = (uint32_t)((last - first + b.stretch - 1) / b.stretch);
        const unsigned bin_blocks = (n_stretches + 7) / 8 * 8 * p.n_levels;
        int rc = TNN_OK;
        if constexpr (F == 2 && !std::is_same<G, float>::value) {
            if (reduce) { // (one part: bins_take_reduction)
                const unsigned taken = (reduce->blocks() + 7) / 8 * 8;
                const auto both = grid_bin_kernel<D, F, G, TrainReduce>;
                if (!reserve_lds(reinterpret_cast<const void *>(both), bin_lds)) return fail(TNN_ERR_HIP, "cannot reserve %zu bytes of LDS", bin_lds);
                TNN_LAUNCH(both, dim3(taken + bin_blocks), dim3(b.threads), bin_lds, s, gp, p, dl, x, order, (const G *)dLdy, runs, records, (long long)first,
                           (long long)last, n_stretches, b.pitch, b.room, *reduce, taken);
                if ((rc = check_launch("grid_bin_kernel with a reduction"))) return rc;
            }
        }
        if ((stage & kBinning) && !reduce) {
            TNN_LAUNCH(bin, dim3(bin_blocks), dim3(b.threads), bin_lds, s, gp, p, dl, x, order, (const G *)dLdy, runs, records, (long long)first, (long long)last,
                       n_stretches, b.pitch, b.room, std::false_type{}, 0u);
            if ((rc = check_launch("grid_bin_kernel"))) return rc;
        }
        if (!(stage & kSums)) continue;
        TNN_LAUNCH(sum, dim3((unsigned)sum_blocks), dim3(sum_threads), sum_lds, s, p, (const uint32_t *)runs, (const BinRecord<F> *)records, grad,
                   n_stretches, b.pitch, (int)(overwrite && first == 0));
        if ((rc = check_launch("grid_bin_sum_kernel"))) return rc;
    }
    return TNN_OK;
}

// The binning is one launch, the threads hold all partials at once, and dL/dy is of the network's type, as the training kernel writes it.
bool bins_take_reduction(const BinPlan &p, uint32_t n_features, int dy_dtype, size_t M, const TrainReduce &r) {
    return n_features == 2 && dy_dtype != TNN_FP32 && M <= p.batch && r.n_partials <= 256;
}

int launch_grid_binned(const BinPlan &p, const GridParams &gp, const GradLayout &dl, uint32_t n_dims, uint32_t n_features, const float *x,
                       const float4 *order, const void *dLdy, int dy_dtype, float *grad, bool overwrite, size_t M, void *scratch, hipStream_t s, BinStage stage,
                       const TrainReduce *reduce) {
#define TNN_BIN_G(D, F)                                                                                                                    \
    switch (dy_dtype) {                                                                                                                    \
    case TNN_FP32: return launch_binned<D, F, float>(p, gp, dl, x, order, dLdy, grad, overwrite, M, scratch, s, stage, reduce); \
    case TNN_BF16: return launch_binned<D, F, bf16_t>(p, gp, dl, x, order, dLdy, grad, overwrite, M, scratch, s, stage, reduce); \
    case TNN_FP16: return launch_binned<D, F, fp16_t>(p, gp, dl, x, order, dLdy, grad, overwrite, M, scratch, s, stage, reduce); \
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

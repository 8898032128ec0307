// Device-side building blocks shared by the fused MLP kernels (gfx950): the per-wave 32-row tile in
// MFMA B-operand order, the weight-fragment product, and the activation / rounding steps.
//
// Register layout: lane (j = lane % 32, h = lane / 32) owns batch row j of the wave's tile; for every
// block kb of 16 features it holds the 8 features 16*kb + 8*h + [0, 8): one aligned 16-byte piece of
// the row-major row. Loads, stores and MFMA B operands all use this layout.
#pragma once

#include "tnn_internal.h"

namespace tnn {

constexpr int kFwdThreads = 256;   // streaming kernels: 4 waves per workgroup share one LDS copy of the weights
constexpr int kTrainThreads = 512; // fused training step: 8 waves per workgroup
constexpr int kWaveSize = 64;

// ------------------------------------------------------------------------------------------
// Device helpers
// ------------------------------------------------------------------------------------------

template <int ACT> __device__ __forceinline__ float act_f32(float v) {
    if (ACT == TNN_ACT_RELU) return fmaxf(v, 0.0f);
    if (ACT == TNN_ACT_SIGMOID) return __builtin_amdgcn_rcpf(1.0f + __expf(-v));
    return v;
}

typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
template <typename T> struct Pair;
template <> struct Pair<bf16_t> { typedef bf16x2 type; };
template <> struct Pair<fp16_t> { typedef fp16x2 type; };

// Two fp32 -> one dword holding two values of T (round to nearest even): one packed convert.
template <typename T> __device__ __forceinline__ unsigned int cvt_pair(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(unsigned int, __builtin_convertvector(v, typename Pair<T>::type));
}

// max(v, 0) on two 2-byte floats with one packed 16-bit integer instruction: a negative bf16/fp16 has
// its sign bit set, i.e. is a negative int16, and every non-negative one is a non-negative int16.
__device__ __forceinline__ unsigned int relu_pair(unsigned int v) {
    const s16x2 b = __builtin_elementwise_max(__builtin_bit_cast(s16x2, v), s16x2{0, 0});
    return __builtin_bit_cast(unsigned int, b);
}

// Hides from the optimiser what a value is (here: that a mask is 0 or 1 per half, which it would turn back into
// per-half compares and selects). The statement emits no instruction: the value stays in the register the compiler
// gave it. Instructions written out in inline asm are not an option in these kernels: their destination registers are
// invisible to the compiler's hazard bookkeeping, and one that lands in the unused part of the destination of an MFMA
// still in flight is overwritten when the MFMA retires.
__device__ __forceinline__ unsigned int opaque(unsigned int v) {
    asm("" : "+v"(v));
    return v;
}

// g where fwd > 0, else 0, with packed 16-bit integer instructions: m = min(max(fwd, 0), 1) is 1 exactly
// for the positive values of fwd (as int16), and g * m keeps or clears the bit pattern of g
// (v_pk_max_i16, v_pk_min_i16, v_pk_mul_lo_u16).
__device__ __forceinline__ unsigned int relu_gate_pair(unsigned int g, unsigned int fwd) {
    s16x2 m = __builtin_elementwise_max(__builtin_bit_cast(s16x2, fwd), s16x2{0, 0});
    m = __builtin_elementwise_min(m, __builtin_bit_cast(s16x2, opaque(0x00010001u)));
    const u16x2 r = __builtin_bit_cast(u16x2, g) * __builtin_bit_cast(u16x2, opaque(__builtin_bit_cast(unsigned int, m)));
    return __builtin_bit_cast(unsigned int, r);
}

// The same gate when fwd is known to be the output of relu_pair (never negative, never -0): min(fwd, 1)
// as unsigned 16-bit integers is already the 0/1 mask (v_pk_min_u16, v_pk_mul_lo_u16).
__device__ __forceinline__ unsigned int relu_gate_pair_nonneg(unsigned int g, unsigned int fwd) {
    const u16x2 m = __builtin_elementwise_min(__builtin_bit_cast(u16x2, fwd), __builtin_bit_cast(u16x2, opaque(0x00010001u)));
    const u16x2 r = __builtin_bit_cast(u16x2, g) * __builtin_bit_cast(u16x2, opaque(__builtin_bit_cast(unsigned int, m)));
    return __builtin_bit_cast(unsigned int, r);
}

// Accumulator half (8 fp32 of one 32x32 tile) -> activation -> 8 values of T.
// ReLU before or after the rounding gives the same value (rounding keeps the sign), so it is applied to
// the rounded values, two per instruction.
template <typename T, int ACT, int HALF>
__device__ __forceinline__ typename Storage<T>::vec8 act_convert(const f32x16 &c) {
    u32x4 r;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        float a = c[HALF * 8 + 2 * p], b = c[HALF * 8 + 2 * p + 1];
        if (ACT == TNN_ACT_SIGMOID) {
            a = act_f32<ACT>(a);
            b = act_f32<ACT>(b);
        }
        unsigned int u = cvt_pair<T>(a, b);
        if (ACT == TNN_ACT_RELU) u = relu_pair(u);
        r[p] = u;
    }
    return __builtin_bit_cast(typename Storage<T>::vec8, r);
}

// Backward: fp32 accumulator, masked / scaled by the stored forward activation, then rounded
// (zeroing before or after the rounding is the same). NONNEG: the activation was produced by this
// library's own ReLU in the same kernel.
template <typename T, int ACT, int HALF, bool NONNEG = false>
__device__ __forceinline__ typename Storage<T>::vec8 bwd_convert(const f32x16 &c,
                                                                 const typename Storage<T>::vec8 &fwd) {
    const u32x4 fw = __builtin_bit_cast(u32x4, fwd);
    u32x4 r;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        float a = c[HALF * 8 + 2 * p], b = c[HALF * 8 + 2 * p + 1];
        if (ACT == TNN_ACT_SIGMOID) {
            const float fa = (float)fwd[2 * p], fb = (float)fwd[2 * p + 1];
            a = as_fp32(a * (fa * (1.0f - fa)));
            b = as_fp32(b * (fb * (1.0f - fb)));
        }
        unsigned int u = cvt_pair<T>(a, b);
        if (ACT == TNN_ACT_RELU) u = NONNEG ? relu_gate_pair_nonneg(u, fw[p]) : relu_gate_pair(u, fw[p]);
        r[p] = u;
    }
    return __builtin_bit_cast(typename Storage<T>::vec8, r);
}

// Every value times `by`, rounded to T.
template <typename T> __device__ __forceinline__ typename Storage<T>::vec8 scaled(const typename Storage<T>::vec8 v, float by) {
    f32x8 f = __builtin_convertvector(v, f32x8);
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = as_fp32(f[e] * by);
    return __builtin_convertvector(f, typename Storage<T>::vec8);
}

// "nt" bit of a buffer store: the line is written through instead of staying dirty in L2 until the kernel ends. Only
// with stores that cover whole 128-byte lines; with partial lines it costs more than it saves.
constexpr int kStreamingStore = 2;

template <typename T, int W> struct Tile {
    static constexpr int NK = W / 16;
    static constexpr int NI = (W + 31) / 32;
    typedef typename Storage<T>::vec8 vec8;

    // Row-major row `row` of an M x W matrix -> the lane's NK 16-byte pieces.
    static __device__ __forceinline__ void load(vec8 (&r)[NK], const T *__restrict__ base, long long row, int h,
                                                bool valid) {
        const vec8 *p = reinterpret_cast<const vec8 *>(base + row * W) + h;
#pragma unroll
        for (int kb = 0; kb < NK; ++kb) {
            if (valid)
                r[kb] = p[2 * kb];
            else
                r[kb] = vec8{};
        }
    }
    static __device__ __forceinline__ void store(const vec8 (&r)[NK], T *__restrict__ base, long long row, int h,
                                                 bool valid) {
        vec8 *p = reinterpret_cast<vec8 *>(base + row * W) + h;
        if (valid) {
#pragma unroll
            for (int kb = 0; kb < NK; ++kb) p[2 * kb] = r[kb];
        }
    }

    // The first `cols` columns of the rows, into a matrix of that many columns.
    static __device__ __forceinline__ void store_columns(const vec8 (&r)[NK], T *__restrict__ base, int cols, long long row, int h, bool valid) {
        if (!valid) return;
        T *p = base + row * cols;
#pragma unroll
        for (int kb = 0; kb < NK; ++kb) {
            const int c = 16 * kb + 8 * h;
            if ((cols & 7) == 0) {
                if (c < cols) *reinterpret_cast<vec8 *>(p + c) = r[kb];
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (c + e < cols) p[c + e] = r[kb][e];
            }
        }
    }
    // A row of `cols` columns of T or fp32 (rounded to T), the others `fill`.
    static __device__ __forceinline__ void load_columns(vec8 (&r)[NK], const void *__restrict__ base, bool fp32, int cols, T fill, long long row, int h,
                                                        bool valid) {
        if (!valid) row = 0;
        const float *pf = static_cast<const float *>(base) + row * cols;
        const T *pt = static_cast<const T *>(base) + row * cols;
#pragma unroll
        for (int kb = 0; kb < NK; ++kb) {
            const int c = 16 * kb + 8 * h;
            if (fp32 && (cols & 7) == 0 && c < cols) {
                const f32x4 a = *reinterpret_cast<const f32x4 *>(pf + c), b = *reinterpret_cast<const f32x4 *>(pf + c + 4);
#pragma unroll
                for (int e = 0; e < 8; ++e) r[kb][e] = (T)(e < 4 ? a[e & 3] : b[e & 3]);
            } else if (!fp32 && (cols & 7) == 0 && c < cols) {
                r[kb] = *reinterpret_cast<const vec8 *>(pt + c);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    r[kb][e] = fill;
                    if (c + e < cols) r[kb][e] = fp32 ? (T)pf[c + e] : pt[c + e];
                }
            }
        }
    }

    // The same rows through a buffer resource whose range is the matrix (`rows_of`): a lane outside the matrix passes
    // `kNoRow`, its loads return zeros and its stores are dropped by the range check, so the instructions issue
    // unconditionally and the waits on them can count exactly (a load under a branch forces a wait for everything).
    static constexpr unsigned int kNoRow = 0xFFFFFF00u;
    static constexpr unsigned long long kMaxBufferBytes = 1ull << 31;
    static __device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_of(const T *base, long long M) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(base), 0, (int)(unsigned int)(M * W * (long long)sizeof(T)), 0x00020000);
    }
    static __device__ __forceinline__ unsigned int row_offset(long long row, int h, bool valid) {
        return valid ? (unsigned int)(row * (W * (long long)sizeof(T))) + 16u * h : kNoRow;
    }
    template <int AUX = 0>
    static __device__ __forceinline__ void load(vec8 (&r)[NK], __amdgpu_buffer_rsrc_t rows, unsigned int off) {
#pragma unroll
        for (int kb = 0; kb < NK; ++kb) r[kb] = __builtin_bit_cast(vec8, __builtin_amdgcn_raw_buffer_load_b128(rows, off + 32 * kb, 0, AUX));
    }
    template <int AUX = 0>
    static __device__ __forceinline__ void store(const vec8 (&r)[NK], __amdgpu_buffer_rsrc_t rows, unsigned int off) {
#pragma unroll
        for (int kb = 0; kb < NK; ++kb) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, r[kb]), rows, off + 32 * kb, 0, AUX);
    }

    // Stores of a tile as whole rows: the lane's pieces go to a row-major copy of the tile in LDS (32 rows of PITCH
    // bytes, owned by the wave) and come back with W/8 neighbouring lanes holding one row, so that a store instruction
    // writes complete 128-byte lines instead of 32 bytes of each of 32 lines (measured: 10 % on the backward pass).
    static constexpr int PITCH = W * 2 + 16;  // bytes per staged row (16-byte skew against bank conflicts)
    static constexpr int TILE_BYTES = 32 * PITCH;
    static constexpr int LPR = W / 8;          // lanes per row of 16-byte pieces
    static constexpr int RPI = kWaveSize / LPR; // rows per store instruction; NK instructions per tile
    static __device__ __forceinline__ void row_offsets(unsigned int (&o)[NK], long long tile, int lane, long long M) {
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const long long r = tile * 32 + i * RPI + lane / LPR;
            o[i] = (r < M) ? (unsigned int)(r * (W * (long long)sizeof(T))) + (lane % LPR) * 16 : kNoRow;
        }
    }
    static __device__ __forceinline__ void stage(const vec8 (&r)[NK], unsigned char *tile_lds, int j, int h) {
#pragma unroll
        for (int kb = 0; kb < NK; ++kb) *reinterpret_cast<vec8 *>(tile_lds + j * PITCH + h * 16 + 32 * kb) = r[kb];
    }
    // AUX: cache policy bits of the store; kStreamingStore marks data that this GPU does not read again soon.
    template <int AUX = 0>
    static __device__ __forceinline__ void store_staged(const unsigned char *tile_lds, int lane, __amdgpu_buffer_rsrc_t rows,
                                                        const unsigned int (&o)[NK]) {
#pragma unroll
        for (int i = 0; i < NK; ++i)
            __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4 *>(tile_lds + (i * RPI + lane / LPR) * PITCH + (lane % LPR) * 16),
                                                   rows, o[i], 0, AUX);
    }

    // The same store from one offset per tile (that of the lane's 16 bytes in the first of its rows) and a constant per
    // instruction. Rows past the end of the matrix need no flag: their offsets lie past the end of the buffer resource and the
    // range check drops them (the resource covers less than 2^31 bytes, so an offset cannot wrap back into range).
    // The constant is part of the lane's offset, not the scalar one: behind a store whose offset is a scalar register the compiler leaves no
    // wait states before the data may be overwritten, and gfx950 needs them there, too (a v_mov into the fourth register right behind the last
    // store: now and then 16 of the 64 lanes stored what the v_mov had written).
    static __device__ __forceinline__ unsigned int staged_base(long long tile, int lane) {
        return (unsigned int)((tile * 32 + lane / LPR) * (W * (long long)sizeof(T))) + (lane % LPR) * 16;
    }
    template <int AUX = 0>
    static __device__ __forceinline__ void store_staged_at(const unsigned char *tile_lds, int lane, __amdgpu_buffer_rsrc_t rows, unsigned int base) {
#pragma unroll
        for (int i = 0; i < NK; ++i)
            __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4 *>(tile_lds + (i * RPI + lane / LPR) * PITCH + (lane % LPR) * 16),
                                                   rows, base + i * RPI * W * (int)sizeof(T), 0, AUX);
    }

    static constexpr int NF = NI * NK; // weight fragments per matrix and lane

    // The lane's NF operand fragments of matrix l (LDS or global, already in operand order).
    static __device__ __forceinline__ void load_frags(vec8 (&f)[NF], const vec8 *__restrict__ w, int l, int lane) {
        const vec8 *p = w + (size_t)l * (NF * kWaveSize) + lane;
#pragma unroll
        for (int i = 0; i < NF; ++i) f[i] = p[i * kWaveSize];
    }

    // acc[a] = sum_kb frag(a, kb) * b[kb]
    static __device__ __forceinline__ void mma(f32x16 (&acc)[NI], const vec8 (&b)[NK], const vec8 (&f)[NF]) {
#pragma unroll
        for (int a = 0; a < NI; ++a) acc[a] = f32x16{};
#pragma unroll
        for (int kb = 0; kb < NK; ++kb) {
#pragma unroll
            for (int a = 0; a < NI; ++a) acc[a] = Storage<T>::mfma(f[a * NK + kb], b[kb], acc[a]);
        }
    }

    // acc[a] = sum_kb frag(l, a, kb) * b[kb]
    template <bool W_IN_LDS>
    static __device__ __forceinline__ void matmul(f32x16 (&acc)[NI], const vec8 (&b)[NK], const vec8 *__restrict__ lds_w,
                                                  const vec8 *__restrict__ glb_w, int l, int lane) {
        const vec8 *w = (W_IN_LDS ? lds_w : glb_w) + (size_t)l * (NI * NK * kWaveSize) + lane;
#pragma unroll
        for (int a = 0; a < NI; ++a) acc[a] = f32x16{};
#pragma unroll
        for (int kb = 0; kb < NK; ++kb) {
#pragma unroll
            for (int a = 0; a < NI; ++a) {
                const vec8 frag = w[(a * NK + kb) * kWaveSize];
                acc[a] = Storage<T>::mfma(frag, b[kb], acc[a]);
            }
        }
    }

    template <int ACT> static __device__ __forceinline__ void repack(vec8 (&r)[NK], const f32x16 (&acc)[NI]) {
#pragma unroll
        for (int a = 0; a < NI; ++a) {
            r[2 * a] = act_convert<T, ACT, 0>(acc[a]);
            if (2 * a + 1 < NK) r[2 * a + 1] = act_convert<T, ACT, 1>(acc[a]);
        }
    }
    static __device__ __forceinline__ void repack_rt(vec8 (&r)[NK], const f32x16 (&acc)[NI], int act) {
        if (act == TNN_ACT_RELU)
            repack<TNN_ACT_RELU>(r, acc);
        else if (act == TNN_ACT_SIGMOID)
            repack<TNN_ACT_SIGMOID>(r, acc);
        else
            repack<TNN_ACT_NONE>(r, acc);
    }

    template <int ACT, bool NONNEG = false>
    static __device__ __forceinline__ void bwd_repack(vec8 (&r)[NK], const f32x16 (&acc)[NI], const vec8 (&fwd)[NK]) {
#pragma unroll
        for (int a = 0; a < NI; ++a) {
            r[2 * a] = bwd_convert<T, ACT, 0, NONNEG>(acc[a], fwd[2 * a]);
            if (2 * a + 1 < NK) r[2 * a + 1] = bwd_convert<T, ACT, 1, NONNEG>(acc[a], fwd[2 * a + 1 < NK ? 2 * a + 1 : 0]);
        }
    }
};

// A forward pass that takes the parameters where the optimiser left them (fp32, packed layout) instead of prepared operands,
// and leaves everything tnn_mlp_set_packed_weights derives from them behind: the launch of its own that the push was took 2.5 to
// 5 us in front of every forward pass. Every workgroup that computes stages its weights from the parameters (twice the bytes
// of the prepared operands, out of L2); the copies are written by workgroups [first, ...), which are those that compute when
// there are enough of them, and additional ones behind them otherwise (a small batch occupies few CUs).
struct WeightPush {
    const float *master = nullptr; // null: no push, the kernel reads prepared operands
    void *packed = nullptr, *packed_t = nullptr, *fwd = nullptr, *bwd = nullptr;
    int live_in = 0, live_out = 0; // rows of the first matrix / columns of the last one from here on only see padding
    int blocks = 0;                // workgroups that compute
    int first = 0;                 // first workgroup that writes copies
};

// A weight of matrix l as set_packed_weights takes it.
template <typename T> __device__ __forceinline__ T pushed_weight(const WeightPush &p, float v, int l, int k, int n, int n_mats) {
    return ((l == 0 && k >= p.live_in) || (l == n_mats - 1 && n >= p.live_out)) ? (T)0.0f : (T)v;
}

// One forward operand fragment (8 values of T): f counts fragments over all matrices and lanes.
template <typename T, int W> struct PushedFragment {
    f32x2 raw[4];
    __device__ __forceinline__ void request(const WeightPush &p, int f) {
        constexpr int NK = W / 16, per_mat = ((W + 31) / 32) * NK * kWaveSize;
        const int l = f / per_mat, r = f % per_mat, lane = r & 63;
        const int outer = 32 * ((r >> 6) / NK) + swap23(lane & 31), k0 = 16 * ((r >> 6) % NK) + 8 * (lane >> 5);
        const float *src = p.master + (size_t)l * W * W + 2 * (outer < W ? outer : 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) raw[q] = *reinterpret_cast<const f32x2 *>(src + (k0 + 2 * q) * W); // rows k0 + 2 q and the next, side by side
    }
    __device__ __forceinline__ typename Storage<T>::vec8 convert(const WeightPush &p, int f, int n_mats) const {
        constexpr int NK = W / 16, per_mat = ((W + 31) / 32) * NK * kWaveSize;
        const int l = f / per_mat, r = f % per_mat, lane = r & 63;
        const int outer = 32 * ((r >> 6) / NK) + swap23(lane & 31), k0 = 16 * ((r >> 6) % NK) + 8 * (lane >> 5);
        typename Storage<T>::vec8 v = {};
#pragma unroll
        for (int t = 0; t < 8; ++t)
            if (outer < W) v[t] = pushed_weight<T>(p, raw[t >> 1][t & 1], l, k0 + t, outer, n_mats);
        return v;
    }
};

// One slot of the operand-order index space of all matrices (it covers every matrix element once, plus the empty half-tile
// at width 16): the element's place in the packed copy, its transpose and both operand orders.
template <typename T, typename SRC, typename WEIGHT>
__device__ __forceinline__ void write_weight_copies(int idx, const SRC *__restrict__ src, T *__restrict__ packed, T *__restrict__ packed_t, T *__restrict__ fwd,
                                                    T *__restrict__ bwd, int W, WEIGHT weight) {
    const int NI = (W + 31) / 32, NK = W / 16;
    const int per_mat = NI * NK * 512;
    const int l = idx / per_mat;
    int r = idx % per_mat;
    const int t = r & 7;
    const int lane = (r >> 3) & 63;
    r >>= 9;
    const int kb = r % NK, a = r / NK;
    const int h = lane >> 5, i = lane & 31;
    const int outer = 32 * a + swap23(i), inner = 16 * kb + 8 * h + t;
    T vf = (T)0.0f, vb = (T)0.0f;
    if (outer < W) {
        const size_t m = (size_t)l * W * W;
        vf = weight((float)src[m + packed_coord(inner, outer, W)], l, inner, outer);
        vb = weight((float)src[m + packed_coord(outer, inner, W)], l, outer, inner);
        packed[m + packed_coord(inner, outer, W)] = vf;
        packed_t[m + packed_coord(outer, inner, W)] = vf; // element (k, n) of W is element (n, k) of its transpose
    }
    fwd[idx] = vf;
    bwd[idx] = vb;
}

template <typename T, int W> __device__ __forceinline__ void push_copies(const WeightPush &p, int n_mats) {
    if ((int)blockIdx.x < p.first) return;
    const int total = n_mats * ((W + 31) / 32) * (W / 16) * 512, step = ((int)gridDim.x - p.first) * (int)blockDim.x;
    for (int idx = ((int)blockIdx.x - p.first) * (int)blockDim.x + (int)threadIdx.x; idx < total; idx += step)
        write_weight_copies<T>(idx, p.master, static_cast<T *>(p.packed), static_cast<T *>(p.packed_t), static_cast<T *>(p.fwd), static_cast<T *>(p.bwd), W,
                               [&](float v, int l, int k, int n) { return pushed_weight<T>(p, v, l, k, n, n_mats); });
}

// Weights of the forward pass into LDS, from prepared operands or from the parameters.
template <typename T, int W>
__device__ __forceinline__ void stage_weights(typename Storage<T>::vec8 *lds_w, const typename Storage<T>::vec8 *__restrict__ glb_w, int n_mats,
                                              const WeightPush &p) {
    constexpr int per_mat = Tile<T, W>::NI * Tile<T, W>::NK * kWaveSize;
    const int n = n_mats * per_mat;
    if (!p.master) {
        for (int f = threadIdx.x; f < n; f += blockDim.x) lds_w[f] = glb_w[f];
    } else {
        for (int f = threadIdx.x; f < n; f += 2 * blockDim.x) {
            const int g = f + (int)blockDim.x < n ? f + (int)blockDim.x : f;
            PushedFragment<T, W> a, b;
            a.request(p, f);
            b.request(p, g);
            lds_w[f] = a.convert(p, f, n_mats);
            lds_w[g] = b.convert(p, g, n_mats);
        }
    }
    __syncthreads();
}

template <typename T, int W>
__device__ __forceinline__ void stage_weights(typename Storage<T>::vec8 *lds_w,
                                              const typename Storage<T>::vec8 *__restrict__ glb_w, int n_mats) {
    constexpr int per_mat = Tile<T, W>::NI * Tile<T, W>::NK * kWaveSize;
    const int n = n_mats * per_mat;
    for (int f = threadIdx.x; f < n; f += blockDim.x) lds_w[f] = glb_w[f];
    __syncthreads();
}


struct DeviceInfo {
    int n_cu = 0;
    size_t max_lds = 0;
    bool ok = false;
};
const DeviceInfo &device_info();

// The grid of a forward pass with a push and the rest of its plan; `blocks` workgroups compute.
inline int push_grid(WeightPush *p, int blocks, int threads, size_t prepared_elements) {
    p->blocks = blocks;
    if (!p->master) return blocks;
    p->first = blocks >= 64 ? 0 : blocks;
    return blocks >= 64 ? blocks : blocks + (int)((prepared_elements + threads - 1) / threads);
}

inline size_t prepared_elems(const tnn_mlp_desc *d) {
    const int W = d->width, NI = (W + 31) / 32, NK = W / 16;
    return (size_t)(d->n_hidden_layers + 1) * NI * NK * 512;
}

} // namespace tnn

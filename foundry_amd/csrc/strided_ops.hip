// Strided entry points for the reference's non-quantized Ops
// (src/nn/primitive.rs:48-68), the rest of what Device::run and
// Device::run_in_place need (src/metal/mod.rs:639-725): copy, dtype
// conversion, unary and binary elementwise ops, row reductions, matmul,
// index_select, cat and slice_scatter, each over strided views.
//
// Elementwise ops and moves take 16-byte pieces where the views allow it and
// single elements otherwise; reductions run a block or a wavefront per output
// element; the matmul runs on the fp32 matrix cores. All with the Metal
// kernels' arithmetic: values decoded to fp32, the op in fp32, one rounding on
// the way out (src/metal/kernels/common.metal:29-43). They serve the model code
// that runs op by op; the decoder's hot path has its own fused kernels.
#include <type_traits>

#include "device.hpp"
#include "q4_common.hpp"

namespace fh {
namespace {

constexpr int kRank = 4;
constexpr uint32_t kThreads = 256;
// src/nn/shape.rs:13: a shape holds at most 2^31 - 1 elements, so a linear
// element index fits 32 bits.
constexpr int64_t kMaxNumel = 0x7FFFFFFF;

// fh_view as the kernels take it (by value), dims past ndim padded with 1.
struct View {
    int64_t offset;
    int64_t strides[kRank];
    uint32_t dims[kRank];
    int32_t ndim;
};

// Element index of the view's linear (row-major) element `i`, the
// decomposition StridedArgs describes (src/metal/kernels/common.metal:13-21).
__device__ __forceinline__ int64_t at(uint32_t i, const View &v) {
    int64_t idx = v.offset;
#pragma unroll
    for (int d = kRank - 1; d >= 0; --d) {
        if (d >= v.ndim) continue;
        const uint32_t size = v.dims[d];
        idx += static_cast<int64_t>(i % size) * v.strides[d];
        i /= size;
    }
    return idx;
}

__device__ __forceinline__ uint32_t gid() { return blockIdx.x * kThreads + threadIdx.x; }

// Float element access by fh_dtype: F32 as is, BF16 decoded exactly and
// written with the reference's RNE.
template <int DT>
struct Float;
template <>
struct Float<FH_F32> {
    using T = float;
    __device__ static float get(const T *p, int64_t i) { return p[i]; }
    __device__ static void put(T *p, int64_t i, float v) { p[i] = v; }
};
template <>
struct Float<FH_BF16> {
    using T = uint16_t;
    __device__ static float get(const T *p, int64_t i) { return bf16_to_f32(p[i]); }
    __device__ static void put(T *p, int64_t i, float v) { p[i] = static_cast<uint16_t>(f32_to_bf16_rne(v)); }
};

// N views of the same dims for an elementwise kernel, after the host has
// dropped dims of size one and merged neighbours that every view steps
// through evenly (walk_of). With `pieces` the last dim counts pieces of
// consecutive elements instead of elements: the views are then read 16 bytes
// (or one broadcast element) at a time. mul and shift divide by dims[d]
// (i / d = (mulhi(mul, i) + i) >> shift for i < 2^31), since a hardware
// division per dim and element was most of these kernels' time.
template <int N>
struct Walk {
    uint32_t ndim;
    uint32_t dims[kRank], mul[kRank], shift[kRank];
    int64_t offset[N], strides[N][kRank];
    bool pieces;
    uint32_t single;  // elements a thread takes without pieces, a block's width apart
};

// Element index, in every view, of element (or piece) i.
template <int N>
__device__ __forceinline__ void walk(uint32_t i, const Walk<N> &w, int64_t (&at)[N]) {
#pragma unroll
    for (int v = 0; v < N; ++v) at[v] = w.offset[v];
#pragma unroll
    for (int d = kRank - 1; d >= 0; --d) {
        if (d >= static_cast<int>(w.ndim)) continue;
        const uint32_t q = (__umulhi(w.mul[d], i) + i) >> w.shift[d];
        const uint32_t r = i - q * w.dims[d];
#pragma unroll
        for (int v = 0; v < N; ++v) at[v] += static_cast<int64_t>(r) * w.strides[v][d];
        i = q;
    }
}

// 8 consecutive values from 16-byte aligned memory.
template <int DT>
__device__ __forceinline__ void load8(const typename Float<DT>::T *p, float (&v)[8]) {
    if constexpr (DT == FH_BF16) {
        const uint4 u = *reinterpret_cast<const uint4 *>(p);
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[2 * e] = __uint_as_float(w[e] << 16);
            v[2 * e + 1] = __uint_as_float(w[e] & 0xFFFF0000u);
        }
    } else {
        const float4 lo = *reinterpret_cast<const float4 *>(p), hi = *reinterpret_cast<const float4 *>(p + 4);
        v[0] = lo.x, v[1] = lo.y, v[2] = lo.z, v[3] = lo.w;
        v[4] = hi.x, v[5] = hi.y, v[6] = hi.z, v[7] = hi.w;
    }
}

template <int DT>
__device__ __forceinline__ void store8(typename Float<DT>::T *p, const float (&v)[8]) {
    if constexpr (DT == FH_BF16) {
        *reinterpret_cast<uint4 *>(p) =
            make_uint4(f32x2_to_bf16x2_rne(v[0], v[1]), f32x2_to_bf16x2_rne(v[2], v[3]),
                       f32x2_to_bf16x2_rne(v[4], v[5]), f32x2_to_bf16x2_rne(v[6], v[7]));
    } else {
        *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4 *>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
    }
}

// src's elements, bit for bit, to dst's (copy, cat, slice_scatter); a piece
// is 16 bytes.
template <typename T>
__global__ __launch_bounds__(kThreads) void move_kernel(const T *__restrict__ src, T *__restrict__ dst, Walk<2> w,
                                                        uint32_t n) {
    int64_t at[2];
    if (w.pieces) {
        const uint32_t i = gid();
        if (i >= n) return;
        walk(i, w, at);
        *reinterpret_cast<uint4 *>(dst + at[1]) = *reinterpret_cast<const uint4 *>(src + at[0]);
        return;
    }
    for (uint32_t u = 0; u < w.single; ++u) {
        const uint32_t i = (blockIdx.x * w.single + u) * kThreads + threadIdx.x;
        if (i >= n) return;
        walk(i, w, at);
        dst[at[1]] = src[at[0]];
    }
}

struct Identity {
    __device__ float operator()(float x) const { return x; }
};

struct UnaryOf {
    int op;
    __device__ float operator()(float x) const {
        switch (op) {
            case FH_NEG: return -x;
            case FH_EXP: return expf(x);
            case FH_SQRT: return sqrtf(x);
            default: return 1.0f / x;
        }
    }
};

struct BinaryOf {
    int op;
    __device__ float operator()(float a, float b) const {
        switch (op) {
            case FH_ADD: return a + b;
            case FH_SUB: return a - b;
            case FH_MUL: return a * b;
            default: return a / b;
        }
    }
};

// dst[i] = f(a[i]) or f(a[i], b[i]) over one or two views of dtype IN, dst
// contiguous of dtype OUT. A piece is 8 elements: each view gives 8
// consecutive values or one for all 8 (its last stride 0).
// Bounded by memory. [24, 512, 512] f32, before (an element a thread, a
// division per dim) and now: add 33.5 -> 10.9 us, exp 20 -> 10.9 us, to
// bf16 18 -> 6.8 us.
template <int IN, int OUT, int N, class F>
__global__ __launch_bounds__(kThreads) void map_kernel(const typename Float<IN>::T *__restrict__ a,
                                                       const typename Float<IN>::T *__restrict__ b,
                                                       typename Float<OUT>::T *__restrict__ dst, Walk<N> w, uint32_t n,
                                                       F f) {
    const typename Float<IN>::T *const src[2] = {a, b};
    int64_t at[N];
    if (w.pieces) {
        const uint32_t i = gid();
        if (i >= n) return;
        walk(i, w, at);
        float v[N][8];
#pragma unroll
        for (int s = 0; s < N; ++s) {
            if (w.strides[s][w.ndim - 1] != 0) {
                load8<IN>(src[s] + at[s], v[s]);
            } else {
                const float x = Float<IN>::get(src[s], at[s]);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[s][e] = x;
            }
        }
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if constexpr (N == 1)
                o[e] = f(v[0][e]);
            else
                o[e] = f(v[0][e], v[1][e]);
        }
        store8<OUT>(dst + static_cast<uint64_t>(i) * 8, o);
        return;
    }
    for (uint32_t u = 0; u < w.single; ++u) {
        const uint32_t i = (blockIdx.x * w.single + u) * kThreads + threadIdx.x;
        if (i >= n) return;
        walk(i, w, at);
        if constexpr (N == 1)
            Float<OUT>::put(dst, i, f(Float<IN>::get(a, at[0])));
        else
            Float<OUT>::put(dst, i, f(Float<IN>::get(a, at[0]), Float<IN>::get(b, at[1])));
    }
}

// One block per output element. Thread t folds elements t, t + 256, ... of
// the reduced dim in order, then the 256 partials meet in a halving tree
// (width 128, 64, ..., 1), the order reduce_rows uses
// (src/metal/kernels/reduce.metal:17-40), so sums round as the reference's do.
template <int DT, bool AMAX>
__global__ __launch_bounds__(kThreads) void reduce_kernel(const typename Float<DT>::T *__restrict__ src, View rows,
                                                          uint32_t dim_size, int64_t dim_stride,
                                                          typename Float<DT>::T *__restrict__ dst,
                                                          uint32_t n_rows) {
    __shared__ float part[kThreads];
    const uint32_t t = threadIdx.x;
    // blocks stride over the output rows: the grid is capped so that its
    // work-item count stays below 2^32 however many rows there are
    for (uint32_t row = blockIdx.x; row < n_rows; row += gridDim.x) {
        const int64_t base = at(row, rows);
        float acc = AMAX ? -INFINITY : 0.0f;
        for (uint32_t k = t; k < dim_size; k += kThreads) {
            const float x = Float<DT>::get(src, base + static_cast<int64_t>(k) * dim_stride);
            acc = AMAX ? fmaxf(acc, x) : acc + x;
        }
        __syncthreads();  // the previous row's tree has read part[]
        part[t] = acc;
        __syncthreads();
        for (uint32_t w = kThreads / 2; w > 0; w /= 2) {
            if (t < w) part[t] = AMAX ? fmaxf(part[t], part[t + w]) : part[t] + part[t + w];
            __syncthreads();
        }
        if (t == 0) Float<DT>::put(dst, row, part[0]);
    }
}

// The same sums a wavefront per output element: lane l holds the partials of
// threads l, l + 64, l + 128 and l + 192 and the tree's first two levels are
// its own, the rest lane exchanges, so no barrier. For many rows (a block per
// row spends its time in the tree's eight barriers): 12288 rows of 512 f32
// 16.4 -> 7.6 us.
template <int DT, bool AMAX>
__global__ __launch_bounds__(kThreads) void reduce_wave_kernel(const typename Float<DT>::T *__restrict__ src,
                                                               View rows, uint32_t dim_size, int64_t dim_stride,
                                                               typename Float<DT>::T *__restrict__ dst,
                                                               uint32_t n_rows) {
    const uint32_t lane = threadIdx.x & 63;
    auto op = [](float a, float b) { return AMAX ? fmaxf(a, b) : a + b; };
    // whole wavefronts leave together; blocks stride over the rows as in
    // reduce_kernel
    for (uint64_t row = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6); row < n_rows;
         row += gridDim.x * (kThreads / 64)) {
        const int64_t base = at(static_cast<uint32_t>(row), rows);
        auto get = [&](uint32_t k) { return Float<DT>::get(src, base + static_cast<int64_t>(k) * dim_stride); };
        float acc[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = AMAX ? -INFINITY : 0.0f;
        uint32_t k = lane;
        for (; k + 192 < dim_size; k += kThreads) {
            float x[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) x[q] = get(k + q * 64);
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[q] = op(acc[q], x[q]);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (k + q * 64 < dim_size) acc[q] = op(acc[q], get(k + q * 64));
        float v = op(op(acc[0], acc[2]), op(acc[1], acc[3]));
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) v = op(v, __shfl_down(v, d, 64));
        if (lane == 0) Float<DT>::put(dst, static_cast<int64_t>(row), v);
    }
}

// argmax_rows (src/metal/kernels/reduce.metal:42-78): a thread keeps its
// first strict maximum; the tree prefers the larger value, then the lower
// index. A NaN never wins; a row with no larger value than -inf gives 0.
template <int DT>
__global__ __launch_bounds__(kThreads) void argmax_kernel(const typename Float<DT>::T *__restrict__ src, View rows,
                                                          uint32_t dim_size, int64_t dim_stride,
                                                          uint32_t *__restrict__ dst, uint32_t n_rows) {
    __shared__ float val[kThreads];
    __shared__ uint32_t idx[kThreads];
    const uint32_t t = threadIdx.x;
    for (uint32_t row = blockIdx.x; row < n_rows; row += gridDim.x) {  // as reduce_kernel
        const int64_t base = at(row, rows);
        float best = -INFINITY;
        uint32_t best_i = 0;
        for (uint32_t k = t; k < dim_size; k += kThreads) {
            const float x = Float<DT>::get(src, base + static_cast<int64_t>(k) * dim_stride);
            if (x > best) best = x, best_i = k;
        }
        __syncthreads();  // the previous row's tree has read val[], idx[]
        val[t] = best;
        idx[t] = best_i;
        __syncthreads();
        for (uint32_t w = kThreads / 2; w > 0; w /= 2) {
            if (t < w) {
                const float o = val[t + w];
                const uint32_t oi = idx[t + w];
                if (o > val[t] || (o == val[t] && oi < idx[t])) val[t] = o, idx[t] = oi;
            }
            __syncthreads();
        }
        if (t == 0) dst[row] = idx[0];
    }
}

// Batched matmul over strided operands on the matrix cores, in fp32:
// v_mfma_f32_16x16x4_f32 adds its four products to the accumulator one fma at
// a time in order of k, so every sum is the chain of fmas over k that
// matmul_tiled forms (src/metal/kernels/matmul.metal:42-64), also for huge,
// tiny, denormal, infinite and NaN values.
// A block of four wavefronts (WM x WN) owns WM * 16 T rows x WN * 16 T columns
// of one batch entry; operand tiles of 32 along k go through LDS as fp32, the
// next tile's global loads in flight while one is computed. In LDS a row's (or
// column's) 32 values lie by k % 4, then k / 4, 8 together: a lane's operands
// of 8 MFMAs are two conflict-free 16-byte reads. Values past k are filled
// with +0 (lhs) and -0 (rhs), whose product leaves every sum as it is.
// Before, a thread kept 2 x 2 sums fed by scalar LDS reads. bf16, before and
// now: 24 x [512, 128] x [128, 512] (keys transposed in place) 69.2 -> 26.5 us
// (61 TFLOP/s, 0.39 of the fp32 matrix-core rate), 24 x [512, 512] x [512, 128]
// 73.9 -> 34.2 us, [16, 3072] x [3072, 8192] 224.6 -> 74.4 us. Neither that rate
// nor memory bounds it but the chain of steps: two barriers around one LDS
// buffer per 32 of k (the last shape: 96 steps of 0.78 us in a block per CU).
struct MatmulShape {
    uint32_t m, n, k, batch_ndim;
    uint32_t batch_dims[2];
    int64_t l_off, l_rs, l_cs, l_bs[2];
    int64_t r_off, r_rs, r_cs, r_bs[2];
    int l_mode, r_mode;  // Stage
};

constexpr uint32_t kMmK = 32;
constexpr uint32_t kMmPitch = kMmK + 4;

// How an operand's tile is read: single values with threads along k or along
// the rows, or 8 values at once where the dim is contiguous, its extent a
// multiple of 8 and every piece 16-byte aligned.
enum Stage { kAlongK, kAlongRows, kPiecesK, kPiecesRows };

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

// One operand's R x 32 tile on its way from memory to LDS: R * 4 pieces of 8
// values over the block's threads. PIECES: the mode is one of the two that
// read 8 values at once (the gathers' addresses cost the kernel 60 registers).
template <int DT, int R, bool PIECES>
struct MmTile {
    using T = typename Float<DT>::T;
    static constexpr int kItems = (R * 4 + static_cast<int>(kThreads) - 1) / static_cast<int>(kThreads);
    static constexpr int kSingles = R * static_cast<int>(kMmK) / static_cast<int>(kThreads);
    static_assert(kSingles <= kItems * 8, "single values fit the pieces' registers");
    float v[kItems * 8];

    // Row and first k of a piece, or row and k of a single value.
    __device__ static void piece(int mode, uint32_t item, uint32_t *r, uint32_t *kk) {
        if (mode == kPiecesK)
            *r = item / 4, *kk = item % 4 * 8;
        else
            *kk = item / (R / 8), *r = item % (R / 8) * 8;
    }
    __device__ static void single(int mode, uint32_t i, uint32_t *r, uint32_t *kk) {
        if (mode == kAlongK)
            *r = i / kMmK, *kk = i % kMmK;
        else
            *kk = i / R, *r = i % R;
    }
    __device__ void load(const T *p, int64_t base, int64_t rs, int64_t ks, uint32_t row0, uint32_t rows, uint32_t k0,
                         uint32_t k, int mode, float fill) {
        uint32_t r, kk;
        if (PIECES || mode >= kPiecesK) {
#pragma unroll
            for (int i = 0; i < kItems; ++i) {
                const uint32_t item = threadIdx.x + i * kThreads;
                if (R * 4 % kThreads != 0 && item >= R * 4) break;
                piece(mode, item, &r, &kk);
                // the extents are multiples of 8: a piece is inside or outside
                float(&o)[8] = *reinterpret_cast<float(*)[8]>(v + i * 8);
                if (row0 + r < rows && k0 + kk < k)
                    load8<DT>(p + base + static_cast<int64_t>(row0 + r) * rs + static_cast<int64_t>(k0 + kk) * ks, o);
                else
#pragma unroll
                    for (int e = 0; e < 8; ++e) o[e] = fill;
            }
            return;
        }
        // requested without a branch each (a value outside reads the first)
#pragma unroll
        for (int e = 0; e < kSingles; ++e) {
            single(mode, threadIdx.x + e * kThreads, &r, &kk);
            const bool in = row0 + r < rows && k0 + kk < k;
            const int64_t at = base + static_cast<int64_t>(row0 + r) * rs + static_cast<int64_t>(k0 + kk) * ks;
            const float x = Float<DT>::get(p, in ? at : base);
            v[e] = in ? x : fill;
        }
    }
    __device__ void store(float *lds, int mode) const {
        uint32_t r, kk;
        if (!PIECES && mode < kPiecesK) {
#pragma unroll
            for (int e = 0; e < kSingles; ++e) {
                single(mode, threadIdx.x + e * kThreads, &r, &kk);
                lds[r * kMmPitch + kk % 4 * 8 + kk / 4] = v[e];
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            const uint32_t item = threadIdx.x + i * kThreads;
            if (R * 4 % kThreads != 0 && item >= R * 4) break;
            piece(mode, item, &r, &kk);
            const float *const o = v + i * 8;
            if (mode == kPiecesK) {
                float *d = lds + r * kMmPitch + kk / 4;  // k % 4 = 0..3, k / 4 and k / 4 + 1
#pragma unroll
                for (int q = 0; q < 4; ++q) *reinterpret_cast<float2 *>(d + q * 8) = make_float2(o[q], o[q + 4]);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) lds[(r + e) * kMmPitch + kk % 4 * 8 + kk / 4] = o[e];
            }
        }
    }
};

template <int DT, int WM, int WN, int T, bool PIECES>
__global__ __launch_bounds__(kThreads) void matmul_kernel(const typename Float<DT>::T *__restrict__ lhs,
                                                          const typename Float<DT>::T *__restrict__ rhs, MatmulShape s,
                                                          typename Float<DT>::T *__restrict__ dst) {
    constexpr int kBM = WM * 16 * T, kBN = WN * 16 * T;
    static_assert(WM * WN * 64 == static_cast<int>(kThreads), "four wavefronts");
    __shared__ __attribute__((aligned(16))) float lt[kBM * kMmPitch];
    __shared__ __attribute__((aligned(16))) float rt[kBN * kMmPitch];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t row0 = blockIdx.y * kBM, col0 = blockIdx.x * kBN;
    // batch entry -> each operand's base offset (batch dims row-major)
    int64_t lb = s.l_off, rb = s.r_off;
    uint32_t b = blockIdx.z;
    for (int d = static_cast<int>(s.batch_ndim) - 1; d >= 0; --d) {
        const uint32_t size = s.batch_dims[d];
        lb += static_cast<int64_t>(b % size) * s.l_bs[d];
        rb += static_cast<int64_t>(b % size) * s.r_bs[d];
        b /= size;
    }
    f32x4_t acc[T][T];
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;
    MmTile<DT, kBM, PIECES> lv;
    MmTile<DT, kBN, PIECES> rv;
    const float *const la = lt + ((wave / WN) * 16 * T + (lane & 15)) * kMmPitch + (lane >> 4) * 8;
    const float *const ra = rt + ((wave % WN) * 16 * T + (lane & 15)) * kMmPitch + (lane >> 4) * 8;
    if (s.k > 0) {
        lv.load(lhs, lb, s.l_rs, s.l_cs, row0, s.m, 0, s.k, s.l_mode, 0.f);
        rv.load(rhs, rb, s.r_cs, s.r_rs, col0, s.n, 0, s.k, s.r_mode, -0.f);
    }
    for (uint32_t k0 = 0; k0 < s.k; k0 += kMmK) {
        __syncthreads();  // the previous tile's reads are done
        lv.store(lt, s.l_mode);
        rv.store(rt, s.r_mode);
        __syncthreads();
        if (k0 + kMmK < s.k) {
            lv.load(lhs, lb, s.l_rs, s.l_cs, row0, s.m, k0 + kMmK, s.k, s.l_mode, 0.f);
            rv.load(rhs, rb, s.r_cs, s.r_rs, col0, s.n, k0 + kMmK, s.k, s.r_mode, -0.f);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            f32x4_t a[T], c[T];
#pragma unroll
            for (int i = 0; i < T; ++i) a[i] = *reinterpret_cast<const f32x4_t *>(la + i * 16 * kMmPitch + h * 4);
#pragma unroll
            for (int j = 0; j < T; ++j) c[j] = *reinterpret_cast<const f32x4_t *>(ra + j * 16 * kMmPitch + h * 4);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < T; ++i)
#pragma unroll
                    for (int j = 0; j < T; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][e], c[j][e], acc[i][j], 0, 0, 0);
        }
    }
    const uint64_t out_base = static_cast<uint64_t>(blockIdx.z) * s.m * s.n;
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t row = row0 + ((wave / WN) * T + i) * 16 + 4 * (lane >> 4) + r;
                const uint32_t col = col0 + ((wave % WN) * T + j) * 16 + (lane & 15);
                if (row < s.m && col < s.n)
                    Float<DT>::put(dst, static_cast<int64_t>(out_base + static_cast<uint64_t>(row) * s.n + col),
                                   acc[i][j][r]);
            }
}

// How an operand's tile is read: rs, ks its strides along the rows (columns
// for rhs) and k, `base` the address of its first element.
int stage_mode(const void *base, int size, int64_t rs, int64_t ks, int64_t rows, int64_t k, const int64_t *bs,
               uint32_t batch_ndim) {
    bool pieces = reinterpret_cast<uintptr_t>(base) % 16 == 0;  // and every batch entry's first element
    const int64_t per = 16 / size;                              // elements in 16 bytes
    for (uint32_t d = 0; d < batch_ndim; ++d) pieces = pieces && bs[d] % per == 0;
    if (pieces && ks == 1 && k % 8 == 0 && (rs % per == 0 || rows == 1)) return kPiecesK;
    if (pieces && rs == 1 && rows % 8 == 0 && (ks % per == 0 || k == 1)) return kPiecesRows;
    return ks <= rs ? kAlongK : kAlongRows;
}

// Launches the tile for the shape: 64 x 64 outputs a block; 32 x 128 or 128 x
// 32 where one extent is at most 32; 32 x 32 (a quarter of the sums a
// wavefront) where the larger ones would give fewer blocks than CUs (24 x
// [512, 512] x [512, 128], 384 blocks of 64 x 64: 43 us against 64 us in 1536
// of 32 x 32).
template <int DT>
void launch_matmul(hipStream_t stream, uint32_t cus, const void *lhs, const void *rhs, const MatmulShape &s,
                   uint32_t batch, void *dst) {
    using E = typename Float<DT>::T;
    auto go = [&](auto kernel, uint32_t bm, uint32_t bn) {
        hipLaunchKernelGGL(kernel, dim3((s.n + bn - 1) / bn, (s.m + bm - 1) / bm, batch), dim3(kThreads), 0, stream,
                           static_cast<const E *>(lhs), static_cast<const E *>(rhs), s, static_cast<E *>(dst));
    };
    const uint32_t bm = s.m <= 32 ? 32 : s.n <= 32 ? 128 : 64, bn = s.m <= 32 ? 128 : s.n <= 32 ? 32 : 64;
    const uint64_t blocks = static_cast<uint64_t>((s.m + bm - 1) / bm) * ((s.n + bn - 1) / bn) * batch;
    auto pick = [&](auto pieces) {
        constexpr bool P = decltype(pieces)::value;
        if (blocks < cus)
            go(matmul_kernel<DT, 2, 2, 1, P>, 32, 32);
        else if (bm == 32)
            go(matmul_kernel<DT, 1, 4, 2, P>, 32, 128);
        else if (bn == 32)
            go(matmul_kernel<DT, 4, 1, 2, P>, 128, 32);
        else
            go(matmul_kernel<DT, 2, 2, 2, P>, 64, 64);
    };
    if (s.l_mode >= kPiecesK && s.r_mode >= kPiecesK)
        pick(std::true_type{});
    else
        pick(std::false_type{});
}

// index_select_rows (src/metal/kernels/index_select.metal:11-29): an id at
// or past the table's rows gives a zero row.
template <typename T>
__global__ __launch_bounds__(kThreads) void index_select_kernel(const T *__restrict__ table, int64_t t_off,
                                                                int64_t t_rs, int64_t t_cs, uint32_t rows,
                                                                uint32_t cols, const uint32_t *__restrict__ ids,
                                                                View iv, T *__restrict__ dst, uint32_t n) {
    const uint32_t i = gid();
    if (i >= n) return;
    const uint32_t r = i / cols, c = i % cols;
    const uint32_t id = ids[at(r, iv)];
    dst[i] = id < rows ? table[t_off + static_cast<int64_t>(id) * t_rs + static_cast<int64_t>(c) * t_cs] : T(0);
}

// ---- host side ----

int itemsize(int dtype) { return dtype == FH_BF16 ? 2 : 4; }

bool valid_dtype(int dtype) { return dtype == FH_F32 || dtype == FH_BF16 || dtype == FH_U32; }

int require_float(const char *fn, int dtype) {
    if (dtype != FH_F32 && dtype != FH_BF16)
        return fail(FH_ERR_DTYPE, "%s: dtype %d is not a float dtype (TensorError::DTypeNotFloat)", fn, dtype);
    return FH_OK;
}

int64_t numel_of(const fh_view &v) {
    int64_t n = 1;
    for (int d = 0; d < v.ndim; ++d) n *= v.dims[d];
    return n;
}

// Checks a view (rank, sizes, strides, element count) and that every element
// it addresses lies inside one live allocation; fills the kernel's View.
int check_view(const fh_device *dev, const char *fn, const char *what, const void *base, const fh_view *v, int dtype,
               View *out) {
    if (!v) return fail(FH_ERR_INVALID_ARGUMENT, "%s: %s view is null", fn, what);
    if (v->ndim < 0 || v->ndim > kRank)
        return fail(FH_ERR_INVALID_ARGUMENT, "%s: %s has rank %d (TensorError::RankTooLarge)", fn, what, v->ndim);
    if (v->offset < 0) return fail(FH_ERR_INVALID_ARGUMENT, "%s: %s has a negative offset", fn, what);
    unsigned __int128 numel = 1, last = static_cast<unsigned __int128>(v->offset);
    for (int d = 0; d < v->ndim; ++d) {
        if (v->dims[d] < 0 || v->dims[d] > kMaxNumel || v->strides[d] < 0)
            return fail(FH_ERR_INVALID_ARGUMENT, "%s: %s dim %d has size %lld, stride %lld", fn, what, d,
                        (long long)v->dims[d], (long long)v->strides[d]);
        numel *= static_cast<uint64_t>(v->dims[d]);
        if (v->dims[d] > 0) last += static_cast<unsigned __int128>(v->dims[d] - 1) * static_cast<uint64_t>(v->strides[d]);
    }
    if (numel > static_cast<unsigned __int128>(kMaxNumel))
        return fail(FH_ERR_INDEX_TOO_LARGE, "%s: %s has more than 2^31 - 1 elements (TensorError::NumelOverflow)", fn,
                    what);
    const int size = itemsize(dtype);
    if (reinterpret_cast<uintptr_t>(base) % size != 0)
        return fail(FH_ERR_INVALID_ARGUMENT, "%s: %s is misaligned for its dtype", fn, what);
    if (numel > 0) {
        const unsigned __int128 bytes = (last + 1) * static_cast<unsigned>(size);
        if (bytes > static_cast<unsigned __int128>(UINT64_MAX >> 1))
            return fail(FH_ERR_OUT_OF_BOUNDS, "%s: %s addresses past any allocation", fn, what);
        if (int rc = check_range(dev, base, static_cast<uint64_t>(bytes), fn, what)) return rc;
    }
    out->offset = v->offset;
    out->ndim = v->ndim;
    for (int d = 0; d < kRank; ++d) {
        out->dims[d] = d < v->ndim ? static_cast<uint32_t>(v->dims[d]) : 1u;
        out->strides[d] = d < v->ndim ? v->strides[d] : 0;
    }
    return FH_OK;
}

int check_out(const fh_device *dev, const char *fn, void *dst, int64_t numel, int dtype) {
    if (reinterpret_cast<uintptr_t>(dst) % itemsize(dtype) != 0)
        return fail(FH_ERR_INVALID_ARGUMENT, "%s: dst is misaligned for its dtype", fn);
    return check_range(dev, dst, static_cast<uint64_t>(numel) * itemsize(dtype), fn, "dst");
}

int begin(fh_device *dev, const char *fn) {
    if (int rc = check_usable(dev, fn)) return rc;
    return FH_OK;
}

uint32_t blocks_for(int64_t n) { return static_cast<uint32_t>((n + kThreads - 1) / kThreads); }

// A contiguous view of `dims` at `offset` (the layout of a fresh output).
View contiguous(const int64_t *dims, int ndim, int64_t offset) {
    View v{};
    v.offset = offset;
    v.ndim = ndim;
    int64_t stride = 1;
    for (int d = kRank - 1; d >= 0; --d) {
        v.dims[d] = d < ndim ? static_cast<uint32_t>(dims[d]) : 1u;
        v.strides[d] = d < ndim ? stride : 0;
        if (d < ndim) stride *= dims[d];
    }
    return v;
}

// The common walk of N views of the same dims. base[v] is the address of view
// v's storage (element size `size`); a view may be read in pieces of
// `per_piece` elements where it is contiguous along the last walked dim (or,
// with `broadcast`, constant along it) and every piece is 16-byte aligned.
// allow: the caller's own operand allows pieces.
template <int N>
Walk<N> walk_of(const View *const (&views)[N], const void *const (&base)[N], int size, uint32_t per_piece,
                bool broadcast, bool allow) {
    Walk<N> w{};
    for (int v = 0; v < N; ++v) w.offset[v] = views[v]->offset;
    for (int d = 0; d < views[0]->ndim; ++d) {
        const uint32_t n = views[0]->dims[d];
        if (n == 1) continue;
        bool merge = w.ndim > 0;
        for (int v = 0; v < N && merge; ++v)
            merge = w.strides[v][w.ndim - 1] == views[v]->strides[d] * static_cast<int64_t>(n);
        if (merge) {
            w.dims[w.ndim - 1] *= n;
        } else {
            w.dims[w.ndim] = n;
            ++w.ndim;
        }
        for (int v = 0; v < N; ++v) w.strides[v][w.ndim - 1] = views[v]->strides[d];
    }
    if (w.ndim == 0) w.dims[w.ndim++] = 1;  // one element
    const uint32_t last = w.ndim - 1;
    const int64_t per16 = 16 / size;  // elements in 16 bytes
    bool pieces = allow && w.dims[last] % per_piece == 0;
    for (int v = 0; v < N && pieces; ++v) {
        if (broadcast && w.strides[v][last] == 0) continue;
        pieces = w.strides[v][last] == 1 &&
                 (reinterpret_cast<uintptr_t>(base[v]) + static_cast<uint64_t>(w.offset[v]) * size) % 16 == 0;
        for (uint32_t d = 0; d < last && pieces; ++d) pieces = w.strides[v][d] % per16 == 0;
    }
    w.pieces = pieces;
    // one element a thread where a view steps by more than one along the
    // last dim: more blocks then share the cache lines it touches
    // ([3072, 512] f32 read transposed: 8.8 us, 16.6 us with four)
    w.single = 4;
    for (int v = 0; v < N; ++v)
        if (w.strides[v][last] > 1) w.single = 1;
    if (pieces) {
        w.dims[last] /= per_piece;
        for (int v = 0; v < N; ++v) w.strides[v][last] *= per_piece;
    }
    for (uint32_t d = 0; d < w.ndim; ++d) {
        const uint32_t shift = w.dims[d] > 1 ? 32 - static_cast<uint32_t>(__builtin_clz(w.dims[d] - 1)) : 0;
        w.shift[d] = shift;
        w.mul[d] = static_cast<uint32_t>(((1ull << 32) * ((1ull << shift) - w.dims[d])) / w.dims[d] + 1);
    }
    return w;
}

// Threads' worth of work and the grid for it.
template <int N>
uint32_t walk_items(const Walk<N> &w, int64_t n, uint32_t per_piece) {
    return static_cast<uint32_t>(w.pieces ? n / per_piece : n);
}
template <int N>
uint32_t walk_blocks(const Walk<N> &w, uint32_t items) {
    return blocks_for(w.pieces ? items : (static_cast<int64_t>(items) + w.single - 1) / w.single);
}

// Launches the move of every element of src (view sv, n elements) into the
// window wv of dst.
int scatter(fh_device *dev, const char *fn, int dtype, const void *src, const View &sv, void *dst, const View &wv,
            int64_t n) {
    if (n == 0) return FH_OK;
    const int size = itemsize(dtype);
    const uint32_t per = 16 / size;
    const View *const views[2] = {&sv, &wv};
    const void *const base[2] = {src, dst};
    const Walk<2> w = walk_of<2>(views, base, size, per, false, true);
    const uint32_t items = walk_items(w, n, per);
    return dispatch(dev, fn, [&] {
        if (dtype == FH_BF16)
            hipLaunchKernelGGL(move_kernel<uint16_t>, dim3(walk_blocks(w, items)), dim3(kThreads), 0, dev->stream,
                               static_cast<const uint16_t *>(src), static_cast<uint16_t *>(dst), w, items);
        else
            hipLaunchKernelGGL(move_kernel<uint32_t>, dim3(walk_blocks(w, items)), dim3(kThreads), 0, dev->stream,
                               static_cast<const uint32_t *>(src), static_cast<uint32_t *>(dst), w, items);
    });
}

// dst = f over one or two views of dtype IN.
template <int IN, int OUT, int N, class F>
int map(fh_device *dev, const char *fn, const View *const (&views)[N], const void *const (&src)[N], void *dst,
        int64_t n, F f) {
    using TI = typename Float<IN>::T;
    using TO = typename Float<OUT>::T;
    const Walk<N> w = walk_of<N>(views, src, static_cast<int>(sizeof(TI)), 8, true,
                                 reinterpret_cast<uintptr_t>(dst) % 16 == 0);
    const uint32_t items = walk_items(w, n, 8);
    return dispatch(dev, fn, [&] {
        hipLaunchKernelGGL((map_kernel<IN, OUT, N, F>), dim3(walk_blocks(w, items)), dim3(kThreads), 0, dev->stream,
                           static_cast<const TI *>(src[0]), static_cast<const TI *>(src[N - 1]),
                           static_cast<TO *>(dst), w, items, f);
    });
}

// dims equal except at `dim` (src/nn/primitive.rs:356-367)
bool dims_equal_except(const fh_view &a, const fh_view &b, int dim) {
    if (a.ndim != b.ndim) return false;
    for (int d = 0; d < a.ndim; ++d)
        if (d != dim && a.dims[d] != b.dims[d]) return false;
    return true;
}

}  // namespace
}  // namespace fh

using namespace fh;

extern "C" int fh_copy_strided(fh_device *dev, int dtype, const void *src, const fh_view *view, void *dst) {
    const char *fn = "fh_copy_strided";
    if (int rc = begin(dev, fn)) return rc;
    if (!valid_dtype(dtype)) return fail(FH_ERR_DTYPE, "%s: unknown dtype %d", fn, dtype);
    View v;
    if (int rc = check_view(dev, fn, "src", src, view, dtype, &v)) return rc;
    const int64_t n = numel_of(*view);
    if (int rc = check_out(dev, fn, dst, n, dtype)) return rc;
    if (n == 0) return FH_OK;
    if (int rc = set_current(dev, fn)) return rc;
    const View out = contiguous(view->dims, view->ndim, 0);
    return scatter(dev, fn, dtype, src, v, dst, out, n);
}

extern "C" int fh_to_dtype(fh_device *dev, int from, const void *src, const fh_view *view, int to, void *dst) {
    const char *fn = "fh_to_dtype";
    if (int rc = begin(dev, fn)) return rc;
    if (int rc = require_float(fn, from)) return rc;
    if (int rc = require_float(fn, to)) return rc;
    if (from == to) return fh_copy_strided(dev, from, src, view, dst);
    View v;
    if (int rc = check_view(dev, fn, "src", src, view, from, &v)) return rc;
    const int64_t n = numel_of(*view);
    if (int rc = check_out(dev, fn, dst, n, to)) return rc;
    if (n == 0) return FH_OK;
    if (int rc = set_current(dev, fn)) return rc;
    const View *const views[1] = {&v};
    const void *const base[1] = {src};
    if (from == FH_F32) return map<FH_F32, FH_BF16, 1>(dev, fn, views, base, dst, n, Identity{});
    return map<FH_BF16, FH_F32, 1>(dev, fn, views, base, dst, n, Identity{});
}

extern "C" int fh_unary(fh_device *dev, int op, int dtype, const void *src, const fh_view *view, void *dst) {
    const char *fn = "fh_unary";
    if (int rc = begin(dev, fn)) return rc;
    if (op < FH_NEG || op > FH_RECIPROCAL) return fail(FH_ERR_INVALID_ARGUMENT, "%s: unknown unary op %d", fn, op);
    if (int rc = require_float(fn, dtype)) return rc;
    View v;
    if (int rc = check_view(dev, fn, "src", src, view, dtype, &v)) return rc;
    const int64_t n = numel_of(*view);
    if (int rc = check_out(dev, fn, dst, n, dtype)) return rc;
    if (n == 0) return FH_OK;
    if (int rc = set_current(dev, fn)) return rc;
    const View *const views[1] = {&v};
    const void *const base[1] = {src};
    if (dtype == FH_F32) return map<FH_F32, FH_F32, 1>(dev, fn, views, base, dst, n, UnaryOf{op});
    return map<FH_BF16, FH_BF16, 1>(dev, fn, views, base, dst, n, UnaryOf{op});
}

extern "C" int fh_binary(fh_device *dev, int op, int dtype, const void *lhs, const fh_view *lhs_view,
                         const void *rhs, const fh_view *rhs_view, void *dst) {
    const char *fn = "fh_binary";
    if (int rc = begin(dev, fn)) return rc;
    if (op < FH_ADD || op > FH_DIV) return fail(FH_ERR_INVALID_ARGUMENT, "%s: unknown binary op %d", fn, op);
    if (int rc = require_float(fn, dtype)) return rc;
    View lv, rv;
    if (int rc = check_view(dev, fn, "lhs", lhs, lhs_view, dtype, &lv)) return rc;
    if (int rc = check_view(dev, fn, "rhs", rhs, rhs_view, dtype, &rv)) return rc;
    if (!dims_equal_except(*lhs_view, *rhs_view, -1))
        return fail(FH_ERR_INVALID_ARGUMENT, "%s: lhs and rhs views must have the output's dims (broadcast first)",
                    fn);
    const int64_t n = numel_of(*lhs_view);
    if (int rc = check_out(dev, fn, dst, n, dtype)) return rc;
    if (n == 0) return FH_OK;
    if (int rc = set_current(dev, fn)) return rc;
    const View *const views[2] = {&lv, &rv};
    const void *const base[2] = {lhs, rhs};
    if (dtype == FH_F32) return map<FH_F32, FH_F32, 2>(dev, fn, views, base, dst, n, BinaryOf{op});
    return map<FH_BF16, FH_BF16, 2>(dev, fn, views, base, dst, n, BinaryOf{op});
}

extern "C" int fh_reduce(fh_device *dev, int op, int dtype, const void *src, const fh_view *view, int32_t dim,
                         void *dst) {
    const char *fn = "fh_reduce";
    if (int rc = begin(dev, fn)) return rc;
    if (op < FH_SUM || op > FH_ARGMAX) return fail(FH_ERR_INVALID_ARGUMENT, "%s: unknown reduce op %d", fn, op);
    if (int rc = require_float(fn, dtype)) return rc;
    View v;
    if (int rc = check_view(dev, fn, "src", src, view, dtype, &v)) return rc;
    if (dim < 0 || dim >= view->ndim)
        return fail(FH_ERR_INVALID_ARGUMENT, "%s: dim %d of a rank-%d view (TensorError::DimOutOfRange)", fn, dim,
                    view->ndim);
    const int64_t dim_size = view->dims[dim];
    if (op != FH_SUM && dim_size == 0)
        return fail(FH_ERR_INVALID_ARGUMENT, "%s: reduction over an empty dim (TensorError::EmptyReduction)", fn);
    int64_t rows = 1;
    for (int d = 0; d < view->ndim; ++d) rows *= d == dim ? 1 : view->dims[d];
    const int out_dtype = op == FH_ARGMAX ? FH_U32 : dtype;
    if (int rc = check_out(dev, fn, dst, rows, out_dtype)) return rc;
    if (rows == 0) return FH_OK;
    if (int rc = set_current(dev, fn)) return rc;
    View rv = v;  // the input's strides over the output's dims
    rv.dims[dim] = 1;
    const int64_t stride = view->strides[dim];
    const uint32_t size = static_cast<uint32_t>(dim_size);
    // A wavefront per row where the rows alone give every CU 4 blocks of
    // them, else a block per row. Sums of 4096 rows, block / wavefront per row:
    // f32 512 long 5.9 / 3.7 us, 8192 27.9 / 20.7, 128256 583 / 363; bf16 512
    // 5.9 / 3.9, 128256 530 / 294. Along a strided dim also (8192 rows of 64 f32
    // 8.6 / 4.1, of 4096 225 / 178), except f32 rows of 256 to 2047 values while
    // there are fewer than 256 rows a CU: 4096 of 512 12.5 / 14.2, 8192 of 1024
    // 38.9 / 47.3 (65536 of 256 81.2 / 79.3).
    const bool block_strided = dtype == FH_F32 && stride > 1 && size >= 256 && size < 2048 &&
                               rows < 256ll * dev->compute_units;
    if (op != FH_ARGMAX && rows >= 16ll * dev->compute_units && !block_strided) {
        return dispatch(dev, fn, [&] {
            const uint32_t n_rows = static_cast<uint32_t>(rows);
            const uint32_t blocks = n_rows / 4 + 1;
            const dim3 grid(blocks < (1u << 20) ? blocks : (1u << 20)), block(kThreads);
            auto go = [&](auto kernel, auto *s) {
                hipLaunchKernelGGL(kernel, grid, block, 0, dev->stream, s, rv, size, stride,
                                   static_cast<std::remove_const_t<std::remove_pointer_t<decltype(s)>> *>(dst), n_rows);
            };
            if (dtype == FH_F32 && op == FH_SUM)
                go(reduce_wave_kernel<FH_F32, false>, static_cast<const float *>(src));
            else if (dtype == FH_F32)
                go(reduce_wave_kernel<FH_F32, true>, static_cast<const float *>(src));
            else if (op == FH_SUM)
                go(reduce_wave_kernel<FH_BF16, false>, static_cast<const uint16_t *>(src));
            else
                go(reduce_wave_kernel<FH_BF16, true>, static_cast<const uint16_t *>(src));
        });
    }
    return dispatch(dev, fn, [&] {
        // at most 2^20 blocks (2^28 work-items); the kernels stride over the rest
        const uint32_t n_rows = static_cast<uint32_t>(rows);
        const dim3 grid(n_rows < (1u << 20) ? n_rows : (1u << 20)), block(kThreads);
        if (dtype == FH_F32) {
            auto *s = static_cast<const float *>(src);
            if (op == FH_SUM)
                hipLaunchKernelGGL((reduce_kernel<FH_F32, false>), grid, block, 0, dev->stream, s, rv, size, stride,
                                   static_cast<float *>(dst), n_rows);
            else if (op == FH_AMAX)
                hipLaunchKernelGGL((reduce_kernel<FH_F32, true>), grid, block, 0, dev->stream, s, rv, size, stride,
                                   static_cast<float *>(dst), n_rows);
            else
                hipLaunchKernelGGL(argmax_kernel<FH_F32>, grid, block, 0, dev->stream, s, rv, size, stride,
                                   static_cast<uint32_t *>(dst), n_rows);
        } else {
            auto *s = static_cast<const uint16_t *>(src);
            if (op == FH_SUM)
                hipLaunchKernelGGL((reduce_kernel<FH_BF16, false>), grid, block, 0, dev->stream, s, rv, size, stride,
                                   static_cast<uint16_t *>(dst), n_rows);
            else if (op == FH_AMAX)
                hipLaunchKernelGGL((reduce_kernel<FH_BF16, true>), grid, block, 0, dev->stream, s, rv, size, stride,
                                   static_cast<uint16_t *>(dst), n_rows);
            else
                hipLaunchKernelGGL(argmax_kernel<FH_BF16>, grid, block, 0, dev->stream, s, rv, size, stride,
                                   static_cast<uint32_t *>(dst), n_rows);
        }
    });
}

extern "C" int fh_matmul(fh_device *dev, int dtype, const void *lhs, const fh_view *lhs_view, const void *rhs,
                         const fh_view *rhs_view, void *dst) {
    const char *fn = "fh_matmul";
    if (int rc = begin(dev, fn)) return rc;
    if (int rc = require_float(fn, dtype)) return rc;
    View lv, rv;
    if (int rc = check_view(dev, fn, "lhs", lhs, lhs_view, dtype, &lv)) return rc;
    if (int rc = check_view(dev, fn, "rhs", rhs, rhs_view, dtype, &rv)) return rc;
    // src/nn/primitive.rs:209-233: [..., m, k] x [..., k, n], equal batch dims
    const int nd = lhs_view->ndim;
    if (nd < 2 || rhs_view->ndim != nd || lhs_view->dims[nd - 1] != rhs_view->dims[nd - 2])
        return fail(FH_ERR_INVALID_ARGUMENT, "%s: shapes cannot be multiplied (TensorError::MatmulIncompatible)", fn);
    for (int d = 0; d < nd - 2; ++d)
        if (lhs_view->dims[d] != rhs_view->dims[d])
            return fail(FH_ERR_INVALID_ARGUMENT, "%s: batch dims differ (TensorError::MatmulIncompatible)", fn);
    MatmulShape s{};
    s.m = static_cast<uint32_t>(lhs_view->dims[nd - 2]);
    s.k = static_cast<uint32_t>(lhs_view->dims[nd - 1]);
    s.n = static_cast<uint32_t>(rhs_view->dims[nd - 1]);
    s.batch_ndim = static_cast<uint32_t>(nd - 2);
    int64_t batch = 1;
    for (int d = 0; d < nd - 2; ++d) {
        s.batch_dims[d] = static_cast<uint32_t>(lhs_view->dims[d]);
        s.l_bs[d] = lhs_view->strides[d];
        s.r_bs[d] = rhs_view->strides[d];
        batch *= lhs_view->dims[d];
    }
    s.l_off = lhs_view->offset, s.l_rs = lhs_view->strides[nd - 2], s.l_cs = lhs_view->strides[nd - 1];
    s.r_off = rhs_view->offset, s.r_rs = rhs_view->strides[nd - 2], s.r_cs = rhs_view->strides[nd - 1];
    const int64_t out = batch * s.m * s.n;
    if (out > kMaxNumel) return fail(FH_ERR_INDEX_TOO_LARGE, "%s: output exceeds 2^31 - 1 elements", fn);
    if (int rc = check_out(dev, fn, dst, out, dtype)) return rc;
    if (out == 0) return FH_OK;
    if (batch > 65535) return fail(FH_ERR_INDEX_TOO_LARGE, "%s: %lld batch entries exceed the grid", fn,
                                   (long long)batch);
    if (int rc = set_current(dev, fn)) return rc;
    // the limits of a grid of 32 x 32 tiles: rows in grid.y, and grid.x * 256
    // work-items below 2^32
    if ((s.m + 31) / 32 > 65535) return fail(FH_ERR_INDEX_TOO_LARGE, "%s: m=%u exceeds the grid", fn, s.m);
    if (static_cast<uint64_t>((s.n + 31) / 32) * kThreads > 0xFFFFFFFFull)
        return fail(FH_ERR_INDEX_TOO_LARGE, "%s: n=%u exceeds the grid", fn, s.n);
    const int size = itemsize(dtype);
    s.l_mode = stage_mode(static_cast<const char *>(lhs) + s.l_off * size, size, s.l_rs, s.l_cs, s.m, s.k, s.l_bs,
                          s.batch_ndim);
    s.r_mode = stage_mode(static_cast<const char *>(rhs) + s.r_off * size, size, s.r_cs, s.r_rs, s.n, s.k, s.r_bs,
                          s.batch_ndim);
    return dispatch(dev, fn, [&] {
        if (dtype == FH_F32)
            launch_matmul<FH_F32>(dev->stream, dev->compute_units, lhs, rhs, s, static_cast<uint32_t>(batch), dst);
        else
            launch_matmul<FH_BF16>(dev->stream, dev->compute_units, lhs, rhs, s, static_cast<uint32_t>(batch), dst);
    });
}

extern "C" int fh_index_select(fh_device *dev, int dtype, const void *table, const fh_view *table_view,
                               const uint32_t *ids, const fh_view *ids_view, void *dst) {
    const char *fn = "fh_index_select";
    if (int rc = begin(dev, fn)) return rc;
    if (int rc = require_float(fn, dtype)) return rc;
    View tv, iv;
    if (int rc = check_view(dev, fn, "table", table, table_view, dtype, &tv)) return rc;
    if (int rc = check_view(dev, fn, "ids", ids, ids_view, FH_U32, &iv)) return rc;
    if (table_view->ndim != 2 || ids_view->ndim != 1)
        return fail(FH_ERR_INVALID_ARGUMENT, "%s: a 2-D table and 1-D ids (TensorError::IndexSelectIncompatible)",
                    fn);
    const int64_t rows = table_view->dims[0], cols = table_view->dims[1], count = ids_view->dims[0];
    const int64_t n = count * cols;
    if (n > kMaxNumel) return fail(FH_ERR_INDEX_TOO_LARGE, "%s: output exceeds 2^31 - 1 elements", fn);
    if (int rc = check_out(dev, fn, dst, n, dtype)) return rc;
    if (n == 0) return FH_OK;
    if (int rc = set_current(dev, fn)) return rc;
    return dispatch(dev, fn, [&] {
        if (dtype == FH_BF16)
            hipLaunchKernelGGL(index_select_kernel<uint16_t>, dim3(blocks_for(n)), dim3(kThreads), 0, dev->stream,
                               static_cast<const uint16_t *>(table), tv.offset, tv.strides[0], tv.strides[1],
                               static_cast<uint32_t>(rows), static_cast<uint32_t>(cols), ids, iv,
                               static_cast<uint16_t *>(dst), static_cast<uint32_t>(n));
        else
            hipLaunchKernelGGL(index_select_kernel<uint32_t>, dim3(blocks_for(n)), dim3(kThreads), 0, dev->stream,
                               static_cast<const uint32_t *>(table), tv.offset, tv.strides[0], tv.strides[1],
                               static_cast<uint32_t>(rows), static_cast<uint32_t>(cols), ids, iv,
                               static_cast<uint32_t *>(dst), static_cast<uint32_t>(n));
    });
}

extern "C" int fh_cat(fh_device *dev, int dtype, int32_t dim, const void *lhs, const fh_view *lhs_view,
                      const void *rhs, const fh_view *rhs_view, void *dst) {
    const char *fn = "fh_cat";
    if (int rc = begin(dev, fn)) return rc;
    if (int rc = require_float(fn, dtype)) return rc;
    View lv, rv;
    if (int rc = check_view(dev, fn, "lhs", lhs, lhs_view, dtype, &lv)) return rc;
    if (int rc = check_view(dev, fn, "rhs", rhs, rhs_view, dtype, &rv)) return rc;
    if (dim < 0 || dim >= lhs_view->ndim)
        return fail(FH_ERR_INVALID_ARGUMENT, "%s: dim %d (TensorError::DimOutOfRange)", fn, dim);
    if (!dims_equal_except(*lhs_view, *rhs_view, dim))
        return fail(FH_ERR_INVALID_ARGUMENT, "%s: shapes cannot be concatenated (TensorError::CatIncompatible)", fn);
    int64_t dims[kRank];
    for (int d = 0; d < lhs_view->ndim; ++d) dims[d] = lhs_view->dims[d];
    dims[dim] = lhs_view->dims[dim] + rhs_view->dims[dim];
    if (dims[dim] > kMaxNumel) return fail(FH_ERR_INVALID_ARGUMENT, "%s: dim %d overflows", fn, dim);
    const int64_t nl = numel_of(*lhs_view), nr = numel_of(*rhs_view);
    if (nl + nr > kMaxNumel) return fail(FH_ERR_INDEX_TOO_LARGE, "%s: output exceeds 2^31 - 1 elements", fn);
    if (int rc = check_out(dev, fn, dst, nl + nr, dtype)) return rc;
    if (nl + nr == 0) return FH_OK;
    if (int rc = set_current(dev, fn)) return rc;
    // MetalDevice::cat: both inputs scatter into windows of the contiguous
    // output, rhs from lhs.dims[dim] along dim
    const View out = contiguous(dims, lhs_view->ndim, 0);
    View lw = out, rw = out;
    for (int d = 0; d < lhs_view->ndim; ++d) lw.dims[d] = static_cast<uint32_t>(lhs_view->dims[d]);
    for (int d = 0; d < lhs_view->ndim; ++d) rw.dims[d] = static_cast<uint32_t>(rhs_view->dims[d]);
    rw.offset = lhs_view->dims[dim] * out.strides[dim];
    if (int rc = scatter(dev, fn, dtype, lhs, lv, dst, lw, nl)) return rc;
    return scatter(dev, fn, dtype, rhs, rv, dst, rw, nr);
}

extern "C" int fh_slice_scatter(fh_device *dev, int dtype, int32_t dim, int64_t start, void *target,
                                const fh_view *target_view, const void *src, const fh_view *src_view) {
    const char *fn = "fh_slice_scatter";
    if (int rc = begin(dev, fn)) return rc;
    if (int rc = require_float(fn, dtype)) return rc;
    View tv, sv;
    if (int rc = check_view(dev, fn, "target", target, target_view, dtype, &tv)) return rc;
    if (int rc = check_view(dev, fn, "src", src, src_view, dtype, &sv)) return rc;
    if (dim < 0 || dim >= target_view->ndim)
        return fail(FH_ERR_INVALID_ARGUMENT, "%s: dim %d (TensorError::DimOutOfRange)", fn, dim);
    // src/nn/primitive.rs:314-335: src fits the target from start along dim
    if (start < 0 || !dims_equal_except(*target_view, *src_view, dim) ||
        start + src_view->dims[dim] > target_view->dims[dim])
        return fail(FH_ERR_INVALID_ARGUMENT, "%s: slice does not fit the target (TensorError::SliceScatterOutOfBounds)",
                    fn);
    const View want = contiguous(target_view->dims, target_view->ndim, target_view->offset);
    for (int d = 0; d < target_view->ndim; ++d)
        if (target_view->dims[d] != 1 && target_view->strides[d] != want.strides[d])
            return fail(FH_ERR_INVALID_ARGUMENT,
                        "%s: the target must be contiguous (TensorError::SliceScatterNonContiguous)", fn);
    const int64_t n = numel_of(*src_view);
    if (n == 0) return FH_OK;
    if (int rc = set_current(dev, fn)) return rc;
    View window = tv;  // the target's strides over src's dims, from start along dim
    for (int d = 0; d < target_view->ndim; ++d) window.dims[d] = static_cast<uint32_t>(src_view->dims[d]);
    window.offset = target_view->offset + start * target_view->strides[dim];
    return scatter(dev, fn, dtype, src, sv, target, window, n);
}

// q4 GEMM for few rows (9 up to a few hundred: batched decode above the
// GEMV's 8 rows, short prompts):
// Y[m, r] = sum_j X[m, j] * RNE_bf16(s[r, j/64] * q[r, j] + b[r, j/64]).
// Replaces matmul_tiled (src/metal/kernels/matmul.metal:29-65) behind
// Linear::forward (src/nn/linear.rs:22-35), as q4_gemm.hip does for prompts.
//
// With so few rows the weight stream and its dequantisation are the work; a
// 256-row tile spends its matrix-core time and X traffic on padding, and its
// few blocks leave CUs idle or need f32 partials in memory. Design for CDNA4:
// - A block owns RT x 16 rows and CT x 16 columns over ALL of K. Its eight
//   wavefronts split K into contiguous ranges, each computing the whole tile
//   over its range (v_mfma_f32_16x16x32_bf16, RT x CT accumulators), so every
//   weight of the block is loaded and dequantised once, and nothing but the
//   final sum is shared: the main loop has no block barrier.
// - The host picks CT so that the column tiles split evenly over the CUs
//   (28672 columns are 1792 tiles, 7 a CU; 5120 are 320).
// - Weights go straight to registers: a lane loads 16 bytes of its column's
//   row, 64 contiguous bytes per column and 128-value chunk of K. A 4 x 4
//   transpose over the four lanes of a column (four permlane swaps per 4
//   words) then gives MFMA sub-step j the words of k = 32 j .. 32 j + 31 in
//   natural order.
// - X goes through LDS by DMA into the wavefront's own two buffers of 8 KB,
//   one in use while the next is in flight; rows' 16-byte pieces are
//   XOR-swizzled so that fragment reads are conflict-free.
// - The eight partial tiles meet in LDS and are added in K order, then
//   rounded once: results do not depend on timing.
// What bounds it (per-wavefront stamps, 32 x 28672 x 4096, weights cold): the
// weights' arrival, 59 MB in about 11 us, and the dequantisation, about 27
// VALU instructions per packed word of which a wavefront issues one per 8
// clocks (two wavefronts per SIMD: one per 4.6), about 12 us; the two overlap
// only partly. Measured against the 256-row kernels it replaces there: 32 x
// 28672 x 4096 60.8 -> 24.9 us, 64 x 16384 x 3072 37.2 -> 16.0, 128 x 5120 x
// 3072 25.0 -> 12.9, 16 x 28672 x 4096 72.5 -> 24.2 (cold). Tried and no
// faster: two blocks of 80 KB LDS per CU, 128-row blocks, the fp16-denormal
// form of the dequantisation (v_fma_mix, 17 instead of 23 instructions per
// word: 1 us).
#include <type_traits>

#include "decoder_common.hpp"
#include "device.hpp"
#include "q4_common.hpp"
#include "q4_gemm.hpp"

namespace fh {

namespace {

constexpr int kRWaves = 8;
constexpr int kRThreads = 64 * kRWaves;
// scale and bias bytes a wavefront keeps in LDS: 8 slots of 16 columns x 8
// groups of each
constexpr uint32_t kRSbBytes = 4096;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;

__device__ __forceinline__ uint32_t rows_low_nibbles(uint32_t w) {
    uint32_t r;
    asm("v_and_b32 %0, 0x0f0f0f0f, %1" : "=v"(r) : "v"(w));
    return r;
}

template <int I>
__device__ __forceinline__ float rows_ubyte(uint32_t v) {
    return static_cast<float>((v >> (8 * I)) & 0xFFu);
}

// 8 weights of one packed word -> bf16x8 in order: fma(s, q, b) of the exact
// nibble, RNE to bf16, the fh_q4_dequant value whenever s * q is finite.
__device__ __forceinline__ bf16x8_t rows_dequant8(uint32_t w, float s, float b) {
    const uint32_t lo = rows_low_nibbles(w), hi = rows_low_nibbles(w >> 4);
    uint4 o;
    o.x = f32x2_to_bf16x2_rne(fmaf(s, rows_ubyte<0>(lo), b), fmaf(s, rows_ubyte<0>(hi), b));
    o.y = f32x2_to_bf16x2_rne(fmaf(s, rows_ubyte<1>(lo), b), fmaf(s, rows_ubyte<1>(hi), b));
    o.z = f32x2_to_bf16x2_rne(fmaf(s, rows_ubyte<2>(lo), b), fmaf(s, rows_ubyte<2>(hi), b));
    o.w = f32x2_to_bf16x2_rne(fmaf(s, rows_ubyte<3>(lo), b), fmaf(s, rows_ubyte<3>(hi), b));
    return __builtin_bit_cast(bf16x8_t, o);
}

// a's odd 16-lane rows and b's even ones change places (32: a's upper half
// and b's lower half).
__device__ __forceinline__ void swap16(uint32_t &a, uint32_t &b) {
    const u32x2_t r = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_permlane16_swap(a, b, false, false));
    a = r.x, b = r.y;
}
__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b) {
    const u32x2_t r = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_permlane32_swap(a, b, false, false));
    a = r.x, b = r.y;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const void *p, uint64_t bytes) {
    const uint32_t records = bytes < 0xFFFFFFFFull ? static_cast<uint32_t>(bytes) : 0xFFFFFFFFu;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), static_cast<short>(0), static_cast<int>(records),
                                             0x00020000);
}

}  // namespace

// Block L -> its row block and column block. Blocks go round-robin over the 8
// XCDs; the row blocks of one column block stay on one XCD, whose L2 then
// serves their weights once (columns of the last, partial group of 8 are
// dealt in order).
__device__ __forceinline__ void rows_block(uint32_t L, uint32_t row_blocks, uint32_t col_blocks, uint32_t *row,
                                           uint32_t *col) {
    const uint32_t whole = col_blocks / 8 * 8 * row_blocks;
    if (L < whole) {
        const uint32_t g = L / (8 * row_blocks), r = L % (8 * row_blocks);
        *col = g * 8 + r % 8;
        *row = r / 8;
    } else {
        *col = col_blocks / 8 * 8 + (L - whole) / row_blocks;
        *row = (L - whole) % row_blocks;
    }
}

// X buffer bytes of one wavefront (it has two).
template <int RT>
struct RowsCfg {
    static constexpr uint32_t kBuf = RT == 1 ? 4096 : 8192;
    static constexpr uint32_t kXLds = kRWaves * 2 * kBuf;
    static constexpr uint32_t kLds = kXLds + kRWaves * kRSbBytes;
    static constexpr int kSub = static_cast<int>(kBuf) / (RT * 16 * 64);  // MFMA sub-steps (32 values of K) per buffer
    static constexpr int kUnits = 4 / kSub;                              // buffers per 128-value chunk
    static constexpr int kPieces = 4 * kSub;                             // 16-byte pieces per buffered row
    static constexpr int kDma = static_cast<int>(kBuf) / 1024;           // DMA instructions per buffer
    static constexpr int kBatch = kXLds / (kRWaves * 1024);              // accumulator tiles summed per round
    static_assert((kPieces == 16 || kPieces == 8) && kUnits <= 2, "the swizzle, and the waits of a chunk");
};

// y_is_f32: 1 stores the f32 sums, 0 their RNE to bf16.
template <int RT, int CT>
__global__ __launch_bounds__(kRThreads, 2) void q4_gemm_rows_kernel(
    const uint16_t *__restrict__ x, uint32_t x_ld, const uint32_t *__restrict__ wq,
    const uint16_t *__restrict__ scales, const uint16_t *__restrict__ biases, uint32_t m, uint32_t n, uint32_t k,
    void *__restrict__ y, int y_is_f32) {
    using C = RowsCfg<RT>;
    constexpr int kSub = C::kSub, kUnits = C::kUnits, kPieces = C::kPieces, kDma = C::kDma;
    constexpr int kRBatch = C::kBatch;
    extern __shared__ __attribute__((aligned(16))) char rows_smem[];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t c16 = lane & 15, quarter = lane >> 4;
    uint32_t row_block, col_block;
    rows_block(blockIdx.x, (m + RT * 16 - 1) / (RT * 16), (n + CT * 16 - 1) / (CT * 16), &row_block, &col_block);
    const uint32_t m0 = row_block * (RT * 16), n0 = col_block * (CT * 16);
    const uint32_t chunks = k / 128;
    const uint32_t c0 = wave * chunks / kRWaves, c1 = (wave + 1) * chunks / kRWaves;

    char *const xbuf = rows_smem + wave * (2 * C::kBuf);
    char *const sbl = rows_smem + C::kXLds + wave * kRSbBytes;
    // slot of piece p in buffered row r: 16 rows of one fragment read hit
    // all 64 banks once
    auto slot_of = [](uint32_t r, uint32_t p) { return kPieces == 16 ? p ^ (r & 15) : p ^ ((r >> 1) & 7); };
    // DMA instruction d brings 64 / kPieces rows: lane i -> row, slot
    uint32_t xoff[kDma];
#pragma unroll
    for (int d = 0; d < kDma; ++d) {
        const uint32_t r = d * (64 / kPieces) + lane / kPieces, slot = lane % kPieces;
        uint32_t row = m0 + r;
        row = row < m ? row : m - 1;  // rows past m feed outputs that are not stored
        xoff[d] = (row * x_ld + slot_of(r, slot) * 8) * 2;
    }
    uint32_t woff[CT];
#pragma unroll
    for (int t = 0; t < CT; ++t) {
        uint32_t col = n0 + t * 16 + c16;
        col = col < n ? col : 0;
        woff[t] = col * (k / 2) + quarter * 16;
    }
    // Chunks past the wavefront's range are requested through a descriptor
    // of no records: they read as zeros and cost no traffic.
    const uint64_t xbytes = (static_cast<uint64_t>(m - 1) * x_ld + k) * 2, wbytes = static_cast<uint64_t>(n) * k / 2;
    auto dma_x = [&](uint32_t unit, uint32_t buf) {
        const __amdgpu_buffer_rsrc_t rx = rows_rsrc(x, unit < c1 * kUnits ? xbytes : 0);
        const uint32_t so = __builtin_amdgcn_readfirstlane(unit * (kSub * 64));
#pragma unroll
        for (int d = 0; d < kDma; ++d)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rx, (__attribute__((address_space(3))) void *)(xbuf + buf * C::kBuf + d * 1024), 16,
                static_cast<int>(xoff[d]), static_cast<int>(so), 0, 0);
    };
    struct WSet {
        uint4 w[CT];
    };
    auto load_w = [&](WSet &ws, uint32_t c) {
        const __amdgpu_buffer_rsrc_t rw = rows_rsrc(wq, c < c1 ? wbytes : 0);
        const uint32_t so = __builtin_amdgcn_readfirstlane(c * 64);
#pragma unroll
        for (int t = 0; t < CT; ++t)
            ws.w[t] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
                                                    rw, static_cast<int>(woff[t]), static_cast<int>(so), 0));
    };
    // Scales and biases of the wavefront's K range, once, by LDS DMA: slot s
    // holds 8 groups (4 chunks, 16 bytes) of column tile s % CT's 16 columns,
    // scales in the first half of the area, biases in the second; an
    // instruction brings four slots. (As a dword per lane and chunk beside
    // each weight load they took a quarter of the kernel.) Bytes past a table
    // read as zeros.
    auto stage_sb = [&]() {
        const uint64_t sbytes = static_cast<uint64_t>(n) * (k / kGroup) * 2;
        const __amdgpu_buffer_rsrc_t rs = rows_rsrc(scales, sbytes), rb = rows_rsrc(biases, sbytes);
        const uint32_t slots = (c1 - c0 + 3) / 4 * CT;
        for (uint32_t s0 = 0; s0 < slots; s0 += 4) {
            const uint32_t s = s0 + quarter;
            uint32_t col = n0 + s % CT * 16 + c16;
            col = col < n ? col : 0;
            const int off = static_cast<int>((col * (k / kGroup) + 2 * c0 + s / CT * 8) * 2);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rs, (__attribute__((address_space(3))) void *)(sbl + s0 * 256), 16, off, 0, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rb, (__attribute__((address_space(3))) void *)(sbl + kRSbBytes / 2 + s0 * 256), 16, off, 0, 0, 0);
        }
    };

    f32x4_t acc[RT][CT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][t][r] = 0.f;

    // One chunk: X of the next buffer and the next chunk's weights are
    // requested before this one is computed.
    auto chunk = [&](uint32_t c, const WSet &ws, WSet &next) {
        uint4 w[CT];
#pragma unroll
        for (int u = 0; u < kUnits; ++u) {
            const uint32_t buf = kUnits == 1 ? (c - c0) & 1 : u & 1;
            dma_x(c * kUnits + u + 1, buf ^ 1);
            __builtin_amdgcn_sched_barrier(0);
            if (u == 0) load_w(next, c + 1);
            __builtin_amdgcn_sched_barrier(0);
            // this buffer's X has landed: only the requests just made (and,
            // in a chunk's second unit, the next weights) are younger
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kDma + CT) : "memory");
            __builtin_amdgcn_sched_barrier(0);
            if (u == 0) {
#pragma unroll
                for (int t = 0; t < CT; ++t) {
                    w[t] = ws.w[t];
                    swap32(w[t].x, w[t].z);
                    swap32(w[t].y, w[t].w);
                    swap16(w[t].x, w[t].y);
                    swap16(w[t].z, w[t].w);
                }
            }
            const char *const sbc = sbl + (c - c0) / 4 * (CT * 256) + (c - c0) % 4 * 4 + c16 * 16;
#pragma unroll
            for (int s = 0; s < kSub; ++s) {
                const int j = u * kSub + s;  // sub-step of the chunk
                bf16x8_t a[RT];
#pragma unroll
                for (int i = 0; i < RT; ++i)
                    a[i] = *reinterpret_cast<const bf16x8_t *>(
                        xbuf + buf * C::kBuf + (i * 16 + c16) * (kPieces * 16) +
                        slot_of(i * 16 + c16, 4 * s + quarter) * 16);
#pragma unroll
                for (int t = 0; t < CT; ++t) {
                    const char *p = sbc + t * 256 + j / 2 * 2;
                    const float sf = bf(*reinterpret_cast<const uint16_t *>(p));
                    const float bs = bf(*reinterpret_cast<const uint16_t *>(p + kRSbBytes / 2));
                    const bf16x8_t b =
                        rows_dequant8(j == 0 ? w[t].x : j == 1 ? w[t].y : j == 2 ? w[t].z : w[t].w, sf, bs);
#pragma unroll
                    for (int i = 0; i < RT; ++i)
                        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b, acc[i][t], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            // the reads of this buffer are done before it is overwritten
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (c0 < c1) {
        WSet ws, next;
        stage_sb();
        dma_x(c0 * kUnits, 0);
        __builtin_amdgcn_sched_barrier(0);
        load_w(ws, c0);
        __builtin_amdgcn_sched_barrier(0);
        // one body, the weights handed on in registers: a load whose only use
        // lies past a loop exit would be sunk there, out of flight. (Weights
        // three chunks ahead measured no faster: 28.6 against 29.6 us for
        // 32 x 28672 x 4096, 9.4 against 11.0 us for 32 x 6144 x 4096.)
        uint32_t c = c0;
        do {
            chunk(c, ws, next);
            ws = next;
        } while (++c < c1);
    }
    // the last requests have landed before the LDS is reused
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // The partial tiles, kRBatch accumulator tiles a round: every wavefront
    // stores its own, then thread t adds the eight values of an output in K
    // order. Tiles are taken row tile by row tile, so consecutive threads
    // write consecutive columns.
    float *const red = reinterpret_cast<float *>(rows_smem);
    constexpr int kRowsPerRound = kRBatch / CT;  // row tiles a round
    static_assert(kRowsPerRound >= 1, "a round holds whole row tiles");
#pragma unroll
    for (int i0 = 0; i0 < RT; i0 += kRowsPerRound) {
        constexpr int kAll = RT;
        const int rows = kAll - i0 < kRowsPerRound ? kAll - i0 : kRowsPerRound;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kRowsPerRound; ++i)
            if (i0 + i < RT)
#pragma unroll
                for (int t = 0; t < CT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        red[(wave * kRBatch + i * CT + t) * 256 + r * 64 + lane] = acc[i0 + i][t][r];
        __syncthreads();
#pragma unroll 4
        for (uint32_t e = tid; e < static_cast<uint32_t>(rows) * CT * 256; e += kRThreads) {
            const uint32_t col = e % (CT * 16), row = e / (CT * 16);  // row of the round
            const uint32_t tile = (row / 16) * CT + col / 16, r16 = row % 16;
            const float *p = red + tile * 256 + (r16 % 4) * 64 + (r16 / 4) * 16 + col % 16;
            float sum = p[0];
#pragma unroll
            for (int v = 1; v < kRWaves; ++v) sum += p[v * kRBatch * 256];
            const uint32_t gr = m0 + i0 * 16 + row, gc = n0 + col;
            if (gr < m && gc < n) {
                const uint64_t o = static_cast<uint64_t>(gr) * n + gc;
                if (y_is_f32)
                    static_cast<float *>(y)[o] = sum;
                else
                    static_cast<uint16_t *>(y)[o] = rne(sum);
            }
        }
    }
}

template <int RT, int CT>
static void launch_rows(hipStream_t stream, const uint16_t *x, uint32_t x_ld, const uint32_t *wq, const uint16_t *s,
                        const uint16_t *b, uint32_t m, uint32_t n, uint32_t k, void *y, int y_is_f32) {
    static const hipError_t opt_in =
        hipFuncSetAttribute(reinterpret_cast<const void *>(q4_gemm_rows_kernel<RT, CT>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, RowsCfg<RT>::kLds);
    (void)opt_in;
    const uint32_t blocks = (n + CT * 16 - 1) / (CT * 16) * ((m + RT * 16 - 1) / (RT * 16));
    hipLaunchKernelGGL((q4_gemm_rows_kernel<RT, CT>), dim3(blocks), dim3(kRThreads), RowsCfg<RT>::kLds, stream, x,
                       x_ld, wq, s, b, m, n, k, y, y_is_f32);
}

// The column tiles per block that give the least estimated time, and that
// time in us (0 tiles: the kernel does not take the shape). Blocks run in
// rounds of one per CU. A block takes about 2 us to start and finish, 0.24 us
// per 16 rows of X and 1000 of K, and for each column tile 0.48 us per 1000 of
// K plus 0.3 us per 16 rows (its part of the final sums). Within 17% of 117
// measured shapes (33..1024 rows; for instance one round of 64-row blocks, K =
// 4096: 8.8, 11.6, 15.1, 18.2, 21.9, 24.8, 31.3 us for 1..7 tiles).
RowsPlan plan_q4_gemm_rows(uint32_t cus, uint32_t x_ld, const uint16_t *s, const uint16_t *b, uint32_t m, uint32_t n,
                           uint32_t k) {
    RowsPlan plan;
    // whole 128-value chunks; dword-aligned scale/bias pieces; 32-bit offsets
    if (m == 0 || n == 0 || k == 0 || k % 128 != 0) return plan;
    if ((reinterpret_cast<uintptr_t>(s) | reinterpret_cast<uintptr_t>(b)) & 3) return plan;
    if (static_cast<uint64_t>(m) * x_ld * 2 >= (1ull << 32) || static_cast<uint64_t>(n) * k / 2 >= (1ull << 32))
        return plan;
    const uint32_t rt = m <= 16 ? 1 : m <= 32 ? 2 : 4;
    const uint64_t row_blocks = (m + rt * 16 - 1) / (rt * 16), tiles = (n + 15) / 16;
    const uint32_t quads = ((k / 128 + kRWaves - 1) / kRWaves + 3) / 4;
    for (uint32_t ct = 1; ct <= 7; ++ct) {
        if (ct * quads * 512 > kRSbBytes) break;  // the scale/bias slots of a wavefront's K range
        const uint64_t blocks = (tiles + ct - 1) / ct * row_blocks;
        if (blocks > 0x7FFFFFull) continue;
        const double rounds = static_cast<double>((blocks + cus - 1) / cus);
        double us = rounds * (2.0 + 0.24e-3 * rt * k + ct * (0.3 * rt + 0.48e-3 * k));
        if (rt == 4 && ct == 7) us *= 1.07;  // at the register limit
        if (plan.ct == 0 || us < plan.us) plan = {rt, ct, us};
    }
    return plan;
}

void launch_q4_gemm_rows(hipStream_t stream, const RowsPlan &plan, const uint16_t *x, uint32_t x_ld,
                         const uint32_t *wq, const uint16_t *s, const uint16_t *b, uint32_t m, uint32_t n, uint32_t k,
                         void *y, int y_is_f32) {
    switch (plan.rt * 8 + plan.ct) {
#define FH_ROWS(R, C) \
    case R * 8 + C: return launch_rows<R, C>(stream, x, x_ld, wq, s, b, m, n, k, y, y_is_f32);
#define FH_ROWS_ALL(R) \
    FH_ROWS(R, 1) FH_ROWS(R, 2) FH_ROWS(R, 3) FH_ROWS(R, 4) FH_ROWS(R, 5) FH_ROWS(R, 6) FH_ROWS(R, 7)
        FH_ROWS_ALL(1)
        FH_ROWS_ALL(2)
        FH_ROWS_ALL(4)
#undef FH_ROWS_ALL
#undef FH_ROWS
    }
}

}  // namespace fh

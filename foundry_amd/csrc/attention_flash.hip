// Prefill attention in one pass per query tile, with the reference's
// rounding points: the counterpart of scaled_dot_product_attention
// (src/nn/attention.rs:23-60) under the causal mask (src/nn/masking.rs:11-32)
// for head_dim 64 and 128. Scores s_j = RNE(q.k_j) * scale (fp32 dot products,
// bf16 rounding, fp32 scale), M = max_j s_j, S = sum_j exp(s_j - M), probabilities
// p_j = RNE(exp(s_j - M) / S) -- from the row's GLOBAL max and sum, as the
// reference rounds them before P.V -- and out = RNE(sum_j p_j v_j).
//
// Design for CDNA4: block (KV head, tile of 256 / G query rows), 8 wavefronts;
// the tile's (row, head) pairs are the columns of the score tiles, 32 per
// wavefront. (With few tiles, heads of 128 take blocks of 4 wavefronts, and
// heads of 64 split their keys over 2 or 4 wavefronts; a block then holds 128
// or 64 pairs.) The keys are walked twice, 64 or 128 at a time through LDS:
//   pass 1: S^T = K Q^T on the matrix cores (v_mfma_f32_32x32x16_bf16, the
//     keys as A rows, the pairs' q as B columns held in registers for the
//     whole block), so a lane holds 16 keys of ONE pair: the running max and
//     sum of exp need no cross-lane work until the two half-wavefronts that
//     share a pair combine them once, at the end;
//   pass 2: the same scores again, p_j rounded from the final M and S, and
//     P.V on the matrix cores: the lane's 16 probabilities of a 32-key tile
//     are already an A fragment pair (keys in the order the score layout
//     gives them), and V is staged transposed in LDS with its keys in that
//     same order, so each B fragment is one 16-byte read.
// No scores or statistics leave the CU (the two-kernel path writes both
// through a workspace), and every key and value is read from L2 once per
// block. What bounds it is VALU issue: about 21 instructions per score, of
// which a wavefront issues one per 8 clocks and a SIMD one per 4.6. Every sum
// runs in a fixed order, so results do not change from run to run.
#include <type_traits>

#include "decoder_common.hpp"

namespace fh {

namespace {

constexpr int kFlKeys = 64;  // keys per LDS block

// Shape of a block: head size, wavefronts W, and over how many of them KS the
// keys of a (row, head) pair are split (1, 2 or 4).
template <int HD, int W, int KS>
struct FlCfg {
    static constexpr int kThreads = 64 * W;
    static constexpr int kPairGroups = W / KS;             // wavefronts of 32 pairs each
    static constexpr uint32_t kPairs = 32 * kPairGroups;   // of the block
    static constexpr uint32_t kParts = 8 / W;              // blocks that share a query tile
    static constexpr int kBlocks = KS == 1 ? 1 : 2;        // LDS blocks of 64 keys per trip
    static constexpr uint32_t kKeys = kFlKeys * kBlocks;   // keys per trip
    static constexpr int kTiles = KS == 4 ? 1 : 2;         // 32-key tiles a wavefront takes of them
    static constexpr uint32_t kBuf = kKeys * HD;           // bf16 per K or V buffer (two of each)
    static constexpr uint32_t kLds = 4 * kBuf * 2;         // bytes
};

typedef __attribute__((ext_vector_type(8))) __bf16 fl_bf16x8_t;
typedef __attribute__((ext_vector_type(16))) float fl_f32x16_t;

__device__ __forceinline__ fl_f32x16_t fl_mfma(const uint4 a, const uint4 b, const fl_f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(fl_bf16x8_t, a), __builtin_bit_cast(fl_bf16x8_t, b),
                                                   c, 0, 0, 0);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t fl_rsrc(const void *p, uint64_t bytes) {
    const uint32_t records = bytes < 0xFFFFFFFFull ? static_cast<uint32_t>(bytes) : 0xFFFFFFFFu;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), static_cast<short>(0), static_cast<int>(records),
                                             0x00020000);
}

// Slot of key k (0..63 of a block) in a V^T row: within each 16-key group,
// keys 0-3 and 8-11 (the first half-wavefront's keys of an MFMA k step) fill
// slots 0-7, keys 4-7 and 12-15 slots 8-15.
__device__ __forceinline__ uint32_t fl_slot(uint32_t k) {
    const uint32_t o = k & 15u;
    return (k & ~15u) + 8u * ((o >> 2) & 1u) + (o & 3u) + 4u * (o >> 3);
}

// exp of the softmax arguments, and each probability from it and the sum.
// The reference compiles its Metal kernels with the default options
// (src/metal/mod.rs:109-128: no MTLCompileOptions), under which Metal's fast
// math is on: its exp (unary.metal:6) and divide (binary.metal:14) are not
// the correctly rounded functions. Here exp(s - m) is v_exp_f32 of one fma,
// b * (scale log2 e) - mb * (scale log2 e) for s = b * scale (b = RNE(q.k))
// and m = mb * scale, and p = e * (1 / S): the same class of approximation.
// With expf of s - m and a true division the one-pass kernel takes 1.8x as
// long (the VALU work per score bounds it). FH_FLASH_EXP2=0 / FH_FLASH_RCP=0
// select those.
#ifndef FH_FLASH_EXP2
#define FH_FLASH_EXP2 1
#endif
#ifndef FH_FLASH_RCP
#define FH_FLASH_RCP 1
#endif
// exp(b * scale - mb * scale) as ex(b, ex.base(mb)); b may be -inf, mb
// is finite
struct FlExp {
    float scale, c1;  // c1 = scale * log2(e)
    __device__ float base(float mb) const {
#if FH_FLASH_EXP2
        return -(mb * c1);
#else
        return __fmul_rn(mb, scale);
#endif
    }
    __device__ float operator()(float b, float base_) const {
#if FH_FLASH_EXP2
        return __builtin_amdgcn_exp2f(fmaf(b, c1, base_));
#else
        return expf(__fmul_rn(b, scale) - base_);
#endif
    }
};

}  // namespace

// Block (KV head, sequence, query tile): rows r0 .. r0 + QT - 1 (QT = pairs of
// the block / G) of sequence blockIdx.y (`rows` rows each, its cache seq_cache
// elements after the previous one's; K tiled in groups of 16 keys, k_tile; V
// [max_len][HD]) over its cache. positions[r]: the row's position; it attends
// keys 0 .. min(pos, max_len - 1). Tiles go out last first: a prompt's later
// rows attend more keys, and the longest blocks then start first.
// With W = 4 a block holds half of the pairs of a 256-pair tile. It walks the
// whole tile's keys, so a pair's sums are those of the block of 8: a running
// sum is rescaled at every trip, also past the pair's last key, and that can
// move it by an ulp.
// With KS > 1 wavefront w holds pairs 32 (w % (W / KS)) .. + 31 and every KS-th
// run of 64 (KS = 4: 32) keys; the splits' statistics, and at the end their
// sums of P.V, meet in LDS and are added in split order. Two blocks share a CU
// where their registers allow it (heads of 64, 128 of them a lane: 2048 rows
// after 1024 108 us, 124 at 130 registers).
template <int HD, int G, int W, int KS>
__global__ __launch_bounds__(64 * W, HD == 64 && KS > 1 ? 4 : 2) void attn_flash_kernel(
    const uint16_t *__restrict__ q, const uint32_t *__restrict__ positions, uint32_t rows,
    const uint16_t *__restrict__ k_cache, const uint16_t *__restrict__ v_cache, uint64_t seq_cache, uint32_t n_heads,
    uint32_t max_len, float scale, uint16_t *__restrict__ out) {
    using C = FlCfg<HD, W, KS>;
    constexpr uint32_t PARTS = C::kParts;          // blocks per query tile
    constexpr uint32_t QT = C::kPairs * PARTS / G;  // query rows per tile
    constexpr uint32_t LIVE = QT * G;               // (row, head) pairs of the tile
    constexpr int QS = HD / 16;             // MFMA k steps of a score
    constexpr int DT = HD / 32;             // 32-dim tiles of the output
    constexpr uint32_t PP = HD / 8;         // 16-byte pieces per key
    // K buffers: [key][PP pieces of 8 dims], piece slot s of key k holding
    // piece s ^ swz(k); V^T buffers: blocks of [dim][64 key slots], 16-byte
    // piece slot s of dim d holding piece s ^ ((d / 2) % 8). Both are
    // conflict-free for the fragment reads below.
    extern __shared__ __align__(16) uint16_t fl_smem[];
    // set when V of a key that not every row attends is inf or NaN: such a
    // value is staged as 0, since its probability of 0 would make the other
    // rows' sums NaN, and added for the rows that do attend it at the end
    __shared__ uint32_t v_special;
    uint16_t *const kls = fl_smem, *const vls = fl_smem + 2 * C::kBuf;
    auto swz = [](uint32_t k) { return HD == 128 ? k & 15u : (k >> 1) & 7u; };
    // the wavefronts' longest contexts, then the splits' statistics: read
    // before V^T buffer 1 is first written
    uint32_t *const wmax = reinterpret_cast<uint32_t *>(vls + C::kBuf);
    const uint32_t tid = threadIdx.x, lane = tid & 63, h = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t pg = wave % C::kPairGroups, split = wave / C::kPairGroups;
    // this wavefront's keys of a trip: LDS block and first 32-key tile in it
    const uint32_t kblk = KS == 4 ? split / 2 : split, t0 = KS == 4 ? split % 2 : 0;
    const uint32_t order = gridDim.z - 1 - blockIdx.z, p0 = order % PARTS * C::kPairs;
    const uint32_t kvh = blockIdx.x, sq = blockIdx.y, r0 = order / PARTS * QT, h0 = kvh * G;
    if (r0 + p0 / G >= rows) return;  // no live pair (uniform over the block)
    {
        const uint64_t rows0 = static_cast<uint64_t>(sq) * rows;  // the sequence's first row
        q += rows0 * n_heads * HD;
        out += rows0 * n_heads * HD;
        positions += rows0;
        k_cache += sq * seq_cache;
        v_cache += sq * seq_cache;
    }
    const uint16_t *const kc = k_cache + static_cast<uint64_t>(kvh) * max_len * HD;
    const uint16_t *const vc = v_cache + static_cast<uint64_t>(kvh) * max_len * HD;

    // this lane's pair: column l % 32 of its wavefront's score tiles
    const uint32_t pb = pg * 32 + (lane & 31), p = p0 + pb;  // in the block, in the tile
    const bool alive = p < LIVE && r0 + p / G < rows;
    const uint32_t prow = alive ? r0 + p / G : 0, phead = h0 + (alive ? p % G : 0);
    const uint32_t pos = alive ? positions[prow] : 0u;
    const uint32_t ctx = alive ? (pos < max_len ? pos + 1 : max_len) : 0u;
    if (tid == 0) v_special = 0;
    // the tile's longest and the block's shortest live contexts: key blocks
    // below the shortest need no mask
    {
        uint32_t most = ctx;
        if constexpr (PARTS > 1) {  // the other half's pair
            const uint32_t o = (p + C::kPairs) % (PARTS * C::kPairs);
            const uint32_t orow = r0 + o / G;
            if (o < LIVE && orow < rows) {
                const uint32_t opos = positions[orow];
                const uint32_t octx = opos < max_len ? opos + 1 : max_len;
                most = octx > most ? octx : most;
            }
        }
        const float mx = wave_max(static_cast<float>(most));
        const float mn = -wave_max(alive ? -static_cast<float>(ctx) : -static_cast<float>(max_len));
        if (lane == 0) wmax[wave] = static_cast<uint32_t>(mx), wmax[W + wave] = static_cast<uint32_t>(mn);
    }
    // q of the pair as B fragments: dims 16 s + 8 h .. + 7
    uint4 qf[QS];
    {
        const uint16_t *qp = q + (static_cast<uint64_t>(prow) * n_heads + phead) * HD + 8 * h;
#pragma unroll
        for (int s = 0; s < QS; ++s) {
            const uint4 v = *reinterpret_cast<const uint4 *>(qp + 16 * s);
            qf[s] = alive ? v : make_uint4(0u, 0u, 0u, 0u);
        }
    }
    __syncthreads();
    uint32_t kmax = 0, kmin = max_len;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        kmax = wmax[w] > kmax ? wmax[w] : kmax;
        kmin = wmax[W + w] < kmin ? wmax[W + w] : kmin;
    }
    const uint32_t trips = (kmax + C::kKeys - 1) / C::kKeys;

    // trip it's keys into LDS by DMA: wavefront w brings kKeys / W of them in
    // 1 KiB instructions (64 / PP keys x PP slots); keys past the block's
    // longest context read key kmax - 1 (valid, never used)
    const __amdgpu_buffer_rsrc_t rk = fl_rsrc(kc, static_cast<uint64_t>(max_len) * HD * 2);
    constexpr uint32_t kPerWave = C::kKeys / W, kPerInst = 64 / PP;
    auto stage_k = [&](uint32_t it, uint32_t buf) {
#pragma unroll
        for (uint32_t c = 0; c < kPerWave / kPerInst; ++c) {
            const uint32_t k0 = wave * kPerWave + c * kPerInst;
            const uint32_t kl = k0 + lane / PP;  // key within the trip
            uint32_t key = it * C::kKeys + kl;
            key = key < kmax ? key : kmax - 1;
            const uint32_t piece = (lane % PP) ^ swz(kl);
            const uint32_t off = static_cast<uint32_t>(k_offset(key, 8 * piece, max_len, HD)) * 2;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rk, (__attribute__((address_space(3))) void *)(kls + buf * C::kBuf + k0 * HD), 16,
                static_cast<int>(off), 0, 0, 0);
        }
    };
    // trip it's V: item (key pair i, dim piece c) loads keys 2 i, 2 i + 1 of
    // dims 8 c .. 8 c + 7, then writes dword (v[2i][d], v[2i+1][d]) of each
    // dim d to V^T
    constexpr uint32_t kVPairs = C::kKeys / 2, kVItems = kVPairs * PP;
    constexpr int kVRounds = kVItems > C::kThreads ? kVItems / C::kThreads : 1;
    auto load_v = [&](uint32_t it, uint4 (&v)[kVRounds][2]) {
#pragma unroll
        for (int r = 0; r < kVRounds; ++r) {
            const uint32_t item = (tid + r * C::kThreads) % kVItems, i = item % kVPairs, c = item / kVPairs;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                uint32_t key = it * C::kKeys + 2 * i + e;
                key = key < kmax ? key : kmax - 1;
                v[r][e] = *reinterpret_cast<const uint4 *>(vc + static_cast<uint64_t>(key) * HD + 8 * c);
            }
        }
    };
    // masked: some row does not attend all of the trip's keys
    auto store_v = [&](uint4 (&v)[kVRounds][2], uint32_t buf, bool masked) {
        if (kVItems < C::kThreads && tid >= kVItems) return;
        if (masked) {
#pragma unroll
            for (int r = 0; r < kVRounds; ++r) {
                const bool x = clear_specials(v[r][0]), y = clear_specials(v[r][1]);
                if (x || y) v_special = 1;
            }
        }
#pragma unroll
        for (int r = 0; r < kVRounds; ++r) {
            const uint32_t item = tid + r * C::kThreads, i = item % kVPairs, c = item / kVPairs;
            uint16_t *const blk = vls + buf * C::kBuf + i / 32 * (kFlKeys * HD);
            const uint32_t slot = fl_slot(2 * (i % 32));  // even; key 2 i + 1 is the next slot
            const uint32_t a[4] = {v[r][0].x, v[r][0].y, v[r][0].z, v[r][0].w};
            const uint32_t b[4] = {v[r][1].x, v[r][1].y, v[r][1].z, v[r][1].w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t d = 8 * c + e;
                const uint32_t lo = (a[e / 2] >> (16 * (e % 2))) & 0xFFFFu, hi = (b[e / 2] >> (16 * (e % 2))) & 0xFFFFu;
                const uint32_t at = d * kFlKeys + (((slot >> 3) ^ ((d >> 1) & 7u)) << 3) + (slot & 7u);
                *reinterpret_cast<uint32_t *>(blk + at) = lo | (hi << 16);
            }
        }
    };
    // S^T of 32-key tile t of this wavefront's block of a buffer: rows = keys
    // 32 t + 8 (r / 4) + 4 h + r % 4, column = this lane's pair
    auto scores = [&](uint32_t buf, uint32_t t) {
        const uint32_t kl = 32 * t + (lane & 31);
        const uint16_t *kr = kls + buf * C::kBuf + (kblk * kFlKeys + kl) * HD;
        fl_f32x16_t d;
#pragma unroll
        for (int r = 0; r < 16; ++r) d[r] = 0.f;
#pragma unroll
        for (int s = 0; s < QS; ++s) {
            const uint4 a = *reinterpret_cast<const uint4 *>(kr + (((2 * s + h) ^ swz(kl)) << 3));
            d = fl_mfma(a, qf[s], d);
        }
        return d;
    };
    // b_j = RNE(q.k_j) (the score is s_j = b_j * scale; the scale is applied
    // inside the exp argument, and the max over b is the max over s), or -inf
    // past the pair's context (MASK: the block reaches past some live pair's
    // context)
    const FlExp ex{scale, scale * 1.44269504088896341f};
    auto score_of = [&](const fl_f32x16_t &d, uint32_t it, uint32_t t, int r, auto mask) {
        const float sv = bf(rne(d[r]));
        if constexpr (decltype(mask)::value) {
            const uint32_t j = it * C::kKeys + kblk * kFlKeys + 32 * t + 8 * (r / 4) + 4 * h + (r % 4);
            return j < ctx ? sv : -INFINITY;
        }
        return sv;
    };
    using Masked = std::integral_constant<bool, true>;
    using Unmasked = std::integral_constant<bool, false>;

    // Pass 1: running (max of b, sum of exp(s - m)) over this lane's keys of the pair
    float m = -INFINITY, l = 0.f;
    stage_k(0, 0);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    __syncthreads();
    for (uint32_t it = 0; it < trips; ++it) {
        const uint32_t buf = it & 1;
        if (it + 1 < trips) stage_k(it + 1, buf ^ 1);
        auto stats = [&](auto mask) {
#pragma unroll
            for (int tt = 0; tt < C::kTiles; ++tt) {
                const uint32_t t = t0 + tt;
                const fl_f32x16_t d = scores(buf, t);
                float sv[16], mt = -INFINITY;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    sv[r] = score_of(d, it, t, r, mask);
                    mt = fmaxf(mt, sv[r]);
                }
                const float mn = fmaxf(m, mt);
                if (mn != -INFINITY) {
                    const float o = ex.base(mn);
                    float sum = 0.f;
#pragma unroll
                    for (int r = 0; r < 16; ++r) sum += ex(sv[r], o);
                    l = l * ex(m, o) + sum;
                    m = mn;
                }
            }
        };
        if ((it + 1) * C::kKeys <= kmin)
            stats(Unmasked{});
        else
            stats(Masked{});
        __builtin_amdgcn_s_waitcnt(0x0f70);  // the next block's DMA has landed
        __syncthreads();
    }
    // two statistics of disjoint keys of a pair, the first one's keys first
    auto meet = [&](float m0, float l0, float m1, float l1, float *mo, float *lo) {
        const float mm = fmaxf(m0, m1);
        const float o = mm == -INFINITY ? 0.f : ex.base(mm);
        *mo = mm;
        *lo = (m0 == -INFINITY ? 0.f : l0 * ex(m0, o)) + (m1 == -INFINITY ? 0.f : l1 * ex(m1, o));
    };
    // the pair's two halves (lanes l and l ^ 32), the h = 0 half first, then
    // its splits in order
    float M, S;
    {
        const float mo = __shfl_xor(m, 32, 64), lo = __shfl_xor(l, 32, 64);
        meet(h ? mo : m, h ? lo : l, h ? m : mo, h ? l : lo, &M, &S);
        if constexpr (KS > 1) {
            float2 *const st = reinterpret_cast<float2 *>(wmax);  // [split][pair]
            if (h == 0) st[split * C::kPairs + pb] = make_float2(M, S);
            __syncthreads();
            float2 v = st[pb];
            M = v.x, S = v.y;
#pragma unroll
            for (int k = 1; k < KS; ++k) {
                v = st[k * C::kPairs + pb];
                meet(M, S, v.x, v.y, &M, &S);
            }
        }
        // every score -inf: exp(-inf + inf) is NaN for a live pair; a dead lane,
        // with no key, gets exp(-inf) = 0 everywhere
        if (M == -INFINITY) S = alive ? NAN : 1.f;
    }
    const float oM = M == -INFINITY ? 0.f : ex.base(M);
#if FH_FLASH_RCP
    const float rS = 1.f / S;
#endif

    // Pass 2: p_j = RNE(exp(s_j - M) / S) (masked keys: exp(-inf) = 0), acc +=
    // P V over DT tiles of 32 dims
    fl_f32x16_t acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[dt][r] = 0.f;
    {
        uint4 vr[kVRounds][2];
        stage_k(0, 0);
        load_v(0, vr);
        store_v(vr, 0, C::kKeys > kmin);
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    fl_f32x16_t dsc;  // the current score tile
    for (uint32_t it = 0; it < trips; ++it) {
        const uint32_t buf = it & 1;
        uint4 vr[kVRounds][2];
        const bool next = it + 1 < trips;
        if (next) {
            stage_k(it + 1, buf ^ 1);
            load_v(it + 1, vr);
        }
        auto probs = [&](uint32_t t, uint32_t (&pw)[8], auto mask) {
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const fl_f32x16_t &d = dsc;
                const float s0 = score_of(d, it, t, r, mask), s1 = score_of(d, it, t, r + 1, mask);
#if FH_FLASH_RCP
                const float p0 = ex(s0, oM) * rS, p1 = ex(s1, oM) * rS;
#else
                const float p0 = ex(s0, oM) / S, p1 = ex(s1, oM) / S;
#endif
                pw[r / 2] = f32x2_to_bf16x2_rne(p0, p1);
            }
        };
        const bool full = (it + 1) * C::kKeys <= kmin;
#pragma unroll
        for (int tt = 0; tt < C::kTiles; ++tt) {
            const uint32_t t = t0 + tt;
            dsc = scores(buf, t);
            uint32_t pw[8];  // probabilities as bf16 pairs, in register order
            if (full)
                probs(t, pw, Unmasked{});
            else
                probs(t, pw, Masked{});
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const uint4 a = make_uint4(pw[4 * ks], pw[4 * ks + 1], pw[4 * ks + 2], pw[4 * ks + 3]);
                const uint32_t piece = 2 * (2 * t + ks) + h;  // slots 16 (2 t + ks) + 8 h .. + 7
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    const uint32_t dd = 32 * dt + (lane & 31);
                    const uint4 b = *reinterpret_cast<const uint4 *>(
                        vls + buf * C::kBuf + kblk * (kFlKeys * HD) + dd * kFlKeys +
                        ((piece ^ ((dd >> 1) & 7u)) << 3));
                    acc[dt] = fl_mfma(a, b, acc[dt]);
                }
            }
        }
        if (next) store_v(vr, buf ^ 1, (it + 2) * C::kKeys > kmin);  // buffer buf ^ 1 was last read before the previous barrier
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();
    }

    // the splits' sums, in split order (the last trip's barrier is behind)
    if constexpr (KS > 1) {
        float *const red = reinterpret_cast<float *>(fl_smem);  // [split - 1][pair group][dt][r][lane]
        constexpr uint32_t kWaveSums = DT * 16 * 64;
        if (split > 0) {
            float *const mine = red + ((split - 1) * C::kPairGroups + pg) * kWaveSums + lane;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) mine[(dt * 16 + r) * 64] = acc[dt][r];
        }
        __syncthreads();
#pragma unroll
        for (int k = 1; k < KS; ++k) {
            const float *const part = red + ((k - 1) * C::kPairGroups + pg) * kWaveSums + lane;
            if (split == 0) {
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[dt][r] += part[(dt * 16 + r) * 64];
            }
        }
    }

    // out[row][head][dim]: lane holds dim 32 dt + l % 32 of pairs 8 (r / 4) + 4 h + r % 4
    if (split == 0) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint32_t pp = p0 + pg * 32 + 8 * (r / 4) + 4 * h + (r % 4);
            if (pp >= LIVE || r0 + pp / G >= rows) continue;
            uint16_t *orow = out + (static_cast<uint64_t>(r0 + pp / G) * n_heads + h0 + pp % G) * HD + (lane & 31);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) orow[32 * dt] = rne(acc[dt][r]);
        }
    }
    if (!v_special) return;  // uniform: last written before a barrier of the loop

    // inf and NaN of V in the trips that some row attends in part: p v for
    // the rows that attend the key, p from the score again
    __syncthreads();  // the outputs are written, the sums above read
    float2 *const st = reinterpret_cast<float2 *>(fl_smem);
    if (split == 0 && h == 0) st[pb] = make_float2(oM, S);
    __syncthreads();
    for (uint32_t o = tid; o < C::kPairs * HD; o += C::kThreads) {
        const uint32_t pi = o / HD, pp = p0 + pi, d = o % HD, row = r0 + pp / G;
        if (pp >= LIVE || row >= rows) continue;
        const uint64_t at = (static_cast<uint64_t>(row) * n_heads + h0 + pp % G) * HD;
        const uint32_t rpos = positions[row], rctx = rpos < max_len ? rpos + 1 : max_len;
        float sum = 0.f;
        bool any = false;
        for (uint32_t j = kmin / C::kKeys * C::kKeys; j < rctx; ++j) {
            const uint32_t v = vc[static_cast<uint64_t>(j) * HD + d];
            if (!bf16_specials(v)) continue;
            float qk = 0.f;
            for (uint32_t e = 0; e < HD; ++e) qk = fmaf(bf(q[at + e]), bf(kc[k_offset(j, e, max_len, HD)]), qk);
            sum += bf(rne(ex(bf(rne(qk)), st[pi].x) / st[pi].y)) * bf(static_cast<uint16_t>(v));
            any = true;
        }
        if (any) out[at + d] = rne(bf(out[at + d]) + sum);
    }
}

// The block shape the one-pass kernel takes for `batch` sequences of `rows`
// prompt rows (waves = 0: it does not take them). Whether it does, and over how
// many wavefronts a pair's keys are split, goes by one sequence alone, so a
// batch gives what a call per sequence gives.
struct FlPlan {
    uint32_t waves = 0, ks = 1;
};

static FlPlan flash_plan(uint32_t cus, uint32_t batch, uint32_t rows, uint32_t n_heads, uint32_t n_kv,
                         uint32_t head_dim, uint32_t max_len, float scale) {
    FlPlan p;
    // the maximum is taken before the scale, which has to be positive; contexts
    // are compared as floats and keys addressed by 32-bit byte offsets
    if (!(scale > 0.f && scale * 1.5f < INFINITY) || max_len >= 1u << 24) return p;
    if ((head_dim != 64 && head_dim != 128) || n_kv == 0 || n_heads % n_kv != 0) return p;
    const uint32_t g = n_heads / n_kv;
    if (g < 1 || g > 8) return p;
    auto tiles = [&](uint32_t pairs) { return (static_cast<uint64_t>(rows) + pairs / g - 1) / (pairs / g); };
    const uint64_t blocks = tiles(256) * n_kv;  // of one sequence, in blocks of 256 pairs
    if (head_dim == 128) {
        // Query tiles for half the CUs. Below that the two-kernel path: 512
        // rows of 24 heads, 8 KV heads, take 36.1 us there and 34.8 here. (With
        // the keys split over wavefronts they take 24.7, but then round the
        // sums otherwise, and a prompt's logits move by 3.5e-4.)
        if (2 * blocks < cus || tiles(256) > 65535) return p;
        // Blocks of 4 wavefronts where 8 would not make two rounds of CUs: two
        // share a CU, so one with few keys can run beside one with many. 8 KV
        // heads, in blocks of 8 and 4: 2048 rows of 32 heads 126.8 / 105.9 us
        // (after 1024 189.7 / 165.0), 1024 rows 64.8 / 50.2.
        p.waves = blocks * batch >= 2ull * cus ? 8 : 4;
        return p;
    }
    // Query tiles for half the CUs, or a prompt of at least 16 rows that is not
    // short against the cache, since a block walks all of its rows' keys.
    // Measured against the two-kernel path, 32 heads, 8 KV heads: 24 rows after
    // 300 keys 10.9 / 14.9 us, 2048 after 1024 108 / 603.8. The keys over 2
    // wavefronts where that gives more than a block per CU, 4 otherwise, none
    // from two rounds on.
    if (2 * blocks < cus && (rows < 16 || max_len > 16ull * rows)) return p;
    p.ks = blocks >= 2ull * cus ? 1 : tiles(128) * n_kv > cus ? 2 : 4;
    p.waves = tiles(256 / p.ks) > 65535 ? 0 : 8;
    return p;
}

// Whether fh_attention takes the one-pass kernel for `rows` prompt rows of a
// sequence.
bool attention_flash_applies(uint32_t cus, uint32_t rows, uint32_t n_heads, uint32_t n_kv, uint32_t head_dim,
                             uint32_t max_len, float scale) {
    return flash_plan(cus, 1, rows, n_heads, n_kv, head_dim, max_len, scale).waves != 0;
}

template <int HD, int G, int W, int KS>
static void launch_flash(hipStream_t stream, const uint16_t *q, const uint32_t *positions, uint32_t rows,
                         const uint16_t *k_cache, const uint16_t *v_cache, uint32_t n_heads, uint32_t n_kv,
                         uint32_t max_len, float scale, uint16_t *out, uint32_t batch, uint64_t seq_cache) {
    using C = FlCfg<HD, W, KS>;
    static const hipError_t opt_in =
        hipFuncSetAttribute(reinterpret_cast<const void *>(attn_flash_kernel<HD, G, W, KS>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, C::kLds);
    (void)opt_in;
    constexpr uint32_t QT = C::kPairs * C::kParts / G;
    hipLaunchKernelGGL((attn_flash_kernel<HD, G, W, KS>), dim3(n_kv, batch, (rows + QT - 1) / QT * C::kParts),
                       dim3(C::kThreads), C::kLds, stream, q, positions, rows, k_cache, v_cache, seq_cache, n_heads,
                       max_len, scale, out);
}

// Launches the one-pass kernel over `batch` sequences of `rows` rows (q, out
// and positions consecutive per sequence, caches seq_cache elements apart)
// when attention_flash_applies; returns false otherwise (the caller takes the
// two-kernel path). The outputs are those of a launch per sequence.
bool launch_attention_flash(hipStream_t stream, uint32_t cus, const uint16_t *q, const uint32_t *positions,
                            uint32_t rows, const uint16_t *k_cache, const uint16_t *v_cache, uint32_t n_heads,
                            uint32_t n_kv, uint32_t head_dim, uint32_t max_len, float scale, uint16_t *out,
                            uint32_t batch, uint64_t seq_cache) {
    if (batch == 0 || batch > 65535) return false;
    const FlPlan p = flash_plan(cus, batch, rows, n_heads, n_kv, head_dim, max_len, scale);
    if (p.waves == 0) return false;
    const uint32_t g = n_heads / n_kv;
#define FH_FLASH(HH, GG, WW, SS)                                                                                  \
    if (head_dim == HH && g == GG && p.waves == WW && p.ks == SS) {                                               \
        launch_flash<HH, GG, WW, SS>(stream, q, positions, rows, k_cache, v_cache, n_heads, n_kv, max_len, scale, \
                                     out, batch, seq_cache);                                                      \
        return true;                                                                                              \
    }
#define FH_FLASH_G(GG)                                                       \
    FH_FLASH(64, GG, 8, 1) FH_FLASH(64, GG, 8, 2) FH_FLASH(64, GG, 8, 4)     \
    FH_FLASH(128, GG, 8, 1) FH_FLASH(128, GG, 4, 1)
    FH_FLASH_G(1)
    FH_FLASH_G(2)
    FH_FLASH_G(3)
    FH_FLASH_G(4)
    FH_FLASH_G(5)
    FH_FLASH_G(6)
    FH_FLASH_G(7)
    FH_FLASH_G(8)
#undef FH_FLASH_G
#undef FH_FLASH
    return false;
}

}  // namespace fh

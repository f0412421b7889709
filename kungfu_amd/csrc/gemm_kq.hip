// Tile GEMM on native q4_K, q5_K and q6_K bytes, from a few rows to prefill, one matrix or the grouped experts:
// y[m][n] = sum over super-blocks b of dx[m][b] * (d[n][b] * S_b[m][n] - dmin[n][b] * mins_b[m][n]) (+ bias[n] + res[m][n]),
// with S_b the reference's exact super-block integer:
//   * q4_K, q5_K (crates/kf-quant/src/types/q4_k.rs:10-58, q5_k.rs): S_b = sum_g sc_g I_g over the eight 32-column groups,
//     I_g the int32 dot of the group's values with the int8 activations; mins_b = sum_g m_g bsum_g;
//   * q6_K (crates/kf-quant/src/types/q6_k.rs): S_b = sum_s sc_s (dot_s - 32 bsum_s) over the sixteen 16-column
//     sub-blocks with int8 scales, formed as sum_s sc_s dot'_s with the operand q - 32; no mins term.
// It replaces the reference's unpack + KF8 GEMM for these types (crates/kf-backend-cuda/src/kernels/quant.cuh:585-601,
// kf8.cu:116-369, 400-416), reading the native bytes directly.
//
// Arithmetic: the product scale x value of every weight, v, is exact in two int8 planes, v = lo + (hi << SHIFT): q4_K's
// nibble times the 6-bit scale's two 3-bit halves, q5_K's and q6_K's 16-bit product split into its signed low byte and
// the rest. Two v_mfma_i32_32x32x32_i8 chains a 32 x 32 tile run through the super-block, so S_b needs no work per group;
// mins_b is one exact v_mfma_f32_32x32x16_f16 against quant_act's split sums, and the float rescale runs once per
// super-block and output (five VALU instructions). A form with one MFMA a group and the scales applied to its results by
// multiply-adds spent 2-3 times the vector work of this one on q5_K and q6_K.
//
// Schedule: eight waves (two a SIMD), one block a CU, block tile 32 TM x 256, each wave a column of TM 32 x 32 tiles, so a
// weight operand is expanded once for TM tiles. The operands of a whole super-block stay in registers (64) and the tiles
// run one after another, eight group steps each: a step's two MFMAs go with an eighth of the previous tile's rescale
// and, in the last tile, with the expansion of the next super-block's operands, so no phase of a wave is without MFMAs
// and the two waves of a SIMD need no offset. What bounds it at TM = 4 (2048 rows of q4_K): MFMA busy 47-53% and
// VALU issue 56-61% of the cycles, which overlap only in part, and LDS and DMA waits (29-33% of a wave's cycles). Choices that measured (2048 rows, us): reloads of spilled registers
// in the K loop wait for every load in flight (446 -> 295, 4096 -> 14336 q4_K); the loads of a super-block spread over
// the steps instead of all at its start, where eight waves queue them behind each other, and each step's LDS
// reads one step ahead (267 -> 241, 14336 -> 4096 q4_K).
// Weights land by DMA in each wave's own LDS buffers ([row 32][WROW]; q6_K: the 16-byte aligned window around the 210-byte
// block, whose rows may start at any even byte, so every width of whole super-blocks is taken), activations in buffers all
// waves share ([tile][row 32][256] with the 16-byte chunk swizzle c ^ (row % 16)); every wait is explicit. Blocks run in
// XCD order, so the blocks in flight on an XCD share their weight tiles in its L2.
// Measured, us, before (the one-MFMA form on q5_K / q6_K, a 128 x 256 tile kernel without the interleaved rescale on q4_K, the
// per-lane product on q6_K rows off 16 bytes) and now, 4096 -> 14336 / 14336 -> 4096: 2048 rows q4_K 291 / 266 -> 285 / 245, q5_K
// 348 / 322 -> 316 / 278, q6_K 629 / 609 -> 338 / 291; 128 rows q4_K 36 / 48 -> 33 / 32, q5_K 38 / 51 -> 36 / 34, q6_K
// 58 / 86 -> 38 / 37; 63 rows of q6_K 2816 -> 7052 273 -> 22. On 64-row tiles of q5_K the expansion of two planes costs more than the
// one-MFMA form did: 378 rows of 1792 -> 10584 32.7 -> 36.8 with the quantization, 510 of 3072 -> 8192 46.7 -> 52.5.
#include "kf_knobs.h"
#include "kf_blocks.h"
#include "kf_device.h"
#include "kf_host.h"

#include <algorithm>
#include <cmath>
#include <optional>
#include <type_traits>

// The K loop relies on gfx950's LDS DMA and vmcnt order: build for gfx950 only.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "the DMA waits assume gfx950"
#endif

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));

constexpr int KQ_WAVES = 8, KQ_THREADS = 64 * KQ_WAVES;
constexpr int KQ_BN = 32 * KQ_WAVES;  // 256: one 32-column tile per wave
constexpr int KQ_LDS = 160 * 1024;
constexpr int KQ_EPI = 256;  // LDS for the parked state
// Cost model of a launch (MI355X, us; least squares over 4-2048 rows at 2048 -> 6144, 4096 -> 4096, 4096 -> 14336 and
// 14336 -> 4096, rms 3-8%): 1.8 for the launch, KQ_ROUND_US a round of the CUs (a block's first loads and its stores), the
// super-blocks of the rounds, and the partial tiles' way through memory where the tail is split (per CU's worth of them).
// The tile height is the cheapest by it: few rows take short tiles (32 rows of 14336 -> 4096 q4_K: 19 / 22 / 29 us with 1 / 2 / 4
// tiles), 2048 tall ones (373 / 292 / 239).
constexpr double KQ_ROUND_US[3] = {4.2, 4.8, 5.6};                                               // [1, 2, 4 tiles]
constexpr double KQ_SB_US[3][3] = {{1.60, 2.44, 4.01}, {2.46, 3.23, 4.66}, {3.03, 3.83, 5.03}};  // [q4_K, q5_K, q6_K][1, 2, 4 tiles]
constexpr double KQ_PART_US[3] = {6.2, 4.5, 2.4};                                                // per tile row, [1, 2, 4 tiles]

// LDS of a block of TM 32-row tiles: NA buffers of a super-block's activations ([tile][row 32][256]), NW buffers a wave of
// its 32 weight rows' super-block ([row 32][WROW]), NS records of a super-block's activation scales and mins operands.
template <uint32_t TY, int TM>
struct KqGeo {
    static constexpr bool Q6 = TY == KF_TYPE_Q6_K, Q4 = TY == KF_TYPE_Q4_K, Q5 = TY == KF_TYPE_Q5_K;
    static constexpr int BM = 32 * TM;
    static constexpr int SBB = Q6 ? KF_Q6_K_BYTES : Q4 ? KF_Q4_K_BYTES : KF_Q5_K_BYTES;  // bytes of a super-block
    static constexpr int WROW = Q6 ? 224 : SBB;   // LDS bytes of a weight row's super-block (q6_K: its 16-byte aligned window)
    static constexpr int QS = Q4 ? 16 : 48;       // q4_K / q5_K: the nibbles' offset
    static constexpr int PR = WROW / 16;          // 16-byte pieces of a row's super-block
    static constexpr int PW = 32 * PR;            // pieces of a wave's rows
    static constexpr int NWI = (PW + 63) / 64;    // weight DMA instructions a wave and super-block
    static constexpr int NSI = Q6 ? 1 : 2;        // record DMA instructions a wave and super-block
    static constexpr int SHIFT = Q4 ? 3 : 8;      // S = S_lo + (S_hi << SHIFT)
    static constexpr int ABUF = BM * 256;
    static constexpr int WBUF = 32 * WROW;        // one wave's
    static constexpr int REC = BM * (Q6 ? 4 : 36);  // dx f32 [BM], then the mins operands f16 [BM][16]
    static constexpr int NA = TM == 1 ? 3 : 2;
    static constexpr int NS = NA + 1;             // one more than ahead: a tile is rescaled one super-block late
    static constexpr int ROOM = KQ_LDS - KQ_EPI - NA * ABUF - NS * REC;
    static constexpr int NW = ROOM >= 3 * KQ_WAVES * WBUF ? 3 : ROOM >= 2 * KQ_WAVES * WBUF ? 2 : 1;
    static constexpr int A = 0, W = A + NA * ABUF, R = W + NW * KQ_WAVES * WBUF, LDS = R + NS * REC;
    static_assert(LDS + KQ_EPI <= KQ_LDS, "the buffers fit the LDS");
    // vector memory operations issued after the loads that the next super-block needs, where they are waited for
    static constexpr int wait(int TL) {
        const int batch = NSI + TL + NWI;
        const int w = (NW - 1) * batch, a = NWI + (NA - 2) * batch;
        return w < a ? w : a;
    }
};

// XCD-aware order over T work items: block b < T runs item (b % 8) (T / 8) + b / 8, so XCD x (blocks go to the eight
// XCDs round-robin) works through a contiguous range of weight tiles against every activation panel. Identity when T is
// not a multiple of eight.
__device__ __forceinline__ int kq_order(int T, int b) { return (T & 7) ? b : (b & 7) * (T >> 3) + (b >> 3); }

// A tile whose super-blocks several range blocks shared: its rows and columns and how many partial tiles make it (0: none)
struct KqDesc {
    int m0, m_end, n0, count;
};

// The launch's work besides whole tiles. Partial tiles go to `part` ([slot][register][thread]) and kq_reduce_kernel adds
// them.
//  * One matrix: tiles below `full` (whole rounds of the CUs) are a block each; the others run as S blocks each, over S
//    consecutive ranges of K (slot S t + range for the t-th of them). part == nullptr: every tile is a block.
//  * Grouped: the tiles of all slots are laid end to end, super-block after super-block, and cut into G equal ranges, a
//    block each, so that every CU gets the same work however the pairs fall on the slots; a tile weighs its number of
//    32-row parts plus one (the weight side). A tile inside a range is stored directly; of a tile that is cut, every
//    block leaves its part (slot 2 b + 1 for the part with the tile's first super-block, 2 b otherwise: a range has at
//    most one of each) and the block with its start describes it in desc[b]. part == nullptr: every tile weighs one and
//    is a block of its own, for grids where the parts' way through memory costs more than the rounds it evens out.
struct KqWork {
    float* part;
    KqDesc* desc;
    int full, S;  // grouped: full is unused, S is G
};

// The grouped (MoE) form: the activation rows are routed pairs in group order (slot s: rows offsets[s]..offsets[s + 1]),
// slot s multiplies its own expert matrix (w + s expert_bytes; with w2, output columns from n_split on come from
// w2 + s expert_bytes, row n - n_split), and output row p goes to y row out_rows[p] (or p).
struct KqMoe {
    const int32_t* offsets;
    const int32_t* out_rows;
    const uint8_t* w2;
    int64_t expert_bytes;
    int n_slots, n_split;
};

// kf_adma16 / kf_adma4 by the first LANES lanes only: the mask is set around the one instruction instead of by a branch,
// which would cut the K loop's steps into small basic blocks (70 spilled registers). For uniform control flow of whole
// waves.
template <int LANES>
__device__ __forceinline__ void kq_adma16(kf_arsrc_t r, int voff, int soff, const void* lds) {
    static_assert(LANES > 0 && LANES < 64, "a part of the wave");
    asm volatile("s_mov_b32 m0, %3\n\ts_mov_b64 exec, %4\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds\n\ts_mov_b64 exec, -1" ::"v"(voff),
                 "s"(r), "s"(soff), "s"(kf_lds_addr(lds)), "s"((1ull << LANES) - 1)
                 : "memory", "m0");
}
template <int LANES>
__device__ __forceinline__ void kq_adma4(kf_arsrc_t r, int voff, int soff, const void* lds) {
    static_assert(LANES > 0 && LANES < 64, "a part of the wave");
    asm volatile("s_mov_b32 m0, %3\n\ts_mov_b64 exec, %4\n\tbuffer_load_dword %0, %1, %2 offen lds\n\ts_mov_b64 exec, -1" ::"v"(voff),
                 "s"(r), "s"(soff), "s"(kf_lds_addr(lds)), "s"((1ull << LANES) - 1)
                 : "memory", "m0");
}

// Grouped form: a block's arguments and the state of its range, parked in LDS while a K loop runs (kept in scalar registers
// across the loop they would spill). Written by thread 0 between barriers, read as wave-uniform values.
struct KqState {
    const uint8_t *w, *w2;
    const int8_t* xq;
    const _Float16* xa;
    const float* xd;
    float* y;
    const int32_t *offsets, *out_rows;
    float* part;
    KqDesc* desc;
    int64_t row_bytes, expert_bytes;
    int N, K, n_slots, n_split;
    int b, G, U, u, u_end, slots_w;     // the range block, the ranges, their total, this block's position and end
    int m0, m_end, n0, s0, s1, next;    // the tile in hand, its super-blocks here and where the next one starts
    int count;                          // partial tiles of a tile that starts here and goes on
};
static_assert(sizeof(KqState) <= KQ_EPI, "the parked state fits");

__device__ __forceinline__ int kq_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t kq_uniform(int64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
    return (int64_t)((uint64_t)hi << 32 | lo);
}
template <typename T>
__device__ __forceinline__ T* kq_uniform(T* p) {
    return reinterpret_cast<T*>(kq_uniform((int64_t)reinterpret_cast<uint64_t>(p)));
}

// Grouped form: the weight of a slot of `rows` rows (per super-block and column tile) in tiles of TM 32-row parts, or
// (whole) its number of tiles
template <int TM>
__device__ __forceinline__ int kq_slot_w(int rows, bool whole) {
    if (whole) return (rows + 32 * TM - 1) / (32 * TM);
    const int full = rows / (32 * TM), rest = rows - full * 32 * TM;
    return full * (TM + 1) + (rest > 0 ? (rest + 31) / 32 + 1 : 0);
}

// The sum of the slots' weights (every lane of the wave calls it)
template <int TM>
__device__ int kq_slots_w(const int32_t* __restrict__ offsets, int n_slots, bool whole) {
    int t = 0;
    for (int s = threadIdx.x & 63; s < n_slots; s += 64) t += kq_slot_w<TM>(offsets[s + 1] - offsets[s], whole);
    return kq_uniform(kf_wave_isum(t));
}

// The slot whose weight range holds position q, and the position inside it
template <int TM>
__device__ int kq_find_slot(const int32_t* __restrict__ offsets, int n_slots, bool whole, int& q) {
    const int lane = threadIdx.x & 63;
    for (int base = 0;; base += 64) {
        const int s = base + lane;
        int v = s < n_slots ? kq_slot_w<TM>(offsets[s + 1] - offsets[s], whole) : 0;
        const int own = v;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(v, o, 64);
            if (lane >= o) v += u;
        }
        const uint64_t hit = __ballot(v > q);
        if (hit || base + 64 >= n_slots) {
            const int l = hit ? __builtin_ctzll(hit) : 63;
            q -= __builtin_amdgcn_readlane(v, l) - __builtin_amdgcn_readlane(own, l);
            return min(base + l, n_slots - 1);
        }
        q -= __builtin_amdgcn_readlane(v, 63);
    }
}

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t kq_pk_mul(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b)));
}
__device__ __forceinline__ uint32_t kq_pk_mad(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b) + __builtin_bit_cast(u16x2, c)));
}

// Bytes 1 and 3 of v as 16-bit pairs
__device__ __forceinline__ uint32_t kq_odd(uint32_t v) { return __builtin_amdgcn_perm(v, v, 0x0c030c01u); }

// Byte B of v in both 16-bit halves, zero- or sign-extended
template <int B>
__device__ __forceinline__ uint32_t kq_pair(uint32_t v) {
    return __builtin_amdgcn_perm(v, v, 0x0c000c00u | (uint32_t)B << 16 | B);
}
template <int B>
__device__ __forceinline__ uint32_t kq_pair_signed(uint32_t v) {
    typedef short i16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, (i16x2)(__builtin_bit_cast(i16x2, __builtin_amdgcn_perm(v, v, 0x000c000cu | (uint32_t)B << 24 | B << 8)) >> (short)8));
}

// The two int8 operand planes of one group for a lane: its 16 columns' products v = scale x value, v = lo + (hi << SHIFT)
struct KqPlanes {
    v4i lo, hi;
};

// Four products v + 128 as 16-bit pairs (e: bytes 0 and 2, o: bytes 1 and 3 of the four), split into the signed low byte
// and the rest: v + 128 = 256 hi + b, v = 256 hi + (b - 128)
__device__ __forceinline__ int kq_low16(uint32_t e, uint32_t o) { return (int)(__builtin_amdgcn_perm(o, e, 0x06020400u) ^ 0x80808080u); }
__device__ __forceinline__ int kq_high16(uint32_t e, uint32_t o) { return (int)__builtin_amdgcn_perm(o, e, 0x07030501u); }

// A wave's weight column (32 lanes a tile, each lane half the group's columns) being expanded, one super-block at a time
template <uint32_t TY, int TM>
struct KqWeight {
    using G = KqGeo<TY, TM>;
    uint32_t sc[2], sh[2], mn[2];  // q4_K / q5_K: the eight 6-bit scales (q4_K: their low and high three bits) and mins
    uint32_t sw[4];               // q6_K: the sixteen int8 scales, shifted so that group g's is byte 2 (g % 2) of word g / 2
    uint32_t d16;                 // d (low), dmin (high)
    uint4 raw, raw2, qh;

    // the header, and the first group's bytes
    __device__ __forceinline__ void begin(const uint8_t* wr, int half) {
        if constexpr (G::Q6) {
            const u32x4_a2 s = *reinterpret_cast<const u32x4_a2*>(wr + 192);
#pragma unroll
            for (int k = 0; k < 4; k++) sw[k] = s[k] >> (8 * half);
            d16 = *reinterpret_cast<const uint16_t*>(wr + 208);
        } else {
            const uint4 hd = *reinterpret_cast<const uint4*>(wr);
            kf_q4k_scales8(hd.y, hd.z, hd.w, sc, mn);
            if constexpr (G::Q4) {
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    sh[k] = (sc[k] >> 3) & 0x07070707u;
                    sc[k] &= 0x07070707u;
                }
            }
            d16 = hd.x;
            if constexpr (G::Q5) qh = *reinterpret_cast<const uint4*>(wr + 16 + 16 * half);
        }
        fetch<0>(wr, half);
    }

    // group g's bytes into registers (q4_K / q5_K: a pair of groups shares its 16 bytes; q6_K: four groups share 48)
    template <int g>
    __device__ __forceinline__ void fetch(const uint8_t* wr, int half) {
        if constexpr (G::Q6) {
            if constexpr (g % 4 == 0) {
                const u32x4_a2 a = *reinterpret_cast<const u32x4_a2*>(wr + 16 * g + 16 * half);
                const u32x4_a2 b = *reinterpret_cast<const u32x4_a2*>(wr + 16 * g + 32 + 16 * half);
                const u32x4_a2 h = *reinterpret_cast<const u32x4_a2*>(wr + 128 + 8 * g + 16 * half);
                raw = make_uint4(a.x, a.y, a.z, a.w);
                raw2 = make_uint4(b.x, b.y, b.z, b.w);
                qh = make_uint4(h.x, h.y, h.z, h.w);
            }
        } else if constexpr (g % 2 == 0) {
            raw = *reinterpret_cast<const uint4*>(wr + G::QS + 16 * g + 16 * half);
        }
    }

    template <int g>
    __device__ __forceinline__ KqPlanes planes() const {
        KqPlanes p;
        const uint32_t m4 = 0x0f0f0f0fu, mb = 0x00ff00ffu;
        if constexpr (G::Q4) {
            // 6-bit scale 8 sh + sl: the nibble products q sl and q sh (at most 105) are bytes, two to a 16-bit product
            const uint32_t v[4] = {raw.x, raw.y, raw.z, raw.w};
            const uint32_t s0 = kq_pair<g & 3>(sc[g >> 2]), s1 = kq_pair<g & 3>(sh[g >> 2]);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t q = ((g & 1) ? v[e] >> 4 : v[e]) & m4;
                p.lo[e] = (int)kq_pk_mul(q, s0);
                p.hi[e] = (int)kq_pk_mul(q, s1);
            }
        } else if constexpr (G::Q5) {
            const uint32_t v[4] = {raw.x, raw.y, raw.z, raw.w}, h[4] = {qh.x, qh.y, qh.z, qh.w};
            const uint32_t s = kq_pair<g & 3>(sc[g >> 2]);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t q = (((g & 1) ? v[e] >> 4 : v[e]) & m4) | ((g < 4 ? h[e] << (4 - g) : h[e] >> (g - 4)) & 0x10101010u);
                const uint32_t ev = kq_pk_mad(q & mb, s, 0x00800080u), ov = kq_pk_mad(kq_odd(q), s, 0x00800080u);
                p.lo[e] = kq_low16(ev, ov);
                p.hi[e] = kq_high16(ev, ov);
            }
        } else {
            // q6_K group 4 h + k: the low (k < 2) or high nibbles of run k % 2 and bits 2 k.. of qh; v = sc (q - 32)
            const uint32_t v[4] = {(g & 1) ? raw2.x : raw.x, (g & 1) ? raw2.y : raw.y, (g & 1) ? raw2.z : raw.z, (g & 1) ? raw2.w : raw.w};
            const uint32_t h[4] = {qh.x, qh.y, qh.z, qh.w};
            const uint32_t s = kq_pair_signed<2 * (g & 1)>(sw[g >> 1]);
            const uint32_t c = kq_pk_mad(s, 0xffe0ffe0u, 0x00800080u);  // 128 - 32 sc
            constexpr int k = g & 3;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t lo = ((k & 2) ? v[e] >> 4 : v[e]) & m4;
                const uint32_t q = lo | (((h[e] >> (2 * k)) & 0x03030303u) << 4);
                const uint32_t ev = kq_pk_mad(q & mb, s, c), ov = kq_pk_mad(kq_odd(q), s, c);
                p.lo[e] = kq_low16(ev, ov);
                p.hi[e] = kq_high16(ev, ov);
            }
        }
        return p;
    }

    // the mins operand: per lane the eight mins, times 64 for the lanes that meet the high parts of the group sums
    __device__ __forceinline__ v8h mins(int half) const {
        // 1024 + m as f16 bits, less 1024, times f: exact
        typedef _Float16 v2h __attribute__((ext_vector_type(2)));
        const _Float16 f = half ? (_Float16)1.0f : (_Float16)64.0f;
        v8h mo;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t u = __builtin_amdgcn_perm(0x64646464u, mn[k >> 1], (k & 1) ? 0x04030402u : 0x04010400u);
            const v2h m = __builtin_bit_cast(v2h, u) - (v2h){(_Float16)1024.0f, (_Float16)1024.0f};
            mo[2 * k] = m[0] * f;
            mo[2 * k + 1] = m[1] * f;
        }
        return mo;
    }
};

// WIDE: the outputs' sums over the super-blocks in 64 bits
struct KqSums64 {
    double v[16];
    __device__ __forceinline__ double& operator[](int r) { return v[r]; }
};

template <uint32_t TY, int TM, bool MOE, bool WIDE>
__global__ void __launch_bounds__(KQ_THREADS, 2) gemm_kq_kernel(const uint8_t* w_, int64_t row_bytes_, const int8_t* xq_, const _Float16* xa_,
                                                                 const float* xd_, const float* bias_, const float* res_, float* y_, int M_, int N_,
                                                                 int K_, KqWork work, KqMoe moe) {
    using G = KqGeo<TY, TM>;
    constexpr int BM = G::BM;
    extern __shared__ __align__(256) uint8_t lds[];
    KqState& st = *reinterpret_cast<KqState*>(lds + G::LDS);
    if constexpr (MOE) {
        // positions are super-blocks times tile weights, from the first tile of all (whole tiles: tiles)
        const bool whole = !work.part;
        const int unit = whole ? 1 : K_ >> 8, NT = (N_ + KQ_BN - 1) / KQ_BN;
        const int sw = kq_slots_w<TM>(moe.offsets, moe.n_slots, whole), U = NT * unit * sw;
        // at least a few super-blocks a range, where tiles are cut
        const int Gr = whole ? min(work.S, U) : max(min(work.S, U / (4 * (TM + 1))), U > 0 ? 1 : 0);
        const bool idle = (int)blockIdx.x >= Gr;
        const int b = idle ? blockIdx.x : kq_order(Gr, blockIdx.x);
        if (threadIdx.x == 0 && work.desc) work.desc[b].count = 0;
        if (idle) return;  // nothing to do: whole block, before any barrier
        if (threadIdx.x == 0)
            st = KqState{w_, moe.w2, xq_, xa_, xd_, y_, moe.offsets, moe.out_rows, work.part, work.desc, row_bytes_, moe.expert_bytes, N_, K_,
                         moe.n_slots, moe.n_split, b, Gr, U, (int)((int64_t)U * b / Gr), (int)((int64_t)U * (b + 1) / Gr), sw, 0, 0, 0, 0, 0, 0, 0};
    }
    for (;;) {  // grouped: a range's tiles; otherwise one pass
    if constexpr (MOE) __syncthreads();  // the state is written, and every wave is done with the LDS of the tile before
    // the thread's indices, made anew for each tile: what derives from them is not kept from tile to tile
    int tid = threadIdx.x;
    if constexpr (MOE) __asm__ volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, r32 = lane & 31;
    const int N = MOE ? kq_uniform(st.N) : N_, K = MOE ? kq_uniform(st.K) : K_;
    const int64_t row_bytes = MOE ? kq_uniform(st.row_bytes) : row_bytes_;
    const int kg = K >> 5, nsb = K >> 8;
    int s0 = 0, s1 = nsb, m0, m_end, n0, nr0, n_rows = N, slot = -1;  // slot: the partial tile's place (-1: a whole tile)
    const uint8_t* wt = MOE ? kq_uniform(st.w) : w_;
    if constexpr (MOE) {
        // the tile at the range's position
        const int u = kq_uniform(st.u), u_end = kq_uniform(st.u_end);
        const bool whole = !kq_uniform(st.part);
        const int unit = whole ? 1 : nsb, tw = whole ? 1 : TM + 1;  // of a full tile
        const int sw = kq_uniform(st.slots_w), per = sw * unit;
        const int tn = u / per;
        const int q = u - tn * per, q0 = q / unit;
        int qs = q0;
        const int32_t* offsets = kq_uniform(st.offsets);
        const int sl = kq_find_slot<TM>(offsets, kq_uniform(st.n_slots), whole, qs);
        const int r0 = kq_uniform(offsets[sl]), r1 = kq_uniform(offsets[sl + 1]);
        const int slot_pos = (q0 - qs) * unit;  // the slot's first position in the column tile
        const int i = min((q - slot_pos) / (unit * tw), (r1 - r0) / BM);
        m0 = r0 + i * BM;
        m_end = r1;
        const int wgt = whole ? 1 : (min(r1 - m0, BM) + 31) / 32 + 1;
        const int start = tn * per + slot_pos + i * unit * tw, end = start + unit * wgt;
        n0 = tn * KQ_BN;
        nr0 = n0;
        const uint8_t* w2 = kq_uniform(st.w2);
        if (w2) {
            const int split = kq_uniform(st.n_split);
            n_rows = split;
            if (n0 >= split) {
                wt = w2;
                nr0 = n0 - split;
                n_rows = N - split;
            }
        }
        wt += sl * kq_uniform(st.expert_bytes);
        s0 = (u - start) / wgt;
        s1 = u_end >= end ? nsb : (u_end - start) / wgt;
        int count = 0;
        if (s0 == 0 && s1 < nsb) {
            // the blocks after this one, up to the one that reaches the tile's end
            const int b = kq_uniform(st.b), Gr = kq_uniform(st.G), U = kq_uniform(st.U);
            count = 2;
            while ((int64_t)U * (b + count) / Gr < end) count++;
        }
        s0 = kq_uniform(s0);
        s1 = kq_uniform(s1);
        m0 = kq_uniform(m0);
        m_end = kq_uniform(m_end);
        n0 = kq_uniform(n0);
        __syncthreads();  // every wave has read the position
        if (tid == 0) {
            st.m0 = m0;
            st.m_end = m_end;
            st.n0 = n0;
            st.s0 = s0;
            st.s1 = s1;
            st.next = end;
            st.count = count;
        }
    } else {
        const int mt = (M_ + BM - 1) / BM;
        int t;
        if (work.part && (int)blockIdx.x >= work.full) {
            slot = blockIdx.x - work.full;
            const int tt = slot / work.S, sp = slot - tt * work.S;
            t = work.full + tt;
            s0 = nsb * sp / work.S;
            s1 = nsb * (sp + 1) / work.S;
        } else {
            t = kq_order(work.full, blockIdx.x);
        }
        const int tn = t / mt;
        m0 = (t - tn * mt) * BM;
        m_end = M_;
        n0 = tn * KQ_BN;
        nr0 = n0;
        s0 = kq_uniform(s0);
        s1 = kq_uniform(s1);
    }
    if (!MOE || s0 < s1) {
    // The wave's weight rows: a buffer from the 16-byte piece its first row starts in to the piece the matrix ends in
    // (reads stay inside that piece's 16 bytes; rows past the matrix read as zeros through the hardware range check).
    // Waves wholly past the matrix get an empty one.
    const int wr0 = nr0 + 32 * wave;
    const int64_t wb0 = (int64_t)wr0 * row_bytes;
    const int wsh = (int)(wb0 & 15);  // q6_K rows start at any even byte
    const int64_t wlen = ((int64_t)n_rows * row_bytes + 15) / 16 * 16 - (wb0 - wsh);
    const kf_arsrc_t rw = kf_arsrc(wt + (wr0 < n_rows ? wb0 - wsh : 0), wr0 < n_rows ? (uint64_t)wlen : 0);
    const kf_arsrc_t rx = kf_arsrc((MOE ? kq_uniform(st.xq) : xq_) + (int64_t)m0 * K, (uint64_t)(m_end - m0) * K);
    const kf_arsrc_t rs = kf_arsrc((MOE ? kq_uniform(st.xa) : xa_) + (int64_t)m0 * nsb * 16, (uint64_t)(m_end - m0) * nsb * 32);
    const kf_arsrc_t rd = kf_arsrc((MOE ? kq_uniform(st.xd) : xd_) + (int64_t)m0 * kg, (uint64_t)(m_end - m0) * kg * 4);
    // past the range's end the loads run with an empty buffer: no traffic, and the counts of the waits hold
    auto off = [](kf_arsrc_t r, bool on) __attribute__((always_inline)) {
        if (!on) r[2] = 0;
        return r;
    };
    // record part k: the activation scales, the mins operands; each wave moves its eighth of the block's rows
    auto dma_rec = [&](int sb, int k) __attribute__((always_inline)) {
        uint8_t* rec = lds + G::R + (sb % G::NS) * G::REC;
        constexpr int RW = BM / KQ_WAVES;
        if (k == 0) {
            kq_adma4<RW>(off(rd, sb < s1), (wave * RW + lane) * kg * 4, sb * 32, rec + wave * RW * 4);
        } else {
            kq_adma16<2 * RW>(off(rs, sb < s1), (wave * RW + (lane >> 1)) * nsb * 32 + (lane & 1) * 16, sb * 32, rec + BM * 4 + wave * RW * 32);
        }
    };
    // The wave's rows 4 w.. of activation tile i: lane l takes chunk (l % 16) ^ (row % 16) of row 4 w + l / 16 and writes
    // it at position l % 16, so the MFMA operand reads below hit distinct banks. With four tiles the addresses are made
    // anew each time (an opaque lane index): kept across the K loop they would spill.
    auto dma_a = [&](int sb, int i) __attribute__((always_inline)) {
        int ln = lane;
        if constexpr (TM > 2) __asm__("" : "+v"(ln));
        const int arow = 4 * wave + (ln >> 4);
        kf_adma16(off(rx, sb < s1), (arow + 32 * i) * K + 16 * ((ln & 15) ^ (arow & 15)), sb * 256,
                  lds + G::A + (sb % G::NA) * G::ABUF + wave * 1024 + i * 8192);
    };
    // 64 of the pieces of the wave's 32 weight rows
    auto dma_w = [&](int sb, int k) __attribute__((always_inline)) {
        int ln = lane;
        if constexpr (TM > 2) __asm__("" : "+v"(ln));
        const int q = 64 * k + ln, row = q / G::PR, piece = q - G::PR * row;
        const int start = row * (int)row_bytes + (G::Q6 ? wsh + sb * G::SBB : 0);
        const int vo = (G::Q6 ? start & ~15 : start) + 16 * piece;
        uint8_t* buf = lds + G::W + (sb % G::NW * KQ_WAVES + wave) * G::WBUF;
        if (64 * k + 64 <= G::PW)
            kf_adma16(off(rw, sb < s1), vo, G::Q6 ? 0 : sb * G::SBB, buf + k * 1024);
        else
            kq_adma16<(G::PW & 63) ? (G::PW & 63) : 1>(off(rw, sb < s1), vo, G::Q6 ? 0 : sb * G::SBB, buf + k * 1024);
    };

    using Sums = std::conditional_t<WIDE, KqSums64, v16f>;
    Sums acc[TM];
#pragma unroll
    for (int i = 0; i < TM; i++) acc[i] = Sums{};

    // The K loop over TLC 32-row tiles (a grouped tile with fewer rows skips the empty ones). Per super-block the tiles
    // run one after another, each as eight group steps: the step's two MFMAs, one eighth of the previous tile's rescale
    // and, in the last tile, the expansion of the same group of the next super-block into the operand registers the
    // step has just used. So every step mixes matrix-core and vector work and no phase of a wave is without MFMAs.
    auto kloop = [&](auto tlc) __attribute__((always_inline)) {
        constexpr int TL = decltype(tlc)::value;
        // An even number of tiles carries the last tile's rescale over into the next super-block's first tile; an odd
        // one, whose parities would alternate, rescales it at the super-block's end.
        constexpr bool LAG = TL % 2 == 0;
        constexpr bool SLOTS = TL > 1;
        constexpr int SPER = (G::NSI + TL + G::NWI + 8 * (TL - 1) - 1) / (8 * (TL > 1 ? TL - 1 : 1));  // loads a step, done before the last tile
        KqPlanes B[8];
        KqWeight<TY, TM> kw;
        float d = 0.0f, dm = 0.0f, dp = 0.0f, dmp = 0.0f;  // this super-block's column scales, and the previous one's
        v8h mo = v8h{};
        auto wrow = [&](int sb) __attribute__((always_inline)) {
            const uint8_t* p = lds + G::W + (sb % G::NW * KQ_WAVES + wave) * G::WBUF + r32 * G::WROW;
            return G::Q6 ? p + ((r32 * (int)row_bytes + wsh + sb * G::SBB) & 15) : p;
        };
        auto take = [&]() __attribute__((always_inline)) {
            d = kf_h2f(kw.d16 & 0xffffu);
            if constexpr (!G::Q6) {
                dm = kf_h2f(kw.d16 >> 16);
                __asm__("" : "+v"(dm));  // kept in f32: mixed-precision multiply-adds need wait states here
            }
        };
        // group g's activation operand of tile i: chunk 2 g + half of the lane's row, stored at (2 g + half) ^ (row % 16),
        // i.e. 32 g exclusive-or'ed into the address of group 0's
        const uint32_t a0 = kf_lds_addr(lds + G::A) + r32 * 256 + 16 * (half ^ (r32 & 15));
        auto aop = [&](uint32_t at, int g, int i) __attribute__((always_inline)) {
            const uint32_t p = ((at + a0) ^ (32u * g)) + i * 8192;
            return *reinterpret_cast<const __attribute__((address_space(3))) v4i*>(p);
        };
        v16i S[2][2];  // [tile parity][lo, hi]; lo becomes S once a tile is done
        v16f mins = v16f{};
        // The rescale of tile i in eight parts: S = lo + (hi << SHIFT) in the first two, the mins product, then rows
        // rat[g].. of acc += dx (d S - dmin mins); accumulator register r holds row (r % 4) + 8 (r / 4) + 4 (lane / 32). The
        // LDS operands of part g are read by load(g) one step earlier.
        constexpr int rat[9] = {0, 0, 0, 4, 6, 8, 12, 14, 16};
        float dxn[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        auto load = [&](auto gc, const uint8_t* rec, int i) __attribute__((always_inline)) {
            constexpr int g = decltype(gc)::value;
            if constexpr (g >= 2 && g < 8) {
#pragma unroll
                for (int r = rat[g]; r < rat[g + 1]; r++) dxn[r - rat[g]] = reinterpret_cast<const float*>(rec)[i * 32 + half * 4 + 8 * (r >> 2) + (r & 3)];
            }
        };
        auto rescale = [&](auto pc, auto gc, Sums& a, const float (&dx)[4], const uint8_t* rec, int i, float ds, float dms) __attribute__((always_inline)) {
            constexpr int p = decltype(pc)::value, g = decltype(gc)::value;
            if constexpr (g < 2) {
#pragma unroll
                for (int r = 8 * g; r < 8 * g + 8; r++) S[p][0][r] += (int)((uint32_t)S[p][1][r] << G::SHIFT);
                if constexpr (g == 1 && !G::Q6) {
                    const v8h xo = *reinterpret_cast<const v8h*>(rec + BM * 4 + (i * 32 + r32) * 32 + half * 16);
                    mins = __builtin_amdgcn_mfma_f32_32x32x16_f16(xo, mo, v16f{}, 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int r = rat[g]; r < rat[g + 1]; r++) {
                    const float sf = (float)S[p][0][r];
                    const float t = G::Q6 ? ds * sf : fmaf(-dms, mins[r], ds * sf);
                    if constexpr (WIDE)
                        a[r] += (double)(t * dx[r - rat[g]]);
                    else
                        a[r] = fmaf(t, dx[r - rat[g]], a[r]);
                }
            }
        };
        // one tile's eight steps; `prev`: the tile rescaled meanwhile (its index and parity), sbn: the super-block
        // expanded meanwhile (EXP)
        auto tile = [&](auto ic, auto pc, auto expc, auto firstc, uint32_t at, const uint8_t* prec, const uint8_t* wn, auto issue)
            __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value, p = decltype(pc)::value;
            constexpr bool EXP = decltype(expc)::value, FIRST = decltype(firstc)::value;
            constexpr int pi = i == 0 ? TL - 1 : i - 1;  // the tile before this one
            if constexpr (i == 0 && !LAG && !G::Q6) mo = kw.mins(half);
            if constexpr (EXP) kw.begin(wn, half);
            v4i a = aop(at, 0, i);
            auto step = [&](auto gc) __attribute__((always_inline)) {
                constexpr int g = decltype(gc)::value;
                // the next step's LDS reads go first, this step's matrix and vector work hides their latency
                v4i an = a;
                if constexpr (g < 7) an = aop(at, g + 1, i);
                const float dx[4] = {dxn[0], dxn[1], dxn[2], dxn[3]};
                if constexpr (!FIRST && g < 7) load(std::integral_constant<int, g + 1>{}, prec, pi);
                if constexpr (SLOTS) {
#pragma unroll
                    for (int k = SPER * (8 * i + g); k < SPER * (8 * i + g + 1); k++) issue(k);
                }
                __builtin_amdgcn_sched_barrier(0);
                const KqPlanes b = B[g];
                S[p][0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b.lo, g == 0 ? v16i{} : S[p][0], 0, 0, 0);
                S[p][1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b.hi, g == 0 ? v16i{} : S[p][1], 0, 0, 0);
                if constexpr (!FIRST) rescale(std::integral_constant<int, 1 - p>{}, gc, acc[pi], dx, prec, pi, i == 0 ? dp : d, i == 0 ? dmp : dm);
                if constexpr (EXP) {
                    B[g] = kw.template planes<g>();
                    if constexpr (g < 7) kw.template fetch<g + 1>(wn, half);
                }
                // the previous super-block's mins operand has had its last use
                if constexpr (i == 0 && g == 2 && LAG && !G::Q6) mo = kw.mins(half);
                a = an;
                __builtin_amdgcn_sched_barrier(0);
            };
            step(std::integral_constant<int, 0>{});
            step(std::integral_constant<int, 1>{});
            step(std::integral_constant<int, 2>{});
            step(std::integral_constant<int, 3>{});
            step(std::integral_constant<int, 4>{});
            step(std::integral_constant<int, 5>{});
            step(std::integral_constant<int, 6>{});
            step(std::integral_constant<int, 7>{});
        };
        // the rescale of a super-block's last tile by itself
        auto finish = [&](int sb) __attribute__((always_inline)) {
            const uint8_t* rec = lds + G::R + (sb % G::NS) * G::REC;
            auto all = [&](auto gc) __attribute__((always_inline)) {
                load(gc, rec, TL - 1);
                rescale(std::integral_constant<int, (TL - 1) & 1>{}, gc, acc[TL - 1], dxn, rec, TL - 1, dp, dmp);
            };
            all(std::integral_constant<int, 0>{});
            all(std::integral_constant<int, 1>{});
            all(std::integral_constant<int, 2>{});
            all(std::integral_constant<int, 3>{});
            all(std::integral_constant<int, 4>{});
            all(std::integral_constant<int, 5>{});
            all(std::integral_constant<int, 6>{});
            all(std::integral_constant<int, 7>{});
        };
        // One super-block (FIRST: no tile before it to rescale)
        auto sblock = [&](auto firstc, int sbv) __attribute__((always_inline)) {
            constexpr bool FIRST = decltype(firstc)::value || !LAG;
            const int sb = __builtin_amdgcn_readfirstlane(sbv);
            // The loads ahead: all at once with one tile, which waits for them right away; with more, SPER of them a step
            // from the first, so that the eight waves' requests do not queue in front of each other.
            auto issue = [&](int k) __attribute__((always_inline)) {
                if (k < G::NSI)
                    dma_rec(sb + G::NA - 1, k);
                else if (k < G::NSI + TL)
                    dma_a(sb + G::NA - 1, k - G::NSI);
                else if (k < G::NSI + TL + G::NWI)
                    dma_w(sb + G::NW, k - G::NSI - TL);
            };
            if constexpr (!SLOTS) {
#pragma unroll
                for (int k = 0; k < G::NSI + TL + G::NWI; k++) issue(k);
            }
            const uint32_t at = (sb % G::NA) * G::ABUF;
            const uint8_t* rec = lds + G::R + (sb % G::NS) * G::REC;
            const uint8_t* prec = FIRST ? rec : lds + G::R + ((sb - 1) % G::NS) * G::REC;
            const uint8_t* wn = wrow(sb + 1);
            auto one = [&](auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value;
                if constexpr (i < TL) {
                    if constexpr (i == TL - 1) __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(G::wait(TL)) : "memory");
                    tile(ic, std::integral_constant<int, i & 1>{}, std::integral_constant<bool, i == TL - 1>{},
                         std::integral_constant<bool, FIRST && i == 0>{}, at, i == 0 ? prec : rec, wn, issue);
                }
            };
            one(std::integral_constant<int, 0>{});
            one(std::integral_constant<int, 1>{});
            one(std::integral_constant<int, 2>{});
            one(std::integral_constant<int, 3>{});
            dp = d;
            dmp = dm;
            take();
            if constexpr (!LAG) finish(sb);
            __syncthreads();
        };
#pragma unroll
        for (int b = 0; b < G::NA - 1; b++) {
#pragma unroll
            for (int k = 0; k < G::NSI; k++) dma_rec(s0 + b, k);
#pragma unroll
            for (int i = 0; i < TL; i++) dma_a(s0 + b, i);
        }
#pragma unroll
        for (int b = 0; b < G::NW; b++)
#pragma unroll
            for (int k = 0; k < G::NWI; k++) dma_w(s0 + b, k);
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        {
            const uint8_t* wr = wrow(s0);
            kw.begin(wr, half);
            auto ex = [&](auto gc) __attribute__((always_inline)) {
                constexpr int g = decltype(gc)::value;
                B[g] = kw.template planes<g>();
                if constexpr (g < 7) kw.template fetch<g + 1>(wr, half);
            };
            ex(std::integral_constant<int, 0>{});
            ex(std::integral_constant<int, 1>{});
            ex(std::integral_constant<int, 2>{});
            ex(std::integral_constant<int, 3>{});
            ex(std::integral_constant<int, 4>{});
            ex(std::integral_constant<int, 5>{});
            ex(std::integral_constant<int, 6>{});
            ex(std::integral_constant<int, 7>{});
            take();
            __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        using std::false_type;
        using std::true_type;
        sblock(true_type{}, s0);
#pragma unroll 1
        for (int sb = s0 + 1; sb < s1; sb++) sblock(false_type{}, sb);
        if constexpr (LAG) finish(s1 - 1);
    };
    if constexpr (MOE) {
        const int tl = (min(m_end - m0, BM) + 31) / 32;
        if (TM >= 4 && tl == 4)
            kloop(std::integral_constant<int, TM < 4 ? TM : 4>{});
        else if (TM >= 4 && tl == 3)
            kloop(std::integral_constant<int, TM < 3 ? TM : 3>{});
        else if (TM >= 2 && tl == 2)
            kloop(std::integral_constant<int, TM < 2 ? TM : 2>{});
        else
            kloop(std::integral_constant<int, 1>{});
    } else {
        kloop(std::integral_constant<int, TM>{});
    }

    // the tile, or the part of it that is this block's
    float* y = y_;
    float* part = work.part;
    const float *bias = bias_, *res = res_;
    const int32_t* out_rows = nullptr;
    int Nn = N_, me = m_end, mb = m0, n = n0;
    if constexpr (MOE) {
        const bool starts = kq_uniform(st.s0) == 0, ends = kq_uniform(st.s1) == kq_uniform(st.K) >> 8;
        if (!starts || !ends) {
            const int b = kq_uniform(st.b);
            slot = 2 * b + (starts ? 1 : 0);
            if (starts && tid == 0) kq_uniform(st.desc)[b] = KqDesc{st.m0, st.m_end, st.n0, st.count};
        }
        y = kq_uniform(st.y);
        part = kq_uniform(st.part);
        out_rows = kq_uniform(st.out_rows);
        bias = res = nullptr;
        Nn = kq_uniform(st.N);
        me = kq_uniform(st.m_end);
        mb = kq_uniform(st.m0);
        n = kq_uniform(st.n0);
    }
    if (slot >= 0) {
        float* pp = part + (size_t)slot * (TM * 16) * KQ_THREADS + tid;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) pp[(i * 16 + r) * KQ_THREADS] = (float)acc[i][r];
    } else {
        n += wave * 32 + r32;
        const float bn = bias && n < Nn ? bias[n] : 0.0f;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = mb + i * 32 + (r & 3) + 8 * (r >> 2) + 4 * half;
                if (m >= me || n >= Nn) continue;
                const int64_t o = (int64_t)(out_rows ? out_rows[m] : m) * Nn + n;
                y[o] = (float)acc[i][r] + bn + (res ? res[o] : 0.0f);
            }
    }
    }
    if constexpr (!MOE) return;
    __syncthreads();  // the state is written (an empty part runs no K loop, whose barriers would order it)
    if (kq_uniform(st.next) >= kq_uniform(st.u_end)) return;
    __syncthreads();  // every wave has read the state
    if (threadIdx.x == 0) st.u = st.next;
    }
}

// Adds the partial tiles of the tiles that several blocks shared, in K order (four at a time by themselves), with bias and residual. One thread an output;
// a block takes RED of the TM * 16 (register, 512 threads) slices of a tile, so every load and store is a run of whole
// lines: one slice with one matrix, whose few tiles have many parts (four made 32 rows of 4096 x 4096 14.2 us, 12.7 with
// one), four in the grouped form, where most blocks have nothing to add. A launch of its own: the last block to arrive adding them by itself took 10-40 us with 16 partial tiles, as
// one CU reads them all.
template <int TM, bool MOE, int RED>
__global__ void __launch_bounds__(KQ_THREADS) kq_reduce_kernel(KqWork work, const float* __restrict__ bias, const float* __restrict__ res,
                                                                const int32_t* __restrict__ out_rows, float* __restrict__ y, int M, int N) {
    constexpr int R = TM * 16;
    const int b = blockIdx.x / (R / RED), e0 = (blockIdx.x - b * (R / RED)) * RED, tid = threadIdx.x;
    KqDesc d;
    size_t first, step;  // the first partial tile's slot, and from the second on the distance
    if constexpr (MOE) {
        d = work.desc[b];
        if (d.count == 0) return;
        first = 2 * b + 1;  // then range block b + 1's slot 2 (b + 1), b + 2's ...
        step = 2;
    } else {
        const int mt = (M + 32 * TM - 1) / (32 * TM), t = work.full + b, tn = t / mt;
        d = KqDesc{(t - tn * mt) * 32 * TM, M, tn * KQ_BN, work.S};
        first = (size_t)b * work.S;
        step = 1;
    }
    const int n = d.n0 + (tid >> 6) * 32 + (tid & 31);
    // registers 4 q.. hold rows 8 q..
    const int mb = d.m0 + (e0 >> 4) * 32 + 8 * ((e0 & 15) >> 2) + (e0 & 3) + 4 * ((tid >> 5) & 1);
    if (mb >= d.m_end || n >= N) return;
    const float* p = work.part + (first * R + e0) * KQ_THREADS + tid;
    float v[RED] = {};
    for (int k = 0; k < d.count; k += 4) {
        float a[4][RED];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const size_t at = k + u > 0 ? 1 + (k + u - 1) * step : 0;
#pragma unroll
            for (int e = 0; e < RED; e++) a[u][e] = k + u < d.count ? p[(at * R + e) * KQ_THREADS] : 0.0f;
        }
#pragma unroll
        for (int e = 0; e < RED; e++) v[e] += ((a[0][e] + a[1][e]) + a[2][e]) + a[3][e];
    }
    const float bn = bias ? bias[n] : 0.0f;
#pragma unroll
    for (int e = 0; e < RED; e++) {
        if (mb + e >= d.m_end) break;
        const int64_t o = (int64_t)(out_rows ? out_rows[mb + e] : mb + e) * N + n;
        y[o] = v[e] + bn + (res ? res[o] : 0.0f);
    }
}

}  // namespace

// Whether the GEMM takes these weights: K a multiple of 256, rows of whole super-blocks from a 16-byte aligned base
bool kf_gemm_kq_ok(uint32_t ty, const void* w, int64_t row_bytes, int K, int N) {
    (void)N;
    return (ty == KF_TYPE_Q4_K || ty == KF_TYPE_Q5_K || ty == KF_TYPE_Q6_K) && K % 256 == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0 &&
           row_bytes == (int64_t)(K / 256) * (ty == KF_TYPE_Q4_K ? KF_Q4_K_BYTES : ty == KF_TYPE_Q5_K ? KF_Q5_K_BYTES : KF_Q6_K_BYTES);
}

namespace {

// Descriptors and partial tiles in the split scratch
constexpr size_t KQ_DESC_BYTES = 16384;
static_assert(KF_SPLIT_SCRATCH >= KF_SPLIT_TICKETS * 4 + KQ_DESC_BYTES, "room for the descriptors");

// Grouped: most range blocks, each with two partial tiles: one a CU, within the scratch
int kq_max_ranges(int tm, int cus) {
    const size_t room = (KF_SPLIT_SCRATCH - (size_t)KF_SPLIT_TICKETS * 4 - KQ_DESC_BYTES) / ((size_t)2 * tm * 16 * KQ_THREADS * 4);
    int G = kf_knob_or(KF_KNOB_KQ_G, cus);
    if ((size_t)G > room) G = (int)room;
    if (G > (int)(KQ_DESC_BYTES / sizeof(KqDesc))) G = (int)(KQ_DESC_BYTES / sizeof(KqDesc));
    return G;
}

// One matrix: most partial tiles, one a CU, within the smaller of the scratch's slots
int kq_max_parts(int tm, int cus) {
    const size_t room = (std::min(KF_SPLIT_SCRATCH, KF_SPLIT_SPARE) - (size_t)KF_SPLIT_TICKETS * 4 - KQ_DESC_BYTES) / ((size_t)tm * 16 * KQ_THREADS * 4);
    return (int)std::min((size_t)kf_knob_or(KF_KNOB_KQ_G, cus), room);
}

// A block's f32 sum of more super-blocks than kq_long is kept in 64 bits instead (WIDE), where the tile's registers have
// room: 16 super-blocks of q4_K are 9.7e-8 from the 64-bit result with f32 sums and 7.3e-8 with these, 51 of q6_K 1.32e-7
// and 4.4e-8, at 10% (q4_K), 6% (q5_K) and 3% (q6_K) of the K loop; priced higher on q4_K, as plans with K ranges in its place
// measured 3-5% less than the model has (500 rows of 4096 -> 4096: 36.2 us in two ranges, 39.0 wide). The few-row products,
// and the 64-row kernel in two or four K ranges, that these blocks replace had 8e-8 to 9.1e-8; where that kernel had whole
// rounds of tiles it summed as many in f32. 128-row tiles, and 64-row ones of q5_K (four registers spilled), keep the f32
// sum, as the tile kernels did whose whole rounds they took over; widths of q6_K that had no tile kernel before (rows
// that are not whole 16-byte pieces) leave them out instead: 2048 rows of 13056 -> 4096 take 426 us in place of 294,
// 6400 -> 2304 145 and 144, and 19.6 and 6.5 ms on the per-lane product.
int kq_long(bool ragged, int M, int N, int nsb, int cus) {
    const int T = ((N + KQ_BN - 1) / KQ_BN) * ((M + 63) / 64);  // tiles of the 64-row kernel
    if (ragged) return 12;
    return std::max(12, T >= cus ? nsb : 4 * T <= cus ? (nsb + 3) / 4 : 2 * T <= cus ? (nsb + 1) / 2 : nsb);
}
constexpr double KQ_WIDE_COST[3] = {1.25, 1.06, 1.03};  // [q4_K, q5_K, q6_K]

struct KqPlan {
    int tm, T, full, S;
    bool wide;
    double us;
};

KqPlan kq_plan_tm(uint32_t ty, int tm, int M, int N, int K, bool split) {
    KqPlan p;
    p.tm = tm;
    const int cus = kf_cu_count(), nsb = K / 256;
    p.T = ((N + KQ_BN - 1) / KQ_BN) * ((M + 32 * tm - 1) / (32 * tm));
    const int rem = p.T % cus, t = tm >> 1, max_g = kq_max_parts(tm, cus), k = ty == KF_TYPE_Q4_K ? 0 : ty == KF_TYPE_Q5_K ? 1 : 2;
    const double sb = KQ_SB_US[k][t];
    const bool fits = tm == 1 || (tm == 2 && ty != KF_TYPE_Q5_K), ragged = ty == KF_TYPE_Q6_K && K % 2048 != 0;
    const int longest = kq_long(ragged, M, N, nsb, cus);
    // a block of n super-blocks, in a launch whose longest one has `most`
    auto cost = [&](int n, int most) {
        if (most > longest && ragged && !fits) return 1e30;
        return KQ_ROUND_US[t] + sb * n * (most > longest && fits ? KQ_WIDE_COST[k] : 1.0);
    };
    const int rounds = p.T / cus;
    p.full = p.T;
    p.S = 1;
    p.us = (rounds + (rem ? 1 : 0)) * cost(nsb, nsb);
    // the tiles of the last round as S blocks each, S the cheapest that fits the CUs with two super-blocks a block or more; up
    // to KF_FEW_ROWS rows two or four, whichever fits, and f32 sums (the order a decoded batch keeps)
    const bool few = M <= KF_FEW_ROWS && !ragged;
    for (int S = 2; split && rem && rem * S <= max_g && 2 * S <= nsb; S++) {
        const int n = (nsb + S - 1) / S, most = rounds ? nsb : n;
        const double part = rounds * cost(nsb, most) + KQ_PART_US[t] * tm * rem * S / cus, us = part + cost(n, most);
        if (few ? S > 4 : part + cost(2, 2) >= p.us) break;
        if (few ? S != 3 : us < p.us) {
            p.us = us;
            p.full = p.T - rem;
            p.S = S;
        }
    }
    p.us += 1.8;
    p.wide = fits && !few && (p.full > 0 ? nsb : (nsb + p.S - 1) / p.S) > longest;
    return p;
}

// `split`: the tiles of the last round may be split (KF_GEMM_NO_TAIL: never, a comparison knob)
KqPlan kq_plan(uint32_t ty, int M, int N, int K, bool split) {
    split = split && !kf_knob_on(KF_KNOB_GEMM_NO_TAIL);
    const int forced = ty == KF_TYPE_Q4_K && kf_knob_on(KF_KNOB_Q4K_KQ) ? (kf_knob(KF_KNOB_Q4K_KQ) ? 2 : 4) : kf_knob_or(KF_KNOB_KQ_TM, 0);
    if (forced) return kq_plan_tm(ty, forced == 1 || forced == 2 ? forced : 4, M, N, K, split);
    KqPlan best = kq_plan_tm(ty, 1, M, N, K, split);
    for (int tm = 2; tm <= 4; tm *= 2) {
        const KqPlan p = kq_plan_tm(ty, tm, M, N, K, split);
        if (p.us < best.us) best = p;
    }
    return best;
}

// Grouped: the tile height, and whether the tiles are cut into one range a CU (the height then by a slot's pairs) or run whole,
// by the cost at the slots' average share of the pairs: the counts are on the device. Cutting pays for the partial tiles'
// way through memory, a second launch and ranges of a few super-blocks, too much for small experts: layers of 512 columns
// 1024 -> 512 -> 1024 with 202 tokens on two of four 104 us cut, 44 whole (59 on the 64-row kernel in K halves that the
// ranges replaced); 8 of 1280 -> 768 with 209 tokens 74, 45 and 53. Large ones gain by it: 512 tokens on two of 8
// of 4096 -> 14336 599 us cut, 652 whole.
struct KqMoePlan {
    int tm;
    bool cut;
    double us;
};

KqMoePlan kq_moe_plan(int pairs, int n_slots, int N, int K, int forced, bool may_cut) {
    const int cus = kf_cu_count(), nsb = K / 256, slots = std::min(pairs, n_slots);
    const double avg = (double)pairs / n_slots;
    const int cut_tm = avg < 32 ? 1 : avg < 65 ? 2 : 4;
    constexpr double cut_us[3] = {8.0, 17.5, 18.4};  // the parts and the reduce launch
    KqMoePlan best{0, false, 1e30};
    for (int tm = 1; tm <= 4; tm *= 2) {
        if (forced && tm != (forced == 1 || forced == 2 ? forced : 4)) continue;
        const int t = tm >> 1;
        // tiles, and the 32-row parts of one (the empty ones are skipped): a slot's last tile is half full on average
        const double T = (double)((N + KQ_BN - 1) / KQ_BN) * slots * std::max(1.0, avg / (32 * tm) + 0.5);
        const double sb = 0.8 + 0.8 * std::min((double)tm, std::max(1.0, avg / 32 + 0.5));
        const double whole = std::ceil(T / cus) * (KQ_ROUND_US[t] + sb * nsb);
        if (whole < best.us) best = KqMoePlan{tm, false, whole};
        const double cut = KQ_ROUND_US[t] + sb * std::max(4.0, nsb * T / cus) + cut_us[t];
        if (may_cut && (forced || tm == cut_tm) && cut < best.us) best = KqMoePlan{tm, true, cut};
    }
    return best;
}

// The scratch's range area, null when the stream has none
KqWork kq_work(const KfSplit& split, int full, int S) {
    KqWork w{nullptr, nullptr, full, S};
    if (char* scr = split.get()) {
        w.desc = reinterpret_cast<KqDesc*>(scr + (size_t)KF_SPLIT_TICKETS * 4);
        w.part = reinterpret_cast<float*>(scr + (size_t)KF_SPLIT_TICKETS * 4 + KQ_DESC_BYTES);
    }
    return w;
}

template <uint32_t TY, int TM, bool MOE, bool WIDE>
hipError_t kq_run(int blocks, hipStream_t s, const uint8_t* w, int64_t row_bytes, const int8_t* xq, const _Float16* xa, const float* xd,
                  const float* bias, const float* res, float* y, int M, int N, int K, KqWork work, KqMoe moe) {
    const auto fn = gemm_kq_kernel<TY, TM, MOE, WIDE>;
    constexpr int bytes = KqGeo<TY, TM>::LDS + KQ_EPI;
    const hipError_t e = kf_raise_lds(reinterpret_cast<const void*>(fn), bytes);
    if (e != hipSuccess) return e;
    fn<<<blocks, KQ_THREADS, bytes, s>>>(w, row_bytes, xq, xa, xd, bias, res, y, M, N, K, work, moe);
    const int shared = MOE ? work.S : (blocks - work.full) / work.S;  // tiles that may have partial ones
    constexpr int RED = MOE ? 4 : 1;
    if (work.part) kq_reduce_kernel<TM, MOE, RED><<<shared * (TM * 16 / RED), KQ_THREADS, 0, s>>>(work, bias, res, moe.out_rows, y, M, N);
    return hipGetLastError();
}

}  // namespace

// Whether the product costs less than `us` on stream `s`, with the split scratch if it can have it. What no plan goes below comes first: the plan's search would cost the shortest
// products a noticeable part of their launch.
bool kf_gemm_kq_below(uint32_t ty, int M, int N, int K, double us, hipStream_t s, bool graph) {
    const double least = std::min(K / 256 * KQ_SB_US[0][0], 2.0 + 2 * KQ_SB_US[0][0]);  // unsplit, split
    if (1.8 + KQ_ROUND_US[0] + least >= us) return false;
    const KqPlan p = kq_plan(ty, M, N, K, true);
    if (p.us + (p.S > 1 ? 2.0 : 0.0) >= us) return false;  // the second launch's host work, which a short product does not hide
    return p.S == 1 || KfSplit::ready(s, graph) || kq_plan(ty, M, N, K, false).us < us;
}

// Host launcher, validated by the caller (kf_gemm_kq_ok; Q8K-kind activations in `act`); `graph`: under graph capture the
// product may use the graph slot of the split scratch
hipError_t kf_launch_gemm_kq(uint32_t ty, const void* w, int64_t row_bytes, const void* act, const float* bias, const float* res, float* y,
                             int M, int N, int K, hipStream_t s, bool graph) {
    const kf_act_offsets o = kf_act_layout((size_t)M, (size_t)K);
    const char* base = static_cast<const char*>(act);
    // whole rounds of the CUs, then the split tiles; these need the scratch, without it the plan is one of whole tiles (the split
    // plan's tile height run whole left 64 rows of 14336 -> 4096 on 16 or 32 blocks)
    KqPlan p = kq_plan(ty, M, N, K, true);
    std::optional<KfSplit> split;
    KqWork work{nullptr, nullptr, p.T, 1};
    if (p.S > 1) {
        work = kq_work(split.emplace(s, graph), p.full, p.S);
        if (!work.part) {
            p = kq_plan(ty, M, N, K, false);
            work = KqWork{nullptr, nullptr, p.T, 1};
        }
    }
    const int blocks = work.full + (p.T - work.full) * work.S;
    const auto* wb = static_cast<const uint8_t*>(w);
    const auto* xq = reinterpret_cast<const int8_t*>(base + o.q);
    const auto* xa = reinterpret_cast<const _Float16*>(base + o.xa);
    const auto* xd = reinterpret_cast<const float*>(base + o.d32);
#define KQ_GO(TY, TM, WIDE) return kq_run<TY, TM, false, WIDE>(blocks, s, wb, row_bytes, xq, xa, xd, bias, res, y, M, N, K, work, KqMoe{})
#define KQ_TMS(TY)                                                     \
    {                                                                  \
        if (p.tm == 1 && p.wide) KQ_GO(TY, 1, true);                   \
        if (p.tm == 1) KQ_GO(TY, 1, false);                            \
        if (p.tm == 2 && p.wide) KQ_GO(TY, 2, (TY != KF_TYPE_Q5_K));   \
        if (p.tm == 2) KQ_GO(TY, 2, false);                            \
        KQ_GO(TY, 4, false);                                           \
    }
    if (ty == KF_TYPE_Q4_K) KQ_TMS(KF_TYPE_Q4_K)
    if (ty == KF_TYPE_Q5_K) KQ_TMS(KF_TYPE_Q5_K)
    KQ_TMS(KF_TYPE_Q6_K)
#undef KQ_TMS
#undef KQ_GO
}

// Grouped (MoE) form on q4_K experts: `act` holds `pairs` activation rows in group order (slot s: rows
// offsets[s]..offsets[s + 1], device offsets), slot s multiplies w + s expert_bytes (N output columns; with w2,
// columns n_split.. from w2), output row p goes to y row out_rows[p] (nullable: p). Validated by the caller: K a
// multiple of 256, n_split a multiple of 256, 16-byte aligned matrices and rows.
hipError_t kf_launch_gemm_kq_moe(const void* w, const void* w2, int64_t expert_bytes, int64_t row_bytes, int n_split, const void* act, int pairs,
                                 int n_slots, const int32_t* offsets, const int32_t* out_rows, float* y, int N, int K, hipStream_t s) {
    const kf_act_offsets o = kf_act_layout((size_t)pairs, (size_t)K);
    const char* base = static_cast<const char*>(act);
    // KF_MOE_KQ = 0 / 1: 128- or 64-row tiles (a comparison knob); KF_GEMM_NO_TAIL: whole tiles, without the scratch (another)
    const int forced = kf_knob_on(KF_KNOB_MOE_KQ) ? (kf_knob(KF_KNOB_MOE_KQ) ? 2 : 4) : kf_knob_or(KF_KNOB_KQ_TM, 0);
    KqMoePlan p = kq_moe_plan(pairs, n_slots, N, K, forced, !kf_knob_on(KF_KNOB_GEMM_NO_TAIL));
    if (kf_knob_on(KF_KNOB_KQ_G)) p.cut = true;  // KF_KQ_G: the number of ranges (a third)
    std::optional<KfSplit> split;
    KqWork work{nullptr, nullptr, 0, 0};
    if (p.cut) {
        work = kq_work(split.emplace(s, true), 0, kq_max_ranges(p.tm, kf_cu_count()));
        if (!work.part) p = kq_moe_plan(pairs, n_slots, N, K, forced, false);
    }
    // whole tiles: as many blocks as there may be tiles
    if (!work.part) work.S = ((N + KQ_BN - 1) / KQ_BN) * (pairs / (32 * p.tm) + std::min(n_slots, pairs));
    const int G = work.S, tm = p.tm;
    const KqMoe moe{offsets, out_rows, static_cast<const uint8_t*>(w2), expert_bytes, n_slots, n_split};
#define KQ_GO(TM)                                                                                                                             \
    return kq_run<KF_TYPE_Q4_K, TM, true, (TM == 1)>(G, s, static_cast<const uint8_t*>(w), row_bytes, reinterpret_cast<const int8_t*>(base + o.q),      \
                                          reinterpret_cast<const _Float16*>(base + o.xa), reinterpret_cast<const float*>(base + o.d32),      \
                                          nullptr, nullptr, y, pairs, N, K, work, moe)
    if (tm == 1) KQ_GO(1);
    if (tm == 2) KQ_GO(2);
    KQ_GO(4);
#undef KQ_GO
}

// Tile GEMM on native q8_0 bytes, any width of whole blocks: y[m][n] = sum over 32-column groups g of
// (dx[m][g] dw[n][g]) I_g[m][n] (+ bias[n] + res[m][n]), I_g the exact int32 dot of the group's int8 values (dot_i8,
// crates/kf-quant/src/types/q8_0.rs:10-29). In place of the reference's unpack + KF8 GEMM
// (crates/kf-backend-cuda/src/kernels/kf8.cu:375-395).
//
// Arithmetic, per group and 32 x 32 tile: one v_mfma_i32_32x32x32_i8 (I_g), one v_mfma_f32_32x32x16_f16 with a single non-zero
// k slot (the outer product dx (x) dw of f16 scales, exact in f32), then a conversion and a multiply-add an output.
//
// What bounds it: those two vector instructions an output and group, 128 cycles a tile and group on a SIMD beside 64 of
// matrix work. So the schedule only has to keep the vector unit fed: eight waves (two a SIMD), each a column of TM 32 x 32
// tiles; a step is one tile and group, and its two MFMAs go with the conversions and multiply-adds of the step before, so
// both run at once and neither waits for the other. The LDS reads of a step are issued one step ahead, the loads of a
// later stage one or two a step.
//
// Tile: 32 TM x 256; K advances 128 columns (four groups) a stage through NST LDS buffers of activations [row][128]
// (16-byte chunk c at c ^ (row / 2 % 8), so the operand reads hit distinct banks), weights [row][176] (the 16-byte aligned
// window around the row's 136 bytes, which may start at any even byte: rows of an odd number of blocks need no
// alignment; 176 keeps 16 rows on distinct banks) and activation scales [row][4]. Columns past the row's end read as zero
// activations and zero scales.
//
// Sums: f32 over the range's groups; where that would be less exact than the products this one replaces, f32 over a few
// stages and from there into 64-bit totals (q8_ragged and Q8_LONG).
//
// Measured (MI355X, one product, with the tiles, split and form the plan picks; before: the 128 x 128 kernel, the 64-row
// small-batch kernel, or for rows that are not 16-byte aligned the multi-row product of kf_hip_gemv):
// 14336 -> 4096 at 2048 rows 359 -> 322 us, 128 rows 60 -> 36, 64 rows 30 -> 25 (4096 -> 14336: 370 -> 368 at 2048 rows, 30 ->
// 26 at 64); 4160 -> 6000 at 64 rows 226 -> 21, 16 rows 60 -> 17.
#include "kf_device.h"
#include "kf_host.h"
#include "kf_knobs.h"
#include "kf_layout.h"

#include <algorithm>
#include <optional>
#include <type_traits>

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef int v4i_a2 __attribute__((ext_vector_type(4), aligned(2)));

constexpr int Q8_BN = 256;     // eight waves of 32 columns
constexpr int Q8_G = 4;        // groups a stage
constexpr int Q8_WB = Q8_G * KF_Q8_0_BYTES;  // 136 weight bytes a row and stage
constexpr int Q8_PR = 11;      // 16-byte pieces of a row's window, the last one only padding
constexpr int Q8_WROW = Q8_PR * 16;
constexpr int Q8_OOB = 0x7fffff00;  // an offset past every buffer: reads as zero

constexpr int Q8_WAVES = 8, Q8_THREADS = 64 * Q8_WAVES;

template <int TM>
struct Q8Geo {
    static constexpr int BM = 32 * TM;
    static constexpr int A = 0, W = BM * 128, DX = W + Q8_BN * Q8_WROW, STAGE = DX + BM * 16;
    static constexpr int PAD = 1024;  // zeros: where the weight instructions past a stage's own write
    static constexpr int NST = 3 * STAGE + PAD <= 160 * 1024 ? 3 : 2;
    static constexpr int LDS = NST * STAGE + PAD;
    static constexpr int NA = BM * 128 / 1024, NW = Q8_BN * Q8_PR / 64, ND = BM * 4 / 64;  // DMA instructions a stage
    // and a wave: every wave issues the same number, so the waits can count
    static constexpr int CA = (NA + Q8_WAVES - 1) / Q8_WAVES, CW = (NW + Q8_WAVES - 1) / Q8_WAVES, CD = (ND + Q8_WAVES - 1) / Q8_WAVES;
    static constexpr int BATCH = CA + CW + CD, STEPS = Q8_G * TM, PER = (BATCH + STEPS - 1) / STEPS;
    static constexpr int R = TM * 16;
    static_assert(NW % Q8_WAVES != 0, "some instruction of every stage fills the pad");
};

// Tiles below `full` are a block each, the others S blocks each over S ranges of K, whose partial tiles ([slot][register]
// [thread]) q8_reduce_kernel adds
struct Q8Work {
    float* part;
    int full, S;
    int fold;  // stages (a power of two, less one) after which the f32 sums go into the 64-bit ones
};

// FOLD: the f32 sums go into 64-bit ones after every few stages (32- and 64-row tiles: taller ones have no registers for these)
template <int TM, bool FOLD>
__global__ void __launch_bounds__(Q8_THREADS, 2) gemm_q8_kernel(const uint8_t* __restrict__ w, int64_t row_bytes, const int8_t* __restrict__ xq,
                                                                          const float* __restrict__ xd32, const float* __restrict__ bias,
                                                                          const float* __restrict__ res, float* __restrict__ y, int M, int N, int K,
                                                                          Q8Work work) {
    using G = Q8Geo<TM>;
    extern __shared__ __align__(256) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, r32 = lane & 31;
    const int kg = K >> 5, nst = (kg + Q8_G - 1) / Q8_G;
    const int mt = (M + G::BM - 1) / G::BM;
    int t, s0 = 0, s1 = nst, slot = -1;
    if ((int)blockIdx.x >= work.full) {
        slot = blockIdx.x - work.full;
        const int tt = slot / work.S, sp = slot - tt * work.S;
        t = work.full + tt;
        s0 = nst * sp / work.S;
        s1 = nst * (sp + 1) / work.S;
    } else {
        // XCD order: XCD x (blocks go to the eight XCDs round-robin) takes a contiguous range of tiles, M fastest
        const int b = blockIdx.x;
        t = (work.full & 7) ? b : (b & 7) * (work.full >> 3) + (b >> 3);
    }
    s0 = __builtin_amdgcn_readfirstlane(s0);
    s1 = __builtin_amdgcn_readfirstlane(s1);
    const int tn = t / mt, m0 = (t - tn * mt) * G::BM, n0 = tn * Q8_BN;

    // the tile's weight rows, from the 16-byte piece row n0 starts in to the piece the last one ends in (reads stay inside
    // that piece's 16 bytes)
    const int64_t wb0 = (int64_t)n0 * row_bytes;
    const int wsh = (int)(wb0 & 15), wrows = min(N - n0, Q8_BN), arows = min(M - m0, G::BM);
    const kf_arsrc_t rw = kf_arsrc(w + (wb0 - wsh), (uint64_t)((wrows * row_bytes + wsh + 15) / 16 * 16));
    const kf_arsrc_t rx = kf_arsrc(xq + (int64_t)m0 * K, (uint64_t)arows * K);
    const kf_arsrc_t rd = kf_arsrc(xd32 + (int64_t)m0 * kg, (uint64_t)arows * kg * 4);

    // Instruction k of a wave's loads of stage st. A stage is 128 activation columns and 136 weight bytes, eight past a whole
    // number of 16-byte pieces, so the weight offsets repeat every two stages: they are kept for an even and an odd one.
    // Past the range the loads run with an empty buffer, past a row's end at an offset outside it: zeros without traffic.
    int va[G::CA], vw[2][G::CW], vd[G::CD];
#pragma unroll
    for (int k = 0; k < G::CA; k++) {
        const int i = wave + Q8_WAVES * k, row = 8 * i + (lane >> 3);
        va[k] = i < G::NA ? row * K + 16 * ((lane & 7) ^ ((row >> 1) & 7)) : Q8_OOB;
    }
#pragma unroll
    for (int k = 0; k < G::CW; k++) {
        const int i = wave + Q8_WAVES * k, q = 64 * i + lane, row = q / Q8_PR, piece = q - Q8_PR * row;
        const int start = row * (int)row_bytes + wsh;
        const bool in = (i < G::NW) & (piece < Q8_PR - 1);
        vw[0][k] = in ? (start & ~15) + 16 * piece : Q8_OOB;
        vw[1][k] = in ? ((start + 8) & ~15) + 16 * piece : Q8_OOB;
    }
#pragma unroll
    for (int k = 0; k < G::CD; k++) {
        const int i = wave + Q8_WAVES * k, e = 64 * i + lane;
        vd[k] = i < G::ND ? ((e >> 2) * kg + (e & 3)) * 4 : Q8_OOB;
    }
    const int acol = 16 * ((lane & 7) ^ ((lane >> 4) & 3) ^ (wave & 1 ? 4 : 0));
    auto dma = [&](auto oddc, int st, int k) __attribute__((always_inline)) {
        constexpr int odd = decltype(oddc)::value;
        uint8_t* buf = lds + (st % G::NST) * G::STAGE;
        uint8_t* pad = lds + G::NST * G::STAGE;
        auto off = [&](kf_arsrc_t r) __attribute__((always_inline)) {
            if (st >= s1) r[2] = 0;
            return r;
        };
        if (k < G::CA) {
            const int i = wave + Q8_WAVES * k;
            kf_adma16(off(rx), acol < K - st * 128 ? va[k] : Q8_OOB, st * 128, i < G::NA ? buf + G::A + i * 1024 : pad);
        } else if (k < G::CA + G::CW) {
            const int j = k - G::CA, i = wave + Q8_WAVES * j;
            kf_adma16(off(rw), vw[odd][j], st * Q8_WB - 8 * odd, i < G::NW ? buf + G::W + i * 1024 : pad);
        } else if (k < G::BATCH) {
            const int j = k - G::CA - G::CW, i = wave + Q8_WAVES * j;
            kf_adma4(off(rd), (lane & 3) < kg - st * Q8_G ? vd[j] : Q8_OOB, st * Q8_G * 4, i < G::ND ? buf + G::DX + i * 256 : pad);
        }
    };

    v16f acc[TM];
#pragma unroll
    for (int i = 0; i < TM; i++) acc[i] = v16f{};
    double tot[FOLD ? TM : 1][16] = {};
    const uint32_t a0 = kf_lds_addr(lds) + r32 * 128 + 16 * (half ^ ((r32 >> 1) & 7));
    const int wrow = wave * 32 + r32;
    const uint32_t w0 = kf_lds_addr(lds) + G::W + wrow * Q8_WROW;
    const int sh0 = wsh + wrow * (int)row_bytes;                // the window's shift before the stage's bytes
    const uint32_t hmask = half ? 0u : 0xffffu;

    auto aop = [&](uint32_t at, int g, int i) __attribute__((always_inline)) {
        return *reinterpret_cast<const __attribute__((address_space(3))) v4i*>(((at + a0) ^ (32u * g)) + i * 4096);
    };
    auto wop = [&](uint32_t at, int g) __attribute__((always_inline)) {
        return (v4i) * reinterpret_cast<const __attribute__((address_space(3))) v4i_a2*>(at + 34 * g + 2 + 16 * half);
    };
    auto wsc = [&](uint32_t at, int g, int st) __attribute__((always_inline)) {
        const uint32_t v = *reinterpret_cast<const __attribute__((address_space(3))) uint16_t*>(at + 34 * g);
        return v & (st * Q8_G + g < kg ? hmask : 0u);
    };

    // the step in hand and the one before it: the group dots and the scale products
    v16i I[2] = {v16i{}, v16i{}};
    v16f S[2] = {v16f{}, v16f{}};
    auto rescale = [&](int p, v16f& c) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; r++) c[r] = fmaf((float)I[p][r], S[p][r], c[r]);
    };

    // a stage of parity P, while the loads of stage st + NST - 1 are issued
    auto stage = [&](auto Pc, int st) __attribute__((always_inline)) {
        constexpr int P = decltype(Pc)::value;
        const uint32_t at = (st % G::NST) * G::STAGE;
        const uint32_t wat = w0 + at + ((sh0 + st * Q8_WB) & 15);
        float dx[TM][4];
#pragma unroll
        for (int i = 0; i < TM; i++) {
            // the scale operand's second half of k slots is zero (from the pad), not a copy: an infinite scale would meet
            // the weight side's zeros there
            const float4 d = *reinterpret_cast<const float4*>(lds + (half ? G::NST * G::STAGE : at + G::DX + (r32 + 32 * i) * 16));
            dx[i][0] = d.x;
            dx[i][1] = d.y;
            dx[i][2] = d.z;
            dx[i][3] = d.w;
        }
        v4i b = wop(wat, 0), a = aop(at, 0, 0);
        uint32_t ws = wsc(wat, 0, st);
        auto step = [&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            if constexpr (k < G::STEPS) {
                constexpr int g = k / TM, i = k % TM, gn = (k + 1) / TM, in = (k + 1) % TM;
                v4i an = a, bn = b;
                uint32_t wsn = ws;
                if constexpr (k + 1 < G::STEPS) {
                    an = aop(at, gn, in);
                    if constexpr (in == 0) {
                        bn = wop(wat, gn);
                        wsn = wsc(wat, gn, st);
                    }
                }
#pragma unroll
                for (int e = 0; e < G::PER; e++) dma(std::integral_constant<int, (P + G::NST - 1) & 1>{}, st + G::NST - 1, G::PER * k + e);
                __builtin_amdgcn_sched_barrier(0);
                // (dx, 0) in one truncating conversion: dx is f16-rounded already
                const v4i xs = {__builtin_bit_cast(int, __builtin_amdgcn_cvt_pkrtz(dx[i][g], 0.0f)), 0, 0, 0}, wv = {(int)ws, 0, 0, 0};
                I[k & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, v16i{}, 0, 0, 0);
                S[k & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, xs), __builtin_bit_cast(v8h, wv), v16f{}, 0, 0, 0);
                rescale((k + 1) & 1, acc[(i + TM - 1) % TM]);
                a = an;
                b = bn;
                ws = wsn;
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
        step(std::integral_constant<int, 4>{});
        step(std::integral_constant<int, 5>{});
        step(std::integral_constant<int, 6>{});
        step(std::integral_constant<int, 7>{});
        step(std::integral_constant<int, 8>{});
        step(std::integral_constant<int, 9>{});
        step(std::integral_constant<int, 10>{});
        step(std::integral_constant<int, 11>{});
        step(std::integral_constant<int, 12>{});
        step(std::integral_constant<int, 13>{});
        step(std::integral_constant<int, 14>{});
        step(std::integral_constant<int, 15>{});
    };
    using even = std::integral_constant<int, 0>;
    using odd = std::integral_constant<int, 1>;
    // the range's stages, by the parity of their number
    auto first = [&](auto Pc) __attribute__((always_inline)) {
        constexpr int P = decltype(Pc)::value;
#pragma unroll
        for (int k = 0; k < G::BATCH; k++) dma(std::integral_constant<int, P>{}, s0, k);
        if constexpr (G::NST == 3) {
#pragma unroll
            for (int k = 0; k < G::BATCH; k++) dma(std::integral_constant<int, 1 - P>{}, s0 + 1, k);
        }
    };
    auto one = [&](auto Pc, int st) __attribute__((always_inline)) {
        // stage st has landed once only the later stages' loads are in flight; the barrier also frees the buffer of stage
        // st - 1, which the next loads take
        __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"((G::NST - 2) * G::BATCH) : "memory");
        __syncthreads();
        stage(Pc, __builtin_amdgcn_readfirstlane(st));
        // (the last step of the stage still waits for its rescale: it goes into the next sum)
        if constexpr (FOLD)
            if (((st - s0 + 1) & work.fold) == 0) {
#pragma unroll
                for (int i = 0; i < TM; i++) {
#pragma unroll
                    for (int r = 0; r < 16; r++) tot[i][r] += (double)acc[i][r];
                    acc[i] = v16f{};
                }
            }
    };
    int st = s0;
    if (s0 & 1) {
        first(odd{});
        one(odd{}, st++);
    } else {
        first(even{});
    }
#pragma unroll 1
    for (; st + 1 < s1; st += 2) {
        one(even{}, st);
        one(odd{}, st + 1);
    }
    if (st < s1) one(even{}, st);
    rescale(1, acc[TM - 1]);  // the last step's (an even number of them a stage)
    if constexpr (FOLD) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][r] = (float)(tot[i][r] + (double)acc[i][r]);
    }

    const int n = n0 + wave * 32 + r32;
    if (slot >= 0) {
        float* pp = work.part + (size_t)slot * G::R * Q8_THREADS + tid;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) pp[(i * 16 + r) * Q8_THREADS] = acc[i][r];
        return;
    }
    if (n >= N) return;
    const float bn = bias ? bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int m = m0 + i * 32 + (r & 3) + 8 * (r >> 2) + 4 * half;
            if (m >= M) continue;
            const int64_t o = (int64_t)m * N + n;
            y[o] = acc[i][r] + bn + (res ? res[o] : 0.0f);
        }
}

// Adds the S partial tiles of each split tile, eight at a time as a tree, or in 64 bits for a FOLD product (1-2.5 us more a
// launch), with bias and residual: one (register, block) slice a block, one thread an output
template <int TM, bool FOLD>
__global__ void __launch_bounds__(Q8_THREADS) q8_reduce_kernel(Q8Work work, const float* __restrict__ bias, const float* __restrict__ res,
                                                                            float* __restrict__ y, int M, int N) {
    using G = Q8Geo<TM>;
    const int tt = blockIdx.x / G::R, e = blockIdx.x - tt * G::R, tid = threadIdx.x, wave = tid >> 6;
    const int mt = (M + G::BM - 1) / G::BM, t = work.full + tt, tn = t / mt;
    const int r = e & 15;
    const int m = (t - tn * mt) * G::BM + (e >> 4) * 32 + (r & 3) + 8 * (r >> 2) + 4 * ((tid >> 5) & 1);
    const int n = tn * Q8_BN + wave * 32 + (tid & 31);
    if (m >= M || n >= N) return;
    const float* p = work.part + ((size_t)tt * work.S * G::R + e) * Q8_THREADS + tid;
    std::conditional_t<FOLD, double, float> v = 0.0f;
    for (int k = 0; k < work.S; k += 8) {
        float a[8];
#pragma unroll
        for (int u = 0; u < 8; u++) a[u] = k + u < work.S ? p[(size_t)(k + u) * G::R * Q8_THREADS] : 0.0f;
        if constexpr (FOLD) {
#pragma unroll
            for (int u = 0; u < 8; u++) v += (double)a[u];
        } else {
            v += ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
        }
    }
    const int64_t o = (int64_t)m * N + n;
    y[o] = (float)v + (bias ? bias[n] : 0.0f) + (res ? res[o] : 0.0f);
}

// Widths that are no whole number of 128-column steps. Before this kernel they ran the multi-row product, whose 64 lanes'
// sums meet in a tree (7e-8 from the 64-bit result at 33-130 groups, 9e-8 at 449, against 2e-7 and 3.8e-7 for one f32 sum
// over all of them), so here every second stage goes into the 64-bit sums (6-7e-8) and tiles without room for these are
// left out: 2048 rows of 14368 -> 4096 take 472 us instead of 352, 300 rows 93 instead of 84, and 56 and 4.3 ms on the
// multi-row product.
bool q8_ragged(int K) { return K % (32 * Q8_G) != 0; }

// Other widths had one f32 sum over all groups, or over half of them and less where the older kernels split K. So only
// sums of more stages than half of 14336 columns go into 64-bit ones here, every eight stages (3% of the time at 64 rows of 4096 ->
// 14336, 1e-7 where one sum over 14336 columns has 3.8e-7); 128-row tiles keep the one sum.
constexpr int Q8_LONG = 56;

template <int TM, bool FOLD = false>
hipError_t q8_run(const uint8_t* w, int64_t row_bytes, const int8_t* xq, const float* xd, const float* bias, const float* res, float* y, int M, int N,
                  int K, int S, float* part, hipStream_t s) {
    using G = Q8Geo<TM>;
    if constexpr (TM <= 2 && !FOLD)
        if (q8_ragged(K) || (K / 32 + Q8_G - 1) / Q8_G > Q8_LONG * S) return q8_run<TM, true>(w, row_bytes, xq, xd, bias, res, y, M, N, K, S, part, s);
    const auto fn = gemm_q8_kernel<TM, FOLD>;
    const hipError_t e = kf_raise_lds(reinterpret_cast<const void*>(fn), G::LDS);
    if (e != hipSuccess) return e;
    const int T = ((N + Q8_BN - 1) / Q8_BN) * ((M + G::BM - 1) / G::BM), rem = T % kf_cu_count();
    const int fold = q8_ragged(K) ? 1 : 7;
    Q8Work work{nullptr, T, 1, fold};
    if (part) work = Q8Work{part, T - rem, S, fold};
    const int split = T - work.full;
    fn<<<work.full + split * work.S, Q8_THREADS, G::LDS, s>>>(w, row_bytes, xq, xd, bias, res, y, M, N, K, work);
    if (split) q8_reduce_kernel<TM, FOLD><<<split * G::R, Q8_THREADS, 0, s>>>(work, bias, res, y, M, N);
    return hipGetLastError();
}

// Cost model of a launch (MI355X, us; least squares over 4-2048 rows at 2048 -> 6144, 2080 -> 1000, 4096 -> 4096, 4160 -> 6000,
// 4096 -> 14336 and 14336 -> 4096, rms 4-7%): a launch, a round of the CUs (a block's first loads and its stores), a
// 128-column stage, and the partial tiles' way through memory where tiles are split. The tile height is the cheapest by it: 32
// rows of 14336 -> 4096 took 23 / 26 / 34 us with 32 / 64 / 128-row tiles, 2048 rows 603 / 392 / 318. A product without the
// scratch plans whole tiles: a split plan's tile height run whole left 64 rows on 16 blocks.
constexpr int Q8_BMS[3] = {32, 64, 128};
constexpr double Q8_LAUNCH_US[3] = {3.5, 1.0, 0.0}, Q8_ROUND_US[3] = {2.0, 3.9, 5.0}, Q8_ST_US[3] = {1.37, 1.80, 2.86}, Q8_PART_US[3] = {4.9, 7.3, 8.7};

struct Q8Plan {
    int v, S;
    double us;
};

constexpr size_t Q8_PART_ROOM = std::min(KF_SPLIT_SCRATCH, KF_SPLIT_SPARE) - (size_t)KF_SPLIT_TICKETS * 4;

Q8Plan q8_plan_v(int v, int M, int N, int K, bool split) {
    const int cus = kf_cu_count(), nst = (K / 32 + Q8_G - 1) / Q8_G;
    const int T = ((N + Q8_BN - 1) / Q8_BN) * ((M + Q8_BMS[v] - 1) / Q8_BMS[v]), rem = T % cus;
    Q8Plan p{v, 1, 0.0};
    double tail = rem ? Q8_ROUND_US[v] + Q8_ST_US[v] * nst : 0.0;
    for (int S = 2; split && rem && rem * S <= cus && 2 * S <= nst; S++) {
        if ((size_t)rem * S * Q8_BMS[v] * Q8_BN * 4 > Q8_PART_ROOM) break;
        const double part = Q8_ROUND_US[v] + Q8_PART_US[v] * rem * S / cus, us = part + Q8_ST_US[v] * ((nst + S - 1) / S);
        if (part + 2 * Q8_ST_US[v] >= tail) break;
        if (us < tail) {
            tail = us;
            p.S = S;
        }
    }
    p.us = Q8_LAUNCH_US[v] + (T / cus) * (Q8_ROUND_US[v] + Q8_ST_US[v] * nst) + tail;
    return p;
}

// `split`: the tiles of the last round may be split (KF_GEMM_NO_TAIL: never, a comparison knob)
Q8Plan q8_plan(int M, int N, int K, bool split) {
    split = split && !kf_knob_on(KF_KNOB_GEMM_NO_TAIL);
    const int forced = kf_knob_or(KF_KNOB_Q8_V, -1);
    if (forced >= 0 && forced < 3) return q8_plan_v(forced, M, N, K, split);
    Q8Plan best = q8_plan_v(0, M, N, K, split);
    for (int v = 1; v < (q8_ragged(K) ? 2 : 3); v++) {
        const Q8Plan p = q8_plan_v(v, M, N, K, split);
        if (p.us < best.us) best = p;
    }
    return best;
}

}  // namespace

// Whether the product costs less than `us` on stream `s`, with the split scratch if it can have it. What no plan goes below comes first: the plan's search would cost the shortest
// products a noticeable part of their launch.
bool kf_gemm_q8_below(int M, int N, int K, double us, hipStream_t s, bool graph) {
    const int nst = (K / 32 + Q8_G - 1) / Q8_G;
    bool may = false;
    for (int v = 0; v < 3; v++) may |= Q8_LAUNCH_US[v] + Q8_ROUND_US[v] + std::min(nst * Q8_ST_US[v], 2.0 + 2 * Q8_ST_US[v]) < us;  // unsplit, split
    if (!may) return false;
    const Q8Plan p = q8_plan(M, N, K, true);
    if (p.us + (p.S > 1 ? 2.0 : 0.0) >= us) return false;  // the second launch's host work, which a short product does not hide
    return p.S == 1 || KfSplit::ready(s, graph) || q8_plan(M, N, K, false).us < us;
}

// Host launcher: K a multiple of 32, Q8_0-kind activations in `act`, weights 16-byte aligned; `graph`: under graph capture
// the product may use the graph slot of the split scratch
hipError_t kf_launch_gemm_q8(const void* w, int64_t row_bytes, const void* act, const float* bias, const float* res, float* y, int M, int N, int K,
                             hipStream_t s, bool graph) {
    const kf_act_offsets o = kf_act_layout((size_t)M, (size_t)K);
    const char* base = static_cast<const char*>(act);
    const auto* xq = reinterpret_cast<const int8_t*>(base + o.q);
    const auto* xd = reinterpret_cast<const float*>(base + o.d32);
    const auto* wb = static_cast<const uint8_t*>(w);
    Q8Plan p = q8_plan(M, N, K, true);
    std::optional<KfSplit> split;
    float* part = nullptr;
    if (p.S > 1) {
        if (char* scr = split.emplace(s, graph).get())
            part = reinterpret_cast<float*>(scr + (size_t)KF_SPLIT_TICKETS * 4);
        else
            p = q8_plan(M, N, K, false);
    }
    if (p.v == 0) return q8_run<1>(wb, row_bytes, xq, xd, bias, res, y, M, N, K, p.S, part, s);
    if (p.v == 1) return q8_run<2>(wb, row_bytes, xq, xd, bias, res, y, M, N, K, p.S, part, s);
    return q8_run<4>(wb, row_bytes, xq, xd, bias, res, y, M, N, K, p.S, part, s);
}

/*
 * gemm_f32_split.h - block-format x fp32 products without rounding to 16 bits, on the matrix cores:
 *
 *   Y[t*ldy + r] = sum_k X[t*ldx + k] * decode(W)[r][k]      X fp32, Y fp32, fp32 accumulate
 *
 * The weights are never decoded to memory and never rounded: their codes are integers of at most 8 bits, exact in fp16,
 * and where code * sub-block scale is an integer of at most 11 bits (kFold) that product is exact too. An activation goes
 * in as two fp16 numbers: with the token scaled by a power of two so that its largest element lies in [2^14, 2^15),
 * hi = fp16(x) and lo = fp16(x - hi) are within 2^-23 of x (23 bits; three quarters of all fp32 numbers are kept whole), for
 * elements below 2^-16 of the token's largest within 2^-39 of that: lo's subnormals end there. v_mfma_f32_32x32x16_f16 then does the work twice, at sixteen times the rate of the fp32 matrix
 * instructions; block scales are applied to the sums in fp32. A minimum (Q4_K, Q5_K, Q2_K) is a product of its 6-bit
 * integers with the sub-blocks' sums of activations (summed in 64 bits, two fp16 numbers as well), one more instruction per
 * 32 x 32 x 256.
 *
 * Launches of a call:
 *   f32_token_exp   the power of two of every token (kF32NotFinite for one that holds an infinity or a NaN); rows of up to
 *                   2048 elements, or up to 4096 in a small X: one launch for both
 *   f32_split       X -> operand fragments of 1 KB (lane l: token l & 31, elements 8 (l >> 5) ..), so that the product's
 *                   requests and LDS reads are linear; the sub-block sums the same way
 *   gemm_f32_split  four waves per workgroup, each 32 TN rows x 32 TM tokens; a wave copies a super-block of its rows to
 *                   an image of its own by load-to-LDS requests, the fragments of 32 elements come into a ring of
 *                   stages that the waves share, one barrier per stage. K is divided over workgroups where the tiles alone
 *                   do not fill the chip; every part writes its sums to the workspace
 *   f32_finish      adds the parts in order, takes the power of two back; tokens that are not finite get what
 *                   the plain fp32 sum gives: infinities and NaN
 *
 * What bounds it: a wave multiplies for a third of its time, the rest are waits at the stage barrier and for the matrix
 * unit's results, with two waves per SIMD to fill them (Q4_K 512 tokens 14336 x 4096: 438 TFLOP/s counted once, 876 of
 * matrix instructions). Tried and without effect: two stages ahead instead of four, codes made fp16 by two instructions
 * instead of four, the next operands made between the matrix instructions instead of ahead of them (4 % at 14336 rows).
 * Measured, us, before (weights decoded to fp32 in the workspace, the library's fp32 product) / now, Q4_K: 8 tokens
 * 4096 x 4096 38 / 16, 64 tokens 45 / 27, 320 tokens 114 / 49, 320 tokens 14336 x 4096 389 / 112 and 4096 x 14336 352 / 101,
 * 2048 tokens 4096 x 4096 478 / 168; Q6_K 320 tokens 110 / 58, 377 / 150, 349 / 141. Error against 64 bits, before / now:
 * 320 tokens Q4_K K = 4096 1.1e-6 / 1.9e-7, K = 14336 2.1e-6 / 2.1e-7, Q6_K 1.1e-6 / 1.8e-7, 2.1e-6 / 3.2e-7; 8 tokens
 * 5.8e-7 / 2.0e-7.
 */
#ifndef QLIN_GEMM_F32_SPLIT_H
#define QLIN_GEMM_F32_SPLIT_H

#include "gemm_image_formats.h"
#include "qlin_codecs_ext.h"
#include "qlin_internal.h"

namespace qlin {

using namespace kq;

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kStageBytes = 4096; /* 32 tokens x 32 elements: [hi, lo][step of 16][64 lanes][16 bytes] */

QLIN_INL half8 join(half2v a, half2v b, half2v c, half2v d) { return half8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]}; }
QLIN_INL half2v as_half2(uint32_t v) { return __builtin_bit_cast(half2v, v); }
QLIN_INL half2v both(float f) { return half2v{(_Float16)f, (_Float16)f}; }
/* codes (bytes) less OFFSET as fp16: 1024 + q has q in its low byte */
template <int OFFSET> QLIN_INL half8 codes_f16(uint32_t a, uint32_t b) {
    constexpr uint32_t hi = 0x64646464u, lo_pair = 0x07010700u, hi_pair = 0x07030702u;
    const half2v o = both(-1024.0f - OFFSET);
    return join(as_half2(__builtin_amdgcn_perm(hi, a, lo_pair)) + o, as_half2(__builtin_amdgcn_perm(hi, a, hi_pair)) + o,
                as_half2(__builtin_amdgcn_perm(hi, b, lo_pair)) + o, as_half2(__builtin_amdgcn_perm(hi, b, hi_pair)) + o);
}
/* code * scale * 2^-14 of codes without an offset, scale below 64: a code alone is the subnormal q * 2^-24, and its product
 * with scale * 2^10 an integer of at most 11 bits in units of 2^-14, exact */
constexpr float kFoldUnit = 16384.0f;
QLIN_INL half8 codes_scaled_f16(uint32_t a, uint32_t b, float scale) {
    constexpr uint32_t lo_pair = 0x0C010C00u, hi_pair = 0x0C030C02u; /* 0C: a zero byte */
    const half2v f = both(scale * 1024.0f);
    return join(as_half2(__builtin_amdgcn_perm(0u, a, lo_pair)) * f, as_half2(__builtin_amdgcn_perm(0u, a, hi_pair)) * f,
                as_half2(__builtin_amdgcn_perm(0u, b, lo_pair)) * f, as_half2(__builtin_amdgcn_perm(0u, b, hi_pair)) * f);
}

/* kFold: block(hdr) * iscale<U>(hdr) is the factor of a lane's elements, iscale an integer with |iscale * code| <= 2048;
 * min_factor(hdr) and min_bytes(hdr, half, a, b): the integers of the minimum, of sub-blocks 0 .. 7 (32 elements each) or
 * 8 half .. + 7 (16 each) */
template <class F> struct Fold {
    static constexpr bool kFold = false;
    template <int U> static QLIN_INL float iscale(const typename F::Hdr &) { return 0.0f; }
    static QLIN_INL float block(const typename F::Hdr &) { return 0.0f; }
};
struct FoldK4 {
    static constexpr bool kFold = true;
    template <int U> static QLIN_INL float iscale(const HdrK4 &h) { return ubyte_f32<U & 3>(U < 4 ? h.sc_lo : h.sc_hi); }
    static QLIN_INL float block(const HdrK4 &h) { return h.d; }
    static QLIN_INL float min_factor(const HdrK4 &h) { return h.dmin; }
    static QLIN_INL void min_bytes(const HdrK4 &h, int, uint32_t &a, uint32_t &b) { a = h.mn_lo; b = h.mn_hi; }
};
template <> struct Fold<TQ4K> : FoldK4 {};
template <> struct Fold<TQ5K> : FoldK4 {};
template <> struct Fold<TQ2K> {
    static constexpr bool kFold = true;
    template <int U> static QLIN_INL float iscale(const TQ2K::Hdr &h) { return (float)((h.sc[U >> 1] >> (16 * (U & 1))) & 15u); }
    static QLIN_INL float block(const TQ2K::Hdr &h) { return h.d; }
    static QLIN_INL float min_factor(const TQ2K::Hdr &h) { return h.dmin; }
    static QLIN_INL void min_bytes(const TQ2K::Hdr &h, int half, uint32_t &a, uint32_t &b) { /* of the first scale group's header */
        a = ((half ? h.sc[2] : h.sc[0]) >> 4) & 0x0F0F0F0Fu;
        b = ((half ? h.sc[3] : h.sc[1]) >> 4) & 0x0F0F0F0Fu;
    }
};
template <> struct Fold<TQ3K> {
    static constexpr bool kFold = true;
    template <int U> static QLIN_INL float iscale(const TQ3K::Hdr &h) { return ubyte_f32<2 * (U & 1)>(h.sc[U >> 1]) - 32.0f; }
    static QLIN_INL float block(const TQ3K::Hdr &h) { return h.d; }
};
template <> struct Fold<TIQ3S> {
    static constexpr bool kFold = true;
    template <int U> static QLIN_INL float iscale(const TIQ3S::Hdr &h) { return (float)(1u + 2u * ((h.sc >> (4 * U)) & 15u)); }
    static QLIN_INL float block(const TIQ3S::Hdr &h) { return h.d; }
};
template <> struct Fold<TIQ2XXS> { /* 0.25 d (0.5 + s) = 0.125 d (1 + 2 s) */
    static constexpr bool kFold = true;
    template <int U> static QLIN_INL float iscale(const TIQ2XXS::Hdr &h) { return (float)(1u + 2u * (uint32_t)(h.row[TIQ2XXS::at(U) + 7] >> 4)); }
    static QLIN_INL float block(const TIQ2XXS::Hdr &h) { return 0.5f * h.d; }
};

QLIN_INL f32x16 mma16(half8 a, half8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
template <int N> QLIN_INL void wait_and_meet() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory");
}

/* TM x 32 tokens by TN x 32 rows per wave. TN = 2 reads a fragment from LDS once for two matrix instructions; the formats
 * with large blocks take one row tile so that two workgroups fit a compute unit's LDS */
template <class F, int TM> struct SplitShape {
    static constexpr int TN = F::kPieces <= 11 ? 2 : 1;
    static constexpr int kRows = 4 * 32 * TN, kTokens = 32 * TM;
    static constexpr int kStage = TM * kStageBytes;
    static constexpr int kSums = F::kHasMin ? TM * (F::kGroup16 ? 2 : 1) : 0; /* KB, and requests, of a super-block's sums */
    static constexpr int kImage = TN * 32 * F::kPieces * 16, kWReq = (kImage + 1023) / 1024;
    /* stages of the ring: what is left of half a compute unit's LDS, at most six, and one of them is being read */
    static constexpr int kFixed = kSums * 1024 + 4 * kImage + 4 * F::kTable;
    static constexpr int kRing = (80 * 1024 - kFixed) / kStage < 6 ? (80 * 1024 - kFixed) / kStage : 6, kAhead = kRing - 1;
    static constexpr int kLds = kRing * kStage + kFixed;
    static_assert(kAhead >= 3, "the order of the requests is counted on");
    /* Requests that a wave has made since those of group U's stage, in their order: per group its stage, behind that of group
     * 0 the sums and behind that of group 6 the next image. Group 0 also waits for the image */
    static constexpr int since(int u) {
        if (u == 0) return TM;
        return (kAhead - 1) * TM + (u <= kAhead ? kSums : 0) + (u + 2 <= kAhead || u == 7 ? kWReq : 0);
    }
};

struct SplitArgs {
    const uint8_t *W, *frags, *sums;
    float *out;                 /* parts: [part][n_tok][n_rows]; one part: Y */
    const int *token_exp;
    int n_rows, n_tok, n_sb, parts, row_tiles, token_tiles, ldo;
};

template <class F, int TM>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
gemm_f32_split_kernel(SplitArgs p) {
    using S = SplitShape<F, TM>;
    using D = Fold<F>;
    constexpr int TN = S::TN, kRow = F::kPieces * 16, kSteps = F::kGroup16 ? 2 : 1; /* scales per 32 elements */
    constexpr uint32_t kPastEnd = 0xFFFFFFF0u; /* an offset outside every buffer: the request returns zeros */
    extern __shared__ __attribute__((aligned(1024))) uint8_t split_lds[];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 31, half = lane >> 5;
    /* items with the token tile fastest, an eighth of them in a row on each XCD (workgroups go to the XCDs in turn), so
     * that the token tiles of one row tile find its blocks in their L2 */
    const int items = p.row_tiles * p.token_tiles * p.parts, per_xcd = (items + 7) >> 3;
    const int item = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || item >= items) return;
    auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); }; /* (divisions run in vector registers) */
    const int rest = uniform(item / p.token_tiles), token_tile = item - rest * p.token_tiles;
    const int part = uniform(rest / p.row_tiles), row_tile = rest - part * p.row_tiles;
    const int sb0 = uniform((int)((unsigned)(p.n_sb * part) / (unsigned)p.parts)), sb1 = uniform((int)((unsigned)(p.n_sb * (part + 1)) / (unsigned)p.parts));
    const int row0 = uniform(row_tile * S::kRows + wv * (32 * TN));
    const int rows_here = uniform(max(0, min(32 * TN, p.n_rows - row0)));
    const uint32_t row_bytes = (uint32_t)p.n_sb * F::kBlock;

    uint8_t *stages = split_lds, *sums = stages + S::kRing * S::kStage, *img = sums + S::kSums * 1024 + wv * S::kImage;
    uint32_t *tab = reinterpret_cast<uint32_t *>(split_lds + S::kRing * S::kStage + S::kSums * 1024 + 4 * S::kImage);
    const uint32_t stages_at = (uint32_t)(uintptr_t)(lds_void *)stages, sums_at = (uint32_t)(uintptr_t)(lds_void *)sums,
                   img_at = (uint32_t)(uintptr_t)(lds_void *)img;

    /* weights: as in the few-token kernel, piece 64 q + lane of the image is part id % kPieces of row id / kPieces */
    /* Past the part's last super-block the requests are made all the same, so that they stay countable, and touch no memory: a
     * buffer of no bytes, read from its start - every offset is past its end, whichever way a scalar offset is counted */
    auto w_rsrc = [&](bool any) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(p.W) + (size_t)(rows_here ? row0 : 0) * row_bytes, 0,
                                                 any ? (int)(rows_here * row_bytes) : 0, 0x00020000);
    };
    uint32_t w_off[S::kWReq];
#pragma unroll
    for (int q = 0; q < S::kWReq; q++) {
        const uint32_t id = 64u * q + lane, row = id / F::kPieces, piece = id % F::kPieces, src = F::piece_src(piece);
        w_off[q] = row < (uint32_t)rows_here && src != kNoPiece ? row * row_bytes + src : kPastEnd;
    }
    const bool w_last = 64 * (S::kWReq - 1) + lane < S::kImage / 16;
    auto request_w = [&](int sb) {
        const uint32_t at = sb < sb1 ? (uint32_t)sb * (uint32_t)F::kBlock : 0u;
#pragma unroll
        for (int q = 0; q < S::kWReq; q++)
            if (q + 1 < S::kWReq || w_last) request16(img_at + 1024u * q, w_off[q], w_rsrc(sb < sb1), at);
    };
    /* fragments: wave w brings the w-th KB of each 32 tokens' stage; the last stage is asked for again past the end */
    const int n_groups = 8 * p.n_sb, last_group = 8 * sb1 - 1;
    const size_t tile_bytes = (size_t)n_groups * kStageBytes;
    __amdgpu_buffer_rsrc_t x_rsrc[TM];
#pragma unroll
    for (int m = 0; m < TM; m++)
        x_rsrc[m] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(p.frags) + (size_t)(token_tile * TM + m) * tile_bytes, 0, (int)tile_bytes,
                                                      0x00020000);
    const uint32_t x_off = 1024u * wv + 16u * lane;
    auto request_x = [&](int group, int slot) {
        const uint32_t at = (uint32_t)min(group, last_group) * (uint32_t)kStageBytes;
#pragma unroll
        for (int m = 0; m < TM; m++) request16(stages_at + (uint32_t)(slot * S::kStage + m * kStageBytes) + 1024u * wv, x_off, x_rsrc[m], at);
    };
    constexpr int kSumsPer = F::kGroup16 ? 2048 : 1024;
    auto request_sums = [&](int sb) { /* every wave the whole of it: the requests stay countable */
        const uint8_t *src = p.sums + ((size_t)token_tile * TM * p.n_sb + sb) * kSumsPer;
#pragma unroll
        for (int q = 0; q < S::kSums; q++) {
            const int m = q / (kSumsPer / 1024), within = q % (kSumsPer / 1024);
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<uint8_t *>(src) + (size_t)m * p.n_sb * kSumsPer + 1024 * within, 0, 1024, 0x00020000);
            request16(sums_at + 1024u * q, 16u * lane, r, 0);
        }
    };

    request_w(sb0);
    for (int g = 0; g < S::kAhead; g++) request_x(8 * sb0 + g, g);
    if constexpr (F::kTable > 0)
        for (int i = threadIdx.x; i < F::kTable; i += blockDim.x) tab[i] = F::table()[i];

    f32x16 acc[TM][TN];
#pragma unroll
    for (int m = 0; m < TM; m++)
#pragma unroll
        for (int n = 0; n < TN; n++) acc[m][n] = f32x16{};

    int slot = 0; /* of the group at hand in the ring */
    for (int sb = sb0; sb < sb1; sb++) {
        typename F::Hdr hdr[TN][kSteps];
        f32x16 c[TM][TN]; /* kFold: the super-block's sums */
        half8 w[2][TN][2]; /* of the group at hand and, made while its products run, the next one's */
        float scale[2][TN][kSteps];
        each<8>([&](auto group) {
            constexpr int U = decltype(group)::value;
            wait_and_meet<S::since(U)>();
            request_x(8 * sb + U + S::kAhead, slot == 0 ? S::kAhead : slot - 1); /* its place was read a group ago, and all waves have met since */
            if constexpr (U == 0) {
                request_sums(sb);
#pragma unroll
                for (int n = 0; n < TN; n++)
#pragma unroll
                    for (int s = 0; s < kSteps; s++) hdr[n][s] = F::header(img + (32 * n + j) * kRow, 2 * s);
            }
            half8 x[TM][2][2]; /* [hi, lo][step] */
#pragma unroll
            for (int m = 0; m < TM; m++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    x[m][q >> 1][q & 1] = *reinterpret_cast<const half8 *>(stages + slot * S::kStage + m * kStageBytes + 1024 * q + 16 * lane);
            auto weights = [&](auto of, half8 (&to)[TN][2], float (&sc)[TN][kSteps]) {
                constexpr int V = decltype(of)::value;
#pragma unroll
                for (int n = 0; n < TN; n++) {
                    const uint8_t *row = img + (32 * n + j) * kRow;
#pragma unroll
                    for (int s = 0; s < 2; s++) {
                        uint32_t a, b;
                        F::template codes<V>(row, 2 * s + half, tab, a, b);
                        const typename F::Hdr &h = hdr[n][s % kSteps];
                        if constexpr (D::kFold && F::kOffset == 0) to[n][s] = codes_scaled_f16(a, b, D::template iscale<V>(h));
                        else to[n][s] = codes_f16<F::kOffset>(a, b);
                        if constexpr (D::kFold && F::kOffset != 0) {
                            const _Float16 f = (_Float16)D::template iscale<V>(h);
                            to[n][s] *= half8{f, f, f, f, f, f, f, f};
                        }
                        if constexpr (!D::kFold) sc[n][s % kSteps] = F::template scale<V>(h, 2 * s);
                    }
                }
            };
            if constexpr (U == 0) weights(group, w[0], scale[0]);
            if constexpr (U < 7) weights(std::integral_constant<int, U + 1>{}, w[(U + 1) & 1], scale[(U + 1) & 1]);
            if constexpr (U == 6) { /* that was the last of the image: the next super-block's takes its place */
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                request_w(sb + 1);
            }
            constexpr int P = U & 1;
#pragma unroll
            for (int n = 0; n < TN; n++)
#pragma unroll
                for (int m = 0; m < TM; m++) {
                    if constexpr (D::kFold) {
                        f32x16 v = U == 0 ? f32x16{} : c[m][n];
#pragma unroll
                        for (int s = 0; s < 2; s++) v = mma16(x[m][0][s], w[P][n][s], mma16(x[m][1][s], w[P][n][s], v));
                        c[m][n] = v;
                    } else if constexpr (kSteps == 2) {
#pragma unroll
                        for (int s = 0; s < 2; s++) {
                            const f32x16 v = mma16(x[m][0][s], w[P][n][s], mma16(x[m][1][s], w[P][n][s], f32x16{}));
#pragma unroll
                            for (int i = 0; i < 16; i++) acc[m][n][i] = fmaf(scale[P][n][s], v[i], acc[m][n][i]);
                        }
                    } else {
                        f32x16 v = f32x16{};
#pragma unroll
                        for (int s = 0; s < 2; s++) v = mma16(x[m][0][s], w[P][n][s], mma16(x[m][1][s], w[P][n][s], v));
#pragma unroll
                        for (int i = 0; i < 16; i++) acc[m][n][i] = fmaf(scale[P][n][0], v[i], acc[m][n][i]);
                    }
                }
            if constexpr (!D::kFold) { /* left alone the compiler puts the scale steps off and runs out of registers */
#pragma unroll
                for (int n = 0; n < TN; n++)
#pragma unroll
                    for (int m = 0; m < TM; m++) asm volatile("" : "+v"(acc[m][n]));
            }
            /* a wave alone would make the next operands first and multiply afterwards */
            constexpr int kPerTile = kSteps == 2 && !D::kFold ? 2 : 1, kMma = 4 / kPerTile, kValu = D::kFold ? 16 : 24;
            each<TM * TN * kPerTile>([&](auto) {
                if constexpr (D::kFold) {
                    each<4>([&](auto) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, kValu / 4, 0);
                    });
                } else {
                    __builtin_amdgcn_sched_group_barrier(0x008, kMma, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, kValu, 0);
                }
            });
            slot = slot == S::kAhead ? 0 : slot + 1;
        });
        if constexpr (D::kFold) {
#pragma unroll
            for (int n = 0; n < TN; n++) {
                const float d = D::block(hdr[n][0]) * (F::kOffset == 0 ? kFoldUnit : 1.0f);
#pragma unroll
                for (int m = 0; m < TM; m++)
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[m][n][i] = fmaf(d, c[m][n][i], acc[m][n][i]);
                if constexpr (F::kHasMin) {
                    uint32_t a, b;
                    D::min_bytes(hdr[n][0], half, a, b);
                    const half8 mins = codes_f16<0>(a, b);
                    const float f = -32.0f * D::min_factor(hdr[n][0]); /* the sums are stored as 1/32 of themselves */
#pragma unroll
                    for (int m = 0; m < TM; m++) {
                        f32x16 v = f32x16{};
#pragma unroll
                        for (int q = 0; q < kSumsPer / 1024; q++)
                            v = mma16(*reinterpret_cast<const half8 *>(sums + m * kSumsPer + 1024 * q + 16 * lane), mins, v);
#pragma unroll
                        for (int i = 0; i < 16; i++) acc[m][n][i] = fmaf(f, v[i], acc[m][n][i]);
                    }
                }
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); /* nothing may arrive in LDS that is no longer this workgroup's */

    float *out = p.out + (size_t)part * (size_t)(p.parts > 1 ? p.n_tok : 0) * (size_t)p.ldo;
#pragma unroll
    for (int m = 0; m < TM; m++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int t = (token_tile * TM + m) * 32 + 8 * (i >> 2) + 4 * half + (i & 3);
            if (t >= p.n_tok) continue;
            const int e = p.parts > 1 ? 0 : -p.token_exp[t];
#pragma unroll
            for (int n = 0; n < TN; n++)
                if (32 * n + j < rows_here) out[(size_t)t * p.ldo + row0 + 32 * n + j] = __builtin_ldexpf(acc[m][n][i], e);
        }
}

/* Adds the parts of K in order (one part: the product has written Y itself) and completes the tokens that hold an infinity
 * or a NaN, whose fragments are zeros. Only those elements decide such a result - an infinity, or a NaN where the products
 * with them do not agree - so a workgroup collects them a stretch of K at a time and decodes no more than their weights, a
 * row only until it is NaN (64 tokens 4096 x 4096, one token not finite: a thread walking whole rows 845 us, now 38). Rows with
 * weights that are not finite have a NaN from the product. A thread has R rows: four where rows of Y and of the parts allow
 * 16-byte accesses. */
template <uint32_t T, int R>
__global__ void __launch_bounds__(256) f32_finish_kernel(const uint8_t *__restrict__ W, const float *__restrict__ X, const float *__restrict__ part,
                                                        const int *__restrict__ token_exp, float *__restrict__ Y, int n_rows, int n_cols, int n_tok,
                                                        int parts, int ldx, int ldy) {
    using C = Codec<T>;
    typedef float vec __attribute__((ext_vector_type(R)));
    const int row = (blockIdx.x * 256 + threadIdx.x) * R, t = blockIdx.y;
    const int e = token_exp[t];
    if (parts == 1 && e != kF32NotFinite) return;
    vec *out = reinterpret_cast<vec *>(Y + (size_t)t * ldy + row);
    vec sum = 0.0f;
    if (row < n_rows) {
        if (parts == 1) sum = *out;
        const float *at = part + (size_t)t * n_rows + row;
        if (parts > 1) {
#pragma unroll 4
            for (int s = 0; s < parts; s++) sum += *reinterpret_cast<const vec *>(at + (size_t)s * n_tok * n_rows);
        }
    }
    if (e != kF32NotFinite) {
#pragma unroll
        for (int i = 0; i < R; i++) sum[i] = __builtin_ldexpf(sum[i], -e);
    } else { /* the same for the whole workgroup */
        constexpr int kStretch = 1024;
        __shared__ int found[kStretch], n_found;
        const uint32_t *x = reinterpret_cast<const uint32_t *>(X + (size_t)t * ldx);
        for (int k0 = 0; k0 < n_cols; k0 += kStretch) {
            if (threadIdx.x == 0) n_found = 0;
            __syncthreads();
            for (int k = k0 + threadIdx.x; k < min(k0 + kStretch, n_cols); k += 256)
                if ((x[k] & 0x7F800000u) == 0x7F800000u) found[atomicAdd(&n_found, 1)] = k;
            __syncthreads();
            bool open = row < n_rows; /* a result that is not NaN yet */
            for (int n = 0; n < n_found && open; n++) {
                const int k = found[n];
                open = false;
                for (int i = 0; i < R; i++) {
                    if (sum[i] != sum[i]) continue;
                    open = true;
                    float v[8], w = 0.0f;
                    C::decode8(W + (size_t)(row + i) * ((size_t)(n_cols / C::BE) * C::BB) + (size_t)(k / C::BE) * C::BB, k % C::BE & ~7, v);
#pragma unroll
                    for (int l = 0; l < 8; l++) w = (k & 7) == l ? v[l] : w;
                    sum[i] += w * __uint_as_float(x[k]);
                }
            }
            if (!__syncthreads_or(open)) break;
        }
    }
    if (row < n_rows) *out = sum;
}

template <class F, int TM> hipError_t split_launch(const F32SplitCall &c, const SplitArgs &base) {
    using S = SplitShape<F, TM>;
    static OnceFlag lds_raised;
    const auto kernel = gemm_f32_split_kernel<F, TM>;
    if (!lds_raised.is_set()) {
        const hipError_t e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);
        if (e != hipSuccess) return e;
        lds_raised.set();
    }
    SplitArgs p = base;
    p.row_tiles = (c.n_rows + S::kRows - 1) / S::kRows;
    p.token_tiles = (c.n_tok + S::kTokens - 1) / S::kTokens;
    const int items = p.row_tiles * p.token_tiles * p.parts;
    hipLaunchKernelGGL(kernel, dim3(8 * ((items + 7) / 8)), dim3(256), S::kLds, c.stream, p);
    return hipGetLastError();
}

template <class F, uint32_t T> hipError_t split_format(const F32SplitCall &c) {
    const F32SplitPlan plan = f32_split_plan(T, c.n_rows, c.n_cols, c.n_tok, c.workspace_bytes);
    constexpr int kSumGroup = F::kHasMin ? (F::kGroup16 ? 16 : 32) : 0;
    if (const hipError_t e = launch_f32_split(c, plan, kSumGroup); e != hipSuccess) return e;
    uint8_t *ws = (uint8_t *)c.workspace;
    SplitArgs p = {};
    p.W = (const uint8_t *)c.W;
    p.frags = ws;
    p.sums = ws + plan.sums_at;
    p.token_exp = (const int *)(ws + plan.exp_at);
    p.parts = plan.parts;
    p.out = plan.parts > 1 ? (float *)(ws + plan.parts_at) : c.Y;
    p.ldo = plan.parts > 1 ? c.n_rows : c.ldy;
    p.n_rows = c.n_rows;
    p.n_tok = c.n_tok;
    p.n_sb = c.n_cols / 256;
    if (const hipError_t e = plan.token_blocks == 1 ? split_launch<F, 1>(c, p) : split_launch<F, 2>(c, p); e != hipSuccess) return e;
    const bool wide = c.n_rows % 4 == 0 && c.ldy % 4 == 0 && ((uintptr_t)c.Y & 15) == 0;
    const int per_block = 256 * (wide ? 4 : 1);
    const dim3 grid((c.n_rows + per_block - 1) / per_block, c.n_tok);
    const auto finish = wide ? f32_finish_kernel<T, 4> : f32_finish_kernel<T, 1>;
    hipLaunchKernelGGL(finish, grid, dim3(256), 0, c.stream, (const uint8_t *)c.W, c.X, (const float *)(ws + plan.parts_at), p.token_exp, c.Y,
                       c.n_rows, c.n_cols, c.n_tok, plan.parts, c.ldx, c.ldy);
    return hipGetLastError();
}

}  // namespace
}  // namespace qlin
#endif

/*
 * gemm_fewtok.h - block-format x bf16 products for up to 128 tokens: a batch of decoding sequences, a speculative
 * verify, a short prompt. The kernel and its launch as templates over the format; gemm_fewtok*.hip instantiate them.
 *
 *   Y[t*ldy + r] = sum_k X[t*ldx + k] * decode(W)[r][k]      X bf16, Y fp32, fp32 accumulate
 *
 * With this few tokens the weights' own bytes are what a launch cannot do without, so the kernel has the structure of
 * the matvec (gemv_q4k.hip) and not that of a tile product: a workgroup owns NT * 16 rows, its eight waves split K - wave
 * w takes super-blocks w, w + 8, ... (seven waves where LDS is short) - and meet once, in LDS, for the sum over K. A wave copies a super-block of all its
 * rows by load-to-LDS requests into an image of its own (whole blocks, consecutive lanes consecutive 16-byte pieces,
 * source addresses of any alignment) and the activations of those 256 elements the same way, chunk by chunk, the next
 * chunk on its way while one is multiplied; it waits by counting its own requests and needs no barrier before the final
 * sum. Matrix instruction: v_mfma_f32_16x16x32_bf16, A = tokens: lane (j, kg) holds elements 8 kg .. + 7 of token j;
 * B = weights: the same elements of row j, cut out of the image.
 *
 * Two forms of the arithmetic:
 *   exact    the codes go through the matrix instruction as they are - integers of up to 8 bits are exact in bf16 - and
 *            the block scales are applied to the 32-element sums in fp32 (formats with a scale per 16 elements: the
 *            token operand holds zeros in the lanes of the other 16, eight tokens per instruction). A minimum goes in as a
 *            second sum. 4-bit codes become bf16 two at a time through the fp8 conversion; 5- and 6-bit codes by a byte
 *            permute that puts a fixed high byte on top (32 + q and 64 + q have all their low bits in the low byte). Such
 *            a 32 or 64, and what the format itself subtracts from its codes, comes off as the instruction's C operand, a
 *            product of the activations with that constant: before the scale, where the sum is as long as its terms
 *            (Q5_K's 32 taken off with the minimum, after 32 s had been rounded: error 1.2e-7 at K = 1024, now 8.8e-8).
 *            8-bit codes go through the byte-to-float conversion signed (as unsigned numbers with 128 taken off, the
 *            magnitudes of IQ3_S, at most 15, drowned in it: 1.8e-7, now 6.5e-8).
 *   rounded  the weights are decoded in fp32 as the codec does and rounded once to bf16: the vector work per weight then
 *            does not depend on the number of tokens.
 *
 * What bounds it: activations and weights share a compute unit's load path (64 bytes per clock), which returns in order,
 * so that tokens * K * 2 bytes of activations per compute unit come on top of the weights' time: 4096 x 14336 at 16
 * tokens 13.8 us, of which 5.5 are the weights' bytes from HBM, 4 the activations through that path and 2 the launch. At
 * high row counts the vector ALU: about 180 instructions per 16 rows x 256 elements and 16 tokens (Q4_K).
 * Measured, us, before (a four-wave kernel with 16 or 32 rows per workgroup, one launch per tensor, 16 tokens at a time;
 * small-tile kernel from 33 tokens) / now: Q4_K 16 tokens 4096 x 4096 9.9 / 5.6, 4096 + 1024 + 1024 rows x 4096 31 / 8,
 * 14336 x 4096 14.3 / 12.0, 4096 x 14336 27 / 13.8; Q6_K 16 tokens 14.5 / 7.7, 14336 x 4096 32 / 18, 4096 x 14336
 * 38 / 18.5; Q8_0 32 tokens 4096 x 14336 103 / 25; IQ4_XS 16 tokens 4096 x 4096 (decode + dense product) 21 / 6.6; 77
 * tokens 2560 x 6912 Q6_K 41 / 18, Q4_K 26 / 13.6.
 */
#ifndef QLIN_GEMM_FEWTOK_H
#define QLIN_GEMM_FEWTOK_H

#include "gemm_image_formats.h"
#include "qlin_internal.h"

namespace qlin {

using namespace kq;

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

QLIN_INL f32x4 mma(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
template <int V> QLIN_INL bf16x8 const_bf16() {
    constexpr float f = (float)V; /* a power of two or a small integer: exact */
    const uint32_t h = __builtin_bit_cast(uint32_t, f) >> 16;
    const uint32_t w = h | (h << 16);
    const u32x4 v = {w, w, w, w};
    return __builtin_bit_cast(bf16x8, v);
}
QLIN_INL uint32_t upper_halves(float lo, float hi) { return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u); }
/* eight codes (unsigned bytes) as bf16, exact */
template <bool SMALL> QLIN_INL bf16x8 codes_bf16(uint32_t a, uint32_t b) {
    u32x4 r;
    if constexpr (SMALL) { /* a byte 0x0q read as E4M3 is q * 2^-9 */
        r.x = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 512.0f, false));
        r.y = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 512.0f, true));
        r.z = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 512.0f, false));
        r.w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 512.0f, true));
    } else { /* integers up to 255 have no bits below bf16's */
        r.x = upper_halves(ubyte_f32<0>(a), ubyte_f32<1>(a));
        r.y = upper_halves(ubyte_f32<2>(a), ubyte_f32<3>(a));
        r.z = upper_halves(ubyte_f32<0>(b), ubyte_f32<1>(b));
        r.w = upper_halves(ubyte_f32<2>(b), ubyte_f32<3>(b));
    }
    return __builtin_bit_cast(bf16x8, r);
}
/* eight codes less 128 as bf16, exact */
QLIN_INL bf16x8 signed_bf16(uint32_t a, uint32_t b) {
    a ^= 0x80808080u;
    b ^= 0x80808080u;
    const u32x4 r = {upper_halves(signed_byte(a, 0), signed_byte(a, 8)), upper_halves(signed_byte(a, 16), signed_byte(a, 24)),
                     upper_halves(signed_byte(b, 0), signed_byte(b, 8)), upper_halves(signed_byte(b, 16), signed_byte(b, 24))};
    return __builtin_bit_cast(bf16x8, r);
}
template <int HI> QLIN_INL bf16x8 ready_bf16(uint32_t a, uint32_t b) {
    constexpr uint32_t hi = HI * 0x01010101u;
    const u32x4 r = {__builtin_amdgcn_perm(hi, a, 0x07010700u), __builtin_amdgcn_perm(hi, a, 0x07030702u),
                     __builtin_amdgcn_perm(hi, b, 0x07010700u), __builtin_amdgcn_perm(hi, b, 0x07030702u)};
    return __builtin_bit_cast(bf16x8, r);
}
/* code * s - o rounded to bf16 */
template <bool SMALL> QLIN_INL bf16x8 weights_bf16(uint32_t a, uint32_t b, float s, float o) {
    float f[8];
    if constexpr (SMALL) {
        const float2v p0 = fp8_pair_lo(a), p1 = fp8_pair_hi(a), p2 = fp8_pair_lo(b), p3 = fp8_pair_hi(b);
        f[0] = p0.x; f[1] = p0.y; f[2] = p1.x; f[3] = p1.y; f[4] = p2.x; f[5] = p2.y; f[6] = p3.x; f[7] = p3.y;
        s *= 512.0f;
    } else {
        f[0] = ubyte_f32<0>(a); f[1] = ubyte_f32<1>(a); f[2] = ubyte_f32<2>(a); f[3] = ubyte_f32<3>(a);
        f[4] = ubyte_f32<0>(b); f[5] = ubyte_f32<1>(b); f[6] = ubyte_f32<2>(b); f[7] = ubyte_f32<3>(b);
    }
#pragma unroll
    for (int i = 0; i < 8; i++) f[i] = fmaf(f[i], s, -o);
    const u32x4 r = {pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]), pack_bf16(f[4], f[5]), pack_bf16(f[6], f[7])};
    return __builtin_bit_cast(bf16x8, r);
}

/* Shape of an instance: NT 16-row tiles, up to 8 TT tokens. kXSteps: 32-element steps whose activations are fetched and
 * held at a time - short chunks leave LDS for a second workgroup per compute unit, which measured more than longer ones
 * (Q4_K, 32 tokens, 14336 x 4096: chunks of two steps 16.3 us, of four 18.8); with eight tokens and one row tile whole
 * super-blocks (4096 x 14336, 8 tokens: 11.5 against 12.9); single steps where two row tiles and more than 96 tokens fill
 * the LDS. A second chunk or image ahead measured no gain. */
template <class F, int NT, int TT, bool EXACT> struct Shape {
    static constexpr bool kDiag = EXACT && F::kGroup16;      /* eight tokens per instruction */
    static constexpr int kOps = kDiag ? TT : (TT + 1) / 2;   /* token operands */
    static constexpr int kXSteps = NT == 2 && TT > 12 ? 1 : TT == 1 ? (NT == 1 ? 8 : 4) : TT == 2 ? (NT == 1 ? 4 : 2) : kDiag && NT == 2 ? 4 : 2;
    static constexpr int kParts = 8 / kXSteps;               /* chunks per super-block */
    static constexpr int kXReq = TT * kXSteps / 2, kXChunk = kXReq * 1024; /* requests and bytes of a chunk of activations */
    static constexpr int kImage = NT * 16 * F::kPieces * 16, kWReq = (kImage + 1023) / 1024; /* of a wave's image */
    static constexpr int kPart = NT * kOps * 1024;           /* bytes of a wave's partial sums, in the same place */
    static constexpr int kWaveLds = kXChunk + kImage > kPart ? kXChunk + kImage : kPart;
    /* the same for every NT, so that a row's sum does not depend on how many rows a launch has */
    static constexpr int kWaves = 8 * (TT * 1024 + 16 * F::kPieces * 16) + 4 * F::kTable <= 160 * 1024 ? 8 : 7;
    /* Chains of fp32 sums that a wave's share of K is divided over. The formats with few unrounded tokens come from the
     * matvec, which sums 64 short shares; their error at K = 14336, 3 tokens, against 64 bits with one chain / four 1.5e-7 /
     * 9.7e-8 (the matvec 8.4e-8). Q4_0 has registers for two without giving up a workgroup per compute unit (151936 x 4096
     * 71 us, with four 87). The other formats keep one (the kernel they come from had half as many waves: Q4_K 2.7e-7,
     * now 2.0e-7). */
    static constexpr int kChains = EXACT && F::kUnrounded <= 4 ? (F::kSmall ? 2 : 4) : 1;
    /* four waves per SIMD - a wave alone issues a vector instruction every five cycles, four together one every 2.4 to
     * 4.3 - where the registers allow; two otherwise */
    static constexpr int kPerSimd = kChains > 2 && NT > 1 ? 6 : TT <= 2 ? 4 : EXACT ? (NT == 1 || kDiag ? 2 : 4) : TT <= 6 ? 4 : 2;
    static constexpr bool kStepwise = NT > 1 || (TT >= 4 && !EXACT) || (kDiag && F::kHasMin); /* see the end of a step */
    static_assert(TT * kXSteps % 2 == 0 && kWaves * kWaveLds + 4 * F::kTable <= 160 * 1024, "whole requests; LDS");
};

template <class F, int NT, int TT, bool EXACT>
__global__ void __launch_bounds__((64 * Shape<F, NT, TT, EXACT>::kWaves))
    __attribute__((amdgpu_waves_per_eu((Shape<F, NT, TT, EXACT>::kPerSimd))))
gemm_fewtok_kernel(TileSet set, const uint16_t *__restrict__ X, int n_sb, int n_tok, int ldx) {
    using S = Shape<F, NT, TT, EXACT>;
    constexpr int kOps = S::kOps, kRow = F::kPieces * 16, XS = S::kXSteps;
    /* codes of eight bits go in signed; the other formats' constants as the instruction's C operand */
    constexpr bool kSigned = F::kOffset == 128, kAsC = F::kOffset != 0 && !kSigned;
    constexpr uint32_t kPastEnd = 0xFFFFFFF0u; /* an offset outside every buffer: the request returns zeros */
    extern __shared__ __attribute__((aligned(1024))) uint8_t fewtok_lds[];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n_waves = blockDim.x >> 6;
    const int j = lane & 15, kg = lane >> 4;
    const TileOf t = tile_of(set, blockIdx.x);
    const int row0 = t.tile * (16 * NT);
    const int rows_here = min(16 * NT, t.n_rows - row0);
    const uint32_t row_bytes = (uint32_t)n_sb * F::kBlock;
    uint8_t *xst = fewtok_lds + wv * S::kWaveLds, *img = xst + S::kXChunk;
    uint32_t *tab = reinterpret_cast<uint32_t *>(fewtok_lds + n_waves * S::kWaveLds);

    /* weights: piece 64 q + lane of an image is part id % kPieces of row id / kPieces; rows past the end arrive as zeros */
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(t.W) + (size_t)row0 * row_bytes, 0,
                                                                            (int)(rows_here * row_bytes), 0x00020000);
    uint32_t w_off[S::kWReq];
#pragma unroll
    for (int q = 0; q < S::kWReq; q++) {
        const uint32_t id = 64u * q + lane, row = id / F::kPieces, part = id % F::kPieces, src = F::piece_src(part);
        const uint32_t off = row * row_bytes + src;
        w_off[q] = row < (uint32_t)rows_here && src != kNoPiece ? off : kPastEnd;
    }
    const bool w_last = 64 * (S::kWReq - 1) + lane < S::kImage / 16; /* lanes past the image's last piece stay out */
    /* activations: a chunk is [8 TT tokens][XS * 4 pieces of 16 bytes], piece c of token t at position c ^ swizzle(t), so
     * that the 16 tokens of an operand read fall into 16 bank groups; tokens past the end arrive as zeros */
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(X), 0,
                                                                            ((n_tok - 1) * ldx + n_sb * 256) * 2, 0x00020000);
    auto swizzle = [](int tok) { return XS == 1 ? (tok >> 2) & 3 : XS == 2 ? (tok >> 1) & 7 : S::kDiag || TT == 1 ? tok & 7 : tok & 15; };
    uint32_t x_off[S::kXReq];
#pragma unroll
    for (int q = 0; q < S::kXReq; q++) {
        const int tok = q * (16 / XS) + lane / (4 * XS);
        const uint32_t off = (uint32_t)tok * (uint32_t)(2 * ldx) + 16u * (uint32_t)((lane % (4 * XS)) ^ swizzle(tok));
        x_off[q] = tok < n_tok ? off : kPastEnd;
    }
    const uint32_t x_at = (uint32_t)(uintptr_t)(lds_void *)xst, w_at = (uint32_t)(uintptr_t)(lds_void *)img;
    auto request_x = [&](int sb, int part) {
#pragma unroll
        for (int q = 0; q < S::kXReq; q++) request16(x_at + 1024u * q, x_off[q], x_rsrc, (uint32_t)sb * 512u + (uint32_t)part * (64u * XS));
    };
    auto request_w = [&](int sb) {
#pragma unroll
        for (int q = 0; q < S::kWReq; q++)
            if (q + 1 < S::kWReq || w_last) request16(w_at + 1024u * q, w_off[q], w_rsrc, (uint32_t)sb * (uint32_t)F::kBlock);
    };
    request_x(wv, 0);
    request_w(wv);
    if constexpr (F::kTable > 0) {
        for (int i = threadIdx.x; i < F::kTable; i += blockDim.x) tab[i] = F::table()[i];
        __syncthreads();
    }

    const bool live = !S::kDiag || (kg >> 1) == (j >> 3);
    const int tok0 = S::kDiag || TT == 1 ? j & 7 : j; /* operand o holds token 16 o (8 o) + tok0 */
    const uint32_t x_rd = (uint32_t)(tok0 * (64 * XS) + ((kg ^ swizzle(tok0)) << 4));
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int CH = S::kChains;
    f32x4 acc[NT][kOps][CH];
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int o = 0; o < kOps; o++)
#pragma unroll
            for (int i = 0; i < CH; i++) acc[nt][o][i] = zero;

    for (int sb = wv; sb < n_sb; sb += n_waves) {
        typename F::Hdr hdr[NT];
        each<S::kParts>([&](auto part) {
            constexpr int pt = decltype(part)::value, u0 = pt * XS;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); /* the chunk is in, and the image ahead of the first */
            u32x4 xa[kOps][XS];
#pragma unroll
            for (int o = 0; o < kOps; o++)
#pragma unroll
                for (int u = 0; u < XS; u++) {
                    /* (two-step chunks: the swizzle of an odd eight-token operand is 4 higher) */
                    u32x4 v = *reinterpret_cast<const u32x4 *>(xst + (x_rd ^ (64u * (u ^ (S::kDiag && XS == 2 ? o & 1 : 0)))) +
                                                               o * (S::kDiag ? 512 : 1024) * XS);
                    if (S::kDiag && !live) v = u32x4{0u, 0u, 0u, 0u};
                    xa[o][u] = v;
                }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* read, so its place can take the next one */
            if constexpr (pt + 1 < S::kParts) request_x(sb, pt + 1);
            else if (sb + n_waves < n_sb) request_x(sb + n_waves, 0);
            if constexpr (pt == 0) {
#pragma unroll
                for (int nt = 0; nt < NT; nt++) hdr[nt] = F::header(img + (16 * nt + j) * kRow, kg);
            }
            each<XS>([&](auto step) {
                constexpr int u = decltype(step)::value, U = u0 + u;
                f32x4 xs[kOps]; /* sums of the activations, or their products with the constant to be subtracted */
                if constexpr (EXACT && (F::kHasMin || kAsC)) {
#pragma unroll
                    for (int o = 0; o < kOps; o++)
                        xs[o] = mma(__builtin_bit_cast(bf16x8, xa[o][u]), const_bf16<(F::kHasMin ? 1 : -F::kOffset - F::kBase)>(), zero);
                }
                f32x4 c0[kOps]; /* where the instruction starts */
#pragma unroll
                for (int o = 0; o < kOps; o++) {
                    if constexpr (EXACT && kAsC) c0[o] = xs[o];
                    else if constexpr (EXACT && F::kHasMin && F::kBase != 0 && TT == 1) c0[o] = mma(__builtin_bit_cast(bf16x8, xa[o][u]), const_bf16<-F::kBase>(), zero);
                    else if constexpr (EXACT && F::kHasMin && F::kBase != 0) c0[o] = xs[o] * (float)-F::kBase; /* (the same numbers) */
                    else c0[o] = zero;
                }
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    const uint8_t *row = img + (16 * nt + j) * kRow;
                    uint32_t a, b;
                    if constexpr (EXACT && F::kReady != 0) F::template ready<U>(row, kg, tab, a, b);
                    else F::template codes<U>(row, kg, tab, a, b);
                    const float s = F::template scale<U>(hdr[nt], kg);
                    if constexpr (EXACT) {
                        bf16x8 w;
                        if constexpr (kSigned) w = signed_bf16(a, b);
                        else if constexpr (F::kReady != 0) w = ready_bf16<F::kReady>(a, b);
                        else w = codes_bf16<F::kSmall>(a, b);
#pragma unroll
                        for (int o = 0; o < kOps; o++) {
                            const f32x4 c = mma(__builtin_bit_cast(bf16x8, xa[o][u]), w, c0[o]);
#pragma unroll
                            for (int v = 0; v < 4; v++) acc[nt][o][U % CH][v] = fmaf(s, c[v], acc[nt][o][U % CH][v]);
                        }
                        if constexpr (F::kHasMin) {
                            const float m = F::template minimum<U>(hdr[nt], kg);
#pragma unroll
                            for (int o = 0; o < kOps; o++)
#pragma unroll
                                for (int v = 0; v < 4; v++) acc[nt][o][U % CH][v] = fmaf(-m, xs[o][v], acc[nt][o][U % CH][v]);
                        }
                    } else {
                        const float off = F::kHasMin ? F::template minimum<U>(hdr[nt], kg) : s * (float)F::kOffset;
                        const bf16x8 w = weights_bf16<F::kSmall>(a, b, s, off);
#pragma unroll
                        for (int o = 0; o < kOps; o++) acc[nt][o][0] = mma(__builtin_bit_cast(bf16x8, xa[o][u]), w, acc[nt][o][0]);
                    }
                }
                /* no further ahead than the steps that share loads: left alone the compiler fetches the whole image first,
                 * keeps the scale steps for the end and runs out of registers (170 instead of 75 with two row tiles). One
                 * row tile and few tokens fit anyway, and are faster its way */
                if constexpr (S::kStepwise && (u + 1) % F::kShare == 0) {
#pragma unroll
                    for (int nt = 0; nt < NT; nt++)
#pragma unroll
                        for (int o = 0; o < kOps; o++) asm volatile("" : "+v"(acc[nt][o][U % CH]));
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
        });
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* the image has been read */
        if (sb + n_waves < n_sb) request_w(sb + n_waves);
    }

    /* the waves' shares of K meet: a wave's partial sums take the place of its chunk and image */
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    f32x4 *mine = reinterpret_cast<f32x4 *>(xst);
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int o = 0; o < kOps; o++) {
#pragma unroll
            for (int n = CH / 2; n > 0; n /= 2)
#pragma unroll
                for (int i = 0; i < n; i++) acc[nt][o][i] += acc[nt][o][i + n];
            f32x4 v = acc[nt][o][0];
            if constexpr (S::kDiag) {
#pragma unroll
                for (int i = 0; i < 4; i++) v[i] = add_lane32(v[i]); /* the two scale groups */
            }
            mine[(nt * kOps + o) * 64 + lane] = v;
        }
    __syncthreads();
    for (int idx = threadIdx.x; idx < NT * kOps * 256; idx += blockDim.x) {
        const int v = idx & 3, ln = (idx >> 2) & 63, o = (idx >> 8) % kOps, nt = (idx >> 8) / kOps;
        if (S::kDiag && ln >= 32) continue;
        float sum = 0.0f;
        for (int w = 0; w < n_waves; w++) sum += *reinterpret_cast<const float *>(fewtok_lds + w * S::kWaveLds + 4 * idx);
        const int tok = (S::kDiag ? 8 : 16) * o + 4 * (ln >> 4) + v, row = 16 * nt + (ln & 15);
        if (tok < n_tok && row < rows_here) t.Y[(size_t)tok * t.ldy + row0 + row] = sum;
    }
}

template <class F, int NT, int TT, bool EXACT> hipError_t fewtok_launch(const FewtokCall &c) {
    using S = Shape<F, NT, TT, EXACT>;
    static OnceFlag lds_raised;
    const auto kernel = gemm_fewtok_kernel<F, NT, TT, EXACT>;
    if (!lds_raised.is_set()) {
        const hipError_t e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
        lds_raised.set();
    }
    const int n_sb = c.n_cols / 256, waves = n_sb < S::kWaves ? n_sb : S::kWaves;
    TileSet set;
    const int grid = fill_tile_set(set, c.n_mat, c.W, c.Y, c.n_rows, c.ldy, 16 * NT);
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * waves), (size_t)waves * S::kWaveLds + 4 * F::kTable, c.stream, set, c.X, n_sb,
                       c.n_tok, c.ldx);
    return hipGetLastError();
}

/* One row tile per workgroup up to a tile for every compute unit and a few over; two beyond, which read the activations
 * once for both (us, 16 tokens, one / two: Q4_K 256 tiles 5.6 / 6.8, 384 tiles 8.4 / 7.6, 864 tiles 12.4 / 9.9; Q6_K 7.8 /
 * 11.4, 11.6 / 11.9, 16.8 / 14.4). Q8_0 with eight tokens: two images leave no room for a second workgroup (13.3 / 16), and
 * from 65 tokens on they do not fit at all. Rows of up to four super-blocks have as many waves, and a compute unit holds
 * more of those workgroups, so that one tile reaches further (24 tokens 9216 x 1024 Q6_K, one / two: 7.1 / 8.9, 64 tokens
 * 14336 x 256 Q4_K 6.2 / 9.1) - except 17 and more unrounded tokens of Q4_K and Q5_K, whose waves want many registers
 * (32 tokens 9216 x 1024 Q4_K 7.1 / 6.2). From 65 tokens on a workgroup of eight waves fills a compute unit (320 tiles x
 * 4096, one / two: 96 tokens Q4_K 18.4 / 12.5, 128 tokens 23.4 / 18.2; 288 tiles x 2048 at 128 15.1 / 11.1). */
template <class F, int TT, bool EXACT> hipError_t fewtok_rows(const FewtokCall &c) {
    if constexpr (TT <= 8 || F::kPieces < 17) {
        constexpr bool kSmallGroups = !(EXACT && TT >= 3 && F::kHasMin && !F::kGroup16);
        const int n_sb = c.n_cols / 256, waves = kSmallGroups && n_sb <= 4 ? n_sb : 8;
        long long tiles = 0;
        for (int i = 0; i < c.n_mat; i++) tiles += (c.n_rows[i] + 15) / 16;
        if (tiles * waves > (TT <= 8 ? 288 : 256) * 8 && !(F::kPieces >= 17 && TT == 1 && tiles > 512)) return fewtok_launch<F, 2, TT, EXACT>(c);
    }
    return fewtok_launch<F, 1, TT, EXACT>(c);
}

template <class F> hipError_t fewtok_format(const FewtokCall &c) {
    constexpr int EXACT_MAX = F::kUnrounded;
    const int n = c.n_tok;
    if (n <= EXACT_MAX) {
        if constexpr (EXACT_MAX <= 8) return fewtok_rows<F, 1, true>(c);
        else {
            if (n <= 8) return fewtok_rows<F, 1, true>(c);
            if (n <= 16) return fewtok_rows<F, 2, true>(c);
            return fewtok_rows<F, EXACT_MAX / 8, true>(c);
        }
    }
    if constexpr (EXACT_MAX <= 8) {
        if (n <= 8) return fewtok_rows<F, 1, false>(c);
        if (n <= 16) return fewtok_rows<F, 2, false>(c);
    }
    if constexpr (EXACT_MAX < 32) {
        if (n <= 32) return fewtok_rows<F, 4, false>(c);
    }
    if (n <= 48) return fewtok_rows<F, 6, false>(c);
    if (n <= 64) return fewtok_rows<F, 8, false>(c);
    if constexpr (F::kTable > 0) return hipErrorInvalidValue; /* the grid formats end here */
    else if (n <= 80) return fewtok_rows<F, 10, false>(c);
    else if (n <= 96) return fewtok_rows<F, 12, false>(c);
    else return fewtok_rows<F, 16, false>(c);
}

}  // namespace
}  // namespace qlin
#endif

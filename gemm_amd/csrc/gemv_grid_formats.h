/*
 * gemv_grid_formats.h - block formats as the matvecs on the 8-bit integer matrix instruction see them (gemv_grid.hip,
 * gemv_dma.hip): what a lane reads of a block, its item - sixteen rows times 256 elements - and the x operand that
 * the items multiply by.
 */
#ifndef QLIN_GEMV_GRID_FORMATS_H
#define QLIN_GEMV_GRID_FORMATS_H

#include "qlin_codebooks.h"
#include "qlin_codebooks_ext.h"
#include "qlin_device.h"
#include "qlin_internal.h"

namespace qlin {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));

constexpr int kXScratch = 1152;   /* per wave: 3 digit planes x 256 B, 128 zero bytes, (at 1024) 8 x 2^(e-22), (at 1056) 16 sums of 16 x */

/* x operand of one super-block: A[s] for instruction s. The other two things an item needs stay in the wave's
 * scratch until the next super-block is prepared: meta[G] = 2^(e-22) of 32-element group G, meta[8 + S] = the sum
 * of x over 16-element group S (formats with a constant offset per code). */
struct XOperand {
    v4i A[4];             /* formats whose items keep LDS busy with table lookups hold the operand in registers */
    const uint8_t *arows; /* the others read it per item: instruction s at arows + F::kStep * s (zeros for a dead lane) */
    const float *meta;
};

template <int CTRL> __device__ __forceinline__ uint32_t dpp_movu(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}

/* sixteen bytes at p (2-byte aligned, inside a block that starts at least two bytes before p): the aligned
 * dwords around them and, where p sits in the middle of a dword, the two bytes behind the last full one */
struct Raw16 {
    u32x4_a4 q;
    uint32_t tail;
};
__device__ __forceinline__ Raw16 load16(const uint8_t *p) {
    Raw16 r;
    const uint32_t odd = (uint32_t)(uintptr_t)p & 2u;
    r.q = *reinterpret_cast<const u32x4_a4 *>(p - odd);
    r.tail = 0;
    if (odd) r.tail = *reinterpret_cast<const uint16_t *>(p + 14);
    return r;
}
__device__ __forceinline__ void bytes16(const Raw16 &r, uint32_t sh, uint32_t (&w)[4]) { /* sh = 0 or 16 */
    w[0] = __builtin_amdgcn_alignbit(r.q.y, r.q.x, sh);
    w[1] = __builtin_amdgcn_alignbit(r.q.z, r.q.y, sh);
    w[2] = __builtin_amdgcn_alignbit(r.q.w, r.q.z, sh);
    w[3] = __builtin_amdgcn_alignbit(r.tail, r.q.w, sh);
}
struct Raw8 {
    u32x2_a4 q;
    uint32_t tail;
};
__device__ __forceinline__ Raw8 load8(const uint8_t *p) {
    Raw8 r;
    const uint32_t odd = (uint32_t)(uintptr_t)p & 2u;
    r.q = *reinterpret_cast<const u32x2_a4 *>(p - odd);
    r.tail = 0;
    if (odd) r.tail = *reinterpret_cast<const uint16_t *>(p + 6);
    return r;
}
__device__ __forceinline__ void bytes8(const Raw8 &r, uint32_t sh, uint32_t (&w)[2]) {
    w[0] = __builtin_amdgcn_alignbit(r.q.y, r.q.x, sh);
    w[1] = __builtin_amdgcn_alignbit(r.tail, r.q.y, sh);
}

/* the tables in LDS: the format's grid, and the sign masks (0xFF per negative element, two dwords per sign
 * byte): 256 entries by sign byte, then 128 by the seven stored bits of the formats that keep a parity bit */
struct Tables {
    const uint32_t *grid;
    const uint2 *sign256, *sign128;
};

/* magnitudes m (four bytes, each 1..127: no grid of these formats holds a zero) with the signs of mask s
 * (0xFF = negative) -> signed bytes: (m ^ s) + (s & 1) per byte; a nonzero m keeps the +1 inside its byte */
__device__ __forceinline__ int apply_signs(uint32_t m, uint32_t s) { return (int)((m ^ s) + (s & 0x01010101u)); }
__device__ __forceinline__ uint32_t spread4(uint32_t v) { return ((v & 15u) * 0x00204081u) & 0x01010101u; }

/* digit sums of one group (top, middle, low) -> the group's integer inner product as a float */
__device__ __forceinline__ float join_digits(v4i c) {
    return fmaf((float)c.x, 65536.0f, (float)((c.y << 8) + c.z));
}

template <uint32_t T> struct GridFmt;

/* IQ2_XXS [d][8 x (4 grid indices, 4 x 7 sign bits + 4-bit scale)]: d*(0.5+s)*0.25 * grid byte * sign, an
 * eight-byte grid entry per index (common/ggml_dequant.h:2793-2816); 66-byte blocks */
template <> struct GridFmt<T_IQ2_XXS> {
    static constexpr int kBlock = 66, kGridBytes = 2048;
    static constexpr int kAlign = 2; /* what the loads want of the matrix address and the row pitch */
    static constexpr int kStep = 16; /* bytes between the x rows of consecutive instructions */
    static constexpr bool kAInRegs = true;
    static constexpr int kPiece = 2; /* every piece a lane reads starts 2 (mod 4) bytes into the block */
    static constexpr bool kSums = false;
    /* lane group g takes elements [64 g, 64 g + 64) in order, 16 per instruction */
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    __device__ static const uint32_t *grid_src() { return reinterpret_cast<const uint32_t *>(qlin_iq2xxs_grid); }
    struct Raw {
        Raw16 a; /* groups 2g, 2g+1: [indices, signs + scale] each */
        uint32_t d;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        r.a = load16(blk + 2 + 16 * g);
        r.d = *reinterpret_cast<const uint16_t *>(blk);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t sh, const Tables &t, int g) {
        uint32_t w[4];
        bytes16(r.a, sh, w);
        const uint2 *grid = reinterpret_cast<const uint2 *>(t.grid);
        const float d = half_bits_fast(r.d) * 0.25f;
        float acc = 0.0f;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t a0 = w[2 * h], a1 = w[2 * h + 1];
            v4i c = {0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const uint2 m0 = grid[(a0 >> (16 * q)) & 255u], m1 = grid[(a0 >> (16 * q + 8)) & 255u];
                const uint2 s0 = t.sign128[(a1 >> (14 * q)) & 127u], s1 = t.sign128[(a1 >> (14 * q + 7)) & 127u];
                const v4i b = {apply_signs(m0.x, s0.x), apply_signs(m0.y, s0.y), apply_signs(m1.x, s1.x), apply_signs(m1.y, s1.y)};
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(xo.A[2 * h + q], b, c, 0, 0, 0);
            }
            acc = fmaf(join_digits(c) * xo.meta[2 * g + h], 0.5f + (float)(a1 >> 28), acc);
        }
        return d * acc;
    }
};

/* IQ3_XXS [d][qs 64][8 x (4 x 7 sign bits + 4-bit scale)]: d*(0.5+s)*0.5 * grid byte * sign, a four-byte
 * grid entry per index byte (:2916-2940); 98-byte blocks */
template <> struct GridFmt<T_IQ3_XXS> {
    static constexpr int kBlock = 98, kGridBytes = 1024;
    static constexpr int kAlign = 2; /* what the loads want of the matrix address and the row pitch */
    static constexpr int kStep = 16; /* bytes between the x rows of consecutive instructions */
    static constexpr bool kAInRegs = true;
    static constexpr int kPiece = 2; /* every piece a lane reads starts 2 (mod 4) bytes into the block */
    static constexpr bool kSums = false;
    /* lane group g takes elements [64 g, 64 g + 64) in order, 16 per instruction */
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    __device__ static const uint32_t *grid_src() { return qlin_iq3xxs_grid; }
    struct Raw {
        Raw16 qs; /* index bytes of groups 2g, 2g+1 */
        Raw8 sc;  /* their sign + scale words */
        uint32_t d;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        r.qs = load16(blk + 2 + 16 * g);
        r.sc = load8(blk + 66 + 8 * g);
        r.d = *reinterpret_cast<const uint16_t *>(blk);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t sh, const Tables &t, int g) {
        uint32_t qs[4], sc[2];
        bytes16(r.qs, sh, qs);
        bytes8(r.sc, sh, sc);
        const float d = half_bits_fast(r.d) * 0.5f;
        float acc = 0.0f;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t a1 = sc[h];
            v4i c = {0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const uint32_t ix = qs[2 * h + q];
                const uint2 s0 = t.sign128[(a1 >> (14 * q)) & 127u], s1 = t.sign128[(a1 >> (14 * q + 7)) & 127u];
                const v4i b = {apply_signs(t.grid[ix & 255u], s0.x), apply_signs(t.grid[(ix >> 8) & 255u], s0.y),
                               apply_signs(t.grid[(ix >> 16) & 255u], s1.x), apply_signs(t.grid[ix >> 24], s1.y)};
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(xo.A[2 * h + q], b, c, 0, 0, 0);
            }
            acc = fmaf(join_digits(c) * xo.meta[2 * g + h], 0.5f + (float)(a1 >> 28), acc);
        }
        return d * acc;
    }
};

/* IQ3_S [d][qs 64][qh 8][signs 32][scales 4]: d*(1+2s) * grid byte * sign, 9-bit grid indices (:3022-3058);
 * 110-byte blocks */
template <> struct GridFmt<T_IQ3_S> {
    static constexpr int kBlock = 110, kGridBytes = 2048;
    static constexpr int kAlign = 2; /* what the loads want of the matrix address and the row pitch */
    static constexpr int kStep = 16; /* bytes between the x rows of consecutive instructions */
    static constexpr bool kAInRegs = true;
    static constexpr int kPiece = 2; /* every piece a lane reads starts 2 (mod 4) bytes into the block */
    static constexpr bool kSums = false;
    /* lane group g takes elements [64 g, 64 g + 64) in order, 16 per instruction */
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    __device__ static const uint32_t *grid_src() { return qlin_iq3s_grid; }
    struct Raw {
        Raw16 qs;  /* low index bytes of groups 2g, 2g+1 */
        Raw8 sg;   /* their sign bytes */
        uint32_t qh, scales, d; /* the ninth index bits (a byte per group), the byte with both 4-bit scales */
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        r.qs = load16(blk + 2 + 16 * g);
        r.sg = load8(blk + 74 + 8 * g);
        r.qh = *reinterpret_cast<const uint16_t *>(blk + 66 + 2 * g);
        r.scales = blk[106 + g];
        r.d = *reinterpret_cast<const uint16_t *>(blk);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t sh, const Tables &t, int g) {
        uint32_t qs[4], sg[2];
        bytes16(r.qs, sh, qs);
        bytes8(r.sg, sh, sg);
        const float d = half_bits_fast(r.d);
        float acc = 0.0f;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            v4i c = {0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const uint32_t ix = qs[2 * h + q];
                const uint32_t hb = r.qh >> (8 * h + 4 * q); /* bits 0..3: the ninth bits of these four indices */
                const uint2 s0 = t.sign256[(sg[h] >> (16 * q)) & 255u], s1 = t.sign256[(sg[h] >> (16 * q + 8)) & 255u];
                const uint32_t i0 = (ix & 255u) | ((hb & 1u) << 8), i1 = ((ix >> 8) & 255u) | ((hb & 2u) << 7);
                const uint32_t i2 = ((ix >> 16) & 255u) | ((hb & 4u) << 6), i3 = (ix >> 24) | ((hb & 8u) << 5);
                const v4i b = {apply_signs(t.grid[i0], s0.x), apply_signs(t.grid[i1], s0.y),
                               apply_signs(t.grid[i2], s1.x), apply_signs(t.grid[i3], s1.y)};
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(xo.A[2 * h + q], b, c, 0, 0, 0);
            }
            const uint32_t nib = (r.scales >> (4 * h)) & 15u;
            acc = fmaf(join_digits(c) * xo.meta[2 * g + h], (float)(1u + 2u * nib), acc);
        }
        return d * acc;
    }
};

/* IQ2_XS [d][32 x (9-bit grid index | 7 sign bits << 9)][8 scale bytes] (common/ggml_dequant.h:2975-2994), 74 bytes:
 * d * (0.5 + nibble) * 0.25 * grid byte * sign, an eight-byte grid entry per 16-bit code, one scale nibble per 16
 * elements. Lane group g takes groups 2g, 2g + 1: eight codes; an instruction is the two codes of one nibble. */
template <> struct GridFmt<T_IQ2_XS> {
    static constexpr int kBlock = 74, kGridBytes = 4096;
    static constexpr int kAlign = 2, kPiece = 2;
    static constexpr int kStep = 16;
    static constexpr bool kAInRegs = true, kSums = false;
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    __device__ static const uint32_t *grid_src() { return reinterpret_cast<const uint32_t *>(qlin_iq2xs_grid); }
    struct Raw {
        Raw16 qs;
        uint32_t sc, d;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        r.qs = load16(blk + 2 + 16 * g);
        r.sc = *reinterpret_cast<const uint16_t *>(blk + 66 + 2 * g);
        r.d = *reinterpret_cast<const uint16_t *>(blk);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t sh, const Tables &t, int g) {
        uint32_t w[4];
        bytes16(r.qs, sh, w);
        const uint2 *grid = reinterpret_cast<const uint2 *>(t.grid);
        float acc = 0.0f;
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const uint32_t u0 = w[st] & 0xFFFFu, u1 = w[st] >> 16;
            const uint2 m0 = grid[u0 & 511u], m1 = grid[u1 & 511u];
            const uint2 s0 = t.sign128[u0 >> 9], s1 = t.sign128[u1 >> 9];
            const v4i b = {apply_signs(m0.x, s0.x), apply_signs(m0.y, s0.y), apply_signs(m1.x, s1.x), apply_signs(m1.y, s1.y)};
            const v4i zero = {0, 0, 0, 0};
            const v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(xo.A[st], b, zero, 0, 0, 0);
            const uint32_t nib = (r.sc >> (8 * (st >> 1) + 4 * (st & 1))) & 15u;
            acc = fmaf(join_digits(c) * xo.meta[2 * g + (st >> 1)], 0.5f + (float)nib, acc);
        }
        return half_bits_fast(r.d) * 0.25f * acc;
    }
};

/* IQ2_S [d][32 index bytes][32 sign bytes][qh 8][8 scale bytes] (:2996-3020), 82 bytes: as IQ2_XS with a 10-bit
 * index (two high bits per code in qh) into a 1024-entry grid and explicit sign bytes. */
template <> struct GridFmt<T_IQ2_S> {
    static constexpr int kBlock = 82, kGridBytes = 8192;
    static constexpr int kAlign = 2, kPiece = 2;
    static constexpr int kStep = 16;
    static constexpr bool kAInRegs = true, kSums = false;
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    __device__ static const uint32_t *grid_src() { return reinterpret_cast<const uint32_t *>(qlin_iq2s_grid); }
    struct Raw {
        Raw8 qs, sg;
        uint32_t qh, sc, d;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        r.qs = load8(blk + 2 + 8 * g);
        r.sg = load8(blk + 34 + 8 * g);
        r.qh = *reinterpret_cast<const uint16_t *>(blk + 66 + 2 * g);
        r.sc = *reinterpret_cast<const uint16_t *>(blk + 74 + 2 * g);
        r.d = *reinterpret_cast<const uint16_t *>(blk);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t sh, const Tables &t, int g) {
        uint32_t q[2], sg[2];
        bytes8(r.qs, sh, q);
        bytes8(r.sg, sh, sg);
        const uint2 *grid = reinterpret_cast<const uint2 *>(t.grid);
        float acc = 0.0f;
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const int h = st >> 1, l0 = 2 * (st & 1);
            const uint32_t qhb = (r.qh >> (8 * h)) & 0xFFu;
            const uint32_t i0 = ((q[h] >> (8 * l0)) & 0xFFu) | ((qhb << (8 - 2 * l0)) & 0x300u);
            const uint32_t i1 = ((q[h] >> (8 * l0 + 8)) & 0xFFu) | ((qhb << (6 - 2 * l0)) & 0x300u);
            const uint2 m0 = grid[i0], m1 = grid[i1];
            const uint2 s0 = t.sign256[(sg[h] >> (8 * l0)) & 0xFFu], s1 = t.sign256[(sg[h] >> (8 * l0 + 8)) & 0xFFu];
            const v4i b = {apply_signs(m0.x, s0.x), apply_signs(m0.y, s0.y), apply_signs(m1.x, s1.x), apply_signs(m1.y, s1.y)};
            const v4i zero = {0, 0, 0, 0};
            const v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(xo.A[st], b, zero, 0, 0, 0);
            const uint32_t nib = (r.sc >> (8 * h + 4 * (st & 1))) & 15u;
            acc = fmaf(join_digits(c) * xo.meta[2 * g + h], 0.5f + (float)nib, acc);
        }
        return half_bits_fast(r.d) * 0.25f * acc;
    }
};

/* IQ1_S [d][32 index bytes][8 x u16: 4 x 3 high index bits, 3-bit scale, shift sign] (common/ggml_dequant.h:3062-3083),
 * 50 bytes: d * (2 s + 1) * (t + delta), t in {-1, 0, 1} from an eight-byte entry of a 2048-entry grid, delta = +-1/8
 * per 32 elements. The grid bytes are the signed codes; delta goes onto the sum of x. */
template <> struct GridFmt<T_IQ1_S> {
    static constexpr int kBlock = 50, kGridBytes = 16384;
    static constexpr int kAlign = 2, kPiece = 2;
    static constexpr int kStep = 16;
    static constexpr bool kAInRegs = true, kSums = true;
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    __device__ static const uint32_t *grid_src() { return reinterpret_cast<const uint32_t *>(qlin_iq1s_grid); }
    struct Raw {
        Raw8 qs;
        uint32_t qh_q, qh_tail, d; /* the two u16 of groups 2g, 2g + 1: aligned dword and, off the grid, the tail */
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        r.qs = load8(blk + 2 + 8 * g);
        const uint8_t *p = blk + 34 + 4 * g;
        const uint32_t odd = (uint32_t)(uintptr_t)p & 2u;
        r.qh_q = *reinterpret_cast<const uint32_t *>(p - odd);
        r.qh_tail = 0;
        if (odd) r.qh_tail = *reinterpret_cast<const uint16_t *>(p + 2);
        r.d = *reinterpret_cast<const uint16_t *>(blk);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t sh, const Tables &t, int g) {
        uint32_t q[2];
        bytes8(r.qs, sh, q);
        const uint32_t qh2 = __builtin_amdgcn_alignbit(r.qh_tail, r.qh_q, sh);
        const uint2 *grid = reinterpret_cast<const uint2 *>(t.grid);
        float acc = 0.0f;
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const int h = st >> 1, l0 = 2 * (st & 1);
            const uint32_t qh = (qh2 >> (16 * h)) & 0xFFFFu;
            const uint32_t i0 = ((q[h] >> (8 * l0)) & 0xFFu) | (((qh >> (3 * l0)) & 7u) << 8);
            const uint32_t i1 = ((q[h] >> (8 * l0 + 8)) & 0xFFu) | (((qh >> (3 * l0 + 3)) & 7u) << 8);
            const uint2 m0 = grid[i0], m1 = grid[i1];
            const v4i b = {(int)m0.x, (int)m0.y, (int)m1.x, (int)m1.y};
            const v4i zero = {0, 0, 0, 0};
            const v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(xo.A[st], b, zero, 0, 0, 0);
            const float dl = (float)(2u * ((qh >> 12) & 7u) + 1u);
            const float delta = (qh & 0x8000u) ? -0.125f : 0.125f;
            const int e0 = elem0(g, st);
            acc = fmaf(dl, fmaf(join_digits(c), xo.meta[e0 >> 5], delta * xo.meta[8 + (e0 >> 4)]), acc);
        }
        return half_bits_fast(r.d) * acc;
    }
};

/* IQ1_M [32 index bytes][qh 16][8 scale bytes] (common/ggml_dequant.h:3084-3126), 56 bytes and no d field (its
 * four nibbles sit on top of the four scale words): d * (2 s + 1) * (t + delta) with the IQ1_S grid, a 3-bit scale
 * per 16 elements and delta = +-1/8 per 8. The codes are 8 t + (+-1), signed bytes picked from a four-byte table by
 * the grid byte's two low bits (t = -1, 0, 1 are 0xFF, 0, 1), and the scale carries the 1/8. */
template <> struct GridFmt<T_IQ1_M> {
    static constexpr int kBlock = 56, kGridBytes = 16384;
    static constexpr int kAlign = 4, kPiece = 0;
    static constexpr int kStep = 16;
    static constexpr bool kAInRegs = true, kSums = false;
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    __device__ static const uint32_t *grid_src() { return reinterpret_cast<const uint32_t *>(qlin_iq1s_grid); }
    struct Raw {
        u32x2_a4 qs, sc;
        uint32_t qh;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        r.qs = *reinterpret_cast<const u32x2_a4 *>(blk + 8 * g);
        r.qh = *reinterpret_cast<const uint32_t *>(blk + 32 + 4 * g);
        r.sc = *reinterpret_cast<const u32x2_a4 *>(blk + 48);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t, const Tables &t, int g) {
        const uint32_t q[2] = {r.qs.x, r.qs.y};
        const uint2 *grid = reinterpret_cast<const uint2 *>(t.grid);
        const uint32_t dbits = ((r.sc.x >> 12) & 0x000Fu) | ((r.sc.x >> 24) & 0x00F0u) | ((r.sc.y >> 4) & 0x0F00u) | ((r.sc.y >> 16) & 0xF000u);
        const uint32_t scg = ((g & 2) ? r.sc.y : r.sc.x) >> (16 * (g & 1)); /* scale word g: groups 2g and 2g + 1 */
        /* codes of t = 0, 1, (unused), -1 for delta = +1/8 and -1/8, as 8 t + (+-1) */
        constexpr uint32_t kPlus = 0xF9000901u, kMinus = 0xF70007FFu;
        float acc = 0.0f;
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const int h = st >> 1, l0 = 2 * (st & 1);
            const uint32_t qb = (r.qh >> (8 * (2 * h + (st & 1)))) & 0xFFu;
            const uint32_t i0 = ((q[h] >> (8 * l0)) & 0xFFu) | ((qb << 8) & 0x700u);
            const uint32_t i1 = ((q[h] >> (8 * l0 + 8)) & 0xFFu) | ((qb << 4) & 0x700u);
            const uint2 m0 = grid[i0], m1 = grid[i1];
            const uint32_t t0 = (qb & 0x08u) ? kMinus : kPlus, t1 = (qb & 0x80u) ? kMinus : kPlus;
            const v4i b = {(int)__builtin_amdgcn_perm(0u, t0, m0.x & 0x03030303u), (int)__builtin_amdgcn_perm(0u, t0, m0.y & 0x03030303u),
                           (int)__builtin_amdgcn_perm(0u, t1, m1.x & 0x03030303u), (int)__builtin_amdgcn_perm(0u, t1, m1.y & 0x03030303u)};
            const v4i zero = {0, 0, 0, 0};
            const v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(xo.A[st], b, zero, 0, 0, 0);
            const uint32_t s3 = (scg >> (6 * h + 3 * (st & 1))) & 7u;
            acc = fmaf((float)(2u * s3 + 1u), join_digits(c) * xo.meta[2 * g + h], acc);
        }
        return half_bits_fast(dbits) * 0.125f * acc;
    }
};

/* Q6_K [ql 128][qh 64][16 int8 scales][d]: d * sc * (q - 32), q = low nibble | two high bits << 4, one scale per
 * 16 elements (common/ggml_dequant.h:1653-1687); 210-byte blocks. Element 128 h + 32 q + l (h = half, q = 0..3,
 * l < 32) has its nibble in ql[64 h + 32 (q & 1) + l] (the high one for q >= 2) and its high bits in
 * qh[32 h + l] >> 2 q. Lane group g = (h, p) takes l in [16 p, 16 p + 16) of all four q: instruction q, sixteen
 * elements of one scale. The codes stay unsigned (0..63); the -32 goes onto the sum of x. */
template <> struct GridFmt<T_Q6_K> {
    static constexpr int kBlock = 210, kGridBytes = 0;
    static constexpr int kAlign = 2; /* what the loads want of the matrix address and the row pitch */
    static constexpr int kStep = 32;
    static constexpr bool kAInRegs = false; /* no table lookups: LDS has time to deliver the x operand per item */
    static constexpr int kPiece = 0;
    static constexpr bool kSums = true;
    __device__ static const uint32_t *grid_src() { return nullptr; }
    __device__ static int elem0(int g, int st) { return 128 * (g >> 1) + 32 * st + 16 * (g & 1); }
    struct Raw {
        Raw16 qa, qb, qh; /* ql[64 h + 16 p ..], ql[64 h + 32 + 16 p ..], qh[32 h + 16 p ..] */
        Raw8 sc;          /* the eight scales of the half */
        uint32_t d;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        const int h = g >> 1, p = g & 1;
        r.qa = load16(blk + 64 * h + 16 * p);
        r.qb = load16(blk + 64 * h + 32 + 16 * p);
        r.qh = load16(blk + 128 + 32 * h + 16 * p);
        r.sc = load8(blk + 192 + 8 * h);
        r.d = *reinterpret_cast<const uint16_t *>(blk + 208);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t sh, const Tables &, int g) {
        uint32_t qa[4], qb[4], qh[4], sc[2];
        bytes16(r.qa, sh, qa);
        bytes16(r.qb, sh, qb);
        bytes16(r.qh, sh, qh);
        bytes8(r.sc, sh, sc);
        const uint32_t scp = (g & 1) ? (sc[0] >> 8) | (sc[1] << 24) : sc[0]; /* byte 2 q (q < 2): scale of (q, p) */
        const uint32_t scq = (g & 1) ? sc[1] >> 8 : sc[1];                  /* byte 2 (q - 2) for q >= 2 */
        float acc = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t(&ql)[4] = (q & 1) ? qb : qa;
            v4i b;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t lo = (ql[i] >> (4 * (q >> 1))) & 0x0F0F0F0Fu;
                const uint32_t hi = ((qh[i] >> (2 * q)) & 0x03030303u) << 4;
                b[i] = (int)(lo | hi);
            }
            const v4i zero = {0, 0, 0, 0};
            const uint4 av = *reinterpret_cast<const uint4 *>(xo.arows + kStep * q);
            const v4i a = {(int)av.x, (int)av.y, (int)av.z, (int)av.w};
            const v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, zero, 0, 0, 0);
            const uint32_t w = q < 2 ? scp >> (16 * q) : scq >> (16 * (q - 2));
            const float scale = (float)(int)(int8_t)(w & 0xFFu);
            const int e0 = elem0(g, q);
            acc = fmaf(scale, fmaf(join_digits(c), xo.meta[e0 >> 5], -32.0f * xo.meta[8 + (e0 >> 4)]), acc);
        }
        return half_bits_fast(r.d) * acc;
    }
};

/* Q8_0 [d][32 x int8] x 8 per 256 elements (common/ggml_dequant.h:1479-1489): 272 bytes, so a row of whole
 * 256-element groups keeps the alignment of the matrix. Lane group g takes blocks 2g, 2g+1: 68 bytes, 17 dwords. */
template <> struct GridFmt<T_Q8_0> {
    static constexpr int kBlock = 272, kGridBytes = 0;
    static constexpr int kPiece = 0, kAlign = 4;
    static constexpr int kStep = 16;
    static constexpr bool kSums = false, kAInRegs = false;
    __device__ static const uint32_t *grid_src() { return nullptr; }
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    struct Raw {
        u32x4_a4 a, b, c, d;
        uint32_t e;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        const uint8_t *p = blk + 68 * g;
        r.a = *reinterpret_cast<const u32x4_a4 *>(p);
        r.b = *reinterpret_cast<const u32x4_a4 *>(p + 16);
        r.c = *reinterpret_cast<const u32x4_a4 *>(p + 32);
        r.d = *reinterpret_cast<const u32x4_a4 *>(p + 48);
        r.e = *reinterpret_cast<const uint32_t *>(p + 64);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t, const Tables &, int g) {
        const uint32_t w[17] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w, r.c.x,
                                r.c.y, r.c.z, r.c.w, r.d.x, r.d.y, r.d.z, r.d.w, r.e};
        float acc = 0.0f;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            v4i c = {0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < 2; q++) {
                v4i b;
#pragma unroll
                for (int i = 0; i < 4; i++) /* block 0: the codes start 2 bytes into dword 0; block 1: at dword 9 */
                    b[i] = h == 0 ? (int)__builtin_amdgcn_alignbit(w[4 * q + i + 1], w[4 * q + i], 16) : (int)w[9 + 4 * q + i];
                const uint4 av = *reinterpret_cast<const uint4 *>(xo.arows + kStep * (2 * h + q));
                const v4i a = {(int)av.x, (int)av.y, (int)av.z, (int)av.w};
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
            }
            const float d = half_bits_fast(h == 0 ? w[0] & 0xFFFFu : w[8] >> 16);
            acc = fmaf(join_digits(c) * xo.meta[2 * g + h], d, acc);
        }
        return acc;
    }
};

/* Q5_K [d][dmin][12 bytes of 6-bit scales and mins][qh 32][qs 128] (:1620-1651), 176 bytes: element 64 j + 32 u + l
 * has its nibble in qs[32 j + l] (the high one for u = 1) and its fifth bit in qh[l] >> (2 j + u); (d sc) q - dmin m
 * with one scale and min per 32 elements. Lane group g takes j = g: low nibbles, then high nibbles. */
template <> struct GridFmt<T_Q5_K> {
    static constexpr int kBlock = 176, kGridBytes = 0;
    static constexpr int kPiece = 0, kAlign = 16;
    static constexpr int kStep = 16;
    static constexpr bool kSums = true, kAInRegs = false;
    __device__ static const uint32_t *grid_src() { return nullptr; }
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    struct Raw {
        uint4 hd, qh0, qh1, qs0, qs1;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        r.hd = *reinterpret_cast<const uint4 *>(blk);
        r.qh0 = *reinterpret_cast<const uint4 *>(blk + 16);
        r.qh1 = *reinterpret_cast<const uint4 *>(blk + 32);
        r.qs0 = *reinterpret_cast<const uint4 *>(blk + 48 + 32 * g);
        r.qs1 = *reinterpret_cast<const uint4 *>(blk + 64 + 32 * g);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t, const Tables &, int g) {
        const uint32_t qs[8] = {r.qs0.x, r.qs0.y, r.qs0.z, r.qs0.w, r.qs1.x, r.qs1.y, r.qs1.z, r.qs1.w};
        const uint32_t qh[8] = {r.qh0.x, r.qh0.y, r.qh0.z, r.qh0.w, r.qh1.x, r.qh1.y, r.qh1.z, r.qh1.w};
        float dots = 0.0f, mins = 0.0f;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            v4i c = {0, 0, 0, 0};
#pragma unroll
            for (int hf = 0; hf < 2; hf++) {
                v4i b;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t lo = (qs[4 * hf + i] >> (4 * u)) & 0x0F0F0F0Fu;
                    const uint32_t hi = ((qh[4 * hf + i] >> (2 * g + u)) & 0x01010101u) << 4;
                    b[i] = (int)(lo | hi);
                }
                const uint4 av = *reinterpret_cast<const uint4 *>(xo.arows + kStep * (2 * u + hf));
                const v4i a = {(int)av.x, (int)av.y, (int)av.z, (int)av.w};
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
            }
            /* get_scale_min_k4 (:1582-1590) for sub-block j = 2g + u, from the header's registers */
            const int j = 2 * g + u;
            const uint32_t at = 8u * (uint32_t)(j & 3);
            const uint32_t yb = __builtin_amdgcn_ubfe(r.hd.y, at, 8), zb = __builtin_amdgcn_ubfe(r.hd.z, at, 8);
            const uint32_t wb = __builtin_amdgcn_ubfe(r.hd.w, at, 8);
            const uint32_t sc = j < 4 ? yb & 63u : (wb & 15u) | ((yb >> 6) << 4);
            const uint32_t mn = j < 4 ? zb & 63u : (wb >> 4) | ((zb >> 6) << 4);
            dots = fmaf((float)sc, join_digits(c) * xo.meta[j], dots);
            mins = fmaf((float)mn, xo.meta[8 + 2 * j] + xo.meta[8 + 2 * j + 1], mins);
        }
        return half_bits_fast(r.hd.x & 0xFFFFu) * dots - half_bits_fast(r.hd.x >> 16) * mins;
    }
};

/* Q2_K [16 scale bytes][qs 64][d][dmin] (common/ggml_dequant.h:1505-1534), 84 bytes: element 128 h + 32 j + l
 * (l < 32) is bits 2j, 2j+1 of qs[32 h + l], scaled by d * (low nibble) and offset by -dmin * (high nibble) of
 * scale byte 8 h + 2 j + l / 16. Lane group g = (h, p) takes l in [16 p, 16 p + 16) of all four j, as Q6_K. */
template <> struct GridFmt<T_Q2_K> {
    static constexpr int kBlock = 84, kGridBytes = 0;
    static constexpr int kPiece = 0, kAlign = 4;
    static constexpr int kStep = 32;
    static constexpr bool kSums = true, kAInRegs = false;
    __device__ static const uint32_t *grid_src() { return nullptr; }
    __device__ static int elem0(int g, int st) { return 128 * (g >> 1) + 32 * st + 16 * (g & 1); }
    struct Raw {
        u32x4_a4 qs;
        u32x2_a4 sc; /* the eight scale bytes of the half */
        uint32_t dd;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        r.qs = *reinterpret_cast<const u32x4_a4 *>(blk + 16 + 16 * g);
        r.sc = *reinterpret_cast<const u32x2_a4 *>(blk + 8 * (g >> 1));
        r.dd = *reinterpret_cast<const uint32_t *>(blk + 80);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t, const Tables &, int g) {
        const uint32_t qs[4] = {r.qs.x, r.qs.y, r.qs.z, r.qs.w};
        const uint32_t scp = (g & 1) ? (r.sc.x >> 8) | (r.sc.y << 24) : r.sc.x; /* byte 2 j (j < 2): scale of (j, p) */
        const uint32_t scq = (g & 1) ? r.sc.y >> 8 : r.sc.y;                    /* byte 2 (j - 2) for j >= 2 */
        float dots = 0.0f, mins = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            v4i b;
#pragma unroll
            for (int i = 0; i < 4; i++) b[i] = (int)((qs[i] >> (2 * j)) & 0x03030303u);
            const v4i zero = {0, 0, 0, 0};
            const uint4 av = *reinterpret_cast<const uint4 *>(xo.arows + kStep * j);
            const v4i a = {(int)av.x, (int)av.y, (int)av.z, (int)av.w};
            const v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, zero, 0, 0, 0);
            const uint32_t w = (j < 2 ? scp >> (16 * j) : scq >> (16 * (j - 2))) & 0xFFu;
            const int e0 = elem0(g, j);
            dots = fmaf((float)(w & 15u), join_digits(c) * xo.meta[e0 >> 5], dots);
            mins = fmaf((float)(w >> 4), xo.meta[8 + (e0 >> 4)], mins);
        }
        return half_bits_fast(r.dd & 0xFFFFu) * dots - half_bits_fast(r.dd >> 16) * mins;
    }
};

/* TQ2_0 [qs 64][d] (common/ggml_dequant.h:3161-3176), 66 bytes: element 128 h + 32 l + m (m < 32) is bits 2l, 2l+1
 * of qs[32 h + m], minus 1, times d. Lane group g = (h, p) takes m in [16 p, 16 p + 16) of all four l, as Q6_K; the
 * codes stay unsigned (0..2) and the -1 goes onto the sum of x. */
template <> struct GridFmt<T_TQ2_0> {
    static constexpr int kBlock = 66, kGridBytes = 0;
    static constexpr int kPiece = 0, kAlign = 2;
    static constexpr int kStep = 32;
    static constexpr bool kSums = true, kAInRegs = false;
    __device__ static const uint32_t *grid_src() { return nullptr; }
    __device__ static int elem0(int g, int st) { return 128 * (g >> 1) + 32 * st + 16 * (g & 1); }
    struct Raw {
        Raw16 qs;
        uint32_t d;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        r.qs = load16(blk + 16 * g);
        r.d = *reinterpret_cast<const uint16_t *>(blk + 64);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t sh, const Tables &, int g) {
        uint32_t qs[4];
        bytes16(r.qs, sh, qs);
        float acc = 0.0f;
#pragma unroll
        for (int l = 0; l < 4; l++) {
            v4i b;
#pragma unroll
            for (int i = 0; i < 4; i++) b[i] = (int)((qs[i] >> (2 * l)) & 0x03030303u);
            const v4i zero = {0, 0, 0, 0};
            const uint4 av = *reinterpret_cast<const uint4 *>(xo.arows + kStep * l);
            const v4i a = {(int)av.x, (int)av.y, (int)av.z, (int)av.w};
            const v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, zero, 0, 0, 0);
            const int e0 = elem0(g, l);
            acc += fmaf(join_digits(c), xo.meta[e0 >> 5], -xo.meta[8 + (e0 >> 4)]);
        }
        return half_bits_fast(r.d) * acc;
    }
};

/* Q1_0 [d][128 bits] per 128 elements (common/ggml_dequant.h:1491-1503), 18 bytes: bit set -> +d, clear -> -d; 36
 * bytes per 256 elements. Lane group g takes 64 bits of block g / 2, which start 2 (mod 4) bytes into the 36 for the
 * first block: aligned dwords and a funnel shift there. The codes are the bits; 2 * (bits . x) - sum of x. */
template <> struct GridFmt<T_Q1_0> {
    static constexpr int kBlock = 36, kGridBytes = 0;
    static constexpr int kPiece = 0, kAlign = 4;
    static constexpr int kStep = 16;
    static constexpr bool kSums = true, kAInRegs = false;
    __device__ static const uint32_t *grid_src() { return nullptr; }
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    struct Raw {
        u32x2_a4 q;
        uint32_t tail, d;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        const int off = 18 * (g >> 1) + 2 + 8 * (g & 1); /* 2, 10, 20, 28 */
        const uint8_t *p = blk + (off & ~3);
        r.q = *reinterpret_cast<const u32x2_a4 *>(p);
        r.tail = 0;
        if (g < 2) r.tail = *reinterpret_cast<const uint32_t *>(p + 8); /* the second block's bits start on a dword */
        r.d = *reinterpret_cast<const uint16_t *>(blk + 18 * (g >> 1));
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t, const Tables &, int g) {
        const uint32_t sh = g < 2 ? 16u : 0u;
        const uint32_t bits[2] = {__builtin_amdgcn_alignbit(r.q.y, r.q.x, sh), __builtin_amdgcn_alignbit(r.tail, r.q.y, sh)};
        float acc = 0.0f;
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const uint32_t b16 = bits[st >> 1] >> (16 * (st & 1));
            const v4i b = {(int)spread4(b16), (int)spread4(b16 >> 4), (int)spread4(b16 >> 8), (int)spread4(b16 >> 12)};
            const v4i zero = {0, 0, 0, 0};
            const uint4 av = *reinterpret_cast<const uint4 *>(xo.arows + kStep * st);
            const v4i a = {(int)av.x, (int)av.y, (int)av.z, (int)av.w};
            const v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, zero, 0, 0, 0);
            const int e0 = elem0(g, st);
            acc += fmaf(2.0f * join_digits(c), xo.meta[e0 >> 5], -xo.meta[8 + (e0 >> 4)]);
        }
        return half_bits_fast(r.d) * acc;
    }
};

/* four bytes at p (2-byte aligned, at least two bytes into a block) */
struct Raw4 {
    uint32_t q, tail;
};
__device__ __forceinline__ Raw4 load4(const uint8_t *p) {
    Raw4 r;
    const uint32_t odd = (uint32_t)(uintptr_t)p & 2u;
    r.q = *reinterpret_cast<const uint32_t *>(p - odd);
    r.tail = 0;
    if (odd) r.tail = *reinterpret_cast<const uint16_t *>(p + 2);
    return r;
}

/* TQ1_0 [qs 48][qh 4][d] (common/ggml_dequant.h:3127-3160), 54 bytes: base-3 digits, five to a byte of qs and four to
 * a byte of qh; digit n of byte b is ((uint8)(b * 3^n) * 3) >> 8, the value (digit - 1) * d. Elements in runs of 16:
 * runs 0..9 are digit n = run / 2 of qs[16 (run % 2) ..], runs 10..14 digit run - 10 of qs[32..48), run 15 the digits
 * 0..3 of qh[0..4) (element 4 n + j = digit n of qh[j]). Lane group g takes runs 4g..4g + 3; every lane reads the
 * three 16-byte pieces of qs and qh and picks. The codes stay unsigned (0..2); the -1 goes onto the sum of x. */
template <> struct GridFmt<T_TQ1_0> {
    static constexpr int kBlock = 54, kGridBytes = 0;
    static constexpr int kPiece = 0, kAlign = 2;
    static constexpr int kStep = 16;
    static constexpr bool kSums = true, kAInRegs = false;
    __device__ static const uint32_t *grid_src() { return nullptr; }
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    struct Raw {
        Raw16 a, b, c;
        Raw4 qh;
        uint32_t d;
    };
    __device__ static Raw load(const uint8_t *blk, int) {
        Raw r;
        r.a = load16(blk);
        r.b = load16(blk + 16);
        r.c = load16(blk + 32);
        r.qh = load4(blk + 48);
        r.d = *reinterpret_cast<const uint16_t *>(blk + 52);
        return r;
    }
    /* digit of four bytes: ((b * pw) mod 256) * 3 >> 8, two bytes at a time in the halves of a dword */
    __device__ static uint32_t digits4(uint32_t w, uint32_t pw) {
        const uint32_t lo = (((w & 0x00FF00FFu) * pw) & 0x00FF00FFu) * 3u, hi = ((((w >> 8) & 0x00FF00FFu) * pw) & 0x00FF00FFu) * 3u;
        return ((lo >> 8) & 0x00030003u) | (hi & 0x03000300u);
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t sh, const Tables &, int g) {
        uint32_t a[4], b[4], c[4];
        bytes16(r.a, sh, a);
        bytes16(r.b, sh, b);
        bytes16(r.c, sh, c);
        const uint32_t qh = __builtin_amdgcn_alignbit(r.qh.tail, r.qh.q, sh);
        /* power of 3 of run 4g + st: runs 0..9 -> run / 2, runs 10..14 -> run - 10 */
        float acc = 0.0f;
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const int run = 4 * g + st;
            const bool from_c = run >= 10, special = run == 15;
            const int n = from_c ? run - 10 : run >> 1;
            const uint32_t pw = n == 0 ? 1u : n == 1 ? 3u : n == 2 ? 9u : n == 3 ? 27u : 81u;
            v4i code;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t src = special ? qh : from_c ? c[i] : (run & 1) ? b[i] : a[i];
                const uint32_t p = special ? (i == 0 ? 1u : i == 1 ? 3u : i == 2 ? 9u : 27u) : pw;
                code[i] = (int)digits4(src, p);
            }
            const v4i zero = {0, 0, 0, 0};
            const uint4 av = *reinterpret_cast<const uint4 *>(xo.arows + kStep * st);
            const v4i av4 = {(int)av.x, (int)av.y, (int)av.z, (int)av.w};
            const v4i cc = __builtin_amdgcn_mfma_i32_16x16x64_i8(av4, code, zero, 0, 0, 0);
            const int e0 = elem0(g, st);
            acc += fmaf(join_digits(cc), xo.meta[e0 >> 5], -xo.meta[8 + (e0 >> 4)]);
        }
        return half_bits_fast(r.d) * acc;
    }
};

/* Q3_K [hmask 32][qs 64][12 packed scale bytes][d] (:1536-1580), 110 bytes: element 128 h + 32 j + l (l < 32) is
 * bits 2j, 2j+1 of qs[32 h + l], minus 4 unless bit 4 h + j of hmask[l] is set, times d * (6-bit scale - 32) of
 * index 8 h + 2 j + l / 16: low nibbles in bytes 0..7 (index & 7, the high nibble for indices 8..15), the two high
 * bits of index i in byte 8 + (i & 3) at bit 2 (i >> 2). Lane group g = (h, p) as Q6_K; the codes stay unsigned
 * (0..7) and the -4 goes onto the sum of x. */
template <> struct GridFmt<T_Q3_K> {
    static constexpr int kBlock = 110, kGridBytes = 0;
    static constexpr int kPiece = 0, kAlign = 2;
    static constexpr int kStep = 32;
    static constexpr bool kSums = true, kAInRegs = false;
    __device__ static const uint32_t *grid_src() { return nullptr; }
    __device__ static int elem0(int g, int st) { return 128 * (g >> 1) + 32 * st + 16 * (g & 1); }
    struct Raw {
        Raw16 qs, hm;
        Raw8 lo; /* scale bytes 0..7 */
        Raw4 hi; /* scale bytes 8..11 */
        uint32_t d;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        r.qs = load16(blk + 32 + 16 * g);
        r.hm = load16(blk + 16 * (g & 1));
        r.lo = load8(blk + 96);
        r.hi = load4(blk + 104);
        r.d = *reinterpret_cast<const uint16_t *>(blk + 108);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t sh, const Tables &, int g) {
        uint32_t qs[4], hm[4], lo[2];
        bytes16(r.qs, sh, qs);
        bytes16(r.hm, sh, hm);
        bytes8(r.lo, sh, lo);
        const uint32_t hi = __builtin_amdgcn_alignbit(r.hi.tail, r.hi.q, sh);
        const int h = g >> 1, p = g & 1;
        const uint32_t scp = p ? (lo[0] >> 8) | (lo[1] << 24) : lo[0]; /* byte 2 j (j < 2) */
        const uint32_t scq = p ? lo[1] >> 8 : lo[1];                   /* byte 2 (j - 2) for j >= 2 */
        float acc = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            v4i b;
#pragma unroll
            for (int i = 0; i < 4; i++)
                b[i] = (int)(((qs[i] >> (2 * j)) & 0x03030303u) | (((hm[i] >> (4 * h + j)) & 0x01010101u) << 2));
            const v4i zero = {0, 0, 0, 0};
            const uint4 av = *reinterpret_cast<const uint4 *>(xo.arows + kStep * j);
            const v4i a = {(int)av.x, (int)av.y, (int)av.z, (int)av.w};
            const v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, zero, 0, 0, 0);
            const uint32_t w = j < 2 ? scp >> (16 * j) : scq >> (16 * (j - 2));
            const uint32_t low = (w >> (4 * h)) & 15u;
            const uint32_t high = (hi >> (8 * (2 * (j & 1) + p) + 2 * (2 * h + (j >> 1)))) & 3u;
            const float scale = (float)((int)(low | (high << 4)) - 32);
            const int e0 = elem0(g, j);
            acc = fmaf(scale, fmaf(join_digits(c), xo.meta[e0 >> 5], -4.0f * xo.meta[8 + (e0 >> 4)]), acc);
        }
        return half_bits_fast(r.d) * acc;
    }
};

/* the sixteen signed bytes of the IQ4 codebook (common/ggml_dequant.h:2942-2954) in four registers, and its
 * lookup for four nibbles at once: two byte permutes and a select by the nibbles' top bits */
struct Table16 {
    uint32_t t0, t1, t2, t3;
};
__device__ __forceinline__ Table16 table16(const int8_t *values) {
    const uint4 v = *reinterpret_cast<const uint4 *>(values);
    const Table16 t = {v.x, v.y, v.z, v.w};
    return t;
}
__device__ __forceinline__ int look4(uint32_t n, const Table16 &t) {
    const uint32_t sel = n & 0x07070707u;
    const uint32_t lo = __builtin_amdgcn_perm(t.t1, t.t0, sel), hi = __builtin_amdgcn_perm(t.t3, t.t2, sel);
    const uint32_t m = ((n >> 3) & 0x01010101u) * 0xFFu;
    return (int)((hi & m) | (lo & ~m));
}

/* IQ4_NL [d][16 bytes of nibbles] x 8 per 256 elements (:2942-2954): d * table[nibble]; element l of a block is the
 * low nibble of byte l, element 16 + l the high one. 144 bytes per 256 elements; lane group g takes blocks 2g, 2g+1:
 * 36 bytes, nine dwords. Q4_0 (:2850-2862) has the same layout with d * (nibble - 8): its codes stay unsigned and
 * the -8 goes onto the sum of x. */
template <uint32_t T> struct Nibble18 {
    static constexpr int kBlock = 144, kGridBytes = 0;
    static constexpr int kPiece = 0, kAlign = 4;
    static constexpr int kStep = 16;
    static constexpr bool kSums = T == T_Q4_0, kAInRegs = false;
    __device__ static const uint32_t *grid_src() { return nullptr; }
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    struct Raw {
        u32x4_a4 a, b;
        uint32_t c;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        const uint8_t *p = blk + 36 * g;
        r.a = *reinterpret_cast<const u32x4_a4 *>(p);
        r.b = *reinterpret_cast<const u32x4_a4 *>(p + 16);
        r.c = *reinterpret_cast<const uint32_t *>(p + 32);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t, const Tables &, int g) {
        const uint32_t w[9] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w, r.c};
        const Table16 tab = table16(qlin_iq4nl_values);
        float acc = 0.0f;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint32_t qs[4]; /* block 0: the nibble bytes start 2 bytes into dword 0; block 1: at dword 5 */
#pragma unroll
            for (int i = 0; i < 4; i++) qs[i] = h == 0 ? __builtin_amdgcn_alignbit(w[i + 1], w[i], 16) : w[5 + i];
            v4i c = {0, 0, 0, 0};
#pragma unroll
            for (int u = 0; u < 2; u++) {
                v4i b;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t nib = (qs[i] >> (4 * u)) & 0x0F0F0F0Fu;
                    b[i] = T == T_Q4_0 ? (int)nib : look4(nib, tab);
                }
                const uint4 av = *reinterpret_cast<const uint4 *>(xo.arows + kStep * (2 * h + u));
                const v4i a = {(int)av.x, (int)av.y, (int)av.z, (int)av.w};
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
            }
            const float d = half_bits_fast(h == 0 ? w[0] & 0xFFFFu : w[4] >> 16);
            const int G = 2 * g + h;
            float dot = join_digits(c) * xo.meta[G];
            if (T == T_Q4_0) dot = fmaf(-8.0f, xo.meta[8 + 2 * G] + xo.meta[8 + 2 * G + 1], dot);
            acc = fmaf(dot, d, acc);
        }
        return acc;
    }
};
template <> struct GridFmt<T_IQ4_NL> : Nibble18<T_IQ4_NL> {};
template <> struct GridFmt<T_Q4_0> : Nibble18<T_Q4_0> {};

/* MXFP4 [e][16 nibble bytes] (common/ggml_dequant.h:2818-2830), 17 bytes: table[nibble] * 2^(e - 127) / 2, low
 * nibbles first as in IQ4_NL; 136 bytes per 256 elements. Lane group g takes blocks 2g and 2g + 1, the 34 bytes from
 * byte 34 g - which is 2 (mod 4) for odd g: nine aligned dwords from two bytes earlier there, and byte shifts. */
template <> struct GridFmt<T_MXFP4> {
    static constexpr int kBlock = 136, kGridBytes = 0;
    static constexpr int kPiece = 0, kAlign = 4;
    static constexpr int kStep = 16;
    static constexpr bool kSums = false, kAInRegs = false;
    __device__ static const uint32_t *grid_src() { return nullptr; }
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    struct Raw {
        u32x4_a4 a, b;
        uint32_t c;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        const uint8_t *p = blk + 34 * g - 2 * (g & 1);
        r.a = *reinterpret_cast<const u32x4_a4 *>(p);
        r.b = *reinterpret_cast<const u32x4_a4 *>(p + 16);
        r.c = *reinterpret_cast<const uint32_t *>(p + 32);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t, const Tables &, int g) {
        const uint32_t w[9] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w, r.c};
        const Table16 tab = table16(qlin_mxfp4_values);
        const uint32_t odd = (uint32_t)g & 1u; /* the piece starts two bytes into w */
        float acc = 0.0f;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint32_t qs[4]; /* block 0: the nibble bytes start 1 (3) bytes into dword 0; block 1: 2 bytes into dword 4 (at dword 5) */
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if (h == 0) qs[i] = __builtin_amdgcn_alignbit(w[i + 1], w[i], 8u + 16u * odd);
                else qs[i] = odd ? w[5 + i] : __builtin_amdgcn_alignbit(w[5 + i], w[4 + i], 16);
            }
            v4i c = {0, 0, 0, 0};
#pragma unroll
            for (int u = 0; u < 2; u++) {
                v4i b;
#pragma unroll
                for (int i = 0; i < 4; i++) b[i] = look4((qs[i] >> (4 * u)) & 0x0F0F0F0Fu, tab);
                const uint4 av = *reinterpret_cast<const uint4 *>(xo.arows + kStep * (2 * h + u));
                const v4i a = {(int)av.x, (int)av.y, (int)av.z, (int)av.w};
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
            }
            const uint32_t e = (h == 0 ? w[0] >> (16u * odd) : w[4] >> (8u + 16u * odd)) & 0xFFu;
            acc = fmaf(join_digits(c) * xo.meta[2 * g + h], e8m0_half(e), acc);
        }
        return acc;
    }
};

/* NVFP4 [4 x ue4m3 scale][32 nibble bytes] per 64 elements (common/ggml_dequant.h:2832-2848), 36 bytes: sub-block s
 * of 16 elements is table[nibble] * scale_s over bytes 8 s .. 8 s + 7, low nibbles first. Lane group g takes block g
 * of the 256 elements, nine dwords; an instruction is one sub-block. */
template <> struct GridFmt<T_NVFP4> {
    static constexpr int kBlock = 144, kGridBytes = 0;
    static constexpr int kPiece = 0, kAlign = 4;
    static constexpr int kStep = 16;
    static constexpr bool kSums = false, kAInRegs = false;
    __device__ static const uint32_t *grid_src() { return nullptr; }
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    struct Raw {
        u32x4_a4 a, b;
        uint32_t c;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        const uint8_t *p = blk + 36 * g;
        r.a = *reinterpret_cast<const u32x4_a4 *>(p);
        r.b = *reinterpret_cast<const u32x4_a4 *>(p + 16);
        r.c = *reinterpret_cast<const uint32_t *>(p + 32);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t, const Tables &, int g) {
        const uint32_t w[9] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w, r.c};
        const Table16 tab = table16(qlin_mxfp4_values);
        float acc = 0.0f;
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const uint32_t q0 = w[1 + 2 * st], q1 = w[2 + 2 * st];
            const v4i b = {look4(q0 & 0x0F0F0F0Fu, tab), look4(q1 & 0x0F0F0F0Fu, tab), look4((q0 >> 4) & 0x0F0F0F0Fu, tab),
                           look4((q1 >> 4) & 0x0F0F0F0Fu, tab)};
            const v4i zero = {0, 0, 0, 0};
            const uint4 av = *reinterpret_cast<const uint4 *>(xo.arows + kStep * st);
            const v4i a = {(int)av.x, (int)av.y, (int)av.z, (int)av.w};
            const v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, zero, 0, 0, 0);
            acc = fmaf(join_digits(c) * xo.meta[2 * g + (st >> 1)], ue4m3_half((w[0] >> (8 * st)) & 0xFFu), acc);
        }
        return acc;
    }
};

/* Q4_1 [d][m][16 nibble bytes] (common/ggml_dequant.h:2864-2877), Q5_0 [d][qh 4][16] (:2879-2895) and Q5_1
 * [d][m][qh 4][16] (:2897-2915): blocks of 32 elements in 20, 22 and 24 bytes; element l < 16 is the low nibble of
 * byte l (+ 16 x bit l of qh), element 16 + l the high nibble (+ 16 x bit 16 + l); Q4_1 and Q5_1 add m, Q5_0
 * subtracts 16. Lane group g takes blocks 2g and 2g + 1 as 10, 11 or 12 dwords; the codes stay unsigned and m or
 * -16 d goes onto the sum of x. */
template <uint32_t T> struct Legacy32 {
    static constexpr int kBytes = T == T_Q4_1 ? 20 : T == T_Q5_0 ? 22 : 24;
    static constexpr int kDw = kBytes / 2; /* dwords of two blocks */
    static constexpr bool kHigh = T != T_Q4_1, kMin = T != T_Q5_0;
    static constexpr int kBlock = 8 * kBytes, kGridBytes = 0;
    static constexpr int kPiece = 0, kAlign = 4;
    static constexpr int kStep = 16;
    static constexpr bool kSums = true, kAInRegs = false;
    __device__ static const uint32_t *grid_src() { return nullptr; }
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    struct Raw {
        uint32_t w[kDw];
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        const uint8_t *p = blk + 2 * kBytes * g;
#pragma unroll
        for (int i = 0; i + 4 <= kDw; i += 4) {
            const u32x4_a4 v = *reinterpret_cast<const u32x4_a4 *>(p + 4 * i);
            r.w[i] = v.x; r.w[i + 1] = v.y; r.w[i + 2] = v.z; r.w[i + 3] = v.w;
        }
        if (kDw % 4 >= 2) {
            const u32x2_a4 v = *reinterpret_cast<const u32x2_a4 *>(p + 4 * (kDw & ~3));
            r.w[kDw & ~3] = v.x; r.w[(kDw & ~3) + 1] = v.y;
        }
        if (kDw % 2) r.w[kDw - 1] = *reinterpret_cast<const uint32_t *>(p + 4 * (kDw - 1));
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t, const Tables &, int g) {
        const uint32_t(&w)[kDw] = r.w;
        float acc = 0.0f;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint32_t dm, qh = 0, qs[4];
            if (T == T_Q5_0) { /* the second block starts in the middle of dword 5 */
                dm = h == 0 ? w[0] & 0xFFFFu : w[5] >> 16;
                qh = h == 0 ? __builtin_amdgcn_alignbit(w[1], w[0], 16) : w[6];
#pragma unroll
                for (int i = 0; i < 4; i++) qs[i] = h == 0 ? __builtin_amdgcn_alignbit(w[i + 2], w[i + 1], 16) : w[7 + i];
            } else {
                constexpr int kHead = kHigh ? 2 : 1;
                const int b = (kDw / 2) * h;
                dm = w[b];
                if (kHigh) qh = w[b + 1];
#pragma unroll
                for (int i = 0; i < 4; i++) qs[i] = w[b + kHead + i];
            }
            v4i c = {0, 0, 0, 0};
#pragma unroll
            for (int u = 0; u < 2; u++) {
                v4i b;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    uint32_t code = (qs[i] >> (4 * u)) & 0x0F0F0F0Fu;
                    if (kHigh) code |= spread4(qh >> (16 * u + 4 * i)) << 4;
                    b[i] = (int)code;
                }
                const uint4 av = *reinterpret_cast<const uint4 *>(xo.arows + kStep * (2 * h + u));
                const v4i a = {(int)av.x, (int)av.y, (int)av.z, (int)av.w};
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
            }
            const int G = 2 * g + h;
            const float sum = xo.meta[8 + 2 * G] + xo.meta[8 + 2 * G + 1];
            const float d = half_bits_fast(dm & 0xFFFFu);
            float dot = join_digits(c) * xo.meta[G];
            if (!kMin) dot = fmaf(-16.0f, sum, dot);
            acc = fmaf(dot, d, acc);
            if (kMin) acc = fmaf(half_bits_fast(dm >> 16), sum, acc);
        }
        return acc;
    }
};
template <> struct GridFmt<T_Q4_1> : Legacy32<T_Q4_1> {};
template <> struct GridFmt<T_Q5_0> : Legacy32<T_Q5_0> {};
template <> struct GridFmt<T_Q5_1> : Legacy32<T_Q5_1> {};

/* IQ4_XS [d][scales_h 2][scales_l 4][qs 128] (:2956-2973), 136 bytes: group j of 32 elements has its nibbles in
 * qs[16 j ..] (low nibbles first, as IQ4_NL) and a 6-bit scale - 32. Lane group g takes groups 2g, 2g+1. */
template <> struct GridFmt<T_IQ4_XS> {
    static constexpr int kBlock = 136, kGridBytes = 0;
    static constexpr int kPiece = 0, kAlign = 4;
    static constexpr int kStep = 16;
    static constexpr bool kSums = false, kAInRegs = false;
    __device__ static const uint32_t *grid_src() { return nullptr; }
    __device__ static int elem0(int g, int st) { return 64 * g + 16 * st; }
    struct Raw {
        u32x4_a4 a, b;
        u32x2_a4 hd;
    };
    __device__ static Raw load(const uint8_t *blk, int g) {
        Raw r;
        r.hd = *reinterpret_cast<const u32x2_a4 *>(blk);
        r.a = *reinterpret_cast<const u32x4_a4 *>(blk + 8 + 32 * g);
        r.b = *reinterpret_cast<const u32x4_a4 *>(blk + 24 + 32 * g);
        return r;
    }
    __device__ static float item(const XOperand &xo, const Raw &r, uint32_t, const Tables &, int g) {
        const uint32_t qs[8] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w};
        const Table16 tab = table16(qlin_iq4nl_values);
        float acc = 0.0f;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            v4i c = {0, 0, 0, 0};
#pragma unroll
            for (int u = 0; u < 2; u++) {
                v4i b;
#pragma unroll
                for (int i = 0; i < 4; i++) b[i] = look4((qs[4 * h + i] >> (4 * u)) & 0x0F0F0F0Fu, tab);
                const uint4 av = *reinterpret_cast<const uint4 *>(xo.arows + kStep * (2 * h + u));
                const v4i a = {(int)av.x, (int)av.y, (int)av.z, (int)av.w};
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
            }
            const int j = 2 * g + h;
            const uint32_t ls = ((r.hd.y >> (4 * j)) & 15u) | ((((r.hd.x >> 16) >> (2 * j)) & 3u) << 4);
            acc = fmaf(join_digits(c) * xo.meta[j], (float)((int)ls - 32), acc);
        }
        return half_bits_fast(r.hd.x & 0xFFFFu) * acc;
    }
};

/* x -> signed digit planes -> A operands, in the wave's own scratch xs; v: the lane's four elements of the 256 */
template <class F> __device__ __forceinline__ void prepare_x(v4f v, uint8_t *xs, int lane, XOperand &xo) {
    const int n = lane & 15, g = lane >> 4;
    /* the largest |x| of the group as a bit pattern: an integer maximum keeps a NaN or an Inf on top */
    constexpr uint32_t kAbs = 0x7FFFFFFFu;
    uint32_t amax = max(max(__float_as_uint(v.x) & kAbs, __float_as_uint(v.y) & kAbs),
                        max(__float_as_uint(v.z) & kAbs, __float_as_uint(v.w) & kAbs));
    /* 8 consecutive lanes share one 32-element group */
    amax = max(amax, dpp_movu<0xB1>(amax));
    amax = max(amax, dpp_movu<0x4E>(amax));
    amax = max(amax, dpp_movu<0x141>(amax));
    int e = (int)(amax >> 23) - 126; /* amax in [2^(e-1), 2^e) */
    if (e < -96) e = -96;            /* zero and tiny groups */
    const float up = __uint_as_float((uint32_t)(127 + 22 - e) << 23);
    float down = __uint_as_float((uint32_t)(127 - 22 + e) << 23);
    if (amax >= 0x7F800000u) down = __uint_as_float(0x7FC00000u); /* Inf/NaN in x: poison every row */
    const int X[4] = {__float2int_rn(v.x * up), __float2int_rn(v.y * up), __float2int_rn(v.z * up),
                      __float2int_rn(v.w * up)};
    /* The three signed base-256 digits of X (X = 256*X1 + d0 with d0 = (int8)X, X1 = 256*X2 + d1, X2 in
     * [-64, 64]) are bytes 0..2 of (X + 0x8080) ^ 0x8080: adding 128 at a byte makes its digit unsigned and
     * carries exactly when the digit is negative, the xor takes the 128 off again. */
    uint32_t Z[4];
#pragma unroll
    for (int k = 0; k < 4; k++) Z[k] = ((uint32_t)X[k] + 0x00008080u) ^ 0x00008080u;
    /* byte transpose: plane j = byte j of Z[0..3] (selector 0-3: second operand, 4-7: first) */
    const uint32_t lo01 = __builtin_amdgcn_perm(Z[1], Z[0], 0x05010400u), lo23 = __builtin_amdgcn_perm(Z[3], Z[2], 0x05010400u);
    const uint32_t hi01 = __builtin_amdgcn_perm(Z[1], Z[0], 0x07030602u), hi23 = __builtin_amdgcn_perm(Z[3], Z[2], 0x07030602u);
    uint32_t *pl = reinterpret_cast<uint32_t *>(xs);
    pl[lane] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);       /* digit 2 (top) */
    pl[64 + lane] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);  /* digit 1 */
    pl[128 + lane] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u); /* digit 0 */
    if ((lane & 7) == 0) reinterpret_cast<float *>(xs + 1024)[lane >> 3] = down;
    if (F::kSums) { /* the sum of x over each 16 elements: four lanes */
        float sum = (v.x + v.y) + (v.z + v.w);
        sum += dpp_mov<0xB1>(sum);
        sum += dpp_mov<0x4E>(sum);
        if ((lane & 3) == 0) reinterpret_cast<float *>(xs + 1056)[lane >> 2] = sum;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    /* A operand: x row i = lane%16 = 4*g' + plane (plane 3 unused) is live in lane group g' only and holds,
     * for instruction s, the digits of the 16 elements from F::elem0(g', s) on. Every other lane reads zeros. */
    const int plane = n & 3;
    const bool live = (n >> 2) == g && plane < 3;
    xo.arows = xs + (live ? plane * 256 + F::elem0(g, 0) : 768);
    if (F::kAInRegs) {
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const uint4 d = *reinterpret_cast<const uint4 *>(xo.arows + F::kStep * st);
            const v4i a = {(int)d.x, (int)d.y, (int)d.z, (int)d.w};
            xo.A[st] = a;
        }
    }
    xo.meta = reinterpret_cast<const float *>(xs + 1024);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

}  // namespace
}  // namespace qlin
#endif

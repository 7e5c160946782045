/*
 * gemv_q4k_item.h - the Q4_K matvecs' arithmetic (described in gemv_q4k.hip): x of a super-block as the operand of the 8-bit
 * integer matrix instruction, and sixteen rows of a super-block times it. For gemv_q4k.hip and gemv_dma.hip.
 */
#ifndef QLIN_GEMV_Q4K_ITEM_H
#define QLIN_GEMV_Q4K_ITEM_H

#include "qlin_device.h"

namespace qlin {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kQ4KScratch = 1088; /* 4 digit planes x 256 B + 8 x (2^(e-30), sum) */
/* x operand of one super-block: A[2p+h] for chain p, instruction h; scale[p] = 2^(e-30) and
 * sum[p] = sum of x for sub-block 4p + lane/16 */
struct Q4KOperand {
    v4i A[4];
    float scale[2], sum[2];
};

/* x -> signed digit planes -> A operands, wave-private (xs: the wave's kQ4KScratch bytes of LDS) */
__device__ __forceinline__ void q4k_prepare(v4f v, Q4KOperand &xo, uint8_t *xs, int lane) {
    const int n = lane & 15, g = lane >> 4;
    float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    float sum = (v.x + v.y) + (v.z + v.w);
    /* 8 consecutive lanes share one 32-element sub-block */
    amax = fmaxf(amax, dpp_mov<0xB1>(amax));
    amax = fmaxf(amax, dpp_mov<0x4E>(amax));
    amax = fmaxf(amax, dpp_mov<0x141>(amax));
    sum += dpp_mov<0xB1>(sum);
    sum += dpp_mov<0x4E>(sum);
    sum += dpp_mov<0x141>(sum);
    int e = (int)(__float_as_uint(amax) >> 23) - 126; /* amax in [2^(e-1), 2^e) */
    if (e < -96) e = -96;                              /* zero and tiny sub-blocks */
    const float up = __uint_as_float((uint32_t)(127 + 30 - e) << 23);
    float down = __uint_as_float((uint32_t)(127 - 30 + e) << 23);
    if (!(amax <= 3.0e38f)) down = __uint_as_float(0x7FC00000u); /* Inf/NaN in x: poison every row */
    const int X[4] = {__float2int_rn(v.x * up), __float2int_rn(v.y * up), __float2int_rn(v.z * up),
                      __float2int_rn(v.w * up)};
    /* The four signed base-256 digits of X (X = 256*X1 + d0 with d0 = (int8)X, X1 = 256*X2 + d1, ...;
     * the top one in [-64, 64]) are the bytes of (X + 0x00808080) ^ 0x00808080: adding 128 at a byte makes its
     * digit unsigned and carries exactly when the digit is negative, the xor takes the 128 off again. */
    uint32_t Z[4];
#pragma unroll
    for (int k = 0; k < 4; k++) Z[k] = ((uint32_t)X[k] + 0x00808080u) ^ 0x00808080u;
    /* byte transpose: plane j = byte j of Z[0..3] (selector 0-3: second operand, 4-7: first) */
    const uint32_t lo01 = __builtin_amdgcn_perm(Z[1], Z[0], 0x05010400u), lo23 = __builtin_amdgcn_perm(Z[3], Z[2], 0x05010400u);
    const uint32_t hi01 = __builtin_amdgcn_perm(Z[1], Z[0], 0x07030602u), hi23 = __builtin_amdgcn_perm(Z[3], Z[2], 0x07030602u);
    uint32_t *pl = reinterpret_cast<uint32_t *>(xs);
    pl[lane] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);       /* digit 3 (top) */
    pl[64 + lane] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);  /* digit 2 */
    pl[128 + lane] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u); /* digit 1 */
    pl[192 + lane] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u); /* digit 0 */
    if ((lane & 7) == 0) reinterpret_cast<float2 *>(xs + 1024)[lane >> 3] = make_float2(down, sum);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    /* A operand: x-row i = lane%16 = 4*s' + plane; k group lane/16 carries sub-blocks 2*(g>>1)
     * (registers 0-1) and 2*(g>>1)+1 (registers 2-3) of the chain, elements 16*(g&1) + 8h .. +7 */
    const int sq = n >> 2, plane = n & 3;
    const bool live = (g >> 1) == (sq >> 1);
    const uint8_t *src = xs + plane * 256 + 32 * sq + 16 * (g & 1);
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint2 d = *reinterpret_cast<const uint2 *>(src + 128 * p + 8 * h);
            const bool lo = live && !(sq & 1), hi = live && (sq & 1);
            v4i a;
            a.x = lo ? (int)d.x : 0;
            a.y = lo ? (int)d.y : 0;
            a.z = hi ? (int)d.x : 0;
            a.w = hi ? (int)d.y : 0;
            xo.A[2 * p + h] = a;
        }
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const float2 m = reinterpret_cast<const float2 *>(xs + 1024)[4 * p + g];
        xo.scale[p] = m.x;
        xo.sum[p] = m.y;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

/* one super-block of 16 rows: header hh, code bytes qa (chain 0) and qb (chain 1) of this lane; g = lane / 16 */
__device__ __forceinline__ float q4k_item(const Q4KOperand &xo, const uint4 hh, const uint4 qa, const uint4 qb, int g) {
    constexpr uint32_t M = 0x0F0F0F0Fu;
    v4i c0 = {0, 0, 0, 0}, c1 = {0, 0, 0, 0};
    v4i b;
    b.x = (int)(qa.x & M); b.y = (int)(qa.y & M); b.z = (int)((qa.x >> 4) & M); b.w = (int)((qa.y >> 4) & M);
    c0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(xo.A[0], b, c0, 0, 0, 0);
    b.x = (int)(qb.x & M); b.y = (int)(qb.y & M); b.z = (int)((qb.x >> 4) & M); b.w = (int)((qb.y >> 4) & M);
    c1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(xo.A[2], b, c1, 0, 0, 0);
    b.x = (int)(qa.z & M); b.y = (int)(qa.w & M); b.z = (int)((qa.z >> 4) & M); b.w = (int)((qa.w >> 4) & M);
    c0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(xo.A[1], b, c0, 0, 0, 0);
    b.x = (int)(qb.z & M); b.y = (int)(qb.w & M); b.z = (int)((qb.z >> 4) & M); b.w = (int)((qb.w >> 4) & M);
    c1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(xo.A[3], b, c1, 0, 0, 0);
    /* 6-bit scale and min of sub-blocks g (chain 0) and 4+g (chain 1) */
    const uint32_t sh = 8u * (uint32_t)g;
    const uint32_t sc0 = __builtin_amdgcn_ubfe(hh.y, sh, 6), mn0 = __builtin_amdgcn_ubfe(hh.z, sh, 6);
    const uint32_t sc1 = __builtin_amdgcn_ubfe(hh.w, sh, 4) | (__builtin_amdgcn_ubfe(hh.y, sh + 6, 2) << 4);
    const uint32_t mn1 = __builtin_amdgcn_ubfe(hh.w, sh + 4, 4) | (__builtin_amdgcn_ubfe(hh.z, sh + 6, 2) << 4);
    const float d = half_bits_fast(hh.x & 0xFFFFu), dmin = half_bits_fast(hh.x >> 16);
    /* digit sums: |top| <= 32*15*64, the others <= 32*15*128, so each pair below is an integer of less
     * than 24 bits and its conversion is exact; one rounding in the multiply-add that joins them */
    const float s0 = fmaf((float)((c0.x << 8) + c0.y), 65536.0f, (float)((c0.z << 8) + c0.w));
    const float s1 = fmaf((float)((c1.x << 8) + c1.y), 65536.0f, (float)((c1.z << 8) + c1.w));
    const float z0 = s0 * xo.scale[0], z1 = s1 * xo.scale[1];
    const float dots = (float)sc0 * z0 + (float)sc1 * z1;
    const float mins = (float)mn0 * xo.sum[0] + (float)mn1 * xo.sum[1];
    return d * dots - dmin * mins;
}

}  // namespace
}  // namespace qlin
#endif

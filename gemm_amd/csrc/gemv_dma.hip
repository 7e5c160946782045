/*
 * gemv_dma.hip - batch-1 matvec for eleven block formats with the blocks fetched by the load-to-LDS path, one to three
 * matrices or a gate and up pair per launch.
 *
 * The arithmetic is that of gemv_grid.hip (Q4_K: gemv_q4k.hip): x as signed base-256 digits, v_mfma_i32_16x16x64_i8, a wave owns a
 * super-block column of the workgroup's rows. What differs is how the blocks come and what an item costs:
 *   - A wave copies whole blocks of a row group by 1 KB requests (consecutive lanes consecutive 16-byte pieces, source addresses
 *     of any alignment) into an image of its own, two images in turn, and cuts its codes out of the image at compile-time offsets.
 *     Loads of the operand layout scatter 64 lanes over 16 rows, and blocks of 210, 110 or 66 bytes need a funnel shift per dword there.
 *   - The x operand and the factors that go with it stay in registers for all row groups of a super-block: an item of Q6_K is 105
 *     vector and 6 LDS instructions, on operand-layout loads and an operand in LDS 150 and 20. This is what bounds the smaller formats.
 *   - The digits of x are made while the first blocks are on their way: requests complete in order and x is the first of them.
 *   - A pair's row group is eight rows of gate and eight of up, so 56 rows of either per compute unit are seven whole items.
 *   - Rows of up to 4096 elements start as many waves as they have super-blocks.
 * What bounds it now: at 4096 x 4096 and below the launch (3.5 us without work); in large tensors the load path, whose 1 KB requests
 * touch four blocks, that is twelve 128-byte lines instead of eight (Q6_K 14336 x 4096: 12.5 us, with the arithmetic removed
 * 12.4, with 16-byte aligned pieces, which cost more instructions than they save, 11.0; a bare read 8.6). Three images, eight
 * or twelve waves and two workgroups per compute unit measured no faster.
 * Measured, us, before (gemv_grid.hip, gemv_int.hip) / now: Q6_K 4096 x 14336 15.5 / 13.1, 14336 x 4096 14.1 / 12.5, 2048 x 5632 8.8 / 5.0, 32003 x
 * 2048 16.5 / 12.9; Q5_K 151936 x 4096 88 / 78; Q8_0 2 x 5632 x 2048 7.9 / 6.1, 2048 x 5632 6.8 / 5.1; Q3_K 14336 x 4096 12.1 / 8.9;
 * IQ3_S 2 x 14336 x 4096 18.5 / 15.6; IQ4_NL 2 x 14336 x 2048 11.5 / 9.2; Q2_K 2 x 14336 x 1024 11.3 / 5.8. Error against 64 bits as before.
 *
 * A non-finite x makes every output NaN (the fixed-point form cannot carry Inf).
 */
#include "gemv_grid_formats.h"
#include "gemv_q4k_item.h"

namespace qlin {

namespace {

constexpr int kMaxWaves = 16;
constexpr uint32_t kNone = 0xFFFFFFFFu;    /* a piece of an image row that is padding */
constexpr uint32_t kPastEnd = 0xFFFFFFF0u; /* an offset outside every buffer: the request returns zeros */
typedef __attribute__((address_space(3))) void lds_void;

/* the x operand of a super-block: what an item multiplies by, in registers (Q4_K has its own) */
struct XRegs {
    v4i A[4];
    float m[4]; /* 2^(e-22) of the instruction's 16 elements */
    float o[4]; /* and the sum of x over them */
};

__device__ __forceinline__ uint4 lds16(const uint8_t *p) { return *reinterpret_cast<const uint4 *>(p); }
__device__ __forceinline__ uint32_t lds4(const uint8_t *p) { return *reinterpret_cast<const uint32_t *>(p); }

template <class F> __device__ __forceinline__ void prepare_regs(v4f v, uint8_t *xs, int lane, float off, XRegs &x) {
    const int g = lane >> 4;
    if (lane < 32) reinterpret_cast<uint32_t *>(xs + 768)[lane] = 0u; /* what the dead lanes of the operand read */
    XOperand xo;
    prepare_x<F>(v, xs, lane, xo);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint4 a = lds16(xo.arows + F::kStep * q);
        x.A[q] = v4i{(int)a.x, (int)a.y, (int)a.z, (int)a.w};
        const int e0 = F::elem0(g, q);
        x.m[q] = xo.meta[e0 >> 5];
        x.o[q] = F::kSums ? off * xo.meta[8 + (e0 >> 4)] : 0.0f;
    }
}

/* A format's image row: kPieces 16-byte pieces, odd so that sixteen rows fall into sixteen bank groups; piece_src gives a
 * piece's place in the block, the last one ends with the block. item: sixteen rows times 256 elements from the image. The elements
 * and the arithmetic are those of GridFmt (gemv_grid_formats.h). */
template <uint32_t T> struct DmaFmt;

template <> struct DmaFmt<T_Q4_K> {
    static constexpr int kBlock = 144, kAlign = 16, kGridBytes = 0, kPieces = 9;
    typedef Q4KOperand X;
    __device__ static uint32_t piece_src(uint32_t p) { return 16u * p; }
    __device__ static void prepare(v4f v, uint8_t *xs, int lane, X &x) { q4k_prepare(v, x, xs, lane); }
    __device__ static float item(const X &x, const uint8_t *row, int g, const Tables &) {
        return q4k_item(x, lds16(row), lds16(row + 16 + 16 * g), lds16(row + 80 + 16 * g), g);
    }
};

template <> struct DmaFmt<T_Q6_K> : GridFmt<T_Q6_K> {
    typedef XRegs X;
    __device__ static void prepare(v4f v, uint8_t *xs, int lane, X &x) { prepare_regs<GridFmt<T_Q6_K>>(v, xs, lane, kOff, x); }
    static constexpr int kPieces = 15;
    __device__ static uint32_t piece_src(uint32_t p) { return p < 13 ? 16u * p : p == 13 ? 194u : kNone; }
    static constexpr float kOff = -32.0f;
    __device__ static float item(const XRegs &x, const uint8_t *row, int g, const Tables &) {
        const int h = g >> 1, p = g & 1;
        const uint4 a4 = lds16(row + 64 * h + 16 * p), b4 = lds16(row + 64 * h + 32 + 16 * p), h4 = lds16(row + 128 + 32 * h + 16 * p);
        const uint2 sc = *reinterpret_cast<const uint2 *>(row + 192 + 8 * h);
        const float d = half_bits_fast(*reinterpret_cast<const uint16_t *>(row + 222));
        const uint32_t qa[4] = {a4.x, a4.y, a4.z, a4.w}, qb[4] = {b4.x, b4.y, b4.z, b4.w}, qh[4] = {h4.x, h4.y, h4.z, h4.w};
        const uint32_t s[2] = {__builtin_amdgcn_alignbit(sc.y, sc.x, 8u * (uint32_t)p), sc.y >> (8 * p)}; /* bytes 0 and 2: the lane's scales */
        float acc = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t(&ql)[4] = (q & 1) ? qb : qa;
            v4i b;
#pragma unroll
            for (int i = 0; i < 4; i++)
                b[i] = (int)(((ql[i] >> (4 * (q >> 1))) & 0x0F0F0F0Fu) | ((q < 2 ? qh[i] << (4 - 2 * q) : qh[i] >> (2 * q - 4)) & 0x30303030u));
            const v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.A[q], b, v4i{0, 0, 0, 0}, 0, 0, 0);
            const float scale = (float)(int)(int8_t)(s[q >> 1] >> (16 * (q & 1)));
            acc = fmaf(scale, fmaf(join_digits(c), x.m[q], x.o[q]), acc);
        }
        return d * acc;
    }
};

template <> struct DmaFmt<T_Q3_K> : GridFmt<T_Q3_K> {
    typedef XRegs X;
    __device__ static void prepare(v4f v, uint8_t *xs, int lane, X &x) { prepare_regs<GridFmt<T_Q3_K>>(v, xs, lane, kOff, x); }
    static constexpr int kPieces = 7;
    __device__ static uint32_t piece_src(uint32_t p) { return p < 6 ? 16u * p : 94u; }
    static constexpr float kOff = -4.0f;
    __device__ static float item(const XRegs &x, const uint8_t *row, int g, const Tables &) {
        const int h = g >> 1, p = g & 1;
        const uint4 q4 = lds16(row + 32 + 16 * g), m4 = lds16(row + 16 * p), t = lds16(row + 96); /* t: the block's last 16 bytes */
        const uint32_t qs[4] = {q4.x, q4.y, q4.z, q4.w}, hm[4] = {m4.x >> (4 * h), m4.y >> (4 * h), m4.z >> (4 * h), m4.w >> (4 * h)};
        const uint32_t lo0 = __builtin_amdgcn_alignbyte(t.y, t.x, 2), lo1 = __builtin_amdgcn_alignbyte(t.z, t.y, 2);
        const uint32_t hi = __builtin_amdgcn_alignbyte(t.w, t.z, 2);
        /* the four 6-bit scales of the lane: indices 8 h + 2 j + p; low nibbles in bytes 2 j + p of lo (high nibble for h), two
         * bits each in byte (2 j + p) & 3 of hi at 2 (2 h + (j >> 1)) */
        const uint32_t sh = 8u * (uint32_t)p + 4u * (uint32_t)h;
        const uint32_t l01 = __builtin_amdgcn_alignbit(lo1, lo0, sh), l23 = lo1 >> sh; /* bytes 0 and 2, low nibbles */
        const uint32_t h01 = hi >> (8 * p + 4 * h), h23 = hi >> (8 * p + 4 * h + 2);
        const uint32_t s[2] = {(l01 & 0x000F000Fu) | ((h01 & 0x00030003u) << 4), (l23 & 0x000F000Fu) | ((h23 & 0x00030003u) << 4)};
        float acc = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            v4i b;
#pragma unroll
            for (int i = 0; i < 4; i++) b[i] = (int)(((qs[i] >> (2 * j)) & 0x03030303u) | ((j < 2 ? hm[i] << (2 - j) : hm[i] >> (j - 2)) & 0x04040404u));
            const v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.A[j], b, v4i{0, 0, 0, 0}, 0, 0, 0);
            const float scale = (float)((int)((s[j >> 1] >> (16 * (j & 1))) & 0xFFu) - 32);
            acc = fmaf(scale, fmaf(join_digits(c), x.m[j], x.o[j]), acc);
        }
        return half_bits_fast(t.w >> 16) * acc;
    }
};

template <> struct DmaFmt<T_Q8_0> : GridFmt<T_Q8_0> {
    typedef XRegs X;
    __device__ static void prepare(v4f v, uint8_t *xs, int lane, X &x) { prepare_regs<GridFmt<T_Q8_0>>(v, xs, lane, kOff, x); }
    static constexpr int kPieces = 17;
    __device__ static uint32_t piece_src(uint32_t p) { return 16u * p; }
    static constexpr float kOff = 1.0f;
    __device__ static float item(const XRegs &x, const uint8_t *row, int g, const Tables &) {
        uint32_t w[17];
#pragma unroll
        for (int i = 0; i < 17; i++) w[i] = lds4(row + 68 * g + 4 * i);
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
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.A[2 * h + q], b, c, 0, 0, 0);
            }
            acc = fmaf(join_digits(c) * x.m[2 * h], half_bits_fast(h == 0 ? w[0] & 0xFFFFu : w[8] >> 16), acc);
        }
        return acc;
    }
};

template <> struct DmaFmt<T_Q5_K> : GridFmt<T_Q5_K> {
    typedef XRegs X;
    __device__ static void prepare(v4f v, uint8_t *xs, int lane, X &x) { prepare_regs<GridFmt<T_Q5_K>>(v, xs, lane, kOff, x); }
    static constexpr int kPieces = 11;
    __device__ static uint32_t piece_src(uint32_t p) { return 16u * p; }
    static constexpr float kOff = 1.0f;
    __device__ static float item(const XRegs &x, const uint8_t *row, int g, const Tables &) {
        const uint4 hd = lds16(row), h0 = lds16(row + 16), h1 = lds16(row + 32), q0 = lds16(row + 48 + 32 * g), q1 = lds16(row + 64 + 32 * g);
        const uint32_t sh = 2u * (uint32_t)g;
        const uint32_t qs[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
        const uint32_t qh[8] = {h0.x >> sh, h0.y >> sh, h0.z >> sh, h0.w >> sh, h1.x >> sh, h1.y >> sh, h1.z >> sh, h1.w >> sh};
        /* get_scale_min_k4 (common/ggml_dequant.h:1582-1590) of sub-blocks 2 g and 2 g + 1: bytes 0 and 1 of sc and mn */
        const uint32_t at = 16u * (uint32_t)(g & 1);
        const uint32_t y = hd.y >> at, z = hd.z >> at, w = hd.w >> at;
        const bool high = g >= 2;
        const uint32_t sc = high ? (w & 0x0F0Fu) | ((y >> 2) & 0x3030u) : y & 0x3F3Fu;
        const uint32_t mn = high ? ((w >> 4) & 0x0F0Fu) | ((z >> 2) & 0x3030u) : z & 0x3F3Fu;
        float dots = 0.0f, mins = 0.0f;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            v4i c = {0, 0, 0, 0};
#pragma unroll
            for (int hf = 0; hf < 2; hf++) {
                v4i b;
#pragma unroll
                for (int i = 0; i < 4; i++)
                    b[i] = (int)(((qs[4 * hf + i] >> (4 * u)) & 0x0F0F0F0Fu) | ((qh[4 * hf + i] << (4 - u)) & 0x10101010u));
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.A[2 * u + hf], b, c, 0, 0, 0);
            }
            dots = fmaf((float)((sc >> (8 * u)) & 0xFFu), join_digits(c) * x.m[2 * u], dots);
            mins = fmaf((float)((mn >> (8 * u)) & 0xFFu), x.o[2 * u] + x.o[2 * u + 1], mins);
        }
        return half_bits_fast(hd.x & 0xFFFFu) * dots - half_bits_fast(hd.x >> 16) * mins;
    }
};

template <> struct DmaFmt<T_Q2_K> : GridFmt<T_Q2_K> {
    typedef XRegs X;
    __device__ static void prepare(v4f v, uint8_t *xs, int lane, X &x) { prepare_regs<GridFmt<T_Q2_K>>(v, xs, lane, kOff, x); }
    static constexpr int kPieces = 7;
    __device__ static uint32_t piece_src(uint32_t p) { return p < 5 ? 16u * p : p == 5 ? 68u : kNone; }
    static constexpr float kOff = 1.0f;
    __device__ static float item(const XRegs &x, const uint8_t *row, int g, const Tables &) {
        const int h = g >> 1, p = g & 1;
        const uint4 q4 = lds16(row + 16 + 16 * g);
        const uint2 sc = *reinterpret_cast<const uint2 *>(row + 8 * h);
        const uint32_t dd = lds4(row + 92);
        const uint32_t qs[4] = {q4.x, q4.y, q4.z, q4.w};
        const uint32_t s[2] = {__builtin_amdgcn_alignbit(sc.y, sc.x, 8u * (uint32_t)p), sc.y >> (8 * p)}; /* bytes 0 and 2 */
        float dots = 0.0f, mins = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            v4i b;
#pragma unroll
            for (int i = 0; i < 4; i++) b[i] = (int)((qs[i] >> (2 * j)) & 0x03030303u);
            const v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.A[j], b, v4i{0, 0, 0, 0}, 0, 0, 0);
            const uint32_t w = s[j >> 1] >> (16 * (j & 1));
            dots = fmaf((float)(w & 15u), join_digits(c) * x.m[j], dots);
            mins = fmaf((float)((w >> 4) & 15u), x.o[j], mins);
        }
        return half_bits_fast(dd & 0xFFFFu) * dots - half_bits_fast(dd >> 16) * mins;
    }
};

/* IQ4_NL and Q4_0 */
template <uint32_t T> struct DmaNibble18 : GridFmt<T> {
    typedef XRegs X;
    __device__ static void prepare(v4f v, uint8_t *xs, int lane, X &x) { prepare_regs<GridFmt<T>>(v, xs, lane, kOff, x); }
    static constexpr int kPieces = 9;
    __device__ static uint32_t piece_src(uint32_t p) { return 16u * p; }
    static constexpr float kOff = -8.0f;
    __device__ static float item(const XRegs &x, const uint8_t *row, int g, const Tables &) {
        uint32_t w[9];
#pragma unroll
        for (int i = 0; i < 9; i++) w[i] = lds4(row + 36 * g + 4 * i);
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
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.A[2 * h + u], b, c, 0, 0, 0);
            }
            float dot = join_digits(c) * x.m[2 * h];
            if (T == T_Q4_0) dot += x.o[2 * h] + x.o[2 * h + 1];
            acc = fmaf(dot, half_bits_fast(h == 0 ? w[0] & 0xFFFFu : w[4] >> 16), acc);
        }
        return acc;
    }
};
template <> struct DmaFmt<T_Q4_0> : DmaNibble18<T_Q4_0> {};
template <> struct DmaFmt<T_IQ4_NL> : DmaNibble18<T_IQ4_NL> {};

template <> struct DmaFmt<T_IQ4_XS> : GridFmt<T_IQ4_XS> {
    typedef XRegs X;
    __device__ static void prepare(v4f v, uint8_t *xs, int lane, X &x) { prepare_regs<GridFmt<T_IQ4_XS>>(v, xs, lane, kOff, x); }
    static constexpr int kPieces = 9;
    __device__ static uint32_t piece_src(uint32_t p) { return p < 8 ? 16u * p : 120u; }
    static constexpr float kOff = 1.0f;
    __device__ static float item(const XRegs &x, const uint8_t *row, int g, const Tables &) {
        const uint2 hd = *reinterpret_cast<const uint2 *>(row);
        const uint8_t *q = row + 8 + 32 * g;
        /* the block's last eight bytes lie in the last piece, eight bytes further on */
        const uint2 c0 = *reinterpret_cast<const uint2 *>(q), c1 = *reinterpret_cast<const uint2 *>(q + 8), c2 = *reinterpret_cast<const uint2 *>(q + 16),
                    c3 = *reinterpret_cast<const uint2 *>(g == 3 ? row + 136 : q + 24);
        const uint32_t qs[8] = {c0.x, c0.y, c1.x, c1.y, c2.x, c2.y, c3.x, c3.y};
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
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.A[2 * h + u], b, c, 0, 0, 0);
            }
            const int j = 2 * g + h;
            const uint32_t ls = ((hd.y >> (4 * j)) & 15u) | (((hd.x >> (16 + 2 * j)) & 3u) << 4);
            acc = fmaf(join_digits(c) * x.m[2 * h], (float)((int)ls - 32), acc);
        }
        return half_bits_fast(hd.x & 0xFFFFu) * acc;
    }
};

template <> struct DmaFmt<T_IQ2_XXS> : GridFmt<T_IQ2_XXS> {
    typedef XRegs X;
    __device__ static void prepare(v4f v, uint8_t *xs, int lane, X &x) { prepare_regs<GridFmt<T_IQ2_XXS>>(v, xs, lane, kOff, x); }
    static constexpr int kPieces = 5;
    __device__ static uint32_t piece_src(uint32_t p) { return p < 4 ? 16u * p : 50u; }
    static constexpr float kOff = 1.0f;
    __device__ static float item(const XRegs &x, const uint8_t *row, int g, const Tables &t) {
        uint32_t w[5]; /* from byte 16 g on: the codes start two bytes in, those of lane group 3 end in the last piece */
#pragma unroll
        for (int i = 0; i < 4; i++) w[i] = lds4(row + 16 * g + 4 * i);
        w[4] = lds4(row + (g == 3 ? 76 : 16 * g + 16));
        if (g == 3) w[4] >>= 16;
        const float d = half_bits_fast(*reinterpret_cast<const uint16_t *>(row)) * 0.25f;
        const uint2 *grid = reinterpret_cast<const uint2 *>(t.grid);
        float acc = 0.0f;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t a0 = __builtin_amdgcn_alignbit(w[2 * h + 1], w[2 * h], 16), a1 = __builtin_amdgcn_alignbit(w[2 * h + 2], w[2 * h + 1], 16);
            v4i c = {0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const uint2 m0 = grid[(a0 >> (16 * q)) & 255u], m1 = grid[(a0 >> (16 * q + 8)) & 255u];
                const uint2 s0 = t.sign128[(a1 >> (14 * q)) & 127u], s1 = t.sign128[(a1 >> (14 * q + 7)) & 127u];
                const v4i b = {apply_signs(m0.x, s0.x), apply_signs(m0.y, s0.y), apply_signs(m1.x, s1.x), apply_signs(m1.y, s1.y)};
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.A[2 * h + q], b, c, 0, 0, 0);
            }
            acc = fmaf(join_digits(c) * x.m[2 * h], 0.5f + (float)(a1 >> 28), acc);
        }
        return d * acc;
    }
};

template <> struct DmaFmt<T_IQ3_S> : GridFmt<T_IQ3_S> {
    typedef XRegs X;
    __device__ static void prepare(v4f v, uint8_t *xs, int lane, X &x) { prepare_regs<GridFmt<T_IQ3_S>>(v, xs, lane, kOff, x); }
    static constexpr int kPieces = 7;
    __device__ static uint32_t piece_src(uint32_t p) { return p < 6 ? 16u * p : 94u; }
    static constexpr float kOff = 1.0f;
    __device__ static float item(const XRegs &x, const uint8_t *row, int g, const Tables &t) {
        uint32_t w[5], v[3];
#pragma unroll
        for (int i = 0; i < 5; i++) w[i] = lds4(row + 16 * g + 4 * i); /* index bytes from 2 on */
        /* sign bytes 74 + 8 g ..: from byte 94 on the image has the block's bytes two further on */
#pragma unroll
        for (int i = 0; i < 3; i++) v[i] = lds4(row + 72 + 8 * g + 4 * i + (g == 3 ? 4 : 0));
        const uint32_t ssh = g == 3 ? 0u : 16u;
        const uint32_t sg[2] = {__builtin_amdgcn_alignbit(v[1], v[0], ssh), g == 2 ? v[2] : __builtin_amdgcn_alignbit(v[2], v[1], ssh)};
        const uint32_t qh = *reinterpret_cast<const uint16_t *>(row + 66 + 2 * g), scales = row[108 + g];
        const float d = half_bits_fast(*reinterpret_cast<const uint16_t *>(row));
        float acc = 0.0f;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            v4i c = {0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const uint32_t ix = __builtin_amdgcn_alignbit(w[2 * h + q + 1], w[2 * h + q], 16);
                const uint32_t hb = qh >> (8 * h + 4 * q); /* bits 0..3: the ninth bits of these four indices */
                const uint2 s0 = t.sign256[(sg[h] >> (16 * q)) & 255u], s1 = t.sign256[(sg[h] >> (16 * q + 8)) & 255u];
                const uint32_t i0 = (ix & 255u) | ((hb & 1u) << 8), i1 = ((ix >> 8) & 255u) | ((hb & 2u) << 7);
                const uint32_t i2 = ((ix >> 16) & 255u) | ((hb & 4u) << 6), i3 = (ix >> 24) | ((hb & 8u) << 5);
                const v4i b = {apply_signs(t.grid[i0], s0.x), apply_signs(t.grid[i1], s0.y), apply_signs(t.grid[i2], s1.x), apply_signs(t.grid[i3], s1.y)};
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.A[2 * h + q], b, c, 0, 0, 0);
            }
            acc = fmaf(join_digits(c) * x.m[2 * h], (float)(1u + 2u * ((scales >> (4 * h)) & 15u)), acc);
        }
        return d * acc;
    }
};

template <int N> __device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }

__device__ __forceinline__ void request16(uint32_t lds_at, uint32_t voff, __amdgpu_buffer_rsrc_t rsrc, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds_at)), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory");
}

/* RG: rows of a group, 16 or 8; S: images of a wave; LONG: a wave has several super-blocks of a row */
template <class F, int RG, int S, bool LONG> struct DmaShape {
    static constexpr int kImage = RG * F::kPieces * 16;
    static constexpr int kXSlots = LONG ? S : 1;
    static constexpr int kWaveLds = S * kImage + kXSlots * kXScratch;
    static constexpr int kBudget = 160 * 1024 - 1024 - (F::kGridBytes > 0 ? F::kGridBytes + 384 * 8 : 0); /* of the dynamic LDS */
};

/* KIND: one matrix, several whose rows follow each other (whole row groups of 16 each), or a gate and up pair - a row group is then
 * eight rows of either */
enum Kind : int { kOne, kSeveral, kPair };

template <class F, int RG, int S, bool LONG, Kind KIND>
__global__ void __launch_bounds__(kMaxWaves * 64)
gemv_dma_kernel(const JobView job, const float *__restrict__ x, int n_sb, int rows_per_wg, uint32_t row_bytes) {
    using D = DmaShape<F, RG, S, LONG>;
    constexpr int kRow = F::kPieces * 16, NQ = ((KIND == kPair ? 8 : RG) * kRow + 1023) / 1024, NI = KIND == kPair ? 2 * NQ : NQ; /* requests of an image */
    extern __shared__ __attribute__((aligned(1024))) uint8_t dma_lds[];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n_waves = blockDim.x >> 6;
    const int n = lane & 15, g = lane >> 4;
    constexpr int R = KIND == kPair ? 8 : RG; /* rows of a matrix in a group */
    const int n0 = job.n0, n1 = job.n1, n2 = job.n2;
    const int row0 = blockIdx.x * rows_per_wg;
    const int rows_here = min(rows_per_wg, (KIND == kSeveral ? n0 + n1 + n2 : n0) - row0);
    const int n_rg = (rows_here + R - 1) / R;
    const int n_kc = LONG ? (n_sb - wv + n_waves - 1) / n_waves : 1, n_items = n_kc * n_rg;

    uint8_t *img = dma_lds + wv * D::kWaveLds, *xs = img + S * D::kImage;
    float *partial = reinterpret_cast<float *>(dma_lds + n_waves * D::kWaveLds);
    const int cap = n_rg * RG; /* partial sums: [wave][row] */
    const uint32_t img_at = (uint32_t)(uintptr_t)(lds_void *)img, xs_at = img_at + S * D::kImage;

    uint32_t voff[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const uint32_t id = 64u * q + lane, row = id / F::kPieces, src = F::piece_src(id % F::kPieces);
        voff[q] = src != kNone ? row * row_bytes + src : kPastEnd;
    }
    const bool w_last = 64 * (NQ - 1) + lane < R * F::kPieces; /* lanes past the image stay out */
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(x), 0, n_sb * 1024, 0x00020000);
    /* the codebook comes the same way, ahead of everything else; the sign masks are built */
    __shared__ __attribute__((aligned(1024))) uint32_t grid_lds[F::kGridBytes > 0 ? F::kGridBytes / 4 : 4];
    __shared__ __attribute__((aligned(16))) uint2 sign_lds[F::kGridBytes > 0 ? 256 + 128 : 2];
    const Tables tab = {grid_lds, sign_lds, sign_lds + (F::kGridBytes > 0 ? 256 : 0)};
    if constexpr (F::kGridBytes > 0) {
        static_assert(F::kGridBytes % 1024 == 0, "whole requests");
        const __amdgpu_buffer_rsrc_t t_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t *>(F::grid_src()), 0, F::kGridBytes, 0x00020000);
        for (int k = wv; k < F::kGridBytes / 1024; k += n_waves)
            request16((uint32_t)(uintptr_t)(lds_void *)grid_lds + 1024u * k, 16u * lane, t_rsrc, 1024u * k);
    }
    int rq_kc = 0, rq_rg = 0, rq_slot = 0; /* of the item to be requested next */
    auto request = [&]() {
        if (rq_rg == 0)
            request16(xs_at + (uint32_t)(LONG ? rq_kc % D::kXSlots * kXScratch : 0), 16u * lane, x_rsrc, (uint32_t)(wv + n_waves * rq_kc) * 1024u);
        const uint8_t *base = job.W0;
        int r = row0 + rq_rg * R, lim = row0 + rows_here;
        if (KIND == kSeveral) {
            if (r < n0) {
                lim = min(lim, n0);
            } else if (r < n0 + n1) {
                base = job.W1;
                r -= n0;
                lim = min(lim - n0, n1);
            } else {
                base = job.W2;
                r -= n0 + n1;
                lim -= n0 + n1;
            }
        }
        const int bytes = (int)((uint32_t)(min(R, lim - r) - 1) * row_bytes + (uint32_t)n_sb * F::kBlock);
        const uint32_t soff = (uint32_t)(wv + n_waves * rq_kc) * (uint32_t)F::kBlock, at = img_at + (uint32_t)(rq_slot * D::kImage);
#pragma unroll
        for (int m = 0; m < (KIND == kPair ? 2 : 1); m++) {
            const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<uint8_t *>(m ? job.W1 : base) + (size_t)r * row_bytes, 0, bytes, 0x00020000);
#pragma unroll
            for (int q = 0; q < NQ; q++)
                if (q + 1 < NQ || w_last) request16(at + (uint32_t)(m * R * kRow) + 1024u * q, voff[q], rsrc, soff);
        }
        rq_slot = rq_slot + 1 == S ? 0 : rq_slot + 1;
        if (++rq_rg == n_rg) {
            rq_rg = 0;
            rq_kc++;
        }
    };
#pragma unroll
    for (int s = 0; s < S; s++)
        if (s < n_items) request();

    if constexpr (F::kGridBytes > 0) {
        for (int i = threadIdx.x; i < 384; i += blockDim.x) {
            const uint32_t sb = i < 256 ? (uint32_t)i : iq_sign_byte(i - 256);
            sign_lds[i] = make_uint2(spread4(sb) * 0xFFu, spread4(sb >> 4) * 0xFFu);
        }
        if (S < n_items) wait_vm<S * NI>(); /* the codebook was asked for first */
        else wait_vm<0>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    typename F::X xr;
    int slot = 0, left = n_items;
    float lone = 0.0f; /* LONG with one row group: the row's shares stay in a register */
    for (int kc = 0; kc < n_kc; kc++) {
        for (int rg = 0; rg < n_rg; rg++, left--) {
            if (rg == 0) {
                if (kc == 0) { /* x came first: its digits are made while the blocks are on their way */
                    if (n_items < S) wait_vm<NI>();
                    else if (LONG && n_rg == 1) wait_vm<S * NI + S - 1>();
                    else wait_vm<S * NI>();
                } else {
                    if (left < S) wait_vm<0>();
                    else if (LONG && n_rg == 1) wait_vm<(S - 1) * (NI + 1)>();
                    else wait_vm<(S - 1) * NI>();
                }
                uint8_t *xp = xs + (LONG ? kc % D::kXSlots * kXScratch : 0);
                v4f v = *reinterpret_cast<const v4f *>(xp + 16 * lane);
                asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v) : : "memory"); /* read before the digits take its place */
                F::prepare(v, xp, lane, xr);
            }
            if (left < S) wait_vm<0>();
            else if (LONG && n_rg == 1) wait_vm<(S - 1) * (NI + 1)>();
            else wait_vm<(S - 1) * NI>();
            const float v = sum_lane_groups(F::item(xr, img + slot * D::kImage + (n & (RG - 1)) * kRow, g, tab));
            if (LONG && n_rg == 1) lone += v;
            else if (lane < RG) {
                float *p = partial + wv * cap + rg * RG + n;
                *p = LONG && kc > 0 ? *p + v : v;
            }
            slot = slot + 1 == S ? 0 : slot + 1;
            if (left > S) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* the slot has been read before it is refilled */
                request();
            }
        }
    }
    if (LONG && n_rg == 1 && lane < RG) partial[wv * cap + n] = lone;
    __syncthreads();
    auto row_total = [&](int lr) { /* all sixteen reads at once; a loop over the waves waited for each (0.3 to 0.6 us) */
        float v[kMaxWaves], s = 0.0f;
#pragma unroll
        for (int k = 0; k < kMaxWaves; k++) v[k] = partial[min(k, n_waves - 1) * cap + lr];
#pragma unroll
        for (int k = 0; k < kMaxWaves; k++) v[k] = k < n_waves ? v[k] : 0.0f;
#pragma unroll
        for (int k = 0; k < kMaxWaves; k += 4) s += (v[k] + v[k + 1]) + (v[k + 2] + v[k + 3]);
        return s;
    };
    for (int lr = threadIdx.x; lr < rows_here; lr += blockDim.x) {
        if (KIND == kPair) {
            const int at = (lr >> 3) * 16 + (lr & 7);
            job.y0[row0 + lr] = silu_times(row_total(at), row_total(at + 8));
            continue;
        }
        const float s = row_total(lr);
        if (KIND == kOne) {
            job.y0[row0 + lr] = job.mode == 1 ? job.y0[row0 + lr] + s : s;
        } else {
            const uint8_t *Wm;
            float *ym;
            int r;
            job_locate(job, row0 + lr, Wm, ym, r);
            ym[r] = job.mode == 1 ? ym[r] + s : s;
        }
    }
}

template <class F, int RG, int S, bool LONG, Kind KIND>
hipError_t dma_launch(const GemvJob &job, const float *x, int n_sb, int rows_per_wg, int waves, size_t pitch, hipStream_t stream) {
    using D = DmaShape<F, RG, S, LONG>;
    const auto kernel = gemv_dma_kernel<F, RG, S, LONG, KIND>;
    static OnceFlag lds_raised;
    if (!lds_raised.is_set()) {
        const hipError_t e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, D::kBudget);
        if (e != hipSuccess) return e;
        lds_raised.set();
    }
    constexpr int R = KIND == kPair ? 8 : RG;
    const int n_rows = KIND == kPair ? job.n_rows[0] : job.total_rows();
    const size_t lds = (size_t)waves * (D::kWaveLds + (size_t)((rows_per_wg + R - 1) / R) * RG * sizeof(float));
    hipLaunchKernelGGL(kernel, dim3((n_rows + rows_per_wg - 1) / rows_per_wg), dim3(64 * waves), lds, stream, job_view(job), x, n_sb, rows_per_wg,
                       (uint32_t)pitch);
    return hipGetLastError();
}

/* Where this kernel measured faster than the one that would run instead (gemv_grid.hip, gemv_int.hip); us, that one / this, rows x
 * columns, 2 x: a gate and up pair. Over 512 to 32000 rows x 1024 to 14336 columns the choice costs 0.1 to 0.5 % of the better one's time in
 * the geometric mean by format, 1.1 % with IQ2_XXS tensors alone.
 *   Q4_K, whose own kernels (gemv_q4k.hip) have this structure for one matrix and the same items: many rows of up to 2048 columns (32000 x
 *     1024 8.5 / 6.7, 2 x 14336 x 2048 9.2 / 8.3) and of 17 to 24 super-blocks (2 x 32000 x 5632 43.6 / 40.1; 9216 x 3072 5.3 / 5.9)
 *   Q6_K, Q5_K, Q3_K everywhere (256 to 151936 rows x 1024 to 14336: 1.21, 1.23 and 1.41 times faster in the mean, pairs 1.29, 1.34, 1.62)
 *   Nine to fifteen super-blocks: as many waves with an item or two each, which do not make up for the start, until a wave has several;
 *     with one row group each it is even or better again
 *       Q8_0 tensors of 3073 to 8192 rows (6144 x 2560 1.07 times the time), pairs of 1537 to 4096 (2 x 4096 x 2304 1.09; 2 x 512 x 2304 0.77)
 *       Q4_0, IQ4_NL, IQ4_XS, Q2_K from eight on: tensors of up to 9216 rows (6144 x 2560 Q4_0 4.1 / 4.5, IQ4_XS 1.04 times the time), pairs of up
 *         to 6144 (2 x 4096 x 2560 4.4 / 4.9, 1.12 times; IQ4_XS 2 x 2048 x 2048 1.07)
 *   Q8_0 of twelve to sixteen super-blocks and many rows, which its own kernel streams row by row: 32000 x 4096 24.7 / 25.8; pairs of
 *     eleven to sixteen from 8193 rows on (2 x 9216 x 4096 15.7 / 18.8, 2 x 14336 x 3072 1.06 times the time, 2 x 14336 x 4096 1.12)
 *   Q2_K, IQ4_XS: few rows of more than 10240 and 12288 columns, whose blocks are small beside the x that every workgroup prepares (1024
 *     x 14336 7.2 / 7.7, 8.7 / 9.1)
 *   IQ3_S, IQ2_XXS, whose workgroups wait for their tables together, which rows must be many enough to cover: IQ3_S 6144 x 4096 7.4 / 7.8,
 *     4096 x 6144 1.09 times the time, 2 x 512 x 4096 1.10, IQ2_XXS 4096 x 11008 7.2 / 8.7, 2 x 4096 x 4096 1.24, 2 x 4096 x 6144 1.21, but
 *     32000 x 2048 14.2 / 10.4, 11.4 / 8.7, 2 x 14336 x 8192 43 / 28, 24 / 21 */
bool dma_pays(uint32_t type, Kind kind, int n_rows, int n_sb) {
    const bool pair = kind == kPair, narrow = n_sb >= 9 && n_sb <= 15;
    switch (type) {
    case T_Q4_K: {
        const long long rows = (pair ? 2 : 1) * (long long)n_rows;
        return (n_sb <= 8 && rows >= 16384) || (n_sb >= 17 && n_sb <= 24 && rows >= 12288);
    }
    case T_Q6_K: case T_Q5_K: case T_Q3_K: return true;
    case T_Q8_0:
        if (pair) return !(narrow && n_rows > 1536 && n_rows <= 4096) && !(n_sb >= 11 && n_sb <= 16 && n_rows > 8192);
        return !(narrow && n_rows > 3072 && n_rows <= 8192) && !(n_sb >= 12 && n_sb <= 16 && n_rows > 16384);
    case T_Q4_0: case T_IQ4_NL: case T_IQ4_XS: case T_Q2_K:
        if ((narrow || n_sb == 8) && n_rows <= (pair ? 6144 : 9216)) return false;
        return pair || n_rows > 4096 || !((type == T_Q2_K && n_sb > 40) || (type == T_IQ4_XS && n_sb > 48));
    case T_IQ3_S: return pair ? !(n_sb >= 9 && n_sb <= 16 && n_rows <= 4096) : !(n_sb >= 9 && n_sb <= 24 && n_rows > 3072 && n_rows <= 8192);
    case T_IQ2_XXS:
        if (n_sb < 8) return true;
        if (n_sb <= 12) return n_rows >= (pair ? 9216 : 14336);
        return pair && n_sb > 16 && !(n_sb <= 24 && n_rows > 2048 && n_rows <= 4096);
    default: return false;
    }
}

/* how a call runs here: waves of a workgroup and its rows; waves 0: it does not */
struct DmaPlan { int waves, rows_per_wg, rounds; bool lng; };

template <uint32_t T> DmaPlan dma_plan(Kind kind, int n_mat, const int *n_rows_of, int n_cols, size_t pitch, int n_cu) {
    using Short = DmaShape<DmaFmt<T>, 16, 2, false>;
    using Long = DmaShape<DmaFmt<T>, 16, 2, true>;
    const DmaPlan none = {0, 0, 0, false};
    const int n_sb = n_cols / 256;
    if (n_cols % 256 != 0 || n_sb < 1 || n_sb > 64 || pitch > (1u << 24)) return none;
    int n_rows = n_rows_of[0];
    if (kind == kSeveral)
        for (int m = 1; m < n_mat; m++) {
            if (n_rows_of[m - 1] % 16) return none; /* a row group would hold rows of two matrices */
            n_rows += n_rows_of[m];
        }
    if (n_rows == 0 || !dma_pays(T, kind, n_rows, n_sb)) return none;
    DmaPlan p;
    p.waves = n_sb < kMaxWaves ? n_sb : kMaxWaves;
    while (p.waves < n_sb && p.waves * Long::kWaveLds > Long::kBudget - 1024) p.waves--; /* Q8_0: 14 */
    p.lng = p.waves < n_sb;
    /* one workgroup per compute unit where its partial sums fit in LDS, else so many equal rounds of workgroups that they do */
    const int unit = kind == kSeveral ? 16 : kind == kPair ? 8 : 1, group = kind == kPair ? 8 : 16;
    const int max_rows = (Long::kBudget - p.waves * (p.lng ? Long::kWaveLds : Short::kWaveLds)) / (16 * p.waves * (int)sizeof(float)) * group;
    const int per_cu = (n_rows + n_cu - 1) / n_cu;
    p.rounds = (per_cu + max_rows - 1) / max_rows;
    p.rows_per_wg = ((n_rows + n_cu * p.rounds - 1) / (n_cu * p.rounds) + unit - 1) / unit * unit;
    return p;
}

template <uint32_t T>
bool dma_typed(const GemvJob &job, const float *x, int n_cols, int n_cu, hipStream_t stream, hipError_t *err, size_t row_stride) {
    using F = DmaFmt<T>;
    if ((uintptr_t)x & 15 || row_stride % F::kAlign) return false;
    for (int m = 0; m < job.n_mat; m++)
        if ((uintptr_t)job.W[m] % F::kAlign) return false;
    const Kind kind = job.mode == kSiluMul ? kPair : job.n_mat > 1 ? kSeveral : kOne;
    const size_t pitch = row_stride ? row_stride : (size_t)(n_cols / 256) * F::kBlock;
    const DmaPlan p = dma_plan<T>(kind, job.n_mat, job.n_rows, n_cols, pitch, n_cu);
    if (!p.waves) return false;
    const auto go = [&](auto launch) { *err = launch(job, x, n_cols / 256, p.rows_per_wg, p.waves, pitch, stream); };
    if (kind == kPair) p.lng ? go(dma_launch<F, 16, 2, true, kPair>) : go(dma_launch<F, 16, 2, false, kPair>);
    else if (kind == kSeveral) p.lng ? go(dma_launch<F, 16, 2, true, kSeveral>) : go(dma_launch<F, 16, 2, false, kSeveral>);
    else if (p.rows_per_wg <= 8) p.lng ? go(dma_launch<F, 8, 2, true, kOne>) : go(dma_launch<F, 8, 2, false, kOne>);
    else p.lng ? go(dma_launch<F, 16, 2, true, kOne>) : go(dma_launch<F, 16, 2, false, kOne>);
    return true;
}

template <uint32_t T> int dma_probe(bool pair, int n_mat, const int *n_rows, int n_cols, int n_cu) {
    const DmaPlan p = dma_plan<T>(pair ? kPair : n_mat > 1 ? kSeveral : kOne, n_mat, n_rows, n_cols, (size_t)(n_cols / 256) * DmaFmt<T>::kBlock, n_cu);
    return p.waves + 100 * p.rounds;
}

}  // namespace

bool launch_gemv_dma(uint32_t type, const GemvJob &job, const float *x, int n_cols, int n_cu, hipStream_t stream, hipError_t *err,
                     size_t row_stride) {
    *err = hipSuccess;
    switch (type) {
    case T_Q4_K: return dma_typed<T_Q4_K>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q6_K: return dma_typed<T_Q6_K>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q8_0: return dma_typed<T_Q8_0>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q5_K: return dma_typed<T_Q5_K>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q2_K: return dma_typed<T_Q2_K>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q3_K: return dma_typed<T_Q3_K>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q4_0: return dma_typed<T_Q4_0>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_IQ4_NL: return dma_typed<T_IQ4_NL>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_IQ4_XS: return dma_typed<T_IQ4_XS>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_IQ2_XXS: return dma_typed<T_IQ2_XXS>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_IQ3_S: return dma_typed<T_IQ3_S>(job, x, n_cols, n_cu, stream, err, row_stride);
    default: return false;
    }
}

int probe_gemv_dma(uint32_t type, bool pair, int n_mat, const int *n_rows, int n_cols, int n_cu) {
    switch (type) {
    case T_Q4_K: return dma_probe<T_Q4_K>(pair, n_mat, n_rows, n_cols, n_cu);
    case T_Q6_K: return dma_probe<T_Q6_K>(pair, n_mat, n_rows, n_cols, n_cu);
    case T_Q8_0: return dma_probe<T_Q8_0>(pair, n_mat, n_rows, n_cols, n_cu);
    case T_Q5_K: return dma_probe<T_Q5_K>(pair, n_mat, n_rows, n_cols, n_cu);
    case T_Q2_K: return dma_probe<T_Q2_K>(pair, n_mat, n_rows, n_cols, n_cu);
    case T_Q3_K: return dma_probe<T_Q3_K>(pair, n_mat, n_rows, n_cols, n_cu);
    case T_Q4_0: return dma_probe<T_Q4_0>(pair, n_mat, n_rows, n_cols, n_cu);
    case T_IQ4_NL: return dma_probe<T_IQ4_NL>(pair, n_mat, n_rows, n_cols, n_cu);
    case T_IQ4_XS: return dma_probe<T_IQ4_XS>(pair, n_mat, n_rows, n_cols, n_cu);
    case T_IQ2_XXS: return dma_probe<T_IQ2_XXS>(pair, n_mat, n_rows, n_cols, n_cu);
    case T_IQ3_S: return dma_probe<T_IQ3_S>(pair, n_mat, n_rows, n_cols, n_cu);
    default: return 0;
    }
}

}  // namespace qlin

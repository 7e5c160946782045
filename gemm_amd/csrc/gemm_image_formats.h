/*
 * gemm_image_formats.h - eleven block formats as the kernels see them that copy whole blocks into an LDS image and cut
 * the codes of eight elements out of it (gemm_fewtok.h, gemm_f32_split.h).
 */
#ifndef QLIN_GEMM_IMAGE_FORMATS_H
#define QLIN_GEMM_IMAGE_FORMATS_H

#include <utility>

#include "gemm_kq_formats.h"

namespace qlin {

using namespace kq;

namespace {

QLIN_INL uint32_t lds_u32(const uint8_t *p) { return *reinterpret_cast<const uint32_t *>(p); }
QLIN_INL uint32_t lds_u16(const uint8_t *p) { return *reinterpret_cast<const uint16_t *>(p); }
/* eight bytes from byte offset AT + var of an image row (16-byte aligned), var a multiple of 4 */
template <int AT> QLIN_INL void lds_bytes8(const uint8_t *row, int var, uint32_t &a, uint32_t &b) {
    const uint8_t *p = row + (AT & ~3) + var;
    if constexpr ((AT & 3) == 0) {
        a = lds_u32(p);
        b = lds_u32(p + 4);
    } else {
        const uint32_t w0 = lds_u32(p), w1 = lds_u32(p + 4), w2 = lds_u32(p + 8);
        a = __builtin_amdgcn_alignbyte(w1, w0, AT & 3);
        b = __builtin_amdgcn_alignbyte(w2, w1, AT & 3);
    }
}
/* byte 0xFF for every set bit of the low four bits of v */
QLIN_INL uint32_t mask_bytes(uint32_t v) { return (((v & 15u) * 0x00204081u) & 0x01010101u) * 255u; }
QLIN_INL uint32_t with_signs(uint32_t mag, uint32_t m) { return ((mag ^ m) + (m & 0x01010101u)) ^ 0x80808080u; } /* + 128 */
template <int N> QLIN_INL uint32_t shifted(uint32_t v) { /* v >> N, v << -N */
    if constexpr (N >= 0) return v >> N;
    else return v << -N;
}
QLIN_INL float signed_byte(uint32_t w, int at) { return (float)(int)(int8_t)(w >> at); }

/* What the kernel needs to know of a format. `row` is a lane's block in its wave's image; 256 elements (a super-block or
 * as many blocks) are the unit; lane (j, kg) owns elements 32 u + 8 kg .. + 7.
 *   kPieces     16-byte pieces of a row's image, odd so that 16 rows fall into 16 different bank groups; piece_src gives
 *               a piece's place in the block - the last one ends with the block, so that no request leaves the tensor -
 *               or kNoPiece for padding
 *   codes<u>    the lane's eight codes as unsigned bytes; kSmall: all below 16
 *   ready<u>    (kReady > 0) the low bytes of bf16 numbers kBase + code, whose high bytes are all kReady
 *   kOffset     what the format subtracts from a code
 *   scale<u>    the factor of the lane's elements; minimum<u> (kHasMin): what is subtracted after that
 *   kGroup16    the factor belongs to 16 elements, not 32
 *   kShare      steps u that are scheduled together
 *   kUnrounded  token count up to which the few-token kernel leaves the codes unrounded */
constexpr uint32_t kNoPiece = 0xFFFFFFFFu;

struct HdrK4 { float d, dmin; uint32_t sc_lo, sc_hi, mn_lo, mn_hi; };
QLIN_INL HdrK4 k4_header(const uint8_t *row) {
    const u32x4 h = *reinterpret_cast<const u32x4 *>(row);
    HdrK4 r;
    r.d = half_bits_fast(h.x & 0xFFFFu);
    r.dmin = half_bits_fast(h.x >> 16);
    r.sc_lo = h.y & 0x3F3F3F3Fu;
    r.mn_lo = h.z & 0x3F3F3F3Fu;
    r.sc_hi = (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u);
    r.mn_hi = ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u);
    return r;
}
struct TQ4K {
    static constexpr int kBlock = 144, kPieces = 9, kOffset = 0, kTable = 0, kReady = 0, kBase = 0, kShare = 2, kUnrounded = 32;
    static constexpr bool kSmall = true, kHasMin = true, kGroup16 = false;
    static QLIN_INL uint32_t piece_src(uint32_t p) { return 16u * p; }
    typedef HdrK4 Hdr;
    static QLIN_INL Hdr header(const uint8_t *row, int) { return k4_header(row); }
    template <int U> static QLIN_INL void codes(const uint8_t *row, int kg, const uint32_t *, uint32_t &a, uint32_t &b) {
        lds_bytes8<16 + 32 * (U >> 1)>(row, 8 * kg, a, b);
        a = (a >> (4 * (U & 1))) & 0x0F0F0F0Fu;
        b = (b >> (4 * (U & 1))) & 0x0F0F0F0Fu;
    }
    template <int U> static QLIN_INL float scale(const Hdr &h, int) { return h.d * ubyte_f32<U & 3>(U < 4 ? h.sc_lo : h.sc_hi); }
    template <int U> static QLIN_INL float minimum(const Hdr &h, int) { return h.dmin * ubyte_f32<U & 3>(U < 4 ? h.mn_lo : h.mn_hi); }
};
struct TQ5K {
    static constexpr int kBlock = 176, kPieces = 11, kOffset = 0, kTable = 0, kReady = 0x42, kBase = 32, kShare = 2, kUnrounded = 24;
    static constexpr bool kSmall = false, kHasMin = true, kGroup16 = false;
    static QLIN_INL uint32_t piece_src(uint32_t p) { return 16u * p; }
    typedef HdrK4 Hdr;
    static QLIN_INL Hdr header(const uint8_t *row, int) { return k4_header(row); }
    template <int U> static QLIN_INL void codes(const uint8_t *row, int kg, const uint32_t *, uint32_t &a, uint32_t &b) {
        uint32_t h0, h1;
        lds_bytes8<16>(row, 8 * kg, h0, h1);
        lds_bytes8<48 + 32 * (U >> 1)>(row, 8 * kg, a, b);
        a = ((a >> (4 * (U & 1))) & 0x0F0F0F0Fu) | (((h0 >> U) & 0x01010101u) << 4);
        b = ((b >> (4 * (U & 1))) & 0x0F0F0F0Fu) | (((h1 >> U) & 0x01010101u) << 4);
    }
    /* 32 + code = 2^5 (1 + 4 code / 128) */
    template <int U> static QLIN_INL void ready(const uint8_t *row, int kg, const uint32_t *, uint32_t &a, uint32_t &b) {
        uint32_t h0, h1;
        lds_bytes8<16>(row, 8 * kg, h0, h1);
        lds_bytes8<48 + 32 * (U >> 1)>(row, 8 * kg, a, b);
        a = (shifted<U & 1 ? 2 : -2>(a) & 0x3C3C3C3Cu) | (shifted<U - 6>(h0) & 0x40404040u);
        b = (shifted<U & 1 ? 2 : -2>(b) & 0x3C3C3C3Cu) | (shifted<U - 6>(h1) & 0x40404040u);
    }
    template <int U> static QLIN_INL float scale(const Hdr &h, int kg) { return TQ4K::scale<U>(h, kg); }
    template <int U> static QLIN_INL float minimum(const Hdr &h, int kg) { return TQ4K::minimum<U>(h, kg); }
};
struct TQ6K {
    static constexpr int kBlock = 210, kPieces = 15, kOffset = 32, kTable = 0, kReady = 0x42, kBase = 64, kShare = 2, kUnrounded = 24;
    static constexpr bool kSmall = false, kHasMin = false, kGroup16 = true;
    static QLIN_INL uint32_t piece_src(uint32_t p) { return p < 13 ? 16u * p : p == 13 ? 194u : kNoPiece; }
    struct Hdr { float d; u32x4 sc; }; /* the scales shifted so that the lane's are bytes 0 and 2 of a dword */
    static QLIN_INL Hdr header(const uint8_t *row, int kg) {
        Hdr h;
        h.sc = *reinterpret_cast<const u32x4 *>(row + 192) >> (uint32_t)(8 * (kg >> 1));
        h.d = half_bits_fast(lds_u32(row + 220) >> 16);
        return h;
    }
    template <int U> static QLIN_INL void codes(const uint8_t *row, int kg, const uint32_t *, uint32_t &a, uint32_t &b) {
        constexpr int n = U >> 2, q = U & 3;
        uint32_t h0, h1;
        lds_bytes8<64 * n + 32 * (q & 1)>(row, 8 * kg, a, b);
        lds_bytes8<128 + 32 * n>(row, 8 * kg, h0, h1);
        a = ((a >> (4 * (q >> 1))) & 0x0F0F0F0Fu) | (((h0 >> (2 * q)) & 0x03030303u) << 4);
        b = ((b >> (4 * (q >> 1))) & 0x0F0F0F0Fu) | (((h1 >> (2 * q)) & 0x03030303u) << 4);
    }
    /* 64 + code = 2^6 (1 + 2 code / 128) */
    template <int U> static QLIN_INL void ready(const uint8_t *row, int kg, const uint32_t *, uint32_t &a, uint32_t &b) {
        constexpr int n = U >> 2, q = U & 3;
        uint32_t h0, h1;
        lds_bytes8<64 * n + 32 * (q & 1)>(row, 8 * kg, a, b);
        lds_bytes8<128 + 32 * n>(row, 8 * kg, h0, h1);
        a = (shifted<(q >> 1 ? 3 : -1)>(a) & 0x1E1E1E1Eu) | (shifted<2 * q - 5>(h0) & 0x60606060u) | 0x80808080u;
        b = (shifted<(q >> 1 ? 3 : -1)>(b) & 0x1E1E1E1Eu) | (shifted<2 * q - 5>(h1) & 0x60606060u) | 0x80808080u;
    }
    template <int U> static QLIN_INL float scale(const Hdr &h, int) { return h.d * signed_byte(h.sc[U >> 1], 16 * (U & 1)); }
    template <int U> static QLIN_INL float minimum(const Hdr &, int) { return 0.0f; }
};
struct TQ8_0 {
    static constexpr int kBlock = 272, kPieces = 17, kOffset = 128, kTable = 0, kReady = 0, kBase = 0, kShare = 1, kUnrounded = 24;
    static constexpr bool kSmall = false, kHasMin = false, kGroup16 = false;
    static QLIN_INL uint32_t piece_src(uint32_t p) { return 16u * p; }
    struct Hdr { const uint8_t *row; };
    static QLIN_INL Hdr header(const uint8_t *row, int) { return Hdr{row}; }
    template <int U> static QLIN_INL void codes(const uint8_t *row, int kg, const uint32_t *, uint32_t &a, uint32_t &b) {
        lds_bytes8<34 * U + 2>(row, 8 * kg, a, b);
        a ^= 0x80808080u;
        b ^= 0x80808080u;
    }
    template <int U> static QLIN_INL float scale(const Hdr &h, int) { return half_bits_fast(lds_u16(h.row + 34 * U)); }
    template <int U> static QLIN_INL float minimum(const Hdr &, int) { return 0.0f; }
};
struct TQ2K {
    static constexpr int kBlock = 84, kPieces = 7, kOffset = 0, kTable = 0, kReady = 0, kBase = 0, kShare = 2, kUnrounded = 24;
    static constexpr bool kSmall = true, kHasMin = true, kGroup16 = true;
    static QLIN_INL uint32_t piece_src(uint32_t p) { return p < 5 ? 16u * p : p == 5 ? 68u : kNoPiece; }
    struct Hdr { float d, dmin; u32x4 sc; };
    static QLIN_INL Hdr header(const uint8_t *row, int kg) {
        Hdr h;
        h.sc = *reinterpret_cast<const u32x4 *>(row) >> (uint32_t)(8 * (kg >> 1));
        const uint32_t dd = lds_u32(row + 92);
        h.d = half_bits_fast(dd & 0xFFFFu);
        h.dmin = half_bits_fast(dd >> 16);
        return h;
    }
    template <int U> static QLIN_INL void codes(const uint8_t *row, int kg, const uint32_t *, uint32_t &a, uint32_t &b) {
        lds_bytes8<16 + 32 * (U >> 2)>(row, 8 * kg, a, b);
        a = (a >> (2 * (U & 3))) & 0x03030303u;
        b = (b >> (2 * (U & 3))) & 0x03030303u;
    }
    template <int U> static QLIN_INL float scale(const Hdr &h, int) { return h.d * (float)((h.sc[U >> 1] >> (16 * (U & 1))) & 15u); }
    template <int U> static QLIN_INL float minimum(const Hdr &h, int) { return h.dmin * (float)((h.sc[U >> 1] >> (16 * (U & 1) + 4)) & 15u); }
};
struct TQ3K {
    static constexpr int kBlock = 110, kPieces = 7, kOffset = 4, kTable = 0, kReady = 0, kBase = 0, kShare = 2, kUnrounded = 24;
    static constexpr bool kSmall = true, kHasMin = false, kGroup16 = true;
    static QLIN_INL uint32_t piece_src(uint32_t p) { return p < 6 ? 16u * p : 94u; }
    struct Hdr { float d; uint32_t sc[4]; }; /* byte u of the eight in sc[0..1] / sc[2..3]: 6-bit scales 2 u (+ 1: the lane's) */
    static QLIN_INL Hdr header(const uint8_t *row, int kg) {
        /* bytes 96..107 (98.. of the image): scale is = low nibble of byte is (8 and up: high nibble of byte is - 8),
         * bits 4, 5 = bits 2 (is / 4) of byte 8 + is % 4 */
        const uint32_t w0 = lds_u32(row + 96), w1 = lds_u32(row + 100), w2 = lds_u32(row + 104), w3 = lds_u32(row + 108);
        const uint32_t a = __builtin_amdgcn_alignbyte(w1, w0, 2), b = __builtin_amdgcn_alignbyte(w2, w1, 2), c = __builtin_amdgcn_alignbyte(w3, w2, 2);
        const uint32_t sh = 8u * (uint32_t)(kg >> 1);
        Hdr h;
        h.sc[0] = ((a & 0x0F0F0F0Fu) | ((c & 0x03030303u) << 4)) >> sh;
        h.sc[1] = ((b & 0x0F0F0F0Fu) | (((c >> 2) & 0x03030303u) << 4)) >> sh;
        h.sc[2] = (((a >> 4) & 0x0F0F0F0Fu) | (((c >> 4) & 0x03030303u) << 4)) >> sh;
        h.sc[3] = (((b >> 4) & 0x0F0F0F0Fu) | (((c >> 6) & 0x03030303u) << 4)) >> sh;
        h.d = half_bits_fast(w3 >> 16);
        return h;
    }
    template <int U> static QLIN_INL void codes(const uint8_t *row, int kg, const uint32_t *, uint32_t &a, uint32_t &b) {
        uint32_t h0, h1;
        lds_bytes8<32 + 32 * (U >> 2)>(row, 8 * kg, a, b);
        lds_bytes8<0>(row, 8 * kg, h0, h1);
        a = ((a >> (2 * (U & 3))) & 0x03030303u) | (((h0 >> U) & 0x01010101u) << 2);
        b = ((b >> (2 * (U & 3))) & 0x03030303u) | (((h1 >> U) & 0x01010101u) << 2);
    }
    template <int U> static QLIN_INL float scale(const Hdr &h, int) {
        return h.d * (ubyte_f32<2 * (U & 1)>(h.sc[U >> 1]) - 32.0f);
    }
    template <int U> static QLIN_INL float minimum(const Hdr &, int) { return 0.0f; }
};
struct TQ4_0 {
    static constexpr int kBlock = 144, kPieces = 9, kOffset = 8, kTable = 0, kReady = 0, kBase = 0, kShare = 1, kUnrounded = 4;
    static constexpr bool kSmall = true, kHasMin = false, kGroup16 = false;
    static QLIN_INL uint32_t piece_src(uint32_t p) { return 16u * p; }
    struct Hdr { const uint8_t *row; };
    static QLIN_INL Hdr header(const uint8_t *row, int) { return Hdr{row}; }
    template <int U> static QLIN_INL void codes(const uint8_t *row, int kg, const uint32_t *, uint32_t &a, uint32_t &b) {
        lds_bytes8<18 * U + 2>(row, 8 * (kg & 1), a, b);
        const uint32_t sh = 4u * (uint32_t)(kg >> 1);
        a = (a >> sh) & 0x0F0F0F0Fu;
        b = (b >> sh) & 0x0F0F0F0Fu;
    }
    template <int U> static QLIN_INL float scale(const Hdr &h, int) { return half_bits_fast(lds_u16(h.row + 18 * U)); }
    template <int U> static QLIN_INL float minimum(const Hdr &, int) { return 0.0f; }
};
struct TIQ4NL {
    static constexpr int kBlock = 144, kPieces = 9, kOffset = 128, kTable = 0, kReady = 0, kBase = 0, kShare = 1, kUnrounded = 4;
    static constexpr bool kSmall = false, kHasMin = false, kGroup16 = false;
    static QLIN_INL uint32_t piece_src(uint32_t p) { return 16u * p; }
    typedef TQ4_0::Hdr Hdr;
    static QLIN_INL Hdr header(const uint8_t *row, int) { return Hdr{row}; }
    template <int U> static QLIN_INL void codes(const uint8_t *row, int kg, const uint32_t *t, uint32_t &a, uint32_t &b) {
        TQ4_0::codes<U>(row, kg, t, a, b);
        a = iq4_table_bytes(a);
        b = iq4_table_bytes(b);
    }
    template <int U> static QLIN_INL float scale(const Hdr &h, int kg) { return TQ4_0::scale<U>(h, kg); }
    template <int U> static QLIN_INL float minimum(const Hdr &, int) { return 0.0f; }
};
struct TIQ4XS {
    static constexpr int kBlock = 136, kPieces = 9, kOffset = 128, kTable = 0, kReady = 0, kBase = 0, kShare = 1, kUnrounded = 4;
    static constexpr bool kSmall = false, kHasMin = false, kGroup16 = false;
    static QLIN_INL uint32_t piece_src(uint32_t p) { return p < 8 ? 16u * p : 120u; }
    struct Hdr { float d; uint32_t hi, lo; };
    static QLIN_INL Hdr header(const uint8_t *row, int) {
        Hdr h;
        const uint32_t w = lds_u32(row);
        h.d = half_bits_fast(w & 0xFFFFu);
        h.hi = w >> 16;
        h.lo = lds_u32(row + 4);
        return h;
    }
    template <int U> static QLIN_INL void codes(const uint8_t *row, int kg, const uint32_t *, uint32_t &a, uint32_t &b) {
        lds_bytes8<(U < 7 ? 8 + 16 * U : 128)>(row, 8 * (kg & 1), a, b);
        const uint32_t sh = 4u * (uint32_t)(kg >> 1);
        a = iq4_table_bytes((a >> sh) & 0x0F0F0F0Fu);
        b = iq4_table_bytes((b >> sh) & 0x0F0F0F0Fu);
    }
    template <int U> static QLIN_INL float scale(const Hdr &h, int) {
        const uint32_t ls = ((h.lo >> (4 * U)) & 15u) | (((h.hi >> (2 * U)) & 3u) << 4);
        return h.d * (float)((int)ls - 32);
    }
    template <int U> static QLIN_INL float minimum(const Hdr &, int) { return 0.0f; }
};
/* the grid formats look their magnitudes up in a table that the workgroup stages in LDS */
struct TIQ3S {
    static constexpr int kBlock = 110, kPieces = 7, kOffset = 128, kTable = 512, kReady = 0, kBase = 0, kShare = 1, kUnrounded = 4;
    static constexpr bool kSmall = false, kHasMin = false, kGroup16 = false;
    static QLIN_INL const uint32_t *table() { return qlin_iq3s_grid; }
    static QLIN_INL uint32_t piece_src(uint32_t p) { return p < 6 ? 16u * p : 94u; }
    struct Hdr { float d; uint32_t sc; };
    static QLIN_INL Hdr header(const uint8_t *row, int) { return Hdr{half_bits_fast(lds_u16(row)), lds_u32(row + 108)}; }
    template <int U> static QLIN_INL void codes(const uint8_t *row, int kg, const uint32_t *t, uint32_t &a, uint32_t &b) {
        const uint32_t ix = lds_u16(row + 2 + 8 * U + 2 * kg), qh = (uint32_t)row[66 + U] >> (2 * kg);
        const uint32_t sg = row[(U < 5 ? 74 + 4 * U : 76 + 4 * U) + kg];
        a = with_signs(t[(ix & 255u) | ((qh & 1u) << 8)], mask_bytes(sg));
        b = with_signs(t[(ix >> 8) | ((qh & 2u) << 7)], mask_bytes(sg >> 4));
    }
    template <int U> static QLIN_INL float scale(const Hdr &h, int) { return h.d * (float)(1u + 2u * ((h.sc >> (4 * U)) & 15u)); }
    template <int U> static QLIN_INL float minimum(const Hdr &, int) { return 0.0f; }
};
struct TIQ2XXS {
    static constexpr int kBlock = 66, kPieces = 5, kOffset = 128, kTable = 512, kReady = 0, kBase = 0, kShare = 1, kUnrounded = 4;
    static constexpr bool kSmall = false, kHasMin = false, kGroup16 = false;
    static QLIN_INL const uint32_t *table() { return reinterpret_cast<const uint32_t *>(qlin_iq2xxs_grid); }
    static QLIN_INL uint32_t piece_src(uint32_t p) { return p < 4 ? 16u * p : 50u; }
    struct Hdr { float d; const uint8_t *row; };
    static QLIN_INL Hdr header(const uint8_t *row, int) { return Hdr{half_bits_fast(lds_u16(row)) * 0.25f, row}; }
    static constexpr int at(int u) { return u < 7 ? 2 + 8 * u : 72; } /* index bytes | signs and scale */
    template <int U> static QLIN_INL void codes(const uint8_t *row, int kg, const uint32_t *t, uint32_t &a, uint32_t &b) {
        const uint32_t ix = row[at(U) + kg];
        const uint32_t i7 = ((lds_u16(row + at(U) + 4) | (lds_u16(row + at(U) + 6) << 16)) >> (7 * kg)) & 127u;
        const uint32_t sg = iq_sign_byte(i7);
        a = with_signs(t[2 * ix], mask_bytes(sg));
        b = with_signs(t[2 * ix + 1], mask_bytes(sg >> 4));
    }
    template <int U> static QLIN_INL float scale(const Hdr &h, int) { return h.d * (0.5f + (float)(h.row[at(U) + 7] >> 4)); }
    template <int U> static QLIN_INL float minimum(const Hdr &, int) { return 0.0f; }
};

/* compile-time loop over 0 .. N - 1 */
template <class Fn, int... I> QLIN_INL void each_impl(Fn &&fn, std::integer_sequence<int, I...>) { (fn(std::integral_constant<int, I>{}), ...); }
template <int N, class Fn> QLIN_INL void each(Fn &&fn) { each_impl(fn, std::make_integer_sequence<int, N>{}); }

/* kq::dma16 in inline asm: around the builtin the compiler waits for every outstanding request before an LDS read that it
 * cannot tell apart from its target (52 waits more in the instances of Q4_K and Q5_K), where these kernels count their own */
QLIN_INL void request16(uint32_t lds_at, uint32_t voff, __amdgpu_buffer_rsrc_t rsrc, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds_at)), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory");
}

}  // namespace
}  // namespace qlin
#endif

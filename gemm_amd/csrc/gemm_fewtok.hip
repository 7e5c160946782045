/*
 * gemm_fewtok.hip - which products the few-token kernel (gemm_fewtok.h) takes, and its launch by format.
 */
#include "qlin_internal.h"

namespace qlin {

bool fewtok_has(uint32_t type) {
    switch (type) {
    case T_Q4_K: case T_Q5_K: case T_Q6_K: case T_Q2_K: case T_Q3_K: case T_Q8_0: case T_Q4_0: case T_IQ4_NL: case T_IQ4_XS:
    case T_IQ3_S: case T_IQ2_XXS: return true;
    default: return false;
    }
}

int fewtok_unrounded(uint32_t type) {
    switch (type) {
    case T_Q4_K: return 32;
    case T_Q5_K: case T_Q6_K: case T_Q2_K: case T_Q3_K: case T_Q8_0: return 24;
    default: return 4;
    }
}

/* Unrounded tokens always. With rounded weights the small-tile kernel, whose workgroup takes 64 rows, computes the same;
 * it is the faster one where this kernel's workgroups no longer run in one go (us, this kernel / small tiles):
 *   49 to 64 tokens, more than 512 row tiles of rows below 4096 elements: 64 tokens 8192 x 2048 Q4_K 7.1 / 10.7, but 8704 x
 *     2048 11.9 / 10.9, 9216 x 2560 Q5_K 15.8 / 13.3; longer rows are even or better here (16384 x 4096 Q4_K 20.0 / 21.0). Not
 *     Q8_0, whose decode costs the tile kernel more (9216 x 2048 14.2 / 17.1), and not from 1593 row tiles on, where 200
 *     large tiles would be chosen, a quarter full (32000 x 2048 Q4_K 26 / 30; 1024 elements from 1200 on, 24576 x 1024 11.1 /
 *     11.8; five to seven super-blocks, a wave for each, from 3000 on, 32000 x 1536 Q4_K 24.2 / 22.4, but 50000 x 1536
 *     31.9 / 36.9)
 *     Rows of 2304 to 4864 elements from 1400 tiles on: the chip takes the small tiles in few enough goes (us, 64 tokens,
 *     this kernel / small tiles, 26624 x 2560 Q4_K 33 / 25, 28672 x 4096 42.8 / 38.4, Q6_K 53.9 / 48.7; at 1280 tiles even;
 *     8192 elements even everywhere)
 *   65 to 128 tokens, more than 320: 80 tokens Q4_K 4096 x 4096 9.2 / 17.3, 5120 x 4096 11.2 / 17.6, but 77 tokens
 *     13824 x 2560 19.6 / 16.8. (A tensor alone gains up to 512: 80 tokens Q4_K 8192 x 4096 12.7 / 20.3. Pairs of such tensors, gate
 *     and up, which share a launch and whose results are those of a call each, lose: 2 x 6144 x 2560 at 96 18.7 / 13.8.) Past 96 tokens,
 *     rows below 2048 (Q8_0: 4096) elements: 256 (128 tokens 5120 x 1024 Q4_K 9.5 / 7.9)
 *   rows so short that one or two waves do all of K: 256 elements from 49 tokens on (64 tokens 4096 x 256 5.6 / 5.1), 512
 *     from 97 on (128 tokens 4096 x 512 Q4_K 7.0 / 6.1; with more than 256 row tiles from 81 on)
 * The grid formats, which have no tile kernel, end at 64 (IQ3_S 13824 x 2560 at 64 tokens 23 us, decode + dense product
 * 63): beyond, their product is that of a cached bf16 copy bit for bit. */
bool fewtok_takes(uint32_t type, int n_rows, int n_cols, int n_tok, int ldx) {
    if (!fewtok_has(type) || n_cols % 256 != 0 || n_tok > 128 || ldx >= (1 << 22)) return false;
    if (n_tok <= fewtok_unrounded(type)) return true;
    if (!gemm_kq_wave4_covers(type)) return n_tok <= 64;
    const int tiles = n_rows / 16 + (n_rows % 16 != 0), n_sb = n_cols / 256;
    if (n_tok <= 48) return true;
    if (n_sb == 1) return false;
    if (n_tok <= 64) {
        if (tiles <= 512 || type == T_Q8_0) return true;
        if (n_sb > 8) return n_sb >= 20 || (n_sb >= 16 && tiles < 1400);
        return tiles >= (n_sb < 4 || n_sb > 7 ? 1593 : n_sb == 4 ? 1200 : 3000);
    }
    if (n_tok <= 80) return tiles <= 320;
    if (n_tok <= 96) return tiles <= (n_sb == 2 ? 256 : 320);
    if (type == T_Q8_0) return tiles <= (n_sb < 16 ? 256 : 320);
    return n_sb > 2 && tiles <= (n_sb < 8 ? 256 : 320);
}

/* Tokens that go one by one through the matvec instead (whose bar is the same, exact weights): the formats that multiply up
 * to four tokens unrounded, where the tensor is so large that the matvec's own launch is cheaper by size (us, this kernel /
 * widening x and a matvec per token; long: rows of 12288 elements and more, of which a wave here walks an eighth alone).
 *   one token   IQ4_NL, IQ4_XS from 32 M weights (4096 x 4096 5.3 / 7.0, 9216 x 4096 12.4 / 9.6, 14336 x 4096 13.1 / 11.0) and
 *               long rows (2048 x 14336 12.5 / 11.3); IQ3_S from 16 M and 4608 rows (5120 x 2048 6.6 / 7.2, 9216 x 4096 15.3 / 11.1)
 *               and long rows; Q4_0 above 64 M (9216 x 8192 13.7 / 13.2, 28672 x 4096 15.1 / 14.1); IQ2_XXS, whose table
 *               every workgroup fills, from 3072 elements or 4608 rows (4096 x 2048 6.0 / 6.7, 4096 x 4096 8.9 / 7.0,
 *               28672 x 4096 36.3 / 13.1)
 *   two         IQ2_XXS above 32 M (4096 x 4096 8.7 / 10.9, 9216 x 4096 20.3 / 14.6) and long rows (4096 x 14336 22.1 / 17.8)
 *   three       IQ2_XXS above 64 M and 8192 rows (8192 x 8192 21.5 / 25.6, 9216 x 14336 60.2 / 47.5)
 * Rows of up to 1024 elements stay (28672 x 1024 IQ4_NL 8.3 / 14.5). */
bool fewtok_leaves_to_matvec(uint32_t type, int n_rows, int n_cols, int n_tok) {
    const long long weights = (long long)n_rows * n_cols, M = 1 << 20;
    if (n_cols <= 1024) return false;
    const bool long_rows = n_cols >= 12288;
    switch (type) {
    case T_IQ4_NL: case T_IQ4_XS: return n_tok == 1 && (long_rows || weights >= 32 * M);
    case T_IQ3_S: return n_tok == 1 && (long_rows || (weights > 16 * M && n_rows >= 4608));
    case T_Q4_0: return n_tok == 1 && weights > 64 * M;
    case T_IQ2_XXS:
        return (n_tok == 1 && (n_cols >= 3072 || n_rows >= 4608)) || (n_tok == 2 && (long_rows || weights > 32 * M)) ||
               (n_tok == 3 && weights > 64 * M && n_rows > 8192);
    default: return false;
    }
}

hipError_t launch_gemm_fewtok(uint32_t type, const FewtokCall &c) {
    switch (type) {
    case T_Q4_K: return fewtok_q4k(c);
    case T_Q5_K: return fewtok_q5k(c);
    case T_Q6_K: return fewtok_q6k(c);
    case T_Q2_K: return fewtok_q2k(c);
    case T_Q3_K: return fewtok_q3k(c);
    case T_Q8_0: return fewtok_q8_0(c);
    case T_Q4_0: return fewtok_q4_0(c);
    case T_IQ4_NL: return fewtok_iq4nl(c);
    case T_IQ4_XS: return fewtok_iq4xs(c);
    case T_IQ3_S: return fewtok_iq3s(c);
    case T_IQ2_XXS: return fewtok_iq2xxs(c);
    default: return hipErrorInvalidValue;
    }
}

/* rows of X so far apart that the kernel's 32-bit offsets do not hold them: the tokens one by one */
hipError_t launch_gemm_fewtok_one_by_one(uint32_t type, const FewtokCall &c) {
    for (int t = 0; t < c.n_tok; t++) {
        float *Y[3];
        for (int i = 0; i < c.n_mat; i++) Y[i] = c.Y[i] + (size_t)t * c.ldy[i];
        FewtokCall one = c;
        one.X = c.X + (size_t)t * c.ldx;
        one.Y = Y;
        one.n_tok = 1;
        one.ldx = c.n_cols;
        if (const hipError_t e = launch_gemm_fewtok(type, one); e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace qlin

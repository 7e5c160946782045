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

/* Up to 64 tokens always; up to 128 while there are few row tiles (320 of 16 rows): the kernel reads the activations once
 * per 16 rows then, where the small-tile kernel, whose workgroup takes 64 rows, fills the chip from about 14000 rows on
 * (us, this kernel / small tiles, 77 tokens: Q4_K 3840 x 2560 8.6 / 12.5, 4096 x 4096 10.2 / 17.5, 2560 x 6912
 * 13.6 / 25.8, but 13824 x 2560 19.6 / 16.8; Q6_K 9.5 / 16.3, 12.9 / 26.5, 18 / 41, 24 / 21; 128 tokens Q4_K 11.4 / 13,
 * 15.2 / 18, 19.9 / 26.6, 40 / 17). The grid formats, which have no tile kernel, end at 64 (IQ3_S 13824 x 2560 at 64
 * tokens 23 us, decode + dense product 63): beyond, their product is that of a cached bf16 copy bit for bit. */
bool fewtok_takes(uint32_t type, int n_rows, int n_cols, int n_tok, int ldx) {
    if (!fewtok_has(type) || n_cols % 256 != 0 || n_tok > 128 || ldx >= (1 << 22)) return false;
    return n_tok <= 64 || ((n_rows + 15) / 16 <= 320 && gemm_kq_wave4_covers(type));
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

/*
 * gemv_grid.hip - batch-1 matvec for rows of more than 4096 elements (and, where it measured faster, of 2048 to
 * 4096) on gfx950, for the codebook ("grid") formats
 * IQ1_S, IQ1_M, IQ2_XXS, IQ2_XS, IQ2_S, IQ3_XXS and IQ3_S and for Q6_K, Q5_K, Q8_0, Q4_0, Q4_1, Q5_0, Q5_1, IQ4_NL, IQ4_XS, MXFP4, NVFP4, TQ1_0, TQ2_0, Q1_0, Q2_K and Q3_K: the inner products run on the 8-bit
 * integer matrix instruction; the grid formats look their codebook and sign masks up in LDS, the others build their
 * codes in registers and read the x operand from LDS for every item.
 *
 * y[r] = sum over 16- or 32-element groups of scale(r, group) * (codes . x_group) (- offset * sum of x_group), with
 * the codes of common/ggml_dequant.h:2793-2816, :2916-2940, :3022-3058 (grid formats), :1653-1687 (Q6_K),
 * :1620-1651 (Q5_K), :1479-1489 (Q8_0), :2850-2862 (Q4_0), :2942-2954 (IQ4_NL), :2956-2973 (IQ4_XS),
 * :1505-1534 (Q2_K), :1536-1580 (Q3_K), :2864-2915 (Q4_1, Q5_0, Q5_1), :2818-2830 (MXFP4) and
 * :2832-2848 (NVFP4), :3161-3176 (TQ2_0), :2975-3020 (IQ2_XS, IQ2_S), :1491-1503 (Q1_0),
 * :3062-3126 (IQ1_S, IQ1_M), :3127-3160 (TQ1_0).
 *
 *  1. x -> fixed point per 32-element group, three signed base-256 digits (the Q4_K matvec, gemv_q4k.hip,
 *     keeps four): X = rint(x * 2^(22-e)), e the exponent of the group's largest |x|; the error is at most
 *     2^-23 of that largest |x| per element.
 *  2. v_mfma_i32_16x16x64_i8: 16 weight rows (B operand: one code byte per element) against 16 "x rows"
 *     (A operand). Lane group g = lane/16 of a wave owns 64 elements of the wave's super-block, 16 per
 *     instruction s = 0..3 (F::elem0(g, s): elements [64 g + 16 s, +16) for most formats; Q6_K takes the 16
 *     elements of one scale). The A operand is block-diagonal to match: x row 4g + digit (digit 0..2; row 4g+3
 *     stays zero) holds that digit plane of lane group g's 16 elements at lane group g's k positions and zeros
 *     elsewhere, so result register v of lane (n, g) is digit plane v of lane group g's elements for weight
 *     row n. Which k position carries which element is free as long as both operands agree.
 *  3. Wave w of the 16-wave workgroup owns super-block w (w+16, ...) of every row of the workgroup, prepares
 *     only its own 256 elements of x, and reads its bytes of a block straight from HBM: lane (n, g) takes
 *     the bytes of its 64 elements of row n (blocks of the grid formats and Q6_K are 2-byte aligned:
 *     dword-aligned loads, a 16-bit tail and a funnel shift). The waves' shares of a row meet in LDS at the end.
 *
 * What a lane of a grid format spends per element is one table lookup per 4-8 elements for the grid, one per 8
 * for the sign mask, two vector instructions per 4 elements to apply the signs and a sixteenth of a matrix
 * instruction; the v_dot4 formulation (gemv_int.hip) spends an instruction per element on the products alone.
 *
 * A non-finite x makes every output NaN (the fixed-point form cannot carry Inf).
 */
#include "gemv_grid_formats.h"

namespace qlin {

namespace {

constexpr int kWaves = 16;        /* wavefronts per workgroup */
constexpr int kMaxKc = 4;         /* super-blocks per wave: K <= 16384 */
constexpr int kMaxRowsPerWg = 640; /* local rows (both matrices of a gate+up pair): 40 KB of partial sums, 63 KB in all */

}  // namespace

/* MOE = 0: the matvec. MOE = 1, 2: a token's routed experts (the reference's MoE block for a token,
 * common/transformer.h:4045-4131) on the same kernel, as moe1_q4k_kernel (gemv_q4k.hip) does for Q4_K:
 *   1  gate + up + SiLU of pair blockIdx.y = token * top_k + k: the job's two matrices moved to expert idx[pair], the
 *      result to h[pair], x the token's bf16 activations;
 *   2  down of token blockIdx.y: one matvec over a row of top_k * n_ff elements whose super-blocks sit in different
 *      experts, x = h scaled by the routing weight of the super-block's expert (nothing for an index out of range). */
struct MoeArgs {
    const int32_t *idx;
    const float *wts;
    int top_k, n_expert, sb_per_expert;
    int ldx; /* elements between two tokens' activations (MOE = 1) or rows of h (MOE = 2) */
    size_t expert_bytes;
    int sb0; /* MOE = 2: the launch covers super-blocks sb0, sb0 + 1, ... of the token's row (x points at sb0's) */
};

template <uint32_t T, int NKC, int MOE = 0>
__global__ void __launch_bounds__(kWaves * 64)
gemv_grid_kernel(const JobView job_in, const float *__restrict__ x, int n_sb, int rows_per_wg, size_t row_bytes, const MoeArgs moe,
                 int lone_ahead) {
    using F = GridFmt<T>;
    JobView job = job_in;
    const int32_t *idx = moe.idx;
    const float *wts = moe.wts;
    if (MOE == 1) {
        const int pair = blockIdx.y, e = idx[pair];
        if (e < 0 || e >= moe.n_expert) return; /* uniform over the workgroup */
        job.W0 += (size_t)e * moe.expert_bytes;
        job.W1 += (size_t)e * moe.expert_bytes;
        job.y0 += (size_t)pair * job.n0;
        x = reinterpret_cast<const float *>(reinterpret_cast<const uint16_t *>(x) + (size_t)(pair / moe.top_k) * moe.ldx);
    } else if (MOE == 2) {
        idx += (size_t)blockIdx.y * moe.top_k;
        wts += (size_t)blockIdx.y * moe.top_k;
        x += (size_t)blockIdx.y * moe.ldx;
        job.y0 += (size_t)blockIdx.y * job.n0;
    }
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, g = lane >> 4;

    /* a workgroup owns rows_per_wg rows: of the concatenated matrices, or, where two results are
     * combined (mode 2), the same rows of both matrices (local rows: first matrix, then second) */
    const bool paired = job.mode == 2;
    const int n_mats_here = paired ? 2 : 1;
    const int n_rows = paired ? job.n0 : job.n0 + job.n1 + job.n2;
    const int row0 = blockIdx.x * rows_per_wg;
    int rows_here = n_rows - row0;
    if (rows_here > rows_per_wg) rows_here = rows_per_wg;
    const int n_lrows = rows_here * n_mats_here;
    const int n_rg = (n_lrows + 15) >> 4;
    const int n_kc = wv < n_sb ? ((n_sb - wv + 15) >> 4) : 0; /* this wave's super-blocks: wv, wv+16, ... */

    /* LDS: x scratch per wave, the grid and the sign masks at addresses the compiler knows (a lookup is then a
     * shift, a mask and a read with a constant offset); the partial sums [rows][kWaves] behind them */
    __shared__ __attribute__((aligned(16))) uint8_t xs_all[kWaves * kXScratch];
    __shared__ __attribute__((aligned(16))) uint32_t grid_lds[F::kGridBytes > 0 ? F::kGridBytes / 4 : 4];
    __shared__ __attribute__((aligned(16))) uint2 sign_lds[F::kGridBytes > 0 ? 256 + 128 : 2];
    uint8_t *xs = xs_all + wv * kXScratch;
    float *partial = reinterpret_cast<float *>(lds);
    const Tables tab = {grid_lds, sign_lds, sign_lds + (F::kGridBytes > 0 ? 256 : 0)};

    const bool one_matrix = !paired && job.n1 == 0 && job.n2 == 0; /* a scalar test: no search by row then */
    auto locate = [&](int lr, const uint8_t *&Wm, float *&ym, int &r) {
        if (one_matrix) {
            Wm = job.W0;
            ym = job.y0;
            r = row0 + lr;
        } else if (paired) {
            const bool second = lr >= rows_here;
            Wm = second ? job.W1 : job.W0;
            ym = job.y0;
            r = row0 + (second ? lr - rows_here : lr);
        } else {
            job_locate(job, row0 + lr, Wm, ym, r);
        }
    };
    auto row_pointer = [&](int rg) { /* this lane's row of row group rg (rows past the end: the last one, never stored) */
        int lr = 16 * rg + n;
        if (lr >= n_lrows) lr = n_lrows - 1;
        /* by branches: a choice between the three matrix arguments by selects becomes a load from the argument
         * block, with a full wait, in front of every weight request */
        const uint8_t *Wm;
        float *ym;
        int r;
        locate(lr, Wm, ym, r);
        return Wm + (size_t)r * row_bytes;
    };
    /* where in its row the wave's super-block kc sits (MOE = 2: in which expert's copy of the row, too; an index
     * out of range reads expert 0 and gets zeros for x) */
    auto sb_off = [&](int kc) {
        const int s = wv + 16 * kc;
        if (MOE == 2) {
            const int v = moe.sb0 + s, j = v / moe.sb_per_expert, e = idx[j];
            const bool valid = e >= 0 && e < moe.n_expert;
            return (size_t)(valid ? e : 0) * moe.expert_bytes + (size_t)(v - j * moe.sb_per_expert) * F::kBlock;
        }
        return (size_t)s * F::kBlock;
    };
    auto moe_x = [&](v4f v, int kc) { /* MOE = 2: the routing weight of the super-block's expert goes onto x */
        if (MOE == 2) {
            const int j = (moe.sb0 + wv + 16 * kc) / moe.sb_per_expert, e = idx[j];
            const float wj = wts[j];
            const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
            v = (e >= 0 && e < moe.n_expert) ? v * wj : zero;
        }
        return v;
    };

    /* the wave's first super-block of x; later ones are fetched where they are used */
    auto load_x = [&](int kc) {
        if (MOE == 1) { /* bf16 activations */
            const uint2 b = *reinterpret_cast<const uint2 *>(reinterpret_cast<const uint16_t *>(x) + (size_t)(16 * kc + wv) * 256 + 4 * lane);
            const v4f v = {__uint_as_float(b.x << 16), __uint_as_float(b.x & 0xFFFF0000u), __uint_as_float(b.y << 16),
                           __uint_as_float(b.y & 0xFFFF0000u)};
            return v;
        }
        return *reinterpret_cast<const v4f *>(x + (size_t)(16 * kc + wv) * 256 + 4 * lane);
    };
    v4f xq = {0.0f, 0.0f, 0.0f, 0.0f};
    if (n_kc > 0) xq = load_x(0);

    auto store_partial = [&](int rg, float v, bool add) { /* the four lane groups hold four shares of the same row */
        v = sum_lane_groups(v);
        const int lr = 16 * rg + n;
        if (lane < 16 && lr < n_lrows) {
            float *p = partial + lr * kWaves + wv;
            *p = add ? *p + v : v;
        }
    };

    /* every piece of a block that a lane reads starts F::kPiece (mod 4) bytes into the block: the funnel shift of its bytes */
    auto shift_of = [](const uint8_t *blk) { return (((uint32_t)(uintptr_t)blk + (uint32_t)F::kPiece) & 2u) * 8u; };

    /* the first blocks are requested before the tables are built and x is prepared: the wave's first two
     * super-blocks of a lone row group (long rows), else its first super-block of the first row groups */
    const bool long_rows = NKC > 1 && n_rg < 2 && lone_ahead;
    /* row groups of a super-block column in flight per wave: with sixteen waves per compute unit one is enough, and
     * two or four measured slower for every format (IQ2_XXS 8192 x 28672: 38.8 us with four, 29.6 with one) */
    constexpr int D = 1;
    constexpr int NF = (NKC > 1 && D < 2) ? 2 : D; /* the long-rows path keeps two */
    typename F::Raw first[NF];
    uint32_t first_sh[NF];
    if (n_kc > 0) {
#pragma unroll
        for (int q = 0; q < NF; q++) {
            if (long_rows ? q >= 2 : q >= D) break;
            const uint8_t *blk = long_rows ? row_pointer(0) + sb_off(q < n_kc ? q : 0) : row_pointer(q < n_rg ? q : 0) + sb_off(0);
            first[q] = F::load(blk, g);
            first_sh[q] = shift_of(blk);
        }
    }
    if (lane < 32) reinterpret_cast<uint32_t *>(xs + 768)[lane] = 0u; /* what the dead lanes of the x operand read */
    for (int t = threadIdx.x; t < F::kGridBytes / 4; t += kWaves * 64) grid_lds[t] = F::grid_src()[t];
    if (F::kGridBytes > 0 && threadIdx.x < 384) {
        const uint32_t i = threadIdx.x, sb = i < 256 ? i : iq_sign_byte(i - 256);
        sign_lds[i] = make_uint2(spread4(sb) * 0xFFu, spread4(sb >> 4) * 0xFFu);
    }
    __syncthreads();

    XOperand xo;
    if (n_kc == 0) { /* a wave without a super-block (K < 4096) contributes zeros */
        for (int rg = 0; rg < n_rg; rg++) store_partial(rg, 0.0f, false);
    } else if (long_rows) {
        /* one row group: the wave's super-blocks of it, two requested ahead of the one being multiplied */
        float acc = 0.0f;
        const uint8_t *blk0 = row_pointer(0);
#pragma unroll
        for (int kc = 0; kc < NKC; kc++) {
            if (kc < n_kc) {
                prepare_x<F>(moe_x(xq, kc), xs, lane, xo);
                if (kc + 1 < n_kc) xq = load_x(kc + 1); /* on its way while this super-block is multiplied */
                acc += F::item(xo, first[kc & 1], first_sh[kc & 1], tab, g);
            }
            if (kc + 2 < n_kc) { /* into the registers just used */
                const uint8_t *blk = blk0 + sb_off(kc + 2);
                first[kc & 1] = F::load(blk, g);
                first_sh[kc & 1] = shift_of(blk);
            }
            __builtin_amdgcn_sched_barrier(0); /* one super-block at a time: interleaving them costs registers */
        }
        store_partial(0, acc, false);
    } else {
        for (int kc = 0; kc < n_kc; kc++) {
            v4f v = xq;
            if (kc > 0) v = load_x(kc);
            prepare_x<F>(moe_x(v, kc), xs, lane, xo);
            /* D row groups in flight: a group's registers are refilled as soon as it has been multiplied */
            if (kc > 0) {
#pragma unroll
                for (int q = 0; q < D; q++) {
                    const uint8_t *blk = row_pointer(q < n_rg ? q : 0) + sb_off(kc);
                    first[q] = F::load(blk, g);
                    first_sh[q] = shift_of(blk);
                }
            }
            for (int rg = 0; rg < n_rg; rg += D) {
#pragma unroll
                for (int q = 0; q < D; q++) {
                    if (rg + q < n_rg) store_partial(rg + q, F::item(xo, first[q], first_sh[q], tab, g), kc > 0);
                    if (rg + q + D < n_rg) {
                        const uint8_t *blk = row_pointer(rg + q + D) + sb_off(kc);
                        first[q] = F::load(blk, g);
                        first_sh[q] = shift_of(blk);
                    }
                }
            }
        }
    }
    __syncthreads();

    /* sum the waves' shares of each row and store */
    auto row_total = [&](int lr) {
        const float4 *p = reinterpret_cast<const float4 *>(partial + lr * kWaves);
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < kWaves / 4; k++) {
            const float4 v = p[k];
            s += (v.x + v.y) + (v.z + v.w);
        }
        return s;
    };
    if (paired) {
        for (int lr = threadIdx.x; lr < rows_here; lr += kWaves * 64)
            job.y0[row0 + lr] = silu_times(row_total(lr), row_total(rows_here + lr));
    } else {
        for (int lr = threadIdx.x; lr < n_lrows; lr += kWaves * 64) {
            const uint8_t *Wm;
            float *ym;
            int r;
            locate(lr, Wm, ym, r);
            const float s = row_total(lr);
            ym[r] = job.mode == 1 ? ym[r] + s : s;
        }
    }
}

namespace {

/* Rows of up to 4096 elements, one super-block per wave and one row group per wave in flight (two and four measured
 * slower for every format): where this kernel measured faster than the v_dot4 kernel (gemv_int.hip) over 1024 to
 * 151936 rows of 2048 to 4096 elements. 14336 x 4096, us: IQ4_NL 13.3 -> 10.3, IQ4_XS 12.8 -> 10.6, Q4_0 10.4 -> 8.7,
 * Q2_K 10.0 -> 8.0, IQ2_XXS 11.0 -> 9.0, Q3_K 13.8 -> 12.8, IQ3_S 13.3 -> 12.5, Q5_K 12.8 -> 12.5; 151936 x 4096:
 * IQ2_XXS 82 -> 51, Q2_K 74 -> 54, IQ4_NL 100 -> 79, but Q5_K 90 -> 112, Q6_K 103 -> 141, Q8_0 103 -> 132 (and
 * Q6_K, Q8_0 no faster at 14336 rows or below 4096: they come here for 4096 to 8192 rows only, 4096 x 4096:
 * Q8_0 6.9 -> 6.0, Q6_K 7.1 -> 6.8; 8192 x 4096: 9.3 -> 8.7, 11.1 -> 10.0). With fewer than eight super-blocks more
 * than half of the waves would have nothing to do. Two workgroups per compute unit (the instances of 64 registers
 * or fewer would fit) measured slower for every format. */
bool short_rows_pay(uint32_t type, int n_sb, int n_rows) {
    if (n_sb < 8) return false;
    switch (type) {
    case T_IQ4_NL: case T_IQ4_XS: case T_Q4_0: case T_Q2_K: case T_IQ2_XXS: case T_IQ3_XXS: case T_IQ3_S: return true;
    case T_IQ2_XS: return true; /* 14336: 12.0 -> 10.3, 151936: 90 -> 64; IQ2_S (12.7 against 13.0, 95 against 101) stays */
    case T_TQ1_0: return true; /* 14336: 31.7 -> 15.7, 151936: 306 -> 107 */
    case T_Q1_0: case T_IQ1_S: case T_IQ1_M: return true; /* 14336: 10.9 -> 7.5, 13.9 -> 10.5, 16.0 -> 10.7; 151936: 89 -> 44, 111 -> 75, 135 -> 67 */
    case T_MXFP4: case T_NVFP4: case T_TQ2_0: return true; /* 14336: 13.4 -> 11.2, 17.9 -> 12.5, 11.7 -> 7.4; 151936: 98 -> 74, 162 -> 88, 93 -> 43 */
    case T_Q3_K: return n_rows >= 4096;
    case T_Q5_K: return n_rows <= 16384;
    case T_Q4_1: case T_Q5_0: case T_Q5_1: return n_rows <= 32768; /* 14336: 10.5 -> 9.3, 12.1 -> 10.0, 12.0 -> 10.3; 151936: 67 -> 88 */
    case T_Q6_K: case T_Q8_0: return n_rows >= 4096 && n_rows <= 8192;
    default: return false;
    }
}

template <uint32_t T>
bool grid_typed(const GemvJob &job, const float *x, int n_cols, int n_cu, hipStream_t stream, hipError_t *err,
                size_t row_stride) {
    const int n_sb = n_cols / 256;
    const bool short_rows = n_sb <= 16;
    if (n_cols % 256 != 0 || n_sb > 16 * kMaxKc || ((uintptr_t)x & 15)) return false;
    /* what the format's loads want of the addresses (block sizes are even; the formats whose 256 elements fill a
     * multiple of 4 or 16 bytes read whole dwords or 16-byte groups) */
    for (int m = 0; m < job.n_mat; m++)
        if ((uintptr_t)job.W[m] % GridFmt<T>::kAlign) return false;
    if (row_stride % GridFmt<T>::kAlign) return false;
    const int n_mats_here = job.mode == kSiluMul ? 2 : 1;
    const int n_rows = job.mode == kSiluMul ? job.n_rows[0] : job.total_rows();
    if (n_rows == 0) return false;
    if (short_rows && !short_rows_pay(T, n_sb, n_rows * n_mats_here)) return false;
    /* one workgroup per compute unit where its partial sums fit in LDS (with the lookup tables: in 128 rows' worth,
     * more measured slower for those formats), else so many equal rounds of workgroups that they do (Q2_K 151936 x
     * 4096: 55 -> 48 us, 49152 rows 22.3 -> 17.4) */
    constexpr int max_rows = GridFmt<T>::kGridBytes > 0 ? 128 : kMaxRowsPerWg;
    const int rows_per_cu = (n_rows + n_cu - 1) / n_cu;
    const int rounds = (rows_per_cu * n_mats_here + max_rows - 1) / max_rows;
    int rows_per_wg = (n_rows + n_cu * rounds - 1) / (n_cu * rounds);
    /* long rows: whole row groups, a matrix instruction wants 16 rows anyway; short ones: a workgroup on every
     * compute unit counts for more (14336 rows: 56 each) */
    if (!short_rows) rows_per_wg = (rows_per_wg + 15) & ~15;
    if (rows_per_wg * n_mats_here > max_rows) rows_per_wg = max_rows / n_mats_here;
    const int grid = (n_rows + rows_per_wg - 1) / rows_per_wg;
    const size_t lds_bytes = (size_t)rows_per_wg * n_mats_here * kWaves * 4; /* the partial sums; the rest is static */
    const JobView view = job_view(job);
    const size_t pitch = row_stride ? row_stride : (size_t)n_sb * GridFmt<T>::kBlock;
    const MoeArgs none = {nullptr, nullptr, 0, 0, 0, 0, 0, 0};
    if (short_rows)
        hipLaunchKernelGGL((gemv_grid_kernel<T, 1>), dim3(grid), dim3(kWaves * 64), lds_bytes, stream, view, x, n_sb, rows_per_wg, pitch, none, 1);
    else
        {
        /* a lone row group per workgroup: two super-blocks requested ahead, except for the two formats with the most
         * loads per item where every compute unit has a workgroup - there one super-block at a time measured faster
         * (Q6_K 4096 x 8192: 11.3 -> 9.9 us, 4096 x 14336: 14.9 -> 14.6; IQ3_S 10.7 -> 9.9, 13.5 -> 13.0) */
        const bool one_at_a_time = (T == T_Q6_K || T == T_IQ3_S) && grid >= n_cu;
        hipLaunchKernelGGL((gemv_grid_kernel<T, kMaxKc>), dim3(grid), dim3(kWaves * 64), lds_bytes, stream, view, x, n_sb, rows_per_wg, pitch, none,
                           one_at_a_time ? 0 : 1);
    }
    *err = hipGetLastError();
    return true;
}

}  // namespace

namespace {

template <uint32_t T>
bool moe1_up_typed(const void *gate, const void *up, const uint16_t *X, const int32_t *idx, float *h, int n_tok, int top_k,
                   int n_embd, int n_ff, int n_expert, int n_cu, hipStream_t stream, bool dry, hipError_t *err) {
    using F = GridFmt<T>;
    const int n_sb = n_embd / 256;
    const size_t row_bytes = (size_t)n_sb * F::kBlock, expert_bytes = (size_t)n_ff * row_bytes;
    if (n_embd % 256 != 0 || n_sb > 16 * kMaxKc || n_ff < 1 || top_k < 1 || n_tok < 1) return false;
    if (((uintptr_t)gate | (uintptr_t)up | expert_bytes) % F::kAlign || ((uintptr_t)X & 7) || ((uintptr_t)h & 15)) return false;
    if (dry) return true;
    constexpr int max_rows = F::kGridBytes > 0 ? 128 : kMaxRowsPerWg;
    const int n_pairs = n_tok * top_k;
    const int tiles = n_cu / n_pairs > 0 ? n_cu / n_pairs : 1;
    int rows_per_wg = (n_ff + tiles - 1) / tiles;
    if (2 * rows_per_wg > max_rows) rows_per_wg = max_rows / 2;
    GemvJob job = {};
    job.W[0] = gate; job.W[1] = up; job.y[0] = h;
    job.n_rows[0] = job.n_rows[1] = n_ff;
    job.n_mat = 2;
    job.mode = kSiluMul;
    const MoeArgs moe = {idx, nullptr, top_k, n_expert, n_sb, n_embd, expert_bytes, 0};
    const dim3 grid((n_ff + rows_per_wg - 1) / rows_per_wg, n_pairs);
    const size_t lds_bytes = (size_t)2 * rows_per_wg * kWaves * 4;
    const float *x = reinterpret_cast<const float *>(X);
    if (n_sb <= 16)
        hipLaunchKernelGGL((gemv_grid_kernel<T, 1, 1>), grid, dim3(kWaves * 64), lds_bytes, stream, job_view(job), x, n_sb, rows_per_wg, row_bytes, moe, 1);
    else
        hipLaunchKernelGGL((gemv_grid_kernel<T, kMaxKc, 1>), grid, dim3(kWaves * 64), lds_bytes, stream, job_view(job), x, n_sb, rows_per_wg, row_bytes, moe, 1);
    *err = hipGetLastError();
    return true;
}

template <uint32_t T>
bool moe1_down_typed(const void *down, const float *h, const int32_t *idx, const float *w, float *out, int n_tok, int top_k,
                     int n_embd, int n_ff, int n_expert, int n_cu, hipStream_t stream, bool dry, hipError_t *err) {
    using F = GridFmt<T>;
    const int sbpe = n_ff / 256, n_sb = top_k * sbpe; /* the row of a token: top_k experts' rows side by side */
    const size_t row_bytes = (size_t)sbpe * F::kBlock, expert_bytes = (size_t)n_embd * row_bytes;
    if (n_ff % 256 != 0 || n_embd < 1 || top_k < 1 || n_tok < 1) return false;
    if (((uintptr_t)down | row_bytes) % F::kAlign || ((uintptr_t)h & 15)) return false;
    if (dry) return true;
    constexpr int max_rows = F::kGridBytes > 0 ? 128 : kMaxRowsPerWg;
    const int tiles = n_cu / n_tok > 0 ? n_cu / n_tok : 1;
    int rows_per_wg = (n_embd + tiles - 1) / tiles;
    if (rows_per_wg > max_rows) rows_per_wg = max_rows;
    const dim3 grid((n_embd + rows_per_wg - 1) / rows_per_wg, n_tok);
    const size_t lds_bytes = (size_t)rows_per_wg * kWaves * 4;
    /* a launch takes 64 super-blocks of the row; a longer row (wide experts) goes in ranges, the later ones adding */
    for (int sb0 = 0; sb0 < n_sb; sb0 += 16 * kMaxKc) {
        const int n_here = n_sb - sb0 < 16 * kMaxKc ? n_sb - sb0 : 16 * kMaxKc;
        GemvJob job = single_job(down, out, n_embd, sb0 == 0 ? kStore : kAdd);
        const MoeArgs moe = {idx, w, top_k, n_expert, sbpe, n_sb * 256, expert_bytes, sb0};
        const float *x = h + (size_t)sb0 * 256;
        if (n_here <= 16)
            hipLaunchKernelGGL((gemv_grid_kernel<T, 1, 2>), grid, dim3(kWaves * 64), lds_bytes, stream, job_view(job), x, n_here, rows_per_wg, row_bytes, moe, 1);
        else
            hipLaunchKernelGGL((gemv_grid_kernel<T, kMaxKc, 2>), grid, dim3(kWaves * 64), lds_bytes, stream, job_view(job), x, n_here, rows_per_wg, row_bytes, moe, 1);
    }
    *err = hipGetLastError();
    return true;
}

}  // namespace

/* every format of this kernel (Q4_K experts take moe1_q4k_kernel, gemv_q4k.hip) */
#define QLIN_MOE1_TYPES(X)                                                                                           \
    X(T_Q6_K) X(T_Q5_K) X(T_Q8_0) X(T_Q4_0) X(T_Q4_1) X(T_Q5_0) X(T_Q5_1) X(T_IQ4_NL) X(T_IQ4_XS) X(T_Q2_K) X(T_Q3_K)  \
    X(T_MXFP4) X(T_NVFP4) X(T_TQ2_0) X(T_Q1_0) X(T_IQ2_XXS) X(T_IQ2_XS) X(T_IQ2_S) X(T_IQ3_XXS) X(T_IQ3_S) X(T_IQ1_S) X(T_IQ1_M) X(T_TQ1_0)

bool launch_moe1_grid_up(uint32_t type, const void *gate, const void *up, const uint16_t *X, const int32_t *idx, float *h,
                         int n_tok, int top_k, int n_embd, int n_ff, int n_expert, int n_cu, hipStream_t stream, bool dry,
                         hipError_t *err) {
    *err = hipSuccess;
    switch (type) {
#define QLIN_CASE(TT) case TT: return moe1_up_typed<TT>(gate, up, X, idx, h, n_tok, top_k, n_embd, n_ff, n_expert, n_cu, stream, dry, err);
    QLIN_MOE1_TYPES(QLIN_CASE)
#undef QLIN_CASE
    default: return false;
    }
}

bool launch_moe1_grid_down(uint32_t type, const void *down, const float *h, const int32_t *idx, const float *w, float *out,
                           int n_tok, int top_k, int n_embd, int n_ff, int n_expert, int n_cu, hipStream_t stream, bool dry,
                           hipError_t *err) {
    *err = hipSuccess;
    switch (type) {
#define QLIN_CASE(TT) case TT: return moe1_down_typed<TT>(down, h, idx, w, out, n_tok, top_k, n_embd, n_ff, n_expert, n_cu, stream, dry, err);
    QLIN_MOE1_TYPES(QLIN_CASE)
#undef QLIN_CASE
    default: return false;
    }
}

bool gemv_grid_covers(uint32_t type) {
    return type == T_IQ2_XXS || type == T_IQ3_XXS || type == T_IQ3_S || type == T_Q6_K || type == T_Q5_K || type == T_Q8_0 ||
           type == T_IQ4_NL || type == T_IQ4_XS || type == T_Q4_0 || type == T_Q2_K || type == T_Q3_K ||
           type == T_Q4_1 || type == T_Q5_0 || type == T_Q5_1 || type == T_MXFP4 || type == T_NVFP4 || type == T_TQ2_0 || type == T_IQ2_XS || type == T_IQ2_S || type == T_Q1_0 || type == T_IQ1_S || type == T_IQ1_M || type == T_TQ1_0;
}

bool launch_gemv_grid(uint32_t type, const GemvJob &job, const float *x, int n_cols, int n_cu, hipStream_t stream,
                      hipError_t *err, size_t row_stride) {
    *err = hipSuccess;
    switch (type) {
    case T_IQ2_XXS: return grid_typed<T_IQ2_XXS>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_IQ3_XXS: return grid_typed<T_IQ3_XXS>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_IQ3_S: return grid_typed<T_IQ3_S>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q6_K: return grid_typed<T_Q6_K>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q5_K: return grid_typed<T_Q5_K>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q8_0: return grid_typed<T_Q8_0>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_IQ4_NL: return grid_typed<T_IQ4_NL>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_IQ4_XS: return grid_typed<T_IQ4_XS>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q4_0: return grid_typed<T_Q4_0>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q2_K: return grid_typed<T_Q2_K>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q3_K: return grid_typed<T_Q3_K>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q4_1: return grid_typed<T_Q4_1>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q5_0: return grid_typed<T_Q5_0>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q5_1: return grid_typed<T_Q5_1>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_MXFP4: return grid_typed<T_MXFP4>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_NVFP4: return grid_typed<T_NVFP4>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_TQ2_0: return grid_typed<T_TQ2_0>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_IQ2_XS: return grid_typed<T_IQ2_XS>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_IQ2_S: return grid_typed<T_IQ2_S>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_Q1_0: return grid_typed<T_Q1_0>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_IQ1_S: return grid_typed<T_IQ1_S>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_IQ1_M: return grid_typed<T_IQ1_M>(job, x, n_cols, n_cu, stream, err, row_stride);
    case T_TQ1_0: return grid_typed<T_TQ1_0>(job, x, n_cols, n_cu, stream, err, row_stride);
    default: return false;
    }
}

}  // namespace qlin

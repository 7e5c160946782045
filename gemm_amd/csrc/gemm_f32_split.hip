/*
 * gemm_f32_split.hip - which fp32 products the split kernel (gemm_f32_split.h) takes, how it divides them, and the two
 * kernels that lay the activations out for it.
 */
#include "qlin_internal.h"

namespace qlin {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));

/* n with |x| 2^n in [2^14, 2^15) for a token's largest |x|, given by its bits (which order like the magnitudes, infinities
 * and NaN above all); 0 for a token of zeros */
__device__ __forceinline__ int token_exp_of(uint32_t largest) {
    if (largest >= 0x7F800000u) return kF32NotFinite;
    if (largest >= 0x00800000u) return 14 + 127 - (int)(largest >> 23);
    return largest == 0 ? 0 : 14 + 149 - (31 - __clz((int)largest)); /* subnormal: its leading bit is 2^(bit - 149) */
}

/* one workgroup per token, dword loads: any alignment of X */
__global__ void __launch_bounds__(256) f32_token_exp_kernel(const float *__restrict__ X, int *__restrict__ token_exp, int n_cols, int ldx) {
    __shared__ uint32_t per_wave[4];
    const uint32_t *x = reinterpret_cast<const uint32_t *>(X + (size_t)blockIdx.x * ldx);
    uint32_t largest = 0;
#pragma unroll 8
    for (int k = threadIdx.x; k < n_cols; k += 256) largest = max(largest, x[k] & 0x7FFFFFFFu);
    for (int d = 32; d > 0; d >>= 1) largest = max(largest, (uint32_t)__shfl_xor((int)largest, d, 64));
    if ((threadIdx.x & 63) == 0) per_wave[threadIdx.x >> 6] = largest;
    __syncthreads();
    if (threadIdx.x) return;
    for (int w = 1; w < 4; w++) largest = max(largest, per_wave[w]);
    token_exp[blockIdx.x] = token_exp_of(largest);
}

/* A workgroup lays out 256 elements of 32 tokens: thread (token, 32 elements). The order of its stores is the fragments'
 * (gemm_f32_split.h); tokens past the end are zeros. SUM: elements per sum of activations (0: none). WIDE: 16-byte
 * loads, where X's rows allow them. */
template <int SUM, bool WIDE>
__global__ void __launch_bounds__(256) f32_split_kernel(const float *__restrict__ X, const int *__restrict__ token_exp, uint8_t *__restrict__ frags,
                                                       uint8_t *__restrict__ sums, int n_sb, int n_tok, int ldx) {
    const int j = threadIdx.x >> 3, u = threadIdx.x & 7, sb = blockIdx.x, tb = blockIdx.y, t = 32 * tb + j;
    const int e = t < n_tok ? token_exp[t] : kF32NotFinite;
    const bool live = e != kF32NotFinite;
    const float *x = X + (size_t)(live ? t : 0) * ldx + 256 * sb + 32 * u;
    float v[32];
#pragma unroll
    for (int i = 0; i < 32; i += 4) {
        if constexpr (WIDE) {
            const float4 q = *reinterpret_cast<const float4 *>(x + i);
            v[i] = q.x; v[i + 1] = q.y; v[i + 2] = q.z; v[i + 3] = q.w;
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++) v[i + k] = x[i + k];
        }
    }
#pragma unroll
    for (int i = 0; i < 32; i++) v[i] = live ? __builtin_ldexpf(v[i], e) : 0.0f;
    uint8_t *at = frags + ((size_t)tb * (8 * n_sb) + 8 * sb + u) * 4096 + 16 * j;
#pragma unroll
    for (int c = 0; c < 4; c++) { /* elements 8 c .. + 7: step c >> 1, lane half c & 1 */
        half8 hi, lo;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            hi[i] = (_Float16)v[8 * c + i];
            lo[i] = (_Float16)(v[8 * c + i] - (float)hi[i]);
        }
        *reinterpret_cast<half8 *>(at + 1024 * (c >> 1) + 512 * (c & 1)) = hi;
        *reinterpret_cast<half8 *>(at + 2048 + 1024 * (c >> 1) + 512 * (c & 1)) = lo;
    }
    if constexpr (SUM != 0) {
        constexpr int kPer = SUM == 16 ? 2048 : 1024;
        uint8_t *s_at = sums + ((size_t)tb * n_sb + sb) * kPer + 16 * j;
#pragma unroll
        for (int g = 0; g < 32 / SUM; g++) {
            double s = 0.0;
#pragma unroll
            for (int i = 0; i < SUM; i++) s += (double)v[SUM * g + i];
            s *= 1.0 / 32; /* 32 elements below 2^15 */
            const _Float16 hi = (_Float16)(float)s, lo = (_Float16)(float)(s - (double)(float)hi);
            /* 32: lanes 0 .. 31 hold the eight heads, 32 .. 63 the tails; 16: lane half h sums 8 h .. + 7, heads then tails */
            const int group = SUM == 16 ? 2 * u + g : u;
            uint8_t *to = SUM == 16 ? s_at + 512 * (group >> 3) + 2 * (group & 7) : s_at + 2 * group;
            *reinterpret_cast<_Float16 *>(to) = hi;
            *reinterpret_cast<_Float16 *>(to + (SUM == 16 ? 1024 : 512)) = lo;
        }
    }
}

/* The same for short rows in one launch: a workgroup finds the powers of two of two tokens and lays their rows out, 256 threads
 * a token. Thread i takes pieces i and i + 256 of eight elements, which wait in registers for the largest element, so that X
 * is read once. What bounds it is the launches of a short call: one in place of two, 320 tokens x 4096 into 4096 rows 46.1
 * -> 43.5 us, 8 tokens 17.0 -> 15.4; with four tokens a workgroup 45.2 and 17.0 (too few workgroups), with one 43.6 and 15.5
 * (single 16-byte pieces of a line). */
constexpr int kTokensPer = 2, kHeld = 2;
template <int SUM, bool WIDE>
__global__ void __launch_bounds__(256 * kTokensPer)
f32_split_rows_kernel(const float *__restrict__ X, int *__restrict__ token_exp, uint8_t *__restrict__ frags, uint8_t *__restrict__ sums, int n_sb,
                 int n_tok, int ldx) {
    __shared__ uint32_t per_wave[4 * kTokensPer];
    const int mine = threadIdx.x >> 8, i = threadIdx.x & 255, t = kTokensPer * blockIdx.x + mine, pieces = 32 * n_sb;
    const float *x = X + (size_t)(t < n_tok ? t : 0) * ldx;
    auto load = [&](int p, float (&v)[8]) {
        if constexpr (WIDE) {
            const float4 a = *reinterpret_cast<const float4 *>(x + 8 * p), b = *reinterpret_cast<const float4 *>(x + 8 * p + 4);
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] = x[8 * p + k];
        }
    };
    uint32_t largest = 0;
    auto look = [&](const float (&v)[8]) {
#pragma unroll
        for (int k = 0; k < 8; k++) largest = max(largest, __float_as_uint(v[k]) & 0x7FFFFFFFu);
    };
    float held[kHeld][8];
    if (t < n_tok) {
#pragma unroll
        for (int k = 0; k < kHeld; k++)
            if (i + 256 * k < pieces) load(i + 256 * k, held[k]);
#pragma unroll
        for (int k = 0; k < kHeld; k++)
            if (i + 256 * k < pieces) look(held[k]);
    }
    for (int d = 32; d > 0; d >>= 1) largest = max(largest, (uint32_t)__shfl_xor((int)largest, d, 64));
    if ((threadIdx.x & 63) == 0) per_wave[threadIdx.x >> 6] = largest;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 4; w++) largest = max(largest, per_wave[4 * mine + w]);
    const int e = t < n_tok ? token_exp_of(largest) : kF32NotFinite;
    if (i == 0 && t < n_tok) token_exp[t] = e;
    const bool live = e != kF32NotFinite;
    const int j = t & 31, tb = t >> 5;
    auto lay_out = [&](int p, const float (&in)[8]) {
        half8 hi, lo;
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float v = live ? __builtin_ldexpf(in[k], e) : 0.0f;
            hi[k] = (_Float16)v;
            lo[k] = (_Float16)(v - (float)hi[k]);
            if (SUM != 0) s += (double)v;
        }
        const int group = p >> 2, c = p & 3; /* 32 elements; step c >> 1, lane half c & 1 */
        uint8_t *at = frags + ((size_t)tb * (8 * n_sb) + group) * 4096 + 16 * j + 1024 * (c >> 1) + 512 * (c & 1);
        *reinterpret_cast<half8 *>(at) = hi;
        *reinterpret_cast<half8 *>(at + 2048) = lo;
        if constexpr (SUM != 0) { /* two or four neighbours have the rest of the sum */
            s += __shfl_xor(s, 1, 64);
            if (SUM == 32) s += __shfl_xor(s, 2, 64);
            s *= 1.0 / 32; /* 32 elements below 2^15 */
            const _Float16 head = (_Float16)(float)s, tail = (_Float16)(float)(s - (double)(float)head);
            /* 32: lanes 0 .. 31 hold the eight heads, 32 .. 63 the tails; 16: lane half h sums 8 h .. + 7, heads then tails */
            constexpr int kPer = SUM == 16 ? 2048 : 1024;
            const int of = SUM == 16 ? 2 * (group & 7) + (c >> 1) : group & 7;
            uint8_t *to = sums + ((size_t)tb * n_sb + (group >> 3)) * kPer + 16 * j + (SUM == 16 ? 512 * (of >> 3) + 2 * (of & 7) : 2 * of);
            if ((c & (SUM / 8 - 1)) == 0) {
                *reinterpret_cast<_Float16 *>(to) = head;
                *reinterpret_cast<_Float16 *>(to + kPer / 2) = tail;
            }
        }
    };
#pragma unroll
    for (int k = 0; k < kHeld; k++)
        if (i + 256 * k < pieces) lay_out(i + 256 * k, held[k]);
}

/* One launch for rows of up to 2048 elements; of up to 4096 where 16-byte loads read them and X holds at most 3 * 2^19 elements.
 * Beyond, the pieces of lines that its workgroups store from different compute units cost more than the launch. A call of
 * two launches against one, of n tokens into 1024 rows: 320 x 4096 29.3 us, 27.2; 400 x 4096 29.2, 29.3; 512 x 4096 30.0, 32.8;
 * 600 x 3072 30.0, 30.8; 512 x 4096 with single loads 30.5, 33.4; the layout of 512 x 14336 alone 18.5, 31. */
bool one_launch(int n_cols, int n_tok, bool wide) {
    return n_cols <= 2048 || (n_cols <= 4096 && wide && (size_t)n_tok * n_cols <= (size_t)3 << 19);
}
static_assert(4096 <= 256 * kHeld * 8, "a row waits in registers");

template <int SUM> void launch_split(const F32SplitCall &c, const F32SplitPlan &p) {
    uint8_t *ws = (uint8_t *)c.workspace;
    int *e = (int *)(ws + p.exp_at);
    const int n_sb = c.n_cols / 256, blocks = p.token_tiles * p.token_blocks;
    const bool wide = ((uintptr_t)c.X & 15) == 0 && c.ldx % 4 == 0;
    if (one_launch(c.n_cols, c.n_tok, wide)) {
        const auto kernel = wide ? f32_split_rows_kernel<SUM, true> : f32_split_rows_kernel<SUM, false>;
        hipLaunchKernelGGL(kernel, dim3(blocks * 32 / kTokensPer), dim3(256 * kTokensPer), 0, c.stream, c.X, e, ws, ws + p.sums_at, n_sb, c.n_tok, c.ldx);
        return;
    }
    hipLaunchKernelGGL(f32_token_exp_kernel, dim3(c.n_tok), dim3(256), 0, c.stream, c.X, e, c.n_cols, c.ldx);
    const auto kernel = wide ? f32_split_kernel<SUM, true> : f32_split_kernel<SUM, false>;
    hipLaunchKernelGGL(kernel, dim3(n_sb, blocks), dim3(256), 0, c.stream, c.X, e, ws, ws + p.sums_at, n_sb, c.n_tok, c.ldx);
}

size_t round256(size_t n) { return (n + 255) & ~(size_t)255; }

/* one chunk of tokens */
hipError_t launch_chunk(uint32_t type, const F32SplitCall &c) {
    switch (type) {
    case T_Q4_K: return f32_split_q4k(c);
    case T_Q5_K: return f32_split_q5k(c);
    case T_Q6_K: return f32_split_q6k(c);
    case T_Q2_K: return f32_split_q2k(c);
    case T_Q3_K: return f32_split_q3k(c);
    case T_Q8_0: return f32_split_q8_0(c);
    case T_Q4_0: return f32_split_q4_0(c);
    case T_IQ4_NL: return f32_split_iq4nl(c);
    case T_IQ4_XS: return f32_split_iq4xs(c);
    case T_IQ3_S: return f32_split_iq3s(c);
    case T_IQ2_XXS: return f32_split_iq2xxs(c);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t launch_f32_split(const F32SplitCall &c, const F32SplitPlan &p, int sum_group) {
    if (sum_group == 0) launch_split<0>(c, p);
    else if (sum_group == 16) launch_split<16>(c, p);
    else launch_split<32>(c, p);
    return hipGetLastError();
}

/* How a chunk is divided. Tiles of 64 tokens (32 where there are no more) by 256 rows (128: Q6_K, Q8_0), and K over
 * `parts` workgroups: the number whose estimated time is least, in units of a super-block's time in a compute unit that
 * two workgroups share (6 us) - rounds of workgroups over 512 places, each with its super-blocks and about one more for its
 * start and end, and the parts' way through memory. Measured, us for 1 / 2 / 4 / 8 / 16 parts (Q4_K): 320 tokens 4096 x 4096
 * 90 / 58 / 49 / 51 / 65 (the rule: 3, 50), 14336 x 4096 123 / 116 / 109 / 121 / 147 (3, 113), 4096 x 14336 257 / 145 / 116 /
 * 110 / 110 (6, 100), 8 tokens 4096 x 4096 52 / 32 / 22 / 17 / 16 (16). */
F32SplitPlan f32_split_plan(uint32_t type, int n_rows, int n_cols, int n_tok, size_t workspace_bytes) {
    F32SplitPlan p = {};
    const int n_sb = n_cols / 256, tile_rows = type == T_Q6_K || type == T_Q8_0 ? 128 : 256;
    p.token_blocks = n_tok > 32 ? 2 : 1;
    p.token_tiles = (n_tok + 32 * p.token_blocks - 1) / (32 * p.token_blocks);
    const size_t blocks = (size_t)p.token_tiles * p.token_blocks;
    p.sums_at = blocks * n_sb * (8 * 4096);
    p.exp_at = p.sums_at + blocks * n_sb * 2048;
    p.parts_at = round256(p.exp_at + blocks * 32 * sizeof(int));
    p.fits = p.parts_at <= workspace_bytes;
    if (!p.fits) return p;
    const size_t part_bytes = (size_t)n_tok * n_rows * sizeof(float);
    const long long tiles = (long long)((n_rows + tile_rows - 1) / tile_rows) * p.token_tiles;
    double best = 0.0;
    for (int parts = 1; parts <= n_sb && parts <= 32; parts++) {
        if (parts > 1 && (p.parts_at + parts * part_bytes > workspace_bytes || tiles * parts > 2048)) break;
        const long long items = tiles * parts;
        const double share = items <= 256 ? 0.6 : 1.0;
        const double cost = (double)((items + 511) / 512) * ((n_sb + parts - 1) / parts + 1.0) * share +
                            (parts > 1 ? 0.5 + parts * (double)part_bytes / (24 << 20) : 0.0);
        if (parts == 1 || cost < best) {
            best = cost;
            p.parts = parts;
        }
    }
    return p;
}

/* Whole super-blocks of the formats whose codes an image gives up, in a workspace that holds the fragments of 32 tokens, from
 * 2.25 M weights on (2 M up to 32 tokens): below, four launches cost more than decoding and the library's product do (us,
 * this route / that one, Q4_K: 64 tokens 1536 x 1536 17.8 / 19.4 but 2048 x 1024 16.6 / 16.1 and 512 x 4096 19.5 / 17.2; 512
 * tokens 1024 x 1024 21.5 / 18.3; 32 tokens 512 x 4096 16.1 / 19.7 but 512 x 2048 14.4 / 13.2; Q6_K the same). The 32-bit
 * offsets of a request hold a wave's 64 rows and a token tile's fragments. */
bool f32_split_takes(uint32_t type, int n_rows, int n_cols, int n_tok, size_t workspace_bytes) {
    const long long weights = (long long)n_rows * n_cols;
    if (weights < (n_tok <= 32 ? 8LL << 18 : 9LL << 18)) return false;
    return fewtok_has(type) && n_cols % 256 == 0 && n_cols <= (1 << 22) && f32_split_plan(type, n_rows, n_cols, 32, workspace_bytes).fits;
}

/* in chunks of tokens whose fragments fill at most three quarters of the workspace (the parts of K want some, too) */
hipError_t launch_gemm_f32_split(uint32_t type, const F32SplitCall &call) {
    int chunk = call.n_tok;
    while (chunk > 32 && (chunk > 65535 || !f32_split_plan(type, call.n_rows, call.n_cols, chunk, call.workspace_bytes / 4 * 3).fits))
        chunk = ((chunk + 1) / 2 + 63) / 64 * 64 < chunk ? ((chunk + 1) / 2 + 63) / 64 * 64 : 32;
    for (int t = 0; t < call.n_tok; t += chunk) {
        F32SplitCall c = call;
        c.X = call.X + (size_t)t * call.ldx;
        c.Y = call.Y + (size_t)t * call.ldy;
        c.n_tok = call.n_tok - t < chunk ? call.n_tok - t : chunk;
        if (const hipError_t e = launch_chunk(type, c); e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace qlin

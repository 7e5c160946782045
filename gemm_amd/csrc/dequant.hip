/*
 * dequant.hip - block decoders: raw GGML blocks -> fp32, bit-identical to the reference's
 * scalar decoders (common/ggml_dequant.h:1479-1687, :2793-3058, type switch :3177-3265),
 * and the same rounded once to bf16.
 *
 * One thread decodes groups of eight consecutive elements. What bounds the kernels is the stream of stores (4 or 2 B out
 * per 0.26..1.06 B in) as long as a group costs few instructions: whole rows one after another are taken as one run of
 * blocks, whose block and place in it are shifts of the thread's index, the codes come in by dword loads and are masked
 * four at a time. 14336 x 4096, with 64-bit divisions and byte loads before: Q5_K to bf16 52 -> 38 us (158 MB, 4.2 TB/s),
 * Q6_K to bf16 39 -> 34.5 (165 MB, 4.8 TB/s), to fp32 Q4_K 67 -> 54 (268 MB, 5.0 TB/s), Q6_K 70 -> 46 (5.8 TB/s).
 */
#include "qlin_device.h"
#include "qlin_internal.h"

namespace qlin {

__device__ __forceinline__ void store8(float *o, const float (&y)[8]) {
    reinterpret_cast<float4 *>(o)[0] = make_float4(y[0], y[1], y[2], y[3]);
    reinterpret_cast<float4 *>(o)[1] = make_float4(y[4], y[5], y[6], y[7]);
}
__device__ __forceinline__ void store8(uint16_t *o, const float (&y)[8]) {
    typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
    uint4 v;
    uint32_t *vp = &v.x;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        bf16x2 r;
        r[0] = (__bf16)y[2 * i];
        r[1] = (__bf16)y[2 * i + 1];
        vp[i] = __builtin_bit_cast(uint32_t, r);
    }
    *reinterpret_cast<uint4 *>(o) = v;
}

/* n_groups groups of eight of one run of blocks; out 16-byte aligned. A workgroup takes 512 groups, a thread two of them
 * 256 apart, so that each store of the workgroup is part of a contiguous stretch.
 * fp32: the two float4 of a thread lie 32 bytes from the next thread's, so a wave would write every second 16 bytes of
 * 2 KB per store; it turns them through its own part of LDS and writes 1 KB in one piece (Q6_K 70 us -> 46, Q4_K 66 -> 54
 * by that alone). */
template <uint32_t T, class OUT>
__global__ void __launch_bounds__(256)
dequant_run_kernel(const uint8_t *__restrict__ W, OUT *__restrict__ out, unsigned long long n_groups) {
    using C = Codec<T>;
    constexpr unsigned GPB = C::BE / 8; /* groups per block, a power of two */
    static_assert((GPB & (GPB - 1)) == 0 && 256 % GPB == 0, "blocks do not divide a workgroup's groups");
    const unsigned long long first = (unsigned long long)blockIdx.x * 512;
    const uint8_t *w = W + first / GPB * C::BB;
    OUT *o = out + first * 8;
    const unsigned left = (unsigned)min(n_groups - first, 512ull);
#pragma unroll
    for (unsigned h = 0; h < 2; h++) {
        const unsigned lane = threadIdx.x & 63u, g0 = threadIdx.x - lane + 256 * h, g = g0 + lane;
        if (g0 >= left) return;
        float y[8];
        if (g < left) C::decode8(w + g / GPB * C::BB, (int)(g % GPB) * 8, y);
        if constexpr (sizeof(OUT) == 2) {
            if (g < left) store8(o + g * 8, y);
        } else {
            __shared__ float4 turn[256 * 2];
            float4 *t = turn + (threadIdx.x - lane) * 2;
            t[2 * lane] = make_float4(y[0], y[1], y[2], y[3]);
            t[2 * lane + 1] = make_float4(y[4], y[5], y[6], y[7]);
            __builtin_amdgcn_wave_barrier();
            float4 *ow = reinterpret_cast<float4 *>(o + g0 * 8);
            const unsigned n = 2 * min(64u, left - g0);
            if (lane < n) ow[lane] = t[lane];
            if (lane + 64 < n) ow[lane + 64] = t[lane + 64];
            __builtin_amdgcn_wave_barrier();
        }
    }
}

/* row by row: gathered rows, rows that end inside a block, rows at a distance, outputs that are not aligned. `chunks`
 * workgroups to a row, or several short rows to a workgroup. */
template <uint32_t T, class OUT, bool VEC>
__global__ void __launch_bounds__(256)
dequant_rows_kernel(const uint8_t *__restrict__ W, const int32_t *__restrict__ row_ids, int n_src_rows,
                    OUT *__restrict__ out, int n_rows, int n_cols, size_t row_bytes, unsigned groups_per_row, unsigned chunks) {
    using C = Codec<T>;
    constexpr unsigned GPB = C::BE / 8;
    const unsigned set = blockIdx.x / chunks, g = (blockIdx.x - set * chunks) * blockDim.x + threadIdx.x;
    const unsigned row = set * blockDim.y + threadIdx.y;
    if (row >= (unsigned)n_rows || g >= groups_per_row) return;
    const unsigned blk = g / GPB, k0 = g % GPB * 8;
    float y[8];
    /* output row `row` is source row row_ids[row] when a list is given (embedding lookup); an id
     * outside the table yields a row of zeros */
    const int src_row = row_ids ? row_ids[row] : (int)row;
    if (src_row >= 0 && src_row < n_src_rows) {
        C::decode8(W + (size_t)src_row * row_bytes + (size_t)blk * C::BB, (int)k0, y);
    } else {
#pragma unroll
        for (int i = 0; i < 8; i++) y[i] = 0.0f;
    }
    OUT *o = out + (size_t)row * n_cols + (size_t)blk * C::BE + k0;
    if constexpr (VEC) {
        store8(o, y);
    } else {
#pragma unroll
        for (int i = 0; i < 8; i++) o[i] = y[i];
    }
}

/* F16 / BF16 / F32 rows (common/ggml_dequant.h:3251-3261); output row r = source row row_ids[r]
 * when a list is given */
__global__ void __launch_bounds__(256)
convert_plain_kernel(uint32_t type, const uint8_t *__restrict__ src, const int32_t *__restrict__ row_ids,
                     int n_src_rows, float *__restrict__ out, long long n, int n_cols) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    long long s = i;
    if (row_ids) {
        const long long r = i / n_cols;
        const int id = row_ids[r];
        if (id < 0 || id >= n_src_rows) {
            out[i] = 0.0f;
            return;
        }
        s = (long long)id * n_cols + (i - r * n_cols);
    }
    if (type == T_F32) {
        reinterpret_cast<uint32_t *>(out)[i] = reinterpret_cast<const uint32_t *>(src)[s];
    } else {
        const uint32_t h = reinterpret_cast<const uint16_t *>(src)[s];
        out[i] = (type == T_F16) ? half_bits_exact(h) : __uint_as_float(h << 16);
    }
}

template <uint32_t T, class OUT>
static hipError_t launch_typed(const void *W, const int32_t *row_ids, int n_src_rows, OUT *out, int n_rows,
                               int n_cols, size_t row_bytes, hipStream_t stream) {
    using C = Codec<T>;
    const size_t bpr = n_cols / C::BE, groups_per_row = bpr * (C::BE / 8);
    if (groups_per_row == 0 || n_rows == 0) return hipSuccess;
    const bool aligned = (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
    if (!row_ids && aligned && (n_rows == 1 || ((size_t)n_cols == bpr * C::BE && row_bytes == bpr * C::BB))) {
        const unsigned long long n = (unsigned long long)groups_per_row * n_rows;
        hipLaunchKernelGGL((dequant_run_kernel<T, OUT>), dim3((unsigned)((n + 511) / 512)), dim3(256), 0, stream,
                           (const uint8_t *)W, out, n);
        return hipGetLastError();
    }
    unsigned wide = 1;
    while (wide < 256 && wide < groups_per_row) wide *= 2;
    const unsigned tall = 256 / wide, chunks = (unsigned)((groups_per_row + wide - 1) / wide);
    const dim3 grid(chunks * (((unsigned)n_rows + tall - 1) / tall)), wg(wide, tall);
    if (sizeof(OUT) == 2 || (n_cols % 4 == 0 && aligned)) {
        hipLaunchKernelGGL((dequant_rows_kernel<T, OUT, true>), grid, wg, 0, stream, (const uint8_t *)W, row_ids,
                           n_src_rows, out, n_rows, n_cols, row_bytes, (unsigned)groups_per_row, chunks);
    } else if constexpr (sizeof(OUT) == 4) {
        hipLaunchKernelGGL((dequant_rows_kernel<T, OUT, false>), grid, wg, 0, stream, (const uint8_t *)W, row_ids,
                           n_src_rows, out, n_rows, n_cols, row_bytes, (unsigned)groups_per_row, chunks);
    }
    return hipGetLastError();
}

hipError_t launch_dequant(uint32_t type, const void *W, const int32_t *row_ids, int n_src_rows, float *out,
                          int n_rows, int n_cols, size_t row_bytes, hipStream_t stream) {
    if (!row_ids) n_src_rows = n_rows;
    switch (type) {
#define QLIN_CASE(TT) case TT: return launch_typed<TT>(W, row_ids, n_src_rows, out, n_rows, n_cols, row_bytes, stream);
    QLIN_FOR_EACH_BLOCK_TYPE(QLIN_CASE)
#undef QLIN_CASE
    case T_F32: case T_F16: case T_BF16: {
        const long long n = (long long)n_rows * n_cols;
        if (n == 0) return hipSuccess;
        hipLaunchKernelGGL(convert_plain_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                           type, (const uint8_t *)W, row_ids, n_src_rows, out, n, n_cols);
        return hipGetLastError();
    }
    default: return hipErrorInvalidValue;
    }
}

/* out[r * n_cols + k] = bf16(decode(W)[r][k]); out 16-byte aligned, n_cols a multiple of the block size */
hipError_t launch_dequant_bf16(uint32_t type, const void *W, uint16_t *out, int n_rows, int n_cols, size_t row_bytes,
                               hipStream_t stream) {
    switch (type) {
#define QLIN_CASE(TT) case TT: return launch_typed<TT>(W, nullptr, n_rows, out, n_rows, n_cols, row_bytes, stream);
    QLIN_FOR_EACH_BLOCK_TYPE(QLIN_CASE)
    QLIN_FOR_EACH_DENSE_TYPE(QLIN_CASE)
#undef QLIN_CASE
    default: return hipErrorInvalidValue;
    }
}

}  // namespace qlin

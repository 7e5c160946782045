/*
 * qlinear_bench.h - measurement probes of libqlinear.so. Not part of the engine's interface: bench.py uses
 * them to print what the GPU at hand sustains beside every measured rate.
 */
#ifndef QLINEAR_BENCH_H
#define QLINEAR_BENCH_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* What this GPU sustains on the two resources the kernels are priced against (the
 * reference prints a peak beside every measured rate, rdna4/dequant/bench_dequant.c:1043-1110). All three
 * only enqueue; time them with qlin_timer_begin/end.
 *   qlin_probe_mfma_bf16: register-only loop of the prefill GEMM's matrix instruction on every compute
 *     unit, `iters` x 4 instructions per wave; *flops receives the flops of the launch.
 *   qlin_probe_clocks: waits for the stream, then returns the shader clock (MHz) that the last
 *     qlin_probe_mfma_bf16 launch ran at (cycle counter against the 100 MHz counter).
 *   qlin_probe_hbm_read: streaming read of n_bytes (16-byte aligned) of device memory. */
int qlin_probe_mfma_bf16(int iters, void *stream, double *flops);
int qlin_probe_clocks(void *stream, double *shader_mhz);
int qlin_probe_hbm_read(const void *buf, size_t n_bytes, void *stream);

/* One tile kernel of the fused prefill GEMM by name, whatever the shape-based choice of qlin_gemm_bf16_any_dev would be:
 * tile 0 = 256 tokens x 128 rows, 1 = 128 tokens x 64 rows, 3 to 6 = that many times 32 tokens x 128 rows. Arguments and result as
 * qlin_gemm_bf16_any_dev without a workspace; Q2_K ... Q6_K, Q8_0, IQ4_NL, IQ4_XS, Q4_0; n_cols % 256 == 0. For timing one against the
 * other and for the parity tests of each on small shapes. */
int qlin_probe_gemm_tile(int tile, uint32_t ggml_type, const void *W, const uint16_t *X, float *Y, int n_rows, int n_cols,
                         int n_tok, int ldx, int ldy, void *stream);
/* what qlin_gemm_bf16_any_dev does with a shape: 1 and 2 = a tile kernel, of the class of 256 x 128 or of 128 x 64 tiles (tensors of
 * one class share a launch; which tiles it takes says qlin_probe_gemm_blocks), 3 = the few-token kernel, 0 = none of them (a matvec
 * per token, or decode to bf16 + dense product) */
int qlin_probe_gemm_route(uint32_t ggml_type, int n_rows, int n_cols, int n_tok, int ldx, int have_workspace);
/* over how many workgroups a tile's K is divided, given a workspace of qlin_gemm_bf16_any_workspace_bytes bytes (1: it is not) */
int qlin_probe_gemm_parts(uint32_t ggml_type, int n_rows, int n_cols, int n_tok, int ldx);
/* the kernel whose one launch the tensors of a qlin_gemm_bf16_multi_dev call share, numbered as above (0: a call each) */
int qlin_probe_gemm_multi_route(uint32_t ggml_type, int n_mat, const int *n_rows, int n_cols, int n_tok, int ldx, int have_workspace);
/* the tiles of the one launch that one tensor, or those of a qlin_gemm_bf16_multi_dev call, take: 1 = 128 tokens x 64 rows, 3, 4, 5, 6
 * or 8 = that many times 32 tokens x 128 rows, 0 = not one launch of tiles */
int qlin_probe_gemm_blocks(uint32_t ggml_type, int n_mat, const int *n_rows, int n_cols, int n_tok, int ldx, int have_workspace);
/* whether a matvec on aligned, unpadded operands copies its blocks to LDS (gemv_dma.hip), for one to three matrices or (pair) gate and
 * up: 0, or the waves of a workgroup + 100 x the rounds of workgroups */
int qlin_probe_gemv_lds(uint32_t ggml_type, int pair, int n_mat, const int *n_rows, int n_cols);
/* whether qlin_gemm_f32_any_dev multiplies a shape's codes on the matrix cores (1) or decodes to fp32 for the library's
 * product, or takes the few-token fp32 kernel (0), given a workspace of qlin_gemm_f32_any_workspace_bytes bytes */
int qlin_probe_gemm_f32_route(uint32_t ggml_type, int n_rows, int n_cols, int n_tok);

#ifdef __cplusplus
}
#endif
#endif /* QLINEAR_BENCH_H */

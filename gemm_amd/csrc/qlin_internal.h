/*
 * qlin_internal.h - host-side launchers shared between the translation units of libqlinear.
 * Every launcher validates nothing: the C-ABI layer (qlin_api.hip) checks shapes, alignment
 * and types before it calls in here. All return the hipError_t of the launch.
 */
#ifndef QLIN_INTERNAL_H
#define QLIN_INTERNAL_H

#include <hip/hip_runtime.h>

#include <atomic>
#include <stddef.h>
#include <stdint.h>

#include "qlin_device.h"

namespace qlin {

/* "this kernel's dynamic LDS limit has been raised": set after hipFuncSetAttribute succeeded. Device entry
 * points may be called from several threads; raising the limit twice is harmless, a torn flag is not. */
struct OnceFlag {
    std::atomic<bool> done{false};
    bool is_set() const { return done.load(std::memory_order_acquire); }
    void set() { done.store(true, std::memory_order_release); }
};

/* out[n_rows, n_cols] = decode(W); n_cols may be ragged: only n_cols / block_elems blocks per
 * row are decoded, row r of W starts at r * row_bytes, row r of out at r * n_cols. With row_ids
 * (device, n_rows entries) output row r is decoded from source row row_ids[r] of a table of
 * n_src_rows rows (zeros for an id outside it); without, n_src_rows is ignored. */
hipError_t launch_dequant(uint32_t type, const void *W, const int32_t *row_ids, int n_src_rows, float *out,
                          int n_rows, int n_cols, size_t row_bytes, hipStream_t stream);

/* One matvec launch over up to three matrices of ONE block type that share x and n_cols: the
 * fused call shapes of the reference's decode loop.
 *   kStore    y_m[r] = W_m[r,:] . x for every matrix m (rows of the matrices are concatenated:
 *             tf_qmatvec_fused2_pool, tf_qmatvec_fused_qkv_pool, common/transformer.h:897, :1021)
 *   kAdd      y_m[r] += W_m[r,:] . x   (projection followed by the residual add, :4037)
 *   kSiluMul  two matrices of equal row count: y_0[r] = silu(W_0[r,:].x) * (W_1[r,:].x)
 *             (tf_qmatvec_fused2_silu_pool, :953; silu(g) = g / (1 + exp(-g))) */
enum GemvMode : int { kStore = 0, kAdd = 1, kSiluMul = 2 };
struct GemvJob {
    const void *W[3];
    float *y[3];
    int n_rows[3];
    int n_mat;   /* 1..3; kSiluMul: 2 */
    int mode;    /* GemvMode */
    int total_rows() const { return n_rows[0] + (n_mat > 1 ? n_rows[1] : 0) + (n_mat > 2 ? n_rows[2] : 0); }
};
inline GemvJob single_job(const void *W, float *y, int n_rows, int mode = kStore) {
    GemvJob j = {{W, nullptr, nullptr}, {y, nullptr, nullptr}, {n_rows, 0, 0}, 1, mode};
    return j;
}

inline JobView job_view(const GemvJob &job) {
    const JobView v = {(const uint8_t *)job.W[0], (const uint8_t *)job.W[1], (const uint8_t *)job.W[2],
                       job.y[0], job.y[1], job.y[2],
                       job.n_rows[0], job.n_mat > 1 ? job.n_rows[1] : 0, job.n_mat > 2 ? job.n_rows[2] : 0, job.mode};
    return v;
}

/* one job: y[n_rows] = W . x (or the fused forms above), any supported type and any whole-block shape */
hipError_t launch_gemv_generic(uint32_t type, const GemvJob &job, const float *x, int n_cols, hipStream_t stream);
/* dense F32/F16/BF16 rows of any length and element alignment, one element per lane and step */
hipError_t launch_gemv_dense_ragged(uint32_t type, const GemvJob &job, const float *x, int n_cols, hipStream_t stream);
/* dense rows of 4097..16384 elements in one launch; false: not this kernel's shape */
bool launch_gemv_dense_long(uint32_t type, const GemvJob &job, const float *x, int n_cols, int n_cu, hipStream_t stream,
                            hipError_t *err, size_t row_stride = 0);
/* streaming matvec for every type; returns false if the shape rules of gemv_stream.hip do not
 * hold (nothing was launched), else true with the launch status in *err */
/* row_stride (all four kernels below): bytes between the rows of a matrix; 0 = the rows are packed. Anything else
 * runs the kernel over a column range of longer rows (W then points at the range's first block of row 0). */
bool launch_gemv_stream(uint32_t type, const GemvJob &job, const float *x, int n_cols, int n_cu,
                        hipStream_t stream, hipError_t *err, size_t row_stride = 0);
/* integer-dot matvec (gemv_int.hip) for the formats it covers; same contract as launch_gemv_stream */
bool launch_gemv_int(uint32_t type, const GemvJob &job, const float *x, int n_cols, int n_cu,
                     hipStream_t stream, hipError_t *err, size_t row_stride = 0);
/* the formats whose rows launch_gemv_int reads from any even address (the others want 16-byte boundaries) */
bool gemv_int_takes_any_even_address(uint32_t type);
/* matrix-instruction matvec for the formats of gemv_grid_covers (gemv_grid.hip): n_cols % 256 == 0, n_cols <= 16384,
 * rows of up to 4096 elements only where it measured faster; same contract as launch_gemv_stream */
bool launch_gemv_grid(uint32_t type, const GemvJob &job, const float *x, int n_cols, int n_cu,
                      hipStream_t stream, hipError_t *err, size_t row_stride = 0);
/* matvec on blocks copied to LDS (gemv_dma.hip), where it measured faster than the others; same contract as launch_gemv_stream */
bool launch_gemv_dma(uint32_t type, const GemvJob &job, const float *x, int n_cols, int n_cu, hipStream_t stream, hipError_t *err,
                     size_t row_stride = 0);
/* for the tests: the waves of a workgroup + 100 x the rounds of workgroups that a call takes there (0: another kernel runs) */
int probe_gemv_dma(uint32_t type, bool pair, int n_mat, const int *n_rows, int n_cols, int n_cu);
bool gemv_grid_covers(uint32_t type); /* the formats it has an item for */
/* A few tokens, each on its own, through their top_k experts as two matvec launches: gate + up + SiLU into h
 * (n_tok * top_k * n_ff floats, X [n_tok, n_embd] bf16), then down with the routing weights folded into h. Q4_K experts
 * and the formats of the matrix-instruction matvec (gate and up of one type). false: not a shape for it; dry: only say so. */
bool launch_moe1_q4k_up(const void *gate, const void *up, const uint16_t *X, const int32_t *idx, float *h, int n_tok,
                        int top_k, int n_embd, int n_ff, int n_expert, int n_cu, hipStream_t stream, bool dry, hipError_t *err);
bool launch_moe1_q4k_down(const void *down, const float *h, const int32_t *idx, const float *w, float *out, int n_tok, int top_k,
                          int n_embd, int n_ff, int n_expert, int n_cu, hipStream_t stream, bool dry, hipError_t *err);
bool launch_moe1_grid_up(uint32_t type, const void *gate, const void *up, const uint16_t *X, const int32_t *idx, float *h,
                         int n_tok, int top_k, int n_embd, int n_ff, int n_expert, int n_cu, hipStream_t stream, bool dry,
                         hipError_t *err);
bool launch_moe1_grid_down(uint32_t type, const void *down, const float *h, const int32_t *idx, const float *w, float *out,
                           int n_tok, int top_k, int n_embd, int n_ff, int n_expert, int n_cu, hipStream_t stream, bool dry,
                           hipError_t *err);
/* tuned Q4_K matvec: n_cols % 256 == 0, n_cols <= 16384, W and x 16-byte aligned */
hipError_t launch_gemv_q4k(const GemvJob &job, const float *x, int n_cols, hipStream_t stream, int n_cu,
                           size_t row_stride = 0);

/* Y[t*ldy + r] = dot(W[r,:], X[t*ldx..]) in fp32 */
hipError_t launch_gemm_f32(uint32_t type, const void *W, const float *X, float *Y, int n_rows,
                           int n_cols, int n_tok, int ldx, int ldy, hipStream_t stream);

/* any format: decode to bf16 (dequant.hip), then the dense library GEMM (gemm_dense_lt.hip) */
hipError_t launch_dequant_bf16(uint32_t type, const void *W, uint16_t *out, int n_rows, int n_cols, size_t row_bytes,
                               hipStream_t stream);
constexpr size_t kDenseLibWorkspace = (size_t)32 << 20; /* behind the decoded weights, for the library; up to twice that is used where there is room */
size_t dense_gemm_weight_bytes(int n_rows, int n_cols);
size_t dense_gemm_weight_bytes_f32(int n_rows, int n_cols);
const char *launch_gemm_dense(bool fp32_operands, const void *Wd, const void *X, float *Y, int n_rows, int n_cols,
                              int n_tok, int ldx, int ldy, void *lib_ws, size_t lib_ws_bytes, hipStream_t stream);
const char *launch_gemm_dense_bf16(const uint16_t *Wd, const uint16_t *X, float *Y, int n_rows, int n_cols, int n_tok,
                                   int ldx, int ldy, void *lib_ws, size_t lib_ws_bytes, hipStream_t stream);
/* this library's dense bf16 x bf16 tile kernel (gemm_dense_mfma.hip): n_cols % 256 == 0, Wd and X 16-byte
 * aligned, ldx % 8 == 0 */
hipError_t launch_gemm_dense_own(const uint16_t *Wd, const uint16_t *X, float *Y, int n_rows, int n_cols, int n_tok,
                                 int ldx, int ldy, hipStream_t stream);
/* the few-token kernel (gemm_fewtok.h): up to three tensors of one format and row length against the same activations */
struct FewtokCall {
    int n_mat; /* 1..3 */
    const void *const *W;
    const uint16_t *X;
    float *const *Y;
    const int *n_rows;
    int n_cols, n_tok, ldx;
    const int *ldy;
    hipStream_t stream;
};
bool fewtok_has(uint32_t type);
int fewtok_unrounded(uint32_t type); /* token count up to which the codes stay unrounded */
bool fewtok_takes(uint32_t type, int n_rows, int n_cols, int n_tok, int ldx);
bool fewtok_leaves_to_matvec(uint32_t type, int n_rows, int n_cols, int n_tok);
hipError_t launch_gemm_fewtok(uint32_t type, const FewtokCall &c);
hipError_t launch_gemm_fewtok_one_by_one(uint32_t type, const FewtokCall &c); /* any ldx */
hipError_t fewtok_q4k(const FewtokCall &c);
hipError_t fewtok_q5k(const FewtokCall &c);
hipError_t fewtok_q6k(const FewtokCall &c);
hipError_t fewtok_q2k(const FewtokCall &c);
hipError_t fewtok_q3k(const FewtokCall &c);
hipError_t fewtok_q8_0(const FewtokCall &c);
hipError_t fewtok_q4_0(const FewtokCall &c);
hipError_t fewtok_iq4nl(const FewtokCall &c);
hipError_t fewtok_iq4xs(const FewtokCall &c);
hipError_t fewtok_iq3s(const FewtokCall &c);
hipError_t fewtok_iq2xxs(const FewtokCall &c);
/* fp32 products without rounding on the matrix cores, activations as two fp16 numbers (gemm_f32_split.h) */
constexpr int kF32NotFinite = 1 << 20; /* in place of a token's power of two */
struct F32SplitCall {
    const void *W;
    const float *X;
    float *Y;
    int n_rows, n_cols, n_tok, ldx, ldy;
    void *workspace;
    size_t workspace_bytes;
    hipStream_t stream;
};
/* token tiles of 32 token_blocks tokens, K in `parts` parts, and where the workspace holds what (fragments first) */
struct F32SplitPlan {
    bool fits;
    int token_blocks, token_tiles, parts;
    size_t sums_at, exp_at, parts_at;
};
F32SplitPlan f32_split_plan(uint32_t type, int n_rows, int n_cols, int n_tok, size_t workspace_bytes);
bool f32_split_takes(uint32_t type, int n_rows, int n_cols, int n_tok, size_t workspace_bytes);
hipError_t launch_gemm_f32_split(uint32_t type, const F32SplitCall &c);
hipError_t launch_f32_split(const F32SplitCall &c, const F32SplitPlan &p, int sum_group);
hipError_t f32_split_q4k(const F32SplitCall &c);
hipError_t f32_split_q5k(const F32SplitCall &c);
hipError_t f32_split_q6k(const F32SplitCall &c);
hipError_t f32_split_q2k(const F32SplitCall &c);
hipError_t f32_split_q3k(const F32SplitCall &c);
hipError_t f32_split_q8_0(const F32SplitCall &c);
hipError_t f32_split_q4_0(const F32SplitCall &c);
hipError_t f32_split_iq4nl(const F32SplitCall &c);
hipError_t f32_split_iq4xs(const F32SplitCall &c);
hipError_t f32_split_iq3s(const F32SplitCall &c);
hipError_t f32_split_iq2xxs(const F32SplitCall &c);
constexpr int kMatvecTokens = 4; /* qlin_gemm_bf16_any_dev: up to this many tokens of a format without a few-token kernel go through the matvec */
/* Tiles of 128 rows on four waves, one per SIMD, weights decoded from their blocks into the matrix operand
 * (gemm_kq_wave4.h): the formats of gemm_kq_wave4_covers, n_cols % 256 == 0, ldx < 2^22 */
bool gemm_kq_wave4_covers(uint32_t type);
/* K of a tensor divided over parts[i] workgroups per tile, which write their sums to buf[i], [part][token][row]; launch_k_join adds
 * them up, of all tensors that are divided. One part: the sums go to Y. */
struct KSplit {
    float *buf[3] = {nullptr, nullptr, nullptr};
    int parts[3] = {1, 1, 1};
    bool divides() const { return parts[0] > 1 || parts[1] > 1 || parts[2] > 1; }
};
void launch_k_join(const KSplit &split, int n_mat, float *const *Y, const int *n_rows, int n_tok, const int *ldy, hipStream_t stream);
/* up to three tensors of one format and K in one launch (row tiles numbered through the tensors): tiles of 128 rows x 32 `blocks`
 * tokens, blocks 3, 4, 5, 6 or 8 (8 where K is divided), or of 64 rows x 128 tokens, two workgroups per compute unit (gemm_kq_wave4s.hip).
 * Every shape gives the same bits */
hipError_t launch_gemm_kq_bf16_wave4_multi(uint32_t type, int blocks, int n_mat, const void *const *W, const uint16_t *X,
                                           float *const *Y, const int *n_rows, int n_cols, int n_tok, int ldx,
                                           const int *ldy, hipStream_t stream, KSplit split = {});
hipError_t launch_gemm_kq_bf16_wave4s_multi(uint32_t type, int n_mat, const void *const *W, const uint16_t *X,
                                            float *const *Y, const int *n_rows, int n_cols, int n_tok, int ldx,
                                            const int *ldy, hipStream_t stream, KSplit split = {});
/* the 128-row kernel by format (gemm_kq_wave4_*.hip) */
constexpr int kLargeBlocks = 8;
struct Wave4Call {
    int blocks, n_mat;
    const void *const *W;
    const uint16_t *X;
    float *const *Y;
    const int *n_rows;
    int n_cols, n_tok, ldx;
    const int *ldy;
    KSplit split;
    hipStream_t stream;
};
hipError_t wave4_q4k(const Wave4Call &c);
hipError_t wave4_q5k(const Wave4Call &c);
hipError_t wave4_q2k(const Wave4Call &c);
hipError_t wave4_q6k(const Wave4Call &c);
hipError_t wave4_q3k(const Wave4Call &c);
hipError_t wave4_q8_0(const Wave4Call &c);
hipError_t wave4_q4_0(const Wave4Call &c);
hipError_t wave4_iq4nl(const Wave4Call &c);
hipError_t wave4_iq4xs(const Wave4Call &c);
/* the fused kernel for a shape (kFusedNone: decode + dense product, or the format has none), by the lines between token counts and the
 * estimates of what lies beyond them, or by the lines alone */
enum FusedTile { kFusedNone = 0, kFusedLarge, kFusedSmall };
FusedTile choose_fused_tile(uint32_t type, int n_rows, int n_cols, int n_tok, int ldx, bool have_workspace, bool estimates = true);
/* whether K is divided, and over how many workgroups a tile (1: it is not), given what would take the product whole by the lines alone;
 * the parts lie at the start of the workspace */
struct FusedSplit { FusedTile tile; int parts; };
FusedSplit choose_fused_split(uint32_t type, int n_rows, int n_cols, int n_tok, int ldx, size_t workspace_bytes, FusedTile tile, bool few);
hipError_t launch_fused_split(FusedSplit s, uint32_t type, const void *W, const uint16_t *X, float *Y, int n_rows, int n_cols, int n_tok,
                              int ldx, int ldy, void *workspace, hipStream_t stream);
/* tensors that take a tile kernel each by itself, undivided, in one launch of the tile shape that suits them together */
int choose_token_blocks(uint32_t type, FusedTile tile, int n_mat, const int *n_rows, int n_cols, int n_tok);
hipError_t launch_fused_tiles(FusedTile tile, uint32_t type, int n_mat, const void *const *W, const uint16_t *X, float *const *Y, const int *n_rows,
                              int n_cols, int n_tok, int ldx, const int *ldy, hipStream_t stream);
hipError_t launch_fused_tile(FusedTile tile, uint32_t type, const void *W, const uint16_t *X, float *Y, int n_rows,
                             int n_cols, int n_tok, int ldx, int ldy, hipStream_t stream);
hipError_t launch_gemm_q4k_bf16(const void *W, const uint16_t *X, float *Y, int n_rows, int n_cols,
                                int n_tok, int ldx, int ldy, hipStream_t stream);

/* grouped MoE expert FFN (bf16 activations): Q4_K matrices on the matrix cores, any other format through
 * the bit-exact codec in fp32; the three matrices may have different formats */
size_t moe_workspace_bytes(int n_tok, int top_k, int n_embd, int n_ff, int n_expert);
hipError_t launch_moe_ffn(uint32_t type_gate, uint32_t type_up, uint32_t type_down, const void *gate, const void *up,
                          const void *down, const uint16_t *X, const int32_t *idx, const float *w, float *out, int n_tok,
                          int top_k, int n_embd, int n_ff, int n_expert, int n_cu, void *workspace, hipStream_t stream);

/* the same with the workspace in a device array of the library (at most kMoeStaticScratchBytes); setup once per
 * device with that device current, before the first launch there */
constexpr size_t kMoeStaticScratchBytes = (size_t)16 << 20; /* = QLIN_MOE_STATIC_SCRATCH_BYTES of the public header */
constexpr int kMaxScratchDevices = 64;
hipError_t moe_static_scratch_setup(int device);
hipError_t launch_moe_ffn_static(uint32_t type_gate, uint32_t type_up, uint32_t type_down, const void *gate,
                                 const void *up, const void *down, const uint16_t *X, const int32_t *idx, const float *w,
                                 float *out, int n_tok, int top_k, int n_embd, int n_ff, int n_expert, int device,
                                 int n_cu, hipStream_t stream);

/* MoE pieces */
hipError_t launch_moe_route(const float *logits, int n_tok, int n_expert, int top_k, int32_t *idx,
                            float *w, hipStream_t stream);
hipError_t launch_silu_mul(float *h, const float *gate, const float *up, int n, hipStream_t stream);
/* result[0] = index (as int32 bits) of the first largest of v[0..n), result[1] = that value: the
 * loop `if (v[j] > v[best]) best = j` (server/server_llm.c:224-228). result holds
 * QLIN_ARGMAX_RESULT_BYTES bytes: the rest is scratch for the first stage. */
hipError_t launch_argmax(const float *v, int n, float *result, hipStream_t stream);
/* measurement probes (probe.hip): a register-only MFMA loop (flops issued come back in *flops) with the
 * cycle and 100 MHz counters around it, and a streaming read of a device buffer */
hipError_t launch_probe_mfma(int iters, int n_cu, hipStream_t stream, double *flops);
hipError_t launch_probe_read(const void *buf, size_t n_bytes, hipStream_t stream);
hipError_t read_probe_clocks(uint64_t out[2]);
hipError_t launch_axpy_dev_weight(float *out, const float *q, const float *w, int widx, int n,
                                  int overwrite, hipStream_t stream);

}  // namespace qlin
#endif

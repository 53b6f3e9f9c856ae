/*
 * C ABI of libatorch_amd_fp8.so: hand-written gfx950 (MI355X) kernels for the
 * FP8 grouped-linear MoE expert path.
 *
 * Conventions
 *   - every pointer is a DEVICE pointer owned by the caller (the caller
 *     allocates all outputs and workspaces); nothing here allocates device
 *     memory or synchronises the host with the device (the dual GELU and the
 *     SwiGLU-backward quantisers take four bytes of pinned host memory each
 *     in their first call on a device that is not captured);
 *   - `stream` is a hipStream_t passed as void* (NULL = the default stream);
 *     kernels are only enqueued;
 *   - functions return AAMD_OK (0) or an error code; aamd_last_error() gives
 *     the message of the last failure on the calling thread;
 *   - fp8 tensors are OCP e4m3fn codes, one byte each; scales are fp32
 *     dequantisation scales  s = max(amax, eps) / 448  (0 -> 1);
 *   - `dtype` arguments: AAMD_BF16 or AAMD_F32 (also AAMD_NONE where stated; the inputs of
 *     aamd_quant_1x128, aamd_permute_quant_1x128, aamd_quant_1x128_dual_grouped,
 *     aamd_permute_quant_1x128_dual_grouped and aamd_quant_128x128 may also be AAMD_F16).
 *
 * Each entry point names the reference interface it replaces (paths relative
 * to the reference tree root).
 */
#ifndef ATORCH_AMD_FP8_H
#define ATORCH_AMD_FP8_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif
#pragma GCC visibility push(default) /* the entry points are the only symbols the library exports */

#define AAMD_OK 0
#define AAMD_ERR_ARG 1 /* bad shape / alignment / dtype */
#define AAMD_ERR_HIP 2 /* the HIP runtime refused the launch */

#define AAMD_NONE (-1)
#define AAMD_BF16 0
#define AAMD_F32 1
#define AAMD_F16 2 /* accepted as the input type of the quantisers only */

/* Layouts of the transposed 1x128 codes q_t of R rows (columns of the quantised tensor) and ld_t padded tokens:
 *   AAMD_QT_ROWS     q_t [R, ld_t]: one row of ld_t bytes per column of x;
 *   AAMD_QT_BLOCKED  q_t [ld_t / 128, R, 128]: token-block-major, byte (r, t) at ((t / 128) * R + r) * 128 + t % 128.
 *   AAMD_QT_ROWS_SCALES  as AAMD_QT_ROWS with the scales row-major too, s_t [R, ld_t / 128] (aamd_quant_1x128_dual_grouped only).
 * The second is what the grouped kernels use among themselves: a 128 x 128 tile of codes is 16 KB of consecutive
 * bytes, which the quantisers write as one sequential sweep and the weight-gradient GEMM loads as whole slabs.
 * The scales s_t [ld_t / 128, R] are the same in both. */
#define AAMD_QT_ROWS 0
#define AAMD_QT_BLOCKED 1
#define AAMD_QT_ROWS_SCALES 2

#define AAMD_ABI_VERSION 4

/* Library identity and error text. */
int aamd_abi_version(void);
const char *aamd_last_error(void);

/*
 * 1x128 tile quantisation.
 * Replaces tile_quant / tile_quant_kernel, atorch/modules/fp8/triton_kernel.py:94-140
 * (dispatch: Fp8Quantization.quantize_tilewise, atorch/modules/fp8/quantize.py:176-201).
 *   x [rows, cols] (row stride ldx elements), cols % 128 == 0
 *   q [rows, cols] codes, s [rows, cols/128] fp32, both dense.
 */
int aamd_quant_1x128(const void *x, int x_dtype, int64_t rows, int64_t cols, int64_t ldx, uint8_t *q, float *s,
                     float eps, void *stream);
/* aamd_group_offsets of `counts` [E] in host memory and aamd_quant_1x128, in one launch for up to 64 groups
 * (triton_kernel.py:94-140, quantized_grouped_linear.py:90-101 as there). */
int aamd_quant_1x128_with_offsets(const void *x, int x_dtype, int64_t rows, int64_t cols, int64_t ldx, const int64_t *counts,
                                  int E, int64_t *group_offsets, uint8_t *q, float *s, float eps, void *stream);

/*
 * Token permute fused into the 1x128 quantisation: every token row is read and
 * quantised once and written to its topk destination rows.
 * Replaces permute (atorch/modules/moe/token_dispatcher.py:89-116) followed by the
 * per-expert quantize calls of atorch/modules/fp8/quantized_grouped_linear.py:90-101.
 *   x [T, cols]; row_map [T*topk] int32: destination (permuted) row of flat
 *   index token*topk+slot, or -1 when that copy is dropped;
 *   q [M_out, cols], s [M_out, cols/128] dense; rows no map entry points to are not written.
 */
int aamd_permute_quant_1x128(const void *x, int x_dtype, int64_t T, int64_t cols, int64_t ldx,
                             const int32_t *row_map, int topk, int64_t M_out, uint8_t *q, float *s, float eps,
                             void *stream);

/*
 * Token permute without quantisation (rows of bf16 or fp32 copied to their topk permuted
 * positions, each source row read once).
 * Replaces permute, atorch/modules/moe/token_dispatcher.py:89-116 (index_select on the argsort).
 *   x [T, cols] dense; out [M_out, cols] dense; cols * element size must be a multiple of 16.
 */
int aamd_permute_rows(const void *x, int x_dtype, int64_t T, int64_t cols, const int32_t *row_map, int topk,
                      int64_t M_out, void *out, void *stream);

/*
 * Row-wise AND transposed 1x128 quantisation of ragged groups in one pass over x
 * ("return_transpose=True").
 * Replaces quantize_op.quantize(x_i, params, return_transpose=True) per expert,
 * quantized_grouped_linear.py:90-101 and :200-206; the transposed result is defined
 * in-tree as tile_quant(x_i.t().contiguous()), atorch/modules/fp8/scaled_linear.py:402-414,
 * with a partial last token tile zero padded.
 *   x [M, cols]; group_offsets [E+1] int64 (device) exclusive prefix of rows per group, or NULL for one group of
 *   all rows (then E must be 1);
 *   q [M, cols], s [M, cols/128]              (both may be NULL: transposed only)
 *   q_t, in the layout q_t_layout names: token poff_g + m of column c holds the code of x[off_g + m, c], where
 *       poff_g = sum_{j<g} ceil(M_j/128)*128; pad tokens of a group are written 0
 *   s_t [ld_t/128, cols]: s_t[poff_g/128 + m/128, c]
 *   ld_t % 128 == 0 and ld_t >= poff_E (M + 127*E rounded up to 128 always suffices)
 *   tile_ws: not used (the kernels find their group in group_offsets themselves); may be NULL.
 */
int aamd_quant_1x128_dual_grouped(const void *x, int x_dtype, int64_t M, int64_t cols, int64_t ldx,
                                  const int64_t *group_offsets, int E, int32_t *tile_ws, uint8_t *q, float *s,
                                  uint8_t *q_t, float *s_t, int64_t ld_t, int q_t_layout, float eps, void *stream);

/*
 * The token permute fused into aamd_quant_1x128_dual_grouped: x holds the tokens in their original order and
 * every output row j (expert-contiguous order) is quantised from token sorted_idx[j] / topk, so the permuted
 * bf16 rows are never written or re-read on the way to the grouped GEMMs of a training step.
 * Replaces permute (atorch/modules/moe/token_dispatcher.py:89-116: argsort, index_select on sorted // topk)
 * followed by the per-expert quantize_op.quantize(x_i, x_params, return_transpose=True) calls of
 * atorch/modules/fp8/quantized_grouped_linear.py:90-101.
 *   x [T, cols] (row stride ldx elements); sorted_idx [M] int64 (device): flat index token*topk+slot of
 *   permuted row j, the sorted_idx of aamd_moe_preprocess (M < T*topk when copies were dropped);
 *   T*topk < 2^31; group_offsets [E+1] int64 exclusive prefix of permuted rows per group;
 *   q [M, cols], s [M, cols/128] (both may be NULL), q_t, s_t [ld_t/128, cols], tile_ws, ld_t and q_t_layout
 *   as for aamd_quant_1x128_dual_grouped.  Results equal aamd_permute_rows followed by
 *   aamd_quant_1x128_dual_grouped bit for bit.
 */
int aamd_permute_quant_1x128_dual_grouped(const void *x, int x_dtype, int64_t T, int64_t cols, int64_t ldx,
                                          const int64_t *sorted_idx, int topk, int64_t M,
                                          const int64_t *group_offsets, int E, int32_t *tile_ws, uint8_t *q, float *s,
                                          uint8_t *q_t, float *s_t, int64_t ld_t, int q_t_layout, float eps,
                                          void *stream);

/*
 * The same of the combine's gradient with respect to the permuted rows: row j is bf16(dout[sorted_idx[j] / topk] * probs[sorted_idx[j]]),
 * what aamd_permute_rows_scaled writes for bf16 rows (autograd of token_dispatcher.py:155-159), quantised as aamd_quant_1x128_dual_grouped does (eps 0) without being written.
 * dout [T, cols] bf16 or fp32, dense; probs [T, topk] bf16 or fp32; tile_sums as in aamd_dual_grouped_with_sums, or NULL.
 */
int aamd_combine_grad_quant_1x128_dual_grouped(const void *dout, int dtype, int64_t T, int64_t cols, const int64_t *sorted_idx,
                                               int topk, int64_t M, const void *probs, int probs_dtype,
                                               const int64_t *group_offsets, int E, uint8_t *q, float *s, uint8_t *q_t,
                                               float *s_t, int64_t ld_t, int q_t_layout, float *tile_sums, void *stream);

/*
 * 128x128 block quantisation of E weight matrices, optionally also emitting the
 * transposed codes and scale grid.
 * Replaces block_quant / block_quant_kernel, triton_kernel.py:21-46 (dispatch
 * quantize.py:204-232) and w_fp8.t().contiguous() / scale.t().contiguous(),
 * scaled_linear.py:359-365.
 *   w [E, N, K] (expert stride in elements; rows dense), N % 128 == 0, K % 128 == 0
 *   q [E, N, K], s [E, N/128, K/128]; q_t [E, K, N], s_t [E, K/128, N/128] (q_t/s_t may be NULL).
 */
int aamd_quant_128x128(const void *w, int w_dtype, int64_t E, int64_t N, int64_t K, int64_t expert_stride,
                       uint8_t *q, float *s, uint8_t *q_t, float *s_t, float eps, void *stream);

/*
 * The codes of aamd_quant_128x128 in the transposed orientation only (q_t [E, K, N], s_t [E, K/128, N/128]): a weight whose
 * product reads it that way, where the other product reads the same bytes through aamd_grouped_gemm_fp8_nn.
 * Replaces the transposed half of quantize_square_blockwise, cuda_kernel.py:41-61.
 */
int aamd_quant_128x128_t(const void *w, int w_dtype, int64_t E, int64_t N, int64_t K, int64_t expert_stride,
                         uint8_t *q_t, float *s_t, float eps, void *stream);

/*
 * The codes of aamd_quant_128x128 (q and s, q_t and s_t, or both) for the experts that have rows, group_offsets [E+1] int64 on the
 * device; those of the others, which no product of these groups reads, are left as they are.  For weights that are new in every
 * call, as in gmm (atorch/kernels/extensions/grouped_gemm_exts/grouped_gemm_gmm.py:10-52).
 */
int aamd_quant_128x128_grouped(const void *w, int w_dtype, int64_t E, int64_t N, int64_t K, int64_t expert_stride,
                               const int64_t *group_offsets, uint8_t *q, float *s, uint8_t *q_t, float *s_t, float eps,
                               void *stream);

/*
 * Dequantisation y = code * scale.
 * Replaces dequant, triton_kernel.py:49-91.  tile_scale != 0: s [M, N/128]; else s [M/128, N/128].
 */
int aamd_dequant(const uint8_t *q, const float *s, int64_t M, int64_t N, int tile_scale, void *y, int y_dtype,
                 void *stream);

/*
 * SwiGLU fused into the 1x128 quantisation of the intermediate activations (the step between
 * the two grouped GEMMs of an expert MLP): for rows [a | b] of the first GEMM's output,
 *   h = bf16(bf16(silu(a)) * b)   (silu(x) = x / (1 + exp(-x)) in fp32)
 * is quantised like aamd_quant_1x128 / aamd_quant_1x128_dual_grouped would quantise h, without h
 * making a round trip through memory.
 * Replaces SwiGLUActivatition.forward, atorch/modules/moe/grouped_gemm_moe.py:331-334 (torch.chunk,
 * F.silu, multiply), as used between the gmm calls of compute_moe, :845-850, followed by the
 * per-expert quantize_op.quantize of the next grouped linear, quantized_grouped_linear.py:90-101.
 *   fc1 [rows, 2F] bf16 (row stride ld elements, ld >= 2F), F % 128 == 0
 *   h_out [rows, F] bf16 or NULL (the activation itself, for callers that keep it)
 *   q [rows, F], s [rows, F/128]; the dual form adds q_t / s_t with the layouts, scratch and
 *   group_offsets of aamd_quant_1x128_dual_grouped (q and s may then be NULL).
 */
int aamd_swiglu_quant_1x128(const void *fc1, int64_t rows, int64_t F, int64_t ld, void *h_out, uint8_t *q, float *s,
                            void *stream);
int aamd_swiglu_quant_1x128_dual_grouped(const void *fc1, int64_t M, int64_t F, int64_t ld,
                                         const int64_t *group_offsets, int E, int32_t *tile_ws, void *h_out,
                                         uint8_t *q, float *s, uint8_t *q_t, float *s_t, int64_t ld_t, int q_t_layout,
                                         void *stream);

/*
 * Backward of the gated activation fused into the quantisation of its gradient: for the gradient dh
 * of h and the saved rows [a | b], the rows [da | db] of d(fc1) are quantised 1x128 row-wise and
 * transposed inside the ragged groups without being written in bf16.
 * Replaces what autograd runs for SwiGLUActivatition.forward, atorch/modules/moe/grouped_gemm_moe.py:331-334
 * (the backward of the multiply, then silu_backward) followed by the per-expert quantize_op.quantize
 * calls of the first grouped linear's backward, quantized_grouped_linear.py:202-206.
 *   dh [M, F] bf16 (row stride ld_dh), fc1 [M, 2F] bf16 (row stride ld), F % 128 == 0
 *   g_out [M, 2F] bf16 or NULL (the gradient itself, for callers that keep it)
 *   q [M, 2F], s [M, 2F/128] (both may be NULL), q_t (2F rows), s_t [ld_t/128, 2F];
 *   group_offsets, tile_ws, ld_t, q_t_layout as for aamd_quant_1x128_dual_grouped.
 */
int aamd_swiglu_bwd_quant_1x128_dual_grouped(const void *dh, int64_t ld_dh, const void *fc1, int64_t ld, int64_t M,
                                             int64_t F, const int64_t *group_offsets, int E, int32_t *tile_ws,
                                             void *g_out, uint8_t *q, float *s, uint8_t *q_t, float *s_t,
                                             int64_t ld_t, int q_t_layout, void *stream);

/*
 * GELU, the expert MLP's default activation, fused into the same quantisers:
 *   h = bf16(x/2 * (1 + erf(x / sqrt 2)))  computed in fp32 from bf16 x, quantised like aamd_quant_1x128 /
 *   aamd_quant_1x128_dual_grouped would quantise h; with dh != NULL the dual form quantises the gradient
 *   g = bf16(dh * (cdf(x) + x * pdf(x))) instead (autograd's gelu_backward).
 * Replaces self.activation = torch.nn.functional.gelu, atorch/modules/moe/grouped_gemm_moe.py:449, applied at
 * :849 between the gmm calls, and what autograd runs for it, each followed by the per-expert
 * quantize_op.quantize of the next grouped GEMM's operand (quantized_grouped_linear.py:90-101, 202-206).
 *   x [rows, F] bf16 (row stride ld), F % 128 == 0; dh [rows, F] bf16 with the same row stride ld
 *   h_out [rows, F] bf16 or NULL (h, or g in the backward form); other arguments as the SwiGLU forms.
 */
int aamd_gelu_quant_1x128(const void *x, int64_t rows, int64_t F, int64_t ld, void *h_out, uint8_t *q, float *s,
                          void *stream);
int aamd_gelu_quant_1x128_dual_grouped(const void *x, const void *dh, int64_t M, int64_t F, int64_t ld,
                                       const int64_t *group_offsets, int E, int32_t *tile_ws, void *h_out, uint8_t *q,
                                       float *s, uint8_t *q_t, float *s_t, int64_t ld_t, int q_t_layout, void *stream);

/*
 * Ragged grouped block-scaled GEMM, "NT": for every group g and its rows m,
 *   C[m, n] = sum_kb dot(A[m, kb], B_g[n, kb]) * a_s[m, kb] * b_s_g[n/128 or n, kb]  (+ bias_g[n])
 * fp8 x fp8 MFMA, fp32 accumulation, scales applied per 128-deep block.
 * Replaces fp8_gemm / fp8_gemm_kernel, triton_kernel.py:143-210, and
 * quantize_op.grouped_qgemm for fprop and dgrad, quantized_grouped_linear.py:141-151, 214-223.
 *   a [M, K] codes (row stride lda bytes), a_s [M, K/128]
 *   b [E, N, K] codes dense, b_s [E, N/128, K/128] (b_tile_scaled == 0) or [E, N, K/128] (!= 0)
 *   group_offsets [E+1] int64 device, or NULL for a single group [0, M] (then E must be 1)
 *   c [M, N] of c_dtype (row stride ldc elements, rows 16-byte aligned); rows of empty groups are not touched
 *   bias [E, N] of bias_dtype or NULL (AAMD_NONE); tile_ws: not used; may be NULL.
 *   K % 128 == 0, N % 128 == 0.
 * The kernel is chosen by M, N, K and E, and the one for few rows adds the 128-deep blocks in another order: a row's fp32
 * sum is the same in every launch of one size, and may differ in its last bits between launches of different sizes.
 */
int aamd_grouped_gemm_fp8_nt(const uint8_t *a, int64_t lda, const float *a_s, const uint8_t *b, const float *b_s,
                             int b_tile_scaled, const int64_t *group_offsets, int E, int32_t *tile_ws, int64_t M,
                             int64_t N, int64_t K, void *c, int c_dtype, int64_t ldc, const void *bias,
                             int bias_dtype, void *stream);

/*
 * The same GEMM with the weights stored as their contraction runs down the rows, b [E, K, N] and b_s [E, K/128, N/128]
 * (block scales): C[m, n] = sum_kb dot(A[m, kb], B_g[kb, n]) * a_s[m, kb] * b_s_g[kb, n/128] (+ bias_g[n]).  The gradient of
 * the rows reads the codes of the forward product this way (and a weight stored [E, K, N] those of its own layout), so that
 * one orientation of the codes is written and kept; results are those of aamd_grouped_gemm_fp8_nt on the transposed codes,
 * bit for bit where both take the same kernel.  N < 2^23; everything else as there.
 * Replaces quantize_op.grouped_qgemm for dgrad, quantized_grouped_linear.py:214-223.
 */
int aamd_grouped_gemm_fp8_nn(const uint8_t *a, int64_t lda, const float *a_s, const uint8_t *b, const float *b_s,
                             const int64_t *group_offsets, int E, int64_t M, int64_t N, int64_t K, void *c, int c_dtype,
                             int64_t ldc, const void *bias, int bias_dtype, void *stream);

/*
 * The two GEMMs above (b_rows == 0 as _nt with block scales, else as _nn) with a workspace that lets them share out the
 * contraction of the last output tiles, where fewer of those are left than the card has units.  ws_bytes() says what a
 * launch of this size can use (0: nothing, or not expected to gain by it); ws may be NULL, is 16-byte aligned and belongs to the
 * call until it has run on the stream.  The sum of a row in such a tile is made of up to eight partial sums, added in the order
 * of the contraction.  Which tiles those are depends on the sizes of the groups, so that the last bits of a row may differ with
 * the other rows of a launch, and between a call with a workspace and one without.
 * Replaces fp8_gemm / fp8_gemm_kernel, triton_kernel.py:143-210, and quantize_op.grouped_qgemm for fprop and dgrad,
 * quantized_grouped_linear.py:141-151, 214-223, as they do.
 */
int64_t aamd_grouped_gemm_fp8_ws_bytes(int64_t M, int64_t N, int64_t K, int E, int grouped, int b_rows);
int aamd_grouped_gemm_fp8_ws(const uint8_t *a, int64_t lda, const float *a_s, const uint8_t *b, const float *b_s,
                             int b_rows, const int64_t *group_offsets, int E, int64_t M, int64_t N, int64_t K, void *c,
                             int c_dtype, int64_t ldc, const void *bias, int bias_dtype, float *ws, int64_t ws_bytes,
                             void *stream);

/*
 * Quantise and multiply in one launch, for the few rows of a decoding step: C = Q(rows) B_g^T (+ bias_g), where Q is the 1x128
 * quantiser's result (its codes and scales, which are not written) of
 *   AAMD_ROWS_PERMUTED  row j of the groups is row sorted_idx[j] / topk of `rows` [T, K] bf16, row stride ld elements
 *   AAMD_ROWS_SWIGLU    SwiGLU of `rows` [M, 2 K] bf16 (as aamd_swiglu_quant_1x128)
 *   AAMD_ROWS_GELU      GELU of `rows` [M, K] bf16 (as aamd_gelu_quant_1x128)
 * c [M, N] bf16.  It takes up to 64 rows where the GEMM of codes would use its kernel for few rows; other sizes are
 * AAMD_ERR_ARG.  _fits() says whether it does and is faster than the two launches, `most` being the most rows a group can have.
 * The results are those of the two launches, bit for bit.
 * Replaces tile_quant + grouped_qgemm, quantized_grouped_linear.py:90-101, 141-151 (and the permute in front of them,
 * token_dispatcher.py:89-116).
 */
#define AAMD_ROWS_PERMUTED 0
#define AAMD_ROWS_SWIGLU 1
#define AAMD_ROWS_GELU 2
int aamd_quant_grouped_gemm_fits(int64_t M, int64_t N, int64_t K, int E, int64_t most);
int aamd_quant_grouped_gemm_fp8_nt(int what, const void *rows, int64_t ld, const int64_t *sorted_idx, int topk, int64_t T,
                                   const uint8_t *b, const float *b_s, const int64_t *group_offsets, int E, int64_t M,
                                   int64_t N, int64_t K, void *c, int64_t ldc, const void *bias, int bias_dtype,
                                   void *stream);

/*
 * The same for permuted rows with the routing made in the launch: ids [T, topk] (int64 or int32, row-major) are the router's choices,
 * T topk at most 64 pairs; c has T topk rows, of which those of pairs with an expert in [0, E) are written.  sorted_idx [T topk],
 * row_map [T topk] and group_offsets [E+1] are outputs, what aamd_moe_preprocess gives (token_dispatcher.py:89-116).  Worth it where
 * _fits() says so.
 */
int aamd_route_quant_grouped_gemm_fits(int64_t T, int topk, int64_t N, int64_t K, int E);
int aamd_route_quant_grouped_gemm_fp8_nt(const void *ids, int ids_are_i64, int topk, int64_t T, const void *rows, int64_t ld,
                                         const uint8_t *b, const float *b_s, int E, int64_t N, int64_t K, void *c,
                                         int64_t ldc, const void *bias, int bias_dtype, int64_t *sorted_idx,
                                         int32_t *row_map, int64_t *group_offsets, void *stream);

/*
 * The second GEMM of a decoding step with the weighted combine in it: out[t] = sum over j of probs[t, j] (b[ids[t, j]] act(row_map[t, j]-th
 * of rows)), `what` AAMD_ROWS_SWIGLU or AAMD_ROWS_GELU of `rows` [T topk, 2K or K] bf16 with row stride ld; row_map [T topk] int32, negative
 * for a copy that was dropped; probs [T, topk] bf16 or fp32; out [T, N] of the type of probs.  topk at most 8, T topk at most 64.
 * The results are those of aamd_quant_grouped_gemm_fp8_nt and aamd_unpermute_combine (token_dispatcher.py:119-175), bit for bit, where
 * _fits() says that it is faster than the two.
 */
int aamd_quant_grouped_gemm_combine_fits(int64_t T, int topk, int64_t N, int64_t K, int E);
int aamd_quant_grouped_gemm_combine_fp8_nt(int what, const void *rows, int64_t ld, const void *ids, int ids_are_i64,
                                           const int32_t *row_map, const void *probs, int probs_dtype, int topk, int64_t T,
                                           const uint8_t *b, const float *b_s, int E, int64_t N, int64_t K, void *out,
                                           const void *bias, int bias_dtype, void *stream);

/*
 * aamd_grouped_gemm_fp8_nt for callers that cannot allocate device memory (code under HIP graph
 * capture, tight serving loops, harnesses that forbid hipMalloc): the same arguments without
 * tile_ws.  No counterpart in the reference.  The call allocates and
 * frees nothing; E > AAMD_STATIC_MAX_GROUPS is rejected with AAMD_ERR_ARG.
 */
#define AAMD_STATIC_MAX_GROUPS 4096
int aamd_grouped_gemm_fp8_nt_static(const uint8_t *a, int64_t lda, const float *a_s, const uint8_t *b,
                                    const float *b_s, int b_tile_scaled, const int64_t *group_offsets, int E,
                                    int64_t M, int64_t N, int64_t K, void *c, int c_dtype, int64_t ldc,
                                    const void *bias, int bias_dtype, void *stream);

/*
 * Grouped weight-gradient GEMM: dW_g[n, k] (+)= sum over the tokens m of group g of
 * dY[m, n] * X[m, k], both operands 1x128-scaled along the tokens (layouts of
 * aamd_quant_1x128_dual_grouped's q_t / s_t).
 * Replaces quantize_op.grouped_qgemm(qdy_t, qx_t, mm_wgrad, ..., accumulate=...),
 * quantized_grouped_linear.py:243-253.
 *   dyt (N rows), sdyt [ld_t/128, N]; xt (K rows), sxt [ld_t/128, K]; both code operands in the layout
 *   q_t_layout names (AAMD_QT_ROWS: [N, ld_t] and [K, ld_t]; AAMD_QT_BLOCKED: [ld_t/128, N, 128] and
 *   [ld_t/128, K, 128])
 *   dw [E, N, K] of dw_dtype (expert stride in elements); an empty group gives zeros,
 *   or leaves dw_g untouched when accumulate != 0.
 *   group_offsets NULL: one group over all ld_t tokens (then E must be 1).
 *   ld_t must cover the padded token total sum_g ceil(M_g/128)*128, which only the device knows:
 *   a group whose tokens lie beyond ld_t gets NaN in its dw_g instead of a wrong finite gradient.
 */
int aamd_grouped_gemm_fp8_wgrad(const uint8_t *dyt, const float *sdyt, const uint8_t *xt, const float *sxt,
                                int64_t ld_t, int q_t_layout, const int64_t *group_offsets, int E, int32_t *tile_ws,
                                int64_t N, int64_t K, void *dw, int dw_dtype, int64_t expert_stride, int accumulate,
                                void *stream);

/*
 * Inverse permutation + weighted combine in one gather-reduce pass:
 *   out[t, :] = sum_j probs[t, j] * y[row_map[t*topk + j], :]
 * Replaces unpermute, token_dispatcher.py:119-161 (zeros + index_copy_ + multiply + sum).
 * Each product is rounded to the promoted dtype before the fp32 sum, as the reference's
 * separate multiply and sum do (:156-159); the sum adds in the order of torch's GPU reduction
 * (slot j into accumulator j mod 4, then ((a0 + a1) + a2) + a3).
 *   y [M, H] of y_dtype (bf16 or fp32); row_map [T*topk] int32 (-1 = dropped copy, contributes 0)
 *   probs [T, topk] of probs_dtype, or AAMD_NONE (probs ignored); out [T, H] has the promoted type of
 *   rows and probs: bf16 for bf16 rows with bf16 or no probs, fp32 otherwise; H % 8 == 0.
 */
int aamd_unpermute_combine(const void *y, int y_dtype, int64_t M, int64_t H, const int32_t *row_map,
                           const void *probs, int probs_dtype, int64_t T, int topk, void *out, void *stream);

/*
 * The two gradients of that combine, as autograd derives them from the reference's torch ops
 * (token_dispatcher.py:155-159: index_copy_, multiply by probs, sum over topk):
 *   permute_rows_scaled: d_y[row_map[t*topk+j], :] = (out_dtype)(d_out[t, :] * probs[t, j]), the product
 *     formed in fp32 and rounded once; with probs_dtype == AAMD_NONE it is the plain permute with a
 *     conversion.  x [T, cols] of x_dtype, out [M_out, cols] of out_dtype (bf16 -> bf16, fp32 -> bf16,
 *     fp32 -> fp32); cols % 8 == 0; rows no map entry points to are not written.
 *   unpermute_probs_grad: d_probs[t, j] = sum_h d_out[t, h] * y[row_map[t*topk+j], h] in fp32
 *     (0 for a dropped copy); d_probs [T, topk] fp32, the caller casts.
 */
int aamd_permute_rows_scaled(const void *x, int x_dtype, int64_t T, int64_t cols, const int32_t *row_map, int topk,
                             const void *probs, int probs_dtype, int64_t M_out, void *out, int out_dtype,
                             void *stream);
int aamd_unpermute_probs_grad(const void *dout, int dout_dtype, const void *y, int y_dtype, int64_t M, int64_t H,
                              const int32_t *row_map, int64_t T, int topk, float *dprobs, void *stream);
/* The same in the weights' type (autograd of token_dispatcher.py:156), bf16 or fp32; bf16 needs M > 0. */
int aamd_unpermute_probs_grad_as(const void *dout, int dout_dtype, const void *y, int y_dtype, int64_t M, int64_t H,
                                 const int32_t *row_map, int64_t T, int topk, void *dprobs, int dprobs_dtype, void *stream);

/*
 * The dual quantiser of a gradient that also leaves the column sums of its 128-token tiles, and the sums of those over
 * the groups: a bias gradient without another pass over the gradient (and, where the quantiser computes it, without
 * writing it).  Replaces the row sums per expert beside the quantisation: bias_gather_add_bw
 * (atorch/kernels/triton_jit/bias_gather_add.py:101-127), quantized_grouped_linear.py:84-86, 201.
 *   what: AAMD_SUMS_PLAIN      the bf16 gradient itself, x [M, width]
 *         AAMD_SUMS_GELU_BWD   dh gelu'(x) of x, dh [M, width] bf16
 *         AAMD_SUMS_SWIGLU_BWD [da | db] of x = [a | b] [M, width], dh [M, width/2] bf16
 *   q, s, q_t, s_t, ld_t, q_t_layout as for aamd_quant_1x128_dual_grouped with cols = width; eps 0 but for PLAIN
 *   tile_sums [ld_t/128, width] fp32: row p/128 holds the sums of the tile at padded token p; rows of no tile are not
 *   written
 *   aamd_group_sums: out [E, cols] of out_dtype = sums of tile_sums over each group's tiles (0 for an empty group)
 */
#define AAMD_SUMS_PLAIN 0
#define AAMD_SUMS_SWIGLU_BWD 1
#define AAMD_SUMS_GELU_BWD 2
int aamd_dual_grouped_with_sums(int what, const void *x, const void *dh, int64_t M, int64_t width,
                                const int64_t *group_offsets, int E, uint8_t *q, float *s, uint8_t *q_t, float *s_t,
                                int64_t ld_t, int q_t_layout, float eps, float *tile_sums, void *stream);
int aamd_group_sums(const float *tile_sums, int64_t cols, const int64_t *group_offsets, int E, void *out, int out_dtype,
                    void *stream);

/*
 * Scales [rows, blocks] (row-major, as the dense GEMM's callers hold them, triton_kernel.py:198-210) to the block-major
 * [blocks, rows] that the weight-gradient GEMM reads.
 */
int aamd_transpose_scales(const float *s, int64_t rows, int64_t blocks, float *s_t, void *stream);
/* Two of them, with as many blocks, in one launch (triton_kernel.py:198-210 as above); no size is zero. */
int aamd_transpose_scales_pair(const float *a, int64_t rows_a, float *a_t, const float *b, int64_t rows_b, float *b_t,
                               int64_t blocks, void *stream);

/*
 * Both gradients of the combine in one pass: drows[row_map[t*topk+j]] = dout[t] * probs[t, j] rounded to the rows'
 * type, dprobs[t, j] = sum_h dout[t, h] * y[row_map[t*topk+j], h] (fp32 sums) in the weights' type, 0 for a dropped
 * copy.  What autograd makes of token_dispatcher.py:155-159.
 *   dout [T, H] of the combine's result type (fp32 if rows or weights are), y and drows [M, H] of y_dtype, probs and
 *   dprobs [T, topk] of probs_dtype; rows of drows no map entry points to are not written.
 */
int aamd_unpermute_backward(const void *dout, int dout_dtype, const void *y, int y_dtype, int64_t M, int64_t H,
                            const int32_t *row_map, const void *probs, int probs_dtype, int64_t T, int topk,
                            void *drows, void *dprobs, void *stream);

/*
 * group_offsets [E+1] int64 (device) = exclusive prefix of counts [E] int64, rows per group.  counts_on_host != 0:
 * counts is host memory, read before the call returns, and nothing waits for the device.
 * Replaces the cumulative sums and host copies around the grouped calls (grouped_gemm_moe.py:837,
 * quantized_grouped_linear.py:90-101).
 */
int aamd_group_offsets(const int64_t *counts, int counts_on_host, int E, int64_t *group_offsets, void *stream);

/*
 * Router preprocess on the device, no host round trip: histogram of expert ids,
 * exclusive scan, stable counting sort.
 * Replaces the argsort of permute (token_dispatcher.py:107-112) and the histc + .cpu()
 * of MoEAllToAllTokenDispatcher.preprocess (token_dispatcher.py:297-353).
 *   expert_ids [n] (n = T*topk; int64 when ids_are_i64 != 0, else int32), values in [0, E)
 *   sorted_idx [n] int64: flat index of permuted row j (the reference's sorted_indices); may be NULL
 *   row_map [n] int32: permuted row of flat index i (inverse of sorted_idx)
 *   group_offsets [E+1] int64: exclusive prefix of tokens per expert
 *   ws: aamd_moe_preprocess_ws_ints(n, E) int32 of scratch.
 */
int64_t aamd_moe_preprocess_ws_ints(int64_t n, int E);
int aamd_moe_preprocess(const void *expert_ids, int ids_are_i64, int64_t n, int E, int64_t *sorted_idx,
                        int32_t *row_map, int64_t *group_offsets, int32_t *ws, void *stream);

/*
 * row_map[sorted_idx[j]] = j for j < n_perm, -1 elsewhere (n_flat entries).
 * Adapter from the reference's sorted_indices (token_dispatcher.py:112,136) to row_map.
 */
int aamd_invert_permutation(const int64_t *sorted_idx, int64_t n_perm, int64_t n_flat, int32_t *row_map,
                            void *stream);

/*
 * Per-expert bias on rows tagged with their expert: out[t, :] = inp[t, :] + bias[bin_ids[t], :]
 * (bf16: the fp32 sum rounded to bf16), and its bias gradient bgrad[e, :] = sum of grad[t, :] over
 * the rows with bin_ids[t] == e, accumulated in fp32 (order of the additions unspecified, as with
 * the reference's atomic adds; the caller casts to the gradient's dtype).
 * Replaces bias_gather_add_fw / bias_gather_add_bw, atorch/kernels/triton_jit/bias_gather_add.py:50-66, 101-127.
 *   inp, out, grad [T, H] and bias [E, H] of `dtype`; H * sizeof(dtype) % 16 == 0
 *   bin_ids [T]: int64 when ids_are_i64 != 0, else int32; rows tagged outside [0, E) pass through
 *   unchanged and add nothing to bgrad
 *   bgrad [E, H] fp32, cleared by the call.
 */
int aamd_bias_gather_add(const void *inp, const void *bias, const void *bin_ids, int ids_are_i64, int64_t T,
                         int64_t H, int E, int dtype, void *out, void *stream);
int aamd_bias_gather_add_bgrad(const void *grad, const void *bin_ids, int ids_are_i64, int64_t T, int64_t H, int E,
                               int dtype, float *bgrad, void *stream);

#pragma GCC visibility pop
#ifdef __cplusplus
}
#endif
#endif /* ATORCH_AMD_FP8_H */

/*
 * C-ABI of libpithtrain_hip.so: hand-written gfx950 kernels for PithTrain's FP8
 * grouped-expert path.  Plain pointers and sizes only; every pointer is a device
 * pointer unless it says "host".  All launches go to `stream` (a hipStream_t passed
 * as void*); nothing here synchronises, allocates or frees device memory.
 *
 * Return value: 0 on success, negative PT_ERR_* otherwise; pt_last_error() gives a
 * thread-local message for the last failure.
 *
 * Each entry point names the reference interface it replaces
 * (paths relative to the PithTrain source tree).
 */
#ifndef PITHTRAIN_HIP_H
#define PITHTRAIN_HIP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef void* pt_stream_t;

enum { PT_OK = 0, PT_ERR_INVALID = -1, PT_ERR_LAUNCH = -2, PT_ERR_UNSUPPORTED = -3 };
/* element types of bf16/fp32/fp16 tensors */
enum { PT_BF16 = 0, PT_F32 = 1, PT_F16 = 2 };

const char* pt_last_error(void);
int pt_abi_version(void);

/* ------------------------------------------------------------------------------------------
 * Blockwise FP8 (e4m3fn) quantisation, power-of-two fp32 scales.
 * Replaces pithtrain/operators/deepgemm_quantize.py (six Triton kernels).
 * x is [M,N] with row stride ldx (elements) and unit column stride; dtype PT_BF16, PT_F16 or
 * PT_F32 (the reference's kernels load any float type and convert to fp32,
 * deepgemm_quantize.py:141-152).
 * ------------------------------------------------------------------------------------------ */

/* layout of the colwise twin written by pt_quant_rowwise_colwise */
enum {
  PT_CH_ROWMAJOR = 0,  /* ch_fp8[M,N],  ch_scale[M/128,N]   fp8cast_rowwise_colwise :204-259 */
  PT_CH_TRANSPOSED = 1,/* ch_fp8[N,M],  ch_scale[M/128,N]   (layout of this library's wgrad GEMM) */
  PT_CH_KMAJOR = 2     /* flat per-group (N,K_g) blocks, ch_scale[N,M/128]  fp8cast_rowwise_kmajor :262-333 */
};

/* 1x128 rowwise + 128-row colwise from one read.  M % 128 == 0 (deepgemm_quantize.py:219).
 * offs/num_groups (int32 inclusive row offsets, multiples of 128) give the PT_CH_KMAJOR layout its
 * groups.  For every layout, when offs is given, offs[num_groups-1] is the number of rows that
 * are quantised: M may then be an upper bound known on the host (buffers sized for the largest
 * row count a routing can produce) while the real count stays in device memory, and row tiles at
 * or past it are left untouched.  Without offs all M rows are quantised. */
int pt_quant_rowwise_colwise(const void* x, int dtype, int64_t M, int64_t N, int64_t ldx,
                             void* tok_fp8, float* tok_scale, void* ch_fp8, float* ch_scale,
                             int ch_layout, const int32_t* offs, int32_t num_groups,
                             pt_stream_t stream);
/* The same (PT_CH_TRANSPOSED, all M rows) with tok_scale [ceil(N/128), M], as pt_gemm_m_grouped_by_block reads it. */
int pt_quant_rowwise_colwise_by_block(const void* x, int dtype, int64_t M, int64_t N, int64_t ldx, void* tok_fp8,
                                      float* tok_scale, void* ch_t_fp8, float* ch_scale, pt_stream_t stream);

/* pt_quant_rowwise_colwise on gathered rows: output row r is quantised from source row
 * row_index[r] of x (a negative index gives an all-zero row: zero bytes, the scale of amax 0).
 * M counts output rows.  With row_index = the scatter's source map this is
 * fp8cast_rowwise_colwise(scatter_for_grouped_gemm(x)) without materialising the permuted bf16
 * copy (token_scatter.py:103-153 followed by deepgemm_quantize.py:204-259). */
int pt_quant_rowwise_colwise_rows(const void* x, int dtype, int64_t M, int64_t N, int64_t ldx,
                                  const int32_t* row_index, void* tok_fp8, float* tok_scale,
                                  void* ch_fp8, float* ch_scale, int ch_layout,
                                  const int32_t* offs, int32_t num_groups, pt_stream_t stream);

/* pt_quant_rowwise_colwise_rows with row r read from x[row_index[r] / repeat]: x [rows, N] holds one row per
 * token and routed row i is token i / repeat (the expand of the models' reference_forward,
 * qwen3_moe.py:104-108, without the copies).  rows * repeat^2 < 2^32. */
int pt_quant_rowwise_colwise_rows_repeat(const void* x, int64_t rows, int64_t repeat, int dtype, int64_t M,
                                         int64_t N, int64_t ldx, const int32_t* row_index,
                                         void* tok_fp8, float* tok_scale, void* ch_fp8, float* ch_scale,
                                         int ch_layout, const int32_t* offs, int32_t num_groups,
                                         pt_stream_t stream);

/* The transposed / column-scaled results (ch_fp8, ch_scale) of the row-scaled quantisers above and of the
 * fused SwiGLU forwards below may be left out (both NULL) when no backward reads them. */

/* SwiGLU fused into the activation quantisation (bf16 only).  Forward: h = bf16(silu(gate) * up)
 * with gate = gate_up[:, :half], up = gate_up[:, half:], quantised as pt_quant_rowwise_colwise
 * with the PT_CH_TRANSPOSED twin: tok_fp8[M,half], tok_scale[M,ceil(half/128)], ch_t_fp8[half,M],
 * ch_scale[M/128,half].  Same bits as silu_mul (silu_mul.py:28-49) followed by
 * fp8cast_rowwise_colwise (deepgemm_quantize.py:204-259); h itself is never written.
 * valid_rows (optional, device): *valid_rows rows are processed, the row tiles past them are left
 * untouched (M is then the host-side upper bound the buffers are sized for). */
int pt_silu_mul_quant_rowwise_colwise(const void* gate_up, int64_t M, int64_t half,
                                      int64_t ld_gate_up, void* tok_fp8, float* tok_scale,
                                      void* ch_t_fp8, float* ch_scale, const int32_t* valid_rows,
                                      pt_stream_t stream);
/* Backward twin: [dgate | dup] = silu_mul backward (silu_mul.py:52-87) of grad_h[M,half] at the
 * saved gate_up[M,2*half], rounded to bf16 and quantised to tok_fp8[M,2*half],
 * tok_scale[M,ceil(2*half/128)], ch_t_fp8[2*half,M], ch_scale[M/128,2*half]. */
int pt_silu_mul_bwd_quant_rowwise_colwise(const void* grad_h, int64_t ld_grad_h,
                                          const void* gate_up, int64_t ld_gate_up, int64_t M,
                                          int64_t half, void* tok_fp8, float* tok_scale,
                                          void* ch_t_fp8, float* ch_scale, const int32_t* valid_rows,
                                          pt_stream_t stream);
/* The same pair in the scalings of the dense linears, for any M: forward h as
 * pt_quant_rowwise_blockwise_transpose_ld (blk_t_fp8 and blk_t_scale may both be NULL), backward
 * [dgate | dup] as pt_quant_rowwise_transpose_ld, half a multiple of 128. */
int pt_silu_mul_quant_rowwise_blockwise_transpose_ld(const void* gate_up, int64_t M, int64_t half,
                                                     int64_t ld_gate_up, void* tok_fp8, float* tok_scale,
                                                     void* blk_t_fp8, int64_t ld_t, float* blk_t_scale,
                                                     pt_stream_t stream);
int pt_silu_mul_bwd_quant_rowwise_transpose_ld(const void* grad_h, int64_t ld_grad_h, const void* gate_up,
                                               int64_t ld_gate_up, int64_t M, int64_t half, void* tok_fp8,
                                               float* tok_scale, void* t_fp8, int64_t ld_t, float* t_scale,
                                               pt_stream_t stream);
/* The same pair for the clamped SwiGLU of GPT-OSS (interleaved (gate, up) pairs, alpha, limit):
 * quantises h = clamped_swiglu(gate_up[M,2*half]) (clamped_swiglu.py:18-46) as
 * fp8cast_rowwise_colwise (deepgemm_quantize.py:204-259) would, without writing h:
 * tok_fp8[M,half], tok_scale[M,ceil(half/128)], ch_t_fp8[half,M], ch_scale[M/128,half]. */
int pt_clamped_swiglu_quant_rowwise_colwise(const void* gate_up, int64_t M, int64_t half,
                                            int64_t ld_gate_up, float alpha, float limit,
                                            void* tok_fp8, float* tok_scale, void* ch_t_fp8,
                                            float* ch_scale, const int32_t* valid_rows,
                                            pt_stream_t stream);
/* Backward twin: the gradient of gate_up in its interleaved layout (clamped_swiglu.py:49-89) from
 * grad_h[M,half], rounded to bf16 and quantised to tok_fp8[M,2*half], tok_scale[M,ceil(2*half/128)],
 * ch_t_fp8[2*half,M], ch_scale[M/128,2*half].  col_sum[M/128, 2*half] (fp32) receives the column
 * sums of every 128-row tile of the bf16 gradient: summed over a group's tiles (pt_segment_sum
 * with the group ends divided by 128) they are the bias gradient that _segment_sum_kernel
 * (indexed_bias_add.py:20-51) computes from the materialised gradient. */
int pt_clamped_swiglu_bwd_quant_rowwise_colwise(const void* grad_h, int64_t ld_grad_h,
                                                const void* gate_up, int64_t ld_gate_up, int64_t M,
                                                int64_t half, float alpha, float limit,
                                                void* tok_fp8, float* tok_scale, void* ch_t_fp8,
                                                float* ch_scale, float* col_sum,
                                                const int32_t* valid_rows, pt_stream_t stream);

/* rowwise(x) + rowwise(x^T): t_fp8[N,M], t_scale[N,ceil(M/128)].
 * fp8cast_rowwise_transpose, deepgemm_quantize.py:429-482 */
int pt_quant_rowwise_transpose(const void* x, int dtype, int64_t M, int64_t N, int64_t ldx,
                               void* tok_fp8, float* tok_scale, void* t_fp8, float* t_scale,
                               pt_stream_t stream);
/* The same with a row pitch ld_t >= M (bytes) for t_fp8: a reduction over all tokens reads the
 * transposed operand along rows, and a power-of-two pitch (M = 8192, 32768 tokens) puts those rows
 * on few memory channels.  A pitch that is a multiple of 16 and at least M rounded up to 16 also gets
 * the columns from M to there filled with zeros (a reduction in 16-byte chunks reads them).  No
 * counterpart in the reference (its transposed outputs are packed). */
int pt_quant_rowwise_transpose_ld(const void* x, int dtype, int64_t M, int64_t N, int64_t ldx,
                                  void* tok_fp8, float* tok_scale, void* t_fp8, int64_t ld_t,
                                  float* t_scale, pt_stream_t stream);

/* The same of a bf16 matrix [M, heads * (head_a + head_b)] given as two packed tensors x [M, heads, head_a] and
 * x2 [M, heads, head_b] (dK and dV of an attention's latent projection, ring_attention.py:636-652)
 * instead of their concatenation per head.  Head widths are multiples of 8. */
int pt_quant_heads_rowwise_transpose_ld(const void* x, const void* x2, int64_t M, int64_t heads,
                                        int64_t head_a, int64_t head_b, void* tok_fp8, float* tok_scale,
                                        void* t_fp8, int64_t ld_t, float* t_scale, pt_stream_t stream);

/* The same and pt_quant_rowwise_blockwise_transpose_ld's transposed results alone of a bf16 input [M, K] (row stride
 * ld_input, the same ld_t), in one launch: what the backward of a latent projection quantises. */
int pt_quant_heads_and_input(const void* x, const void* x2, int64_t M, int64_t heads, int64_t head_a, int64_t head_b,
                             void* tok_fp8, float* tok_scale, void* t_fp8, int64_t ld_t, float* t_scale,
                             const void* input, int64_t K, int64_t ld_input, void* blk_t_fp8, float* blk_t_scale,
                             pt_stream_t stream);

/* rowwise(x) + 128x128 blockwise(x^T): blk_t_fp8[K,M], blk_t_scale[ceil(K/128),ceil(M/128)].
 * fp8cast_rowwise_blockwise_transpose, deepgemm_quantize.py:575-629 */
int pt_quant_rowwise_blockwise_transpose(const void* x, int dtype, int64_t M, int64_t K,
                                         int64_t ldx, void* tok_fp8, float* tok_scale,
                                         void* blk_t_fp8, float* blk_t_scale, pt_stream_t stream);
/* The same with a row pitch ld_t >= M (bytes) for blk_t_fp8 (see pt_quant_rowwise_transpose_ld).  One of
 * the two results may be left out (NULL for its bytes and scales). */
int pt_quant_rowwise_blockwise_transpose_ld(const void* x, int dtype, int64_t M, int64_t K,
                                            int64_t ldx, void* tok_fp8, float* tok_scale,
                                            void* blk_t_fp8, int64_t ld_t, float* blk_t_scale,
                                            pt_stream_t stream);

/* pt_quant_rowwise_blockwise_transpose_ld of x [M, K] and pt_quant_blockwise_transpose_batched of up to
 * PT_QUANT_DENSE_MAX weights, all in dtype (bf16 or fp32): one launch, or two when x has more than
 * PT_QUANT_DENSE_INPUT_TILES 128 x 128 tiles.  fp8_t and scale_t of a weight have row pitches t_ld and
 * scale_t_ld (weights side by side in one transposed operand).  blk_t_fp8 and blk_t_scale may both be NULL. */
#define PT_QUANT_DENSE_MAX 3
#define PT_QUANT_DENSE_INPUT_TILES 512
typedef struct {
  const void* w; int64_t N, K, ldw;
  void* fp8; float* scale;
  void* fp8_t; int64_t t_ld; float* scale_t; int64_t scale_t_ld;
} pt_quant_dense_weight;
int pt_quant_dense_operands(const pt_quant_dense_weight* weights /* host */, int32_t n, const void* x,
                            int dtype, int64_t M, int64_t K, int64_t ldx, void* tok_fp8, float* tok_scale,
                            void* blk_t_fp8, int64_t ld_t, float* blk_t_scale, pt_stream_t stream);
/* The same for one weight w [N, K]. */
int pt_quant_linear_operands(const void* x, const void* w, int dtype, int64_t M, int64_t N, int64_t K,
                             int64_t ldx, int64_t ldw, void* tok_fp8, float* tok_scale, void* blk_t_fp8,
                             int64_t ld_t, float* blk_t_scale, void* w_fp8, float* w_scale,
                             void* w_t_fp8, float* w_t_scale, pt_stream_t stream);

/* 128x128 blockwise(x) + blockwise(x^T) for x[G,N,K] (element strides stride_g, stride_row):
 * fp8[G,N,K], scale[G,ceil(N/128),ceil(K/128)], fp8_t[G,K,N], scale_t[G,ceil(K/128),ceil(N/128)].
 * fp8cast_blockwise_transpose (:709-756, G == 1) and fp8cast_blockwise_transpose_batched
 * (:846-899).  fp8_t and scale_t may both be NULL: then only fp8 and scale are written (the
 * transposed twin holds the same bytes and the transposed scale grid, and pt_gemm_m_grouped_nn
 * reads the forward layout directly). */
int pt_quant_blockwise_transpose_batched(const void* x, int dtype, int64_t G, int64_t N, int64_t K,
                                         int64_t stride_g, int64_t stride_row, void* fp8,
                                         float* scale, void* fp8_t, float* scale_t,
                                         pt_stream_t stream);
/* Several weights (up to PT_QUANT_WEIGHTS_MAX, one dtype) quantised in their forward layout by one launch:
 * the projections of an expert block after an optimizer step.  x [G, N, K] with strides in elements;
 * fp8 [G, N, K] and scale [G, ceil(N/128), ceil(K/128)] may be slices of larger tensors (group strides
 * in bytes and in floats).  All fields are 8 bytes wide. */
#define PT_QUANT_WEIGHTS_MAX 4
typedef struct {
  const void* x;
  int64_t G, N, K, stride_g, stride_row;
  void* fp8; int64_t fp8_stride_g;
  float* scale; int64_t scale_stride_g;
} pt_quant_weight;
int pt_quant_weights(const pt_quant_weight* parts /* host */, int32_t n, int dtype, pt_stream_t stream);

/* The same into slices of larger outputs: group strides for fp8 / scale, and for the transposed
 * twin its row pitch t_ld (>= N), group stride, and the row length scale_t_ld of its scale grid.
 * Separate gate and up weights are quantised into one fused [G, 2I, K] operand this way (the up
 * half starts I rows, i.e. I*K bytes / I columns of the twin, further in). */
int pt_quant_blockwise_transpose_batched_into(const void* x, int dtype, int64_t G, int64_t N,
                                              int64_t K, int64_t stride_g, int64_t stride_row,
                                              void* fp8, int64_t fp8_stride_g, float* scale,
                                              int64_t scale_stride_g, void* fp8_t, int64_t t_ld,
                                              int64_t t_stride_g, float* scale_t,
                                              int64_t scale_t_ld, int64_t scale_t_stride_g,
                                              pt_stream_t stream);

/* ------------------------------------------------------------------------------------------
 * FP8 GEMMs (fp32 accumulate on the MFMA units, scales applied in hardware as E8M0).
 * Replace the DeepGEMM call sites of pithtrain/operators/linear.py and grouped_linear.py.
 * ------------------------------------------------------------------------------------------ */

/* out[m,n] = sum_k a[m,k] b[n,k];  a_scale[M,ceil(K/128)] (1x128), b_scale[ceil(N/128),ceil(K/128)]
 * (128x128).  out is bf16 [M,N] (out_dtype PT_BF16) or fp32 (PT_F32).
 * deep_gemm.fp8_fp4_gemm_nt at linear.py:40 (forward :57, dgrad :77, wgrad :80). */
int pt_gemm_nt_dense(const void* a_fp8, const float* a_scale, const void* b_fp8,
                     const float* b_scale, void* out, int out_dtype, int64_t M, int64_t N,
                     int64_t K, pt_stream_t stream);
/* The same for operands with row pitches lda, ldb >= K (bytes, multiples of 16): the padded
 * transposed operands of pt_quant_rowwise_transpose_ld / pt_quant_rowwise_blockwise_transpose_ld. */
int pt_gemm_nt_dense_ld(const void* a_fp8, int64_t lda, const float* a_scale, const void* b_fp8,
                        int64_t ldb, const float* b_scale, void* out, int out_dtype, int64_t M,
                        int64_t N, int64_t K, pt_stream_t stream);
/* Two products in the form of pt_gemm_nt_dense_ld that do not depend on each other (the input and the weight
 * gradient of a dense linear, linear.py:77-80), in one launch where they are small.  All fields are 8
 * bytes wide. */
typedef struct {
  const void* a_fp8; int64_t lda; const float* a_scale;
  const void* b_fp8; int64_t ldb; const float* b_scale;
  void* out;
  int64_t M, N, K;
} pt_dense_gemm;
int pt_gemm_nt_dense_pair(const pt_dense_gemm* two /* host, [2] */, int out_dtype, pt_stream_t stream);

/* pt_gemm_nt_dense (packed operands, bf16 result) whose columns go to two tensors, head by head: result
 * column h * (head_a + head_b) + c is out[:, h * head_a + c] for c < head_a and
 * out2[:, h * head_b + c - head_a] behind it; out [M, heads * head_a], out2 [M, heads * head_b] packed.
 * out2 lies behind out in one allocation, together below 2 GiB; head widths are multiples of 8.
 * The kv split of the MLA decompression (operators/ring_attention.py:428-457) without its copy. */
int pt_gemm_nt_dense_heads(const void* a_fp8, const float* a_scale, const void* b_fp8, const float* b_scale,
                           void* out, void* out2, int64_t head_a, int64_t head_b, int64_t M, int64_t N,
                           int64_t K, pt_stream_t stream);
/* Split-K form of pt_gemm_nt_dense for outputs with too few 256 x 256 tiles to fill the GPU (the
 * weight gradient of a dense linear, linear.py:61-83: M, N = weight dims, K = tokens): the
 * reduction is cut into `splits` ranges of split_len (a multiple of 128), range s is reduced into
 * the fp32 slab partial[s] ([splits, M, N], caller-provided), and pt_sum_partials adds the slabs
 * in the order of s and stores the sum as out_dtype (n = M * N, a multiple of 8). */
int pt_gemm_nt_dense_splitk(const void* a_fp8, const float* a_scale, const void* b_fp8,
                            const float* b_scale, float* partial, int32_t splits, int64_t split_len,
                            int64_t M, int64_t N, int64_t K, pt_stream_t stream);
int pt_gemm_nt_dense_splitk_ld(const void* a_fp8, int64_t lda, const float* a_scale,
                               const void* b_fp8, int64_t ldb, const float* b_scale, float* partial,
                               int32_t splits, int64_t split_len, int64_t M, int64_t N, int64_t K,
                               pt_stream_t stream);
int pt_sum_partials(const float* partial, int32_t splits, int64_t n, void* out, int out_dtype,
                    pt_stream_t stream);

/* Rows [offs[g-1], offs[g]) of a[M,K] use b[g] of b[G,N,K]; every offs[g] is a multiple of 128.
 * Rows at or past offs[G-1] are not written.  out bf16 [M,N].
 * deep_gemm.m_grouped_fp8(_fp4)_gemm_nt_contiguous at grouped_linear.py:88-101 (forward :146-154,
 * dgrad :192-200). */
int pt_gemm_m_grouped_nt(const void* a_fp8, const float* a_scale, const void* b_fp8,
                         const float* b_scale, void* out, int out_dtype, const int32_t* offs,
                         int32_t num_groups, int64_t M, int64_t N, int64_t K, pt_stream_t stream);

/* pt_gemm_m_grouped_nt whose result row r is written to out[out_row_index[r], :] (negative
 * index: the row is dropped); out is bf16 [out_rows, N], N % 8 == 0.  With out_row_index = the
 * scatter's source map this is padded_index_gather(gemm(...), reverse) - the un-permute of
 * token_scatter.py:297-309 (forward) or ScatterForGroupedGemm.backward (:271-284, dgrad) -
 * without the intermediate [M, N] tensor. */
int pt_gemm_m_grouped_nt_scatter(const void* a_fp8, const float* a_scale, const void* b_fp8,
                                 const float* b_scale, void* out, int out_dtype,
                                 const int32_t* offs, int32_t num_groups, int64_t M, int64_t N,
                                 int64_t K, const int32_t* out_row_index, int64_t out_rows,
                                 pt_stream_t stream);

/* pt_gemm_m_grouped_nt and its _scatter / _bias forms (out_row_index, bias: may be NULL) for groups of a few
 * rows each: every offs[g] is a multiple of 64 only, so that less padding is computed (a forward
 * without a backward, whose groups need not be whole 128-row scale blocks). */
int pt_gemm_m_grouped_nt_few_rows(const void* a_fp8, const float* a_scale, const void* b_fp8,
                                  const float* b_scale, void* out, int out_dtype, const int32_t* offs,
                                  int32_t num_groups, int64_t M, int64_t N, int64_t K,
                                  const int32_t* out_row_index, int64_t out_rows, const void* bias,
                                  pt_stream_t stream);

/* pt_gemm_m_grouped_nt with the b operand given reduction-major: b[g] is [K, N] (K = the reduction,
 * row pitch N, N % 16 == 0) with scales [ceil(K/128), ceil(N/128)], i.e. a weight and its
 * 128 x 128 block scales as the forward pass stores them, read by the input-gradient GEMM
 * dX = dY W without the transposed FP8 copy of W that the call at grouped_linear.py:192-200 is given
 * (made by fp8cast_blockwise_transpose_batched, deepgemm_quantize.py:419-456).  Same products, same
 * order of accumulation, same bits as pt_gemm_m_grouped_nt on the transposed operand.  The _scatter
 * form stores result row r to out[out_row_index[r], :] like pt_gemm_m_grouped_nt_scatter. */
int pt_gemm_m_grouped_nn(const void* a_fp8, const float* a_scale, const void* b_fp8,
                         const float* b_scale, void* out, int out_dtype, const int32_t* offs,
                         int32_t num_groups, int64_t M, int64_t N, int64_t K, pt_stream_t stream);
int pt_gemm_m_grouped_nn_scatter(const void* a_fp8, const float* a_scale, const void* b_fp8,
                                 const float* b_scale, void* out, int out_dtype,
                                 const int32_t* offs, int32_t num_groups, int64_t M, int64_t N,
                                 int64_t K, const int32_t* out_row_index, int64_t out_rows,
                                 pt_stream_t stream);
/* The same products from a_scale [ceil(K/128), M]: b as pt_gemm_m_grouped_nt has it, or with b_reduction_major != 0 as
 * pt_gemm_m_grouped_nn; stored through out_row_index (with out_rows) when that is not NULL. */
int pt_gemm_m_grouped_by_block(const void* a_fp8, const float* a_scale, const void* b_fp8, const float* b_scale,
                               int b_reduction_major, void* out, int out_dtype, const int32_t* offs, int32_t num_groups,
                               int64_t M, int64_t N, int64_t K, const int32_t* out_row_index, int64_t out_rows,
                               pt_stream_t stream);
/* The same stored to two outputs: result row r to row out_row_index[r] of out (out_rows rows), an index of -2 - i to row i
 * of out2 (out2_rows rows), -1 nowhere.  The index is not checked against out_rows and out2_rows on the device. */
int pt_gemm_m_grouped_by_block_two(const void* a_fp8, const float* a_scale, const void* b_fp8, const float* b_scale,
                                   int b_reduction_major, void* out, void* out2, int out_dtype, const int32_t* offs,
                                   int32_t num_groups, int64_t M, int64_t N, int64_t K, const int32_t* out_row_index,
                                   int64_t out_rows, int64_t out2_rows, pt_stream_t stream);

/* pt_gemm_m_grouped_nt followed by `out + bias[group of the row]` in the output type (the result
 * is rounded to bf16, then the bias row of its group is added and the sum rounded again): the
 * grouped linear and the indexed_bias_add after it (models/gpt_oss.py:151-156,
 * indexed_bias_add.py:100-104) as one kernel.  bias is [G,N] bf16; N % 8 == 0. */
int pt_gemm_m_grouped_nt_bias(const void* a_fp8, const float* a_scale, const void* b_fp8,
                              const float* b_scale, void* out, int out_dtype, const int32_t* offs,
                              int32_t num_groups, int64_t M, int64_t N, int64_t K,
                              const void* bias, pt_stream_t stream);
/* Both of the above: the bias row of the group is added to the rounded result and the row is
 * stored at out[out_row_index[r]] (grouped linear + indexed_bias_add + the un-permuting
 * padded_index_gather of forward_stage3, models/gpt_oss.py:155-156,318-321, as one kernel). */
int pt_gemm_m_grouped_nt_scatter_bias(const void* a_fp8, const float* a_scale, const void* b_fp8,
                                      const float* b_scale, void* out, int out_dtype,
                                      const int32_t* offs, int32_t num_groups, int64_t M, int64_t N,
                                      int64_t K, const int32_t* out_row_index, int64_t out_rows,
                                      const void* bias, pt_stream_t stream);

/* dW[g][n,k] = sum_{m in group g} dY[m,n] X[m,k] with colwise-quantised operands stored
 * transposed: dy_t[N,M] and x_t[K,M] (PT_CH_TRANSPOSED) and their scales dy_scale[M/128,N],
 * x_scale[M/128,K].  out is [G,N,K]:
 *   out_dtype PT_F32 : fp32, accumulate==0 overwrites, !=0 adds (the `c=` operand)
 *   out_dtype PT_BF16: bf16(sum) rounded once; accumulate!=0 then adds the existing bf16 value
 *                      in fp32 and rounds again (weight.grad += wgrad.to(bf16)).
 * Groups with no rows get zeros (or are left unchanged when accumulating).
 * deep_gemm.k_grouped_fp8_gemm_{tn,nt}_contiguous + grad_weight_fn, grouped_linear.py:202-221. */
int pt_gemm_k_grouped_wgrad(const void* dy_t_fp8, const float* dy_scale, const void* x_t_fp8,
                            const float* x_scale, void* out, int out_dtype, int accumulate,
                            const int32_t* offs, int32_t num_groups, int64_t M, int64_t N,
                            int64_t K, pt_stream_t stream);
/* The same with the row length of the two scale arrays given: dy_scale[M/128, ld_dy_scale] and
 * x_scale[M/128, ld_x_scale] may be column slices of wider arrays (the gate and up halves of a
 * fused projection's colwise twin get their own weight-gradient tensors this way). */
int pt_gemm_k_grouped_wgrad_ld(const void* dy_t_fp8, const float* dy_scale, int64_t ld_dy_scale,
                               const void* x_t_fp8, const float* x_scale, int64_t ld_x_scale,
                               void* out, int out_dtype, int accumulate, const int32_t* offs,
                               int32_t num_groups, int64_t M, int64_t N, int64_t K,
                               pt_stream_t stream);
/* The same for two parameters whose gradients are the first `split` (a multiple of 128) and the remaining
 * rows of every group's [N, K] result: one launch instead of two on halves of dy_t.  out0 [G, split, K],
 * out1 [G, N - split, K]. */
int pt_gemm_k_grouped_wgrad_pair(const void* dy_t_fp8, const float* dy_scale, const void* x_t_fp8,
                                 const float* x_scale, void* out0, void* out1, int64_t split,
                                 int out_dtype, int accumulate, const int32_t* offs, int32_t G,
                                 int64_t M, int64_t N, int64_t K, pt_stream_t stream);

/* Which GEMM kernel the three entry points above launch: "auto" (or NULL: per call from the
 * shape; the default unless the environment variable PT_GEMM_IMPL names one of the others),
 * "r0" persistent kernel, one 256x256 tile after the other per compute unit ("p0", "q0" and "q1", names of
 * main loops that it has replaced, mean the same), "s64" / "s128" one 64x128 / 128x128 tile per workgroup
 * (small problems), "s128d" the latter with one workgroup per compute unit (dense products, else "s128"), "t" one 128x128 tile per workgroup through 64-bit addresses.
 * Every choice computes the same function; this exists for measurements and for tests that
 * cover each kernel.  Process-wide, not synchronised with concurrent GEMM calls.
 * No counterpart in the reference (DeepGEMM selects its kernels internally). */
int pt_gemm_select_kernel(const char* name);

/* ------------------------------------------------------------------------------------------
 * Routing-driven permute / unpermute.  Replace pithtrain/operators/token_scatter.py.
 * ------------------------------------------------------------------------------------------ */

/* Bytes of workspace pt_group_rows needs for m keys and num_groups groups. */
int64_t pt_group_rows_workspace_bytes(int64_t m, int32_t num_groups);

/* Stable counting sort of rows by group with every group padded to `alignment` rows.
 *   keys[m] int64 in [0,num_groups)            (expert_idxs)
 *   offs[G] int32 inclusive cumsum of padded sizes, ks[G] int32 padded sizes
 *   reverse[m] int64: destination row of source row i  (reverse_shuffle_idxs)
 *   src_of[cap] int32: source row of destination row r, -1 for pad rows (r < cap)
 * Canonical order: ascending source row inside a group.  Keys are expected in [0,num_groups); a row
 * whose key is outside belongs to no group: no src_of entry names it and its reverse entry is 0.
 * _compute_group_offsets_kernel + slot assignment of _scatter_for_grouped_gemm_kernel,
 * token_scatter.py:38-101. */
int pt_group_rows(const int64_t* keys, int64_t m, int32_t num_groups, int32_t alignment,
                  int32_t* offs, int32_t* ks, int64_t* reverse, int32_t* src_of, int64_t cap,
                  void* workspace, int64_t workspace_bytes, pt_stream_t stream);

/* pt_group_rows for callers that cannot allocate device memory (code under HIP graph capture,
 * tight serving loops, harnesses that forbid hipMalloc): same arguments, results and errors, but
 * the workspace is a device array built into the library (one copy per GPU, held until the
 * process ends) instead of an argument, and the call allocates and frees nothing.  It refuses
 * problems whose pt_group_rows_workspace_bytes(m, num_groups) exceeds
 * PT_GROUP_ROWS_STATIC_MAX_WORKSPACE (e.g. up to 262144 keys in 256 groups, or 524288 keys in 128).
 * Every call on a GPU uses that GPU's one array: calls that overlap on one GPU (two streams, two
 * threads) race; calls on one stream are ordered and need nothing cleared in between.
 * The first call on a device looks the array's address up (hipGetSymbolAddress, which may load the
 * code object) and must be made outside a graph capture; a captured call records that one
 * address, so two graphs that contain it must not replay at the same time on one GPU either.
 * No counterpart in the reference, which allocates its counters with torch on every call
 * (token_scatter.py:205-207). */
#define PT_GROUP_ROWS_STATIC_MAX_WORKSPACE ((1 << 20) + 8192)
int pt_group_rows_static(const int64_t* keys, int64_t m, int32_t num_groups, int32_t alignment,
                         int32_t* offs, int32_t* ks, int64_t* reverse, int32_t* src_of, int64_t cap,
                         pt_stream_t stream);

/* out[r,:] = src_of[r] >= 0 ? in[pre ? pre[src_of[r]] : src_of[r], :] : 0   for r < rows_out,
 * where rows_out = min(cap, round_up(offs_last[0], tail_alignment)) read on the device when
 * offs_last != NULL, else cap.  Rows in [rows_out, cap) are not touched.  elem_bytes-wide
 * elements, H per row.  `pre` (int64, may be NULL) composes a first gather (the dedup expand)
 * into the same pass.
 * Row copy + pad/tail zeroing of _scatter_for_grouped_gemm_kernel, token_scatter.py:103-153. */
int pt_permute_rows(const void* in, int64_t ld_in, void* out, int64_t ld_out, const int32_t* src_of,
                    const int64_t* pre, const int32_t* offs_last, int32_t tail_alignment,
                    int64_t cap, int64_t H, int32_t elem_bytes, pt_stream_t stream);

/* out[i,:] = in[index[i],:], i < n.  index int64.
 * _PaddedIndexGather.forward (token_scatter.py:297-309), ScatterForGroupedGemm.backward
 * (:271-284). */
int pt_gather_rows(const void* in, int64_t ld_in, void* out, int64_t ld_out, const int64_t* index,
                   int64_t n, int64_t H, int32_t elem_bytes, pt_stream_t stream);

/* Bytes of workspace pt_gather_rows_backward needs. */
int64_t pt_gather_rows_backward_workspace_bytes(int64_t n, int64_t rows);

/* grad_in[r,:] = sum over {j : index[j] == r} of grad_out[j,:], r < rows; summed in fp32 in
 * ascending j, rounded once to the element type (dtype PT_BF16 / PT_F32 / PT_F16).
 * _PaddedIndexGather.backward (scatter_add_), token_scatter.py:311-325. */
int pt_gather_rows_backward(const void* grad_out, int64_t ld_go, void* grad_in, int64_t ld_gi,
                            const int64_t* index, int64_t n, int64_t rows, int64_t H, int dtype,
                            void* workspace, int64_t workspace_bytes, pt_stream_t stream);
/* The same in two parts around the kernel that writes grad_out from grouped rows (a GEMM that un-permutes on the way):
 * _begin fills the workspace from the index and says in dest[q], q < M, where the row of grouped row q belongs, whose
 * index entry is j = row_map[q] (negative: padding): index[j] where no other entry names that row, -2 - j where
 * others do, -1 for padding and for an entry outside [0, rows).  Rows with one source then need no sum: the kernel writes
 * them to grad_in, the others to row j of grad_out (pt_gemm_m_grouped_by_block_two), and _shared adds those up from
 * the same workspace and zeroes the rows that no entry names. */
int pt_gather_rows_backward_begin(const int64_t* index, int64_t n, int64_t rows, void* workspace, int64_t workspace_bytes,
                                  const int32_t* row_map, int32_t* dest, int64_t M, pt_stream_t stream);
int pt_gather_rows_backward_shared(const void* grad_out, int64_t ld_go, void* grad_in, int64_t ld_gi, int64_t n,
                                   int64_t rows, int64_t H, int dtype, void* workspace, int64_t workspace_bytes,
                                   pt_stream_t stream);

/* group_ids[r] = min(#{g : offs[g] <= r}, G-1), r < M; out_dtype_bytes 4 (int32) or 8 (int64).
 * precompute_group_indices, token_scatter.py:370-384; GptOssExperts.forward,
 * models/gpt_oss.py:146-150. */
int pt_group_indices(const int32_t* offs, int32_t num_groups, int64_t M, void* group_ids,
                     int32_t out_dtype_bytes, pt_stream_t stream);
/* out[r] = expand_idx[row_map[r]] (int32) where row_map[r] is in [0, n_expand) and the result in
 * [0, n_src), -1 otherwise.  Composes the scatter's source map with the dedup expand index
 * (models/qwen3_moe.py:222-224 gathers through expand_idx, then scatters), so that the first
 * quantisation of the expert block reads the deduplicated rows directly. */
int pt_compose_row_map(const int32_t* row_map, int64_t n, const int64_t* expand_idx,
                       int64_t n_expand, int64_t n_src, int32_t* out, pt_stream_t stream);

/* ------------------------------------------------------------------------------------------
 * Expert-parallel dispatch index construction with token dedup.
 * Replace the Triton kernels of pithtrain/operators/ep_dispatch.py.
 * ------------------------------------------------------------------------------------------ */

int64_t pt_dedup_workspace_bytes(int64_t m, int32_t k, int32_t num_experts, int32_t ep_size);

/* topk_ids[m,k] int64 (row stride ld_ids) -> tokens_per_ep_rank[ep], dedup_tokens_per_gpu[ep],
 * dispatch_token_idxs[m*ep] (first sum(dedup) valid), idxs[m*k], expand_idx[m*k],
 * send_meta[ep*(epr+1)], all int64.  Canonical order: ascending flat index inside an expert
 * bucket, ascending token id inside an EP-rank chunk.
 * fused_dedup_prepare_dispatch, ep_dispatch.py:271-420. */
int pt_dedup_prepare_dispatch(const int64_t* topk_ids, int64_t ld_ids, int64_t m, int32_t k,
                              int32_t num_experts, int32_t ep_size, int32_t experts_per_rank,
                              int64_t* tokens_per_ep_rank, int64_t* dedup_tokens_per_gpu,
                              int64_t* dispatch_token_idxs, int64_t* idxs, int64_t* expand_idx,
                              int64_t* send_meta, void* workspace, int64_t workspace_bytes,
                              pt_stream_t stream);

/* expert_idxs[s] = e % experts_per_rank for slot s in bucket e (s < sum(counts), s < max_total);
 * output_splits[g] = sum of counts of rank g.   build_expert_idxs, ep_dispatch.py:426-508. */
int pt_build_expert_idxs(const int64_t* tokens_per_expert_group, int32_t num_experts,
                         int32_t ep_size, int32_t experts_per_rank, int64_t max_total,
                         int64_t* expert_idxs, int64_t* output_splits, pt_stream_t stream);

/* out[i] = received[i] + exclusive_cumsum(dedup_counts)[sender(i)], sender from output_splits.
 * dedup_counts has element stride dedup_stride.   adjust_expand_idx, ep_dispatch.py:511-576. */
int pt_adjust_expand_idx(const int64_t* received, int64_t* out, const int64_t* dedup_counts,
                         int64_t dedup_stride, const int64_t* output_splits, int32_t ep_size,
                         int64_t n, pt_stream_t stream);

/* ------------------------------------------------------------------------------------------
 * Fused epilogues.  dtype is the storage type (PT_BF16 / PT_F16 / PT_F32); math in fp32.
 * ------------------------------------------------------------------------------------------ */

/* out = silu(gate) * up over n elements.   _silu_mul_fwd_kernel, silu_mul.py:28-49 */
int pt_silu_mul_fwd(const void* gate, const void* up, void* out, int64_t n, int dtype,
                    pt_stream_t stream);
/* _silu_mul_bwd_kernel, silu_mul.py:52-87 */
int pt_silu_mul_bwd(const void* grad_out, const void* gate, const void* up, void* grad_gate,
                    void* grad_up, int64_t n, int dtype, pt_stream_t stream);
/* The same two kernels on [rows, cols] views with their own leading dimensions (in elements), so
 * that the halves of a fused gate_up buffer are read in place and both gradients land in one
 * [rows, 2*cols] buffer: replaces the .contiguous() copies around silu_mul in
 * Qwen35MoeExperts.forward (models/qwen35_moe.py:196-199) and their autograd backward. */
int pt_silu_mul_fwd_2d(const void* gate, int64_t ld_gate, const void* up, int64_t ld_up, void* out,
                       int64_t ld_out, int64_t rows, int64_t cols, int dtype, pt_stream_t stream);
int pt_silu_mul_bwd_2d(const void* grad_out, int64_t ld_grad_out, const void* gate, int64_t ld_gate,
                       const void* up, int64_t ld_up, void* grad_gate, int64_t ld_grad_gate,
                       void* grad_up, int64_t ld_grad_up, int64_t rows, int64_t cols, int dtype,
                       pt_stream_t stream);
/* gate_up[M,2N] interleaved -> out[M,N]; n = M*N.  _clamped_swiglu_fwd_kernel,
 * clamped_swiglu.py:18-46 */
int pt_clamped_swiglu_fwd(const void* gate_up, void* out, int64_t n, float alpha, float limit,
                          int dtype, pt_stream_t stream);
/* _clamped_swiglu_bwd_kernel, clamped_swiglu.py:49-89 */
int pt_clamped_swiglu_bwd(const void* grad_out, const void* gate_up, void* grad_gate_up, int64_t n,
                          float alpha, float limit, int dtype, pt_stream_t stream);
/* out[r,:] = x[r,:] + bias[group_ids[r],:]  (group_ids int64).  _IndexedBiasAdd.forward,
 * indexed_bias_add.py:100-104 */
int pt_indexed_bias_add_fwd(const void* x, const void* bias, const int64_t* group_ids, void* out,
                            int64_t M, int64_t H, int dtype, pt_stream_t stream);
/* out[g,:] = sum of rows [offs[g-1], min(offs[g],M)) of x, fp32 accumulate, stored as out_dtype.
 * _segment_sum_kernel, indexed_bias_add.py:20-96 */
int pt_segment_sum(const void* x, const int32_t* offs, int32_t num_groups, void* out, int64_t M,
                   int64_t H, int dtype, int out_dtype, pt_stream_t stream);
/* The same sums with grouped row r read from x[row_index[r]] (x [x_rows,H] un-permuted; a negative
 * index is a padding row): the bias gradient of a grouped linear whose output rows were stored
 * through row_index, in the grouped order of the rows (same bits as gathering first). */
int pt_segment_sum_rows(const void* x, int64_t x_rows, const int32_t* row_index, const int32_t* offs,
                        int32_t num_groups, void* out, int64_t M, int64_t H, int dtype,
                        int out_dtype, pt_stream_t stream);
/* pt_segment_sum of fp32 rows that each stand for `unit` grouped rows (per-tile column sums): group g owns
 * rows offs[g-1] / unit .. offs[g] / unit - 1. */
int pt_segment_sum_tiles(const float* x, const int32_t* offs, int32_t unit, int32_t num_groups,
                         void* out, int64_t M, int64_t H, int out_dtype, pt_stream_t stream);

/* ------------------------------------------------------------------------------------------
 * Top-k weighted combine with the residual: the memory-bound step that follows the expert path.
 * forward_stage5, single-rank branch (models/qwen3_moe.py:229-237; the same expression in
 * models/deepseek_v2.py, models/gpt_oss.py, models/qwen35_moe.py).
 * ------------------------------------------------------------------------------------------ */

/* out[t,:] = residual[t,:] + S(sum_j float(moe[t*k+j,:]) * topk_weight[t,j]): fp32 products added in
 * the order j = 0..k-1, the sum rounded to the storage type S (dtype), the addition rounded again.
 * moe is [T*k,H], residual and out [T,H] (leading dimensions in elements), topk_weight fp32 [T,k],
 * 1 <= k <= 16.  residual may be NULL: out is then the rounded sum itself, the weighted sum that
 * ends the single-device MoE forward (models/qwen3_moe.py:119). */
int pt_moe_combine_fwd(const void* moe, int64_t ld_moe, const float* topk_weight,
                       const void* residual, int64_t ld_res, void* out, int64_t ld_out, int64_t T,
                       int32_t k, int64_t H, int dtype, pt_stream_t stream);
/* d_moe[t*k+j,:] = S(float(grad_out[t,:]) * topk_weight[t,j]);
 * d_weight[t,j] = sum_h grad_out[t,h] * moe[t*k+j,h] in fp32 (fixed reduction order);
 * the gradient of the residual is grad_out itself. */
int pt_moe_combine_bwd(const void* grad_out, int64_t ld_go, const void* moe, int64_t ld_moe,
                       const float* topk_weight, void* d_moe, int64_t ld_dmoe, float* d_weight,
                       int64_t T, int32_t k, int64_t H, int dtype, pt_stream_t stream);

/* Gradient of a tensor [T, H] that several branches read: out[t] = sum_j rows[t * k + j] + g0[t] + g1[t] + g2[t]
 * (rows [T * k, H] or NULL, g0 .. g2 [T, H] or NULL), all in dtype, added in fp32 in that order and rounded
 * once.  Replaces the reduction of the expand's backward and the additions autograd does between branches
 * (qwen3_moe.py:104-119).  H % 8 == 0, 16-byte aligned. */
int pt_sum_branches(const void* rows, int32_t k, const void* g0, const void* g1, const void* g2, void* out,
                    int64_t T, int64_t H, int dtype, pt_stream_t stream);

/* Expert-parallel branch of forward_stage5 (models/qwen3_moe.py:238-245, same lines in
 * deepseek_v2.py:351-357, qwen35_moe.py:334-340, gpt_oss.py:334-340): row r of moe [rows,H] belongs
 * to the flat top-k slot local_idxs[r] (token local_idxs[r] / k), every weighted row is rounded to
 * S and added to a zeroed S accumulator, the residual is added last.  The reference's scatter_add_
 * leaves the order of the adds to the device's atomics; here a token's rows are added in ascending
 * r, every partial sum rounded to S (the result of a sequential scatter_add_).
 *
 * pt_moe_combine_ep_index: slot_row[s] = r for s = local_idxs[r], -1 for slots without a row
 * (slot_row int32 [slots], slots = T*k; entries of local_idxs must be distinct, values outside
 * [0, slots) are ignored). */
int pt_moe_combine_ep_index(const int64_t* local_idxs, int64_t rows, int64_t slots,
                            int32_t* slot_row, pt_stream_t stream);
int pt_moe_combine_ep_fwd(const void* moe, int64_t ld_moe, int64_t rows, const int32_t* slot_row,
                          const float* topk_weight, const void* residual, int64_t ld_res, void* out,
                          int64_t ld_out, int64_t T, int32_t k, int64_t H, int dtype,
                          pt_stream_t stream);
/* d_moe[r,:] = S(float(grad_out[t,:]) * topk_weight[t,j]) for r = slot_row[t*k+j];
 * d_weight[t,j] = sum_h grad_out[t,h] * moe[r,h] in fp32, 0 for a slot without a row. */
int pt_moe_combine_ep_bwd(const void* grad_out, int64_t ld_go, const void* moe, int64_t ld_moe,
                          int64_t rows, const int32_t* slot_row, const float* topk_weight,
                          void* d_moe, int64_t ld_dmoe, float* d_weight, int64_t T, int32_t k,
                          int64_t H, int dtype, pt_stream_t stream);

/* Router gate after the logits GEMM: softmax + top-k + weights of the chosen experts, one launch.
 *   mode 0: Qwen3MoeGate.forward (models/qwen3_moe.py:81-88), Qwen35MoeTopKRouter.forward
 *           (models/qwen35_moe.py:216-222) and DeepSeekV2MoEGate.forward (models/deepseek_v2.py:
 *           149-164): scores = softmax(logits) in fp32; with num_group > 1 only the topk_group
 *           groups of E/num_group contiguous experts with the largest maximum keep their scores
 *           (group_limited_greedy), the rest become 0; top-k of the scores; w = scores[topk_idx];
 *           w /= sum(w) if norm_topk_prob; w *= scale (routed_scaling_factor).
 *   mode 1: GptOssTopKRouter.forward (models/gpt_oss.py:176-182): top-k of the logits, then
 *           w = softmax(logits[topk_idx]) in fp32.
 * logits [T,E] in dtype (leading dimension in elements), E <= 512, k <= min(32, E).  topk_idx int64
 * [T,k] comes out sorted by descending value, ties to the lower expert index (torch.topk leaves
 * both open for sorted=False).  forced_idx (router replay, the `router_replay` hook of the same
 * functions) replaces the selection when not null.  scores fp32 [T,E] (what the load-balance loss
 * reads: after the group limit in mode 0, the full softmax in mode 1) is written when not null. */
int pt_router_topk_fwd(const void* logits, int64_t ld_logits, int dtype, int64_t T, int32_t E,
                       int32_t k, int mode, int norm_topk_prob, float scale, int32_t num_group,
                       int32_t topk_group, const int64_t* forced_idx, int64_t* topk_idx,
                       float* topk_weight, float* scores, pt_stream_t stream);
/* Gradient of the logits from d_weight fp32 [T,k] (and d_scores fp32 [T,E] when not null), through
 * the scale, the normalisation, the gather at topk_idx, the group limit and the softmax; the
 * scores are recomputed from the logits.  d_logits [T,E] in dtype. */
int pt_router_topk_bwd(const void* logits, int64_t ld_logits, int dtype, int64_t T, int32_t E,
                       int32_t k, int mode, int norm_topk_prob, float scale, int32_t num_group,
                       int32_t topk_group, const int64_t* topk_idx, const float* d_weight,
                       const float* d_scores, void* d_logits, int64_t ld_dlogits,
                       pt_stream_t stream);

/* Gradients of a gate's logits = x w^T for bf16 x [T,H] and w [E,H] (models/qwen3_moe.py:79; as an fp32 product
 * models/deepseek_v2.py:145-147): d_x = d_logits w and d_w = d_logits^T x from d_logits [T,E] in dtype (fp32
 * or bf16), summed in fp32 and rounded to bf16.  E and H multiples of 8, E <= 256. */
int64_t pt_gate_linear_bwd_workspace_bytes(int64_t T, int32_t E, int64_t H);
int pt_gate_linear_bwd(const void* d_logits, int dtype, const void* x, const void* w, void* d_x, void* d_w,
                       int64_t T, int32_t E, int64_t H, void* workspace, pt_stream_t stream);

/* ------------------------------------------------------------------------------------------
 * Whole steps as one call: the launches of a forward or a backward are prepared and queued here
 * instead of one by one by the caller.  The argument blocks are read on the host during the call;
 * every field is 8 bytes wide.
 * ------------------------------------------------------------------------------------------ */

/* Forward of an expert block (gate_up projection, SwiGLU, down projection; FP8 operands).
 * x bf16 [x_rows, K] (row stride ldx).  With row_map (int32 [M], the scatter's source map, negative =
 * padding) grouped row r is x[row_map[r]], or x[expand_idx[row_map[r]]] with expand_idx (int64
 * [n_expand]); the row count is then read from offs[G-1].  Without it x has M grouped rows.
 * gate_up bf16 [M, 2*half] is an output that the backward reads.  out bf16: row_map'd to
 * [out_rows, H] when scatter != 0, else [M, H].  clamped != 0: the clamped SwiGLU on interleaved pairs
 * (alpha, limit) with the biases gu_bias [G, 2*half] and dn_bias [G, H] (may be NULL) added by the
 * GEMMs' stores; otherwise silu(gate) * up on concatenated halves.  x_t [K, M] and h_t [half, M] bytes with
 * scales [M/128, K] and [M/128, half]: the transposed activations that the weight gradients read (all four
 * NULL: no backward follows).  repeat > 1 (with row_map, without expand_idx): grouped row r is
 * x[row_map[r] / repeat].  few_rows != 0 (no backward): the groups are multiples of 64 rows.  Not
 * needed afterwards: composed_map int32 [M] (with expand_idx), x_fp8 [M, K] and h_fp8 [M, half] with
 * their 1x128 scales. */
typedef struct {
  const void* x; int64_t x_rows, ldx;
  int64_t M, K, half, H, G;
  const int32_t* offs;
  const int32_t* row_map;
  const int64_t* expand_idx; int64_t n_expand;
  int64_t repeat, few_rows;
  const void* gu_fp8; const float* gu_scale; const void* gu_bias;
  const void* dn_fp8; const float* dn_scale; const void* dn_bias;
  void* gate_up;
  void* out; int64_t out_rows, scatter;
  int64_t clamped; double alpha, limit;
  void* x_t; float* x_t_scale; void* h_t; float* h_t_scale;
  int32_t* composed_map; void* x_fp8; float* x_scale; void* h_fp8; float* h_scale;
  pt_stream_t stream;
} pt_experts_forward_args;
int pt_experts_forward(const pt_experts_forward_args* args /* host */);
/* The same step with the scales of its row-scaled operands (x_scale, h_scale; in the backward dy_scale and dgu_scale) as
 * [K/128, M] instead of [M, K/128]: the GEMMs read them in whole lines. */
int pt_experts_forward_by_block(const pt_experts_forward_args* args /* host */);
/* The latter of scattered rows (scatter != 0), which leaves padding out: what stands for it, row_map[r] < 0, in gate_up, x_fp8 and
 * h_fp8 is not defined, and the transposed activations hold zeros for it.  Where a backward follows, without the clamped
 * activation and gu_bias, which make other values of padding, and that backward is pt_experts_backward_without_padding.  row_map
 * is 16-byte aligned. */
int pt_experts_forward_without_padding(const pt_experts_forward_args* args /* host */);

/* Backward of the same block, up to the quantised gradient of gate_up: dgu_fp8 [M, 2*half] and dgu_scale
 * [M, ceil(2*half/128)], from which the input gradient follows with one pt_gemm_m_grouped_nn(_scatter) on
 * the gate_up weight.  grad_out bf16 [grad_rows, H]; out_map: row_map when the forward scattered its
 * result (the gradient arrives un-permuted), else NULL; limit_rows != 0: the row count is offs[G-1] (the
 * forward had a row_map).  dn_dg: the down weight, dn_forward_layout != 0 for the forward-layout tensor, 0
 * for the transposed twin.  dy_t [H, M] and dgu_t [2*half, M] bytes with scales [M/128, .]: the transposed
 * gradients of the weight-gradient GEMMs (kept by the caller when it runs those later).  Not needed
 * afterwards: dy_fp8 [M, H] with 1x128 scales, grad_h bf16 [M, half], col_sum fp32 [M/128, 2*half].
 * dy_fp8 and dy_scale may be the memory of dgu_fp8 and dgu_scale (of the larger size): they have been read
 * before those are written.
 * dw_down [G, H, half] bf16 (NULL = not computed here), dw_gate_up [G, 2*half, K] or, when dw_up is given,
 * [G, half, K] each (pt_experts_weight_gradient only); *_add != 0: added to what is there.  d_gu_bias / d_dn_bias [G, 2*half] /
 * [G, H] in the types given: NULL = none. */
typedef struct {
  const void* grad_out; int64_t grad_rows;
  int64_t M, K, half, H, G;
  const int32_t* offs;
  const int32_t* out_map; int64_t limit_rows;
  const void* dn_dg; const float* dn_dg_scale; int64_t dn_forward_layout;
  const void* gate_up;
  const void* x_t; const float* x_t_scale; const void* h_t; const float* h_t_scale;
  void* dgu_fp8; float* dgu_scale;
  void* dy_t; float* dy_t_scale; void* dgu_t; float* dgu_t_scale;
  void* dy_fp8; float* dy_scale; void* grad_h; float* col_sum;
  void* dw_down; int64_t dw_down_add;
  void* dw_gate_up; int64_t dw_gate_up_add;
  void* dw_up; int64_t dw_up_add;
  int64_t clamped; double alpha, limit;
  void* d_gu_bias; int64_t d_gu_bias_dtype;
  void* d_dn_bias; int64_t d_dn_bias_dtype;
  pt_stream_t stream;
} pt_experts_backward_args;
int pt_experts_backward(const pt_experts_backward_args* args /* host */);
int pt_experts_backward_by_block(const pt_experts_backward_args* args /* host */); /* see pt_experts_forward_by_block; the input gradient is pt_gemm_m_grouped_by_block's */
/* The latter after pt_experts_forward_without_padding (out_map: its row_map, limit_rows != 0): what stands for padding in dy_fp8,
 * dgu_fp8 and grad_h is not defined either, and the transposed gradients hold zeros for it. */
int pt_experts_backward_without_padding(const pt_experts_backward_args* args /* host */);
/* The gate_up weight gradient of the same block from the same arguments (dw_gate_up, dw_up): the last
 * launch of a backward, after the caller has queued the input gradient. */
int pt_experts_weight_gradient(const pt_experts_backward_args* args /* host */);
/* Row pitch (bytes) of a transposed FP8 operand of `rows` columns in a dense linear: what the backward entry points
 * below use for their own, and callers for the ones they keep. */
int64_t pt_transposed_pitch(int64_t rows);
/* Forward of a dense FP8 linear (fp8_act_weight_gemm, operators/linear.py:44-60): x [M, K] in dtype,
 * y [M, N] in y_dtype (PT_BF16 or PT_F32); x_t (row pitch ld_t >= M bytes) and x_t_scale are the transposed
 * operand the weight gradient reads (both NULL: not written).  K % 16 == 0.  y2 != NULL (bf16, splits == 1):
 * the outputs of pt_gemm_nt_dense_heads.  w != NULL (in dtype, row stride ldw): the weight itself, quantised
 * here into w_fp8 [N, K], w_scale, w_t_fp8 [K, N] and w_t_scale (then outputs, with x_t). */
typedef struct {
  const void* x; int64_t dtype, M, K, ldx;
  const void* w; int64_t ldw; void* w_t_fp8; float* w_t_scale;
  const void* w_fp8; const float* w_scale; int64_t N;
  void* y; int64_t y_dtype;
  void* x_t; int64_t ld_t; float* x_t_scale;
  int64_t splits, split_len;
  void* y2; int64_t head_a, head_b;
  void* workspace;
  pt_stream_t stream;
} pt_linear_forward_args;
int64_t pt_linear_forward_workspace_bytes(int64_t M, int64_t N, int64_t K, int64_t splits);
int pt_linear_forward(const pt_linear_forward_args* args /* host */);

/* Backward (fp8_dgrad_wgrad, operators/linear.py:63-83): grad [M, N] in dtype -> grad_x [M, K] through
 * the transposed weight w_t [K, N], grad_w [N, K] through x_t [K, M]; both in out_dtype.  N % 16 == 0;
 * M % 16 == 0 unless x_t was written by pt_linear_forward with a pitch of at least M rounded up to 16
 * (its columns past M are zero).  splits / split_len per GEMM: the reduction ranges of
 * pt_gemm_nt_dense_splitk (1 = not split).  x_t NULL: the input x [M, K] (dtype, row stride ldx) is
 * quantised here (workspace query with from_x != 0).  grad2 != NULL: the gradient's columns come from two
 * tensors as in pt_quant_heads_rowwise_transpose_ld. */
typedef struct {
  const void* grad; int64_t dtype, M, N, ldg;
  const void* w_t_fp8; const float* w_t_scale; int64_t K;
  const void* x_t; int64_t ld_xt; const float* x_t_scale;
  void* grad_x; void* grad_w; int64_t out_dtype;
  int64_t x_splits, x_split_len, w_splits, w_split_len;
  const void* x; int64_t ldx;
  const void* grad2; int64_t head_a, head_b;
  void* workspace;
  pt_stream_t stream;
} pt_linear_backward_args;
int64_t pt_linear_backward_workspace_bytes(int64_t M, int64_t N, int64_t K, int64_t x_splits, int64_t w_splits,
                                           int64_t from_x);
int pt_linear_backward(const pt_linear_backward_args* args /* host */);

/* Forward of a dense SwiGLU MLP (DeepseekV2MLP, models/deepseek_v2.py:94-108), all bf16:
 * gate_up [M, 2 half] = x [M, K] (gate | up)^T, y [M, H] = (silu(gate) * up) down^T.  The gate and up weights
 * [half, K] are one quantised operand gu_fp8 [2 half, K] with scales [2 half / 128, K / 128] and its
 * transposed form gu_t [K, 2 half]; down [H, half] has dn_*.  w_gate, w_up, w_down (row strides ld_*; all or
 * none): the weights, quantised here into those operands.  x_t [K, ld_t], h_t [half, ld_t] and their scales:
 * what the weight gradients read (all NULL: not written).  half % 128 == 0, K % 16 == 0, H % 16 == 0. */
typedef struct {
  const void* x; int64_t M, K, ldx, half, H;
  const void* w_gate; int64_t ld_gate; const void* w_up; int64_t ld_up; const void* w_down; int64_t ld_down;
  void* gu_fp8; float* gu_scale; void* gu_t; float* gu_t_scale;
  void* dn_fp8; float* dn_scale; void* dn_t; float* dn_t_scale;
  void* gate_up; void* y;
  void* x_t; float* x_t_scale; void* h_t; float* h_t_scale; int64_t ld_t;
  int64_t gu_splits, gu_split_len, dn_splits, dn_split_len;
  void* workspace;
  pt_stream_t stream;
} pt_mlp_forward_args;
int64_t pt_mlp_forward_workspace_bytes(int64_t M, int64_t K, int64_t half, int64_t H, int64_t gu_splits,
                                       int64_t dn_splits);
int pt_mlp_forward(const pt_mlp_forward_args* args /* host */);
/* Its backward: grad [M, H] -> grad_x [M, K], grad_gu [2 half, K] (gate | up), grad_dn [H, half], all bf16.
 * splits of the four GEMMs (grad_h, grad_dn, grad_x, grad_gu) as in pt_linear_backward. */
typedef struct {
  const void* grad; int64_t M, K, half, H, ldg;
  const void* gu_t; const float* gu_t_scale; const void* dn_t; const float* dn_t_scale;
  const void* gate_up;
  const void* x_t; const float* x_t_scale; const void* h_t; const float* h_t_scale; int64_t ld_t;
  void* grad_x; void* grad_gu; void* grad_dn;
  int64_t splits[4], split_len[4];
  void* workspace;
  pt_stream_t stream;
} pt_mlp_backward_args;
int64_t pt_mlp_backward_workspace_bytes(int64_t M, int64_t K, int64_t half, int64_t H, const int64_t* splits /* host [4] */);
int pt_mlp_backward(const pt_mlp_backward_args* args /* host */);

/* Measurement: `fn`, when not NULL, is called on the host before (begin = 1) and after (begin = 0) every
 * entry point that the whole-step functions above run, with its name and {M, N, K} of a GEMM or
 * {rows, columns, source rows} of a quantisation. */
typedef void (*pt_observer_t)(const char* name, int begin, int64_t a, int64_t b, int64_t c);
void pt_set_observer(pt_observer_t fn);
/* Reports an entry point that a caller outside this library runs as part of a whole step of its own. */
void pt_observe(const char* name, int begin, int64_t a, int64_t b, int64_t c);

/* In-place fused cross-entropy with mean reduction (CrossEntropy.forward and its Triton kernel
 * cross_entropy_fwd, operators/cross_entropy.py:16-78,86-118): logits [N,V] in dtype are
 * overwritten with the gradient of the mean loss, S((exp(x - max) / sum) / n) and, at the target,
 * S(float(stored) - 1/n), with n = max(1, number of rows whose target is not ignore_index); rows
 * with the ignored target become zero.  loss_rows fp32 [N] receives -(x_y - max - log sum) (0 for
 * ignored rows, NaN for a target outside [0, V)), loss fp32 [1] their sum over n, n_non_ignore
 * int64 [1] n itself.  Three launches on the stream, no host synchronisation. */
int pt_cross_entropy_fwd(void* logits, int64_t ld, int dtype, const int64_t* target, int64_t N,
                         int64_t V, int64_t ignore_index, float* loss_rows, float* loss,
                         int64_t* n_non_ignore, pt_stream_t stream);
/* CrossEntropy.backward (operators/cross_entropy.py:120-124): the stored gradient times the
 * incoming scalar (fp32 on the device, rounded to dtype first), in place. */
int pt_cross_entropy_bwd(void* grad, int64_t ld, int dtype, int64_t N, int64_t V,
                         const float* grad_output, pt_stream_t stream);

#ifdef __cplusplus
}
#endif
#endif /* PITHTRAIN_HIP_H */

// Whole steps as one host call (no kernels here): the forward and the backward of an expert block and
// of a dense linear queue their launches from this file.
//
// A layer with few tokens is bound by the host: a launch costs about 3.5 us of host time, and every
// separate call from Python added 6-10 us of argument conversion, allocation and stream lookup to it
// (toy layer, 22 calls: 400 us a step against 170 us of kernels).  Here a step is one call with one
// block of arguments.
#include "common.h"

namespace pt {

static int64_t up(int64_t x) { return (x + 255) & ~(int64_t)255; }

static pt_observer_t g_observer = nullptr;

// runs one entry point, with the observer around it, and returns from the caller on failure
#define PT_STEP(NAME, A, B, C, ...)                         \
  do {                                                      \
    if (g_observer) g_observer(#NAME, 1, (A), (B), (C));    \
    if (int rc_ = NAME(__VA_ARGS__)) return rc_;            \
    if (g_observer) g_observer(#NAME, 0, (A), (B), (C));    \
  } while (0)

// the same around an internal form of that entry point
#define PT_STEP_AS(NAME, A, B, C, CALL)                     \
  do {                                                      \
    if (g_observer) g_observer(#NAME, 1, (A), (B), (C));    \
    if (int rc_ = CALL) return rc_;                         \
    if (g_observer) g_observer(#NAME, 0, (A), (B), (C));    \
  } while (0)

// Carves consecutive 256-byte aligned pieces out of a buffer (a null buffer gives offsets).
struct Carve {
  uintptr_t p;
  explicit Carve(const void* base) : p((uintptr_t)base) {}
  void* bytes(int64_t n) { void* r = (void*)p; p += (uintptr_t)up(n); return r; }
  float* floats(int64_t n) { return (float*)bytes(4 * n); }
};

}  // namespace pt

using namespace pt;

extern "C" void pt_set_observer(pt_observer_t fn) { g_observer = fn; }
extern "C" void pt_observe(const char* name, int begin, int64_t a, int64_t b, int64_t c) {
  if (g_observer) g_observer(name, begin, a, b, c);
}

static int experts_forward(const pt_experts_forward_args* args, RowScales order, bool without_padding = false) {
  PT_REQUIRE(args, "experts_forward: null arguments");
  const pt_experts_forward_args& a = *args;
  PT_REQUIRE(a.M >= 0 && a.M % 128 == 0 && a.K > 0 && a.half > 0 && a.H > 0 && a.G > 0 && a.G < (1ll << 31), "experts_forward: bad sizes");
  const bool keep = a.x_t != nullptr;  // a backward will read the transposed activations
  PT_REQUIRE(a.offs && a.gate_up && a.out && a.x_fp8 && a.x_scale && a.h_fp8 && a.h_scale && keep == (a.h_t != nullptr) &&
                 keep == (a.x_t_scale != nullptr) && keep == (a.h_t_scale != nullptr), "experts_forward: null pointer");
  PT_REQUIRE(a.repeat >= 1 && (a.repeat == 1 || (a.row_map && !a.expand_idx)), "experts_forward: repeat needs row_map and no expand_idx");
  PT_REQUIRE(!a.few_rows || !keep, "experts_forward: a backward needs groups of whole 128-row blocks");
  PT_REQUIRE(!a.expand_idx || a.composed_map, "experts_forward: expand_idx needs composed_map");
  PT_REQUIRE(a.row_map || (!a.expand_idx && !a.scatter), "experts_forward: expand_idx and scatter need row_map");
  if (a.M == 0) return PT_OK;
  const int32_t G = (int32_t)a.G;
  const int32_t* limit = a.row_map ? a.offs + G - 1 : nullptr;  // rows past it hold nothing
  const int32_t* in_map = a.row_map;
  const bool few = a.few_rows != 0;
  PT_REQUIRE(!without_padding || ((uintptr_t)a.row_map & 15) == 0, "experts_forward_without_padding: row_map must be 16-byte aligned");
  PT_REQUIRE(!without_padding || (a.scatter && (!keep || (!a.gu_bias && !a.clamped))),
             "experts_forward_without_padding: needs scatter, and before a backward a SwiGLU block without a bias");
  const int32_t* used = without_padding ? a.row_map : nullptr;
  if (a.expand_idx) {
    PT_STEP(pt_compose_row_map, a.M, 0, 0, a.row_map, a.M, a.expand_idx, a.n_expand, a.x_rows, a.composed_map, a.stream);
    in_map = a.composed_map;
  }
  const auto quant_x = [&](int64_t repeat, const int32_t* rows_of, const int32_t* ends) {
    return quant_rowwise_colwise(a.x, a.x_rows, repeat, PT_BF16, a.M, a.K, a.ldx, rows_of, a.x_fp8, a.x_scale, order, a.x_t, a.x_t_scale,
                                 PT_CH_TRANSPOSED, ends, ends ? G : 0, a.stream, nullptr, used);
  };
  if (a.repeat > 1)
    PT_STEP_AS(pt_quant_rowwise_colwise_rows_repeat, a.M, a.K, a.x_rows, quant_x(a.repeat, in_map, a.offs));
  else if (in_map)
    PT_STEP_AS(pt_quant_rowwise_colwise_rows, a.M, a.K, a.x_rows, quant_x(1, in_map, a.offs));
  else
    PT_STEP_AS(pt_quant_rowwise_colwise, a.M, a.K, a.x_rows, quant_x(1, nullptr, nullptr));
  const int64_t N = 2 * a.half;
  const auto gate_up = [&](const void* bias) {
    return gemm_m_grouped(a.x_fp8, a.x_scale, order, a.gu_fp8, a.gu_scale, a.gate_up, PT_BF16, a.offs, G, a.M, N, a.K, nullptr, 0, bias, a.stream,
                          false, few, nullptr, 0, used, a.out_rows);
  };
  if (few)
    PT_STEP_AS(pt_gemm_m_grouped_nt_few_rows, a.M, N, a.K, gate_up(a.gu_bias));
  else if (a.gu_bias)
    PT_STEP_AS(pt_gemm_m_grouped_nt_bias, a.M, N, a.K, gate_up(a.gu_bias));
  else
    PT_STEP_AS(pt_gemm_m_grouped_nt, a.M, N, a.K, gate_up(nullptr));
  if (a.clamped)
    PT_STEP_AS(pt_clamped_swiglu_quant_rowwise_colwise, a.M, a.half, 0,
               clamped_swiglu_quant(a.gate_up, a.M, a.half, N, (float)a.alpha, (float)a.limit, a.h_fp8, a.h_scale, a.h_t, a.h_t_scale, limit, order,
                                    a.stream, used));
  else
    PT_STEP_AS(pt_silu_mul_quant_rowwise_colwise, a.M, a.half, 0,
               silu_mul_quant(a.gate_up, a.M, a.half, N, a.h_fp8, a.h_scale, a.h_t, a.h_t_scale, limit, order, a.stream, used));
  const auto down = [&](const void* bias) {
    return gemm_m_grouped(a.h_fp8, a.h_scale, order, a.dn_fp8, a.dn_scale, a.out, PT_BF16, a.offs, G, a.M, a.H, a.half, a.scatter ? a.row_map : nullptr,
                          a.scatter ? a.out_rows : 0, bias, a.stream, false, few, nullptr, 0, used);
  };
  if (few)
    PT_STEP_AS(pt_gemm_m_grouped_nt_few_rows, a.M, a.H, a.half, down(a.dn_bias));
  else if (a.scatter && a.dn_bias)
    PT_STEP_AS(pt_gemm_m_grouped_nt_scatter_bias, a.M, a.H, a.half, down(a.dn_bias));
  else if (a.scatter)
    PT_STEP_AS(pt_gemm_m_grouped_nt_scatter, a.M, a.H, a.half, down(nullptr));
  else if (a.dn_bias)
    PT_STEP_AS(pt_gemm_m_grouped_nt_bias, a.M, a.H, a.half, down(a.dn_bias));
  else
    PT_STEP_AS(pt_gemm_m_grouped_nt, a.M, a.H, a.half, down(nullptr));
  return PT_OK;
}

static int experts_backward(const pt_experts_backward_args* args, RowScales order, bool without_padding = false) {
  PT_REQUIRE(args, "experts_backward: null arguments");
  const pt_experts_backward_args& a = *args;
  PT_REQUIRE(a.M >= 0 && a.M % 128 == 0 && a.K > 0 && a.half > 0 && a.H > 0 && a.G > 0 && a.G < (1ll << 31), "experts_backward: bad sizes");
  PT_REQUIRE(a.grad_out && a.offs && a.gate_up && a.h_t && a.h_t_scale && a.dy_fp8 && a.dy_scale && a.dy_t && a.dy_t_scale && a.grad_h && a.dgu_fp8 &&
                 a.dgu_scale && a.dgu_t && a.dgu_t_scale, "experts_backward: null pointer");
  if (a.M == 0) return PT_OK;
  const int32_t G = (int32_t)a.G;
  const int32_t* limit = a.limit_rows ? a.offs + G - 1 : nullptr;
  PT_REQUIRE(!without_padding || (a.out_map && a.limit_rows && !a.clamped && !a.d_gu_bias),
             "experts_backward_without_padding: needs out_map and limit_rows of a SwiGLU block without a bias");
  PT_REQUIRE(!without_padding || ((uintptr_t)a.out_map & 15) == 0, "experts_backward_without_padding: out_map must be 16-byte aligned");
  const int32_t* used = without_padding ? a.out_map : nullptr;
  // The gradient of the down bias is the sum of the rows that are quantised here: the kernel that reads them adds up
  // every 128 (groups are whole 128-row tiles) where col_sum, which the activation's backward fills afterwards, has
  // room for those sums (16384 tokens x 4 of 2880 columns: a second pass over the rows took 110 us, the sums here cost
  // 12 and their sum over the tiles 9).
  float* const dy_sums = a.d_dn_bias && a.clamped && a.H <= 2 * a.half ? a.col_sum : nullptr;
  const auto quant_dy = [&](const int32_t* ends) {
    return quant_rowwise_colwise(a.grad_out, a.grad_rows, 1, PT_BF16, a.M, a.H, a.H, a.out_map, a.dy_fp8, a.dy_scale, order, a.dy_t, a.dy_t_scale,
                                 PT_CH_TRANSPOSED, ends, ends ? G : 0, a.stream, dy_sums, used);
  };
  if (a.out_map)
    PT_STEP_AS(pt_quant_rowwise_colwise_rows, a.M, a.H, a.grad_rows, quant_dy(a.offs));
  else
    PT_STEP_AS(pt_quant_rowwise_colwise, a.M, a.H, a.grad_rows, quant_dy(nullptr));
  if (a.d_dn_bias) {
    if (dy_sums)
      PT_STEP(pt_segment_sum_tiles, a.M / 128, a.H, 0, dy_sums, a.offs, 128, G, a.d_dn_bias, a.M / 128, a.H, (int)a.d_dn_bias_dtype, a.stream);
    else if (a.out_map)
      PT_STEP(pt_segment_sum_rows, a.M, a.H, 0, a.grad_out, a.grad_rows, a.out_map, a.offs, G, a.d_dn_bias, a.M, a.H, PT_BF16,
              (int)a.d_dn_bias_dtype, a.stream);
    else
      PT_STEP(pt_segment_sum, a.M, a.H, 0, a.grad_out, a.offs, G, a.d_dn_bias, a.M, a.H, PT_BF16, (int)a.d_dn_bias_dtype, a.stream);
  }
  const auto grad_h = [&] {
    return gemm_m_grouped(a.dy_fp8, a.dy_scale, order, a.dn_dg, a.dn_dg_scale, a.grad_h, PT_BF16, a.offs, G, a.M, a.half, a.H, nullptr, 0, nullptr,
                          a.stream, a.dn_forward_layout != 0, false, nullptr, 0, used, a.grad_rows);
  };
  if (a.dn_forward_layout)
    PT_STEP_AS(pt_gemm_m_grouped_nn, a.M, a.half, a.H, grad_h());
  else
    PT_STEP_AS(pt_gemm_m_grouped_nt, a.M, a.half, a.H, grad_h());
  if (a.dw_down)
    PT_STEP(pt_gemm_k_grouped_wgrad, a.M, a.H, a.half, a.dy_t, a.dy_t_scale, a.h_t, a.h_t_scale, a.dw_down, PT_BF16, (int)a.dw_down_add, a.offs, G,
            a.M, a.H, a.half, a.stream);
  if (a.clamped)
    PT_STEP_AS(pt_clamped_swiglu_bwd_quant_rowwise_colwise, a.M, a.half, 0,
               clamped_swiglu_bwd_quant(a.grad_h, a.half, a.gate_up, 2 * a.half, a.M, a.half, (float)a.alpha, (float)a.limit, a.dgu_fp8, a.dgu_scale,
                                        a.dgu_t, a.dgu_t_scale, a.col_sum, limit, order, a.stream));
  else
    PT_STEP_AS(pt_silu_mul_bwd_quant_rowwise_colwise, a.M, a.half, 0,
               silu_mul_bwd_quant(a.grad_h, a.half, a.gate_up, 2 * a.half, a.M, a.half, a.dgu_fp8, a.dgu_scale, a.dgu_t, a.dgu_t_scale, limit, order,
                                  a.stream, used));
  if (a.d_gu_bias)  // groups are whole 128-row tiles: their ends in tiles index the per-tile column sums
    PT_STEP(pt_segment_sum_tiles, a.M / 128, 2 * a.half, 0, a.col_sum, a.offs, 128, G, a.d_gu_bias, a.M / 128, 2 * a.half,
            (int)a.d_gu_bias_dtype, a.stream);
  return PT_OK;
}

extern "C" int pt_experts_forward(const pt_experts_forward_args* args) { return experts_forward(args, RowScales::BY_ROW); }
extern "C" int pt_experts_forward_by_block(const pt_experts_forward_args* args) { return experts_forward(args, RowScales::BY_BLOCK); }
extern "C" int pt_experts_forward_without_padding(const pt_experts_forward_args* args) { return experts_forward(args, RowScales::BY_BLOCK, true); }
extern "C" int pt_experts_backward(const pt_experts_backward_args* args) { return experts_backward(args, RowScales::BY_ROW); }
extern "C" int pt_experts_backward_by_block(const pt_experts_backward_args* args) { return experts_backward(args, RowScales::BY_BLOCK); }
extern "C" int pt_experts_backward_without_padding(const pt_experts_backward_args* args) { return experts_backward(args, RowScales::BY_BLOCK, true); }

extern "C" int pt_experts_weight_gradient(const pt_experts_backward_args* args) {
  PT_REQUIRE(args, "experts_weight_gradient: null arguments");
  const pt_experts_backward_args& a = *args;
  PT_REQUIRE(a.M >= 0 && a.M % 128 == 0 && a.offs && a.x_t && a.x_t_scale && a.dgu_t && a.dgu_t_scale && a.dw_gate_up, "experts_weight_gradient: bad arguments");
  const int32_t G = (int32_t)a.G;
  if (!a.dw_up)
    PT_STEP(pt_gemm_k_grouped_wgrad, a.M, 2 * a.half, a.K, a.dgu_t, a.dgu_t_scale, a.x_t, a.x_t_scale, a.dw_gate_up, PT_BF16, (int)a.dw_gate_up_add,
            a.offs, G, a.M, 2 * a.half, a.K, a.stream);
  else if ((a.dw_gate_up_add != 0) == (a.dw_up_add != 0) && a.half % 128 == 0)
    PT_STEP(pt_gemm_k_grouped_wgrad_pair, a.M, 2 * a.half, a.K, a.dgu_t, a.dgu_t_scale, a.x_t, a.x_t_scale, a.dw_gate_up, a.dw_up, a.half, PT_BF16,
            (int)a.dw_up_add, a.offs, G, a.M, 2 * a.half, a.K, a.stream);
  else {
    PT_STEP(pt_gemm_k_grouped_wgrad_ld, a.M, a.half, a.K, a.dgu_t, a.dgu_t_scale, 2 * a.half, a.x_t, a.x_t_scale, a.K, a.dw_gate_up, PT_BF16,
            (int)a.dw_gate_up_add, a.offs, G, a.M, a.half, a.K, a.stream);
    PT_STEP(pt_gemm_k_grouped_wgrad_ld, a.M, a.half, a.K, (const uint8_t*)a.dgu_t + a.half * a.M, a.dgu_t_scale + a.half, 2 * a.half, a.x_t,
            a.x_t_scale, a.K, a.dw_up, PT_BF16, (int)a.dw_up_add, a.offs, G, a.M, a.half, a.K, a.stream);
  }
  return PT_OK;
}

// out[m, n] = a b^T, its reduction cut into ranges when splits > 1 (fp32 slabs in `slabs`)
static int dense_gemm(const void* a, int64_t lda, const float* as, const void* b, int64_t ldb, const float* bs, void* out, int out_dtype,
                      int64_t M, int64_t N, int64_t K, int64_t splits, int64_t split_len, float* slabs, pt_stream_t stream) {
  if (splits > 1) {
    PT_STEP(pt_gemm_nt_dense_splitk_ld, M, N, K, a, lda, as, b, ldb, bs, slabs, (int32_t)splits, split_len, M, N, K, stream);
    PT_STEP(pt_sum_partials, M, N, splits, slabs, (int32_t)splits, M * N, out, out_dtype, stream);
  } else {
    PT_STEP(pt_gemm_nt_dense_ld, M, N, K, a, lda, as, b, ldb, bs, out, out_dtype, M, N, K, stream);
  }
  return PT_OK;
}

// two independent products, in one launch where they are small and neither is split
static int dense_gemms(const pt_dense_gemm* two, int out_dtype, const int64_t* splits, const int64_t* lens, float* slabs, pt_stream_t stream) {
  if (splits[0] <= 1 && splits[1] <= 1) {
    PT_STEP(pt_gemm_nt_dense_pair, 2 * two[0].M, two[0].N, two[0].K, two, out_dtype, stream);
    return PT_OK;
  }
  for (int i = 0; i < 2; ++i) {
    const pt_dense_gemm& g = two[i];
    if (int rc = dense_gemm(g.a_fp8, g.lda, g.a_scale, g.b_fp8, g.ldb, g.b_scale, g.out, out_dtype, g.M, g.N, g.K, splits[i], lens[i], slabs, stream)) return rc;
  }
  return PT_OK;
}

extern "C" int64_t pt_linear_forward_workspace_bytes(int64_t M, int64_t N, int64_t K, int64_t splits) {
  return up(M * K) + up(4 * M * cdiv(K, 128)) + (splits > 1 ? up(4 * splits * M * N) : 0);
}

extern "C" int pt_linear_forward(const pt_linear_forward_args* args) {
  PT_REQUIRE(args, "linear_forward: null arguments");
  const pt_linear_forward_args& a = *args;
  PT_REQUIRE(a.M > 0 && a.N > 0 && a.K > 0 && a.x && a.workspace, "linear_forward: bad arguments");
  PT_REQUIRE(!a.w || a.x_t, "linear_forward: a weight is quantised together with the transposed input");
  Carve ws(a.workspace);
  void* x_fp8 = ws.bytes(a.M * a.K);
  float* x_s = ws.floats(a.M * cdiv(a.K, 128));
  if (a.w)
    PT_STEP(pt_quant_linear_operands, a.M, a.N, a.K, a.x, a.w, (int)a.dtype, a.M, a.N, a.K, a.ldx, a.ldw, x_fp8, x_s, a.x_t, a.ld_t, a.x_t_scale,
            const_cast<void*>(a.w_fp8), const_cast<float*>(a.w_scale), a.w_t_fp8, a.w_t_scale, a.stream);
  else
    PT_STEP(pt_quant_rowwise_blockwise_transpose_ld, a.M, a.K, a.M, a.x, (int)a.dtype, a.M, a.K, a.ldx, x_fp8, x_s, a.x_t, a.x_t ? a.ld_t : a.M,
            a.x_t_scale, a.stream);
  if (a.y2) {
    PT_STEP(pt_gemm_nt_dense_heads, a.M, a.N, a.K, x_fp8, x_s, a.w_fp8, a.w_scale, a.y, a.y2, a.head_a, a.head_b, a.M, a.N, a.K, a.stream);
    return PT_OK;
  }
  return dense_gemm(x_fp8, a.K, x_s, a.w_fp8, a.K, a.w_scale, a.y, (int)a.y_dtype, a.M, a.N, a.K, a.splits, a.split_len,
                    (float*)(void*)ws.p, a.stream);
}

// Whole 16-byte chunks; from 2048 on whole 128-byte lines, and no multiple of 256 bytes, which would put the rows
// of a reduction step onto few memory channels.
extern "C" int64_t pt_transposed_pitch(int64_t rows) {
  const int64_t red = (rows + 15) & ~(int64_t)15;
  if (red < 2048) return red;
  const int64_t lines = (red + 127) & ~(int64_t)127;
  return lines % 256 == 0 ? lines + 128 : lines;
}

// workspace: gradient bytes and scales | its transposed form and scales | the input's transposed form and
// scales when it is quantised here | slabs of whichever GEMM is split
extern "C" int64_t pt_linear_backward_workspace_bytes(int64_t M, int64_t N, int64_t K, int64_t x_splits, int64_t w_splits, int64_t from_x) {
  const int64_t sx = x_splits > 1 ? 4 * x_splits * M * K : 0, sw = w_splits > 1 ? 4 * w_splits * N * K : 0;
  return up(M * N) + up(4 * M * cdiv(N, 128)) + up(N * (M + 384)) + up(4 * N * cdiv(M, 128)) + up(sx > sw ? sx : sw) +
         (from_x ? up(K * (M + 384)) + up(4 * cdiv(K, 128) * cdiv(M, 128)) : 0);
}

extern "C" int pt_linear_backward(const pt_linear_backward_args* args) {
  PT_REQUIRE(args, "linear_backward: null arguments");
  const pt_linear_backward_args& a = *args;
  PT_REQUIRE(a.M > 0 && a.N > 0 && a.K > 0 && a.grad && a.workspace && (a.x_t || a.x), "linear_backward: bad arguments");
  const int64_t red = (a.M + 15) & ~(int64_t)15;  // the weight gradient's reduction, zero-filled to whole 16-byte chunks
  PT_REQUIRE(!a.x_t || (a.ld_xt >= red && a.ld_xt % 16 == 0),
             "linear_backward: the transposed input needs a row pitch of %lld or more, a multiple of 16", (long long)red);
  const int64_t ld_t = pt_transposed_pitch(a.M);
  Carve ws(a.workspace);
  void* g_fp8 = ws.bytes(a.M * a.N);
  float* g_s = ws.floats(a.M * cdiv(a.N, 128));
  void* g_t = ws.bytes(a.N * (a.M + 384));
  float* g_ts = ws.floats(a.N * cdiv(a.M, 128));
  const void* x_t = a.x_t;
  const float* x_ts = a.x_t_scale;
  int64_t ld_xt = a.ld_xt;
  bool quantised = false;
  if (!x_t) {
    void* t = ws.bytes(a.K * (a.M + 384));
    float* ts = ws.floats(cdiv(a.K, 128) * cdiv(a.M, 128));
    ld_xt = ld_t;
    quantised = a.grad2 && a.dtype == PT_BF16;  // the gradients with it
    if (quantised)
      PT_STEP(pt_quant_heads_and_input, a.M, a.N, a.M, a.grad, a.grad2, a.M, a.N / (a.head_a + a.head_b), a.head_a, a.head_b, g_fp8, g_s, g_t, ld_t, g_ts,
              a.x, a.K, a.ldx, t, ts, a.stream);
    else
      PT_STEP(pt_quant_rowwise_blockwise_transpose_ld, a.M, a.K, a.M, a.x, (int)a.dtype, a.M, a.K, a.ldx, nullptr, nullptr, t, ld_xt, ts, a.stream);
    x_t = t;
    x_ts = ts;
  }
  float* slabs = (float*)(void*)ws.p;
  if (!quantised && a.grad2)
    PT_STEP(pt_quant_heads_rowwise_transpose_ld, a.M, a.N, a.M, a.grad, a.grad2, a.M, a.N / (a.head_a + a.head_b), a.head_a, a.head_b, g_fp8,
            g_s, g_t, ld_t, g_ts, a.stream);
  else if (!quantised)
    PT_STEP(pt_quant_rowwise_transpose_ld, a.M, a.N, a.M, a.grad, (int)a.dtype, a.M, a.N, a.ldg, g_fp8, g_s, g_t, ld_t, g_ts, a.stream);
  const pt_dense_gemm two[2] = {{g_fp8, a.N, g_s, a.w_t_fp8, a.N, a.w_t_scale, a.grad_x, a.M, a.K, a.N},
                                {g_t, ld_t, g_ts, x_t, ld_xt, x_ts, a.grad_w, a.N, a.K, red}};
  const int64_t splits[2] = {a.x_splits, a.w_splits}, lens[2] = {a.x_split_len, a.w_split_len};
  return dense_gemms(two, (int)a.out_dtype, splits, lens, slabs, a.stream);
}

// ---- dense SwiGLU MLP --------------------------------------------------------------------------
// As three linears, two activations and an addition such a layer quantised its input twice, wrote and read
// h, [dgate | dup] and one of two input gradients as bf16, and took 19 launches from five autograd
// nodes; here it is 4 or 5 and 4 to 7 (block of 8192 tokens with a shared MLP of 2048 x 2816: 3717 -> 3593 us).
struct MlpForwardBuffers {
  void *x_fp8, *h_fp8;
  float *x_s, *h_s, *slabs;
  int64_t bytes;
  MlpForwardBuffers(const void* base, int64_t M, int64_t K, int64_t half, int64_t H, int64_t gu_splits, int64_t dn_splits) {
    Carve ws(base);
    x_fp8 = ws.bytes(M * K);
    x_s = ws.floats(M * cdiv(K, 128));
    h_fp8 = ws.bytes(M * half);
    h_s = ws.floats(M * cdiv(half, 128));
    const int64_t a = gu_splits > 1 ? gu_splits * M * 2 * half : 0, b = dn_splits > 1 ? dn_splits * M * H : 0;
    slabs = ws.floats(a > b ? a : b);
    bytes = (int64_t)(ws.p - (uintptr_t)base);
  }
};
extern "C" int64_t pt_mlp_forward_workspace_bytes(int64_t M, int64_t K, int64_t half, int64_t H, int64_t gu_splits, int64_t dn_splits) {
  return MlpForwardBuffers(nullptr, M, K, half, H, gu_splits, dn_splits).bytes;
}

extern "C" int pt_mlp_forward(const pt_mlp_forward_args* args) {
  PT_REQUIRE(args, "mlp_forward: null arguments");
  const pt_mlp_forward_args& a = *args;
  PT_REQUIRE(a.M > 0 && a.K > 0 && a.half > 0 && a.H > 0 && a.half % 128 == 0 && a.K % 16 == 0 && a.H % 16 == 0 && a.ldx >= a.K, "mlp_forward: bad sizes");
  const bool fresh = a.w_gate != nullptr, keep = a.x_t != nullptr;
  PT_REQUIRE(a.x && a.gu_fp8 && a.gu_scale && a.dn_fp8 && a.dn_scale && a.gate_up && a.y && a.workspace && fresh == (a.w_up != nullptr) &&
                 fresh == (a.w_down != nullptr) && (!fresh || (a.gu_t && a.gu_t_scale && a.dn_t && a.dn_t_scale)) &&
                 keep == (a.x_t_scale != nullptr) && keep == (a.h_t != nullptr) && keep == (a.h_t_scale != nullptr), "mlp_forward: null pointer");
  const MlpForwardBuffers b(a.workspace, a.M, a.K, a.half, a.H, a.gu_splits, a.dn_splits);
  const int64_t N = 2 * a.half, ld_t = keep ? a.ld_t : a.M;
  if (fresh) {
    const int64_t blocks = a.half / 128, kb = cdiv(a.K, 128), hb = cdiv(a.H, 128);
    const pt_quant_dense_weight w[3] = {
        {a.w_gate, a.half, a.K, a.ld_gate, a.gu_fp8, a.gu_scale, a.gu_t, N, a.gu_t_scale, 2 * blocks},
        {a.w_up, a.half, a.K, a.ld_up, (uint8_t*)a.gu_fp8 + a.half * a.K, a.gu_scale + blocks * kb, (uint8_t*)a.gu_t + a.half, N, a.gu_t_scale + blocks,
         2 * blocks},
        {a.w_down, a.H, a.half, a.ld_down, a.dn_fp8, a.dn_scale, a.dn_t, a.H, a.dn_t_scale, hb}};
    PT_STEP(pt_quant_dense_operands, a.M, N, a.K, w, 3, a.x, PT_BF16, a.M, a.K, a.ldx, b.x_fp8, b.x_s, a.x_t, ld_t, a.x_t_scale, a.stream);
  } else {
    PT_STEP(pt_quant_rowwise_blockwise_transpose_ld, a.M, a.K, a.M, a.x, PT_BF16, a.M, a.K, a.ldx, b.x_fp8, b.x_s, a.x_t, ld_t, a.x_t_scale, a.stream);
  }
  if (int rc = dense_gemm(b.x_fp8, a.K, b.x_s, a.gu_fp8, a.K, a.gu_scale, a.gate_up, PT_BF16, a.M, N, a.K, a.gu_splits, a.gu_split_len, b.slabs,
                          a.stream)) return rc;
  PT_STEP(pt_silu_mul_quant_rowwise_blockwise_transpose_ld, a.M, a.half, 0, a.gate_up, a.M, a.half, N, b.h_fp8, b.h_s, a.h_t, ld_t, a.h_t_scale,
          a.stream);
  return dense_gemm(b.h_fp8, a.half, b.h_s, a.dn_fp8, a.half, a.dn_scale, a.y, PT_BF16, a.M, a.H, a.half, a.dn_splits, a.dn_split_len, b.slabs,
                    a.stream);
}

struct MlpBackwardBuffers {
  void *dy, *dy_t, *dh, *dgu, *dgu_t;
  float *dy_s, *dy_ts, *dgu_s, *dgu_ts, *slabs;
  int64_t bytes;
  MlpBackwardBuffers(const void* base, int64_t M, int64_t K, int64_t half, int64_t H, const int64_t* splits) {
    Carve ws(base);
    const int64_t N = 2 * half, mb = cdiv(M, 128);
    dy = ws.bytes(M * H);
    dy_s = ws.floats(M * cdiv(H, 128));
    dy_t = ws.bytes(H * (M + 384));
    dy_ts = ws.floats(H * mb);
    dh = ws.bytes(2 * M * half);
    dgu = ws.bytes(M * N);
    dgu_s = ws.floats(M * cdiv(N, 128));
    dgu_t = ws.bytes(N * (M + 384));
    dgu_ts = ws.floats(N * mb);
    const int64_t outputs[4] = {M * half, H * half, M * K, N * K};
    int64_t most = 0;
    for (int i = 0; i < 4; ++i)
      if (splits[i] > 1 && splits[i] * outputs[i] > most) most = splits[i] * outputs[i];
    slabs = ws.floats(most);
    bytes = (int64_t)(ws.p - (uintptr_t)base);
  }
};
extern "C" int64_t pt_mlp_backward_workspace_bytes(int64_t M, int64_t K, int64_t half, int64_t H, const int64_t* splits) {
  return MlpBackwardBuffers(nullptr, M, K, half, H, splits).bytes;
}

extern "C" int pt_mlp_backward(const pt_mlp_backward_args* args) {
  PT_REQUIRE(args, "mlp_backward: null arguments");
  const pt_mlp_backward_args& a = *args;
  PT_REQUIRE(a.M > 0 && a.K > 0 && a.half > 0 && a.H > 0 && a.half % 128 == 0 && a.K % 16 == 0 && a.H % 16 == 0 && a.ldg >= a.H, "mlp_backward: bad sizes");
  PT_REQUIRE(a.grad && a.gu_t && a.gu_t_scale && a.dn_t && a.dn_t_scale && a.gate_up && a.x_t && a.x_t_scale && a.h_t && a.h_t_scale && a.grad_x &&
                 a.grad_gu && a.grad_dn && a.workspace, "mlp_backward: null pointer");
  const int64_t red = (a.M + 15) & ~(int64_t)15, ld_t = pt_transposed_pitch(a.M), N = 2 * a.half;
  PT_REQUIRE(a.ld_t >= red && a.ld_t % 16 == 0, "mlp_backward: the transposed operands need a row pitch of %lld or more, a multiple of 16", (long long)red);
  const MlpBackwardBuffers b(a.workspace, a.M, a.K, a.half, a.H, a.splits);
  PT_STEP(pt_quant_rowwise_transpose_ld, a.M, a.H, a.M, a.grad, PT_BF16, a.M, a.H, a.ldg, b.dy, b.dy_s, b.dy_t, ld_t, b.dy_ts, a.stream);
  const pt_dense_gemm down[2] = {{b.dy, a.H, b.dy_s, a.dn_t, a.H, a.dn_t_scale, b.dh, a.M, a.half, a.H},
                                 {b.dy_t, ld_t, b.dy_ts, a.h_t, a.ld_t, a.h_t_scale, a.grad_dn, a.H, a.half, red}};
  if (int rc = dense_gemms(down, PT_BF16, a.splits, a.split_len, b.slabs, a.stream)) return rc;
  PT_STEP(pt_silu_mul_bwd_quant_rowwise_transpose_ld, a.M, a.half, 0, b.dh, a.half, a.gate_up, N, a.M, a.half, b.dgu, b.dgu_s, b.dgu_t, ld_t, b.dgu_ts,
          a.stream);
  const pt_dense_gemm up[2] = {{b.dgu, N, b.dgu_s, a.gu_t, N, a.gu_t_scale, a.grad_x, a.M, a.K, N},
                               {b.dgu_t, ld_t, b.dgu_ts, a.x_t, a.ld_t, a.x_t_scale, a.grad_gu, N, a.K, red}};
  return dense_gemms(up, PT_BF16, a.splits + 2, a.split_len + 2, b.slabs, a.stream);
}

// Host side of the hot operators as a Python extension: allocations, argument blocks and the dense linear's
// autograd node in C++, the kernels behind the C-ABI of libpithtrain_hip.so as everywhere else.
//
// Layers of a few thousand tokens are bound by what the host does per step.  Written in Python, preparing
// the launches of an expert block's forward and backward took about 90 us and of a dense linear's 40 us,
// on top of 3.5 us per launch in the runtime; torch's allocator alone costs 1.5 us per tensor from Python
// and 0.7 us from here.
//
// No HIP header and no stream query here: the caller passes the stream it is on, and a backward runs on
// the stream of its forward.
#include <torch/extension.h>

#include <dlfcn.h>

#include <optional>

#include "../../include/pithtrain_hip.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
typedef std::optional<Tensor> Maybe;

namespace {

struct HipError : std::runtime_error {
  using std::runtime_error::runtime_error;
};

struct Library {
#define PT_FN(NAME) decltype(&::NAME) NAME = nullptr
  PT_FN(pt_last_error);
  PT_FN(pt_observe);
  PT_FN(pt_quant_blockwise_transpose_batched);
  PT_FN(pt_quant_weights);
  PT_FN(pt_group_rows_workspace_bytes);
  PT_FN(pt_group_rows);
  PT_FN(pt_experts_forward);
  PT_FN(pt_experts_backward);
  PT_FN(pt_experts_weight_gradient);
  PT_FN(pt_linear_forward_workspace_bytes);
  PT_FN(pt_linear_forward);
  PT_FN(pt_linear_backward_workspace_bytes);
  PT_FN(pt_linear_backward);
#undef PT_FN
} lib;

void init(const std::string& path) {
  void* h = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  if (!h) throw HipError(std::string("cannot load ") + path + ": " + dlerror());
  auto get = [&](const char* name) {
    void* p = dlsym(h, name);
    if (!p) throw HipError(path + " lacks " + name);
    return p;
  };
#define PT_FN(NAME) lib.NAME = (decltype(lib.NAME))get(#NAME)
  PT_FN(pt_last_error);
  PT_FN(pt_observe);
  PT_FN(pt_quant_blockwise_transpose_batched);
  PT_FN(pt_quant_weights);
  PT_FN(pt_group_rows_workspace_bytes);
  PT_FN(pt_group_rows);
  PT_FN(pt_experts_forward);
  PT_FN(pt_experts_backward);
  PT_FN(pt_experts_weight_gradient);
  PT_FN(pt_linear_forward_workspace_bytes);
  PT_FN(pt_linear_forward);
  PT_FN(pt_linear_backward_workspace_bytes);
  PT_FN(pt_linear_backward);
#undef PT_FN
}

void check(int rc, const char* what) {
  if (rc) throw HipError(std::string(what) + " failed (" + std::to_string(rc) + "): " + lib.pt_last_error());
}

constexpr auto kFp8 = at::kFloat8_e4m3fn;

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }
int64_t up256(int64_t n) { return (n + 255) & ~(int64_t)255; }
void* ptr(const Tensor& t) { return t.data_ptr(); }
void* ptr(const Maybe& t) { return t ? t->data_ptr() : nullptr; }
Tensor empty(at::IntArrayRef shape, at::ScalarType type, const at::Device& dev) {
  return at::empty(shape, at::TensorOptions().dtype(type).device(dev));
}
int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return PT_BF16;
    case at::kFloat: return PT_F32;
    case at::kHalf: return PT_F16;
    default: throw py::type_error(std::string("unsupported dtype ") + c10::toString(t));
  }
}
Tensor row_major(const Tensor& t) { return t.size(-1) > 0 && t.stride(-1) != 1 ? t.contiguous() : t; }
void require_cuda(const Tensor& t) {
  if (!t.is_cuda()) throw HipError("pith_train_amd operators run on the GPU only (got a tensor on " + t.device().str() + "); there is no CPU path");
}

// Row pitch of a transposed operand: the rule of deepgemm_quantize.transposed_pitch.
int64_t transposed_pitch(int64_t m) {
  m = (m + 15) / 16 * 16;
  return m >= 2048 && m % 256 == 0 ? m + 128 : m;
}

constexpr int64_t kWorkgroups = 256;  // compute units of the MI355X

// (splits, split_len) for out[m, n] = a[m, k] b[n, k]^T.  An output with fewer 256 x 256 tiles than the GPU
// has compute units leaves most of them idle, so its reduction is cut into ranges of whole scale blocks,
// at least 1024 long, that are computed side by side into fp32 slabs and summed afterwards.  Outputs of
// up to 512 128 x 128 tiles take the library's small-tile kernel: when their 64 x 128 tiles are enough for
// half of the compute units, up to a reduction of 8192 that kernel alone beats the slabs and their sum
// (4096 x 512 x 4096: 18.5 us against 28.6 + 6.4), with a quarter up to 4096 (1001 x 512 x 2048: 10.7 us
// against 8.9 + 3.3 and a launch).
std::pair<int64_t, int64_t> split_k(int64_t m, int64_t n, int64_t k) {
  const int64_t tiles = cdiv(m, 256) * cdiv(n, 256);
  if (tiles * 2 > kWorkgroups || k < 2048 || (m * n) % 8) return {1, k};
  const int64_t small = cdiv(m, 64) * cdiv(n, 128);
  if (cdiv(m, 128) * cdiv(n, 128) <= 512 && ((small * 4 >= kWorkgroups && k < 4096) || (small * 2 >= kWorkgroups && k < 8192))) return {1, k};
  const int64_t want = std::min(kWorkgroups / tiles, k / 1024);
  const int64_t len = cdiv(cdiv(k, want), 128) * 128;
  const int64_t splits = cdiv(k, len);
  return splits > 1 ? std::pair<int64_t, int64_t>{splits, len} : std::pair<int64_t, int64_t>{1, k};
}

// ---------------------------------------------------------------------------------------------------------
// weights
// ---------------------------------------------------------------------------------------------------------
// fp8cast_blockwise_transpose of one weight [N, K]
std::tuple<Tensor, Tensor, Tensor, Tensor> quant_weight(const Tensor& weight, int64_t stream) {
  require_cuda(weight);
  const Tensor x = row_major(weight);
  const int64_t N = x.size(0), K = x.size(1), nb = cdiv(N, 128), kb = cdiv(K, 128);
  const auto dev = x.device();
  Tensor q = empty({N, K}, kFp8, dev), s = empty({nb, kb}, at::kFloat, dev), q_t = empty({K, N}, kFp8, dev), s_t = empty({kb, nb}, at::kFloat, dev);
  lib.pt_observe("pt_quant_blockwise_transpose_batched", 1, N, K, 0);
  check(lib.pt_quant_blockwise_transpose_batched(ptr(x), dtype_code(x.scalar_type()), 1, N, K, N * K, N > 1 ? x.stride(0) : K, ptr(q),
                                                 (float*)ptr(s), ptr(q_t), (float*)ptr(s_t), (pt_stream_t)stream), "pt_quant_blockwise_transpose_batched");
  lib.pt_observe("pt_quant_blockwise_transpose_batched", 0, N, K, 0);
  return {q, s, q_t, s_t};
}

// The fused operands [G, sum N_i, K] of lists of grouped weights, all quantised by one launch (no twins).
std::vector<std::pair<Tensor, Tensor>> quant_grouped_weights(const std::vector<std::vector<Tensor>>& weights, int64_t stream) {
  pt_quant_weight parts[PT_QUANT_WEIGHTS_MAX];
  std::vector<std::pair<Tensor, Tensor>> result;
  std::vector<Tensor> keep;
  int n = 0;
  for (const auto& list : weights) {
    const int64_t G = list[0].size(0), K = list[0].size(2);
    int64_t N = 0;
    for (const auto& w : list) {
      require_cuda(w);
      TORCH_CHECK(w.dim() == 3 && w.size(0) == G && w.size(2) == K, "weights of one operand need the same groups and width");
      N += w.size(1);
    }
    const int64_t nb = cdiv(N, 128), kb = cdiv(K, 128);
    Tensor q = empty({G, N, K}, kFp8, list[0].device()), s = empty({G, nb, kb}, at::kFloat, list[0].device());
    int64_t row = 0;
    for (const auto& w : list) {
      TORCH_CHECK(n < PT_QUANT_WEIGHTS_MAX, "too many weights");
      keep.push_back(row_major(w));
      const Tensor& x = keep.back();
      const int64_t rows = x.size(1);
      parts[n++] = {ptr(x), G, rows, K, G > 1 ? x.stride(0) : rows * K, rows > 1 ? x.stride(1) : K, (uint8_t*)ptr(q) + row * K, N * K,
                    (float*)ptr(s) + row / 128 * kb, nb * kb};
      row += rows;
    }
    result.emplace_back(q, s);
  }
  int64_t elements = 0;
  for (int i = 0; i < n; ++i) elements += parts[i].G * parts[i].N * parts[i].K;
  lib.pt_observe("pt_quant_weights", 1, elements, 1, 0);
  check(lib.pt_quant_weights(parts, n, dtype_code(weights[0][0].scalar_type()), (pt_stream_t)stream), "pt_quant_weights");
  lib.pt_observe("pt_quant_weights", 0, elements, 1, 0);
  return result;
}

// ---------------------------------------------------------------------------------------------------------
// dense linear
// ---------------------------------------------------------------------------------------------------------
// Whether the whole-step entry points take both directions of y[m, n] = x[m, k] W^T.
bool linear_supported(const Tensor& x, const Tensor& w_fp8, const Tensor& w_t) {
  const int64_t m = x.size(0), k = x.size(1), n = w_fp8.size(0);
  return (x.scalar_type() == at::kBFloat16 || x.scalar_type() == at::kFloat) && m > 0 && n > 0 && k > 0 && k % 16 == 0 && n % 16 == 0 &&
         w_fp8.is_contiguous() && w_t.is_contiguous();
}

std::tuple<Tensor, Tensor, Tensor> linear_forward(const Tensor& input, const Tensor& w_fp8, const Tensor& w_s, int64_t stream) {
  const Tensor x = row_major(input);
  const int64_t m = x.size(0), k = x.size(1), n = w_fp8.size(0);
  const auto dev = x.device();
  const int64_t ld_t = transposed_pitch(m);
  Tensor y = empty({m, n}, x.scalar_type(), dev), x_t = empty({k, ld_t}, kFp8, dev), x_ts = empty({cdiv(k, 128), cdiv(m, 128)}, at::kFloat, dev);
  const auto [splits, len] = split_k(m, n, k);
  Tensor ws = empty({lib.pt_linear_forward_workspace_bytes(m, n, k, splits)}, at::kByte, dev);
  const int code = dtype_code(x.scalar_type());
  const pt_linear_forward_args a = {ptr(x), code, m, k, m > 1 ? x.stride(0) : k, ptr(w_fp8), (const float*)ptr(w_s), n, ptr(y), code, ptr(x_t), ld_t,
                                    (float*)ptr(x_ts), splits, len, nullptr, 0, 0, ptr(ws), (pt_stream_t)stream};
  check(lib.pt_linear_forward(&a), "pt_linear_forward");
  return {y, x_t, x_ts};
}

struct LinearFunction : torch::autograd::Function<LinearFunction> {
  // weight is an argument for its gradient's sake; the quantised forms are what is read
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, const Tensor& w_fp8, const Tensor& w_s, const Tensor& w_t,
                        const Tensor& w_ts, int64_t stream) {
    auto [y, x_t, x_ts] = linear_forward(x, w_fp8, w_s, stream);
    ctx->save_for_backward({w_t, w_ts, x_t, x_ts});
    ctx->saved_data["stream"] = stream;
    return y;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &w_t = saved[0], &w_ts = saved[1], &x_t = saved[2], &x_ts = saved[3];
    const Tensor g = row_major(grads[0]);
    const int64_t m = g.size(0), n = g.size(1), k = w_t.size(0);
    const auto dev = g.device();
    const auto type = g.scalar_type() == at::kBFloat16 ? at::kBFloat16 : at::kFloat;
    Tensor gx = empty({m, k}, type, dev), gw = empty({n, k}, type, dev);
    const auto [xs, xl] = split_k(m, k, n);
    const auto [ws, wl] = split_k(n, k, cdiv(m, 16) * 16);
    Tensor work = empty({lib.pt_linear_backward_workspace_bytes(m, n, k, xs, ws, 0)}, at::kByte, dev);
    const pt_linear_backward_args a = {ptr(g), dtype_code(g.scalar_type()), m, n, m > 1 ? g.stride(0) : n, ptr(w_t), (const float*)ptr(w_ts), k, ptr(x_t),
                                       x_t.size(1), (const float*)ptr(x_ts), ptr(gx), ptr(gw), dtype_code(type), xs, xl, ws, wl, nullptr, 0,
                                       nullptr, 0, 0, ptr(work), (pt_stream_t)ctx->saved_data["stream"].toInt()};
    check(lib.pt_linear_backward(&a), "pt_linear_backward");
    if (type != g.scalar_type()) {
      gx = gx.to(g.scalar_type());
      gw = gw.to(g.scalar_type());
    }
    return {gx, gw, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// None where the whole-step entry points do not take the shape.
Maybe linear(const Tensor& x, const Tensor& weight, const Tensor& w_fp8, const Tensor& w_s, const Tensor& w_t, const Tensor& w_ts, int64_t stream) {
  require_cuda(x);
  if (!linear_supported(x, w_fp8, w_t)) return std::nullopt;
  return LinearFunction::apply(x, weight, w_fp8, w_s, w_t, w_ts, stream);
}

// Dense linear on two per-head halves (see operators/linear.py).
std::pair<Tensor, Tensor> linear_heads_forward(const Tensor& input, const Tensor& w_fp8, const Tensor& w_s, int64_t heads, int64_t head_a, int64_t head_b,
                                               int64_t stream) {
  const Tensor x = row_major(input);
  const int64_t m = x.size(0), k = x.size(1), n = w_fp8.size(0), na = m * heads * head_a, nb = m * heads * head_b;
  Tensor y = empty({na + nb}, at::kBFloat16, x.device());  // one allocation: the GEMM stores through one descriptor
  Tensor ws = empty({lib.pt_linear_forward_workspace_bytes(m, n, k, 1)}, at::kByte, x.device());
  const pt_linear_forward_args a = {ptr(x), PT_BF16, m, k, m > 1 ? x.stride(0) : k, ptr(w_fp8), (const float*)ptr(w_s), n, ptr(y), PT_BF16, nullptr, 0,
                                    nullptr, 1, k, (char*)ptr(y) + 2 * na, head_a, head_b, ptr(ws), (pt_stream_t)stream};
  check(lib.pt_linear_forward(&a), "pt_linear_forward");
  return {y.narrow(0, 0, na).view({m, heads, head_a}), y.narrow(0, na, nb).view({m, heads, head_b})};
}

std::pair<Tensor, Tensor> linear_heads_backward(const Tensor& grad_a, const Tensor& grad_b, const Tensor& w_t, const Tensor& w_ts, const Tensor& input,
                                                int64_t stream) {
  const Tensor x = row_major(input);
  const int64_t m = grad_a.size(0), heads = grad_a.size(1), head_a = grad_a.size(2), head_b = grad_b.size(2), n = heads * (head_a + head_b), k = x.size(1);
  Tensor gx = empty({m, k}, at::kFloat, x.device()), gw = empty({n, k}, at::kFloat, x.device());
  const auto [xs, xl] = split_k(m, k, n);
  const auto [ws, wl] = split_k(n, k, cdiv(m, 16) * 16);
  Tensor work = empty({lib.pt_linear_backward_workspace_bytes(m, n, k, xs, ws, 1)}, at::kByte, x.device());
  const pt_linear_backward_args a = {ptr(grad_a), PT_BF16, m, n, n, ptr(w_t), (const float*)ptr(w_ts), k, nullptr, 0, nullptr, ptr(gx), ptr(gw), PT_F32,
                                     xs, xl, ws, wl, ptr(x), m > 1 ? x.stride(0) : k, ptr(grad_b), head_a, head_b, ptr(work), (pt_stream_t)stream};
  check(lib.pt_linear_backward(&a), "pt_linear_backward");
  return {gx, gw};
}

// ---------------------------------------------------------------------------------------------------------
// index half of the scatter
// ---------------------------------------------------------------------------------------------------------
// (reverse i64[m] or None, offs i32[G], ks i32[G], src_of i32[cap]): one allocation for the int32 results and
// the workspace, src_of first.
std::tuple<Maybe, Tensor, Tensor, Tensor> group_rows(const Tensor& keys, int64_t G, int64_t alignment, int64_t cap, bool need_reverse, int64_t stream) {
  const int64_t m = keys.size(0), bytes = lib.pt_group_rows_workspace_bytes(m, (int32_t)G);
  const auto dev = keys.device();
  Maybe reverse;
  if (need_reverse) reverse = empty({m}, at::kLong, dev);
  const int64_t o = cdiv(cap, 4) * 4, ws = cdiv(o + 2 * G, 64) * 64;  // in words; the workspace starts on 256 bytes
  Tensor words = empty({ws + bytes / 4}, at::kInt, dev);
  int32_t* at = (int32_t*)ptr(words);
  lib.pt_observe("pt_group_rows", 1, m, G, 0);
  check(lib.pt_group_rows((const int64_t*)ptr(keys), m, (int32_t)G, (int32_t)alignment, at + o, at + o + G, (int64_t*)ptr(reverse), at, cap,
                          bytes ? at + ws : nullptr, bytes, (pt_stream_t)stream), "pt_group_rows");
  lib.pt_observe("pt_group_rows", 0, m, G, 0);
  return {reverse, words.narrow(0, o, G), words.narrow(0, o + G, G), words.narrow(0, 0, cap)};
}

// ---------------------------------------------------------------------------------------------------------
// expert block
// ---------------------------------------------------------------------------------------------------------
// Buffers of one kind: a single allocation while they are small (an allocation costs the host time), one
// each when they are large.
constexpr int64_t kOneBuffer = 32 << 20;
struct Pieces {
  std::vector<int64_t> sizes;
  std::vector<Tensor> buffers;

  explicit Pieces(std::vector<int64_t> s) : sizes(std::move(s)) {}
  void allocate(const at::Device& dev) {
    int64_t total = 0;
    for (int64_t n : sizes) total += up256(n);
    if (total <= kOneBuffer) buffers.push_back(empty({total}, at::kByte, dev));
    else
      for (int64_t n : sizes) buffers.push_back(empty({n}, at::kByte, dev));
  }
  void* at(size_t i) const {
    if (buffers.size() > 1) return ptr(buffers[i]);
    int64_t o = 0;
    for (size_t q = 0; q < i; ++q) o += up256(sizes[q]);
    return (char*)ptr(buffers[0]) + o;
  }
  Tensor piece(size_t i, int64_t rows, int64_t cols, at::ScalarType type) const {
    if (buffers.size() > 1) return buffers[i].view(type).view({rows, cols});
    int64_t o = 0;
    for (size_t q = 0; q < i; ++q) o += up256(sizes[q]);
    return buffers[0].narrow(0, o, sizes[i]).view(type).view({rows, cols});
  }
};

struct Dims {
  int64_t M, K, half, H, G;
  Pieces kept() const { return Pieces({K * M, M / 128 * K * 4, half * M, M / 128 * half * 4}); }            // x^T, h^T with scales
  Pieces forward_temp(bool map) const {                                                                    // composed map, x, h with scales
    return Pieces({map ? 4 * M : 0, M * K, 4 * M * cdiv(K, 128), M * half, 4 * M * cdiv(half, 128)});
  }
  Pieces twins() const { return Pieces({H * M, M / 128 * H * 4, 2 * half * M, M / 128 * half * 8}); }      // dy^T, d(gate_up)^T with scales
  Pieces backward_temp(bool sums) const {                                                                  // dy with scales, grad_h, column sums
    return Pieces({M * H, 4 * M * cdiv(H, 128), 2 * M * half, sums ? M / 128 * half * 8 : 0});
  }
};

// Forward of an expert block (see fused_experts._forward): (out, gate_up, kept buffers).
std::tuple<Tensor, Tensor, std::vector<Tensor>> experts_forward(const Tensor& x, int64_t repeat, const Maybe& row_map, const Maybe& expand_idx,
                                                                const Tensor& offs, const Tensor& gu, const Tensor& gu_s, const Tensor& dn,
                                                                const Tensor& dn_s, int64_t half, const Maybe& gu_bias, const Maybe& dn_bias, bool scatter,
                                                                bool clamped, double alpha, double limit, bool keep, bool few_rows, int64_t stream) {
  const int64_t src_rows = x.size(0), K = x.size(1);
  const Dims d{row_map ? row_map->size(0) : src_rows, K, half, dn.size(1), dn.size(0)};
  const int64_t routed = expand_idx ? expand_idx->size(0) : src_rows * repeat;
  const auto dev = x.device();
  Pieces kept = d.kept(), temp = d.forward_temp((bool)expand_idx);
  if (keep) kept.allocate(dev);
  temp.allocate(dev);
  Tensor gate_up = empty({d.M, 2 * half}, x.scalar_type(), dev);
  Tensor out = empty({scatter ? routed : d.M, d.H}, x.scalar_type(), dev);
  pt_experts_forward_args a = {};
  a.x = ptr(x); a.x_rows = src_rows; a.ldx = src_rows > 1 ? x.stride(0) : K;
  a.M = d.M; a.K = K; a.half = half; a.H = d.H; a.G = d.G;
  a.offs = (const int32_t*)ptr(offs); a.row_map = (const int32_t*)ptr(row_map);
  a.expand_idx = (const int64_t*)ptr(expand_idx); a.n_expand = expand_idx ? routed : 0;
  a.repeat = repeat; a.few_rows = few_rows;
  a.gu_fp8 = ptr(gu); a.gu_scale = (const float*)ptr(gu_s); a.gu_bias = ptr(gu_bias);
  a.dn_fp8 = ptr(dn); a.dn_scale = (const float*)ptr(dn_s); a.dn_bias = ptr(dn_bias);
  a.gate_up = ptr(gate_up); a.out = ptr(out); a.out_rows = out.size(0); a.scatter = scatter;
  a.clamped = clamped; a.alpha = alpha; a.limit = limit;
  if (keep) { a.x_t = kept.at(0); a.x_t_scale = (float*)kept.at(1); a.h_t = kept.at(2); a.h_t_scale = (float*)kept.at(3); }
  a.composed_map = (int32_t*)temp.at(0); a.x_fp8 = temp.at(1); a.x_scale = (float*)temp.at(2); a.h_fp8 = temp.at(3); a.h_scale = (float*)temp.at(4);
  a.stream = (pt_stream_t)stream;
  check(lib.pt_experts_forward(&a), "pt_experts_forward");
  return {out, gate_up, kept.buffers};
}

// Where a weight gradient goes: an existing bf16 gradient is accumulated into by the GEMM, otherwise a new
// tensor becomes, or is added to, the parameter's gradient once the GEMM is queued.
struct Target {
  Tensor weight, out;
  bool add = false;
  void* at() const { return out.defined() ? ptr(out) : nullptr; }
  void aim(const Tensor& w) {
    weight = w;
    const Tensor& grad = w.grad();
    add = grad.defined() && grad.scalar_type() == at::kBFloat16 && grad.is_contiguous();
    out = add ? grad : empty(w.sizes(), at::kBFloat16, w.device());
  }
  void finish() {
    if (!out.defined() || add) return;
    at::NoGradGuard no_grad;
    if (weight.grad().defined()) weight.mutable_grad().add_(out);
    else weight.mutable_grad() = weight.scalar_type() == at::kBFloat16 ? out : out.to(weight.scalar_type());
  }
};

// Backward of an expert block up to the quantised gradient of gate_up; the caller queues the input gradient from
// it and then weight_gradient().
struct ExpertsBackward {
  Dims d;
  pt_experts_backward_args a = {};
  Pieces kept, twins, temp;
  Tensor grad_out, dgu, dgu_s;
  Maybe d_gu_bias, d_dn_bias;
  Target down, gate_up, up;

  ExpertsBackward(const Tensor& grad, const Dims& dims, const Tensor& offs, const Maybe& row_map, bool scatter, const Tensor& dn_dg, const Tensor& dn_dg_s,
                  bool dn_forward, const Tensor& gate_up_saved, std::vector<Tensor> kept_buffers, bool clamped, double alpha, double limit,
                  const Maybe& gu_bias_like, const Maybe& dn_bias_like, const std::vector<Tensor>& weights /* down, gate_up or gate, up; empty: deferred */,
                  int64_t stream)
      : d(dims), kept(d.kept()), twins(d.twins()), temp(d.backward_temp(clamped)) {
    grad_out = grad.contiguous();
    const auto dev = grad_out.device();
    kept.buffers = std::move(kept_buffers);
    twins.allocate(dev);
    temp.allocate(dev);
    dgu = empty({d.M, 2 * d.half}, kFp8, dev);
    dgu_s = empty({d.M, cdiv(2 * d.half, 128)}, at::kFloat, dev);
    if (gu_bias_like) d_gu_bias = empty({d.G, 2 * d.half}, gu_bias_like->scalar_type(), dev);
    if (dn_bias_like) d_dn_bias = empty({d.G, d.H}, dn_bias_like->scalar_type(), dev);
    if (weights.size() > 0) down.aim(weights[0]);
    if (weights.size() > 1) gate_up.aim(weights[1]);
    if (weights.size() > 2) up.aim(weights[2]);
    a.grad_out = ptr(grad_out); a.grad_rows = grad_out.size(0);
    a.M = d.M; a.K = d.K; a.half = d.half; a.H = d.H; a.G = d.G;
    a.offs = (const int32_t*)ptr(offs); a.out_map = scatter ? (const int32_t*)ptr(row_map) : nullptr; a.limit_rows = (bool)row_map;
    a.dn_dg = ptr(dn_dg); a.dn_dg_scale = (const float*)ptr(dn_dg_s); a.dn_forward_layout = dn_forward;
    a.gate_up = ptr(gate_up_saved);
    a.x_t = kept.at(0); a.x_t_scale = (const float*)kept.at(1); a.h_t = kept.at(2); a.h_t_scale = (const float*)kept.at(3);
    a.dgu_fp8 = ptr(dgu); a.dgu_scale = (float*)ptr(dgu_s);
    a.dy_t = twins.at(0); a.dy_t_scale = (float*)twins.at(1); a.dgu_t = twins.at(2); a.dgu_t_scale = (float*)twins.at(3);
    a.dy_fp8 = temp.at(0); a.dy_scale = (float*)temp.at(1); a.grad_h = temp.at(2); a.col_sum = (float*)temp.at(3);
    a.dw_down = down.at(); a.dw_down_add = down.add;
    a.dw_gate_up = gate_up.at(); a.dw_gate_up_add = gate_up.add;
    a.dw_up = up.at(); a.dw_up_add = up.add;
    a.clamped = clamped; a.alpha = alpha; a.limit = limit;
    a.d_gu_bias = ptr(d_gu_bias); a.d_gu_bias_dtype = d_gu_bias ? dtype_code(d_gu_bias->scalar_type()) : 0;
    a.d_dn_bias = ptr(d_dn_bias); a.d_dn_bias_dtype = d_dn_bias ? dtype_code(d_dn_bias->scalar_type()) : 0;
    a.stream = (pt_stream_t)stream;
    check(lib.pt_experts_backward(&a), "pt_experts_backward");
  }

  void weight_gradient() {
    check(lib.pt_experts_weight_gradient(&a), "pt_experts_weight_gradient");
    down.finish();
    gate_up.finish();
    up.finish();
  }

  // the operands of the deferred weight gradients: dy^T, gate_up's^T, x^T, h^T, each with its scales
  std::vector<std::pair<Tensor, Tensor>> operands() const {
    const int64_t blocks = d.M / 128;
    return {{twins.piece(0, d.H, d.M, kFp8), twins.piece(1, blocks, d.H, at::kFloat)},
            {twins.piece(2, 2 * d.half, d.M, kFp8), twins.piece(3, blocks, 2 * d.half, at::kFloat)},
            {kept.piece(0, d.K, d.M, kFp8), kept.piece(1, blocks, d.K, at::kFloat)},
            {kept.piece(2, d.half, d.M, kFp8), kept.piece(3, blocks, d.half, at::kFloat)}};
  }
};

PyObject* g_error = nullptr;

}  // namespace

PYBIND11_MODULE(_host, m) {
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const HipError& e) {
      PyErr_SetString(g_error ? g_error : PyExc_RuntimeError, e.what());
    }
  });
  m.def("init", [](const std::string& path, py::object error) {
    g_error = error.release().ptr();
    init(path);
  });
  m.def("split_k", &split_k);
  m.def("quant_weight", &quant_weight);
  m.def("quant_grouped_weights", &quant_grouped_weights);
  m.def("linear", &linear);
  m.def("linear_heads_forward", &linear_heads_forward);
  m.def("linear_heads_backward", &linear_heads_backward);
  m.def("group_rows", &group_rows);
  m.def("experts_forward", &experts_forward);
  py::class_<ExpertsBackward>(m, "ExpertsBackward")
      .def(py::init([](const Tensor& grad, std::tuple<int64_t, int64_t, int64_t, int64_t, int64_t> dims, const Tensor& offs, const Maybe& row_map,
                       bool scatter, const Tensor& dn_dg, const Tensor& dn_dg_s, bool dn_forward, const Tensor& gate_up, std::vector<Tensor> kept,
                       bool clamped, double alpha, double limit, const Maybe& gu_bias_like, const Maybe& dn_bias_like,
                       const std::vector<Tensor>& weights, int64_t stream) {
        const auto [M, K, half, H, G] = dims;
        return std::make_unique<ExpertsBackward>(grad, Dims{M, K, half, H, G}, offs, row_map, scatter, dn_dg, dn_dg_s, dn_forward, gate_up,
                                                 std::move(kept), clamped, alpha, limit, gu_bias_like, dn_bias_like, weights, stream);
      }))
      .def("weight_gradient", &ExpertsBackward::weight_gradient)
      .def("operands", &ExpertsBackward::operands)
      .def_readonly("dgu", &ExpertsBackward::dgu)
      .def_readonly("dgu_s", &ExpertsBackward::dgu_s)
      .def_readonly("d_gu_bias", &ExpertsBackward::d_gu_bias)
      .def_readonly("d_dn_bias", &ExpertsBackward::d_dn_bias);
}

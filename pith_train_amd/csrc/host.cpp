// Host side of the hot operators as a Python extension: allocations, argument blocks and autograd nodes in C++, the kernels behind the C-ABI of libpithtrain_hip.so as everywhere else.
//
// Layers of a few thousand tokens are bound by what the host does per step.  Written in Python, preparing
// the launches of an expert block's forward and backward took about 90 us and of a dense linear's 40 us,
// on top of 3.5 us per launch in the runtime; torch's allocator alone costs 1.5 us per tensor from Python
// and 0.7 us from here, an autograd node written in Python 10 to 15 us a direction.
//
// No HIP header and no stream query here: the caller passes the stream it is on, and a backward runs on
// the stream of its forward.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/extension.h>

#include <dlfcn.h>

#include <algorithm>
#include <optional>
#include <sstream>

#include "../../include/pithtrain_hip.h"
#include "gemm_rules.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
typedef std::optional<Tensor> Maybe;

namespace {

struct HipError : std::runtime_error {
  using std::runtime_error::runtime_error;
};
struct AssertionError : std::runtime_error {
  using std::runtime_error::runtime_error;
};

PyObject* g_error = nullptr;  // PithTrainHipError (never released)

// Runs a backward and turns what it throws into the Python error that a node written in Python would raise: the
// engine carries nothing but torch's own exceptions over to the caller's thread unchanged.
template <class F>
auto as_python_errors(F f) {
  const auto carry = [](PyObject* type, const char* what) {
    py::gil_scoped_acquire gil;
    if (type) PyErr_SetString(type, what);
    python_error e;
    e.persist();
    throw std::move(e);
  };
  try {
    return f();
  } catch (const HipError& e) {
    carry(g_error ? g_error : PyExc_RuntimeError, e.what());
  } catch (const AssertionError& e) {
    carry(PyExc_AssertionError, e.what());
  } catch (const py::type_error& e) {
    carry(PyExc_TypeError, e.what());
  } catch (py::error_already_set& e) {  // from a callback
    py::gil_scoped_acquire gil;
    e.restore();
    carry(nullptr, nullptr);
  }
  return decltype(f())();
}

struct Library {
#define PT_FN(NAME) decltype(&::NAME) NAME = nullptr
  PT_FN(pt_last_error);
  PT_FN(pt_observe);
  PT_FN(pt_quant_blockwise_transpose_batched);
  PT_FN(pt_quant_weights);
  PT_FN(pt_group_rows_workspace_bytes);
  PT_FN(pt_group_rows);
  PT_FN(pt_experts_forward_by_block);
  PT_FN(pt_experts_forward_without_padding);
  PT_FN(pt_experts_backward_by_block);
  PT_FN(pt_experts_backward_without_padding);
  PT_FN(pt_experts_weight_gradient);
  PT_FN(pt_transposed_pitch);
  PT_FN(pt_linear_forward_workspace_bytes);
  PT_FN(pt_linear_forward);
  PT_FN(pt_linear_backward_workspace_bytes);
  PT_FN(pt_linear_backward);
  PT_FN(pt_mlp_forward_workspace_bytes);
  PT_FN(pt_mlp_forward);
  PT_FN(pt_mlp_backward_workspace_bytes);
  PT_FN(pt_mlp_backward);
  PT_FN(pt_gather_rows);
  PT_FN(pt_gather_rows_backward_workspace_bytes);
  PT_FN(pt_gather_rows_backward);
  PT_FN(pt_gather_rows_backward_begin);
  PT_FN(pt_gather_rows_backward_shared);
  PT_FN(pt_permute_rows);
  PT_FN(pt_silu_mul_fwd);
  PT_FN(pt_silu_mul_bwd);
  PT_FN(pt_moe_combine_fwd);
  PT_FN(pt_moe_combine_bwd);
  PT_FN(pt_moe_combine_ep_index);
  PT_FN(pt_moe_combine_ep_fwd);
  PT_FN(pt_moe_combine_ep_bwd);
  PT_FN(pt_router_topk_fwd);
  PT_FN(pt_router_topk_bwd);
  PT_FN(pt_gate_linear_bwd_workspace_bytes);
  PT_FN(pt_gate_linear_bwd);
  PT_FN(pt_dedup_workspace_bytes);
  PT_FN(pt_dedup_prepare_dispatch);
  PT_FN(pt_build_expert_idxs);
  PT_FN(pt_adjust_expand_idx);
  PT_FN(pt_quant_rowwise_colwise_by_block);
  PT_FN(pt_gemm_m_grouped_by_block);
  PT_FN(pt_gemm_m_grouped_by_block_two);
  PT_FN(pt_gemm_k_grouped_wgrad);
  PT_FN(pt_sum_branches);
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
  PT_FN(pt_experts_forward_by_block);
  PT_FN(pt_experts_forward_without_padding);
  PT_FN(pt_experts_backward_by_block);
  PT_FN(pt_experts_backward_without_padding);
  PT_FN(pt_experts_weight_gradient);
  PT_FN(pt_transposed_pitch);
  PT_FN(pt_linear_forward_workspace_bytes);
  PT_FN(pt_linear_forward);
  PT_FN(pt_linear_backward_workspace_bytes);
  PT_FN(pt_linear_backward);
  PT_FN(pt_mlp_forward_workspace_bytes);
  PT_FN(pt_mlp_forward);
  PT_FN(pt_mlp_backward_workspace_bytes);
  PT_FN(pt_mlp_backward);
  PT_FN(pt_gather_rows);
  PT_FN(pt_gather_rows_backward_workspace_bytes);
  PT_FN(pt_gather_rows_backward);
  PT_FN(pt_gather_rows_backward_begin);
  PT_FN(pt_gather_rows_backward_shared);
  PT_FN(pt_permute_rows);
  PT_FN(pt_silu_mul_fwd);
  PT_FN(pt_silu_mul_bwd);
  PT_FN(pt_moe_combine_fwd);
  PT_FN(pt_moe_combine_bwd);
  PT_FN(pt_moe_combine_ep_index);
  PT_FN(pt_moe_combine_ep_fwd);
  PT_FN(pt_moe_combine_ep_bwd);
  PT_FN(pt_router_topk_fwd);
  PT_FN(pt_router_topk_bwd);
  PT_FN(pt_gate_linear_bwd_workspace_bytes);
  PT_FN(pt_gate_linear_bwd);
  PT_FN(pt_dedup_workspace_bytes);
  PT_FN(pt_dedup_prepare_dispatch);
  PT_FN(pt_build_expert_idxs);
  PT_FN(pt_adjust_expand_idx);
  PT_FN(pt_quant_rowwise_colwise_by_block);
  PT_FN(pt_gemm_m_grouped_by_block);
  PT_FN(pt_gemm_m_grouped_by_block_two);
  PT_FN(pt_gemm_k_grouped_wgrad);
  PT_FN(pt_sum_branches);
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
// Rows that do not overlap, each contiguous: a sum over the rows hands one row of gradients to all of them (pitch 0).
Tensor row_major(const Tensor& t) {
  const bool overlap = t.dim() == 2 && t.size(0) > 1 && t.stride(0) < t.size(1);
  return t.size(-1) > 0 && (t.stride(-1) != 1 || overlap) ? t.contiguous() : t;
}
// contiguous and on a 16-byte boundary, for kernels that take nothing else (a gradient may be a piece of a wider buffer)
Tensor packed(const Tensor& t) {
  const Tensor c = t.contiguous();
  return (uintptr_t)c.data_ptr() % 16 ? c.clone() : c;
}
void require_cuda(const Tensor& t) {
  if (!t.is_cuda()) throw HipError("pith_train_amd operators run on the GPU only (got a tensor on " + t.device().str() + "); there is no CPU path");
}
// Every other operand of a call lives where its input does (undefined: not given): a kernel gets their addresses.
void require_same_device(const Tensor& x, std::initializer_list<const Tensor*> others) {
  require_cuda(x);
  for (const Tensor* t : others)
    if (t->defined() && t->device() != x.device())
      throw HipError("pith_train_amd operators take all of their tensors on one GPU (got " + x.device().str() + " and " + t->device().str() + ")");
}

bool has_tangent(const Tensor& t) { return t.defined() && t._fw_grad(0).defined(); }
void refuse_tangent(const Tensor& t) {
  TORCH_CHECK_NOT_IMPLEMENTED(!has_tangent(t), "pith_train_amd operators have no forward-mode derivative");
}

// A tensor whose address goes to a kernel that derives every index from the sizes given here.
void require_shape(const Tensor& t, at::IntArrayRef shape, at::ScalarType type, const char* what) {
  if (t.sizes() != shape || t.scalar_type() != type || !t.is_contiguous()) {
    std::ostringstream s;
    s << what << ": expected a contiguous " << c10::toString(type) << " tensor of " << shape << ", got " << c10::toString(t.scalar_type()) << ' '
      << t.sizes() << " with strides " << t.strides();
    throw HipError(s.str());
  }
}
// An index that a kernel reads as 64-bit numbers.
void require_index(const Tensor& t, const char* what) {
  if (t.numel() > 0 && (t.dim() != 1 || t.scalar_type() != at::kLong))
    throw py::type_error(std::string(what) + ": expected a one-dimensional int64 index, got " + c10::toString(t.scalar_type()));
}
// the FP8 bytes [G, N, K] of a grouped weight and the scales of its 128 x 128 blocks
void require_operand(const Tensor& q, const Tensor& scale, int64_t G, int64_t N, int64_t K, const char* what) {
  require_shape(q, {G, N, K}, kFp8, what);
  require_shape(scale, {G, cdiv(N, 128), cdiv(K, 128)}, at::kFloat, what);
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
bool linear_supported(const Tensor& x, int64_t n) {
  const int64_t m = x.size(0), k = x.size(1);
  return (x.scalar_type() == at::kBFloat16 || x.scalar_type() == at::kFloat) && m > 0 && n > 0 && k > 0 && k % 16 == 0 && n % 16 == 0;
}

typedef std::tuple<Tensor, Tensor, Tensor, Tensor> QuantisedWeight;  // bytes, scales, transposed bytes, their scales

// (y, x^T, its scales); `fresh`: the weight itself, to be quantised into `q` in the same call
std::tuple<Tensor, Tensor, Tensor> linear_forward(const Tensor& input, const QuantisedWeight& q, const Tensor* fresh, int64_t stream) {
  const auto& [w_fp8, w_s, w_t, w_ts] = q;
  const Tensor x = row_major(input);
  const int64_t m = x.size(0), k = x.size(1), n = w_fp8.size(0);
  const auto dev = x.device();
  const int64_t ld_t = lib.pt_transposed_pitch(m);
  Tensor y = empty({m, n}, x.scalar_type(), dev), x_t = empty({k, ld_t}, kFp8, dev), x_ts = empty({cdiv(k, 128), cdiv(m, 128)}, at::kFloat, dev);
  const auto [splits, len] = split_k(m, n, k);
  Tensor ws = empty({lib.pt_linear_forward_workspace_bytes(m, n, k, splits)}, at::kByte, dev);
  const int code = dtype_code(x.scalar_type());
  const pt_linear_forward_args a = {ptr(x), code, m, k, m > 1 ? x.stride(0) : k,
                                    fresh ? ptr(*fresh) : nullptr, fresh ? (n > 1 ? fresh->stride(0) : k) : 0, fresh ? ptr(w_t) : nullptr,
                                    fresh ? (float*)ptr(w_ts) : nullptr, ptr(w_fp8), (const float*)ptr(w_s), n, ptr(y), code, ptr(x_t), ld_t,
                                    (float*)ptr(x_ts), splits, len, nullptr, 0, 0, ptr(ws), (pt_stream_t)stream};
  check(lib.pt_linear_forward(&a), "pt_linear_forward");
  return {y, x_t, x_ts};
}

// Dense linear on two per-head halves (see operators/linear.py).
std::pair<Tensor, Tensor> linear_heads_forward(const Tensor& input, const Tensor& w_fp8, const Tensor& w_s, int64_t heads, int64_t head_a, int64_t head_b,
                                               int64_t stream) {
  require_same_device(input, {&w_fp8, &w_s});
  const Tensor x = row_major(input);
  const int64_t m = x.size(0), k = x.size(1), n = w_fp8.size(0), na = m * heads * head_a, nb = m * heads * head_b;
  Tensor y = empty({na + nb}, at::kBFloat16, x.device());  // one allocation: the GEMM stores through one descriptor
  Tensor ws = empty({lib.pt_linear_forward_workspace_bytes(m, n, k, 1)}, at::kByte, x.device());
  const pt_linear_forward_args a = {ptr(x), PT_BF16, m, k, m > 1 ? x.stride(0) : k, nullptr, 0, nullptr, nullptr,
                                    ptr(w_fp8), (const float*)ptr(w_s), n, ptr(y), PT_BF16, nullptr, 0,
                                    nullptr, 1, k, (char*)ptr(y) + 2 * na, head_a, head_b, ptr(ws), (pt_stream_t)stream};
  check(lib.pt_linear_forward(&a), "pt_linear_forward");
  return {y.narrow(0, 0, na).view({m, heads, head_a}), y.narrow(0, na, nb).view({m, heads, head_b})};
}

std::pair<Tensor, Tensor> linear_heads_backward(const Tensor& grad_a, const Tensor& grad_b, const Tensor& w_t, const Tensor& w_ts, const Tensor& input,
                                                int64_t stream) {
  require_same_device(input, {&grad_a, &grad_b, &w_t, &w_ts});
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
  at::AutoDispatchBelowADInplaceOrView separate;  // a caller that writes to one of them does not touch the others
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
  Pieces backward_temp(bool sums) const { return Pieces({2 * M * half, sums ? M / 128 * half * 8 : 0}); }  // grad_h, column sums
};

// Whether a training step of `routed` rows leaves out what stands for padding (the _without_padding steps) when the rows go back
// to their places: up to few_used_rows, where groups of whole 128-row blocks are padding for a good part, us a pass with padding
// written / left out: 128 experts of 2048 x 768, 16 rows each 966 / 903, 48 981 / 942, 96 1013 / 1008; 64 of
// 2048 x 1408, 16 839 / 795, 64 860 / 836; and from 64 groups on, whatever their rows, where the kernel of large tiles looks for it
// (gemm_rowsplit.hip has both sides).  Biases and the clamped activation make other values than zero of padding, which the
// column scales of the transposed activations see: such blocks write it.
bool leaves_padding(const Dims& d, int64_t routed, bool biased) { return !biased && (pt::few_used_rows(routed, d.G) || d.G >= 64); }
bool in_whole_chunks(const Tensor& map) { return ((uintptr_t)ptr(map) & 15) == 0; }

// Forward of an expert block (see fused_experts._forward): (out, gate_up, kept buffers, whether padding was left out).
std::tuple<Tensor, Tensor, std::vector<Tensor>, bool> experts_forward(const Tensor& x, int64_t repeat, const Maybe& row_map, const Maybe& expand_idx,
                                                                const Tensor& offs, const Tensor& gu, const Tensor& gu_s, const Tensor& dn,
                                                                const Tensor& dn_s, int64_t half, const Maybe& gu_bias, const Maybe& dn_bias, bool scatter,
                                                                bool clamped, double alpha, double limit, bool keep, bool few_rows, int64_t stream) {
  const auto given = [](const Maybe& t) { return t.value_or(Tensor()); };
  const Tensor maps[] = {given(row_map), given(expand_idx), given(gu_bias), given(dn_bias)};
  require_same_device(x, {&offs, &gu, &gu_s, &dn, &dn_s, &maps[0], &maps[1], &maps[2], &maps[3]});
  const int64_t src_rows = x.size(0), K = x.size(1);
  const Dims d{row_map ? row_map->size(0) : src_rows, K, half, dn.size(1), dn.size(0)};
  const int64_t routed = expand_idx ? expand_idx->size(0) : src_rows * repeat;
  if (x.scalar_type() != at::kBFloat16) throw HipError("expert block: bf16 rows only");
  refuse_tangent(x);
  require_operand(gu, gu_s, d.G, 2 * half, K, "gate_up weight");
  require_operand(dn, dn_s, d.G, d.H, half, "down weight");
  require_shape(offs, {d.G}, at::kInt, "group ends");
  if (gu_bias) require_shape(*gu_bias, {d.G, 2 * half}, x.scalar_type(), "gate_up bias");
  if (dn_bias) require_shape(*dn_bias, {d.G, d.H}, x.scalar_type(), "down bias");
  if (row_map) require_shape(*row_map, {d.M}, at::kInt, "row map");
  if (expand_idx) require_shape(*expand_idx, {routed}, at::kLong, "expanding index");
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
  // (those steps read the map in 16-byte chunks; a slice of a longer one may start anywhere)
  const bool without_padding = row_map && scatter && in_whole_chunks(*row_map) && (keep ? leaves_padding(d, routed, clamped || gu_bias) : few_rows);
  if (without_padding)
    check(lib.pt_experts_forward_without_padding(&a), "pt_experts_forward_without_padding");
  else
    check(lib.pt_experts_forward_by_block(&a), "pt_experts_forward_by_block");
  return {out, gate_up, kept.buffers, without_padding};
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

// [rows, cols] of `type` in a new buffer that holds at least `other` columns
Tensor shared_rows(int64_t rows, int64_t cols, int64_t other, at::ScalarType type, const at::Device& dev) {
  if (cols >= other) return empty({rows, cols}, type, dev);
  return empty({rows * other}, type, dev).narrow(0, 0, rows * cols).view({rows, cols});
}

// [rows, blocks] scales that lie as [blocks, rows], in a new buffer that holds at least `other` blocks
Tensor scales_by_block(int64_t rows, int64_t blocks, int64_t other, const at::Device& dev) {
  const auto options = at::TensorOptions().dtype(at::kFloat).device(dev);
  if (blocks >= other) return at::empty_strided({rows, blocks}, {1, rows}, options);
  return empty({other, rows}, at::kFloat, dev).narrow(0, 0, blocks).t();
}

// Backward of an expert block up to the quantised gradient of gate_up; the caller queues the input gradient from
// it and then weight_gradient().  A buffer goes back to the allocator when its last reader is queued (the next
// user is behind it on the stream), and the gradient of gate_up is written over the one of the output, which only
// the GEMM before it reads: at 32k tokens these are 0.6 GB each.
struct ExpertsBackward {
  Dims d;
  pt_experts_backward_args a = {};
  Pieces kept, twins;
  std::vector<Tensor> weights;
  Tensor grad_out, dgu, dgu_s;
  Maybe d_gu_bias, d_dn_bias;
  Target down, gate_up, up;

  ExpertsBackward(const Tensor& grad, const Dims& dims, const Tensor& offs, const Maybe& row_map, bool scatter, bool without_padding, const Tensor& dn_dg, const Tensor& dn_dg_s,
                  bool dn_forward, const Tensor& gate_up_saved, std::vector<Tensor> kept_buffers, bool clamped, double alpha, double limit,
                  const Maybe& gu_bias_like, const Maybe& dn_bias_like, std::vector<Tensor> weights_ /* down, gate_up or gate, up; empty: deferred */,
                  int64_t stream)
      : d(dims), kept(d.kept()), twins(d.twins()), weights(std::move(weights_)) {
    Pieces temp = d.backward_temp(clamped);
    grad_out = grad.contiguous();
    const auto dev = grad_out.device();
    kept.buffers = std::move(kept_buffers);
    twins.allocate(dev);
    temp.allocate(dev);
    dgu = shared_rows(d.M, 2 * d.half, d.H, kFp8, dev);
    dgu_s = scales_by_block(d.M, cdiv(2 * d.half, 128), cdiv(d.H, 128), dev);
    if (gu_bias_like) d_gu_bias = empty({d.G, 2 * d.half}, gu_bias_like->scalar_type(), dev);
    if (dn_bias_like) d_dn_bias = empty({d.G, d.H}, dn_bias_like->scalar_type(), dev);
    if (weights.size() > 0) down.aim(weights[0]);
    a.grad_out = ptr(grad_out); a.grad_rows = grad_out.size(0);
    a.M = d.M; a.K = d.K; a.half = d.half; a.H = d.H; a.G = d.G;
    a.offs = (const int32_t*)ptr(offs); a.out_map = scatter ? (const int32_t*)ptr(row_map) : nullptr; a.limit_rows = (bool)row_map;
    a.dn_dg = ptr(dn_dg); a.dn_dg_scale = (const float*)ptr(dn_dg_s); a.dn_forward_layout = dn_forward;
    a.gate_up = ptr(gate_up_saved);
    a.x_t = kept.at(0); a.x_t_scale = (const float*)kept.at(1); a.h_t = kept.at(2); a.h_t_scale = (const float*)kept.at(3);
    a.dgu_fp8 = ptr(dgu); a.dgu_scale = (float*)ptr(dgu_s);
    a.dy_t = twins.at(0); a.dy_t_scale = (float*)twins.at(1); a.dgu_t = twins.at(2); a.dgu_t_scale = (float*)twins.at(3);
    a.dy_fp8 = ptr(dgu); a.dy_scale = (float*)ptr(dgu_s); a.grad_h = temp.at(0); a.col_sum = (float*)temp.at(1);
    a.dw_down = down.at(); a.dw_down_add = down.add;
    a.clamped = clamped; a.alpha = alpha; a.limit = limit;
    a.d_gu_bias = ptr(d_gu_bias); a.d_gu_bias_dtype = d_gu_bias ? dtype_code(d_gu_bias->scalar_type()) : 0;
    a.d_dn_bias = ptr(d_dn_bias); a.d_dn_bias_dtype = d_dn_bias ? dtype_code(d_dn_bias->scalar_type()) : 0;
    a.stream = (pt_stream_t)stream;
    if (without_padding)
      check(lib.pt_experts_backward_without_padding(&a), "pt_experts_backward_without_padding");
    else
      check(lib.pt_experts_backward_by_block(&a), "pt_experts_backward_by_block");
    grad_out.reset();
  }

  void weight_gradient() {
    gate_up.aim(weights[1]);
    if (weights.size() > 2) up.aim(weights[2]);
    a.dw_gate_up = gate_up.at(); a.dw_gate_up_add = gate_up.add;
    a.dw_up = up.at(); a.dw_up_add = up.add;
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

// ---------------------------------------------------------------------------------------------------------
// autograd nodes
// ---------------------------------------------------------------------------------------------------------
// Python objects the nodes call back into (never released: they live as long as the process)
PyObject *g_store = nullptr, *g_schedule = nullptr, *g_dgrad = nullptr;

// A tensor kept for the backward as autograd keeps its own: a write to it before the backward is found out, and
// saved-tensor hooks see it.  What a hook gives back goes to kernels by address, so it has to be what was saved.
struct Saved {
  torch::autograd::SavedVariable v;
  std::vector<int64_t> sizes, strides;  // with hooks only
  at::TensorOptions options;
  Saved() = default;
  Saved(const Tensor& t) : v(t, false) {
    if (!v.has_hooks()) return;
    sizes = t.sizes().vec();
    strides = t.strides().vec();
    options = t.options();
  }
  Tensor get() const {
    const Tensor t = v.unpack();
    if (!v.has_hooks()) return t;
    TORCH_CHECK(t.defined() && t.sizes() == sizes && t.scalar_type() == c10::typeMetaToScalarType(options.dtype()) && t.device() == options.device(),
                "a saved-tensor hook gave back another size, type or device than it was given");
    if (t.strides() == strides) return t;
    Tensor same = at::empty_strided(sizes, strides, options);
    return same.copy_(t.detach());
  }
  void reset() { v.reset_data(); }
};

struct HipNode : torch::autograd::Node {
  pt_stream_t stream = nullptr;
  bool released = false;
  virtual variable_list run(variable_list&& grads) = 0;
  // the gradients as torch's operators make them, for nodes whose backward can be differentiated
  virtual std::optional<variable_list> differentiable(const variable_list& grads) { return std::nullopt; }
  virtual void drop() = 0;
  variable_list apply(variable_list&& grads) override {
    return as_python_errors([&] { return backward(std::move(grads)); });
  }
  variable_list backward(variable_list&& grads) {
    TORCH_CHECK(!released, "the saved tensors of ", name(), " are gone: a second backward needs retain_graph=True for the first one");
    const bool twice = at::GradMode::is_enabled();  // create_graph=True
    if (twice)
      if (auto result = differentiable(grads)) return *result;
    const variable_list given = twice ? grads : variable_list();
    variable_list result;
    {
      at::AutoDispatchBelowADInplaceOrView guard;
      result = run(std::move(grads));
    }
    if (twice) refuse_second(result, given);
    return result;
  }
  // A kernel's result has no graph: differentiating it again raises instead of passing for a constant.
  void refuse_second(variable_list& result, const variable_list& given) {
    for (Tensor& t : result) {
      if (!t.defined() || std::any_of(given.begin(), given.end(), [&](const Tensor& g) { return g.is_same(t); })) continue;
      std::shared_ptr<torch::autograd::Error> error(new torch::autograd::Error("the backward of " + name() + " cannot be differentiated"),
                                                    torch::autograd::deleteNode);
      torch::autograd::set_history(t, error);
    }
  }
  void release_variables() override {
    released = true;
    drop();
  }
};

template <class N, class... Inputs>
std::shared_ptr<N> make_node(int64_t stream, const Inputs&... inputs) {
  std::shared_ptr<N> node(new N(), torch::autograd::deleteNode);
  node->stream = (pt_stream_t)stream;
  node->set_next_edges(torch::autograd::collect_next_edges(inputs...));
  return node;
}

// Runs `compute` below autograd and, when one of the inputs wants a gradient, hangs its result (a fresh
// tensor) on a node that `fill` completes.
template <class N, class Compute, class Fill, class... Inputs>
Tensor with_node(int64_t stream, Compute compute, Fill fill, const Inputs&... inputs) {
  const bool wants = torch::autograd::compute_requires_grad(inputs...);
  (refuse_tangent(inputs), ...);
  Tensor out;
  {
    at::AutoDispatchBelowADInplaceOrView guard;
    out = compute();
  }
  if (wants) {
    auto node = make_node<N>(stream, inputs...);
    fill(*node);
    torch::autograd::set_history(out, node);
  }
  return out;
}

bool deferred_gradients() {  // WeightGradStore.enabled; needs the GIL
  return py::handle(g_store).attr("enabled").cast<bool>();
}

// ---- rows moved through an index --------------------------------------------------------------------------
constexpr int64_t kRowAlignment = 1024;

Tensor gather_into(const Tensor& src, const Tensor& index, const Tensor& out, pt_stream_t stream) {
  const int64_t n = index.size(0);
  if (n > 0 && src.size(1) > 0)
    check(lib.pt_gather_rows(ptr(src), src.stride(0), ptr(out), out.stride(0), (const int64_t*)ptr(index), n, src.size(1), (int32_t)src.element_size(),
                             stream), "pt_gather_rows");
  return out;
}

// Sum of the rows of `grad` that share an index, in a buffer of whole 1024 rows.
Tensor scatter_sum(const Tensor& grad, const Tensor& index, int64_t rows, int64_t alignment, int64_t stream) {
  std::vector<int64_t> shape = grad.sizes().vec();
  shape[0] = cdiv(rows, alignment) * alignment;
  Tensor out = empty(shape, grad.scalar_type(), grad.device());
  const int64_t n = index.size(0);
  int64_t H = 1;
  for (size_t i = 1; i < shape.size(); ++i) H *= shape[i];
  if (rows && H) {
    const Tensor go = grad.contiguous(), idx = index.contiguous();
    const int64_t bytes = lib.pt_gather_rows_backward_workspace_bytes(n, rows);
    Tensor ws = empty({std::max<int64_t>(bytes, 256)}, at::kByte, grad.device());
    check(lib.pt_gather_rows_backward(ptr(go), H, ptr(out), H, (const int64_t*)ptr(idx), n, rows, H, dtype_code(grad.scalar_type()), ptr(ws),
                                      ws.numel(), (pt_stream_t)stream), "pt_gather_rows_backward");
  }
  return out.narrow(0, 0, rows);
}

struct GatherNode : HipNode {
  Saved index;
  int64_t rows, alignment;
  void drop() override { index.reset(); }
  variable_list run(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor()};
    return {scatter_sum(g[0], index.get(), rows, alignment, (int64_t)stream)};
  }
};

Tensor index_gather(const Tensor& input, const Tensor& index, int64_t alignment, int64_t stream) {
  require_same_device(input, {&index});
  require_index(index, "padded_index_gather");
  return with_node<GatherNode>(
      stream,
      [&] {
        const int64_t n = index.size(0);
        std::vector<int64_t> shape = input.sizes().vec();
        shape[0] = cdiv(n, alignment) * alignment;
        Tensor buf = empty(shape, input.scalar_type(), input.device());
        Tensor out = buf.narrow(0, 0, n);
        if (n) {
          const Tensor src = row_major(input.reshape({input.size(0), -1}));
          gather_into(src, index.contiguous(), out.view({n, -1}), (pt_stream_t)stream);
        }
        return out;
      },
      [&](GatherNode& node) {
        node.index = Saved(index);
        node.rows = input.size(0);
        node.alignment = alignment;
      },
      input);
}

// Rows grouped by expert (ScatterForGroupedGemm): the caller sorted the indices; backward: gather.
struct PermuteNode : HipNode {
  Saved reverse, pre;
  bool expanded;
  int64_t in_rows;
  void drop() override { reverse.reset(); pre.reset(); }
  variable_list run(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor()};
    const Tensor go = g[0].contiguous(), index = reverse.get();
    Tensor grad = gather_into(go, index, empty({index.size(0), go.size(1)}, go.scalar_type(), go.device()), stream);
    return {expanded ? scatter_sum(grad, pre.get(), in_rows, kRowAlignment, (int64_t)stream) : grad};
  }
};

Tensor permute_rows(const Tensor& input, const Tensor& src_of, const Tensor& offs, const Tensor& reverse, const Maybe& pre, const Tensor& buffer,
                    int64_t rows, int64_t stream) {
  return with_node<PermuteNode>(
      stream, [&] { return buffer.narrow(0, 0, rows); },
      [&](PermuteNode& node) {
        node.reverse = Saved(reverse);
        node.expanded = (bool)pre;
        if (pre) node.pre = Saved(*pre);
        node.in_rows = input.size(0);
      },
      input);
}
// The row copy itself, queued before the caller waits for the group sizes.
Tensor permute_into_buffer(const Tensor& input, const Tensor& src_of, const Tensor& offs, const Maybe& pre, int64_t stream) {
  const Tensor index = pre.value_or(Tensor());
  require_same_device(input, {&src_of, &offs, &index});
  if (pre) require_index(*pre, "scatter_for_grouped_gemm: pre_index");
  at::AutoDispatchBelowADInplaceOrView guard;
  const Tensor in = row_major(input), through = index.defined() ? index.contiguous() : Tensor();
  Tensor buf = empty({src_of.size(0), in.size(1)}, in.scalar_type(), in.device());
  check(lib.pt_permute_rows(ptr(in), in.stride(0), ptr(buf), buf.stride(0), (const int32_t*)ptr(src_of), index.defined() ? (const int64_t*)ptr(through) : nullptr,
                            (const int32_t*)ptr(offs) + offs.size(0) - 1, (int32_t)kRowAlignment, buf.size(0), in.size(1), (int32_t)in.element_size(),
                            (pt_stream_t)stream), "pt_permute_rows");
  return buf;
}

// ---- SwiGLU -----------------------------------------------------------------------------------------------
struct SiluMulNode : HipNode {
  Saved gate, up;
  void drop() override { gate.reset(); up.reset(); }
  variable_list run(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor(), Tensor()};
    const Tensor a = gate.get(), b = up.get();
    if (g[0].sizes() != a.sizes()) throw AssertionError("grad_output shape != gate shape");
    if (g[0].scalar_type() != a.scalar_type()) throw AssertionError("grad_output dtype differs from gate's");
    if (!g[0].is_contiguous()) throw AssertionError("grad_output must be contiguous");
    Tensor da = empty(a.sizes(), a.scalar_type(), a.device()), db = empty(a.sizes(), a.scalar_type(), a.device());
    check(lib.pt_silu_mul_bwd(ptr(g[0]), ptr(a), ptr(b), ptr(da), ptr(db), a.numel(), dtype_code(a.scalar_type()), stream), "pt_silu_mul_bwd");
    return {da, db};
  }
};

Tensor silu_mul(const Tensor& gate, const Tensor& up, int64_t stream) {
  require_same_device(gate, {&up});
  return with_node<SiluMulNode>(
      stream,
      [&] {
        Tensor out = empty(gate.sizes(), gate.scalar_type(), gate.device());
        check(lib.pt_silu_mul_fwd(ptr(gate), ptr(up), ptr(out), gate.numel(), dtype_code(gate.scalar_type()), (pt_stream_t)stream), "pt_silu_mul_fwd");
        return out;
      },
      [&](SiluMulNode& node) {
        node.gate = Saved(gate);
        node.up = Saved(up);
      },
      gate, up);
}

// ---- dense linear -----------------------------------------------------------------------------------------
struct LinearNode : HipNode {
  Saved weight_t, weight_ts, input_t, input_ts;
  void drop() override { for (Saved* s : {&weight_t, &weight_ts, &input_t, &input_ts}) s->reset(); }
  variable_list run(variable_list&& grads) override {
    if (!grads[0].defined()) return {Tensor(), Tensor()};
    const Tensor w_t = weight_t.get(), w_ts = weight_ts.get(), x_t = input_t.get(), x_ts = input_ts.get(), g = row_major(grads[0]);
    const int64_t m = g.size(0), n = g.size(1), k = w_t.size(0);
    const auto dev = g.device();
    const auto type = g.scalar_type() == at::kBFloat16 ? at::kBFloat16 : at::kFloat;
    Tensor gx = empty({m, k}, type, dev), gw = empty({n, k}, type, dev);
    const auto [xs, xl] = split_k(m, k, n);
    const auto [ws, wl] = split_k(n, k, cdiv(m, 16) * 16);
    Tensor work = empty({lib.pt_linear_backward_workspace_bytes(m, n, k, xs, ws, 0)}, at::kByte, dev);
    const pt_linear_backward_args a = {ptr(g), dtype_code(g.scalar_type()), m, n, m > 1 ? g.stride(0) : n, ptr(w_t), (const float*)ptr(w_ts), k, ptr(x_t),
                                       x_t.size(1), (const float*)ptr(x_ts), ptr(gx), ptr(gw), dtype_code(type), xs, xl, ws, wl, nullptr, 0,
                                       nullptr, 0, 0, ptr(work), stream};
    check(lib.pt_linear_backward(&a), "pt_linear_backward");
    if (type != g.scalar_type()) {
      gx = gx.to(g.scalar_type());
      gw = gw.to(g.scalar_type());
    }
    return {gx, gw};
  }
};

// weight is an argument for its gradient's sake; the quantised forms are what is read
Tensor linear_node(const Tensor& x, const Tensor& weight, const QuantisedWeight& q, const Tensor* fresh, int64_t stream) {
  Tensor x_t, x_ts;
  return with_node<LinearNode>(
      stream,
      [&] {
        Tensor y;
        std::tie(y, x_t, x_ts) = linear_forward(x, q, fresh, stream);
        return y;
      },
      [&](LinearNode& node) {
        node.weight_t = Saved(std::get<2>(q));
        node.weight_ts = Saved(std::get<3>(q));
        node.input_t = Saved(x_t);
        node.input_ts = Saved(x_ts);
      },
      x, weight);
}

// None where the whole-step entry points do not take the shape.
Maybe linear(const Tensor& x, const Tensor& weight, const Tensor& w_fp8, const Tensor& w_s, const Tensor& w_t, const Tensor& w_ts, int64_t stream) {
  require_same_device(x, {&weight, &w_fp8, &w_s, &w_t, &w_ts});
  // the GEMM walks the weight at x's width: a wider input would be multiplied with memory past it
  if (x.size(1) != w_fp8.size(1) || w_t.size(0) != x.size(1) || w_t.size(1) != w_fp8.size(0))
    throw HipError("linear: an input of width " + std::to_string(x.size(1)) + " for a weight of " + std::to_string(w_fp8.size(0)) + " x " +
                   std::to_string(w_fp8.size(1)));
  if (!linear_supported(x, w_fp8.size(0)) || !w_fp8.is_contiguous() || !w_t.is_contiguous()) return std::nullopt;
  const int64_t nb = cdiv(w_fp8.size(0), 128), kb = cdiv(w_fp8.size(1), 128);
  require_shape(w_s, {nb, kb}, at::kFloat, "linear: scales of the quantised weight");
  require_shape(w_ts, {kb, nb}, at::kFloat, "linear: scales of the transposed weight");
  return linear_node(x, weight, QuantisedWeight{w_fp8, w_s, w_t, w_ts}, nullptr, stream);
}

// The same with a weight that has not been quantised yet: (result, its quantised forms), or two Nones.
std::pair<Maybe, std::optional<QuantisedWeight>> linear_fresh(const Tensor& x, const Tensor& weight, int64_t stream) {
  require_same_device(x, {&weight});
  if (weight.dim() != 2 || weight.size(1) != x.size(1) || !linear_supported(x, weight.size(0))) return {std::nullopt, std::nullopt};
  const Tensor w = row_major(weight.detach());
  const int64_t N = w.size(0), K = w.size(1), nb = cdiv(N, 128), kb = cdiv(K, 128);
  const auto dev = w.device();
  QuantisedWeight q{empty({N, K}, kFp8, dev), empty({nb, kb}, at::kFloat, dev), empty({K, N}, kFp8, dev), empty({kb, nb}, at::kFloat, dev)};
  Tensor y = linear_node(x, weight, q, &w, stream);
  return {y, q};
}

// ---- dense SwiGLU MLP -------------------------------------------------------------------------------------
struct MlpNode : HipNode {
  enum { GU_T, GU_TS, DN_T, DN_TS, GATE_UP, X_T, X_TS, H_T, H_TS, COUNT };  // transposed weights, gate_up, transposed activations; scales
  Saved kept[COUNT];
  int64_t M;
  void drop() override { for (Saved& s : kept) s.reset(); }
  variable_list run(variable_list&& grads) override {
    if (!grads[0].defined()) return variable_list(4);
    Tensor t[COUNT];
    for (int i = 0; i < COUNT; ++i) t[i] = kept[i].get();
    const Tensor &x_t = t[X_T], &h_t = t[H_T], g = row_major(grads[0]);
    const int64_t K = x_t.size(0), half = h_t.size(0), H = t[DN_T].size(1);
    const auto dev = g.device();
    Tensor gx = empty({M, K}, at::kBFloat16, dev), ggu = empty({2 * half, K}, at::kBFloat16, dev), gdn = empty({H, half}, at::kBFloat16, dev);
    pt_mlp_backward_args a = {ptr(g), M, K, half, H, M > 1 ? g.stride(0) : H, ptr(t[GU_T]), (const float*)ptr(t[GU_TS]), ptr(t[DN_T]),
                              (const float*)ptr(t[DN_TS]), ptr(t[GATE_UP]), ptr(x_t), (const float*)ptr(t[X_TS]), ptr(h_t), (const float*)ptr(t[H_TS]),
                              x_t.size(1), ptr(gx), ptr(ggu), ptr(gdn), {}, {}, nullptr, stream};
    const int64_t red = cdiv(M, 16) * 16, shapes[4][3] = {{M, half, H}, {H, half, red}, {M, K, 2 * half}, {2 * half, K, red}};
    for (int i = 0; i < 4; ++i) std::tie(a.splits[i], a.split_len[i]) = split_k(shapes[i][0], shapes[i][1], shapes[i][2]);
    Tensor ws = empty({lib.pt_mlp_backward_workspace_bytes(M, K, half, H, a.splits)}, at::kByte, dev);
    a.workspace = ptr(ws);
    check(lib.pt_mlp_backward(&a), "pt_mlp_backward");
    return {gx, ggu.narrow(0, 0, half), ggu.narrow(0, half, half), gdn};
  }
};

// y = down(silu(gate(x)) * up(x)) for bf16 x [M, K]; `cached`: the quantised weights (gate | up as one operand, and down:
// bytes, scales and their transposed forms, eight tensors) when there are any, else they are quantised in the same call.  (y, those tensors), or two Nones where the
// library does not take the shapes.
std::pair<Maybe, std::optional<std::vector<Tensor>>> mlp(const Tensor& input, const Tensor& w_gate, const Tensor& w_up, const Tensor& w_down,
                                                         const std::optional<std::vector<Tensor>>& cached, int64_t stream) {
  require_same_device(input, {&w_gate, &w_up, &w_down});
  if (cached)
    for (const Tensor& q : *cached) require_same_device(input, {&q});
  const int64_t M = input.size(0), K = input.size(1), half = w_gate.size(0), H = w_down.size(0);
  const auto bf16 = at::kBFloat16;
  if (input.scalar_type() != bf16 || w_gate.scalar_type() != bf16 || w_up.scalar_type() != bf16 || w_down.scalar_type() != bf16 || w_gate.dim() != 2 ||
      w_up.sizes() != w_gate.sizes() || w_gate.size(1) != K || w_down.size(1) != half || M == 0 || half == 0 || half % 128 || K == 0 || K % 16 || H == 0 || H % 16)
    return {std::nullopt, std::nullopt};
  const bool keep = torch::autograd::compute_requires_grad(input, w_gate, w_up, w_down);
  if (has_tangent(input) || has_tangent(w_gate) || has_tangent(w_up) || has_tangent(w_down)) return {std::nullopt, std::nullopt};
  std::vector<Tensor> t;
  auto node = keep ? make_node<MlpNode>(stream, input, w_gate, w_up, w_down) : nullptr;
  Tensor y;
  {
    at::AutoDispatchBelowADInplaceOrView guard;
    const auto dev = input.device();
    const int64_t N = 2 * half, nb = cdiv(N, 128), kb = cdiv(K, 128), hb = half / 128, Hb = cdiv(H, 128);
    const Tensor x = row_major(input), wg = row_major(w_gate), wu = row_major(w_up), wd = row_major(w_down);
    if (cached) {
      t = *cached;
      if (t.size() != 8) throw HipError("mlp: eight quantised tensors");
      const int64_t sizes[4][2] = {{N, K}, {K, N}, {H, half}, {half, H}};
      for (int i = 0; i < 4; ++i) {
        require_shape(t[2 * i], {sizes[i][0], sizes[i][1]}, kFp8, "mlp: quantised weight");
        require_shape(t[2 * i + 1], {cdiv(sizes[i][0], 128), cdiv(sizes[i][1], 128)}, at::kFloat, "mlp: scales of a quantised weight");
      }
    } else t = {empty({N, K}, kFp8, dev), empty({nb, kb}, at::kFloat, dev), empty({K, N}, kFp8, dev), empty({kb, nb}, at::kFloat, dev),
              empty({H, half}, kFp8, dev), empty({Hb, hb}, at::kFloat, dev), empty({half, H}, kFp8, dev), empty({hb, Hb}, at::kFloat, dev)};
    const int64_t ld_t = lib.pt_transposed_pitch(M);
    Tensor gate_up = empty({M, N}, bf16, dev), x_t, x_ts, h_t, h_ts;
    y = empty({M, H}, bf16, dev);
    if (keep) {
      x_t = empty({K, ld_t}, kFp8, dev);
      x_ts = empty({kb, cdiv(M, 128)}, at::kFloat, dev);
      h_t = empty({half, ld_t}, kFp8, dev);
      h_ts = empty({hb, cdiv(M, 128)}, at::kFloat, dev);
    }
    const auto [gs, gl] = split_k(M, N, K);
    const auto [ds, dl] = split_k(M, H, half);
    Tensor ws = empty({lib.pt_mlp_forward_workspace_bytes(M, K, half, H, gs, ds)}, at::kByte, dev);
    auto opt = [](const Tensor& v) { return v.defined() ? v.data_ptr() : nullptr; };
    auto pitch = [](const Tensor& v) { return v.size(0) > 1 ? v.stride(0) : v.size(1); };
    const pt_mlp_forward_args a = {ptr(x), M, K, pitch(x), half, H,
                                   cached ? nullptr : ptr(wg), pitch(wg), cached ? nullptr : ptr(wu), pitch(wu), cached ? nullptr : ptr(wd), pitch(wd),
                                   ptr(t[0]), (float*)ptr(t[1]), ptr(t[2]), (float*)ptr(t[3]), ptr(t[4]), (float*)ptr(t[5]), ptr(t[6]), (float*)ptr(t[7]),
                                   ptr(gate_up), ptr(y), opt(x_t), (float*)opt(x_ts), opt(h_t), (float*)opt(h_ts), ld_t, gs, gl, ds, dl, ptr(ws),
                                   (pt_stream_t)stream};
    check(lib.pt_mlp_forward(&a), "pt_mlp_forward");
    if (keep) {
      const Tensor kept[MlpNode::COUNT] = {t[2], t[3], t[6], t[7], gate_up, x_t, x_ts, h_t, h_ts};
      for (int i = 0; i < MlpNode::COUNT; ++i) node->kept[i] = Saved(kept[i]);
      node->M = M;
    }
  }
  if (keep) torch::autograd::set_history(y, node);
  return {y, t};
}

// ---- grouped linear ---------------------------------------------------------------------------------------
// Row- and column-scaled FP8 forms of x [M, N], M % 128 == 0: bytes, scales [N/128, M], transposed bytes, their scales
struct Quantised {
  Tensor q, s, q_t, s_t;
  Quantised() = default;
  Quantised(const Tensor& input, pt_stream_t stream) {
    const Tensor x = row_major(input);
    const int64_t M = x.size(0), N = x.size(1);
    const auto dev = x.device();
    q = empty({M, N}, kFp8, dev);
    s = empty({cdiv(N, 128), M}, at::kFloat, dev);
    q_t = empty({N, M}, kFp8, dev);
    s_t = empty({M / 128, N}, at::kFloat, dev);
    lib.pt_observe("pt_quant_rowwise_colwise", 1, M, N, M);
    check(lib.pt_quant_rowwise_colwise_by_block(ptr(x), dtype_code(x.scalar_type()), M, N, M > 1 ? x.stride(0) : N, ptr(q), (float*)ptr(s), ptr(q_t),
                                                (float*)ptr(s_t), stream), "pt_quant_rowwise_colwise");
    lib.pt_observe("pt_quant_rowwise_colwise", 0, M, N, M);
  }
};

// The GEMM of a fused step's own operand (its row scales lie as [K/128, M]), from Python: b [G, N, K], or reduction-major
// [G, K, N]; result row r at out[rows[r]] when there is a map.
void m_grouped_by_block(const Tensor& a, const Tensor& a_s, const Tensor& b, const Tensor& b_s, bool reduction_major, const Tensor& out, const Tensor& offs,
                        const Maybe& rows, int64_t stream) {
  const int64_t M = a.size(0), K = a.size(1), N = b.size(reduction_major ? 2 : 1), G = b.size(0);
  const char* what = reduction_major ? rows ? "pt_gemm_m_grouped_nn_scatter" : "pt_gemm_m_grouped_nn"
                                     : rows ? "pt_gemm_m_grouped_nt_scatter" : "pt_gemm_m_grouped_nt";
  lib.pt_observe(what, 1, M, N, K);
  check(lib.pt_gemm_m_grouped_by_block(ptr(a), (const float*)ptr(a_s), ptr(b), (const float*)ptr(b_s), reduction_major, ptr(out),
                                       dtype_code(out.scalar_type()), (const int32_t*)ptr(offs), (int32_t)G, M, N, K, (const int32_t*)ptr(rows),
                                       rows ? out.size(0) : 0, (pt_stream_t)stream), what);
  lib.pt_observe(what, 0, M, N, K);
}

struct GroupedLinearNode : HipNode {
  Tensor weight;  // its gradient is written to; its values are not read
  Saved operand, operand_scale, ends, input_t, input_ts;
  bool forward_layout;
  void drop() override { for (Saved* s : {&operand, &operand_scale, &ends, &input_t, &input_ts}) s->reset(); }
  variable_list run(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor(), Tensor()};
    const Tensor dg = operand.get(), dg_s = operand_scale.get(), offs = ends.get(), x_t = input_t.get(), x_ts = input_ts.get();
    const Tensor go = g[0].contiguous();
    const int64_t M = go.size(0), N = go.size(1), K = x_t.size(0), G = offs.size(0);
    Quantised d(go, stream);
    Tensor gx = empty({M, K}, go.scalar_type(), go.device());
    const auto o = (const int32_t*)ptr(offs);
    m_grouped_by_block(d.q, d.s, dg, dg_s, forward_layout, gx, offs, std::nullopt, (int64_t)stream);
    {
      py::gil_scoped_acquire gil;
      if (deferred_gradients()) {
        const py::handle schedule(g_schedule);
        schedule(weight, py::make_tuple(d.q_t, d.s_t), py::make_tuple(x_t, x_ts), offs);
        return {gx, Tensor()};
      }
    }
    Target t;
    t.aim(weight);
    lib.pt_observe("pt_gemm_k_grouped_wgrad", 1, M, N, K);
    check(lib.pt_gemm_k_grouped_wgrad(ptr(d.q_t), (const float*)ptr(d.s_t), ptr(x_t), (const float*)ptr(x_ts), t.at(), PT_BF16, t.add, o, (int32_t)G, M, N,
                                      K, stream), "pt_gemm_k_grouped_wgrad");
    lib.pt_observe("pt_gemm_k_grouped_wgrad", 0, M, N, K);
    t.finish();
    return {gx, Tensor()};  // the weight's gradient went to .grad
  }
};

Tensor grouped_linear(const Tensor& x, const Tensor& weight, const Tensor& offs, const Tensor& w, const Tensor& w_s, const Tensor& dg, const Tensor& dg_s,
                      bool forward_layout, int64_t stream) {
  require_same_device(x, {&weight, &offs, &w, &w_s, &dg, &dg_s});
  Quantised q;
  return with_node<GroupedLinearNode>(
      stream,
      [&] {
        const int64_t M = x.size(0), K = x.size(1), N = w.size(1), G = w.size(0);
        if (weight.sizes() != w.sizes()) throw HipError("grouped linear: the quantised weight has another size than the weight");
        require_operand(w, w_s, G, N, K, "grouped weight");
        require_operand(dg, dg_s, G, forward_layout ? N : K, forward_layout ? K : N, "grouped weight of the input gradient");
        require_shape(offs, {G}, at::kInt, "group ends");
        q = Quantised(x, (pt_stream_t)stream);
        Tensor y = empty({M, N}, x.scalar_type(), x.device());
        lib.pt_observe("pt_gemm_m_grouped_nt", 1, M, N, K);
        check(lib.pt_gemm_m_grouped_by_block(ptr(q.q), (const float*)ptr(q.s), ptr(w), (const float*)ptr(w_s), 0, ptr(y), dtype_code(y.scalar_type()),
                                             (const int32_t*)ptr(offs), (int32_t)G, M, N, K, nullptr, 0, (pt_stream_t)stream), "pt_gemm_m_grouped_nt");
        lib.pt_observe("pt_gemm_m_grouped_nt", 0, M, N, K);
        return y;
      },
      [&](GroupedLinearNode& node) {
        node.weight = weight; node.operand = Saved(dg); node.operand_scale = Saved(dg_s); node.ends = Saved(offs);
        node.input_t = Saved(q.q_t); node.input_ts = Saved(q.s_t); node.forward_layout = forward_layout;
      },
      x, weight);
}

// Input gradient of an expert block whose routed rows expand `src_rows` rows: what the scattering GEMM and the backward of
// the expanding gather after it give, but a row with one routed row goes to its place from the GEMM's store and is not
// read, added to nothing and written again (262 144 rows of 2048, a quarter of them repeats: sum 299 -> 132 us, and 6 for the destinations;
// 32 768 rows that five of eight ranks' tokens share: 39 -> 28 and 5).
Tensor expanded_input_gradient(const Tensor& dgu, const Tensor& dgu_s, const Tensor& w, const Tensor& w_s, bool forward_layout, const Tensor& offs,
                               const Tensor& row_map, const Tensor& expand_idx, int64_t src_rows, int64_t K, int64_t stream) {
  const auto st = (pt_stream_t)stream;
  const auto dev = dgu.device();
  const int64_t n = expand_idx.size(0), M = row_map.size(0), N = dgu.size(1), G = offs.size(0);
  Tensor out = empty({cdiv(src_rows, kRowAlignment) * kRowAlignment, K}, at::kBFloat16, dev), shared = empty({n, K}, at::kBFloat16, dev);
  const int64_t bytes = up256(lib.pt_gather_rows_backward_workspace_bytes(n, src_rows));
  Tensor ws = empty({bytes + 4 * M}, at::kByte, dev);
  int32_t* const dest = (int32_t*)((char*)ptr(ws) + bytes);
  check(lib.pt_gather_rows_backward_begin((const int64_t*)ptr(expand_idx), n, src_rows, ptr(ws), bytes, (const int32_t*)ptr(row_map), dest, M, st),
        "pt_gather_rows_backward_begin");
  const char* what = forward_layout ? "pt_gemm_m_grouped_nn_scatter" : "pt_gemm_m_grouped_nt_scatter";
  lib.pt_observe(what, 1, M, K, N);
  check(lib.pt_gemm_m_grouped_by_block_two(ptr(dgu), (const float*)ptr(dgu_s), ptr(w), (const float*)ptr(w_s), forward_layout, ptr(out), ptr(shared), PT_BF16,
                                           (const int32_t*)ptr(offs), (int32_t)G, M, K, N, dest, src_rows, n, st), what);
  lib.pt_observe(what, 0, M, K, N);
  check(lib.pt_gather_rows_backward_shared(ptr(shared), K, ptr(out), K, n, src_rows, K, PT_BF16, ptr(ws), bytes, st), "pt_gather_rows_backward_shared");
  return out.narrow(0, 0, src_rows);
}

// ---- expert block -----------------------------------------------------------------------------------------
struct ExpertsNode : HipNode {
  Dims d;
  Tensor w_gate, w_up, w_down;  // w_gate: the fused gate_up weight when w_up is not there
  enum { GU_DG, GU_DG_S, DN_DG, DN_DG_S, OFFS, GATE_UP, ROW_MAP, EXPAND_IDX, COUNT };
  Saved saved[COUNT];
  std::vector<Saved> activations;  // x^T, h^T with scales
  Maybe gu_bias, dn_bias;
  bool has_map, has_expand, gu_forward, dn_forward, scatter, without_padding, clamped;
  double alpha, limit;
  int64_t src_rows, routed, repeat;
  void drop() override {
    for (Saved& s : saved) s.reset();
    activations.clear();
  }
  variable_list run(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    const Tensor offs = saved[OFFS].get(), gu_dg = saved[GU_DG].get(), gu_dg_s = saved[GU_DG_S].get();
    Maybe row_map, expand_idx;
    if (has_map) row_map = saved[ROW_MAP].get();
    if (without_padding && !in_whole_chunks(*row_map)) row_map = row_map->clone();  // a saved-tensor hook's
    if (has_expand) expand_idx = saved[EXPAND_IDX].get();
    std::vector<Tensor> kept;
    for (const Saved& s : activations) kept.push_back(s.get());
    bool deferred;
    {
      py::gil_scoped_acquire gil;
      deferred = deferred_gradients();
    }
    std::vector<Tensor> weights;
    if (!deferred) {
      weights = {w_down, w_gate};
      if (w_up.defined()) weights.push_back(w_up);
    }
    ExpertsBackward step(g[0], d, offs, row_map, scatter, without_padding, saved[DN_DG].get(), saved[DN_DG_S].get(), dn_forward, saved[GATE_UP].get(), std::move(kept),
                         clamped, alpha, limit, gu_bias, dn_bias, std::move(weights), (int64_t)stream);
    // Rows that expand the same source row are summed (the backward of the expanding gather), right behind the GEMM
    // that wrote them: after the weight gradient they come from HBM.  Only a sum of bf16 rows below 4 GiB takes two outputs.
    const bool two = expand_idx && row_map && g[0].scalar_type() == at::kBFloat16 && d.K % 8 == 0 && src_rows * d.K < (1ll << 31) &&
                     routed * d.K < (1ll << 31);
    Tensor gx;
    if (two) gx = expanded_input_gradient(step.dgu, step.dgu_s, gu_dg, gu_dg_s, gu_forward, offs, *row_map, *expand_idx, src_rows, d.K, (int64_t)stream);
    else gx = empty({row_map ? routed : d.M, d.K}, g[0].scalar_type(), g[0].device());
    if (!two || deferred) {
      py::gil_scoped_acquire gil;
      if (!two) {
        const py::handle dgrad(g_dgrad);
        dgrad(py::make_tuple(step.dgu, step.dgu_s), gu_dg, gu_dg_s, gu_forward, gx, offs, row_map);
      }
      if (deferred) {
        const auto op = step.operands();
        auto pair = [](const std::pair<Tensor, Tensor>& p) { return py::make_tuple(p.first, p.second); };
        py::handle schedule(g_schedule);
        schedule(w_down, pair(op[0]), pair(op[3]), offs);
        if (w_up.defined()) {
          const Tensor &q = op[1].first, &sc = op[1].second;
          schedule(w_gate, py::make_tuple(q.narrow(0, 0, d.half), sc.narrow(1, 0, d.half)), pair(op[2]), offs);
          schedule(w_up, py::make_tuple(q.narrow(0, d.half, d.half), sc.narrow(1, d.half, d.half)), pair(op[2]), offs);
        } else {
          schedule(w_gate, pair(op[1]), pair(op[2]), offs);
        }
      }
    }
    step.dgu.reset();
    step.dgu_s.reset();
    if (expand_idx && !two) gx = scatter_sum(gx, *expand_idx, src_rows, kRowAlignment, (int64_t)stream);
    if (!deferred) step.weight_gradient();
    if (repeat > 1) gx = gx.view({src_rows, repeat, d.K});
    return {gx, Tensor(), Tensor(), Tensor(), step.d_gu_bias.value_or(Tensor()), step.d_dn_bias.value_or(Tensor())};
  }
};

// (fp8, scale) of the forward operand and (fp8, scale, forward_layout) of the input gradient's
typedef std::tuple<Tensor, Tensor> Operand;
typedef std::tuple<Tensor, Tensor, bool> DgradOperand;

Tensor experts(const Tensor& input, const Tensor& w_gate, const Maybe& w_up, const Tensor& w_down, const Maybe& gu_bias, const Maybe& dn_bias,
               const Tensor& offs, const Operand& gu, const Operand& dn, const DgradOperand& gu_dg, const DgradOperand& dn_dg, const Maybe& row_map,
               const Maybe& expand_idx, bool scatter, std::optional<std::pair<double, double>> clamp, int64_t stream) {
  const Tensor up = w_up.value_or(Tensor()), b0 = gu_bias.value_or(Tensor()), b1 = dn_bias.value_or(Tensor());
  require_same_device(input, {&w_gate, &up, &w_down, &std::get<0>(gu_dg), &std::get<1>(gu_dg), &std::get<0>(dn_dg), &std::get<1>(dn_dg)});
  std::tuple<Tensor, Tensor, std::vector<Tensor>, bool> done;
  Tensor x;
  int64_t repeat = 1;
  const auto [alpha, limit] = clamp.value_or(std::pair<double, double>{0.0, 0.0});
  return with_node<ExpertsNode>(
      stream,
      [&] {
        x = input;
        if (x.dim() == 3) {
          repeat = x.size(1);
          x = x.select(1, 0);
        }
        x = row_major(x);
        Maybe c0, c1;
        if (gu_bias) c0 = gu_bias->contiguous();
        if (dn_bias) c1 = dn_bias->contiguous();
        const int64_t G = w_down.size(0), H = w_down.size(1), half = w_down.size(2), K = x.size(1), N = 2 * half;
        const auto dgrad = [&](const DgradOperand& q, int64_t rows, int64_t cols, const char* what) {  // W as it is, or its transposed twin
          if (!std::get<2>(q)) std::swap(rows, cols);
          require_operand(std::get<0>(q), std::get<1>(q), G, rows, cols, what);
        };
        // the weight gradients are written to tensors of the parameters' sizes
        const bool split = up.defined();
        if (w_gate.sizes() != at::IntArrayRef({G, split ? half : N, K}) || (split && up.sizes() != w_gate.sizes()))
          throw HipError("expert block: gate and up weights of other sizes than the down weight and the rows");
        dgrad(gu_dg, N, K, "gate_up weight of the input gradient");
        dgrad(dn_dg, H, half, "down weight of the input gradient");
        done = experts_forward(x, repeat, row_map, expand_idx, offs, std::get<0>(gu), std::get<1>(gu), std::get<0>(dn), std::get<1>(dn), w_down.size(2), c0,
                               c1, scatter, (bool)clamp, alpha, limit, true, false, stream);
        return std::get<0>(done);
      },
      [&](ExpertsNode& n) {
        n.src_rows = x.size(0);
        n.repeat = repeat;
        n.routed = expand_idx ? expand_idx->size(0) : n.src_rows * repeat;
        n.d = Dims{row_map ? row_map->size(0) : n.src_rows, x.size(1), w_down.size(2), w_down.size(1), w_down.size(0)};
        n.w_gate = w_gate; n.w_up = up; n.w_down = w_down;
        n.gu_forward = std::get<2>(gu_dg);
        n.dn_forward = std::get<2>(dn_dg);
        n.has_map = (bool)row_map;
        n.has_expand = (bool)expand_idx;
        const Tensor keep[] = {std::get<0>(gu_dg), std::get<1>(gu_dg), std::get<0>(dn_dg), std::get<1>(dn_dg), offs, std::get<1>(done),
                               row_map.value_or(Tensor()), expand_idx.value_or(Tensor())};
        for (int i = 0; i < ExpertsNode::COUNT; ++i)
          if (keep[i].defined()) n.saved[i] = Saved(keep[i]);
        for (const Tensor& t : std::get<2>(done)) n.activations.emplace_back(t);
        n.gu_bias = gu_bias; n.dn_bias = dn_bias;
        n.scatter = scatter; n.without_padding = std::get<3>(done); n.clamped = (bool)clamp; n.alpha = alpha; n.limit = limit;
      },
      input, w_gate, up, w_down, b0, b1);
}

// ---- combine ----------------------------------------------------------------------------------------------
struct CombineNode : HipNode {
  Saved outs, weight;
  bool residual;
  void drop() override { outs.reset(); weight.reset(); }
  variable_list run(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor(), Tensor(), Tensor()};
    const Tensor moe = outs.get(), w = weight.get();
    const int64_t T = w.size(0), k = w.size(1), H = moe.size(1);
    const Tensor go = g[0].reshape({T, H}).contiguous();
    Tensor dm = empty(moe.sizes(), moe.scalar_type(), moe.device()), dw = empty({T, k}, at::kFloat, moe.device());
    check(lib.pt_moe_combine_bwd(ptr(go), H, ptr(moe), H, (const float*)ptr(w), ptr(dm), H, (float*)ptr(dw), T, (int32_t)k, H,
                                 dtype_code(moe.scalar_type()), stream), "pt_moe_combine_bwd");
    return {dm, dw, residual ? g[0] : Tensor()};
  }
};

Tensor combine(const Tensor& outs, const Tensor& weight, const Maybe& residual, int64_t stream) {
  const Tensor res = residual.value_or(Tensor());
  require_same_device(outs, {&weight, &res});
  const int64_t T = weight.size(0), k = weight.size(1), H = outs.size(1);
  Tensor moe, w;
  return with_node<CombineNode>(
      stream,
      [&] {
        moe = outs.contiguous();
        w = weight.contiguous();
        Tensor r;
        if (residual) r = res.reshape({T, H}).contiguous();
        Tensor out = empty({T, H}, moe.scalar_type(), moe.device());
        check(lib.pt_moe_combine_fwd(ptr(moe), H, (const float*)ptr(w), residual ? ptr(r) : nullptr, H, ptr(out), H, T, (int32_t)k, H,
                                     dtype_code(moe.scalar_type()), (pt_stream_t)stream), "pt_moe_combine_fwd");
        return residual ? out.view(res.sizes()) : out;
      },
      [&](CombineNode& n) { n.outs = Saved(moe); n.weight = Saved(w); n.residual = (bool)residual; }, outs, weight, res);
}

struct CombineEpNode : HipNode {
  Saved outs, weight, slot_row;
  void drop() override { outs.reset(); weight.reset(); slot_row.reset(); }
  variable_list run(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor(), Tensor(), Tensor()};
    const Tensor moe = outs.get(), w = weight.get(), slots = slot_row.get();
    const int64_t T = w.size(0), k = w.size(1), R = moe.size(0), H = moe.size(1);
    const Tensor go = g[0].reshape({T, H}).contiguous();
    // rows no slot points to (none when the indices are a permutation) get a zero gradient
    Tensor dm = R == T * k ? empty(moe.sizes(), moe.scalar_type(), moe.device()) : at::zeros_like(moe);
    Tensor dw = empty({T, k}, at::kFloat, moe.device());
    check(lib.pt_moe_combine_ep_bwd(ptr(go), H, ptr(moe), H, R, (const int32_t*)ptr(slots), (const float*)ptr(w), ptr(dm), H, (float*)ptr(dw), T,
                                    (int32_t)k, H, dtype_code(moe.scalar_type()), stream), "pt_moe_combine_ep_bwd");
    return {dm, dw, g[0]};
  }
};

Tensor combine_ep(const Tensor& outs, const Tensor& local_idxs, const Tensor& weight, const Tensor& residual, int64_t stream) {
  require_same_device(outs, {&local_idxs, &weight, &residual});
  const int64_t T = weight.size(0), k = weight.size(1), R = outs.size(0), H = outs.size(1);
  const auto st = (pt_stream_t)stream;
  Tensor moe, w, slots;
  return with_node<CombineEpNode>(
      stream,
      [&] {
        moe = outs.contiguous();
        w = weight.contiguous();
        const Tensor r = residual.reshape({T, H}).contiguous(), idx = local_idxs.contiguous();
        slots = empty({T * k}, at::kInt, moe.device());
        check(lib.pt_moe_combine_ep_index((const int64_t*)ptr(idx), R, T * k, (int32_t*)ptr(slots), st), "pt_moe_combine_ep_index");
        Tensor out = empty({T, H}, moe.scalar_type(), moe.device());
        check(lib.pt_moe_combine_ep_fwd(ptr(moe), H, R, (const int32_t*)ptr(slots), (const float*)ptr(w), ptr(r), H, ptr(out), H, T, (int32_t)k, H,
                                        dtype_code(moe.scalar_type()), st), "pt_moe_combine_ep_fwd");
        return out.view(residual.sizes());
      },
      [&](CombineEpNode& n) { n.outs = Saved(moe); n.weight = Saved(w); n.slot_row = Saved(slots); }, outs, weight, residual);
}

// ---- a MoE block's branches (see moe_combine.token_branches) ------------------------------------------------
// The branches are views of x in autograd's eyes as well: they share its version counter, so a branch that
// something saved for its backward is found out when x is written afterwards (hidden += block(hidden)), and
// writing to a branch is refused.  That is what torch's own function template does with views that a
// forward returns; a node of this file would leave it out.
struct BranchesFunction : torch::autograd::Function<BranchesFunction> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, int64_t k, int64_t n, int64_t stream) {
    ctx->set_materialize_grads(false);
    ctx->saved_data["stream"] = stream;
    variable_list out;
    out.push_back(x.unsqueeze(1).expand({-1, k, -1}));
    for (int64_t i = 0; i < n; ++i) out.push_back(x.view_as(x));
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list g) {
    return as_python_errors([&] { return sum(ctx, g); });
  }

  static variable_list sum(AutogradContext* ctx, const variable_list& g) {
    std::vector<Tensor> given;
    bool same = g.size() <= 4;
    for (const Tensor& t : g)
      if (t.defined()) {
        given.push_back(t);
        const auto type = t.scalar_type();
        same = same && t.is_cuda() && t.size(-1) % 8 == 0 && type == given[0].scalar_type() && (type == at::kBFloat16 || type == at::kFloat || type == at::kHalf);
      }
    if (given.empty()) return variable_list(4);
    const bool rows = g[0].defined();
    if (!same || at::GradMode::is_enabled()) {  // a backward that is itself differentiated adds with torch's operators
      Tensor total = rows ? g[0].sum(1) : Tensor();
      for (size_t i = 1; i < g.size(); ++i)
        if (g[i].defined()) total = total.defined() ? total + g[i] : g[i];
      return {total, Tensor(), Tensor(), Tensor()};
    }
    for (Tensor& t : given) t = packed(t);
    const void* at[3] = {};
    for (size_t i = rows, n = 0; i < given.size(); ++i) at[n++] = ptr(given[i]);
    const int64_t T = given[0].size(0), H = given[0].size(-1);
    Tensor out = empty({T, H}, given[0].scalar_type(), given[0].device());
    check(lib.pt_sum_branches(rows ? ptr(given[0]) : nullptr, rows ? (int32_t)given[0].size(1) : 0, at[0], at[1], at[2], ptr(out), T, H,
                              dtype_code(out.scalar_type()), (pt_stream_t)ctx->saved_data["stream"].toInt()), "pt_sum_branches");
    return {out, Tensor(), Tensor(), Tensor()};
  }
};

variable_list branches(const Tensor& x, int64_t k, int64_t n, int64_t stream) { return BranchesFunction::apply(x, k, n, stream); }

// ---- router gate ------------------------------------------------------------------------------------------
struct RouterNode : HipNode {
  Saved input, choice;
  int64_t mode, k, norm, num_group, topk_group;
  double scale;
  void drop() override { input.reset(); choice.reset(); }
  variable_list run(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor()};
    const Tensor logits = input.get(), idx = choice.get();
    const int64_t T = logits.size(0), E = logits.size(1);
    const Tensor dw = g[0].to(at::kFloat).contiguous();
    Tensor d = empty({T, E}, logits.scalar_type(), logits.device());
    check(lib.pt_router_topk_bwd(ptr(logits), logits.stride(0), dtype_code(logits.scalar_type()), T, (int32_t)E, (int32_t)k, (int)mode, (int)norm,
                                 (float)scale, (int32_t)num_group, (int32_t)topk_group, (const int64_t*)ptr(idx), (const float*)ptr(dw), nullptr, ptr(d), E,
                                 stream), "pt_router_topk_bwd");
    return {d};
  }
};

// (topk_idx, topk_weight), without forced choices and without the scores
std::pair<Tensor, Tensor> router_topk(const Tensor& input, int64_t mode, int64_t k, bool norm, double scale, int64_t num_group, int64_t topk_group,
                                      int64_t stream) {
  require_cuda(input);
  Tensor logits, idx;
  Tensor weight = with_node<RouterNode>(
      stream,
      [&] {
        logits = row_major(input);
        const int64_t T = logits.size(0), E = logits.size(1);
        idx = empty({T, k}, at::kLong, logits.device());
        Tensor w = empty({T, k}, at::kFloat, logits.device());
        check(lib.pt_router_topk_fwd(ptr(logits), logits.stride(0), dtype_code(logits.scalar_type()), T, (int32_t)E, (int32_t)k, (int)mode, (int)norm,
                                     (float)scale, (int32_t)num_group, (int32_t)topk_group, nullptr, (int64_t*)ptr(idx), (float*)ptr(w), nullptr,
                                     (pt_stream_t)stream), "pt_router_topk_fwd");
        return w;
      },
      [&](RouterNode& n) {
        n.input = Saved(logits); n.choice = Saved(idx);
        n.mode = mode; n.k = k; n.norm = norm; n.scale = scale; n.num_group = num_group; n.topk_group = topk_group;
      },
      input);
  return {idx, weight};
}

// logits of a gate on bf16 inputs, bf16 or as the product of fp32 copies; the backward is one pass over them (csrc/gate.hip)
struct GateLinearNode : HipNode {
  Saved input, weight;
  void drop() override { input.reset(); weight.reset(); }
  std::optional<variable_list> differentiable(const variable_list& g) override {
    if (!g[0].defined()) return variable_list(2);
    const Tensor x = input.get(), w = weight.get();
    const Tensor dl = g[0].scalar_type() == at::kBFloat16 ? g[0] : g[0].to(at::kFloat);
    const auto type = dl.scalar_type();
    return variable_list{at::matmul(dl, w.to(type)).to(at::kBFloat16), at::matmul(dl.t(), x.to(type)).to(at::kBFloat16)};
  }
  variable_list run(variable_list&& g) override {
    if (!g[0].defined()) return {Tensor(), Tensor()};
    const Tensor x = input.get(), w = weight.get();
    const int64_t T = x.size(0), H = x.size(1), E = w.size(0);
    const Tensor dl = packed(g[0].scalar_type() == at::kBFloat16 ? g[0] : g[0].to(at::kFloat));
    Tensor dx = empty({T, H}, at::kBFloat16, x.device()), dw = empty({E, H}, at::kBFloat16, x.device());
    Tensor ws = empty({lib.pt_gate_linear_bwd_workspace_bytes(T, (int32_t)E, H)}, at::kByte, x.device());
    check(lib.pt_gate_linear_bwd(ptr(dl), dtype_code(dl.scalar_type()), ptr(x), ptr(w), ptr(dx), ptr(dw), T, (int32_t)E, H, ptr(ws), stream), "pt_gate_linear_bwd");
    return {dx, dw};
  }
};

// None where the backward kernel does not take the shapes and types.
Maybe gate_linear(const Tensor& input, const Tensor& weight, bool fp32, int64_t stream) {
  if (!input.is_cuda() || input.device() != weight.device() || input.dim() != 2 || weight.dim() != 2 || input.scalar_type() != at::kBFloat16 || weight.scalar_type() != at::kBFloat16)
    return std::nullopt;
  const int64_t E = weight.size(0);
  const auto plain = [](const Tensor& t) { return t.is_contiguous() && (uintptr_t)ptr(t) % 16 == 0; };
  if (input.numel() == 0 || E % 8 || E > 256 || E == 0 || input.size(1) % 8 || input.size(1) != weight.size(1) || !plain(input) || !plain(weight))
    return std::nullopt;
  if (has_tangent(input) || has_tangent(weight)) return std::nullopt;
  return with_node<GateLinearNode>(
      stream, [&] { return fp32 ? at::linear(input.to(at::kFloat), weight.to(at::kFloat)) : at::linear(input, weight); },
      [&](GateLinearNode& n) {
        n.input = Saved(input);
        n.weight = Saved(weight);
      },
      input, weight);
}

// ---- dispatch of an expert-parallel rank --------------------------------------------------------------------
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor> dedup_prepare_dispatch(const Tensor& ids, int64_t E, int64_t ep, int64_t epr, int64_t stream) {
  const int64_t m = ids.size(0), k = ids.size(1);
  const auto dev = ids.device();
  auto i64 = [&](int64_t n) { return empty({n}, at::kLong, dev); };
  Tensor per_rank = i64(ep), unique = i64(ep), dispatch = i64(m * ep), idxs = i64(m * k), expand = i64(m * k), meta = i64(ep * (epr + 1));
  Tensor ws = empty({std::max<int64_t>(lib.pt_dedup_workspace_bytes(m, (int32_t)k, (int32_t)E, (int32_t)ep), 256)}, at::kByte, dev);
  auto p = [](const Tensor& t) { return (int64_t*)ptr(t); };
  check(lib.pt_dedup_prepare_dispatch(p(ids), ids.stride(0), m, (int32_t)k, (int32_t)E, (int32_t)ep, (int32_t)epr, p(per_rank), p(unique), p(dispatch),
                                      p(idxs), p(expand), p(meta), ptr(ws), ws.numel(), (pt_stream_t)stream), "pt_dedup_prepare_dispatch");
  return {per_rank, unique, dispatch, idxs, expand, meta};
}

std::pair<Tensor, Tensor> build_expert_idxs(const Tensor& counts, int64_t ep, int64_t epr, int64_t max_total, int64_t stream) {
  const Tensor c = counts.to(at::kLong).contiguous();
  Tensor idxs = empty({max_total}, at::kLong, c.device()), splits = empty({ep}, at::kLong, c.device());
  check(lib.pt_build_expert_idxs((const int64_t*)ptr(c), (int32_t)c.size(0), (int32_t)ep, (int32_t)epr, max_total, max_total ? (int64_t*)ptr(idxs) : nullptr,
                                 (int64_t*)ptr(splits), (pt_stream_t)stream), "pt_build_expert_idxs");
  return {idxs, splits};
}

Tensor adjust_expand_idx(const Tensor& received, const Tensor& dedup, const Tensor& splits, int64_t stream) {
  require_same_device(received, {&dedup, &splits});
  require_index(received, "adjust_expand_idx");
  require_index(dedup, "adjust_expand_idx: rows from each rank");
  require_index(splits, "adjust_expand_idx: splits");
  if (splits.size(0) < dedup.size(0)) throw HipError("adjust_expand_idx: fewer splits than ranks");
  const Tensor r = received.contiguous(), sp = splits.contiguous();
  Tensor out = empty(r.sizes(), at::kLong, r.device());
  if (r.size(0))
    check(lib.pt_adjust_expand_idx((const int64_t*)ptr(r), (int64_t*)ptr(out), (const int64_t*)ptr(dedup), dedup.stride(0), (const int64_t*)ptr(sp),
                                   (int32_t)dedup.size(0), r.size(0), (pt_stream_t)stream), "pt_adjust_expand_idx");
  return out;
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const HipError& e) {
      PyErr_SetString(g_error ? g_error : PyExc_RuntimeError, e.what());
    } catch (python_error& e) {  // a saved-tensor hook's
      e.restore();
    } catch (const c10::Error&) {  // by its kind: NotImplementedError, IndexError, ...
      torch::translate_exception_to_python(p);
    }
  });
  m.def("init", [](const std::string& path, py::object error) {
    g_error = error.release().ptr();
    init(path);
  });
  m.def("set_callbacks", [](py::object store, py::object schedule, py::object dgrad) {
    g_store = store.release().ptr();
    g_schedule = schedule.release().ptr();
    g_dgrad = dgrad.release().ptr();
  });
  // without the GIL, as ctypes calls the library: other threads run while a step's launches are queued
  const auto launch = [&m](const char* name, auto* f) { m.def(name, f, py::call_guard<py::gil_scoped_release>()); };
  launch("index_gather", &index_gather);
  launch("scatter_sum", &scatter_sum);
  launch("permute_into_buffer", &permute_into_buffer);
  launch("permute_rows", &permute_rows);
  launch("silu_mul", &silu_mul);
  launch("m_grouped_by_block", &m_grouped_by_block);
  launch("grouped_linear", &grouped_linear);
  launch("experts", &experts);
  launch("combine", &combine);
  launch("combine_ep", &combine_ep);
  launch("branches", &branches);
  launch("router_topk", &router_topk);
  launch("dedup_prepare_dispatch", &dedup_prepare_dispatch);
  launch("build_expert_idxs", &build_expert_idxs);
  launch("adjust_expand_idx", &adjust_expand_idx);
  m.def("split_k", &split_k);
  launch("quant_weight", &quant_weight);
  launch("quant_grouped_weights", &quant_grouped_weights);
  launch("gate_linear", &gate_linear);
  launch("mlp", &mlp);
  launch("linear", &linear);
  launch("linear_fresh", &linear_fresh);
  launch("linear_heads_forward", &linear_heads_forward);
  launch("linear_heads_backward", &linear_heads_backward);
  launch("group_rows", &group_rows);
  launch("experts_forward", &experts_forward);
}

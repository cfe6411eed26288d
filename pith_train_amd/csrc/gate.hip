// Backward of a router gate: d_x = bf16(d_logits w) and d_w = bf16(d_logits^T x) in one pass over x, for bf16
// logits and for fp32 logits of bf16 inputs (logits = float(x) float(w)^T).
//
// The two matrix products that autograd ran for fp32 logits read fp32 copies of x and wrote an fp32 d_x before
// its conversion: 8192 tokens x 2048, 64 experts took 84 us for d_w (64 workgroups over the whole token
// range), 38 us for d_x, 20 us for conversions.  What has to move is x, d_x and the small rest, 70 MB: this
// kernel and the sum of its slabs take 36 + 11 us (block of that size: 3593 -> 3532 us).  With bf16 logits and
// few tokens it was the host that the two library products cost: a block step on 512 tokens x 256 took 300 us
// and takes 260.
//
// Both products run on the bf16 matrix instructions without losing anything: x and w are bf16 already, and an
// fp32 gradient is the exact sum of three bf16 numbers (its 24 significant bits cut in three), so the
// products are exact and are added in fp32 as before.
//
// A workgroup takes 128 columns and a range of tokens, a wave 32 tokens of it at a time:
//   - lane (q, c) = (lane / 16, lane % 16) loads eight 16-byte pieces (columns 8c..8c+7) of eight rows, so a
//     row of the tile is one 256-byte access; byte permutes turn them into the fragments of eight
//     16-column products whose column c stands for 8c + j;
//   - hence a lane ends up with eight neighbouring columns of a result and stores 16 bytes of d_x.
// d_w of the 64 experts of blockIdx.y stays in 128 accumulators over the range; the four waves add theirs through
// LDS in a fixed order, and the ranges are summed by pt_sum_partials.  w is kept in LDS as fragments.
#include "common.h"

namespace pt {

typedef __bf16 gate_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gate_f32x4 __attribute__((ext_vector_type(4)));

static constexpr int kGateCols = 128, kGateExperts = 64, kGateMaxExperts = 256;

struct GateArgs {
  const void* dl;  // [T][E], fp32 or bf16
  const uint16_t *x, *w;
  uint16_t* dx;
  float* partial;  // [ranges][E][H]
  int64_t T, H;
  int32_t E, col_tiles;
  int64_t range;  // tokens per range, a multiple of 128
};

struct GateFrag { uint32_t w[4]; };
__device__ __forceinline__ gate_f32x4 gate_mfma(const GateFrag& a, const GateFrag& b, gate_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gate_bf16x8, a), __builtin_bit_cast(gate_bf16x8, b), c, 0, 0, 0);
}

// Eight rows of eight columns -> the eight rows of column j, as the reduction elements of one lane.
__device__ __forceinline__ GateFrag gate_column(const uint4 (&rows)[8], int j) {
  GateFrag f;
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const uint4 a = rows[2 * m], b = rows[2 * m + 1];
    const int d = j >> 1;
    const uint32_t wa = d == 0 ? a.x : d == 1 ? a.y : d == 2 ? a.z : a.w, wb = d == 0 ? b.x : d == 1 ? b.y : d == 2 ? b.z : b.w;
    f.w[m] = __builtin_amdgcn_perm(wb, wa, (j & 1) ? 0x07060302u : 0x05040100u);
  }
  return f;
}

// The gradients of the logits as operands.  fp32: v = hi + mid + lo exactly, each with at most eight significant
// bits (a NaN stays one in all three, an infinity in the first); bf16: as they are.
template <typename D> struct GateOperand;
template <> struct GateOperand<float> {
  GateFrag hi, mid, lo;
  __device__ __forceinline__ void set(const float (&v)[8]) {
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      uint32_t h[2], d[2], l[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const float f = v[2 * m + u];
        h[u] = __float_as_uint(f);
        const float r = __builtin_isinf(f) ? 0.f : f - __uint_as_float(h[u] & 0xFFFF0000u);  // an infinity is its own first part
        d[u] = __float_as_uint(r);
        l[u] = __float_as_uint(r - __uint_as_float(d[u] & 0xFFFF0000u));
      }
      hi.w[m] = __builtin_amdgcn_perm(h[1], h[0], 0x07060302u);
      mid.w[m] = __builtin_amdgcn_perm(d[1], d[0], 0x07060302u);
      lo.w[m] = __builtin_amdgcn_perm(l[1], l[0], 0x07060302u);
    }
  }
  __device__ __forceinline__ void load_row(const float* p, bool ok) {  // eight neighbours
    float v[8] = {};
    if (ok) {
      const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
      v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    }
    set(v);
  }
  __device__ __forceinline__ void load_column(const float* p, int64_t pitch, int n, const float*) {  // n of eight, one per row
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = k < n ? p[k * pitch] : 0.f;
    set(v);
  }
  __device__ __forceinline__ gate_f32x4 times(const GateFrag& b, gate_f32x4 c) const { return gate_mfma(hi, b, gate_mfma(mid, b, gate_mfma(lo, b, c))); }
};
template <> struct GateOperand<uint16_t> {
  GateFrag v;
  __device__ __forceinline__ void load_row(const uint16_t* p, bool ok) {
    const uint4 u = ok ? *reinterpret_cast<const uint4*>(p) : make_uint4(0, 0, 0, 0);
    v = {{u.x, u.y, u.z, u.w}};
  }
  // From row min(k, n - 1), and `inside` where n is 0, with zeros in place of what is none of the n: behind a condition each 16-bit load
  // waits for the one before it to be merged with zeros (with the sum of the slabs, 8192 tokens x 2048, 128 experts 52.5 -> 46.0 us, 16 384 tokens
  // 85.3 -> 71.6; 32-bit loads are masked without a wait, and selecting their zeros afterwards costs 1 us of 44).
  __device__ __forceinline__ void load_column(const uint16_t* p, int64_t pitch, int n, const uint16_t* inside) {
    uint32_t b[8];
    p = n ? p : inside;
#pragma unroll
    for (int k = 0; k < 8; ++k) b[k] = p[(k < n ? k : n ? n - 1 : 0) * pitch];
#pragma unroll
    for (int k = 0; k < 8; ++k) b[k] = k < n ? b[k] : 0u;
#pragma unroll
    for (int m = 0; m < 4; ++m) v.w[m] = b[2 * m] | (b[2 * m + 1] << 16);
  }
  __device__ __forceinline__ gate_f32x4 times(const GateFrag& b, gate_f32x4 c) const { return gate_mfma(v, b, c); }
};

__device__ __forceinline__ void gate_rows(uint4 (&rows)[8], const uint16_t* base, int64_t row0, int64_t n_rows, int64_t H, bool col_ok) {
#pragma unroll
  for (int k = 0; k < 8; ++k)
    rows[k] = col_ok && row0 + k < n_rows ? *reinterpret_cast<const uint4*>(base + (row0 + k) * H) : make_uint4(0, 0, 0, 0);
}

template <typename D>
__global__ __launch_bounds__(256, 2) void gate_linear_bwd_kernel(GateArgs p) {
  const D* dl = reinterpret_cast<const D*>(p.dl);
  extern __shared__ __attribute__((aligned(16))) uint8_t s_mem[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  const int col_tile = blockIdx.x % p.col_tiles;
  const int64_t range = blockIdx.x / p.col_tiles;
  const int64_t col = (int64_t)col_tile * kGateCols + 8 * c;
  const bool col_ok = col < p.H;  // H % 8 == 0
  const int e0 = blockIdx.y * kGateExperts;
  const bool input_gradient = blockIdx.y == 0;
  const int steps = (p.E + 31) >> 5;

  uint4* s_w = reinterpret_cast<uint4*>(s_mem);  // [steps][8][64]
  if (input_gradient) {
    for (int s = wave; s < steps; s += 4) {
      uint4 rows[8];
      gate_rows(rows, p.w + col, 32 * s + 8 * q, p.E, p.H, col_ok);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const GateFrag f = gate_column(rows, j);
        s_w[(s * 8 + j) * 64 + lane] = make_uint4(f.w[0], f.w[1], f.w[2], f.w[3]);
      }
    }
  }
  __syncthreads();

  gate_f32x4 dw[4][8];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) dw[i][j] = gate_f32x4{0.f, 0.f, 0.f, 0.f};

  const int64_t begin = range * p.range, end = begin + p.range < p.T ? begin + p.range : p.T;
  for (int64_t t0 = begin + 32 * wave; t0 < end; t0 += 128) {
    uint4 rows[8];
    gate_rows(rows, p.x + col, t0 + 8 * q, end, p.H, col_ok);
    if (input_gradient) {
#pragma unroll 1
      for (int half = 0; half < 2; ++half) {
        const int64_t token = t0 + 16 * half + c;
        gate_f32x4 acc[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = gate_f32x4{0.f, 0.f, 0.f, 0.f};
        for (int s = 0; s < steps; ++s) {
          const int e = 32 * s + 8 * q;
          GateOperand<D> g;
          g.load_row(dl + token * p.E + e, token < end && e < p.E);  // E % 8 == 0
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const uint4 u = s_w[(s * 8 + j) * 64 + lane];
            const GateFrag f = {{u.x, u.y, u.z, u.w}};
            acc[j] = g.times(f, acc[j]);
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int64_t row = t0 + 16 * half + 4 * q + i;
          if (row < end && col_ok)
            *reinterpret_cast<uint4*>(p.dx + row * p.H + col) = make_uint4(pack_bf16x2(acc[0][i], acc[1][i]), pack_bf16x2(acc[2][i], acc[3][i]),
                                                                           pack_bf16x2(acc[4][i], acc[5][i]), pack_bf16x2(acc[6][i], acc[7][i]));
        }
      }
    }
    GateFrag fx[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) fx[j] = gate_column(rows, j);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = e0 + 16 * i + c;
      const int64_t row = t0 + 8 * q;
      const int n = e >= p.E || row >= end ? 0 : end - row < 8 ? (int)(end - row) : 8;
      GateOperand<D> g;
      g.load_column(dl + row * p.E + e, p.E, n, dl);
#pragma unroll
      for (int j = 0; j < 8; ++j) dw[i][j] = g.times(fx[j], dw[i][j]);
    }
  }

  float* s_acc = reinterpret_cast<float*>(s_mem);  // [64][128]
  for (int turn = 0; turn < 4; ++turn) {
    __syncthreads();  // the fragments of w, or the wave before, are done
    if (wave != turn) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          float4* at = reinterpret_cast<float4*>(s_acc + (16 * i + 4 * q + r) * kGateCols + 8 * c + 4 * h);
          float4 v = make_float4(dw[i][4 * h][r], dw[i][4 * h + 1][r], dw[i][4 * h + 2][r], dw[i][4 * h + 3][r]);
          if (turn) {
            const float4 o = *at;
            v.x += o.x; v.y += o.y; v.z += o.z; v.w += o.w;
          }
          *at = v;
        }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < kGateExperts * kGateCols / 4; k += 256) {
    const int e = e0 + k / (kGateCols / 4), cc = 4 * (k % (kGateCols / 4));
    const int64_t h = (int64_t)col_tile * kGateCols + cc;
    if (e < p.E && h < p.H) *reinterpret_cast<float4*>(p.partial + (range * p.E + e) * p.H + h) = reinterpret_cast<const float4*>(s_acc)[k];
  }
}

// Ranges of tokens: two workgroups per compute unit, a whole number of 128-token rounds each.
static int64_t gate_range(int64_t T, int64_t E, int64_t H) {
  const int64_t tiles = cdiv(H, kGateCols) * cdiv(E, kGateExperts), want = tiles < 512 ? 512 / tiles : 1;
  return cdiv(cdiv(T, want), 128) * 128;
}

}  // namespace pt

using namespace pt;

extern "C" int64_t pt_gate_linear_bwd_workspace_bytes(int64_t T, int32_t E, int64_t H) {
  if (T <= 0 || E <= 0 || H <= 0) return 0;
  return 4 * cdiv(T, gate_range(T, E, H)) * E * H;
}

extern "C" int pt_gate_linear_bwd(const void* d_logits, int dtype, const void* x, const void* w, void* d_x, void* d_w, int64_t T, int32_t E, int64_t H,
                                  void* workspace, pt_stream_t stream) {
  PT_REQUIRE(T > 0 && E > 0 && H > 0 && E % 8 == 0 && E <= kGateMaxExperts && H % 8 == 0,
             "gate_linear_bwd: %d experts and a width of %lld: both multiples of 8, at most %d experts", E, (long long)H, kGateMaxExperts);
  PT_REQUIRE(d_logits && x && w && d_x && d_w && workspace, "gate_linear_bwd: null pointer");
  PT_REQUIRE((((uintptr_t)d_logits | (uintptr_t)x | (uintptr_t)w | (uintptr_t)d_x | (uintptr_t)d_w | (uintptr_t)workspace) & 15) == 0,
             "gate_linear_bwd: pointers must be 16-byte aligned");
  GateArgs a;
  a.dl = d_logits; a.x = (const uint16_t*)x; a.w = (const uint16_t*)w; a.dx = (uint16_t*)d_x; a.partial = (float*)workspace;
  a.T = T; a.H = H; a.E = E; a.col_tiles = (int32_t)cdiv(H, kGateCols); a.range = gate_range(T, E, H);
  const int64_t ranges = cdiv(T, a.range);
  PT_REQUIRE(ranges * a.col_tiles < (1ll << 31), "gate_linear_bwd: too many tokens");
  const int weights = (int)cdiv(E, 32) * 8 * 64 * 16, sums = kGateExperts * kGateCols * 4;
  const dim3 grid((unsigned)(ranges * a.col_tiles), (unsigned)cdiv(E, kGateExperts)), block(256);
  const int lds = weights > sums ? weights : sums;
  if (dtype == PT_F32) hipLaunchKernelGGL(gate_linear_bwd_kernel<float>, grid, block, lds, (hipStream_t)stream, a);
  else if (dtype == PT_BF16) hipLaunchKernelGGL(gate_linear_bwd_kernel<uint16_t>, grid, block, lds, (hipStream_t)stream, a);
  else PT_REQUIRE(false, "gate_linear_bwd: unsupported dtype %d (fp32 and bf16 only)", dtype);
  if (int rc = check_launch("gate_linear_bwd_kernel")) return rc;
  return pt_sum_partials(a.partial, (int32_t)ranges, (int64_t)E * H, d_w, PT_BF16, stream);
}

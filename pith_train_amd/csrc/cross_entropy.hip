// In-place fused cross-entropy of the loss head: one pass for the row's softmax statistics, one
// that overwrites the logits with the gradient of the mean loss, as the reference's kernel does
// (operators/cross_entropy.py:16-78):
//
//   n    = max(1, #rows with target != ignore_index)
//   m, d = max_i x_i, sum_i exp(x_i - m)                               (fp32)
//   loss_row = -(x_y - m - log d);  ignored rows: loss_row = 0, gradient row = 0
//   x_i <- S((exp(x_i - m) / d) / n);   x_y <- S(float(x_y) - 1/n)      (S = the logits' type)
//   loss = sum(loss_row) / n
//
// One 1024-thread workgroup per row (vocabularies are 32-200 k entries), 16-byte accesses.  Rows of up to 400 KB stay on chip between
// the passes (registers and LDS); the second read of a longer one comes out of the caches, so
// HBM sees one read and one write of the logits.  exp is the hardware's exp2 of x * log2(e): at
// 1.2 G elements per step a library exp would cost as much as the memory traffic.  The row
// statistics combine per-thread (m, d) pairs in a fixed order: the result is the same on every run.
// Backward (CrossEntropy.backward, operators/cross_entropy.py:120-124): the stored gradient times
// the incoming scalar rounded to S, in place.
#include "common.h"
#include <stdlib.h>
#include <string.h>

// Cache policy of the logits' accesses (1 = non-temporal loads, 2 = non-temporal stores; build
// switch, make EXTRA=-DPT_CE_NT=<bits>): a [N, V] logits matrix is larger than every cache and each
// pass touches an element once.  Both on: the in-place backward runs 10 % faster (4096 x 151 936
// bf16: 478 -> 428 us), the forward is level; either one alone changes nothing.
#ifndef PT_CE_NT
#define PT_CE_NT 3
#endif
#if PT_CE_NT & 1
#define PT_CE_LDS_LOAD_NT " nt"
#else
#define PT_CE_LDS_LOAD_NT ""
#endif

namespace pt {

static constexpr int kCeThreads = 1024;
static constexpr float kLog2e = 1.4426950408889634f;

struct CeArgs {
  char* x;
  int64_t ld;  // bytes
  const int64_t* target;
  int64_t N, V, ignore_index;
  float* loss_rows;
  float* loss;
  int64_t* n_non_ignore;
  const float* grad_output;
  int vec;  // rows start at multiples of their element size, as those of any tensor do; a C caller's elsewhere go element by element
};

// A row in 16-byte chunks.  Rows whose length is no multiple of 16 bytes start anywhere in one, so the chunks begin at
// the first boundary; the elements before it and behind the last whole chunk (at most 7 of either, "edges") belong to
// threads 0 .. 7 and 8 .. 15 of the workgroup, one each.
template <typename S>
struct CeRow {
  static constexpr int kPer = 16 / S::kBytes;  // elements of a chunk
  char* x;
  int head, tail;
  uint32_t chunks;
  __device__ __forceinline__ CeRow(char* row, int64_t V) : x(row) {
    const int64_t to_boundary = (int64_t)(-(uintptr_t)row & 15) / S::kBytes;
    head = (int)(to_boundary < V ? to_boundary : V);
    chunks = (uint32_t)((V - head) / kPer);
    tail = (int)((V - head) % kPer);
  }
  __device__ __forceinline__ char* body() const { return x + head * S::kBytes; }
  // whether thread tid has an edge element, and its byte offset in the row
  __device__ __forceinline__ bool edge(int tid) const { return tid < 8 ? tid < head : tid < 8 + tail; }
  __device__ __forceinline__ int64_t edge_at(int tid) const { return (tid < 8 ? tid : head + (int64_t)chunks * kPer + tid - 8) * S::kBytes; }
};

__device__ __forceinline__ float fast_exp(float v) { return __builtin_amdgcn_exp2f(v * kLog2e); }

__global__ __launch_bounds__(1024) void ce_count_kernel(const int64_t* target, int64_t N, int64_t ignore_index,
                                                        int64_t* n_non_ignore) {
  __shared__ int64_t s_part[16];
  int64_t c = 0;
  for (int64_t i = threadIdx.x; i < N; i += 1024) c += target[i] != ignore_index;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) c += __shfl_xor((int)c, d);  // a wave counts at most N / 16 < 2^31 rows
  if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t t = 0;
    for (int w = 0; w < 16; ++w) t += s_part[w];
    *n_non_ignore = t < 1 ? 1 : t;
  }
}

// (m, d) of two disjoint parts of a row -> (m, d) of their union
__device__ __forceinline__ void merge_md(float& m, float& d, float m2, float d2) {
  const float mn = fmaxf(m, m2);
  // a part that saw no more than -inf has m = -inf and d = 0, or the not-a-number that it saw
  const float a = m == -INFINITY ? d : d * fast_exp(m - mn);
  const float b = m2 == -INFINITY ? d2 : d2 * fast_exp(m2 - mn);
  m = mn;
  d = a + b;
}

typedef int ce_v4i __attribute__((ext_vector_type(4)));

template <typename S>
__device__ __forceinline__ void unpack(const ce_v4i& w, float (&v)[CeRow<S>::kPer]) {
  if constexpr (S::kBytes == 2) {
    S::load8(&w, v);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __int_as_float(w[i]);
  }
}
template <typename S>
__device__ __forceinline__ ce_v4i pack(const float (&v)[CeRow<S>::kPer]) {
  ce_v4i w;
  if constexpr (S::kBytes == 2) {
    S::store8(&w, v);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = __float_as_int(v[i]);
  }
  return w;
}
// one chunk (or one edge element) into a thread's running (m, d), rescaled where the maximum grows
template <int N>
__device__ __forceinline__ void absorb(const float (&v)[N], float& m, float& d) {
  float cm = v[0];
#pragma unroll
  for (int i = 1; i < N; ++i) cm = fmaxf(cm, v[i]);
  if (cm > m) {
    d = d * fast_exp(m - cm);  // m = -inf on the first chunk: d is 0 and exp2(-inf) is 0
    m = cm;
  }
  // (a chunk of -inf logits, a masked vocabulary, adds zeros; one of them and a not-a-number, which no maximum shows, adds that)
  const float mb = m == -INFINITY ? 0.f : m * kLog2e;
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) s += __builtin_amdgcn_exp2f(v[i] * kLog2e - mb);
  d += s;
}
// logits into gradients of the mean loss; off: the target's place among them (anything else: not there)
template <typename S, int N, class I>
__device__ __forceinline__ void gradient(float (&v)[N], float mb, float inv_d, float inv_n, I off) {
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = (__builtin_amdgcn_exp2f(v[i] * kLog2e - mb) * inv_d) * inv_n;
  if (off >= 0 && off < N) {
    // the reference stores the softmax term first and corrects the stored value afterwards
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (i == (int)off) v[i] = S::round(v[i]) - inv_n;
  }
}

template <typename S>
__global__ __launch_bounds__(1024) void ce_fwd_kernel(CeArgs p) {
  __shared__ float s_m[16], s_d[16];
  const int64_t row = blockIdx.x;
  char* x = p.x + row * p.ld;
  const int64_t y = p.target[row];
  const int tid = threadIdx.x;
  const CeRow<S> r(x, p.V);
  ce_v4i* body = (ce_v4i*)r.body();
  const bool edge = p.vec && r.edge(tid);
  if (y == p.ignore_index) {
    if (p.vec) {
      const ce_v4i z = {0, 0, 0, 0};
      for (uint32_t c = tid; c < r.chunks; c += kCeThreads) body[c] = z;
      if (edge) S::store1(x + r.edge_at(tid), 0.f);
    } else {
      for (int64_t i = tid; i < p.V; i += kCeThreads) S::store1(x + i * S::kBytes, 0.f);
    }
    if (tid == 0) p.loss_rows[row] = 0.f;
    return;
  }
  // pass 1: per-thread running (m, d), rescaled once per chunk
  float m = -INFINITY, d = 0.f;
  if (p.vec) {
    for (uint32_t c = tid; c < r.chunks; c += kCeThreads) {
      float v[CeRow<S>::kPer];
      unpack<S>(body[c], v);
      absorb(v, m, d);
    }
    if (edge) {
      const float v[1] = {S::load1(x + r.edge_at(tid))};
      absorb(v, m, d);
    }
  } else {
    for (int64_t i = tid; i < p.V; i += kCeThreads) {
      const float v = S::load1(x + i * S::kBytes);
      if (v > m) {
        d = d * fast_exp(m - v);
        m = v;
      }
      d += fast_exp(v - (m == -INFINITY ? 0.f : m));
    }
  }
  // fixed-order combination: xor butterfly inside the wave, then the 16 waves in order
#pragma unroll
  for (int s = 32; s >= 1; s >>= 1) {
    const float m2 = __shfl_xor(m, s), d2 = __shfl_xor(d, s);
    merge_md(m, d, m2, d2);
  }
  if ((tid & 63) == 0) {
    s_m[tid >> 6] = m;
    s_d[tid >> 6] = d;
  }
  __syncthreads();
  m = s_m[0];
  d = s_d[0];
  for (int w = 1; w < 16; ++w) merge_md(m, d, s_m[w], s_d[w]);
  const float n = (float)*p.n_non_ignore;
  const bool y_ok = y >= 0 && y < p.V;
  if (tid == 0) {
    // a target outside the vocabulary (and not the ignore value) has no logit: the loss says so
    const float xy = y_ok ? S::load1(x + y * S::kBytes) : NAN;
    p.loss_rows[row] = -(xy - m - logf(d));
  }
  __syncthreads();  // the target's logit is read before anyone overwrites it
  // pass 2: gradient of the mean loss, in place
  const float mb = m * kLog2e;
  // The two divisions of the reference become multiplications by reciprocals computed once per
  // row: an fp32 division per element costs more issue cycles than everything else in the pass.
  const float inv_d = 1.0f / d, inv_n = 1.0f / n;
  const float neg_inv_n = -1.0f / n;
  if (p.vec) {
    for (uint32_t c = tid; c < r.chunks; c += kCeThreads) {
      float v[CeRow<S>::kPer];
      unpack<S>(body[c], v);
      gradient<S>(v, mb, inv_d, inv_n, y - r.head - (int64_t)c * CeRow<S>::kPer);
      body[c] = pack<S>(v);
    }
    if (edge) {
      char* q = x + r.edge_at(tid);
      float v[1] = {S::load1(q)};
      gradient<S>(v, mb, inv_d, inv_n, y - (q - x) / S::kBytes);
      S::store1(q, v[0]);
    }
  } else {
    for (int64_t i = tid; i < p.V; i += kCeThreads) {
      float g = (fast_exp(S::load1(x + i * S::kBytes) - m) * inv_d) * inv_n;
      if (i == y) g = S::round(g) + neg_inv_n;
      S::store1(x + i * S::kBytes, g);
    }
  }
}

// The same computation with the row held on chip between the passes: up to kCeRegChunks 16-byte
// chunks per thread in registers and the chunks past those in LDS, so the
// logits cross the memory bus once each way (the generic kernel's second read of a 300 KB row
// mostly misses the caches when 256 rows are in flight).
static constexpr int kCeRegChunks = 15;                                  // 15 x 1024 x 16 bytes: 122 880 elements of 16 bits
// Rows of up to 64 KiB leave room for two workgroups a compute unit, one of which reads while the other is between its
// last load and its first store: 4096 x 32 000 bf16 with its copy 380 -> 307 us.  With 8 chunks the kernel spills (358;
// 32 000 float32 593 -> 607).
static constexpr int kCeShortChunks = 4;
static constexpr int kCeLdsChunks = (160 * 1024 - 256) / 16;             // + 81 792 elements in the rest of the 160 KiB of LDS

static constexpr int64_t kCeUnits = 256;  // compute units

// 16 bytes per lane from base + voff (per lane) + soff (uniform) into LDS at lds_off + 16 * lane.
__device__ __forceinline__ void ce_load_to_lds(ce_v4i rsrc, uint32_t voff, uint32_t soff, uint32_t lds_off) {
  soff = (uint32_t)__builtin_amdgcn_readfirstlane((int)soff);
  lds_off = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_off);
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen" PT_CE_LDS_LOAD_NT " lds" ::"v"(voff), "s"(rsrc), "s"(soff),
               "s"(lds_off)
               : "memory");
}

// A workgroup (one per compute unit: the row takes the register file and most of the LDS) walks the rows
// blockIdx, blockIdx + gridDim, ...: as soon as a chunk's gradient is on its way out, the same chunk of
// the next row is requested into its place, so that the memory always has requests; with one workgroup
// per row a compute unit first only read and then only wrote (4096 x 151 936 bf16: 546 us against
// 523 here, where a plain copy of the logits takes 471; what is left is the pause of every row between
// its last load and its first store).
template <typename S, int CHUNKS>
__global__ __launch_bounds__(1024, CHUNKS == kCeRegChunks ? 4 : 8) void ce_fwd_onchip_kernel(CeArgs p) {
  extern __shared__ ce_v4i s_over[];
  __shared__ float s_m[16], s_d[16];
  const int tid = threadIdx.x;
  const uint32_t voff = (uint32_t)tid * 16u;
  ce_v4i cache[CHUNKS];
  // The chunks past the registers go straight from memory into LDS (direct-to-LDS loads: a wave's
  // 64 lanes fill 1 KiB, lane l the 16 bytes of the chunk thread l of that wave owns).
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) ce_v4i*)s_over;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Raw buffer descriptor over a row's chunks: a lane's byte offset is tid * 16 for every chunk, the
  // chunk's i * 16 KiB goes into the uniform offset, and accesses past the last chunk are dropped by
  // the hardware (loads return 0) instead of needing an address and a predicate per chunk.
  auto row_words = [&](const CeRow<S>& r) {
    const uint64_t a = (uint64_t)(uintptr_t)r.body();
    ce_v4i w;
    w[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
    w[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)((a >> 32) & 0xFFFF));
    w[2] = __builtin_amdgcn_readfirstlane((int)(r.chunks * 16));
    w[3] = 0x00020000;
    return w;
  };
  auto edge_logit = [&](const CeRow<S>& r) { return r.edge(tid) ? S::load1(r.x + r.edge_at(tid)) : 0.f; };
  auto target_logit = [&](const char* x, int64_t y) { return y >= 0 && y < p.V ? S::load1(x + y * S::kBytes) : NAN; };

  int64_t row = blockIdx.x;  // the grid has at most as many workgroups as there are rows
  CeRow<S> r(p.x + row * p.ld, p.V);
  int64_t y = p.target[row];
  float xy = target_logit(r.x, y);
  float xe = edge_logit(r);
  {
    const ce_v4i words = row_words(r);
#pragma unroll 1
    for (uint32_t c0 = CHUNKS * kCeThreads + wave * 64; c0 < r.chunks; c0 += kCeThreads)
      ce_load_to_lds(words, (uint32_t)(tid & 63) * 16u, c0 * 16u, lds_base + (c0 - CHUNKS * kCeThreads) * 16u);
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(r.body(), 0, (int)(r.chunks * 16), 0x00020000);
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) cache[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff, i * kCeThreads * 16, (PT_CE_NT & 1) ? 2 : 0);
  }
  const float n = (float)*p.n_non_ignore;
  const float inv_n = 1.0f / n;

#pragma unroll 1
  for (;;) {
    const int64_t next = row + gridDim.x;
    const bool more = next < p.N;
    const bool ignored = y == p.ignore_index;
    float m = -INFINITY, d = 0.f;
    auto absorb_chunk = [&](const ce_v4i& w) {
      float v[CeRow<S>::kPer];
      unpack<S>(w, v);
      absorb(v, m, d);
      __builtin_amdgcn_sched_barrier(0);  // one chunk's temporaries at a time: the cache owns the registers
    };
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i)
      if ((uint32_t)i * kCeThreads + tid < r.chunks) absorb_chunk(cache[i]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the LDS part has landed (each thread reads only its own chunks)
#pragma unroll 1
    for (uint32_t c = CHUNKS * kCeThreads + tid; c < r.chunks; c += kCeThreads) absorb_chunk(s_over[c - CHUNKS * kCeThreads]);
    if (r.edge(tid)) {
      const float v[1] = {xe};
      absorb(v, m, d);
    }
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) {
      const float m2 = __shfl_xor(m, s), d2 = __shfl_xor(d, s);
      merge_md(m, d, m2, d2);
    }
    if ((tid & 63) == 0) {
      s_m[tid >> 6] = m;
      s_d[tid >> 6] = d;
    }
    __syncthreads();
    m = s_m[0];
    d = s_d[0];
    for (int w = 1; w < 16; ++w) merge_md(m, d, s_m[w], s_d[w]);
    __syncthreads();  // (the next row's statistics go to the same place)
    if (tid == 0) p.loss_rows[row] = ignored ? 0.f : -(xy - m - logf(d));
    // the next row's target and logit are requested before its chunks
    const int64_t row2 = more ? next : row;
    const CeRow<S> r2(p.x + row2 * p.ld, p.V);
    const int64_t y2 = p.target[row2];
    const float xy2 = target_logit(r2.x, y2);
    const float xe2 = edge_logit(r2);
    const float mb = m * kLog2e;
    // The two divisions of the reference become multiplications by reciprocals computed once per
    // row: an fp32 division per element costs more issue cycles than everything else in the pass.
    const float inv_d = 1.0f / d;
    // the target's place in the body (before it, where there is none: rows of this kernel are far shorter)
    const int y_body = y >= 0 && y < p.V ? (int)y - r.head : -16;
    // gradient of one chunk, packed for a 16-byte store
    auto grad_of = [&](const ce_v4i& w, uint32_t c) {
      float v[CeRow<S>::kPer];
      unpack<S>(w, v);
      gradient<S>(v, mb, inv_d, inv_n, y_body - (int)c * CeRow<S>::kPer);
      ce_v4i out = pack<S>(v);
      if (ignored) out = ce_v4i{0, 0, 0, 0};
      return out;
    };
    if (r.edge(tid)) {
      float v[1] = {xe};
      gradient<S>(v, mb, inv_d, inv_n, y - r.edge_at(tid) / S::kBytes);
      S::store1(r.x + r.edge_at(tid), ignored ? 0.f : v[0]);
    }
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(r.body(), 0, (int)(r.chunks * 16), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc2 = __builtin_amdgcn_make_buffer_rsrc(r2.body(), 0, more ? (int)(r2.chunks * 16) : 0, 0x00020000);
    // LDS part first: its loads are the slower kind to drain at the end of the next statistics pass
    {
      const ce_v4i words2 = row_words(r2);
      // (the next row may have a chunk more or less than this one)
      const uint32_t most = more && r2.chunks > r.chunks ? r2.chunks : r.chunks;
#pragma unroll 1
      for (uint32_t c0 = CHUNKS * kCeThreads + wave * 64; c0 < most; c0 += kCeThreads) {
        const uint32_t c = c0 + (tid & 63);
        if (c < r.chunks) {
          const ce_v4i g = grad_of(s_over[c - CHUNKS * kCeThreads], c);
          ce_v4i* q = (ce_v4i*)r.body() + c;
          if (PT_CE_NT & 2) __builtin_nontemporal_store(g, q);
          else *q = g;
        }
        // (the wave's reads of these 1 KiB have returned: their values are in the stores above)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (more) ce_load_to_lds(words2, (uint32_t)(tid & 63) * 16u, c0 * 16u, lds_base + (c0 - CHUNKS * kCeThreads) * 16u);
      }
    }
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
      const uint32_t c = (uint32_t)i * kCeThreads + tid;
      asm volatile("" : "+v"(cache[i]));  // unpack again rather than keep 120 values from the statistics pass
      // a chunk past the row's end computes on zeros and its store is dropped by the descriptor
      __builtin_amdgcn_raw_buffer_store_b128(grad_of(cache[i], c), rsrc, voff, i * kCeThreads * 16, (PT_CE_NT & 2) ? 2 : 0);
      cache[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc2, voff, i * kCeThreads * 16, (PT_CE_NT & 1) ? 2 : 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!more) break;
    row = next;
    r = r2;
    y = y2;
    xy = xy2;
    xe = xe2;
  }
}

__global__ __launch_bounds__(1024) void ce_finish_kernel(const float* loss_rows, int64_t N, const int64_t* n_non_ignore,
                                                         float* loss) {
  __shared__ double s_part[16];
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < N; i += 1024) acc += (double)loss_rows[i];
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    const int lo = __shfl_xor(__double2loint(acc), d), hi = __shfl_xor(__double2hiint(acc), d);
    acc += __hiloint2double(hi, lo);
  }
  if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < 16; ++w) t += s_part[w];
    *loss = (float)t / (float)*n_non_ignore;
  }
}

// Backward: four 16-byte chunks per thread, 4 KiB apart, so a wave's accesses stay contiguous and every thread has four loads in
// flight (from clamped places: with a condition around each load 4096 x 151 936 bf16 take 437 us, so 415; a pass of the loss 1407 /
// 1391).  One chunk per thread is faster where it scales (370) and slower where the scale is 1 and every workgroup
// leaves at once, the usual call (66 us instead of 18: four times the waves to start); fixed grids that walk the rows, 410 to 470.
template <typename S>
__global__ __launch_bounds__(256) void ce_scale_kernel(CeArgs p, uint32_t blocks_per_row) {
  const float s = S::round(*p.grad_output);
  if (s == 1.0f) return;  // the stored gradient is already the answer
  const uint32_t row = blockIdx.x / blocks_per_row, rb = blockIdx.x % blocks_per_row;
  char* x = p.x + (int64_t)row * p.ld;
  if (p.vec) {
    const CeRow<S> r(x, p.V);
    ce_v4i* body = (ce_v4i*)r.body();
    const uint32_t c0 = rb * 1024 + threadIdx.x;
    if (rb == 0 && r.edge(threadIdx.x)) {
      char* q = x + r.edge_at(threadIdx.x);
      S::store1(q, S::load1(q) * s);
    }
    ce_v4i w[4];
    if (r.chunks == 0) return;
    // (from a clamped place: behind a condition each load would wait for the one before)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const ce_v4i* from = body + (c0 + q * 256 < r.chunks ? c0 + q * 256 : r.chunks - 1);
      w[q] = (PT_CE_NT & 1) ? __builtin_nontemporal_load(from) : *from;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (c0 + q * 256 < r.chunks) {
        float v[CeRow<S>::kPer];
        unpack<S>(w[q], v);
#pragma unroll
        for (int i = 0; i < CeRow<S>::kPer; ++i) v[i] = v[i] * s;
        const ce_v4i g = pack<S>(v);
        if (PT_CE_NT & 2) __builtin_nontemporal_store(g, body + c0 + q * 256);
        else body[c0 + q * 256] = g;
      }
    }
  } else {
    for (int64_t i = (int64_t)rb * 256 + threadIdx.x; i < p.V; i += (int64_t)blocks_per_row * 256)
      S::store1(x + i * S::kBytes, S::load1(x + i * S::kBytes) * s);
  }
}

static int ce_args(CeArgs& a, const char* who, void* logits, int64_t ld, int dtype, int64_t N, int64_t V) {
  PT_REQUIRE(N >= 0 && V >= 1 && N < (1ll << 31) && V < (1ll << 34), "%s: bad sizes", who);
  PT_REQUIRE(ld >= V, "%s: bad leading dimension", who);
  PT_REQUIRE(dtype == PT_BF16 || dtype == PT_F16 || dtype == PT_F32, "%s: unsupported dtype %d", who, dtype);
  const int eb = dtype == PT_F32 ? 4 : 2;
  a.x = (char*)logits; a.ld = ld * eb; a.N = N; a.V = V;
  a.vec = (uintptr_t)logits % eb == 0;
  return PT_OK;
}

}  // namespace pt

using namespace pt;

extern "C" int pt_cross_entropy_fwd(void* logits, int64_t ld, int dtype, const int64_t* target, int64_t N, int64_t V,
                                    int64_t ignore_index, float* loss_rows, float* loss, int64_t* n_non_ignore,
                                    pt_stream_t stream) {
  CeArgs a = {};
  if (int rc = ce_args(a, "cross_entropy_fwd", logits, ld, dtype, N, V)) return rc;
  PT_REQUIRE(loss && n_non_ignore && (N == 0 || (logits && target && loss_rows)), "cross_entropy_fwd: null pointer");
  a.target = target; a.ignore_index = ignore_index; a.loss_rows = loss_rows; a.loss = loss; a.n_non_ignore = n_non_ignore;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(ce_count_kernel, dim3(1), dim3(1024), 0, s, target, N, ignore_index, n_non_ignore);
  const int64_t chunks = V * (dtype == PT_F32 ? 4 : 2) / 16, over = chunks - (int64_t)kCeRegChunks * kCeThreads;  // at most, of a row
  // PITHTRAIN_CE_KERNEL=twopass keeps the generic kernel for every shape (for measurements)
  static const bool onchip_allowed = [] {
    const char* e = getenv("PITHTRAIN_CE_KERNEL");
    return !(e && strcmp(e, "twopass") == 0);
  }();
  if (N && a.vec && over <= kCeLdsChunks && onchip_allowed) {
    const bool short_rows = chunks <= kCeShortChunks * kCeThreads;
    const size_t lds = over > 0 ? (size_t)over * 16 : 0;
    // more than 64 KiB of dynamic LDS has to be allowed per kernel, once per process
    static const hipError_t allow = [] {
      for (const void* k : {(const void*)ce_fwd_onchip_kernel<st_bf16, kCeRegChunks>, (const void*)ce_fwd_onchip_kernel<st_f16, kCeRegChunks>,
                            (const void*)ce_fwd_onchip_kernel<st_f32, kCeRegChunks>}) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kCeLdsChunks * 16);
        if (e != hipSuccess) return e;
      }
      return hipSuccess;
    }();
    PT_REQUIRE(allow == hipSuccess, "cross_entropy_fwd: hipFuncSetAttribute failed: %s", hipGetErrorString(allow));
    const int64_t most = short_rows ? 2 * kCeUnits : kCeUnits;
    const dim3 blocks((unsigned)(N < most ? N : most)), threads(kCeThreads);
    switch (dtype) {
#define PT_CE_LAUNCH(S)                                                                                        \
  if (short_rows) hipLaunchKernelGGL((ce_fwd_onchip_kernel<S, kCeShortChunks>), blocks, threads, 0, s, a);         \
  else hipLaunchKernelGGL((ce_fwd_onchip_kernel<S, kCeRegChunks>), blocks, threads, lds, s, a);               \
  break;
      case PT_BF16: PT_CE_LAUNCH(st_bf16)
      case PT_F16: PT_CE_LAUNCH(st_f16)
      default: PT_CE_LAUNCH(st_f32)
#undef PT_CE_LAUNCH
    }
  } else if (N) {
    switch (dtype) {
      case PT_BF16: hipLaunchKernelGGL(ce_fwd_kernel<st_bf16>, dim3((unsigned)N), dim3(kCeThreads), 0, s, a); break;
      case PT_F16: hipLaunchKernelGGL(ce_fwd_kernel<st_f16>, dim3((unsigned)N), dim3(kCeThreads), 0, s, a); break;
      default: hipLaunchKernelGGL(ce_fwd_kernel<st_f32>, dim3((unsigned)N), dim3(kCeThreads), 0, s, a); break;
    }
  }
  hipLaunchKernelGGL(ce_finish_kernel, dim3(1), dim3(1024), 0, s, loss_rows, N, n_non_ignore, loss);
  return check_launch("ce_fwd_kernel");
}

extern "C" int pt_cross_entropy_bwd(void* grad, int64_t ld, int dtype, int64_t N, int64_t V, const float* grad_output,
                                    pt_stream_t stream) {
  CeArgs a = {};
  if (int rc = ce_args(a, "cross_entropy_bwd", grad, ld, dtype, N, V)) return rc;
  if (N == 0) return PT_OK;
  PT_REQUIRE(grad && grad_output, "cross_entropy_bwd: null pointer");
  a.grad_output = grad_output;
  const int64_t bx = a.vec ? cdiv(cdiv(V * (dtype == PT_F32 ? 4 : 2), 16), 1024) : (cdiv(V, 256) < 1024 ? cdiv(V, 256) : 1024);
  PT_REQUIRE(N * bx < (1ll << 31), "cross_entropy_bwd: too many rows for one launch");
  const dim3 grid((unsigned)(N * bx));
  switch (dtype) {
    case PT_BF16: hipLaunchKernelGGL(ce_scale_kernel<st_bf16>, grid, dim3(256), 0, (hipStream_t)stream, a, (uint32_t)bx); break;
    case PT_F16: hipLaunchKernelGGL(ce_scale_kernel<st_f16>, grid, dim3(256), 0, (hipStream_t)stream, a, (uint32_t)bx); break;
    default: hipLaunchKernelGGL(ce_scale_kernel<st_f32>, grid, dim3(256), 0, (hipStream_t)stream, a, (uint32_t)bx); break;
  }
  return check_launch("ce_scale_kernel");
}

// Routing-driven permute / unpermute and expert-parallel dedup index construction (gfx950).
//
// Ordering is made deterministic with a stable counting sort: every wavefront owns a contiguous
// chunk of keys, (1) counts them into a private LDS histogram, (2) one workgroup turns the
// [chunk][group] counts into exclusive bases, (3) every wavefront replays its chunk 64 keys at a
// time, ranking equal keys inside the wave with ballot masks (one ballot per key bit) on top of
// its running LDS counters.  Up to 8192 keys one workgroup does all three; more take one launch for (1) and one in which every
// workgroup scans the counts itself before (3), or, with many chunks or groups, a launch each.  No global atomics decide a position, so the result is the
// ascending-source-row order inside every group on every run.
//
// Row movement is a separate pass over the *destination* rows (one wavefront per row, 16-byte
// accesses) so that padding rows are zeroed and data rows copied in one coalesced sweep.
#include "common.h"
#include <mutex>

// Cache policy of the row movers (build switch, make EXTRA=-DPT_PERMUTE_NT=<bits>): 1 = non-temporal
// loads of source rows, 2 = non-temporal stores of destination rows.  Source rows are read once
// (or a few times, close together, by the expanding gather) and the results are the next
// operator's input, so only the loads are non-temporal: 65 536 rows x 4 KiB, timed alone,
// permute 112 -> 104 us, gather 105 -> 80 us, gather backward 133 -> 121 us.
#ifndef PT_PERMUTE_NT
#define PT_PERMUTE_NT 1
#endif

namespace pt {

static constexpr int kWaveKeys = 256;    // keys per wavefront chunk (4 steps of 64)
static constexpr int kMaxGroups = 2048;  // LDS: 4 waves x 2048 x 4 B = 32 KiB

__device__ __forceinline__ uint64_t lanemask_lt() {
  const int lane = threadIdx.x & 63;
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// lanes (among `active`) whose key equals this lane's key
__device__ __forceinline__ uint64_t wave_match(uint32_t key, bool active, int nbits) {
  uint64_t m = __ballot(active);
  for (int b = 0; b < nbits; ++b) {
    const bool bit = (key >> b) & 1u;
    const uint64_t bal = __ballot(active && bit);
    m &= bit ? bal : ~bal;
  }
  return m;
}

static inline int bits_for(int n) { int b = 0; while ((1 << b) < n) ++b; return b < 1 ? 1 : b; }

// ---------------------------------------------------------------------------------------------
// group_rows: counts -> bases -> ranks
// ---------------------------------------------------------------------------------------------
// Also marks every entry of src_of as "no row" (the rank kernel, three launches later, overwrites
// the entries that name one).
__global__ __launch_bounds__(256) void gr_hist_kernel(const int64_t* keys, int64_t m, int G, int32_t* counts /*[W][G]*/,
                                                      int32_t* src_of, int64_t cap) {
  extern __shared__ int32_t s_hist[];  // [4][G]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < cap; i += (int64_t)gridDim.x * 256) src_of[i] = -1;
  int32_t* h = s_hist + wave * G;
  for (int g = lane; g < G; g += 64) h[g] = 0;
  __builtin_amdgcn_wave_barrier();
  const int64_t w = (int64_t)blockIdx.x * 4 + wave;
  const int64_t base = w * kWaveKeys;
  for (int s = 0; s < kWaveKeys; s += 64) {
    const int64_t i = base + s + lane;
    if (i < m) {
      const int64_t k = keys[i];
      if (k >= 0 && k < G) atomicAdd(&h[k], 1);
    }
  }
  __builtin_amdgcn_wave_barrier();
  if (base < m)
    for (int g = lane; g < G; g += 64) counts[w * G + g] = h[g];
}

// counts[W][G] -> exclusive bases over the chunks in place, one wavefront per group (64 chunks per
// step, ranked with a wave prefix sum); the group's total goes to totals[g].
__global__ __launch_bounds__(256) void gr_scan_chunks_kernel(int32_t* counts, int64_t W, int G, int32_t* totals) {
  const int lane = threadIdx.x & 63;
  const int g = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (g >= G) return;
  int32_t run = 0;
  for (int64_t w0 = 0; w0 < W; w0 += 64) {
    const int64_t w = w0 + lane;
    const int32_t c = w < W ? counts[w * G + g] : 0;
    int32_t incl = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t up = __shfl_up(incl, d);
      if (lane >= d) incl += up;
    }
    if (w < W) counts[w * G + g] = run + incl - c;
    run += __shfl(incl, 63);
  }
  if (lane == 0) totals[g] = run;
}

// one workgroup: per-group totals (read from group_start) -> padded sizes, inclusive offsets, starts
__global__ __launch_bounds__(1024) void gr_scan_groups_kernel(int G, int alignment, int32_t* offs, int32_t* ks,
                                                              int32_t* group_start /*[G]: totals in, starts out*/) {
  __shared__ int32_t s_part[1024];
  const int t = threadIdx.x;
  // thread t owns groups 2t and 2t+1 (G <= 2048)
  int32_t p0 = 0, p1 = 0;
  if (2 * t < G) p0 = (int32_t)(((int64_t)group_start[2 * t] + alignment - 1) / alignment * alignment);
  if (2 * t + 1 < G) p1 = (int32_t)(((int64_t)group_start[2 * t + 1] + alignment - 1) / alignment * alignment);
  s_part[t] = p0 + p1;
  __syncthreads();
  for (int d = 1; d < 1024; d <<= 1) {
    const int32_t add = t >= d ? s_part[t - d] : 0;
    __syncthreads();
    s_part[t] += add;
    __syncthreads();
  }
  const int32_t excl = s_part[t] - (p0 + p1);
  if (2 * t < G) {
    group_start[2 * t] = excl;
    offs[2 * t] = excl + p0;
    ks[2 * t] = p0;
  }
  if (2 * t + 1 < G) {
    group_start[2 * t + 1] = excl + p0;
    offs[2 * t + 1] = excl + p0 + p1;
    ks[2 * t + 1] = p1;
  }
}

__global__ __launch_bounds__(256) void gr_rank_kernel(const int64_t* keys, int64_t m, int G, int nbits,
                                                      const int32_t* bases /*[W][G]*/, const int32_t* group_start,
                                                      int64_t* reverse, int32_t* src_of, int64_t cap) {
  extern __shared__ int32_t s_run[];  // [4][G]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int32_t* run = s_run + wave * G;
  const int64_t w = (int64_t)blockIdx.x * 4 + wave;
  const int64_t base = w * kWaveKeys;
  if (base >= m) return;
  for (int g = lane; g < G; g += 64) run[g] = bases[w * G + g] + group_start[g];
  __builtin_amdgcn_wave_barrier();
  const uint64_t lt = lanemask_lt();
  for (int s = 0; s < kWaveKeys; s += 64) {
    const int64_t i = base + s + lane;
    int64_t k = (i < m) ? keys[i] : 0;
    const bool active = (i < m) && k >= 0 && k < G;
    if (!active) k = 0;
    const uint64_t mask = wave_match((uint32_t)k, active, nbits);
    const int rank = __popcll(mask & lt);
    const int32_t b = run[k];
    __builtin_amdgcn_wave_barrier();
    if (active && rank == 0) run[k] = b + __popcll(mask);
    __builtin_amdgcn_wave_barrier();
    if (active) {
      const int64_t pos = (int64_t)b + rank;
      if (reverse) reverse[i] = pos;
      if (pos < cap) src_of[pos] = (int32_t)i;
    } else if (i < m && reverse) {
      // a key outside [0, G) belongs to no group: the row is dropped (no src_of entry names it) and
      // its reverse entry is a valid row, so that a later gather through it stays in bounds
      reverse[i] = 0;
    }
  }
}

// The sort in two launches: the histograms are those of blocks of 1024 keys, and the workgroups of the second launch add up
// the others' themselves, up to kBlockCounts numbers (64 KiB from the L2 each), instead of waiting for two scans in launches
// of their own.  Four launches / two, us: 65 536 keys of 128 groups 15.3 / 12.6, 131 072 18.2 / 17.3, 32 768 of 16 12.8 / 7.7,
// 262 144 of 64 22.5 / 17.0; past the limit 262 144 of 128 24.1 / 25.9.  (One workgroup and two launches: 4096 keys of 128 groups
// 8.5 / 8.7, 8192 12.6 / 9.1; but so short a list belongs to a step that waits for the host, whom a launch costs 4.)
static constexpr int kBlockKeys = 4 * kWaveKeys, kBlockCounts = 16384, kBlockGroups = 256;
__global__ __launch_bounds__(256) void gr_block_hist_kernel(const int64_t* keys, int64_t m, int G, int32_t* counts /*[blocks][G]*/, int32_t* src_of,
                                                            int64_t cap) {
  __shared__ int32_t s_hist[kBlockGroups];
  const int t = threadIdx.x;
  for (int g = t; g < G; g += 256) s_hist[g] = 0;
  int64_t k[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int64_t i = (int64_t)blockIdx.x * kBlockKeys + 256 * u + t;
    k[u] = i < m ? keys[i] : -1;
  }
  for (int64_t i = (int64_t)blockIdx.x * 256 + t; i < cap; i += (int64_t)gridDim.x * 256) src_of[i] = -1;  // (see gr_hist_kernel)
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (k[u] >= 0 && k[u] < G) atomicAdd(&s_hist[k[u]], 1);
  __syncthreads();
  for (int g = t; g < G; g += 256) counts[(int64_t)blockIdx.x * G + g] = s_hist[g];
}

__global__ __launch_bounds__(256) void gr_block_rank_kernel(const int64_t* keys, int64_t m, int G, int nbits, int alignment, const int32_t* counts,
                                                            int32_t* offs, int32_t* ks, int64_t* reverse, int32_t* src_of, int64_t cap) {
  __shared__ int32_t s_run[4 * kBlockGroups], s_total[kBlockGroups], s_before[kBlockGroups], s_w[4];
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, block = blockIdx.x, blocks = gridDim.x;
  int32_t* run = s_run + wave * G;
  const int64_t base = (int64_t)block * kBlockKeys + wave * kWaveKeys;
  int64_t keys4[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int64_t i = base + 64 * u + lane;
    keys4[u] = i < m ? keys[i] : -1;
  }
  for (int g = t; g < G; g += 256) s_total[g] = s_before[g] = 0;
  for (int g = lane; g < G; g += 64) run[g] = 0;
  __syncthreads();
  // every group's keys in all blocks and in those before this one: as many threads to a group as there are
  const int parts = 256 / G, g = t % G, part = t / G;
  if (part < parts) {
    int32_t total = 0, before = 0;
#pragma unroll 16
    for (int b = part; b < blocks; b += parts) {
      const int32_t c = counts[b * G + g];
      total += c;
      before += b < block ? c : 0;
    }
    if (total) {
      atomicAdd(&s_total[g], total);
      if (before) atomicAdd(&s_before[g], before);
    }
  }
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (keys4[u] >= 0 && keys4[u] < G) atomicAdd(&run[keys4[u]], 1);
  __syncthreads();
  // thread g: the group's padded size, where it starts, and where each wave's rows do
  const int32_t size = t < G ? (int32_t)(((int64_t)s_total[t] + alignment - 1) / alignment * alignment) : 0;
  int32_t incl = size;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int32_t up = __shfl_up(incl, d);
    if (lane >= d) incl += up;
  }
  if (lane == 63) s_w[wave] = incl;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 4; ++w) incl += w < wave ? s_w[w] : 0;
  if (t < G) {
    int32_t at = incl - size + s_before[t];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const int32_t c = s_run[w * G + t];
      s_run[w * G + t] = at;
      at += c;
    }
    if (block == 0) {
      offs[t] = incl;
      ks[t] = size;
    }
  }
  __syncthreads();
  const uint64_t lt = lanemask_lt();
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int64_t i = base + 64 * u + lane;
    int64_t k = keys4[u];
    const bool active = i < m && k >= 0 && k < G;
    if (!active) k = 0;
    const uint64_t mask = wave_match((uint32_t)k, active, nbits);
    const int rank = __popcll(mask & lt);
    const int32_t b = run[k];
    __builtin_amdgcn_wave_barrier();
    if (active && rank == 0) run[k] = b + __popcll(mask);
    __builtin_amdgcn_wave_barrier();
    const int64_t pos = active ? (int64_t)b + rank : 0;  // a key outside [0, G): see gr_rank_kernel
    if (i < m && reverse) reverse[i] = pos;
    if (active && pos < cap) src_of[pos] = (int32_t)i;
  }
}

// The whole sort in one workgroup, for lists short enough that three more launches cost more than one
// compute unit's memory path: 16 waves own contiguous segments of the keys; histogram, scan and
// ranks as above, with the [wave][group] counters in LDS and workgroup barriers between the phases.
// Entries of src_of that name no row (a group's padding, the buffer's tail) are filled from the
// group sizes, so that no entry is written twice.  Bound by latency: a wave's step reads 64 keys,
// ranks them with one ballot per key bit and writes two scattered words per key.
static constexpr int kOneGroupMax = 512;     // LDS: 16 waves x 512 x 4 B
__global__ __launch_bounds__(1024) void gr_one_kernel(const int64_t* keys, int64_t m, int G, int nbits, int alignment,
                                                      int32_t* offs, int32_t* ks, int64_t* reverse, int32_t* src_of, int64_t cap) {
  __shared__ int32_t s_cnt[16 * kOneGroupMax];  // [wave][G]: counts, then running positions
  __shared__ int32_t s_start[kOneGroupMax + 1], s_size[kOneGroupMax], s_w[16];
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  int32_t* cnt = s_cnt + wave * G;
  for (int g = lane; g < G; g += 64) cnt[g] = 0;
  const int64_t seg = ((m + 15) / 16 + 63) & ~(int64_t)63;
  const int64_t begin = wave * seg, end = begin + seg < m ? begin + seg : m;
  for (int64_t i0 = begin; i0 < end; i0 += 256) {  // four loads in flight
    int64_t k[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t i = i0 + 64 * u + lane;
      k[u] = i < end ? keys[i] : -1;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k[u] >= 0 && k[u] < G) atomicAdd(&cnt[k[u]], 1);
  }
  __syncthreads();
  // thread g: the group's bases per wave, its total and its padded size; scan of the padded sizes
  int32_t total = 0, padded = 0;
  if (t < G) {
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const int32_t c = s_cnt[w * G + t];
      s_cnt[w * G + t] = total;
      total += c;
    }
    padded = (int32_t)(((int64_t)total + alignment - 1) / alignment * alignment);
  }
  int32_t incl = padded;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int32_t up = __shfl_up(incl, d);
    if (lane >= d) incl += up;
  }
  if (lane == 63) s_w[wave] = incl;
  __syncthreads();
  int32_t before = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) before += w < wave ? s_w[w] : 0;
  incl += before;
  if (t < G) {
    s_start[t] = incl - padded;
    s_size[t] = total;
    offs[t] = incl;
    ks[t] = padded;
    if (t == G - 1) s_start[G] = incl;
  }
  __syncthreads();
  for (int g = wave; g < G; g += 16) {
    const int64_t stop = s_start[g + 1] < cap ? s_start[g + 1] : cap;
    for (int64_t r = s_start[g] + s_size[g] + lane; r < stop; r += 64) src_of[r] = -1;
  }
  for (int64_t r = s_start[G] + t; r < cap; r += 1024) src_of[r] = -1;
  for (int g = lane; g < G; g += 64) cnt[g] += s_start[g];
  __builtin_amdgcn_wave_barrier();
  const uint64_t lt = lanemask_lt();
  int64_t next = begin + lane < end ? keys[begin + lane] : 0;
  for (int64_t i0 = begin; i0 < end; i0 += 64) {
    const int64_t i = i0 + lane;
    int64_t k = next;
    next = i + 64 < end ? keys[i + 64] : 0;  // requested before this step's ranks
    const bool active = i < end && k >= 0 && k < G;
    if (!active) k = 0;
    const uint64_t mask = wave_match((uint32_t)k, active, nbits);
    const int rank = __popcll(mask & lt);
    const int32_t b = cnt[k];
    __builtin_amdgcn_wave_barrier();
    if (active && rank == 0) cnt[k] = b + __popcll(mask);
    __builtin_amdgcn_wave_barrier();
    const int64_t pos = active ? (int64_t)b + rank : 0;  // a key outside [0, G): see gr_rank_kernel
    if (i < end && reverse) reverse[i] = pos;
    if (active && pos < cap) src_of[pos] = (int32_t)i;
  }
}

__global__ void fill_i32_kernel(int32_t* p, int64_t n, int32_t v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ---------------------------------------------------------------------------------------------
// row movement: one wavefront per destination row
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ nt_u4 row_ld(const nt_u4* p) { return (PT_PERMUTE_NT & 1) ? __builtin_nontemporal_load(p) : *p; }
__device__ __forceinline__ void row_st(nt_u4* p, nt_u4 v) {
  if (PT_PERMUTE_NT & 2) __builtin_nontemporal_store(v, p);
  else *p = v;
}
template <bool VEC>
__device__ __forceinline__ void copy_row(const char* src, char* dst, int64_t row_bytes, int lane) {
  if (VEC) {
    const int64_t chunks = row_bytes >> 4;
    int64_t c = lane;
    for (; c + 192 < chunks; c += 256) {  // four 16-byte loads in flight per lane
      const nt_u4 a0 = row_ld((const nt_u4*)src + c), a1 = row_ld((const nt_u4*)src + c + 64);
      const nt_u4 a2 = row_ld((const nt_u4*)src + c + 128), a3 = row_ld((const nt_u4*)src + c + 192);
      row_st((nt_u4*)dst + c, a0); row_st((nt_u4*)dst + c + 64, a1); row_st((nt_u4*)dst + c + 128, a2); row_st((nt_u4*)dst + c + 192, a3);
    }
    for (; c < chunks; c += 64) row_st((nt_u4*)dst + c, row_ld((const nt_u4*)src + c));
  } else {
    for (int64_t b = lane; b < row_bytes; b += 64) dst[b] = src[b];
  }
}
template <bool VEC>
__device__ __forceinline__ void zero_row(char* dst, int64_t row_bytes, int lane) {
  if (VEC) {
    const int64_t chunks = row_bytes >> 4;
    for (int64_t c = lane; c < chunks; c += 64) ((uint4*)dst)[c] = make_uint4(0, 0, 0, 0);
  } else {
    for (int64_t b = lane; b < row_bytes; b += 64) dst[b] = 0;
  }
}

template <bool VEC>
__global__ __launch_bounds__(256) void permute_rows_kernel(const char* in, int64_t ld_in_b, char* out, int64_t ld_out_b,
                                                           const int32_t* src_of, const int64_t* pre,
                                                           const int32_t* offs_last, int tail_alignment, int64_t cap,
                                                           int64_t row_bytes) {
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  int64_t rows_out = cap;
  if (offs_last) {
    const int64_t last = offs_last[0];
    const int64_t rounded = (last + tail_alignment - 1) / tail_alignment * tail_alignment;
    rows_out = rounded < cap ? rounded : cap;
  }
  if (r >= rows_out) return;
  int64_t s = src_of[r];
  char* dst = out + r * ld_out_b;
  if (s < 0) {
    zero_row<VEC>(dst, row_bytes, lane);
  } else {
    if (pre) s = pre[s];
    copy_row<VEC>(in + s * ld_in_b, dst, row_bytes, lane);
  }
}

template <bool VEC>
__global__ __launch_bounds__(256) void gather_rows_kernel(const char* in, int64_t ld_in_b, char* out, int64_t ld_out_b,
                                                          const int64_t* index, int64_t n, int64_t row_bytes) {
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= n) return;
  copy_row<VEC>(in + index[r] * ld_in_b, out + r * ld_out_b, row_bytes, lane);
}

// ---------------------------------------------------------------------------------------------
// gather backward: deterministic sum of the gradient rows that share an index
// ---------------------------------------------------------------------------------------------
// Every destination row has room for kGbSlots source rows; what does not fit is chained.  Counting,
// scanning the counts and filling a list in their order took six launches for what is one pass over
// the indices (262 144 of them: 52 us; 32 768: 28 us).  The order in which the atomics fill the slots does
// not matter: the sum sorts a row's sources.
static constexpr int kGbSlots = 8;
__global__ __launch_bounds__(256) void gb_link_kernel(const int64_t* index, int64_t n, int64_t rows, int32_t* cnt, int32_t* head,
                                                      int32_t* slots /*[rows][kGbSlots]*/, int32_t* next /*[n]*/) {
  const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (j >= n) return;
  const int64_t r = index[j];
  if (r < 0 || r >= rows) return;
  const int32_t at = atomicAdd(&cnt[r], 1);
  if (at < kGbSlots) slots[r * kGbSlots + at] = (int32_t)j;
  else next[j] = atomicExch(&head[r], (int32_t)j + 1);  // links hold source + 1; 0 ends the chain
}

// Where the rows of a grouped tensor go: to their destination row at once when it has no other source (see
// pt_gather_rows_backward_begin).  Of 262 144 rows whose quarter re-uses another one's source, 54 % do; the sum then moves 177 000
// rows instead of 459 000.
__global__ __launch_bounds__(256) void gb_destinations_kernel(const int32_t* row_map, int64_t M, const int64_t* index, int64_t n, int64_t rows,
                                                              const int32_t* cnt, int32_t* dest) {
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (q >= M) return;
  const int32_t j = row_map[q];
  int32_t to = -1;
  if (j >= 0 && j < n) {
    const int64_t r = index[j];
    if (r >= 0 && r < rows) to = cnt[r] == 1 ? (int32_t)r : -2 - j;
  }
  dest[q] = to;
}

// one wavefront per destination row; each lane owns 8-element chunks lane, lane+64, ...  SHARED: rows with one source have
// been written already.
template <typename S, bool VEC, bool SHARED = false>
__global__ __launch_bounds__(256) void gb_sum_kernel(const char* go, int64_t ld_go_b, char* gi, int64_t ld_gi_b,
                                                     const int32_t* cnts, const int32_t* head, const int32_t* slots,
                                                     const int32_t* next, int32_t* list, int32_t* list_end, int64_t rows, int64_t H) {
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  const int32_t cnt = cnts[r];
  if (SHARED && cnt == 1) return;
  // Sources are summed in ascending order.  Up to 64 of them are rank-sorted in registers; a longer
  // row takes its own piece of `list` and a lane-0 insertion sort in it.
  int32_t mine = 0x7FFFFFFF, s0 = 0;
  int rank = -1;
  if (cnt <= 64) {
    if (lane < cnt && lane < kGbSlots) mine = slots[r * kGbSlots + lane];
    if (cnt > kGbSlots) {
      int32_t link = head[r];
      for (int q = kGbSlots; q < cnt; ++q) {
        if (lane == q) mine = link - 1;
        link = next[link - 1];
      }
    }
    rank = 0;
    for (int q = 0; q < cnt; ++q) rank += (__shfl(mine, q) < mine) ? 1 : 0;
    if (lane >= cnt) rank = -1;
  } else {
    if (lane == 0) {
      s0 = atomicAdd(list_end, cnt);  // the rows' counts add up to at most n, the length of the list
      int32_t link = head[r];
      for (int a = 0; a < cnt; ++a) {
        const int32_t v = a < kGbSlots ? slots[r * kGbSlots + a] : link - 1;
        if (a >= kGbSlots) link = next[link - 1];
        int b = a - 1;
        while (b >= 0 && list[s0 + b] > v) { list[s0 + b + 1] = list[s0 + b]; --b; }
        list[s0 + b + 1] = v;
      }
    }
    s0 = __shfl(s0, 0);
    __threadfence();
    __builtin_amdgcn_wave_barrier();
  }
  char* dst = gi + r * ld_gi_b;
  auto source = [&](int q) -> int64_t {
    if (cnt <= 64) {
      const uint64_t b = __ballot(rank == q);
      return __shfl(mine, __ffsll((unsigned long long)b) - 1);
    }
    return ((volatile int32_t*)list)[s0 + q];
  };
  if (VEC) {
    // Four 16-byte chunks per lane and source row in flight (2048 elements of a row per pass): with
    // one, a wave waits a full memory latency per source row.  The additions keep their order:
    // sources ascending, one accumulator per element.
    // (all 64 lanes stay in the loop whatever H is: each may hold a source that the others ask for)
    for (int64_t hb = 0; hb < H; hb += 2048) {
      const int64_t h0 = hb + lane * 8, h_ok = h0 < H ? h0 : 0;
      float acc[4][8];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[u][e] = 0.f;
      for (int q = 0; q < cnt; ++q) {
        const char* src = go + source(q) * ld_go_b;
        // (a chunk past the end of the row reads the lane's first chunk again and is not added:
        // no branch around a load, which would make the wave wait for one before asking for the next)
        float v[4][8];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          load8_policy<S, (PT_PERMUTE_NT & 1) != 0>(src + (h0 + u * 512 < H ? h0 + u * 512 : h_ok) * S::kBytes, v[u]);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[u][e] = h0 + u * 512 < H ? acc[u][e] + v[u][e] : acc[u][e];
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (h0 + u * 512 < H) S::store8(dst + (h0 + u * 512) * S::kBytes, acc[u]);
    }
  } else {
    for (int64_t hb = 0; hb < H; hb += 512) {
      const int64_t h0 = hb + lane * 8;
      float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int q = 0; q < cnt; ++q) {
        const char* src = go + source(q) * ld_go_b;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (h0 + e < H) acc[e] += S::load1(src + (h0 + e) * S::kBytes);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (h0 + e < H) S::store1(dst + (h0 + e) * S::kBytes, acc[e]);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// group indices
// ---------------------------------------------------------------------------------------------
template <typename O>
__global__ void group_indices_kernel(const int32_t* offs, int G, int64_t M, O* out) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= M) return;
  int lo = 0, hi = G;  // first g with offs[g] > r
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if ((int64_t)offs[mid] <= r) lo = mid + 1; else hi = mid;
  }
  out[r] = (O)(lo < G - 1 ? lo : G - 1);
}

// ---------------------------------------------------------------------------------------------
// dedup dispatch
// ---------------------------------------------------------------------------------------------
static constexpr int kWaveTokens = 64;  // tokens per wave of the dedup kernels (one step of 64 lanes)
static constexpr int kMaxExperts = 1024;

__device__ __forceinline__ int64_t topk_at(const int64_t* ids, int64_t ld, int k, int64_t flat) {
  const int64_t t = flat / k;
  return ids[t * ld + (flat - t * k)];
}

__global__ __launch_bounds__(256) void dd_hist_kernel(const int64_t* ids, int64_t ld, int64_t m, int k, int E, int ep,
                                                      int epr, int32_t* cnt_e /*[W][E]*/, int32_t* cnt_g /*[W][ep]*/) {
  extern __shared__ int32_t s_h[];  // [4][E + 32]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int32_t* he = s_h + wave * (E + 32);
  int32_t* hg = he + E;
  for (int e = lane; e < E + 32; e += 64) he[e] = 0;
  __builtin_amdgcn_wave_barrier();
  const int64_t w = (int64_t)blockIdx.x * 4 + wave;
  const int64_t t0 = w * kWaveTokens;
  for (int s = 0; s < kWaveTokens; s += 64) {
    const int64_t t = t0 + s + lane;
    if (t < m) {
      uint32_t visited = 0;
      for (int j = 0; j < k; ++j) {
        const int64_t e = ids[t * ld + j];
        if (e >= 0 && e < E) {
          atomicAdd(&he[e], 1);
          const uint32_t bit = 1u << (uint32_t)(e / epr);
          if (!(visited & bit)) atomicAdd(&hg[e / epr], 1);
          visited |= bit;
        }
      }
    }
  }
  __builtin_amdgcn_wave_barrier();
  if (t0 < m) {
    for (int e = lane; e < E; e += 64) cnt_e[w * E + e] = he[e];
    for (int g = lane; g < ep; g += 64) cnt_g[w * ep + g] = hg[g];
  }
}

// Exclusive scan down one column of the per-wave count tables (column c < E: expert c, else EP rank
// c - E), one wave per column, 64 chunks per step; the column total goes to totals[c].
__global__ __launch_bounds__(256) void dd_scan_cols_kernel(int32_t* cnt_e, int32_t* cnt_g, int64_t W, int E, int ep,
                                                           int32_t* totals /*[E + ep]*/) {
  const int lane = threadIdx.x & 63;
  const int c = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (c >= E + ep) return;
  int32_t* col = c < E ? cnt_e + c : cnt_g + (c - E);
  const int64_t stride = c < E ? E : ep;
  int32_t run = 0;
  for (int64_t w0 = 0; w0 < W; w0 += 64) {
    const int64_t w = w0 + lane;
    const int32_t v = w < W ? col[w * stride] : 0;
    int32_t incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t y = __shfl_up(incl, d);
      if (lane >= d) incl += y;
    }
    if (w < W) col[w * stride] = run + incl - v;
    run += __shfl(incl, 63);
  }
  if (lane == 0) totals[c] = run;
}

// Starts of the experts and of the EP ranks from the column totals, and the per-rank metadata.
__global__ __launch_bounds__(64) void dd_scan_totals_kernel(const int32_t* totals, int E, int ep, int epr,
                                                            int64_t* tokens_per_ep_rank, int64_t* dedup_tokens_per_gpu,
                                                            int64_t* send_meta, int32_t* expert_starts, int32_t* gpu_starts) {
  const int lane = threadIdx.x;  // one wave
  // exclusive scan over the experts, 64 at a time
  int32_t run = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int e = e0 + lane;
    const int32_t c = e < E ? totals[e] : 0;
    int32_t incl = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t y = __shfl_up(incl, d);
      if (lane >= d) incl += y;
    }
    if (e < E) {
      expert_starts[e] = run + incl - c;
      send_meta[(e / epr) * (epr + 1) + (e % epr)] = c;
    }
    run += __shfl(incl, 63);
  }
  // per EP rank: rows routed to it, unique tokens sent to it, start of its slice of the dispatch list
  const int g = lane;
  int32_t sg = 0;
  int64_t rank_total = 0;
  if (g < ep) {
    sg = totals[E + g];
    for (int e = 0; e < epr; ++e) rank_total += totals[g * epr + e];
  }
  int32_t incl = sg;
#pragma unroll
  for (int d = 1; d < 32; d <<= 1) {
    const int32_t y = __shfl_up(incl, d);
    if (lane >= d) incl += y;
  }
  if (g < ep) {
    tokens_per_ep_rank[g] = rank_total;
    dedup_tokens_per_gpu[g] = sg;
    gpu_starts[g] = incl - sg;
    send_meta[g * (epr + 1) + epr] = sg;
  }
}

__global__ __launch_bounds__(256) void dd_rank_kernel(const int64_t* ids, int64_t ld, int64_t m, int k, int E, int ep,
                                                      int epr, int nbits, const int32_t* base_e, const int32_t* base_g,
                                                      const int32_t* expert_starts, const int32_t* gpu_starts,
                                                      int64_t* dispatch, int64_t* idxs, int64_t* expand_idx) {
  extern __shared__ int32_t s_r[];  // per wave: run_e[E], run_g[32], lp[64][ep]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int per_wave = E + 32 + 64 * ep;
  int32_t* run_e = s_r + wave * per_wave;
  int32_t* run_g = run_e + E;
  int32_t* lp = run_g + 32;
  const int64_t w = (int64_t)blockIdx.x * 4 + wave;
  const int64_t t0 = w * kWaveTokens;
  if (t0 >= m) return;
  for (int e = lane; e < E; e += 64) run_e[e] = base_e[w * E + e] + expert_starts[e];
  for (int g = lane; g < ep; g += 64) run_g[g] = base_g[w * ep + g];
  __builtin_amdgcn_wave_barrier();
  const uint64_t lt = lanemask_lt();
  for (int s = 0; s < kWaveTokens; s += 64) {
    const int64_t tb = t0 + s;  // first token of this step
    if (tb >= m) break;
    // ---- phase A: first-visit dedup positions of 64 tokens ----
    const int64_t t = tb + lane;
    uint32_t visited = 0;
    if (t < m)
      for (int j = 0; j < k; ++j) {
        const int64_t e = ids[t * ld + j];
        if (e >= 0 && e < E) visited |= 1u << (uint32_t)(e / epr);
      }
    for (int g = 0; g < ep; ++g) {
      const bool v = (visited >> g) & 1u;
      const uint64_t bal = __ballot(v);
      const int32_t b = run_g[g];
      __builtin_amdgcn_wave_barrier();
      if (v) {
        const int32_t pos = b + __popcll(bal & lt);
        lp[lane * ep + g] = pos;
        dispatch[(int64_t)gpu_starts[g] + pos] = t;
      }
      if (lane == 0) run_g[g] = b + __popcll(bal);
      __builtin_amdgcn_wave_barrier();
    }
    // ---- phase B: stable counting sort of the 64*k flat entries of these tokens ----
    const int64_t ntok = (m - tb) < 64 ? (m - tb) : 64;
    const int64_t nflat = ntok * k;
    for (int64_t q = 0; q < nflat; q += 64) {
      const int64_t fl = q + lane;  // flat index local to this step
      const bool in = fl < nflat;
      const int64_t f = tb * k + fl;
      int64_t e = in ? topk_at(ids, ld, k, f) : 0;
      const bool active = in && e >= 0 && e < E;
      if (!active) e = 0;
      const uint64_t mask = wave_match((uint32_t)e, active, nbits);
      const int rank = __popcll(mask & lt);
      const int32_t b = run_e[e];
      __builtin_amdgcn_wave_barrier();
      if (active && rank == 0) run_e[e] = b + __popcll(mask);
      __builtin_amdgcn_wave_barrier();
      if (active) {
        const int64_t pos = (int64_t)b + rank;
        idxs[pos] = f;
        expand_idx[pos] = lp[(int)(fl / k) * ep + (int)(e / epr)];
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// The same in two launches, up to kBlockCounts numbers in the count table (64 KiB from the L2 for each workgroup of the second
// launch) and kDedupBlockTopK choices a token.  A workgroup takes 256 tokens and loads their choices flat, four a lane in
// flight, instead of a lane the choices of its token one after the other.  What bounds it is the chain of loads, scans and
// ballots.  Four launches / two, us for 128 experts of 8 ranks, 8 choices a token: 256 tokens 22.0 / 14.1, 4096 22.8 / 15.3, 30 000
// 28.3 / 20.3; 65 536 tokens, 4 of 32 experts of 4 ranks 25.5 / 12.8.  (The limits are those of the sort above: past them
// every workgroup reads more counts than the two scans take.)
static constexpr int kDedupBlockTopK = 16;
static bool dedup_in_two_launches(int64_t m, int k, int E, int ep) {
  return k <= kDedupBlockTopK && E + ep <= kBlockGroups && cdiv(m, 4 * kWaveTokens) * (E + ep) <= kBlockCounts;
}

// f(position in the wave's flat list, token of the wave, choice or -1) for the wave's tokens from t0 on
template <typename F>
__device__ __forceinline__ void for_choices(const int64_t* ids, int64_t ld, int64_t m, int k, int E, int64_t t0, F f) {
  const int lane = threadIdx.x & 63;
  const int n = (int)(m - t0 < kWaveTokens ? (m - t0 > 0 ? m - t0 : 0) : kWaveTokens) * k;
  for (int q = lane; q < n; q += 4 * 64) {
    int64_t e[4];
    int token[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {  // (from a clamped place: behind a condition each load would wait for the one before)
      const int fl = q + 64 * u < n ? q + 64 * u : q;
      token[u] = fl / k;
      e[u] = ids[(t0 + token[u]) * ld + (fl - token[u] * k)];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (q + 64 * u < n) f(q + 64 * u, token[u], e[u] >= 0 && e[u] < E ? (int)e[u] : -1);
  }
}

__global__ __launch_bounds__(256) void dd_block_hist_kernel(const int64_t* ids, int64_t ld, int64_t m, int k, int E, int ep, int epr,
                                                            int32_t* counts /*[blocks][E + ep]*/) {
  __shared__ int32_t s_count[kBlockGroups];
  __shared__ uint32_t s_visited[256];
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  s_count[t] = 0;
  s_visited[t] = 0;
  __syncthreads();
  for_choices(ids, ld, m, k, E, ((int64_t)blockIdx.x * 4 + wave) * kWaveTokens, [&](int, int token, int e) {
    if (e < 0) return;
    atomicAdd(&s_count[e], 1);
    atomicOr(&s_visited[wave * 64 + token], 1u << (e / epr));
  });
  __syncthreads();
  const uint32_t visited = s_visited[t];
  for (int g = 0; g < ep; ++g) {
    const int n = __popcll(__ballot((visited >> g) & 1u));
    if (lane == 0 && n) atomicAdd(&s_count[E + g], n);
  }
  __syncthreads();
  if (t < E + ep) counts[(int64_t)blockIdx.x * (E + ep) + t] = s_count[t];
}

__global__ __launch_bounds__(256) void dd_block_rank_kernel(const int64_t* ids, int64_t ld, int64_t m, int k, int E, int ep, int epr, int nbits,
                                                            const int32_t* counts, int64_t* tokens_per_ep_rank,
                                                            int64_t* dedup_tokens_per_gpu, int64_t* send_meta, int64_t* dispatch,
                                                            int64_t* idxs, int64_t* expand_idx) {
  extern __shared__ int32_t s_b[];  // per wave: run[E + ep], lp[64][ep], the choices [64][k]
  __shared__ int32_t s_total[kBlockGroups], s_before[kBlockGroups], s_start[kBlockGroups], s_w[4];
  __shared__ uint32_t s_visited[256];
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, block = blockIdx.x, blocks = gridDim.x, C = E + ep;
  const int per_wave = C + 64 * ep + 64 * k;
  int32_t* run = s_b + wave * per_wave;
  int32_t* lp = run + C;
  int32_t* choice = lp + 64 * ep;
  const int64_t t0 = ((int64_t)block * 4 + wave) * kWaveTokens;
  s_total[t] = s_before[t] = 0;
  s_visited[t] = 0;
  for (int c = lane; c < C; c += 64) run[c] = 0;
  __syncthreads();
  // every column's sum over all blocks and over those before this one: as many threads to a column as there are
  const int parts = 256 / C, col = t % C, part = t / C;
  if (part < parts) {
    int32_t total = 0, before = 0;
#pragma unroll 16
    for (int b = part; b < blocks; b += parts) {
      const int32_t c = counts[b * C + col];
      total += c;
      before += b < block ? c : 0;
    }
    if (total) {
      atomicAdd(&s_total[col], total);
      if (before) atomicAdd(&s_before[col], before);
    }
  }
  for_choices(ids, ld, m, k, E, t0, [&](int fl, int token, int e) {
    choice[fl] = e;
    if (e < 0) return;
    atomicAdd(&run[e], 1);
    atomicOr(&s_visited[wave * 64 + token], 1u << (e / epr));
  });
  __syncthreads();
  const uint32_t visited = s_visited[t];
  for (int g = 0; g < ep; ++g) {
    const int n = __popcll(__ballot((visited >> g) & 1u));
    if (lane == 0) run[E + g] = n;
  }
  const int32_t size = s_total[t];
  int32_t incl = size;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int32_t up = __shfl_up(incl, d);
    if (lane >= d) incl += up;
  }
  if (lane == 63) s_w[wave] = incl;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 4; ++w) incl += w < wave ? s_w[w] : 0;
  s_start[t] = incl - size;  // of the ranks behind all experts: their sum is taken off below
  if (t < C) {
    // where each wave's rows of an expert go, and its unique tokens in the slice of a rank
    int32_t at = (t < E ? incl - size : 0) + s_before[t];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      int32_t* r = s_b + w * per_wave + t;
      const int32_t c = *r;
      *r = at;
      at += c;
    }
  }
  __syncthreads();
  if (block == 0 && t < E) send_meta[(t / epr) * (epr + 1) + t % epr] = size;
  if (block == 0 && t >= E && t < C) {
    const int g = t - E;
    tokens_per_ep_rank[g] = s_start[(g + 1) * epr] - s_start[g * epr];
    dedup_tokens_per_gpu[g] = size;
    send_meta[g * (epr + 1) + epr] = size;
  }
  const uint64_t lt = lanemask_lt();
  for (int g = 0; g < ep; ++g) {
    const bool v = (visited >> g) & 1u;
    const uint64_t bal = __ballot(v);
    if (v) {
      const int32_t pos = run[E + g] + __popcll(bal & lt);
      lp[lane * ep + g] = pos;
      dispatch[(int64_t)(s_start[E + g] - s_start[E]) + pos] = t0 + lane;
    }
  }
  __builtin_amdgcn_wave_barrier();
  const int n = (int)(m - t0 < kWaveTokens ? (m - t0 > 0 ? m - t0 : 0) : kWaveTokens) * k;
  for (int q = 0; q < n; q += 64) {
    const int fl = q + lane;
    int e = fl < n ? choice[fl] : -1;
    const bool active = e >= 0;
    if (!active) e = 0;
    const uint64_t mask = wave_match((uint32_t)e, active, nbits);
    const int rank = __popcll(mask & lt);
    const int32_t b = run[e];
    __builtin_amdgcn_wave_barrier();
    if (active && rank == 0) run[e] = b + __popcll(mask);
    __builtin_amdgcn_wave_barrier();
    if (active) {
      const int64_t pos = (int64_t)b + rank;
      idxs[pos] = t0 * k + fl;
      expand_idx[pos] = lp[(fl / k) * ep + e / epr];
    }
  }
}

__global__ __launch_bounds__(256) void build_expert_idxs_kernel(const int64_t* counts, int E, int ep, int epr,
                                                                int64_t max_total, int64_t* expert_idxs,
                                                                int64_t* output_splits) {
  __shared__ int64_t s_end[kMaxExperts];  // inclusive cumsum
  if (threadIdx.x < 64) {  // one wave, 64 experts a step (one thread alone waited for every count: 9.5 us for 128)
    int64_t run = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + (int)threadIdx.x;
      int64_t incl = e < E ? counts[e] : 0;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int64_t y = __shfl_up((long long)incl, d);
        if ((int)threadIdx.x >= d) incl += y;
      }
      if (e < E) s_end[e] = run + incl;
      run += __shfl((long long)incl, 63);
    }
  }
  __syncthreads();
  if (blockIdx.x == 0)
    for (int g = threadIdx.x; g < ep; g += blockDim.x)
      output_splits[g] = s_end[(g + 1) * epr - 1] - (g == 0 ? 0 : s_end[g * epr - 1]);
  const int64_t total = s_end[E - 1];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total || i >= max_total) return;
  int lo = 0, hi = E;  // first e with s_end[e] > i
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (s_end[mid] <= i) lo = mid + 1; else hi = mid;
  }
  expert_idxs[i] = lo % epr;
}

__global__ __launch_bounds__(256) void adjust_expand_idx_kernel(const int64_t* received, int64_t* out, const int64_t* dedup,
                                                                int64_t dedup_stride, const int64_t* splits, int ep,
                                                                int64_t n) {
  __shared__ int64_t s_bound[33], s_start[33];
  if (threadIdx.x == 0) {
    int64_t b = 0, d = 0;
    for (int g = 0; g < ep; ++g) {
      s_bound[g] = b; s_start[g] = d;
      b += splits[g]; d += dedup[g * dedup_stride];
    }
    s_bound[ep] = b;
  }
  __syncthreads();
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int64_t off = 0;
  for (int g = 0; g < ep; ++g)
    if (i >= s_bound[g] && i < s_bound[g + 1]) off = s_start[g];
  out[i] = received[i] + off;
}

static inline int64_t align_up(int64_t x, int64_t a) { return (x + a - 1) / a * a; }

}  // namespace pt

using namespace pt;

// ------------------------------------------------------------------------------------------------
// Short lists are sorted by one workgroup (gr_one_kernel): 2048 keys in 8 / 128 groups 4.5 / 6.6 us on the
// device against 10.0 / 12.5 for the four launches, 8192 keys 9.4 / 12.8 against 10.4 / 12.7 (and three
// launches less for the host), 16384 keys 16.0 / 20.9 against 10.5 / 12.6.
static bool sorted_by_one_workgroup(int64_t m, int32_t G) { return m <= 8192 && G <= kOneGroupMax; }

extern "C" int64_t pt_group_rows_workspace_bytes(int64_t m, int32_t num_groups) {
  if (sorted_by_one_workgroup(m, num_groups)) return 0;
  const int64_t W = cdiv(m > 0 ? m : 1, kWaveKeys);
  return align_up(W * num_groups * 4, 256) + align_up((int64_t)num_groups * 4, 256);
}

// The two launches of the stable counting sort, or four of a long one (chunk histograms, scan over the chunks, scan over
// the groups, ranks); `workspace` holds the [W][G] chunk counts and the G group starts
// (pt_group_rows_workspace_bytes), every byte of which is written before it is read.  (One kernel
// for both scans, with the last workgroup to finish doing the second, measured slower: the
// device-scope fences it needs write back and invalidate the XCD's L2, 8 us against a 4 us launch.)
static int group_rows_launch(const int64_t* keys, int64_t m, int32_t G, int32_t alignment, int32_t* offs, int32_t* ks,
                             int64_t* reverse, int32_t* src_of, int64_t cap, void* workspace, hipStream_t s) {
  if (sorted_by_one_workgroup(m, G)) {
    gr_one_kernel<<<1, 1024, 0, s>>>(keys, m, G, bits_for(G), alignment, offs, ks, reverse, src_of, cap);
    return check_launch("group_rows");
  }
  const int64_t W = cdiv(m, kWaveKeys), lists = cdiv(m, kBlockKeys);
  int32_t* counts = (int32_t*)workspace;
  if (lists * G <= kBlockCounts && G <= kBlockGroups) {
    gr_block_hist_kernel<<<(unsigned)lists, 256, 0, s>>>(keys, m, G, counts, src_of, cap);
    gr_block_rank_kernel<<<(unsigned)lists, 256, 0, s>>>(keys, m, G, bits_for(G), alignment, counts, offs, ks, reverse, src_of, cap);
    return check_launch("group_rows");
  }
  int32_t* group_start = (int32_t*)((char*)workspace + align_up(W * G * 4, 256));
  const unsigned blocks = (unsigned)cdiv(W, 4);
  const size_t lds = (size_t)4 * G * sizeof(int32_t);
  gr_hist_kernel<<<blocks, 256, lds, s>>>(keys, m, G, counts, src_of, cap);
  gr_scan_chunks_kernel<<<(unsigned)cdiv(G, 4), 256, 0, s>>>(counts, W, G, group_start);
  gr_scan_groups_kernel<<<1, 1024, 0, s>>>(G, alignment, offs, ks, group_start);
  gr_rank_kernel<<<blocks, 256, lds, s>>>(keys, m, G, bits_for(G), counts, group_start, reverse, src_of, cap);
  return check_launch("group_rows");
}

static int group_rows_check(const int64_t* keys, int64_t m, int32_t G, int32_t alignment, const int32_t* offs, const int32_t* ks,
                            const int64_t* reverse, const int32_t* src_of, int64_t cap) {
  PT_REQUIRE(m > 0 && G > 0 && G <= kMaxGroups && alignment > 0, "group_rows: m=%lld G=%d (max %d)", (long long)m, G, kMaxGroups);
  PT_REQUIRE(m + (int64_t)G * (alignment - 1) < (1ll << 31), "group_rows: row count exceeds int32");
  PT_REQUIRE(keys && offs && ks && src_of, "group_rows: null pointer");
  PT_REQUIRE(cap >= m, "group_rows: cap < m");
  return PT_OK;
}

extern "C" int pt_group_rows(const int64_t* keys, int64_t m, int32_t G, int32_t alignment, int32_t* offs, int32_t* ks,
                             int64_t* reverse, int32_t* src_of, int64_t cap, void* workspace, int64_t workspace_bytes,
                             pt_stream_t stream) {
  if (int rc = group_rows_check(keys, m, G, alignment, offs, ks, reverse, src_of, cap)) return rc;
  PT_REQUIRE(workspace || sorted_by_one_workgroup(m, G), "group_rows: null pointer");
  PT_REQUIRE(workspace_bytes >= pt_group_rows_workspace_bytes(m, G), "group_rows: workspace too small");
  return group_rows_launch(keys, m, G, alignment, offs, ks, reverse, src_of, cap, workspace, (hipStream_t)stream);
}

// ---- the same sort for callers that cannot allocate: its workspace is a device array that is
// part of the loaded code object (one copy per GPU, held until the process ends).  The array's
// name is only a host-side handle; the address the kernels get is looked up once per device. ----
static constexpr int64_t kStaticScratchBytes = PT_GROUP_ROWS_STATIC_MAX_WORKSPACE;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
static constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static void* g_scratch_ptr[kMaxDevices];  // device address of `scratch` on device d, null until looked up

static int static_scratch(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    set_error("group_rows_static: no current device (%s)", e != hipSuccess ? hipGetErrorString(e) : "index out of range");
    return PT_ERR_LAUNCH;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      set_error("group_rows_static: cannot find the scratch array on device %d: %s", dev, hipGetErrorString(e));
      return PT_ERR_LAUNCH;
    }
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return PT_OK;
}

extern "C" int pt_group_rows_static(const int64_t* keys, int64_t m, int32_t G, int32_t alignment, int32_t* offs, int32_t* ks,
                                    int64_t* reverse, int32_t* src_of, int64_t cap, pt_stream_t stream) {
  if (int rc = group_rows_check(keys, m, G, alignment, offs, ks, reverse, src_of, cap)) return rc;
  const int64_t need = pt_group_rows_workspace_bytes(m, G);
  PT_REQUIRE(need <= kStaticScratchBytes,
             "group_rows_static: m=%lld keys in %d groups need %lld bytes of scratch, the built-in array holds %lld "
             "(use pt_group_rows with a workspace)",
             (long long)m, G, (long long)need, (long long)kStaticScratchBytes);
  void* ws = nullptr;
  if (int rc = static_scratch(&ws)) return rc;
  return group_rows_launch(keys, m, G, alignment, offs, ks, reverse, src_of, cap, ws, (hipStream_t)stream);
}

extern "C" int pt_permute_rows(const void* in, int64_t ld_in, void* out, int64_t ld_out, const int32_t* src_of,
                               const int64_t* pre, const int32_t* offs_last, int32_t tail_alignment, int64_t cap, int64_t H,
                               int32_t elem_bytes, pt_stream_t stream) {
  if (cap == 0 || H == 0) return PT_OK;
  PT_REQUIRE(cap > 0 && H > 0 && in && out && src_of && elem_bytes > 0 && tail_alignment > 0, "permute_rows: bad arguments");
  const int64_t rb = H * elem_bytes, lib = ld_in * elem_bytes, lob = ld_out * elem_bytes;
  const bool vec = (rb % 16 == 0) && (lib % 16 == 0) && (lob % 16 == 0) && ((uintptr_t)in % 16 == 0) && ((uintptr_t)out % 16 == 0);
  const unsigned blocks = (unsigned)cdiv(cap, 4);
  hipStream_t s = (hipStream_t)stream;
  if (vec) permute_rows_kernel<true><<<blocks, 256, 0, s>>>((const char*)in, lib, (char*)out, lob, src_of, pre, offs_last, tail_alignment, cap, rb);
  else     permute_rows_kernel<false><<<blocks, 256, 0, s>>>((const char*)in, lib, (char*)out, lob, src_of, pre, offs_last, tail_alignment, cap, rb);
  return check_launch("permute_rows");
}

extern "C" int pt_gather_rows(const void* in, int64_t ld_in, void* out, int64_t ld_out, const int64_t* index, int64_t n,
                              int64_t H, int32_t elem_bytes, pt_stream_t stream) {
  if (n == 0 || H == 0) return PT_OK;
  PT_REQUIRE(n > 0 && H > 0 && in && out && index && elem_bytes > 0, "gather_rows: bad arguments");
  const int64_t rb = H * elem_bytes, lib = ld_in * elem_bytes, lob = ld_out * elem_bytes;
  const bool vec = (rb % 16 == 0) && (lib % 16 == 0) && (lob % 16 == 0) && ((uintptr_t)in % 16 == 0) && ((uintptr_t)out % 16 == 0);
  const unsigned blocks = (unsigned)cdiv(n, 4);
  hipStream_t s = (hipStream_t)stream;
  if (vec) gather_rows_kernel<true><<<blocks, 256, 0, s>>>((const char*)in, lib, (char*)out, lob, index, n, rb);
  else     gather_rows_kernel<false><<<blocks, 256, 0, s>>>((const char*)in, lib, (char*)out, lob, index, n, rb);
  return check_launch("gather_rows");
}

// zeroed by one fill: cnt[rows], head[rows], the end of the list | slots[rows][kGbSlots], next[n], list[n]
static int64_t gb_zeroed_words(int64_t rows) { return 2 * rows + 1; }
extern "C" int64_t pt_gather_rows_backward_workspace_bytes(int64_t n, int64_t rows) {
  return align_up(gb_zeroed_words(rows) * 4, 256) + align_up(rows * kGbSlots * 4, 256) + 2 * align_up((n > 0 ? n : 1) * 4, 256);
}

namespace pt {
// the workspace of a gather's backward
struct GatherBackward {
  int32_t *cnt, *head, *slots, *next, *list, *list_end;
  GatherBackward(void* workspace, int64_t n, int64_t rows) {
    char* p = (char*)workspace;
    cnt = (int32_t*)p; p += align_up(gb_zeroed_words(rows) * 4, 256);
    slots = (int32_t*)p; p += align_up(rows * kGbSlots * 4, 256);
    next = (int32_t*)p; p += align_up((n > 0 ? n : 1) * 4, 256);
    list = (int32_t*)p;
    head = cnt + rows;
    list_end = cnt + 2 * rows;
  }
  void link(const int64_t* index, int64_t n, int64_t rows, hipStream_t s) const {
    fill_i32_kernel<<<(unsigned)cdiv(gb_zeroed_words(rows), 256), 256, 0, s>>>(cnt, gb_zeroed_words(rows), 0);
    if (n > 0) gb_link_kernel<<<(unsigned)cdiv(n, 256), 256, 0, s>>>(index, n, rows, cnt, head, slots, next);
  }
  template <bool SHARED>
  int sum(const void* grad_out, int64_t ld_go, void* grad_in, int64_t ld_gi, int64_t rows, int64_t H, int dtype, hipStream_t s) const {
    const unsigned blocks = (unsigned)cdiv(rows, 4);
    const int eb = dtype == PT_F32 ? 4 : 2;
    const bool vec = (H % 8 == 0) && ((ld_go * eb) % 16 == 0) && ((ld_gi * eb) % 16 == 0) && ((uintptr_t)grad_out % 16 == 0) &&
                     ((uintptr_t)grad_in % 16 == 0);
#define PT_GB(S)                                                                                                         \
  do {                                                                                                                   \
    if (vec) gb_sum_kernel<S, true, SHARED><<<blocks, 256, 0, s>>>((const char*)grad_out, ld_go * eb, (char*)grad_in, ld_gi * eb, cnt, head, slots, next, list, list_end, rows, H); \
    else     gb_sum_kernel<S, false, SHARED><<<blocks, 256, 0, s>>>((const char*)grad_out, ld_go * eb, (char*)grad_in, ld_gi * eb, cnt, head, slots, next, list, list_end, rows, H); \
  } while (0)
    switch (dtype) {
      case PT_BF16: PT_GB(st_bf16); break;
      case PT_F16:  PT_GB(st_f16); break;
      case PT_F32:  PT_GB(st_f32); break;
      default: PT_REQUIRE(false, "gather_rows_backward: unsupported dtype %d", dtype);
    }
#undef PT_GB
    return check_launch("gather_rows_backward");
  }
};
}  // namespace pt

extern "C" int pt_gather_rows_backward(const void* grad_out, int64_t ld_go, void* grad_in, int64_t ld_gi,
                                       const int64_t* index, int64_t n, int64_t rows, int64_t H, int dtype, void* workspace,
                                       int64_t workspace_bytes, pt_stream_t stream) {
  if (rows == 0 || H == 0) return PT_OK;
  PT_REQUIRE(rows > 0 && n >= 0 && H > 0 && grad_in && workspace, "gather_rows_backward: bad arguments");
  PT_REQUIRE(n == 0 || (grad_out && index), "gather_rows_backward: null pointer");
  PT_REQUIRE(n < (1ll << 31) && rows < (1ll << 31), "gather_rows_backward: sizes exceed int32");
  PT_REQUIRE(workspace_bytes >= pt_gather_rows_backward_workspace_bytes(n, rows), "gather_rows_backward: workspace too small");
  const GatherBackward b(workspace, n, rows);
  b.link(index, n, rows, (hipStream_t)stream);
  return b.sum<false>(grad_out, ld_go, grad_in, ld_gi, rows, H, dtype, (hipStream_t)stream);
}

extern "C" int pt_gather_rows_backward_begin(const int64_t* index, int64_t n, int64_t rows, void* workspace, int64_t workspace_bytes,
                                             const int32_t* row_map, int32_t* dest, int64_t M, pt_stream_t stream) {
  PT_REQUIRE(n >= 0 && rows >= 0 && M >= 0 && workspace && (n == 0 || index) && (M == 0 || (row_map && dest)), "gather_rows_backward_begin: bad arguments");
  PT_REQUIRE(n < (1ll << 31) - 2 && rows < (1ll << 31) && M < (1ll << 31), "gather_rows_backward_begin: sizes exceed int32");
  PT_REQUIRE(workspace_bytes >= pt_gather_rows_backward_workspace_bytes(n, rows), "gather_rows_backward_begin: workspace too small");
  const GatherBackward b(workspace, n, rows);
  b.link(index, n, rows, (hipStream_t)stream);
  if (M > 0) gb_destinations_kernel<<<(unsigned)cdiv(M, 256), 256, 0, (hipStream_t)stream>>>(row_map, M, index, n, rows, b.cnt, dest);
  return check_launch("gather_rows_backward_begin");
}

extern "C" int pt_gather_rows_backward_shared(const void* grad_out, int64_t ld_go, void* grad_in, int64_t ld_gi, int64_t n, int64_t rows,
                                              int64_t H, int dtype, void* workspace, int64_t workspace_bytes, pt_stream_t stream) {
  if (rows == 0 || H == 0) return PT_OK;
  PT_REQUIRE(rows > 0 && n >= 0 && H > 0 && grad_in && workspace && (n == 0 || grad_out), "gather_rows_backward_shared: bad arguments");
  PT_REQUIRE(workspace_bytes >= pt_gather_rows_backward_workspace_bytes(n, rows), "gather_rows_backward_shared: workspace too small");
  return GatherBackward(workspace, n, rows).sum<true>(grad_out, ld_go, grad_in, ld_gi, rows, H, dtype, (hipStream_t)stream);
}

extern "C" int pt_group_indices(const int32_t* offs, int32_t G, int64_t M, void* group_ids, int32_t out_bytes,
                                pt_stream_t stream) {
  if (M == 0) return PT_OK;
  PT_REQUIRE(M > 0 && G > 0 && offs && group_ids, "group_indices: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  if (out_bytes == 4) group_indices_kernel<int32_t><<<(unsigned)cdiv(M, 256), 256, 0, s>>>(offs, G, M, (int32_t*)group_ids);
  else if (out_bytes == 8) group_indices_kernel<int64_t><<<(unsigned)cdiv(M, 256), 256, 0, s>>>(offs, G, M, (int64_t*)group_ids);
  else PT_REQUIRE(false, "group_indices: out_dtype_bytes must be 4 or 8");
  return check_launch("group_indices");
}

// out[r] = expand_idx[row_map[r]] for row_map[r] in [0, n_expand), -1 otherwise: the source row of
// every grouped row when the routed rows are themselves an expansion of deduplicated rows.
__global__ __launch_bounds__(256) void compose_row_map_kernel(const int32_t* row_map, int64_t n, const int64_t* expand_idx,
                                                              int64_t n_expand, int64_t n_src, int32_t* out) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r >= n) return;
  const int32_t i = row_map[r];
  int64_t s = -1;
  if (i >= 0 && i < n_expand) {
    s = expand_idx[i];
    if (s < 0 || s >= n_src) s = -1;  // an index outside the source rows reads nothing
  }
  out[r] = (int32_t)s;
}

extern "C" int pt_compose_row_map(const int32_t* row_map, int64_t n, const int64_t* expand_idx, int64_t n_expand,
                                  int64_t n_src, int32_t* out, pt_stream_t stream) {
  PT_REQUIRE(n >= 0 && n_expand >= 0 && n_src >= 0 && n_src < (1ll << 31), "compose_row_map: bad sizes");
  if (n == 0) return PT_OK;
  PT_REQUIRE(row_map && out && (expand_idx || n_expand == 0), "compose_row_map: null pointer");
  compose_row_map_kernel<<<(unsigned)cdiv(n, 256), 256, 0, (hipStream_t)stream>>>(row_map, n, expand_idx, n_expand, n_src, out);
  return check_launch("compose_row_map");
}

extern "C" int64_t pt_dedup_workspace_bytes(int64_t m, int32_t k, int32_t E, int32_t ep) {
  (void)k;
  const int64_t W = cdiv(m > 0 ? m : 1, kWaveTokens);
  return align_up(W * E * 4, 256) + align_up(W * ep * 4, 256) + align_up((int64_t)E * 4, 256) + 256 +
         align_up((int64_t)(E + ep) * 4, 256);
}

extern "C" int pt_dedup_prepare_dispatch(const int64_t* topk_ids, int64_t ld_ids, int64_t m, int32_t k, int32_t E,
                                         int32_t ep, int32_t epr, int64_t* tokens_per_ep_rank, int64_t* dedup_tokens_per_gpu,
                                         int64_t* dispatch_token_idxs, int64_t* idxs, int64_t* expand_idx, int64_t* send_meta,
                                         void* workspace, int64_t workspace_bytes, pt_stream_t stream) {
  PT_REQUIRE(m > 0 && k > 0 && E > 0 && E <= kMaxExperts && ep > 0 && ep <= 32 && ep * epr == E,
             "dedup_prepare_dispatch: m=%lld k=%d E=%d ep=%d epr=%d", (long long)m, k, E, ep, epr);
  PT_REQUIRE(m * k < (1ll << 31), "dedup_prepare_dispatch: m*k exceeds int32");
  PT_REQUIRE(topk_ids && tokens_per_ep_rank && dedup_tokens_per_gpu && dispatch_token_idxs && idxs && expand_idx &&
                 send_meta && workspace, "dedup_prepare_dispatch: null pointer");
  PT_REQUIRE(workspace_bytes >= pt_dedup_workspace_bytes(m, k, E, ep), "dedup_prepare_dispatch: workspace too small");
  hipStream_t s = (hipStream_t)stream;
  const int64_t W = cdiv(m, kWaveTokens);
  char* wsp = (char*)workspace;
  int32_t* cnt_e = (int32_t*)wsp; wsp += align_up(W * E * 4, 256);
  int32_t* cnt_g = (int32_t*)wsp; wsp += align_up(W * ep * 4, 256);
  int32_t* expert_starts = (int32_t*)wsp; wsp += align_up((int64_t)E * 4, 256);
  int32_t* gpu_starts = (int32_t*)wsp; wsp += 256;
  int32_t* totals = (int32_t*)wsp;
  const unsigned blocks = (unsigned)cdiv(W, 4);
  if (dedup_in_two_launches(m, k, E, ep)) {
    int32_t* counts = (int32_t*)workspace;  // blocks x (E + ep): less than the two tables
    dd_block_hist_kernel<<<blocks, 256, 0, s>>>(topk_ids, ld_ids, m, k, E, ep, epr, counts);
    dd_block_rank_kernel<<<blocks, 256, (size_t)4 * (E + ep + 64 * ep + 64 * k) * 4, s>>>(
        topk_ids, ld_ids, m, k, E, ep, epr, bits_for(E), counts, tokens_per_ep_rank, dedup_tokens_per_gpu, send_meta, dispatch_token_idxs,
        idxs, expand_idx);
    return check_launch("dedup_prepare_dispatch");
  }
  dd_hist_kernel<<<blocks, 256, (size_t)4 * (E + 32) * 4, s>>>(topk_ids, ld_ids, m, k, E, ep, epr, cnt_e, cnt_g);
  dd_scan_cols_kernel<<<(unsigned)cdiv(E + ep, 4), 256, 0, s>>>(cnt_e, cnt_g, W, E, ep, totals);
  dd_scan_totals_kernel<<<1, 64, 0, s>>>(totals, E, ep, epr, tokens_per_ep_rank, dedup_tokens_per_gpu, send_meta, expert_starts,
                                         gpu_starts);
  const size_t lds = (size_t)4 * (E + 32 + 64 * ep) * 4;
  dd_rank_kernel<<<blocks, 256, lds, s>>>(topk_ids, ld_ids, m, k, E, ep, epr, bits_for(E), cnt_e, cnt_g, expert_starts,
                                          gpu_starts, dispatch_token_idxs, idxs, expand_idx);
  return check_launch("dedup_prepare_dispatch");
}

extern "C" int pt_build_expert_idxs(const int64_t* counts, int32_t E, int32_t ep, int32_t epr, int64_t max_total,
                                    int64_t* expert_idxs, int64_t* output_splits, pt_stream_t stream) {
  PT_REQUIRE(E > 0 && E <= kMaxExperts && ep > 0 && ep * epr == E && counts && output_splits, "build_expert_idxs: bad arguments");
  PT_REQUIRE(max_total == 0 || expert_idxs, "build_expert_idxs: null pointer");
  const unsigned blocks = (unsigned)(max_total > 0 ? cdiv(max_total, 256) : 1);
  build_expert_idxs_kernel<<<blocks, 256, 0, (hipStream_t)stream>>>(counts, E, ep, epr, max_total, expert_idxs, output_splits);
  return check_launch("build_expert_idxs");
}

extern "C" int pt_adjust_expand_idx(const int64_t* received, int64_t* out, const int64_t* dedup_counts, int64_t dedup_stride,
                                    const int64_t* output_splits, int32_t ep, int64_t n, pt_stream_t stream) {
  if (n == 0) return PT_OK;
  PT_REQUIRE(n > 0 && ep > 0 && ep <= 32 && received && out && dedup_counts && output_splits, "adjust_expand_idx: bad arguments");
  adjust_expand_idx_kernel<<<(unsigned)cdiv(n, 256), 256, 0, (hipStream_t)stream>>>(received, out, dedup_counts, dedup_stride,
                                                                                      output_splits, ep, n);
  return check_launch("adjust_expand_idx");
}

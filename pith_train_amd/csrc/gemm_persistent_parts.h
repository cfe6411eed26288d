// Parts of the persistent FP8 GEMM kernel (gemm_rowsplit.hip), some of them shared with the kernel for small
// problems (gemm_small.hip): buffer descriptors and direct-to-LDS loads, the work list (group scan, tile
// geometry), the result stores, and the launch of one workgroup per CU.
#pragma once
#include "common.h"
#include "gemm_args.h"
#include <stdlib.h>

namespace pt {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

static constexpr int kMaxGroupsGemm = 2048;
#ifdef PT_GEMM_ABLATE_STORES
static constexpr bool kAblateStores = true;
#else
static constexpr bool kAblateStores = false;
#endif
static constexpr uint32_t kOob = 0x80000000u;  // per-lane offset that is out of range for every descriptor used here
// Cache-policy bits of the wide result stores (buffer instruction aux operand: 1 = sc0, 2 = nt,
// 16 = sc1), for the weight-gradient mode and for the others.  Non-temporal by default: a GEMM
// launched alone runs the same either way, but inside a training step the results (the weight
// gradients above all: 1.2 GB per step for a 128-expert layer, read by nobody soon) otherwise
// push the next kernels' operands out of the memory-side cache.  Measured on the Qwen3-30B-A3B
// step: weight gradients only -1.7 %, all modes -2.2 %, all but the weight gradients -0.3 %.
#ifndef PT_GEMM_STORE_AUX_WGRAD
#define PT_GEMM_STORE_AUX_WGRAD 2
#endif
#ifndef PT_GEMM_STORE_AUX
#define PT_GEMM_STORE_AUX 2
#endif
template <int MODE> static constexpr int kStoreAux = MODE == GEMM_K_GROUPED ? PT_GEMM_STORE_AUX_WGRAD : PT_GEMM_STORE_AUX;
static constexpr int kRsrcFlags = 0x00020000;  // raw buffer, 32-bit data format

// Raw buffer descriptor over [base, base + bytes) for the inline-assembly loads.
__device__ __forceinline__ v4i make_rsrc(const void* base, uint32_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)base;
  v4i r;
  r[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
  r[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)((a >> 32) & 0xFFFF));
  r[2] = __builtin_amdgcn_readfirstlane((int)bytes);
  r[3] = kRsrcFlags;
  return r;
}

// Direct-to-LDS buffer loads: address = base + voff (per lane) + soff (uniform); lane l's data lands
// at lds_off + 16*l (dwordx4) or lds_off + 4*l (dword).  lds_off is a wave-uniform LDS byte address.
// (PT_GEMM_LOAD_A_MOD / PT_GEMM_LOAD_B_MOD, measurement builds: cache-policy modifiers, e.g. " nt", of
// the row-split kernel's a and b operand loads.)
#ifndef PT_GEMM_LOAD_A_MOD
#define PT_GEMM_LOAD_A_MOD ""
#endif
#ifndef PT_GEMM_LOAD_B_MOD
#define PT_GEMM_LOAD_B_MOD ""
#endif
template <bool NT = false>  // NT: non-temporal
__device__ __forceinline__ void dma16(v4i rsrc, uint32_t voff, uint32_t soff, uint32_t lds_off) {
  soff = (uint32_t)__builtin_amdgcn_readfirstlane((int)soff);  // uniform by construction; pin them to SGPRs
  lds_off = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_off);
  if (NT)
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen nt lds" ::"v"(voff), "s"(rsrc), "s"(soff),
                 "s"(lds_off)
                 : "memory");
  else
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(rsrc), "s"(soff),
                 "s"(lds_off)
                 : "memory");
}
// the same at LDS byte lds_off + OFF; OPERAND 0: a, 1: b
template <int OPERAND, int OFF>
__device__ __forceinline__ void dma16_at(v4i rsrc, uint32_t voff, uint32_t soff, uint32_t lds_off) {
  soff = (uint32_t)__builtin_amdgcn_readfirstlane((int)soff);
  lds_off = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_off);
  if (OPERAND == 0)
    asm volatile("s_add_u32 m0, %3, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen" PT_GEMM_LOAD_A_MOD " lds" ::"v"(voff), "s"(rsrc),
                 "s"(soff), "s"(lds_off), "n"(OFF)
                 : "memory", "scc");
  else
    asm volatile("s_add_u32 m0, %3, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen" PT_GEMM_LOAD_B_MOD " lds" ::"v"(voff), "s"(rsrc),
                 "s"(soff), "s"(lds_off), "n"(OFF)
                 : "memory", "scc");
}
__device__ __forceinline__ void dma4(v4i rsrc, uint32_t voff, uint32_t soff, uint32_t lds_off) {
  soff = (uint32_t)__builtin_amdgcn_readfirstlane((int)soff);
  lds_off = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_off);
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dword %0, %1, %2 offen lds" ::"v"(voff), "s"(rsrc), "s"(soff),
               "s"(lds_off)
               : "memory");
}
__device__ __forceinline__ void wait_all_vmem() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

__device__ __forceinline__ uint32_t pack2_bf16(float lo, float hi) {
  const bf16x2 h = __builtin_convertvector(f32x2{lo, hi}, bf16x2);
  return __builtin_bit_cast(uint32_t, h);
}

// ---- result stores -------------------------------------------------------------------------
// The products are computed with the b fragment as the first MFMA operand, so that a lane holds one row of
// the result: row lane % 32 of a 32x32 block, columns 8 (v / 4) + 4 (lane / 32) + v % 4, i.e. four
// neighbouring columns per register quad.  A wave turns 32 rows x 128 bytes (two blocks of bf16, one of
// fp32) into whole lines through a 4 KiB staging area of its own, four pieces of 8 rows: 8- or 16-byte LDS
// writes, then four times a 16-byte read and a store of eight full lines.  With a lane per column every bf16 pair
// had to be traded with the neighbouring lane first and went to LDS in 4-byte writes: us with that / with
// this / with raw accumulator bits stored instead, 128 groups of 512 rows 1536 x 2048 243 / 238 / 233, 2048 x
// 768 137 / 132 / 128, their weight gradients 297 / 291 / 290 and 135 / 127 / 119.  (Half lines cost a
// tenth of the dense and a quarter of the weight-gradient GEMM's time in the write path; the memory
// pipeline spends the same time on a 4-byte and on a 16-byte store.)
// Only this wave touches its staging area, and the LDS executes one wave's operations in order, so the
// phases need compiler fences only.
struct Staging {
  uint32_t wr;     // the lane's place for row lane % 32, chunk 0 of the swizzle (LDS byte address)
  uint32_t rd[4];  // the lane's 16 bytes of piece q: row 8 q + lane / 8, chunk lane % 8
};
// Chunk c (16 bytes) of row m lies at position c ^ (m / 2) % 8: the 16 rows that an 8-byte write touches
// at a time spread over all banks, and so do the 8 of a 16-byte one.
__device__ __forceinline__ Staging make_staging(const uint32_t (&piece)[4], int lane) {
  Staging s;
  const int m = lane & 31, r = lane >> 3;
  const uint32_t lo = lane & 8 ? piece[1] : piece[0], hi = lane & 8 ? piece[3] : piece[2];
  s.wr = (lane & 16 ? hi : lo) + (m & 7) * 128 + (((m >> 1) & 7) << 4);
#pragma unroll
  for (int q = 0; q < 4; ++q) s.rd[q] = piece[q] + r * 128 + (((lane & 7) ^ ((4 * q + (r >> 1)) & 7)) << 4);
  return s;
}
typedef int v2i __attribute__((ext_vector_type(2)));
#define PT_LDS(TYPE, ADDR) (*(TYPE __attribute__((address_space(3)))*)(uintptr_t)(ADDR))

// A 16-byte store reads its data registers for a few cycles after it issues; the compiler only guards that
// window for stores without a scalar offset, so the registers are held here.
template <int AUX>
__device__ __forceinline__ void store16(v4i w, __amdgpu_buffer_rsrc_t out, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_buffer_store_b128(w, out, voff, soff, AUX);
  asm volatile("s_nop 4" ::"v"(w) : "memory");
}

// Writes two horizontally adjacent blocks as bf16 (one block as fp32) to the staging area, and reads back the
// lane's 16 bytes of each piece.
__device__ __forceinline__ void stage_bf16(const v16f& a0, const v16f& a1, const Staging& stg, int lane) {
  const uint32_t wr = stg.wr + (lane >> 5) * 8;
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const v16f& a = b ? a1 : a0;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      PT_LDS(v2i, wr ^ ((4 * b + q) << 4)) = v2i{(int)pack2_bf16(a[4 * q], a[4 * q + 1]), (int)pack2_bf16(a[4 * q + 2], a[4 * q + 3])};
  }
}
__device__ __forceinline__ void stage_f32(const v16f& a, const Staging& stg, int lane) {
#pragma unroll
  for (int q = 0; q < 4; ++q)
    PT_LDS(v4i, stg.wr ^ ((2 * q + (lane >> 5)) << 4)) =
        v4i{__float_as_int(a[4 * q]), __float_as_int(a[4 * q + 1]), __float_as_int(a[4 * q + 2]), __float_as_int(a[4 * q + 3])};
}
// A column of TM blocks (pairs of them as bf16) through the staging area: emit(i, q, w) gets the 16 bytes of rows
// 8 q + lane / 8 of block row i.  One block row after the other (scheduling barriers: converted all at once they
// would not fit next to the accumulators).
template <bool F32, int TM, int TN, class Emit>
__device__ __forceinline__ void stage_column(const v16f (&acc)[TM][TN], int j, const Staging& stg, int lane, Emit emit) {
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    if (F32) stage_f32(acc[i][j], stg, lane);
    else     stage_bf16(acc[i][j], acc[i][j + 1], stg, lane);
    asm volatile("" ::: "memory");  // the reads alias the writes before and behind them
    v4i w[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) w[q] = PT_LDS(const v4i, stg.rd[q]);
#ifdef PT_GEMM_ABLATE_STAGING
    // measurement build: the stores carry raw accumulator bits, no conversion and no staging
    for (int q = 0; q < 4; ++q) w[q] = v4i{__float_as_int(acc[i][j][4 * q]), __float_as_int(acc[i][j][4 * q + 1]), __float_as_int(acc[i][j][4 * q + 2]), __float_as_int(acc[i][j][4 * q + 3])};
#endif
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < 4; ++q) emit(i, q, w[q]);
    __builtin_amdgcn_sched_barrier(0);
  }
}
// x + y on packed bf16 pairs
__device__ __forceinline__ v4i add_bf16(v4i x, v4i y) {
#pragma unroll
  for (int k = 0; k < 4; ++k)
    x[k] = (int)pack2_bf16(bf16_lo((uint32_t)x[k]) + bf16_lo((uint32_t)y[k]), bf16_hi((uint32_t)x[k]) + bf16_hi((uint32_t)y[k]));
  return x;
}

// One block element by element, for outputs that the wide stores cannot write (a pitch, an end or a base that is
// no multiple of 16 bytes).  voff: byte offset of the lane's row and first column (kOob: no such row); cols:
// columns from the lane's first on that exist.
template <bool F32>
__device__ __forceinline__ void store_elements(const v16f& a, __amdgpu_buffer_rsrc_t out, uint32_t voff, uint32_t soff, int cols, bool accumulate) {
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int c = 8 * (v >> 2) + (v & 3);
    const uint32_t vo = c < cols ? voff : kOob, so = soff + c * (F32 ? 4 : 2);
    if (F32) {
      float x = a[v];
      if (accumulate) x += __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(out, vo, so, 0));
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, x), out, vo, so, 0);
    } else {
      uint32_t r = f32_to_bf16_bits(a[v]);
      if (accumulate) {
        const uint32_t old = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(out, vo, so, 0);
        r = f32_to_bf16_bits(bf16_bits_to_f32(old) + bf16_bits_to_f32(r));
      }
      __builtin_amdgcn_raw_buffer_store_b16((short)r, out, vo, so, 0);
    }
  }
}

// The kernel's arguments read anew from where the launch left them (the kernel takes the block by value as its
// only argument).  What a tile needs once need not stay in scalar registers during its main loop, nor be
// spilled to vector registers: the compiler cannot see that these loads return what it has read before.
__device__ __forceinline__ GemmArgs reload_args() {
#ifdef __HIP_DEVICE_COMPILE__
  typedef const GemmArgs __attribute__((address_space(4))) * ArgsPtr;
  ArgsPtr q = (ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(q));
  return *q;
#else
  return GemmArgs{};
#endif
}

// One tile of the work list; everything is wave-uniform (SGPRs).
struct Tile {
  int a_row0, b_row0, a_lim, b_lim, k_begin, k_len, kb0, g;
};

// Scaled MFMA whose scale bytes are byte `ia` of sa and byte `ib` of sb (byte index = op_sel bit +
// 2 * op_sel_hi bit, one pair per operand).  Issued as volatile inline assembly with a memory
// clobber: the compiler keeps such statements, and every memory operation between them, in source
// order, which is what pins the interleaving of MFMAs, LDS reads and direct-to-LDS loads in the
// main loop.  The accumulators live in ordinary registers ("v"; 128 of them fit next to everything else in the
// 256 a wave has at two waves per SIMD), where the epilogue reads them without a copy.
__device__ __forceinline__ void mfma_sel(const v8i& a, const v8i& b, v16f& c, int ia, int sa, int ib, int sb) {
#define PT_MFMA_TEXT(S0, S1, H0, H1) \
  "v_mfma_scale_f32_32x32x64_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel:[" #S0 "," #S1 ",0] op_sel_hi:[" #H0 "," #H1 ",0]"
#define PT_MFMA(IA, IB, S0, S1, H0, H1)                                                                                  \
  case IA * 4 + IB:                                                                                                      \
    asm volatile(PT_MFMA_TEXT(S0, S1, H0, H1) : "+v"(c) : "v"(a), "v"(b), "v"(sa), "v"(sb) : "memory");                  \
    break;
  switch (ia * 4 + ib) {
    PT_MFMA(0, 0, 0, 0, 0, 0) PT_MFMA(0, 1, 0, 1, 0, 0) PT_MFMA(0, 2, 0, 0, 0, 1) PT_MFMA(0, 3, 0, 1, 0, 1)
    PT_MFMA(1, 0, 1, 0, 0, 0) PT_MFMA(1, 1, 1, 1, 0, 0) PT_MFMA(1, 2, 1, 0, 0, 1) PT_MFMA(1, 3, 1, 1, 0, 1)
    PT_MFMA(2, 0, 0, 0, 1, 0) PT_MFMA(2, 1, 0, 1, 1, 0) PT_MFMA(2, 2, 0, 0, 1, 1) PT_MFMA(2, 3, 0, 1, 1, 1)
    PT_MFMA(3, 0, 1, 0, 1, 0) PT_MFMA(3, 1, 1, 1, 1, 0) PT_MFMA(3, 2, 1, 0, 1, 1) PT_MFMA(3, 3, 1, 1, 1, 1)
  }
#undef PT_MFMA
#undef PT_MFMA_TEXT
}

// s_pref[g] = sum of weight(g') over groups g' < g (s_pref[G] = the total, s_pref[G + 1] = the largest
// weight); computed by the first wave, followed by a workgroup barrier.
template <class E, class W>
__device__ __forceinline__ void scan_groups(const GemmArgs& p, int* s_pref, int tid, int lane, E end_of, W weight) {
  if (tid < 64) {
    // Lane l owns groups [l * per, (l + 1) * per): one global read per group, running sums kept in
    // LDS, then the lanes' totals are scanned and added to each lane's own entries.
    const int per = (p.G + 63) / 64;
    const int g0 = tid * per;
    int sum = 0, mx = 0;
    if (per <= 4) {
      // up to 256 groups: the lane's five group ends are requested together (one memory latency)
      const int last = p.G - 1;
      int e[5];
#pragma unroll
      for (int q = 0; q < 5; ++q) {
        int g = g0 - 1 + q;
        g = g < 0 ? 0 : (g > last ? last : g);
        e[q] = end_of(g);
      }
      if (g0 == 0) e[0] = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int g = g0 + q;
        if (q < per && g < p.G) {
          const int w = weight(e[q + 1] - e[q]);
          sum += w;
          mx = w > mx ? w : mx;
          s_pref[g + 1] = sum;
        }
      }
    } else {
      int prev = (g0 > 0 && g0 <= p.G) ? end_of(g0 - 1) : 0;
      for (int q = 0; q < per; ++q) {
        const int g = g0 + q;
        if (g < p.G) {
          const int cur = end_of(g);
          const int w = weight(cur - prev);
          sum += w;
          mx = w > mx ? w : mx;
          prev = cur;
          s_pref[g + 1] = sum;
        }
      }
    }
    int incl = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(incl, d);
      if (lane >= d) incl += y;
    }
    const int base = incl - sum;
    for (int q = 0; q < per; ++q) {
      const int g = g0 + q;
      if (g < p.G) s_pref[g + 1] += base;
    }
    if (tid == 0) s_pref[0] = 0;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_xor(mx, d);
      mx = y > mx ? y : mx;
    }
    if (tid == 0) s_pref[p.G + 1] = mx;  // the largest weight, after the total
  }
  __syncthreads();
}

// m-grouped: s_pref[g] = number of BM-row tiles of groups < g, from the cumulative group ends.
template <int BM>
__device__ __forceinline__ void scan_group_tiles(const GemmArgs& p, int* s_pref, int tid, int lane) {
  scan_groups(p, s_pref, tid, lane, [&](int g) { return p.offs[g]; }, [](int rows) { return (rows + BM - 1) / BM; });
}

// k-grouped: a tile of group g costs its number of 128-deep reduction blocks plus a fixed share
// for the tile switch and the result store; s_pref[g] = that cost summed over groups < g.
static constexpr int kTileFixedCost = 3;
__device__ __forceinline__ int k_group_tile_cost(int rows) { return ((rows + 127) >> 7) + kTileFixedCost; }
__device__ __forceinline__ void scan_group_costs(const GemmArgs& p, int* s_pref, int tid, int lane) {
  scan_groups(p, s_pref, tid, lane, [&](int g) { return k_group_end(p, g); }, [](int rows) { return k_group_tile_cost(rows); });
}

// Groups of nearly equal cost (largest within a quarter of the mean): the plain cut by count, which
// for a group count that is a multiple of eight also keeps whole groups on one XCD.
__device__ __forceinline__ bool level_groups(const GemmArgs& p, const int* s_pref) {
  return (int64_t)s_pref[p.G + 1] * p.G * 4 <= (int64_t)s_pref[p.G] * 5;
}

// First logical tile of XCD `x` (x in [0, 8]; x = 8 gives the end of the list).  Dense and
// m-grouped tiles all cost the same, so the list is cut into eight equal counts.  k-grouped tiles
// cost in proportion to their group's row count: the list (group-major) is cut where the summed
// cost reaches x/8 of the total, so that skewed group sizes do not leave most XCDs idle while one
// works through the large groups.  Cuts are rounded to multiples of `round`, the number of
// workgroups per XCD.
template <int MODE>
__device__ __forceinline__ int xcd_first_tile(const GemmArgs& p, const int* s_pref, int total_tiles, int x, int round) {
  if (MODE != GEMM_K_GROUPED || level_groups(p, s_pref)) {
    const int per_xcd = (total_tiles + 7) / 8;
    const int t = x * per_xcd;
    return t < total_tiles ? t : total_tiles;
  }
  if (x <= 0) return 0;
  if (x >= 8) return total_tiles;
  const int per_g = p.tiles_a * p.tiles_b;
  const int64_t pos = (int64_t)s_pref[p.G] * per_g * x / 8;
  int lo = 0, hi = p.G - 1;  // last g with s_pref[g] * per_g <= pos
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((int64_t)s_pref[mid] * per_g <= pos) lo = mid; else hi = mid - 1;
  }
  const int cost = s_pref[lo + 1] - s_pref[lo];
  int idx = (int)((pos - (int64_t)s_pref[lo] * per_g) / cost);
  if (idx > per_g) idx = per_g;
  // whole rounds of the XCD's workgroups: a cut a few tiles past a multiple of `round` would
  // leave most of them idle during one more round
  const int t = (lo * per_g + idx + (round >> 1)) / round * round;
  return t < total_tiles ? t : total_tiles;
}

// ---- k-grouped tiles of skewed groups -------------------------------------------------------------
// Tiles of groups of 64 blocks and of one stand in the same list, so a cut of the list by cost that rounds to whole
// rounds of workgroups, and dealing it out by count, leave workgroups idle where the largest tile is a good part of
// a workgroup's share.  There an XCD deals out its big tiles one by one, largest first, to the workgroup that has
// the least, and its workgroups take the small ones in turns, one that has less so far the earlier, as if each took
// the next tile when it is done.  What an XCD's tiles are has two forms:
//   eighths  every XCD takes an eighth of every group (neighbours in the group's order, the remainders of the eighths in
//            turn), so that all have the same to multiply, to store and to fetch from HBM; of groups with tiles enough for it
//   parts    the whole list is cut by cost, as without a schedule but anywhere: an operand is read by one XCD or two,
//            but one whose 32 workgroups get 33 big tiles of nearly a share each takes two rounds for them
// All of it is the same arithmetic in every workgroup (one wave).
static constexpr int kSchedGroups = 256;  // groups it is made for: four a lane
static constexpr int kNoLoad = 0x3fffffff;
struct KSchedule {  // in LDS
  int tiles[kSchedGroups + 1], cost[kSchedGroups + 1];  // of the small groups before g: tiles, and their cost
  int ahead[64];                                        // the XCD's workgroups: cost of their big tiles in small ones
  int big[128];                                         // this workgroup's big tiles: group * 2^22 + place in the group
  int n_big, first, n;                                  // how many; parts: the XCD's first small tile; how many tiles in all
};
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_min(int v) {
  const int o = __builtin_amdgcn_update_dpp(kNoLoad, v, CTRL, ROWS, 0xf, false);
  return o < v ? o : v;
}
__device__ __forceinline__ int wave_min(int v) {
  v = dpp_min<0x111, 0xf>(v); v = dpp_min<0x112, 0xf>(v); v = dpp_min<0x114, 0xf>(v); v = dpp_min<0x118, 0xf>(v);  // row_shr 1, 2, 4, 8
  v = dpp_min<0x142, 0xa>(v);  // row_bcast 15
  v = dpp_min<0x143, 0xc>(v);  // row_bcast 31
  return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ int wave_scan(int v, int lane) {  // sum up to this lane
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) { const int y = __shfl_up(v, d); if (lane >= d) v += y; }
  return v;
}
// eighths: an XCD's tiles of a group, from .. from + number
__device__ __forceinline__ void xcd_share(int per_g, int xcd, int g, int& from, int& number) {
  const int y = (xcd + g) & 7;
  from = per_g * y >> 3;
  number = (per_g * (y + 1) >> 3) - from;
}
// eighths of groups of per_g tiles, in the order of the groups: how many tiles an XCD has, and its tile j (of group h, its
// place there).  Eight groups' eighths are one of each, which together are per_g tiles from the XCD's own eighth on, around.
__device__ __forceinline__ int eighths_tiles(int per_g, int xcd, int groups) {
  const int from = per_g * xcd >> 3, last = xcd + (groups & 7);
  return (groups >> 3) * per_g + (last < 8 ? per_g * last >> 3 : per_g + (per_g * (last - 8) >> 3)) - from;
}
__device__ __forceinline__ void eighths_tile(int per_g, int xcd, int j, int& h, int& place) {
  const int round = j / per_g;
  place = j - round * per_g + (per_g * xcd >> 3);
  if (place >= per_g) place -= per_g;
  const int y = (8 * place + 7 + per_g) / per_g - 1;  // the first eighth that ends behind it
  h = 8 * round + ((y - xcd) & 7);
}
// Which form a launch takes (schedule_of_groups has the lines).  Limits: what the lists above can hold (a workgroup's big tiles are at
// most its share and one tile); sums that stay below 2^29, a workgroup's below 2^22.
__device__ __forceinline__ Schedule schedule_of(const GemmArgs& p, const int* s_pref, int workers) {
  const int64_t per_g = (int64_t)p.tiles_a * p.tiles_b, total = s_pref[p.G] * per_g, all_workers = 8 * workers;
  if (!p.offs || p.G > kSchedGroups || workers > 64 || per_g >= (1 << 22) || total >= (8ll << 22) * workers || total >= (1ll << 29)) return kInOrder;
  if (level_groups(p, s_pref)) return kInOrder;
  return schedule_of_groups(s_pref[p.G + 1], s_pref[p.G], per_g, all_workers);
}
// Place of workgroup `me`'s small tile j in the XCD's part of their list.  ahead: on lane w the big tiles of workgroup w
// in small ones; tiles are taken in the order of (ahead + count so far, workgroup).
__device__ __forceinline__ int small_place(int ahead, int me, int workers, int j) {
  const int time = __builtin_amdgcn_readlane(ahead, me) + j;
  int place = 0;
  for (int w = 0; w < workers; ++w) {
    const int before = time - __builtin_amdgcn_readlane(ahead, w) + (w < me);
    place += before > 0 ? before : 0;
  }
  return place;
}
// By the first wave; the caller waits for the workgroup.  `workers` workgroups an XCD, this one is `me`; parts: the XCD's
// part of the list is t_first .. t_last.
__device__ __forceinline__ void schedule_k_groups(const GemmArgs& p, const int* s_pref, KSchedule& s, bool parts, int xcd, int t_first, int t_last,
                                                  int me, int workers, int lane) {
  const int per_g = p.tiles_a * p.tiles_b;
  const int64_t total = (int64_t)s_pref[p.G] * per_g, all_workers = 8 * workers;
  const int least = (int)(total / (big_tile_parts(parts ? kParts : kEighths, total, all_workers) * all_workers)) + 1;  // cost of a big tile
  int cost[4];
  unsigned left = 0;  // the lane's groups of big tiles that have not been dealt out
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int g = 4 * lane + r;
    cost[r] = g < p.G ? s_pref[g + 1] - s_pref[g] : 0;
    if (cost[r] >= least) left |= 1u << r;
  }
  // ---- the others: their list, and this XCD's part of it ----
  int tiles = 0, sum = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (!(left >> r & 1) && cost[r]) { tiles += per_g; sum += per_g * cost[r]; }
  int tiles0 = wave_scan(tiles, lane), sum0 = wave_scan(sum, lane);
  const int all_tiles = __builtin_amdgcn_readlane(tiles0, 63), all = __builtin_amdgcn_readlane(sum0, 63);
  tiles0 -= tiles;
  sum0 -= sum;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    s.tiles[4 * lane + r] = tiles0;
    s.cost[4 * lane + r] = sum0;
    if (!(left >> r & 1) && cost[r]) { tiles0 += per_g; sum0 += per_g * cost[r]; }
  }
  if (lane == 0) { s.tiles[kSchedGroups] = all_tiles; s.cost[kSchedGroups] = all; }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's own writes
  int part, n_near = all_tiles, cost_near = all;  // the XCD's small tiles; those whose mean cost they have, and their cost
  if (parts) {
    // small tiles before a place of the list, and their cost, on lanes 0 and 1 for the two ends of the part
    const int end = (lane & 1) ? t_last : t_first, g = end / per_g < kSchedGroups ? end / per_g : kSchedGroups - 1;
    const int n = s.tiles[g + 1] - s.tiles[g], in_g = n ? end - g * per_g : 0;
    const int below = s.tiles[g] + in_g, spent = s.cost[g] + (n ? in_g * ((s.cost[g + 1] - s.cost[g]) / n) : 0);
    const int first = __builtin_amdgcn_readlane(below, 0);
    n_near = part = __builtin_amdgcn_readlane(below, 1) - first;
    cost_near = __builtin_amdgcn_readlane(spent, 1) - __builtin_amdgcn_readlane(spent, 0);
    if (lane == 0) s.first = first;
  } else {
    part = eighths_tiles(per_g, xcd, all_tiles / per_g);
  }
  // ---- the big ones ----
  int load = lane < workers ? 0 : kNoLoad, n_big = 0;
  while (__ballot(left != 0)) {
    int most = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (left >> r & 1) most = cost[r] > most ? cost[r] : most;
    const int c = -wave_min(-most);
    int mine = 0;  // the lane's first group of that cost
#pragma unroll
    for (int r = 3; r >= 0; --r)
      if ((left >> r & 1) && cost[r] == c) mine = r;
    const int owner = __builtin_ctzll(__ballot(most == c));
    if (lane == owner) left &= ~(1u << mine);
    const int g = 4 * owner + __builtin_amdgcn_readlane(mine, owner);
    int at, n;
    if (parts) {
      at = t_first - g * per_g > 0 ? t_first - g * per_g : 0;
      n = (t_last - g * per_g < per_g ? t_last - g * per_g : per_g) - at;
    } else {
      xcd_share(per_g, xcd, g, at, n);
    }
    while (n > 0) {
      // every workgroup that would still be ahead of another with one more takes one; if there are too few, those with the least
      const int low = wave_min(load);
      uint64_t takers = __ballot(load < low + c);
      if (__popcll(takers) > n) takers = __ballot(load == low);
      const int k = __popcll(takers), deal = k < n ? k : n;
      const int rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(takers >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)takers, 0));
      if ((takers >> lane & 1) && rank < deal) {
        if (lane == me) s.big[n_big] = g << 22 | (at + rank);
        ++n_big;
        load += c;
      }
      at += deal;
      n -= deal;
    }
  }
  const int ahead = n_near ? (int)((float)load * ((float)n_near / (float)cost_near) + 0.5f) : 0;
  s.ahead[lane] = ahead;
  n_big = __builtin_amdgcn_readlane(n_big, me);
  if (lane == 0) s.n_big = n_big;
  int n = n_big;
  for (int j = lane;; j += 64) {
    const int k = __popcll(__ballot(small_place(ahead, me, workers, j) < part));
    n += k;
    if (k < 64) break;
  }
  if (lane == 0) s.n = n;
}

// the workgroup's tile i, one on every lane of the first wave: its group and its place in it
__device__ __forceinline__ void scheduled_tile(const KSchedule& s, bool parts, int per_g, int xcd, int me, int workers, int lane, int i, int& g, int& idx) {
  const int j = small_place(s.ahead[lane], me, workers, i - s.n_big);
  if (i < s.n_big) {
    g = s.big[i] >> 22;
    idx = s.big[i] & ((1 << 22) - 1);
    return;
  }
  int t, place = 0;  // a tile of the small groups' list
  if (parts) {
    t = s.first + j;
  } else {
    eighths_tile(per_g, xcd, j, t, place);
    t *= per_g;
  }
  int lo = 0, hi = kSchedGroups - 1;  // last g with tiles[g] <= t
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (s.tiles[mid] <= t) lo = mid; else hi = mid - 1;
  }
  g = lo;
  idx = t - s.tiles[lo] + place;
}

// Geometry of logical tile t (k-grouped, with group >= 0: of that group's tile t); plain per-lane arithmetic (every lane
// may ask for a different one).
template <int MODE, int BM, int BN>
__device__ __forceinline__ void decode_tile(const GemmArgs& p, const int* s_pref, int t, Tile& T, int group = -1) {
  // The 32 CUs of an XCD work on 32 consecutive logical tiles at a time.  One side of the tile grid is cut into
  // strips of at most `width` tiles (of nearly equal width), and a strip is walked line by line along the other
  // side: 32 consecutive tiles then share 32 / w tiles of one operand and w of the other in that XCD's L2
  // instead of 32 and 1, whatever the two counts are.
  auto strips = [](int t, int n, int lines, int width, int& tn, int& tl) {  // t -> place tn of the n that are cut, line tl
    const int ns = (n + width - 1) / width;
    const int w0 = n / ns, wide = n - w0 * ns;  // the first `wide` strips have w0 + 1 tiles
    const int per_wide = lines * (w0 + 1);
    int s, r, w, n0;
    if (t < wide * per_wide) { s = t / per_wide; r = t - s * per_wide; w = w0 + 1; n0 = s * w; }
    else { const int t2 = t - wide * per_wide; s = t2 / (lines * w0); r = t2 - s * lines * w0; w = w0; n0 = wide * (w0 + 1) + s * w0; }
    tl = r / w;
    tn = n0 + r - tl * w;
  };
  // A group's tiles: the longer side is cut, so that the operand that is read once per strip is the smaller one, and
  // into strips of 3.  Against row tile by row tile down one column after the other, us: 32 groups of 2048 rows 5760 x
  // 2880 1103 -> 994, their input gradient 1015 -> 974, weight gradient 994 -> 949, 2880 x 2880 586 -> 531; 8 groups of
  // 8192 rows 1178 -> 930, 1251 -> 942, 994 -> 869, 1536 x 2048 193 -> 180; 128 groups of 512 rows level.  Strips
  // of 4 of the columns (windows of 32 tiles are then whole lines and move on all at once) give 1066, 1013 and 601 for the
  // first two and the 2880 x 2880, of 6 997, 989 and 545; the shorter side cut instead loses 2..10 % on 8192 rows.
  // Dense products, which do not change operands every few tiles, are level with 3 and with 8.
  auto group_strips = [&](int t, int na, int nb, int& ta, int& tb) {
    if (na > nb) strips(t, na, nb, 3, ta, tb);
    else strips(t, nb, na, 3, tb, ta);
  };
  if (MODE == GEMM_DENSE) {
    T.g = 0;
    int ta, tb;
    strips(t, p.tiles_b, p.tiles_a, 8, tb, ta);
    T.a_row0 = ta * BM; T.b_row0 = tb * BN;
    T.a_lim = (int)p.rows_a; T.b_lim = (int)p.rows_b; T.k_begin = 0; T.k_len = (int)p.red; T.kb0 = 0;
  } else if (MODE == GEMM_M_GROUPED) {
    const int q = t / p.tiles_b;
    int lo = 1, hi = p.G;  // first j in [1, G] with s_pref[j] > q
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (s_pref[mid] > q) hi = mid; else lo = mid + 1;
    }
    const int g = lo - 1;
    const int pg = s_pref[g], pg1 = s_pref[g + 1];
    const int gs = g ? p.offs[g - 1] : 0;
    const int m_tiles = pg1 - pg;
    const int idx = t - pg * p.tiles_b;
    T.g = g;
    int ta, tb;
    group_strips(idx, m_tiles, p.tiles_b, ta, tb);
    T.a_row0 = gs + ta * BM; T.b_row0 = tb * BN;
    T.a_lim = p.offs[g]; T.b_lim = (int)p.rows_b; T.k_begin = 0; T.k_len = (int)p.red; T.kb0 = 0;
  } else {
    const int per_g = p.tiles_a * p.tiles_b;
    const int g = group >= 0 ? group : t / per_g;
    const int idx = group >= 0 ? t : t % per_g;
    T.g = g;
    int ta, tb;
    if (p.offs) group_strips(idx, p.tiles_a, p.tiles_b, ta, tb);
    else strips(idx, p.tiles_b, p.tiles_a, 8, tb, ta);  // split-K of a dense product: the dense order inside every range
    T.a_row0 = ta * BM; T.b_row0 = tb * BN;
    T.a_lim = (int)p.rows_a; T.b_lim = (int)p.rows_b;
    T.k_begin = g ? k_group_end(p, g - 1) : 0; T.k_len = k_group_end(p, g) - T.k_begin; T.kb0 = T.k_begin >> 7;
  }
}

// Writes one wave's TM x TN blocks of 32 x 32 results of tile T (rows wm0.., columns wn0.. of the
// tile).  `piece`: the LDS addresses of the wave's four 1 KiB pieces of staging.
// PAIR: the result has two outputs (k-grouped: where the arguments say so).
// EXTRAS: the output rows (out_row_index) and the bias of the tile lie in LDS, row wm0 and column wn0 of
// the tile's at LDS bytes rows_lds + 4 wm0 and bias_lds + 2 wn0: a load here would wait for every store before it.
template <int MODE, int TM, int TN, bool ACC, bool PAIR = false, bool EXTRAS = false>
__device__ __forceinline__ void store_tile(const v16f (&acc)[TM][TN], const GemmArgs& p, const Tile& T, int wm0, int wn0, int lane,
                                           const uint32_t (&piece)[4], uint32_t rows_lds = 0, uint32_t bias_lds = 0) {
  const Staging stg = make_staging(piece, lane);
  const uint32_t esz = p.out_dtype == PT_F32 ? 4 : 2;
  const uint32_t pitch = (uint32_t)p.ldo * esz;
  const int whole = p.out_dtype == PT_F32 ? 3 : 7;  // elements of 16 bytes, less one
  const bool wide_ok = (p.ldo & whole) == 0 && (((uintptr_t)p.out) & 15) == 0 && (MODE != GEMM_K_GROUPED || (p.out_stride_g & whole) == 0) &&
                       (T.b_lim & whole) == 0;
  // The descriptor ends after the tile's last valid row: stores to ragged rows are dropped.
  // (PT_GEMM_ABLATE_STORES, measurement builds only: it ends before the first, so every store
  // instruction runs and nothing is written.)
  char* outp = (char*)p.out + (MODE == GEMM_K_GROUPED ? (int64_t)T.g * p.out_stride_g * esz : 0);
  int row0 = T.a_row0 + wm0, row_lim = T.a_lim;
  if (MODE == GEMM_K_GROUPED && PAIR && p.split_row) {  // a wave's rows lie on one side of the split
    if (row0 >= (int)p.split_row) {
      outp = (char*)p.out2 + (int64_t)T.g * p.out2_stride_g * esz;
      row0 -= (int)p.split_row; row_lim -= (int)p.split_row;
    } else {
      row_lim = row_lim < (int)p.split_row ? row_lim : (int)p.split_row;
    }
  }
  const __amdgpu_buffer_rsrc_t rs_out = __builtin_amdgcn_make_buffer_rsrc(outp, 0, kAblateStores ? 0 : (int)((uint32_t)row_lim * pitch), kRsrcFlags);
  const uint32_t s_tile = (uint32_t)row0 * pitch + (uint32_t)(T.b_row0 + wn0) * esz;
  static_assert(TN % 2 == 0, "the bf16 stores take column blocks in pairs");
  constexpr int AUX = kStoreAux<MODE>;
  // bias: the 8 values of the lane's columns, added in the output type after the result has been rounded to it
  // (x + bias[group] as a second operation on the rounded x)
  auto bias_of = [&](int j, int colc) -> v4i {
    if (MODE != GEMM_M_GROUPED || p.bias == nullptr || colc >= T.b_lim) return v4i{0, 0, 0, 0};
    if (EXTRAS) return PT_LDS(const v4i, bias_lds + (wn0 + j * 32 + (lane & 7) * 8) * 2);
    return *(const v4i*)((const char*)p.bias + ((int64_t)T.g * p.rows_b + colc) * 2);
  };
  if (MODE == GEMM_DENSE && p.head_a) {
    // Per-head halves in two tensors: a lane's eight columns lie in one of them (both widths are multiples
    // of 8), so its offset from `out` and its row pitch are all that differ.
    const __amdgpu_buffer_rsrc_t rs_heads = __builtin_amdgcn_make_buffer_rsrc(p.out, 0, kAblateStores ? 0 : (int)p.out_extent, kRsrcFlags);
    const int width = p.head_a + p.head_b, heads = (int)p.rows_b / width;
#pragma unroll
    for (int j = 0; j < TN; j += 2) {
      const int colc = T.b_row0 + wn0 + j * 32 + (lane & 7) * 8;
      const int h = colc / width, c = colc - h * width;
      const bool second = c >= p.head_a;
      const uint32_t at = second ? (uint32_t)((char*)p.out2 - (char*)p.out) + (uint32_t)(h * p.head_b + c - p.head_a) * 2 : (uint32_t)(h * p.head_a + c) * 2;
      const uint32_t pitch_h = (uint32_t)(heads * (second ? p.head_b : p.head_a)) * 2;
      stage_column<false>(acc, j, stg, lane, [&](int i, int q, v4i w) {
        const int r = row0 + i * 32 + q * 8 + (lane >> 3);
        store16<AUX>(w, rs_heads, colc < T.b_lim && r < row_lim ? (uint32_t)r * pitch_h + at : kOob, 0);
      });
    }
  } else if (MODE == GEMM_M_GROUPED && (PAIR || p.out_row_index)) {
    // Result row r goes to output row out_row_index[r] (the un-permute folded into the store);
    // rows of the group's padding map to a negative index and are dropped.
    const __amdgpu_buffer_rsrc_t rs_sc = __builtin_amdgcn_make_buffer_rsrc(p.out, 0, kAblateStores ? 0 : (int)((uint32_t)p.out_rows * pitch), kRsrcFlags);
    // one index per lane and block row (lane -> row lane % 32), handed to the lanes that store the row
    int dst[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int r = T.a_row0 + wm0 + i * 32 + (lane & 31);
      if (EXTRAS) dst[i] = PT_LDS(const int, rows_lds + (wm0 + i * 32 + (lane & 31)) * 4);
      else dst[i] = p.out_row_index[r < T.a_lim ? r : T.a_row0];
      if (r >= T.a_lim) dst[i] = -1;
    }
    if constexpr (PAIR) {
      // Two outputs, -2 - r for row r of the second: 64-bit addresses, since no descriptor spans both.  (Rows of an
      // input gradient that nobody else adds to go to their place at once, see pt_gather_rows_backward_begin.)
      if (kAblateStores) return;
#pragma unroll
      for (int j = 0; j < TN; j += 2) {
        const int colc = T.b_row0 + wn0 + j * 32 + (lane & 7) * 8;
        stage_column<false>(acc, j, stg, lane, [&](int i, int q, v4i w) {
          const int row = __shfl(dst[i], q * 8 + (lane >> 3));
          char* to = (char*)(row >= 0 ? p.out : p.out2) + (uint64_t)(uint32_t)(row >= 0 ? row : -2 - row) * pitch + (uint32_t)colc * 2;
          if (row != -1 && colc < T.b_lim) __builtin_nontemporal_store(w, (v4i*)to);
        });
      }
    } else {
#pragma unroll
      for (int j = 0; j < TN; j += 2) {
        const int colc = T.b_row0 + wn0 + j * 32 + (lane & 7) * 8;
        const v4i bias = bias_of(j, colc);
        stage_column<false>(acc, j, stg, lane, [&](int i, int q, v4i w) {
          const int row = __shfl(dst[i], q * 8 + (lane >> 3));
          store16<AUX>(p.bias ? add_bf16(w, bias) : w, rs_sc, row >= 0 && colc < T.b_lim ? (uint32_t)row * pitch + (uint32_t)(lane & 7) * 16 : kOob,
                       (uint32_t)(T.b_row0 + wn0 + j * 32) * 2);
        });
      }
    }
  } else if (p.out_dtype != PT_F32 && wide_ok) {
    const bool has_bias = MODE == GEMM_M_GROUPED && p.bias != nullptr;
#pragma unroll
    for (int j = 0; j < TN; j += 2) {
      const int colc = T.b_row0 + wn0 + j * 32 + (lane & 7) * 8;
      const v4i bias = bias_of(j, colc);
      const uint32_t v0 = (uint32_t)(lane >> 3) * pitch + (uint32_t)(lane & 7) * 16;
      stage_column<false>(acc, j, stg, lane, [&](int i, int q, v4i w) {
        const uint32_t soff = s_tile + i * 32 * pitch + j * 64;
        const uint32_t voff = colc < T.b_lim ? v0 + q * 8 * pitch : kOob;
        v4i x = has_bias ? add_bf16(w, bias) : w;
        // the result is rounded to bf16 first, then added: the two roundings of `grad += wgrad.to(bf16)`
        if (ACC) x = add_bf16(__builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rs_out, voff, soff, 0)), x);
        store16<AUX>(x, rs_out, voff, soff);
      });
    }
  } else if (wide_ok) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int colc = T.b_row0 + wn0 + j * 32 + (lane & 7) * 4;
      const uint32_t v0 = (uint32_t)(lane >> 3) * pitch + (uint32_t)(lane & 7) * 16;
      stage_column<true>(acc, j, stg, lane, [&](int i, int q, v4i w) {
        const uint32_t soff = s_tile + i * 32 * pitch + j * 128;
        const uint32_t voff = colc < T.b_lim ? v0 + q * 8 * pitch : kOob;
        v4i x = w;
        if (ACC) {
          const v4i old = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rs_out, voff, soff, 0));
#pragma unroll
          for (int k = 0; k < 4; ++k) x[k] = __float_as_int(__int_as_float(x[k]) + __int_as_float(old[k]));
        }
        store16<0>(x, rs_out, voff, soff);
      });
    }
  } else {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = T.b_row0 + wn0 + j * 32 + 4 * (lane >> 5);
      const uint32_t voff = (uint32_t)(lane & 31) * pitch + (uint32_t)(4 * (lane >> 5) + j * 32) * esz;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        if (p.out_dtype == PT_F32) store_elements<true>(acc[i][j], rs_out, voff, s_tile + i * 32 * pitch, T.b_lim - col, ACC);
        else store_elements<false>(acc[i][j], rs_out, voff, s_tile + i * 32 * pitch, T.b_lim - col, ACC);
      }
    }
  }
}

// One workgroup per CU (fewer when there are fewer tiles), in multiples of the 8 XCDs.  `upper` is
// an upper bound of the number of tiles.
template <class Kernel>
static int launch_persistent_grid(Kernel kernel, const char* name, const GemmArgs& a, int64_t upper, int threads, size_t lds,
                                  bool& attr_set, hipStream_t stream) {
  static int num_cus = 0;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) { set_error("gemm: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e)); return PT_ERR_LAUNCH; }
    attr_set = true;
  }
  if (num_cus == 0) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    num_cus = n;
  }
  if (upper == 0) return PT_OK;
  PT_REQUIRE(upper < (1ll << 30), "gemm: too many tiles");
  int64_t blocks = (num_cus + 7) / 8 * 8;
  if (upper < blocks) blocks = (upper + 7) / 8 * 8;
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(threads), lds, stream, a);
  return check_launch(name);
}

// Fills the tile counts of `a` for BM x BN tiles and returns an upper bound of the number of tiles
// (exact except in the m-grouped mode, where the kernel counts them from the group sizes).
static inline int64_t plan_tiles(GemmArgs& a, int BM, int BN) {
  a.tiles_a = (int)cdiv(a.rows_a, BM);
  a.tiles_b = (int)cdiv(a.rows_b, BN);
  if (a.mode == GEMM_DENSE) return a.total_tiles = (int64_t)a.tiles_a * a.tiles_b;
  if (a.mode == GEMM_K_GROUPED) return a.total_tiles = (int64_t)a.tiles_a * a.tiles_b * a.G;
  return ((a.rows_a / 128 + a.G) / 2 + 1) * a.tiles_b;
}

}  // namespace pt

// Persistent FP8 GEMM for gfx950, the kernel of every problem that fills the GPU with 256 x 256 tiles.
//
// The loads of a CU move at most ~70 GB/s out of L2: a 64 KiB stage of a 256 x 256 x 128 tile needs
// about as long to arrive as its MFMAs need to run, so the load path must never idle.  The two MFMA
// steps of a 128-block are therefore cut by rows instead of by reduction depth:
//
//   step X:  A blocks 0,1 (rows 0-63 of the wave's 128) x B blocks 0,1, both 64-deep halves
//   step Y:  A blocks 2,3 (rows 64-127)                 x B blocks 0,1, both halves
//
// and a ring slot is cut the same way: its half E holds the a rows of block rows 0,1 and one half
// of the b part (plus the block's scales), its half O the a rows of block rows 2,3 and the other
// half of the b part.  Inside a step the first 64-deep half comes before the second, which makes
// the a fragments short-lived: four 8-register buffers hold the step's two block rows x two
// halves, and each buffer takes a fragment of the next step as soon as the last MFMA on its old
// content has issued.  With the four b fragments of the block that is 64 fragment registers.  E of block g
// has been read completely when X(g) ends, O(g) when Y(g) ends; either step refills the half it
// finds free with block g + 2's data, 32 KiB per step, requested two steps before the barrier
// behind which it is first read.  One workgroup barrier per step.
//
// What bounds the loop on real (not zero) operands is the power limit: MFMAs alone reach 3.8 PFLOP/s at the
// clock it leaves, with the 192 KiB a block reads from LDS 3.15; this loop runs 8192 x 8192 x 8192 at 2.8
// (392 us; 290 us = 3.8 PFLOP/s with zero operands, where the clock does not fall).  Behind a barrier both waves
// of a SIMD want to issue MFMAs at once, so whatever a wave does there first is time in which the matrix pipe
// idles: the loader's state moves on between the MFMAs of step X, a wave's own waits and its barrier come at the
// end of a step, the addresses of the LDS reads are registers that toggle between the two slots, and what a
// tile needs only once (arguments of the result stores, output rows, bias) is fetched when it is needed instead
// of being kept in spilled scalar registers.  Against the same loop with some 200 scalar instructions between a
// barrier and the first MFMA, us: 8192 x 8192 x 8192 463 -> 392, 32768 x 4096 x 2048 278 -> 217; 128 groups of
// 512 rows 1536 x 2048 297 -> 244, weight gradients of those groups 309 -> 248; 32 groups of 2048 rows 5760 x
// 2880 1175 -> 1141 and their weight gradients 1207 -> 1003.  The loops this kernel replaced for dense products
// and long weight gradients (one barrier per block, all fragments of a 64-deep half in registers): 415, 230
// and 1136 on the same box.
#include "gemm_persistent_parts.h"
#include <type_traits>

// Measurement builds only (never defined by the Makefile's default target): parts of the main loop
// compiled out to see what the rest costs.  PT_GEMM_ABLATE_MFMA: no MFMAs, fragment reads or result
// stores (every wave takes the path of one without rows).  PT_GEMM_ABLATE_LOADS: 1 = every operand and scale
// load is issued out of range (the instruction runs, nothing is fetched), 2 = not issued at all.
// The results of such builds are garbage; only their timing means something.
#ifndef PT_GEMM_ABLATE_MFMA
#define PT_GEMM_ABLATE_MFMA 0
#endif
#ifndef PT_GEMM_ABLATE_LOADS
#define PT_GEMM_ABLATE_LOADS 0
#endif

namespace pt {

// LDS of a workgroup, all of it dynamic, so that the ring starts at byte 0 and a slot is bit 16 of an address:
// two operand stages, two stages of scales, the tile table, the group scan of the work list, the scatter
// indices and the bias of the current tile.  (The waves stage their results in the ring itself.)
static constexpr int kRsStage = 512 * 128;
static constexpr int kRsScales = 2 * kRsStage;
static constexpr int kRsTable = kRsScales + 2 * 512 * 4;
static constexpr int kRsTiles = 48, kRsEntry = 48;
static constexpr int kRsPref = kRsTable + kRsTiles * kRsEntry;
static constexpr int kRsIndex = kRsPref + ((kMaxGroupsGemm + 2) * 4 + 15) / 16 * 16;
static constexpr int kRsBias = kRsIndex + 256 * 4;
static constexpr int kRsSched = kRsBias + 256 * 2;
static constexpr int kRsLds = kRsSched + sizeof(KSchedule);
static_assert(kRsLds <= 160 * 1024 && kRsPref % 16 == 0, "LDS map");

// BT: the b operand is given reduction-major, [red][rows_b] with row pitch ldb (the forward layout of
// a weight, read by its input-gradient GEMM), instead of [rows_b][red].
// PAIR: two outputs (k-grouped: the result rows from split_row on go to the second; m-grouped: out_row_index says which).
// A kernel of its own, so that every other launch keeps its code without a further form of the store.
// TRIM (m-grouped): groups end at their last used row; a kernel of its own likewise (its code took other launches 0.2 to 0.3 us: 8 groups of 256
// rows 256 x 512 11.8 -> 11.5, 16 of 282 1536 x 1024 18.3 -> 18.0).
template <int MODE, int BM, int BN, int WGM, int WGN, bool ACC, bool BT = false, bool PAIR = false, bool TRIM = false>
__global__ __launch_bounds__(WGM * WGN * 64, 1) void fp8_gemm_nt_rowsplit_kernel(GemmArgs) {
  constexpr int NW = WGM * WGN;
  constexpr int WM = BM / WGM, WN = BN / WGN;
  constexpr int TM = WM / 32, TN = WN / 32;
  constexpr int BK = 128;                      // reduction depth of one stage = one scale block = two MFMA steps
  constexpr int STAGE = (BM + BN) * BK;
  static_assert(BM == 256 && BN == 256 && WGM == 2 && WGN == 4 && STAGE == kRsStage, "the row split is written for 8 waves of 128 x 64");
  constexpr int NX = 4, NY = 5;  // loads a wave issues per step: two 1 KiB loads of a rows and two of b rows; with E one of scales
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave / WGN) * WM, wn0 = (wave % WGN) * WN;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  int* const s_pref = (int*)(lds + kRsPref);

  // ---- tile list ----
  const GemmArgs p = reload_args();
  int total_tiles;
  if (MODE == GEMM_M_GROUPED) {
    scan_group_tiles<BM>(p, s_pref, tid, lane);
    total_tiles = __builtin_amdgcn_readfirstlane(s_pref[p.G]) * p.tiles_b;
  } else {
    total_tiles = (int)p.total_tiles;
    if (MODE == GEMM_K_GROUPED) scan_group_costs(p, s_pref, tid, lane);
  }
  const int xcd = blockIdx.x & 7;
  // lanes 0 and 1 find the two ends of this XCD's share of the list side by side
  int t_step = gridDim.x >> 3;
  const Schedule scheduled = MODE == GEMM_K_GROUPED ? schedule_of(p, s_pref, t_step) : kInOrder;
  const int t_cut = xcd_first_tile<MODE>(p, s_pref, total_tiles, xcd + (lane & 1), scheduled ? 1 : t_step);
  int t_end = __builtin_amdgcn_readlane(t_cut, 1);
  int t_next = __builtin_amdgcn_readlane(t_cut, 0) + (blockIdx.x >> 3);
  KSchedule& sched = *(KSchedule*)(lds + kRsSched);
  if (scheduled) {
    if (tid < 64) schedule_k_groups(p, s_pref, sched, scheduled == kParts, xcd, __builtin_amdgcn_readlane(t_cut, 0), t_end, blockIdx.x >> 3, t_step, lane);
    __syncthreads();
    t_next = 0;
    t_end = __builtin_amdgcn_readfirstlane(sched.n);
    t_step = 1;
  }

  // ---- LDS addressing ----
  // A stage holds rows of 128 bytes (8 chunks of 16).  Row r keeps logical chunk c at position
  // c ^ fs(r), fs(r) = (r&7) ^ ((r>>3)&1), which spreads the ds_read_b128 of 8 or 16 consecutive
  // rows over all banks.  Direct-to-LDS wave-load q covers rows 8q..8q+7 (1 KiB, eight full
  // 128-byte lines): lane -> row 8q + lane/8, position lane%8, i.e. logical chunk
  // (lane%8) ^ (lane/8) ^ (q&1).  A wave's loads q = w, w+NW, ... all have the parity of w, so one
  // per-lane offset serves them all and the rest of the address is uniform (scalar offset).
  const int chunk16 = ((lane & 7) ^ (lane >> 3) ^ (wave & 1)) * 16;
  const uint32_t va = (uint32_t)(lane >> 3) * (uint32_t)p.lda + chunk16;
  const int fs_rd = (lane & 7) ^ ((lane >> 3) & 1);
  // per-lane LDS addresses of the fragment reads, in the ring slot that is read next: [MFMA half][chunk of it]
  uint32_t rd_a[2][2], rd_b[2][2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int c = (lane & 31) * 128 + (((ks * 4 + (lane >> 5) * 2 + h) ^ fs_rd) << 4);
      rd_a[ks][h] = lds_base + wm0 * BK + c;
      rd_b[ks][h] = lds_base + (BM + wn0) * BK + c;
    }

  // Reduction-major b operand: its part of a stage holds 128 reduction rows of 256 bytes (the
  // tile's 256 b rows), logical 16-byte chunk c of row k at position c ^ 2 (k & 7): the eight rows
  // that one transposing read touches put a chunk at eight different positions, and the chunks
  // c and c + 1 (c even) of the two halves of a 32-row b block never share one, so such a read
  // spreads over all banks.  A direct-to-LDS
  // wave-load covers four such rows (lane -> row lane / 16, position lane % 16); a wave's loads are
  // row quads Q = w, w + 8, ... of a half, so (k & 7) = 4 (w & 1) + lane / 16 for all of them.
  // Fragments come out of it through the transposing LDS read: in every group of 16 lanes, source
  // lane s supplies the address of 8 bytes and lane l receives byte (l & 7) of source lanes
  // (l >> 3), 2 + (l >> 3), ..., 14 + (l >> 3).  With source lane s pointing at reduction row
  // s / 2 and b rows 8 (s & 1) .. + 7 of the group's 16, lane l gets 8 consecutive reduction
  // elements of b row l % 16: four such reads are the lane's 32 bytes of an MFMA operand.
  if constexpr (BT) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {  // per b block j, for reduction rows 0-7
      const int s16 = lane & 15, g16 = lane >> 4;
      const int c = (wn0 >> 4) + 2 * j + (g16 & 1);
      rd_b[0][j] = lds_base + BM * BK + (uint32_t)((32 * (g16 >> 1) + (s16 >> 1)) * 256 + ((c ^ (2 * (s16 >> 1))) << 4) + 8 * (s16 & 1));
    }
  }
  const int bt_chunk = (lane & 15) ^ (2 * (4 * (wave & 1) + (lane >> 4)));
  const uint32_t vb = BT ? (uint32_t)(lane >> 4) * (uint32_t)p.ldb + bt_chunk * 16 : (uint32_t)(lane >> 3) * (uint32_t)p.ldb + chunk16;
  uint32_t rd_sa = lds_base + kRsScales + (wm0 + (lane & 31)) * 4, rd_sb = lds_base + kRsScales + (BM + wn0 + (lane & 31)) * 4;

  // ---- loader: walks (tile, 128-block, half) triples ahead of the MFMAs ----
  // Half E of a block: a rows 128r + 0..63 and b rows 64c + 0..31 (the A0,A1 and B0 fragments of
  // every wave) plus the block's scales; half O: the other rows.  Reduction-major b: reduction rows
  // 0..63 with E, 64..127 with O.  All of the state is uniform but the three per-lane offsets; it moves on
  // during step X (advance), between MFMAs, so that behind a barrier nothing comes before the next MFMA.
  const uint32_t lda = (uint32_t)p.lda, ldb = (uint32_t)p.ldb;
  // rows of this wave's first load of a half: a 8 wave, b 64 (wave / 4) + 8 (wave % 4) (reduction-major: 4 wave)
  const uint32_t wave_a = (uint32_t)(8 * wave) * lda;
  const uint32_t wave_b = BT ? (uint32_t)(4 * wave) * ldb : (uint32_t)(64 * (wave >> 2) + 8 * (wave & 3)) * ldb;
  const uint32_t a64 = 64 * lda, a128 = 128 * lda;                      // to the O half, to the wave's second load
  const uint32_t b_o = BT ? 64 * ldb : 32 * ldb, b_2 = BT ? 32 * ldb : 128 * ldb;
  const uint32_t b_step = BT ? 128 * ldb : 128;                         // to the next block
  // LDS places of those loads inside a slot
  const uint32_t to_a = lds_base + wave * 1024, to_b = lds_base + BM * BK + (BT ? wave : 8 * (wave >> 2) + (wave & 3)) * 1024;
  constexpr int kToAO = 8 * 1024, kToA2 = 16 * 1024, kToBO = (BT ? 16 : 4) * 1024, kToB2 = (BT ? 8 : 16) * 1024;
  // scales: waves 0-3 load those of 64 a rows each, waves 4-7 those of 64 b rows
  const bool sc_a = wave < 4;
  const int sc_shift = sc_a ? p.sa_shift : p.sb_shift;
  const uint32_t sc_rs = (uint32_t)(sc_a ? p.sa_rs : p.sb_rs) * 4, sc_ks = (uint32_t)(sc_a ? p.sa_ks : p.sb_ks) * 4;
  const uint32_t to_s = lds_base + kRsScales + wave * 256;

  v4i rs_a = make_rsrc(p.a, 0), rs_b = make_rsrc(p.b, (uint32_t)p.b_bytes);
  v4i rs_s = sc_a ? make_rsrc(p.sa, (uint32_t)p.sa_bytes) : make_rsrc(p.sb, (uint32_t)p.sb_bytes);
  int n_tiles = 0, l_n = 0, l_rem = 0;  // tiles in the table, the loader's next one, what is left of its reduction from the current block on
  uint32_t l_slot = STAGE, l_soA = 0, l_soB = 0, l_soS = 0;
  uint32_t l_va = kOob, l_vb = kOob, l_vs = kOob, vs = 0;

  auto advance = [&]() {
    l_slot ^= STAGE;
    l_rem -= BK;
    l_soA += BK; l_soB += b_step; l_soS += sc_ks;
    while (l_rem <= 0) {
      // past the end of the list the loads still run (the counted waits rely on them), out of range
      if (l_n >= n_tiles) { l_rem = 0; break; }
      const int* e = (const int*)(lds + kRsTable + l_n * kRsEntry);
      ++l_n;
      const int4 e0 = *(const int4*)e, e1 = *(const int4*)(e + 4);
      l_rem = __builtin_amdgcn_readfirstlane(e0.w);
      l_soA = (uint32_t)__builtin_amdgcn_readfirstlane(e0.x) + wave_a;
      l_soB = (uint32_t)__builtin_amdgcn_readfirstlane(e0.y) + wave_b;
      l_soS = 0;
      rs_a[2] = __builtin_amdgcn_readfirstlane(e0.z);  // ends behind the tile's last row: rows past a ragged group's end are not fetched
      const int row = sc_a ? __builtin_amdgcn_readfirstlane(e1.z) + 64 * wave : __builtin_amdgcn_readfirstlane(e1.w) + 64 * (wave - 4);
      vs = (uint32_t)((row + lane) >> sc_shift) * sc_rs + (uint32_t)__builtin_amdgcn_readfirstlane(e1.x) * sc_ks;
      if (MODE == GEMM_M_GROUPED) {
        const GemmArgs p = reload_args();
        const int64_t g = __builtin_amdgcn_readfirstlane(e1.y);
        rs_b = make_rsrc(p.b + g * p.b_stride_g, (uint32_t)p.b_bytes);
        if (!sc_a) rs_s = make_rsrc(p.sb + g * p.sb_stride_g, (uint32_t)p.sb_bytes);
      }
    }
    // chunks past the end of a ragged reduction are not fetched.  Reduction-major b: such rows lie past the end
    // of the group's matrix, whose extent is the descriptor's: the hardware returns zeros for them (its range
    // check includes the scalar offset).
    l_va = chunk16 < l_rem ? va : kOob;
    l_vb = (BT ? 0 : chunk16) < l_rem ? vb : kOob;
    l_vs = 0 < l_rem ? vs : kOob;
  };
  // load k of the E half (0 <= k < NY) and of the O half (0 <= k < NX)
  auto issue_e = [&](int k) {
    if (PT_GEMM_ABLATE_LOADS == 2) return;
    const bool off = PT_GEMM_ABLATE_LOADS == 1;
    if (k == 0) dma16_at<0, 0>(rs_a, off ? kOob : l_va, l_soA, to_a + l_slot);
    if (k == 1) dma16_at<0, kToA2>(rs_a, off ? kOob : l_va, l_soA + a128, to_a + l_slot);
    if (k == 2) dma16_at<1, 0>(rs_b, off ? kOob : l_vb, l_soB, to_b + l_slot);
    if (k == 3) dma16_at<1, kToB2>(rs_b, off ? kOob : l_vb, l_soB + b_2, to_b + l_slot);
    if (k == 4) dma4(rs_s, off ? kOob : l_vs, l_soS, to_s + (l_slot >> 5));  // 2 KiB of scales a slot
  };
  auto issue_o = [&](int k) {
    if (PT_GEMM_ABLATE_LOADS == 2) return;
    const bool off = PT_GEMM_ABLATE_LOADS == 1;
    if (k == 0) dma16_at<0, kToAO>(rs_a, off ? kOob : l_va, l_soA + a64, to_a + l_slot);
    if (k == 1) dma16_at<0, kToAO + kToA2>(rs_a, off ? kOob : l_va, l_soA + a64 + a128, to_a + l_slot);
    if (k == 2) dma16_at<1, kToBO>(rs_b, off ? kOob : l_vb, l_soB + b_o, to_b + l_slot);
    if (k == 3) dma16_at<1, kToBO + kToB2>(rs_b, off ? kOob : l_vb, l_soB + b_o + b_2, to_b + l_slot);
  };

  // one 32-row block of fragments, 64 deep, from the slot that the read addresses point at
  auto at = [&](uint32_t addr) { return *(const v4i __attribute__((address_space(3)))*)(uintptr_t)addr; };
  auto read_a = [&](int i, int ks) -> v8i {
    const v4i lo = at(rd_a[ks][0] + i * (32 * BK)), hi = at(rd_a[ks][1] + i * (32 * BK));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  // The b fragments are kept as fb[late][early]: the half of the b part of a slot that is read
  // during step X of its block ("late") against the one read ahead during step Y of the block
  // before.  Row-major b: late = b block j (rows 64c + 32..63), early = 64-deep half.
  // Reduction-major b: late = the 64-deep half (reduction rows 64..127), early = b block j.
  auto read_b = [&](int late, int early) -> v8i {
    if constexpr (BT) {
      typedef int v2i_t __attribute__((ext_vector_type(2)));
      v8i r;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const v2i_t t = __builtin_amdgcn_ds_read_tr8_b64_v2i32((v2i_t __attribute__((address_space(3)))*)(uintptr_t)(rd_b[0][early] + late * (64 * 256) + q * (8 * 256)));
        r[2 * q] = t[0];
        r[2 * q + 1] = t[1];
      }
      return r;
    } else {
      const v4i lo = at(rd_b[early][0] + late * (32 * BK)), hi = at(rd_b[early][1] + late * (32 * BK));
      return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  };
  auto next_slot = [&]() {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int h = 0; h < 2; ++h) { rd_a[ks][h] ^= STAGE; if (!BT || ks == 0) rd_b[ks][h] ^= STAGE; }
    rd_sa ^= STAGE >> 5; rd_sb ^= STAGE >> 5;
  };
  // The E8M0 exponent bytes of a block's scales, packed one byte per 32-row block: the MFMA picks
  // its byte with the opsel immediates, so a whole block costs two registers.
  auto read_scales = [&](int& pa, int& pb) {
    uint32_t a = 0, b = 0;
#pragma unroll
    for (int i = 0; i < TM; ++i) a |= ((*(const uint32_t __attribute__((address_space(3)))*)(uintptr_t)(rd_sa + i * 128) >> 23) & 0xFFu) << (8 * i);
#pragma unroll
    for (int j = 0; j < TN; ++j) b |= ((*(const uint32_t __attribute__((address_space(3)))*)(uintptr_t)(rd_sb + j * 128) >> 23) & 0xFFu) << (8 * j);
    pa = (int)a; pb = (int)b;
  };

  // Fragments.  A: four buffers; the step in progress owns all four (two block rows x two 64-deep
  // halves) and hands each to the next step's fragment as soon as its last MFMA has issued.  B:
  // fb[late][early], both block columns and both halves of the current 128-block.
  v8i fa[4], fb[2][2];
  int sca = 0, scb = 0, sca_n = 0, scb_n = 0;

  // ---- the work list in pieces of kRsTiles tiles: as many lanes decode one each into the table, from which
  // the two cursors (loader, MFMAs) fetch a tile with a few LDS reads; nothing in flight between two pieces ----
  for (bool first_piece = true; t_next < t_end; first_piece = false, t_next += kRsTiles * t_step) {
    const GemmArgs p = reload_args();
    if (!first_piece) {  // the scan of the groups and the schedule have their own LDS and are still there
      wait_all_vmem();
      __syncthreads();
    }
    n_tiles = (t_end - t_next + t_step - 1) / t_step;
    if (n_tiles > kRsTiles) n_tiles = kRsTiles;
    int t = t_next + tid * t_step, group = -1;
    if (scheduled && tid < 64) scheduled_tile(sched, scheduled == kParts, p.tiles_a * p.tiles_b, xcd, blockIdx.x >> 3, gridDim.x >> 3, lane, t, group, t);
    if (tid < n_tiles) {
      Tile T;
      decode_tile<MODE, BM, BN>(p, s_pref, t, T, group);
      const int64_t a_end = (int64_t)T.a_lim * p.lda < p.a_bytes ? (int64_t)T.a_lim * p.lda : p.a_bytes;
      const uint32_t soA = (uint32_t)T.a_row0 * lda + T.k_begin;
      const uint32_t soB = BT ? (uint32_t)T.k_begin * ldb + (uint32_t)T.b_row0 : (uint32_t)T.b_row0 * ldb + T.k_begin;
      int4* e = (int4*)(lds + kRsTable + tid * kRsEntry);
      e[0] = make_int4((int)soA, (int)soB, (int)a_end, T.k_len);
      e[1] = make_int4(T.kb0, T.g, T.a_row0, T.b_row0);
      e[2] = make_int4(T.a_lim, T.b_lim, 0, 0);
    }
    __syncthreads();
    if constexpr (TRIM) {
      // A group ends at its last used row (eight): what is behind it in its last block is neither loaded nor stored.  The
      // waves share the tiles out, the loads of all of them in one latency.  Layers that leave padding out, us a pass without /
      // with this and its like in the quantisers: 128 groups of 512 rows 2048 x 768 1872 / 1860 (0.4 to 0.8 % in other runs), of 128 rows 1160 / 1138; 64
      // skewed groups of 2048 x 1408 with shared experts 3000 / 2987.  It takes a launch 1 to 2 us, which 16 and 32 groups
      // do not bring in (257 / 262, 532 / 537; 64 of 540 rows 1550 / 1550).
      int row[kRsTiles / NW][2], lim[kRsTiles / NW];
#pragma unroll
      for (int k = 0; k < kRsTiles / NW; ++k) {
        const int n = wave + NW * k;
        lim[k] = *(const int*)(lds + kRsTable + (n < n_tiles ? n : 0) * kRsEntry + 32);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int r = lim[k] - 128 + 64 * h + lane;
          row[k][h] = r >= 0 ? p.row_used[r] : -1;
        }
      }
#pragma unroll
      for (int k = 0; k < kRsTiles / NW; ++k) {
        const int n = wave + NW * k;
        int end = lim[k] - 128;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint64_t m = __ballot(PAIR ? row[k][h] != -1 : row[k][h] >= 0);
          if (m) end = lim[k] - 128 + 64 * h + (71 - __builtin_clzll(m)) / 8 * 8;
        }
        if (lane == 0 && n < n_tiles) {
          int* e = (int*)(lds + kRsTable + n * kRsEntry);
          e[2] = (int)((int64_t)end * p.lda < p.a_bytes ? (int64_t)end * p.lda : p.a_bytes);
          e[8] = end;
        }
      }
      __syncthreads();
    }

    // E0, O0, E1 on their way; the first block complete
    // (a piece starts in the slot that the reads point at: both sides toggle once a block)
    l_n = 0; l_rem = 0;
    advance();
#pragma unroll
    for (int k = 0; k < NY; ++k) issue_e(k);
#pragma unroll
    for (int k = 0; k < NX; ++k) issue_o(k);
    advance();
#pragma unroll
    for (int k = 0; k < NY; ++k) issue_e(k);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NY) : "memory");
    __syncthreads();
    read_scales(sca, scb);
    fa[0] = read_a(0, 0);
    fa[1] = read_a(1, 0);
    fb[0][0] = read_b(0, 0);
    fb[0][1] = read_b(0, 1);

#pragma unroll 1
    for (int n = 0; n < n_tiles; ++n) {
      Tile C;
      {
        const int* e = (const int*)(lds + kRsTable + n * kRsEntry);
        const int4 e1 = *(const int4*)(e + 4), e2 = *(const int4*)(e + 8);
        C.k_len = __builtin_amdgcn_readfirstlane(e[3]);
        C.g = __builtin_amdgcn_readfirstlane(e1.y);
        C.a_row0 = __builtin_amdgcn_readfirstlane(e1.z);
        C.b_row0 = __builtin_amdgcn_readfirstlane(e1.w);
        C.a_lim = __builtin_amdgcn_readfirstlane(e2.x);
        C.b_lim = __builtin_amdgcn_readfirstlane(e2.y);
        C.k_begin = 0; C.kb0 = 0;
      }
      const int nk = (C.k_len + 127) >> 7;
      // Waves whose whole row range lies past the end of a ragged group skip the MFMAs, which leaves
      // the matrix pipe to the other wave of their SIMD, and have nothing to store; they still take
      // part in the loads, the fragment reads and the barriers.
      const bool wave_active = C.a_row0 + wm0 < C.a_lim && !PT_GEMM_ABLATE_MFMA;

      v16f acc[TM][TN];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
#pragma unroll 1
      for (int it = 0; it < nk; ++it) {
        // Slot m of a step: MFMA (block row i, block column j, half ks), the first 64-deep half
        // before the second:
        //   m:   0        1        2        3        4        5        6        7
        //   X: (0,0,0)  (1,0,0)  (0,1,0)  (1,1,0)  (0,0,1)  (1,0,1)  (0,1,1)  (1,1,1)
        //   Y: (2,0,0)  (3,0,0)  (2,1,0)  (3,1,0)  (2,0,1)  (3,0,1)  (2,1,1)  (3,1,1)
        // The same accumulator comes back four slots later.  A fragment (i, ks) of the step lives in
        // fa[2 ks + (i & 1)] and is used in slots 4 ks + (i & 1) and 4 ks + 2 + (i & 1): the first
        // half's buffers are free from slot 4 on and take the next step's first-half fragments; the
        // second half's are free when the step ends and take the next step's second-half fragments in
        // its first slots.  B fragments fb[late][early] (row-major b: late = block column, early =
        // half; reduction-major b: the other way round): the "early" part of a block's slot is read
        // during step Y of the block before (fb[0][.], each after its last MFMA), the "late" part in
        // step X (fb[1][.]), every one in the order of its first use.
        // The two halves of a ring slot: E = a rows of block rows 0,1 + the early b part (+ scales),
        // O = a rows of block rows 2,3 + the late b part.  E of block g has been read when X(g) ends
        // and is refilled during Y(g) with block g + 2; O(g) has been read when Y(g) ends and is
        // refilled during X(g + 1).  Every refill is requested two steps before the barrier behind
        // which it is first read, so a step waits until only the previous step's loads are outstanding.
        // ---- step X ----
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          const int i = m & 1, j = (m >> 1) & 1, ks = m >> 2;
          const int late = BT ? ks : j, early = BT ? j : ks;
          if (wave_active) {
            mfma_sel(fb[late][early], fa[2 * ks + i], acc[i][j], j, scb, i, sca);
          }
          if (m < NX) issue_o(m);
          if (m == 0) { if (BT) fa[2] = read_a(0, 1); else fb[1][0] = read_b(1, 0); }
          if (m == 1) { if (BT) fb[1][0] = read_b(1, 0); else fa[2] = read_a(0, 1); }
          if (m == 2) fa[3] = read_a(1, 1);
          if (m == 3) fb[1][1] = read_b(1, 1);
          if (m == 4) fa[0] = read_a(2, 0);
          if (m == 5) fa[1] = read_a(3, 0);
          if (m == 6) advance();
          __builtin_amdgcn_sched_barrier(0);
        }
        // ---- step Y ----
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NX) : "memory");
        __builtin_amdgcn_s_barrier();
        if (MODE == GEMM_M_GROUPED && it == 0) {
          const GemmArgs p = reload_args();
          // what the result stores of this tile need, in LDS by then: the output row of each of its rows and its
          // bias (loaded where they are needed, each would wait for all stores before it, and for the operands in flight)
          if (p.out_row_index && wave < 4)
            dma4(make_rsrc(p.out_row_index, (uint32_t)(p.rows_a * 4)), lane * 4, (uint32_t)(C.a_row0 + 64 * wave) * 4, lds_base + kRsIndex + wave * 256);
          if (p.bias && wave >= 4 && wave < 6)
            dma4(make_rsrc((const uint16_t*)p.bias + (int64_t)C.g * p.rows_b, (uint32_t)p.rows_b * 2), lane * 4, (uint32_t)(C.b_row0 + 128 * (wave - 4)) * 2,
                 lds_base + kRsBias + (wave - 4) * 256);
        }
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          const int i = m & 1, j = (m >> 1) & 1, ks = m >> 2;
          const int late = BT ? ks : j, early = BT ? j : ks;
          if (wave_active) {
            mfma_sel(fb[late][early], fa[2 * ks + i], acc[2 + i][j], j, scb, 2 + i, sca);
          }
          if (m < NY) issue_e(m);
          if (m == 0) fa[2] = read_a(2, 1);
          if (m == 1) { fa[3] = read_a(3, 1); next_slot(); }
          if (m == 2) read_scales(sca_n, scb_n);
          if (m == 3) fb[0][0] = read_b(0, 0);
          if (m == 4) { fa[0] = read_a(0, 0); if (BT) fb[0][1] = read_b(0, 1); }
          if (m == 5) fa[1] = read_a(1, 0);
          if (m == 6 && !BT) fb[0][1] = read_b(0, 1);
          __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NY) : "memory");
        __builtin_amdgcn_s_barrier();
        sca = sca_n; scb = scb_n;
      }
      // the compiler does not see the MFMAs inside the assembly statements: cover the result latency
      // of the last one before the epilogue reads the accumulators
      static_assert(TM == 4 && TN == 2, "all accumulators are operands");
      asm volatile("s_nop 15\n\ts_nop 15"
                   : "+v"(acc[0][0]), "+v"(acc[0][1]), "+v"(acc[1][0]), "+v"(acc[1][1]), "+v"(acc[2][0]), "+v"(acc[2][1]), "+v"(acc[3][0]), "+v"(acc[3][1])
                   :
                   : "memory");

      // ---- epilogue ----
      if (!wave_active) continue;
      if (MODE == GEMM_K_GROUPED && nk == 0 && ACC) continue;
      // a copy of the lane number that the compiler cannot trace: addresses derived from it are worked out here,
      // not kept (or spilled, and reloaded behind a wait for every store so far) across the main loop
      int el = lane;
      asm volatile("" : "+v"(el));
      // staging: the part of the ring that this wave itself refills next (the O half that its step Y has just
      // released), with loads that it issues behind these stores
      const uint32_t piece[4] = {to_a + l_slot + kToAO, to_a + l_slot + kToAO + kToA2, to_b + l_slot + kToBO, to_b + l_slot + kToBO + kToB2};
      store_tile<MODE, TM, TN, ACC, PAIR, true>(acc, reload_args(), C, wm0, wn0, el, piece,
                                                   lds_base + kRsIndex, lds_base + kRsBias);
    }
  }
  wait_all_vmem();  // nothing may still be writing into this workgroup's LDS when it retires
}

template <int MODE, int BM, int BN, int WGM, int WGN, bool ACC, bool BT = false, bool PAIR = false, bool TRIM = false>
static int launch_one(GemmArgs a, hipStream_t stream) {
  constexpr size_t lds = kRsLds;
  static bool attr_set = false;
  const int64_t upper = plan_tiles(a, BM, BN);
  return launch_persistent_grid(fp8_gemm_nt_rowsplit_kernel<MODE, BM, BN, WGM, WGN, ACC, BT, PAIR, TRIM>, "fp8_gemm_nt_rowsplit_kernel", a, upper, WGM * WGN * 64, lds, attr_set, stream);
}

template <int BM, int BN, int WGM, int WGN, bool TRIM>
static int launch_m_grouped(const GemmArgs& a, hipStream_t stream) {
  if (a.out2)
    return a.b_kmajor ? launch_one<GEMM_M_GROUPED, BM, BN, WGM, WGN, false, true, true, TRIM>(a, stream)
                      : launch_one<GEMM_M_GROUPED, BM, BN, WGM, WGN, false, false, true, TRIM>(a, stream);
  return a.b_kmajor ? launch_one<GEMM_M_GROUPED, BM, BN, WGM, WGN, false, true, false, TRIM>(a, stream)
                    : launch_one<GEMM_M_GROUPED, BM, BN, WGM, WGN, false, false, false, TRIM>(a, stream);
}

template <int BM, int BN, int WGM, int WGN>
static int launch_mode(const GemmArgs& a, hipStream_t stream) {
  switch (a.mode) {
    case GEMM_DENSE: return launch_one<GEMM_DENSE, BM, BN, WGM, WGN, false>(a, stream);
    case GEMM_M_GROUPED:
      return a.row_used && a.G >= kPaddedGroups ? launch_m_grouped<BM, BN, WGM, WGN, true>(a, stream) : launch_m_grouped<BM, BN, WGM, WGN, false>(a, stream);
    default:
      if (a.split_row)
        return a.accumulate ? launch_one<GEMM_K_GROUPED, BM, BN, WGM, WGN, true, false, true>(a, stream)
                            : launch_one<GEMM_K_GROUPED, BM, BN, WGM, WGN, false, false, true>(a, stream);
      return a.accumulate ? launch_one<GEMM_K_GROUPED, BM, BN, WGM, WGN, true>(a, stream)
                          : launch_one<GEMM_K_GROUPED, BM, BN, WGM, WGN, false>(a, stream);
  }
}

int launch_gemm_rowsplit(const GemmArgs& a, hipStream_t stream) {
  PT_REQUIRE(a.mode == GEMM_DENSE || a.G <= kMaxGroupsGemm, "gemm: at most %d groups", kMaxGroupsGemm);
  PT_REQUIRE(!a.b_kmajor || a.mode == GEMM_M_GROUPED, "gemm: a reduction-major b operand is built for the m-grouped mode only");
  return launch_mode<256, 256, 2, 4>(a, stream);  // 8 waves, 128 x 64 per wave
}

}  // namespace pt

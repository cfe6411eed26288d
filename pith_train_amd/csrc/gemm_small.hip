// FP8 GEMM for problems that do not fill the GPU with 256 x 256 tiles (gfx950).
//
// A layer with few tokens has a handful of large tiles: most compute units stay idle, and the ones
// that work spend their time waiting for one operand stage after the other.  Here a workgroup of
// four waves owns one BM x 128 tile (BM = 64 or 128) with a ring of two or three 128-deep stages, small
// enough that a compute unit holds two workgroups: while one waits for its first stage, drains its
// pipeline or stores its result, the other multiplies.
// DEEP: where there is one 128-row tile per unit and a long reduction, nobody else fills a workgroup's waits.  There
// eight waves own the tile, two a SIMD, with a ring of four stages (three in flight instead of one): us with two
// stages and four waves / four and four / four and eight, 1001 x 4096 x 2048 20.1 / 16.3 / 15.5, 2048 x 2048 x 4096
// 28.9 / 26.1 / 23.9, 2048 x 2048 x 2816 21.1 / 18.1 / 17.2; 2048 x 1536 x 1024 9.0 / 9.6 / 9.4.  With two tiles per unit
// the two workgroups are the better way (2048 x 4096 x 2048 21.0, deep 29.1).
// There is no persistent loop, no tile table and no scan over the groups (a tile finds its group with
// one ballot over the group ends), which keeps the time before the first load and the code that has to
// be fetched short.  Operand traffic bounds it from the L2 on (tiles x reduction x (BM + 128) bytes): 4096 x 2048 x
// 2048 268 MB in 19.3 us, 4096 x 512 x 4096 201 MB in 18.5, 4096 x 4096 x 512 134 MB in 15.1: 9 to 14 TB/s.
//
// Operand layouts in LDS, direct-to-LDS loads, scale handling and result stores are those of the
// persistent kernel (gemm_rowsplit.hip, gemm_persistent_parts.h); the MFMAs run in the same order, so the results have
// the same bits.
#include "gemm_persistent_parts.h"

namespace pt {

// LDS of a workgroup: the ring of stages, their scales, a sink for scale loads that nobody needs
// (65.3 or 74.5 KiB: two workgroups share a compute unit)
template <int BM> static constexpr int kSmallStages = BM == 64 ? 3 : 2;
static constexpr int kDeepStages = 4;
static constexpr size_t kDeepLds = (size_t)kDeepStages * (128 + 128) * (128 + 4) + 256;
template <int BM> static constexpr size_t kSmallLds = (size_t)kSmallStages<BM> * (BM + 128) * (128 + 4) + 256;

// STREAM: the loads of b pass the memory-side cache by (launch_small_mode has the rule and both sides).  TWO (m-grouped): two outputs.
template <int MODE, int BM, bool ACC, bool BT, bool STREAM = false, bool DEEP = false, bool TWO = false>
__device__ __forceinline__ void small_tile_body(const GemmArgs& p, int block) {
  constexpr int BN = 128, BK = 128, NS = DEEP ? kDeepStages : kSmallStages<BM>, NW = DEEP ? 8 : 4;
  static_assert(DEEP ? BM == 128 && kDeepLds <= 160 * 1024 : 2 * kSmallLds<BM> <= 160 * 1024, "one deep workgroup or two others per compute unit");
  constexpr int TM = BM / (16 * NW), TN = 2;   // waves NW / 2 x 2, each TM x 2 blocks of 32 x 32
  constexpr int STAGE = (BM + BN) * BK;
  constexpr int LA = BM / (8 * NW), LB = BN / (8 * NW);  // 1 KiB loads of a and of b per wave and stage
  constexpr int NP = LA + LB + 1;            // and one of scales
  constexpr int kWait = (NS - 2) * NP;       // loads of the stages after the one a step needs
  static_assert(kWait < 64, "vmcnt is a 6-bit counter");
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];  // [NS][STAGE] | [NS][BM + BN] scales | 256 B sink; the stores' staging takes the first 16 KiB afterwards

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave >> 1) * (32 * TM), wn0 = (wave & 1) * 64;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  const uint32_t sc_base = lds_base + NS * STAGE;

  // ---- which tile: an XCD takes an eighth of the list (its tiles share operand panels in that L2).
  // The m-grouped row count is known on the device only; workgroups past the real list end here. ----
  const int total = MODE == GEMM_M_GROUPED ? p.offs[p.G - 1] / BM * p.tiles_b : (int)p.total_tiles;
  const int per_xcd = (total + 7) >> 3;
  const int idx = block >> 3;
  const int t = (block & 7) * per_xcd + idx;
  if (idx >= per_xcd || t >= total) return;
  Tile T;
  if (MODE == GEMM_M_GROUPED) {
    // Row tile t / tiles_b names the group; inside a group the row tiles of one b panel come first, so
    // that they run together and the panel comes from HBM once.
    const int row = t / p.tiles_b * BM;
    int g = 0;  // groups that end at or before that row; groups are whole tiles
    for (int g0 = 0; g0 < p.G; g0 += 64) {
      const int q = g0 + lane;
      g += __popcll(__ballot(q < p.G && p.offs[q < p.G ? q : 0] <= row));
    }
    T.g = __builtin_amdgcn_readfirstlane(g);
    const int first = __builtin_amdgcn_readfirstlane(T.g ? p.offs[T.g - 1] : 0);
    const int rows_g = (__builtin_amdgcn_readfirstlane(p.offs[T.g]) - first) / BM;
    const int i = t - first / BM * p.tiles_b, col = i / rows_g;
    T.a_row0 = first + (i - col * rows_g) * BM;
    T.b_row0 = col * BN;
    T.a_lim = T.a_row0 + BM; T.b_lim = (int)p.rows_b;
    T.k_begin = 0; T.k_len = (int)p.red; T.kb0 = 0;
  } else {
    const int per_g = p.tiles_a * p.tiles_b;
    const int g = t / per_g, r = t - g * per_g;
    const int ta = r / p.tiles_b;
    T.g = g;
    T.a_row0 = ta * BM; T.b_row0 = (r - ta * p.tiles_b) * BN;
    T.a_lim = (int)p.rows_a; T.b_lim = (int)p.rows_b;
    T.k_begin = 0; T.k_len = (int)p.red; T.kb0 = 0;
    if (MODE == GEMM_K_GROUPED) {
      T.k_begin = __builtin_amdgcn_readfirstlane(g ? k_group_end(p, g - 1) : 0);
      T.k_len = __builtin_amdgcn_readfirstlane(k_group_end(p, g)) - T.k_begin;
      T.kb0 = T.k_begin >> 7;
    }
  }
  const int nk = (T.k_len + 127) >> 7;
  if constexpr (MODE == GEMM_M_GROUPED) {
    // Groups of a few rows end in tiles that are padding for the most part (333 tokens of 8 in 128 experts: 21 of 64 rows):
    // eights of rows behind the last used one are neither loaded nor stored.  Stores between the weights' reads cost 0.7 us a
    // MB: a block of them, gate_up and down 178 -> 158 us a pass; 100 tokens of 4 in 32 experts 2880 x 2880 247 -> 217.
    if (p.row_used) {
      int row[BM / 64];
#pragma unroll
      for (int h = 0; h < BM / 64; ++h) row[h] = p.row_used[T.a_row0 + 64 * h + lane];
      int used = 0;
#pragma unroll
      for (int h = 0; h < BM / 64; ++h) {
        const uint64_t m = __ballot(TWO ? row[h] != -1 : row[h] >= 0);
        if (m) used = 64 * h + (71 - __builtin_clzll(m)) / 8 * 8;
      }
      if (!used) return;
      T.a_lim = T.a_row0 + used;
    }
  }

  // ---- loads (layout and swizzle as in gemm_rowsplit.hip) ----
  const int chunk = (lane & 7) ^ (lane >> 3) ^ (wave & 1);
  const uint32_t va = (uint32_t)(lane >> 3) * (uint32_t)p.lda + chunk * 16;
  // Row-major b as a.  Reduction-major b: a stage holds 128 reduction rows of 128 bytes, logical
  // 16-byte chunk c of row k at position c ^ 2 ((k >> 1) & 3): the eight rows a transposing read
  // touches lie two to a 256-byte bank line, and the four row pairs put a chunk at four positions.
  const int bt_chunk = (lane & 7) ^ (2 * ((lane >> 4) & 3));
  const uint32_t vb = (uint32_t)(lane >> 3) * (uint32_t)p.ldb + (BT ? bt_chunk : chunk) * 16;
  const v4i rs_a = make_rsrc(p.a, (uint32_t)p.a_bytes);
  const v4i rs_b = make_rsrc(p.b + (MODE == GEMM_M_GROUPED ? (int64_t)T.g * p.b_stride_g : 0), (uint32_t)p.b_bytes);
  const v4i rs_sa = make_rsrc(p.sa, (uint32_t)p.sa_bytes);
  const v4i rs_sb = make_rsrc(p.sb + (MODE == GEMM_M_GROUPED ? (int64_t)T.g * p.sb_stride_g : 0), (uint32_t)p.sb_bytes);
  constexpr int SLA = BM / 64;  // scale loads of a (the next two are b's, the fourth of BM = 64 goes to the sink)
  const bool sc_a = wave < SLA, sc_real = wave < SLA + 2;
  uint32_t vs;
  if (sc_a) vs = (uint32_t)(((int64_t)((T.a_row0 + 64 * wave + lane) >> p.sa_shift) * p.sa_rs + (int64_t)T.kb0 * p.sa_ks) * 4);
  else      vs = (uint32_t)(((int64_t)((T.b_row0 + 64 * (wave - SLA) + lane) >> p.sb_shift) * p.sb_rs + (int64_t)T.kb0 * p.sb_ks) * 4);
  const int a_rows = T.a_lim - T.a_row0;
  const uint32_t soA0 = (uint32_t)T.a_row0 * (uint32_t)p.lda + T.k_begin;
  const uint32_t soB0 = BT ? (uint32_t)T.b_row0 : (uint32_t)T.b_row0 * (uint32_t)p.ldb + T.k_begin;
  const bool bt_in = T.b_row0 + bt_chunk * 16 < T.b_lim;

  auto issue_stage = [&](int it) {
    // past the end of the reduction the same loads run out of range, so that every step counts alike
    const int slot = it % NS;
    const uint32_t sA = lds_base + slot * STAGE, sB = sA + BM * BK;
    const bool ok = it < nk;
    const uint32_t koff = (uint32_t)it * BK;
    const bool in = ok && (int)(koff + chunk * 16) < T.k_len;
#pragma unroll
    for (int k = 0; k < LA; ++k) {
      const int q = NW * k + wave;
      dma16(rs_a, in && 8 * q < a_rows ? va : kOob, soA0 + koff + (uint32_t)(8 * q) * (uint32_t)p.lda, sA + q * 1024);
    }
#pragma unroll
    for (int k = 0; k < LB; ++k) {
      const int q = NW * k + wave;
      if constexpr (BT) dma16<STREAM>(rs_b, ok && bt_in ? vb : kOob, soB0 + (koff + 8 * q) * (uint32_t)p.ldb, sB + q * 1024);
      else              dma16<STREAM>(rs_b, in ? vb : kOob, soB0 + koff + (uint32_t)(8 * q) * (uint32_t)p.ldb, sB + q * 1024);
    }
    const uint32_t dst = sc_real ? sc_base + slot * (BM + BN) * 4 + wave * 256 : sc_base + NS * (BM + BN) * 4;
    if (sc_a) dma4(rs_sa, ok ? vs : kOob, (uint32_t)(it * p.sa_ks * 4), dst);
    else      dma4(rs_sb, ok && sc_real ? vs : kOob, (uint32_t)(it * p.sb_ks * 4), dst);
  };

  // ---- fragment reads ----
  const int fs_rd = (lane & 7) ^ ((lane >> 3) & 1);
  int coff[2][2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int h = 0; h < 2; ++h) coff[ks][h] = (lane & 31) * 128 + (((ks * 4 + (lane >> 5) * 2 + h) ^ fs_rd) << 4);
  auto read_frag = [&](const uint8_t* base, int ks) -> v8i {
    const uint4 lo = *(const uint4*)(base + coff[ks][0]);
    const uint4 hi = *(const uint4*)(base + coff[ks][1]);
    return v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
  };
  uint32_t bt_rd[2];  // the lane's byte offset for b block j, reduction rows 0-7 of a 64-deep half
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int s16 = lane & 15, g16 = lane >> 4, k = s16 >> 1;
    const int c = (wn0 >> 4) + 2 * j + (g16 & 1);
    bt_rd[j] = (uint32_t)((32 * (g16 >> 1) + k) * 128 + ((c ^ (2 * ((k >> 1) & 3))) << 4) + 8 * (s16 & 1));
  }
  auto read_b = [&](const uint8_t* sB, int j, int ks) -> v8i {
    if constexpr (BT) {
      typedef int v2i_t __attribute__((ext_vector_type(2)));
      v8i r;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const v2i_t w = __builtin_amdgcn_ds_read_tr8_b64_v2i32((v2i_t __attribute__((address_space(3)))*)(sB + bt_rd[j] + ks * (64 * 128) + q * 8 * 128));
        r[2 * q] = w[0];
        r[2 * q + 1] = w[1];
      }
      return r;
    } else {
      return read_frag(sB + (wn0 + 32 * j) * BK, ks);
    }
  };

  v16f acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

#pragma unroll 1
  for (int s = 0; s < NS - 1; ++s) issue_stage(s);
#pragma unroll 1
  for (int it = 0; it < nk; ++it) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kWait) : "memory");
    __syncthreads();  // stage `it` is complete, and every wave has read the stage whose slot is refilled next
    const uint8_t* sA = lds + (it % NS) * STAGE;
    const uint8_t* sB = sA + BM * BK;
    const float* sc = (const float*)(lds + NS * STAGE) + (it % NS) * (BM + BN);
    uint32_t sca[TM], scb[TN];
    v8i fa[2][TM], fb[2][TN];
    auto read_scales = [&]() {
#pragma unroll
      for (int i = 0; i < TM; ++i) sca[i] = __float_as_uint(sc[wm0 + 32 * i + (lane & 31)]);
#pragma unroll
      for (int j = 0; j < TN; ++j) scb[j] = __float_as_uint(sc[BM + wn0 + 32 * j + (lane & 31)]);
    };
    auto read = [&](int ks) {
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[ks][j] = read_b(sB, j, ks);
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[ks][i] = read_frag(sA + (wm0 + 32 * i) * BK, ks);
    };
    auto multiply = [&](int ks) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fb[ks][j], fa[ks][i], acc[i][j], 0, 0, 0, (int)(scb[j] >> 23), 0, (int)(sca[i] >> 23));
    };
    // Dense products run few steps a workgroup from operands that lie in the L2, so a step is as long as its chain
    // of barrier, reads and MFMAs: the reads go ahead of the next stage's loads, which have two steps to arrive (the
    // gradients of an MLA block's latent projection as a pair, 2048 rows, 512 to 1024 wide: 12.9 -> 12.1 us; its
    // forward product 6.5 -> 6.3).  Weights that come from HBM want their loads out first (few-row groups 74.7 us,
    // 75.2 with the reads ahead; reduction-major 64 x 60 rows of 2048 x 2816: 90.0, 92.9).
    if constexpr (MODE == GEMM_DENSE) {
      read_scales();
      read(0);
      read(1);
      __builtin_amdgcn_sched_barrier(0);
      issue_stage(it + NS - 1);
      multiply(0);
      multiply(1);
    } else {
      issue_stage(it + NS - 1);
      read_scales();
      read(0);
      multiply(0);
      read(1);
      multiply(1);
    }
  }
  wait_all_vmem();  // nothing may still be writing into this workgroup's LDS when it retires
  if (MODE == GEMM_K_GROUPED && nk == 0 && ACC) return;
  __syncthreads();  // every wave has read its last stage and has nothing in flight: the ring's memory is free
  const uint32_t stg = lds_base + wave * 4096, piece[4] = {stg, stg + 1024, stg + 2048, stg + 3072};
  store_tile<MODE, TM, TN, ACC, MODE == GEMM_K_GROUPED || TWO>(acc, p, T, wm0, wn0, lane, piece);
}

template <int MODE, int BM, bool ACC, bool BT, bool STREAM, bool TWO>
__global__ __launch_bounds__(256, 2) void fp8_gemm_small_kernel(GemmArgs p) {
  small_tile_body<MODE, BM, ACC, BT, STREAM, false, TWO>(p, blockIdx.x);
}

__global__ __launch_bounds__(512, 2) void fp8_gemm_deep_kernel(GemmArgs p) {
  small_tile_body<GEMM_DENSE, 128, false, false, false, true>(p, blockIdx.x);
}

// Two products that do not depend on each other (the input and the weight gradient of a dense linear): the
// workgroups past `second` (a multiple of 8) take the second one's tiles, so that compute units which
// either would leave with one workgroup or none hold two.
struct GemmPair { GemmArgs g[2]; int second; };
template <int BM, bool DEEP>
__global__ __launch_bounds__(DEEP ? 512 : 256, 2) void fp8_gemm_small_pair_kernel(GemmPair q) {
  const bool late = (int)blockIdx.x >= q.second;
  small_tile_body<GEMM_DENSE, BM, false, false, false, DEEP>(late ? q.g[1] : q.g[0], (int)blockIdx.x - (late ? q.second : 0));
}

template <int MODE, int BM>
static void count_small_tiles(GemmArgs& a) {
  a.tiles_a = (int)cdiv(a.rows_a, BM);
  a.tiles_b = (int)cdiv(a.rows_b, 128);
  a.total_tiles = (int64_t)a.tiles_a * a.tiles_b * (MODE == GEMM_K_GROUPED ? a.G : 1);
}

template <class Kernel>
static int reserve_lds(Kernel kernel, size_t lds, bool& done) {
  if (done) return PT_OK;
  hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) { set_error("gemm: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e)); return PT_ERR_LAUNCH; }
  done = true;
  return PT_OK;
}

template <int BM, bool DEEP = false>
static int launch_pair(const GemmArgs& a, const GemmArgs& b, hipStream_t stream) {
  constexpr size_t lds = DEEP ? kDeepLds : kSmallLds<BM>;
  static bool reserved = false;
  auto kernel = fp8_gemm_small_pair_kernel<BM, DEEP>;
  if (int rc = reserve_lds(kernel, lds, reserved)) return rc;
  GemmPair q = {{a, b}, 0};
  count_small_tiles<GEMM_DENSE, BM>(q.g[0]);
  count_small_tiles<GEMM_DENSE, BM>(q.g[1]);
  q.second = (int)(cdiv(q.g[0].total_tiles, 8) * 8);
  hipLaunchKernelGGL(kernel, dim3((unsigned)(q.second + cdiv(q.g[1].total_tiles, 8) * 8)), dim3(DEEP ? 512 : 256), lds, stream, q);
  return check_launch("fp8_gemm_small_pair_kernel");
}

int launch_gemm_small_pair(const GemmArgs& a, const GemmArgs& b, int rows, hipStream_t stream) {
  PT_REQUIRE(rows == 64 || rows == 128 || rows == kDeepTile, "gemm: the small-problem kernel has tiles of 64 or 128 rows");
  return rows == 64 ? launch_pair<64>(a, b, stream) : rows == 128 ? launch_pair<128>(a, b, stream) : launch_pair<128, true>(a, b, stream);
}

static int launch_deep(GemmArgs a, hipStream_t stream) {
  static bool reserved = false;
  if (int rc = reserve_lds(fp8_gemm_deep_kernel, kDeepLds, reserved)) return rc;
  count_small_tiles<GEMM_DENSE, 128>(a);
  if (a.total_tiles == 0) return PT_OK;
  hipLaunchKernelGGL(fp8_gemm_deep_kernel, dim3((unsigned)(cdiv(a.total_tiles, 8) * 8)), dim3(512), kDeepLds, stream, a);
  return check_launch("fp8_gemm_deep_kernel");
}

template <int MODE, int BM, bool ACC, bool BT, bool STREAM = false, bool TWO = false>
static int launch_small(GemmArgs a, hipStream_t stream) {
  constexpr size_t lds = kSmallLds<BM>;
  static bool reserved = false;
  auto kernel = fp8_gemm_small_kernel<MODE, BM, ACC, BT, STREAM, TWO>;
  if (int rc = reserve_lds(kernel, lds, reserved)) return rc;
  count_small_tiles<MODE, BM>(a);
  if (a.total_tiles == 0) return PT_OK;
  PT_REQUIRE(a.total_tiles < (1ll << 28), "gemm: too many tiles");
  hipLaunchKernelGGL(kernel, dim3((unsigned)(cdiv(a.total_tiles, 8) * 8)), dim3(256), lds, stream, a);
  return check_launch("fp8_gemm_small_kernel");
}

template <int BM>
static int launch_small_mode(const GemmArgs& a, hipStream_t stream) {
  switch (a.mode) {
    case GEMM_DENSE: return launch_small<GEMM_DENSE, BM, false, false>(a, stream);
    case GEMM_M_GROUPED:
      // Groups of one or two tiles of rows read their weights once or, from the L2, twice.  Past the memory-side cache (256 MiB) they arrive faster, whatever
      // their size, when the weights of other layers are read before they are wanted again, as in a model (1536 x 2048 an
      // expert, us through the cache / past it: 96 MiB 25.7 / 23.8, 129 MiB 36.9 / 33.8, 192 40.9 / 37.9, 384 80.1 / 74.8).
      // A block that runs alone finds what is left of its own last pass, while its two operands fit together (gate_up and
      // a down of half its size in turn, us a product: 129 MiB of gate_up 22.6 / 25.2, 162 26.0 / 28.4, 192 31.8 / 29.9, 258
      // 48.5 / 45.0), and a single product repeated (162 MiB 29.8 / 33.8, 225 39.5 / 46.2, 321 71.6 / 65.8).  A launch
      // sees one operand and not what comes between: from half of the cache on it is taken for the first case, below for
      // the others, so a block alone loses a tenth between 128 and 170 MiB and a model 5 to 8 % below 128.  A row that is
      // no whole 128-byte lines shares one with the next (32 experts of 5760 x 2880: 127 us, 132 past the cache).
      // Training steps, whose weights are read again only after the other layers', through / past, us a pass: 128 experts of
      // 2048 x 768, 16 rows each 903 / 856, 64 964 / 914; 64 of 2048 x 1408, 16 rows 798 / 760; 128 of 2048 x 512, 64 rows 704 /
      // 649; with single operators 128 of 2048 x 768, 48 rows 1217 / 1195.
      if (streams_weights(a)) {
        if (a.out2)
          return a.b_kmajor ? launch_small<GEMM_M_GROUPED, BM, false, true, true, true>(a, stream)
                            : launch_small<GEMM_M_GROUPED, BM, false, false, true, true>(a, stream);
        return a.b_kmajor ? launch_small<GEMM_M_GROUPED, BM, false, true, true>(a, stream)
                          : launch_small<GEMM_M_GROUPED, BM, false, false, true>(a, stream);
      }
      if (a.out2)
        return a.b_kmajor ? launch_small<GEMM_M_GROUPED, BM, false, true, false, true>(a, stream)
                          : launch_small<GEMM_M_GROUPED, BM, false, false, false, true>(a, stream);
      return a.b_kmajor ? launch_small<GEMM_M_GROUPED, BM, false, true>(a, stream)
                        : launch_small<GEMM_M_GROUPED, BM, false, false>(a, stream);
    default:
      return a.accumulate ? launch_small<GEMM_K_GROUPED, BM, true, false>(a, stream)
                          : launch_small<GEMM_K_GROUPED, BM, false, false>(a, stream);
  }
}

int launch_gemm_small(const GemmArgs& a, int rows, hipStream_t stream) {
  if (rows == kDeepTile) {
    if (a.mode == GEMM_DENSE) return launch_deep(a, stream);
    rows = 128;
  }
  PT_REQUIRE(rows == 64 || rows == 128, "gemm: the small-problem kernel has tiles of 64 or 128 rows");
  return rows == 64 ? launch_small_mode<64>(a, stream) : launch_small_mode<128>(a, stream);
}

}  // namespace pt

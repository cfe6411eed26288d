// Lines that a GEMM's dispatch draws by sizes alone: plain arithmetic, the same on the host and on the device.
#pragma once
#include <cstdint>

namespace pt {

enum { GEMM_DENSE = 0, GEMM_M_GROUPED = 1, GEMM_K_GROUPED = 2 };
constexpr int64_t up_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ---- m-grouped: rows that count, whatever the padded rows that hold them (a capacity, or the sizes that a routing has) ---------
// Few enough for 128-row tiles that end at their last used row, in place of large ones.  Layers in training, us a pass in large tiles / in these, with
// buffers as large as the routing could need: 128 experts of 2048 x 768, 100 rows each 1007 / 982, 108 1050 / 1026, 116 1093 / 1075, 124 1118 / 1142, 128 1140 /
// 1170; with exact sizes 116 1078 / 1064, 124 1118 / 1153, 128 1150 / 1190; 128 of 2048 x 512, 116 807 / 802, 124 831 / 842; 64 of 2048 x 1408, 116 931 /
// 932, 124 957 / 946
constexpr bool few_used_rows(int64_t rows, int64_t groups) { return rows <= 120 * groups; }

// Weights that the small-problem kernel loads past the memory-side cache (launch_small_mode has the reasons for their size): those of
// groups of 64 rows, and in tiles of 128 rows up to one and a half of them a group (rows_a, or where that is a capacity half a tile more than the
// rows that count).  Weights that are read again come from that cache; operands from HBM, us through / past it for 1, 2, 3 and 5 row tiles: 8 x 4096 x
// 4096 45 / 43, 62 / 60, 85 / 101, 121 / 139; 32 x 2048 x 2048 38 / 34, 60 / 60, 78 / 82, 118 / 128; reduction-major 43 / 37, 63 / 63, 77 / 81,
// 118 / 130; 128 x 1536 x 2048 97 / 95, 166 / 170, 213 / 240, 320 / 360
template <class Args>
constexpr bool streams_weights(const Args& a) {
  const int64_t groups = a.G, counted = a.used_rows + 64 * groups, rows = a.row_used && counted < a.rows_a ? counted : a.rows_a;
  return a.b_stride_g * groups >= (128ll << 20) && a.ldb % 128 == 0 && (a.few_rows || rows <= 192 * groups);
}

// ---- large or small tiles (Args: GemmArgs) -------------------------------------------------------------------------------------
// Small: 64 or 128 rows x 128 columns, two workgroups per compute unit; kDeepTile: 128 rows, one workgroup (dense products)
constexpr int kDeepTile = 129;

// Problems too small for 256 x 256 tiles to fill 256 compute units evenly go to the kernel with one 64 x 128
// or 128 x 128 tile per workgroup and two workgroups per compute unit (gemm_small.hip): tile rows, or 0
// when the persistent kernel is the better choice.  While all 64-row tiles run at once the smaller tile
// wins (1001 x 512 x 2048: 10.7 us against 12.9 with 128 rows and 21.5 for the large one).  While the 128-row tiles do,
// dense ones with a long reduction take the form with one workgroup per unit (us, two per unit / one: 1001 x 4096 x 1536 14.7 / 13.1,
// 1792 17.3 / 14.0, 2880 27.7 / 20.8; 2048 x 2048 x 1536 11.5 / 11.5, 1792 13.3 / 12.8, 2048 16.4 / 14.0; 4096 x 1024 x 1792 12.1 /
// 12.5, 2048 13.3 / 13.4, 2880 24.1 / 19.0).  Then both
// kinds are priced in rounds of the GPU: a round of 256 large tiles is the unit, a round of 512 small ones
// (a quarter of the area each, half of it in all) costs 0.72 of it in the m-grouped mode, 0.68 in
// the dense one (0.45 up to a reduction of 512, most of it filling and draining), 0.36 for a weight gradient
// over groups of up to 1024 rows (mostly stores, which one workgroup of a unit does while the other loads), 0.65
// over longer ones (16 Zipf-distributed groups of 7600 rows 768 x 2048 and 1536 x 2048: whole step 2540 us, 2623 at
// 0.56).  A partly filled round of small tiles costs half of what it leaves idle.  Fitted to 270
// shapes timed with both kernels, where the choice now loses 0.9 % to the better one in the mean (m-grouped), 0.2 %
// (weight gradients) and nothing (dense).  Us, large / small: m-grouped, K 2048, N 1536: 16 groups of 256 rows
// 25.4 / 19.7, of 512 30.5 / 34.9, of 640 50.1 / 37.4, of 1024 53.0 / 62.8; 64 groups of 128 49.6 / 52.7, of 384
// 89 / 108; reduction-major b, K 1536, N 2048: 16 groups of 256 24.5 / 25.2, of 640 42.2 / 41.2.  Dense
// 4096 x 2048 x 2048 26 / 20, 4096 x 4096 x 512 15.0 / 13.6.  Weight gradients 1536 x 2048 of 8 groups of 512
// rows 26.6 / 23.4, of 1024 35.1 / 32.7; of 16 groups of 512 37.8 / 40.9.  Past two rounds large tiles have
// no round to waste and need half of the operand traffic.
template <class Args>
constexpr int small_tile_rows(const Args& g) {
  const int64_t groups = g.mode == GEMM_K_GROUPED ? g.G : 1;
  const int64_t cols = up_div(g.rows_b, 128) * groups, cols_large = up_div(g.rows_b, 256) * groups;
  if (up_div(g.rows_a, 64) * cols <= 256) return 64;
  // Where padding is known and left out, 128-row tiles, which end at their last used row, up to few_used_rows.  Layers of 128 experts
  // 2048 x 768, us a pass in large tiles / these: 16 rows each 943 / 903, 48 974 / 942, 96 1029 / 1008; in tiles of 64 rows, of which every
  // second finds nothing, 969 at 16.
  if (g.row_used && few_used_rows(g.used_rows, g.G)) return 128;
  // Weights that come from HBM and are read once, mostly: single operators on 128 groups of 48 rows 2048 x 768 1191 / 1182, of 96
  // 1222 / 1209.
  if (g.mode == GEMM_M_GROUPED && streams_weights(g) && g.rows_a <= 140 * (int64_t)g.G) return 128;
  int64_t small = up_div(g.rows_a, 128) * cols;
  if (small <= 256 && g.mode == GEMM_DENSE && g.red >= 1792) return kDeepTile;
  if (small <= 512) return 128;
  int64_t rows_large = up_div(g.rows_a, 256);
  if (g.mode == GEMM_M_GROUPED) {
    // Half of the groups end in half a large tile.  The row count may be a capacity, which exceeds the real
    // one by half a block per group in the mean, or exact: half of that is taken off.
    const int64_t blocks = g.rows_a / 128, least = blocks < g.G ? blocks : g.G;
    rows_large = (blocks + g.G / 2) / 2;
    if (rows_large < least) rows_large = least;
    const int64_t fewer = blocks - g.G / 4;
    small = (fewer > least ? fewer : least) * cols;
  }
  const int64_t large = rows_large * cols_large;
  if (large > 512) return 0;
  const int64_t depth = g.mode == GEMM_K_GROUPED ? g.red / g.G : g.red;
  const int64_t price = g.mode == GEMM_M_GROUPED ? 72 : g.mode == GEMM_K_GROUPED ? (depth <= 1024 ? 36 : 65) : depth <= 512 ? 45 : 68;
  // in units of 1 / (100 * 512 * 2) of a round of large tiles, five percent in favour of those
  return (small + up_div(small, 512) * 512) * price * 105 < up_div(large, 256) * (2 * 512 * 100) * 100 ? 128 : 0;
}

// ---- k-grouped: who computes which tile of skewed groups (gemm_persistent_parts.h has the forms) -------------------------------
enum Schedule { kInOrder, kEighths, kParts };

// A launch of groups that are not level: `largest` and `sum` of the groups' tile costs in blocks, `per_group` tiles each,
// `workgroups` that share them.  S: a workgroup's share of the cost; L: the largest tile in shares.  Weight gradients with
// Zipf-distributed and with single crowded groups whose operands come from HBM, as in a step; time in order over the time of eighths / parts,
// geometric means over the launches of each kind:
//   L >= 1, no XCD has more big tiles than workgroups: parts.  S from 90 on 1.09 / 1.24, 56 to 90 1.02 / 1.10, 36 to 56 0.96 / 1.04;
//     below 36 0.88 / 0.98
//   fewer than 32 tiles a group, of which an XCD's eighth would be two or three: every XCD reads nearly all of an operand for them.  Parts where
//     L >= 0.4, S >= 56: 0.94 / 1.15 (8942 tokens of 8 in 128 groups 512 x 2048 149 us / 167 / 145; 16384, 2048 x 768, 397 / 341 / 264); L below
//     0.87 / 1.03, S below 0.78 / 0.92
//   32 to 39 tiles: eighths where L >= 0.45, S >= 90: 1.04 / 1.00; others 0.90 / 0.97
//   from 40 tiles on: eighths where a group makes a 25th of the work and S >= 56: 1.10 / 1.01 (8192 of 6 in 64, 2816 x 2048 429 / 359 / 421; 10000 of
//     4 in 32, 5760 x 2880 820 / 687 / 781).  A 25th to a 16th 1.06, from an eighth on 1.17; less, up to 120 tiles, 0.98 / 0.99 (8192 of 6 in 64, less
//     skewed, 352 / 380 / 364), from 144 on 1.12 (1200 to 5000 of 8 in 128, 2880 x 2880, hardly skewed 1.14); S below 56 0.92 / 0.93
constexpr Schedule schedule_of_groups(int64_t largest, int64_t sum, int64_t per_group, int64_t workgroups) {
  const int64_t total = sum * per_group, most = largest * workgroups;  // most : total is L
  if (most >= total) return total >= 36 * workgroups ? kParts : kInOrder;
  if (per_group < 32) return 5 * most >= 2 * total && total >= 56 * workgroups ? kParts : kInOrder;
  if (per_group < 40) return 20 * most >= 9 * total && total >= 90 * workgroups ? kEighths : kInOrder;
  return (25 * largest >= sum || per_group >= 128) && total >= 56 * workgroups ? kEighths : kInOrder;
}

// What is dealt out one by one, in parts of a share: an eighth; among eighths of shares from 140 on, which pay for a longer list, a
// sixteenth (in order over eighth / sixteenth, S 56 to 72 1.09 / 1.01, to 110 1.12 / 1.11, to 140 1.12 / 1.13, to 200 1.10 / 1.12, above 1.09 / 1.12; parts
// 1.13 / 1.11)
constexpr int64_t big_tile_parts(Schedule form, int64_t total, int64_t workgroups) { return form == kEighths && total >= 140 * workgroups ? 16 : 8; }

}  // namespace pt

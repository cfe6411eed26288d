// Lines that a GEMM's dispatch draws by sizes alone: plain arithmetic, the same on the host and on the device.
#pragma once
#include <cstdint>

namespace pt {

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

// Argument block shared by the FP8 GEMM kernels.
#pragma once
#include "common.h"
#include "gemm_rules.h"

namespace pt {

struct GemmArgs {
  const uint8_t* a; int64_t lda;          // [rows_a, red] bytes
  const uint8_t* b; int64_t ldb;          // [rows_b, red] bytes
  const float* sa; int64_t sa_rs, sa_ks; int sa_shift;  // scale(row,kb) = sa[(row>>shift)*rs + kb*ks]
  const float* sb; int64_t sb_rs, sb_ks; int sb_shift;
  void* out; int64_t ldo;                 // elements
  int out_dtype; int accumulate;
  int64_t rows_a, rows_b, red;            // output is rows_a x rows_b; red = reduction length (dense / m-grouped)
  const int32_t* offs; int G;
  int mode;
  int64_t b_stride_g, sb_stride_g, out_stride_g;
  int tiles_a, tiles_b;                   // tile counts along rows_a / rows_b
  int64_t a_bytes, b_bytes, sa_bytes, sb_bytes;  // extents of a, one group of b, and their scale arrays
  int64_t total_tiles;
  const int32_t* out_row_index;           // m-grouped only: output row of result row r (negative: dropped); null = identity
  int64_t out_rows;                       // rows of the output when out_row_index is given
  const void* bias;                       // m-grouped only: [G, rows_b] in the output's type, row g added to the rows of group g
  int64_t split_len;                      // k-grouped with offs == null: group g reduces over [g, g + 1) * split_len (split-K)
  void* out2; int64_t split_row;          // m-grouped with out_row_index: row -2 - i of the index goes to row i of out2.
                                          // k-grouped: result rows from split_row on (a multiple of 128; 0 = none) go to out2, a second
                                          // parameter's gradient (group stride out2_stride_g) whose row 0 is row split_row
  int64_t out2_stride_g;
  int head_a, head_b;                     // dense only: result column h * (head_a + head_b) + c is out[h * head_a + c] for c < head_a, else
                                          // out2[h * head_b + c - head_a]; out2 lies behind out in one allocation (head_a == 0: one output)
  int64_t out_extent;                     // with head_a: bytes from out to the end of out2, below 2 GiB
  int few_rows;                           // m-grouped: the group ends are multiples of 64, not of 128
  const int32_t* row_used;                // m-grouped: negative (with out2: -1) where row r of the result is not wanted; row r of a may hold anything there
  int64_t used_rows;                      // with row_used: how many are, at most (rows_a may be a capacity)
  int b_kmajor;                           // m-grouped, row-split kernel: b is [red, rows_b] per group (row pitch ldb) instead of [rows_b, red]
};

// End of group g's reduction range in the k-grouped mode (its start is the end of group g - 1).
__device__ __forceinline__ int k_group_end(const GemmArgs& p, int g) {
  if (p.offs) return p.offs[g];
  const int64_t e = (int64_t)(g + 1) * p.split_len;
  return (int)(e < p.red ? e : p.red);
}


// m-grouped: groups from which on the kernel of large tiles looks for the padding behind each
static constexpr int kPaddedGroups = 64;

// persistent kernel whose two steps per 128-block split the tile by rows (gemm_rowsplit.hip)
int launch_gemm_rowsplit(const GemmArgs& a, hipStream_t stream);
// one tile of 64 or 128 rows x 128 columns per workgroup, for small problems, or kDeepTile (gemm_small.hip)
int launch_gemm_small(const GemmArgs& a, int rows, hipStream_t stream);
// the tiles of two independent dense products in one launch of that kernel
int launch_gemm_small_pair(const GemmArgs& a, const GemmArgs& b, int rows, hipStream_t stream);

}  // namespace pt

// Tile scheduling for the MI355X GEMM kernels: linear workgroup id -> output tile.
//
// Replaces the reference's block remap (mmm.cpp:1219-1236, mmmTensor.cpp:50-65), which
// groups tiles into column strips of 32 but is not a bijection when gridDim.x > 32 and
// gridDim.x % 32 != 0 (tiles are then skipped and others computed twice).
//
// This mapping is a bijection for every grid.  It is built from two bijective steps:
//  1. XCD compaction.  The command processor hands workgroups to the 8 XCDs round-robin
//     (workgroup b runs on XCD b % 8).  Each XCD has its own L2, so workgroups that share
//     operand panels should sit on the same XCD: virtual id v gives XCD x a contiguous
//     range of v.  With q = n / 8 and r = n % 8, XCDs 0..r-1 own q+1 ids and the rest q.
//  2. Grouped ordering.  Virtual ids walk GROUP_M tile-rows down a column before moving to
//     the next column, so 32 consecutive ids (one XCD's 32 CUs) form a 4 x 8 tile patch
//     that shares 4 A panels and 8 B panels in that XCD's L2.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define MMM_HD __host__ __device__ __forceinline__
#else
#define MMM_HD inline
#endif

namespace mmm {

constexpr int kNumXcd = 8;

MMM_HD int xcd_compact(int b, int n) {
  const int q = n / kNumXcd, r = n % kNumXcd;
  const int x = b % kNumXcd, slot = b / kNumXcd;
  return (x < r) ? x * (q + 1) + slot : r * (q + 1) + (x - r) * q + slot;
}

MMM_HD void grouped_tile(int v, int tiles_m, int tiles_n, int group_m, int* tm, int* tn) {
  const int per_group = group_m * tiles_n;
  const int g = v / per_group;
  const int first_m = g * group_m;
  const int rows = (tiles_m - first_m < group_m) ? (tiles_m - first_m) : group_m;
  const int w = v % per_group;
  *tm = first_m + w % rows;
  *tn = w / rows;
}

MMM_HD void tile_of_block(int b, int tiles_m, int tiles_n, int group_m, int* tm, int* tn) {
  grouped_tile(xcd_compact(b, tiles_m * tiles_n), tiles_m, tiles_n, group_m, tm, tn);
}

// A grid in which the tiles from `whole` on run as `splits` K ranges (whole == 0: every tile).  Block b
// of those is K range q of split tile j, block whole + q * split_tiles + j; with every tile split into
// more than two ranges (`major`, split_major), the blocks are numbered so that each XCD takes a contiguous
// run of the items (q, j): it then reads as few K ranges as possible, and a slice of A or B is fetched by one
// or two L2s instead of by every one that holds a tile.  Measured on MI355X (B from HBM): 64 x 4096 x 16384
// 34.5 -> 30.1 us, 128 x 4096 x 4096 20.1 -> 18.2, 2000 x 1000 x 8192 48.6 -> 45.4, 1536^2 x 12288 63.4 ->
// 61.4; with two ranges 128 x 14336 x 4096 38.3 -> 39.3.  Not on 128x128 tiles over ranges of fewer than 16 K
// tiles of operands of 8 to 20 MB, which the L2s hold either way: there 704 x 1024 x 2816 took 17.3 us
// against 13.9, 448 x 2368 x 2816 17.7 against 15.7, and 64 shapes of that kind 2.6% more on average (one,
// three or eight sets of buffers in turn made no difference); smaller operands 2% less, larger ones 7 to 10%.
MMM_HD bool split_major(int whole, int splits, int bm, int bn, int range_k_tiles, int64_t operand_bytes) {
  if (whole != 0 || splits <= 2) return false;
  return !(bm == 128 && bn == 128 && range_k_tiles < 16 && operand_bytes >= 8000000 && operand_bytes < 20000000);
}

MMM_HD void split_item(int b, int whole, int split_tiles, int splits, bool major, int* q, int* j) {
  const int v = major ? xcd_compact(b, split_tiles * splits) : b - whole;
  *q = v / split_tiles;
  *j = v - *q * split_tiles;
}

// The tile of block b (unsplit; j < 0) or of split tile j.
MMM_HD void tile_of_item(int b, int j, int whole, bool major, int tiles_m, int tiles_n, int* tm, int* tn) {
  int v = j < 0 ? b : whole + j;
  if (j < 0 || !major) v = xcd_compact(v, tiles_m * tiles_n);
  grouped_tile(v, tiles_m, tiles_n, 4, tm, tn);
}

}  // namespace mmm

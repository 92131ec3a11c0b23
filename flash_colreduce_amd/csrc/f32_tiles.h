// Tiles of the fp32 sweeps in parts, from sizes alone: plain C++, so that the rules can be tested without a device.
#pragma once

#include <stdint.h>

namespace fcr_tiles {

constexpr int64_t kMaxWorkgroups = 1ll << 24; // of 256 threads: the runtime refuses launches of 2^32 threads or more

// Tiles of the fp32 sweeps in parts (row_lse_f32_kernel, col_reduce_f32_kernel): waves per workgroup (four: two workgroups share a
// CU; eight: one) and resident 16-row groups per wave.  Two groups read a streamed fragment once for two blocks of scores,
// eight waves share the split of a streamed row: 4 x 2 and 8 x 1 are 128 rows, 8 x 2 256, 4 x 1 64.  Per call, fp32:
//   32 heads of 4096 x 4096 x 128   8x2 733 us, 4x2 828, 8x1 927      2 x 16 of 2048 x 2048 x 128 causal   8x1 129, 4x2 140, 8x2 164
//   32 of 1024 x 1024 x 128         8x1 70, 4x2 75, 4x1 85, 8x2 86    8 of 5055 x 5055 x 128 causal        8x1 253, 4x2 298
//   16 of 1500 x 1500 x 96 causal   8x1 63, 4x1 76, 4x2 81, 8x2 89    20 of 2100 x 2100 x 256 causal       8x1 204, 4x2 264
//   32 of 2048 x 2048 x 256         8x2 351, 4x2 410, 8x1 429         32 of 3000 x 3000 x 128 causal       8x2 247, 4x2 255, 8x1 291
//   32 of 2048 x 2048 x 160         8x2 247, 4x2 313, 8x1 330         32 of 512 x 512 x 128                4x1 32, 8x1 36, 4x2 40, 8x2 52
// So: 256 rows where 128-row tiles are more than one per CU (with the mask, which wants some to level it, two), 8 x 1
// where they are at most that, and 64 rows for short sweeps that leave every other CU without a workgroup.  Where most sweeps
// are whole (M and N a factor of 1.5 apart) or of at most 512 streamed rows the mask leaves little to level and 4 x 2 stays (32 heads of 330 x 1294 x 224, maxima, 4x2 67,
// 8x1 75.5; 48 of 1084 x 3477 x 80, maxima, 214, 226; 8 x 12 of 481 x 10807 x 192, sums and maxima, 1425, 1546; 40 of 512 x 900 x 64
// 31.6, 33.2; 32 of 1000 x 1900 x 128 101, 110; but of 1000 x 1300 x 128 73.5, 67.8).  The 256-row forms
// of D > 192 keep some registers in memory (rows up to 12, columns 1, sums and maxima 17 with the mask and 8 without) and are
// the fastest all the same: 40 heads of 3000 x 3000 x 256 causal, sums and maxima, 8x2 569 us, 4x2 619, 8x1 651.
struct F32Tile {
  int waves, groups;
  int rows() const { return 16 * waves * groups; }
};
// Whether the sweeps of a launch differ enough in length to want levelling.
inline bool f32_uneven(int M, int N, int streamed, bool causal) {
  return causal && 2 * (int64_t)N <= 3 * (int64_t)M && 2 * (int64_t)M <= 3 * (int64_t)N && streamed > 512;
}
inline F32Tile f32_tile(int rows, int64_t bh, bool causal, bool uneven, bool short_sweep, int cus) {
  const int64_t tiles = bh * (((int64_t)rows + 127) / 128);   // of 128 rows
  if (rows <= 64 || (short_sweep && 2 * tiles <= cus)) return F32Tile{4, 1};
  if (tiles <= cus) return F32Tile{8, 1};
  if (causal && tiles <= 2 * (int64_t)cus) return uneven ? F32Tile{8, 1} : F32Tile{4, 2};
  // (a launch of 512-thread workgroups reaches 2^32 threads at half as many of them)
  const bool tall_fits = bh * (((int64_t)rows + 255) / 256) < kMaxWorkgroups / 2;
  return tall_fits ? F32Tile{8, 2} : F32Tile{4, 2};
}
// A sweep of at most 128 queries is all prologue: 256-row tiles of four waves each half (32 heads of 64 x 8192 x 128 causal 66 us, with
// 8x2 tiles 73), except where the registers of that form do not reach for sums and maxima (D > 192, 128 x 8192 x 256 171 and 167).  At
// most 64 short queries take four waves for 8 x 1 too (2 heads of 12 x 15478 x 64 19.3, 8x1 20.4; 32 of 64 x 1024 x 64 15.3, 17.3).
inline F32Tile f32_col_tile(int ksteps, bool both, int M, int N, int64_t bh, bool causal, int cus) {
  const F32Tile t = f32_tile(N, bh, causal, f32_uneven(M, N, M, causal), M <= 512, cus);
  if (M <= 64 && ksteps <= 4 && t.waves == 8) return F32Tile{4, 2};
  return M <= 128 && t.waves * t.groups == 16 && !(both && ksteps > 6) ? F32Tile{4, 2} : t;
}
// A row sweep of 16 chunks or more over fewer tiles than CUs is split over the idle CUs (row_splits), two workgroups each.
inline F32Tile f32_row_tile(int M, int N, int64_t bh, bool causal, int cus) {
  const F32Tile t = f32_tile(M, bh, causal, f32_uneven(M, N, N, causal), N <= 15 * 64, cus);
  return t.waves == 8 && t.groups == 1 && N > 15 * 64 && bh * (((int64_t)M + 127) / 128) < cus ? F32Tile{4, 2} : t;
}

}  // namespace fcr_tiles

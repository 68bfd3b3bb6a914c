// Launches of the one-wave-per-SIMD MLA kernels (mla_decode_wide.hip) and the
// rules for when they run; the 8-wave kernels (mla_decode.hip) run otherwise.
#pragma once

#include "mla_common.hpp"

namespace mla {

// What a piece weighs besides its tiles in the balanced plan, in tiles: Q, the
// first tile's scores, the last tile's PV and the stores. Fits over the
// workgroups' ends say 5 to 6 (128 requests of ~4096 tokens: 12.5 us per piece
// and 2.6 per tile at 128 rows, 7.5 and 1.3 at 16; 32 of ~16384, 64 rows: 8.1
// and 1.36); at 8 the shares of one piece end last (171 us, of two 165, of three
// 159). It is 8 because most steps are fastest there. Step (us) at
//                                   2      4      5      6      8      10
//  128 of ~4096, 128 heads        184.8  180.7  178.6  175.0  173.1  176.0
//    the same, s_q = 2            305.3  304.8  302.2  300.1  300.9  301.3
//    the same, 16 heads           109.0  108.5  109.0  109.1  109.7  110.2
//  128 of ~8192, 128 heads        323.0  319.5  319.7  319.3  315.8  317.4
//  64 of ~2000, 128 heads          76.2   73.1   70.6   69.1   68.7   68.8
//  128 of ~1000, 128 heads         82.3   77.9   75.8   73.9   73.5   73.5
//  32 of ~16384, 64 heads         117.3  114.2  114.3  114.6  113.9  113.8
//  16 of ~4096, 128 heads          45.3   43.0   42.5   42.8   43.5   43.7
//  7 of ~3000, 128 heads           33.7   33.6   34.0   33.9   34.2   34.1
// (Even batches, best without: kEvenTiles.)
constexpr int kWidePieceCost = 8;

// (The phase-timing build stamps the 8-wave kernels, and runs them alone.)
#ifndef MLA_PHASE_TIMING
#define MLA_PHASE_TIMING 0
#endif
// Block sizes that are multiples of 8: the 8 rows of a tile that a wave copies
// lie in one block, so its copies need one scalar block id (the per-lane gather
// of other sizes keeps to the 8-wave kernels, which have registers for it).
// 16-token blocks, the gather -> here: one request of 4096 tokens, 128 heads,
// 75.9 -> 20.0 us (its smaller row groups with it); 128 requests of ~4096
// tokens 195.4 -> 179.1 (128 heads) and 144.0 -> 112.0 (16 heads).
inline bool wide_blocks(int block_size) { return !MLA_PHASE_TIMING && block_size % 8 == 0; }
inline int64_t tile_bound(const MlaArgs& a) {  // tiles of the longest sequence
  return ((int64_t)a.max_blocks * a.block_size + kTile - 1) / kTile;
}
// Row groups of `rows` query rows: 16, 32, 64 or 128, no larger than R needs.
inline int wide_rows(int R, int rows) {
  const int most = R <= 16 ? 16 : R <= 32 ? 32 : R <= 64 ? 64 : 128;
  return rows < most ? rows : most;
}
inline int row_groups(int R, int rows) { return (R + rows - 1) / rows; }

// Rows per workgroup of a balanced launch on nwg workgroups. Large row groups
// read the cache once and are the most work per byte; small ones spread little
// work over more CUs (every row group's workgroups read the tiles again, from
// the L2) and have less to load and store per piece. By work, in tiles x 16
// rows of the longest possible batch per workgroup; us at 16 / 32 / 64 / 128
// rows (128 heads; uniform lengths up to 4 requests, varlen beyond):
//    4  1 request of 4096 tokens      20.5   24.5   26.0   31.4
//    8  2 of 4096                     24.6   26.2   28.1   33.3
//   16  4 of 4096                     29.7   28.6   34.6   39.6
//   32  2 of 16384                    43.5   37.3   37.7   42.5
//   64  4 of 16384                    70.6   51.2   47.5   54.0
//  128  16 of ~4096                   90.3   60.5   48.9   56.8
//  512  16 of ~16384                 318.8  193.6  134.1  120.8
// Short requests are not that work but pieces: as long as larger row groups
// leave fewer requests than shares, requests of up to two tiles take them (the
// balanced launch at the rows by work -> here, and the 8-wave kernels: 200
// requests of 16 tokens, 64 heads, 25.2 -> 15.3, 18.8 us; 256 of 64, 128 heads,
// 38.7 -> 28.9, 33.0). Longer ones cost more in one large row group than in two
// rounds of smaller ones, unless every round of large ones is full: 256 of 200
// (500), 128 heads, 45.4 -> 39.8, 43.3 (66.9 -> 63.0, 61.1) us, but 300 of 200
// 60.4 -> 65.4. (256 of ~200, ragged, pay for it: 50.2 -> 54.2, 90.6.)
constexpr int kWorkRows[3] = {12, 28, 160};  // most work of 16, 32 and 64 rows
constexpr int kShortTiles = 2, kFullTiles = 8;
inline int wide_rows_balanced(int B, int R, int64_t tiles, int nwg) {
  const int64_t work = B * tiles * row_groups(R, 16);
  int rows = 16;
  for (int i = 0; i < 3 && work > (int64_t)kWorkRows[i] * nwg; ++i) rows *= 2;
  rows = wide_rows(R, rows);
  const int most = wide_rows(R, 128);
  if (tiles <= kShortTiles)
    while (rows < most && (int64_t)B * row_groups(R, rows) > nwg) rows *= 2;
  if (tiles >= kFullTiles && (int64_t)B * row_groups(R, most) % nwg == 0) rows = most;
  return rows;
}
// Fixed splits: the largest row groups that still give every CU a workgroup.
inline int wide_rows_splitkv(const MlaArgs& a, int cus) {
  const int64_t pieces = (int64_t)a.B * a.num_splits;
  int rows = 128;
  while (rows > 16 && pieces * row_groups(a.R, rows) * 2 <= cus) rows /= 2;
  return wide_rows(a.R, rows);
}

// Whether the wide kernels run. At 128 rows per workgroup the 8-wave kernels
// keep fixed splits (num_splits > 1) of at most 2048 tokens of the longest
// sequence: twice the waves load Q and store the states, which weighs more than
// the tiles there (64 requests of ~1024 tokens at 4 splits, 128 rows: 51.8
// against 55.5 us; of ~4096 tokens: 124.6 against 121.3).
inline bool wide_splitkv(const MlaArgs& a, int rows) {
  return wide_blocks(a.block_size) &&
         (rows < 128 || a.num_splits == 1 || tile_bound(a) * kTile > 2048ll * a.num_splits);
}
// Rows per workgroup of a balanced launch whose longest sequence has at most
// `tiles` tiles, 0 for the 8-wave kernels (they run the other block sizes alone:
// on few workgroups and tiles too they are slower, 512 rows of one request on
// one of 128 rows, 64 tokens 20.9 against 18.2 us, 256 tokens 29.1 against 26.2).
inline int balanced_rows(int B, int R, int block_size, int64_t tiles, int nwg) {
  return wide_blocks(block_size) ? wide_rows_balanced(B, R, tiles, nwg) : 0;
}
// The most tiles, from `tiles` on, for which balanced_rows stays what it is.
inline int64_t balanced_rows_until(int B, int R, int block_size, int64_t tiles, int nwg) {
  const int64_t per_tile = (int64_t)B * row_groups(R, 16);
  const int64_t ends[] = {kShortTiles, kFullTiles - 1,
                          (int64_t)kWorkRows[0] * nwg / per_tile,
                          (int64_t)kWorkRows[1] * nwg / per_tile,
                          (int64_t)kWorkRows[2] * nwg / per_tile};
  const int rows = balanced_rows(B, R, block_size, tiles, nwg);
  int64_t until = INT64_MAX;
  for (const int64_t e : ends)
    if (e >= tiles && e < until && balanced_rows(B, R, block_size, e + 1, nwg) != rows) until = e;
  return until;
}

hipError_t launch_wide_splitkv(const MlaArgs& a, int rows, hipStream_t stream);
hipError_t launch_wide_balanced(const MlaArgs& a, int rows, hipStream_t stream);

}  // namespace mla

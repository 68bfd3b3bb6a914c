// Launches of the one-wave-per-SIMD MLA kernels (mla_decode_wide.hip) and the
// rules for when they run; the 8-wave kernels (mla_decode.hip) run otherwise.
#pragma once

#include "mla_common.hpp"

namespace mla {

// What a piece weighs besides its tiles in the balanced plan, in tiles: Q, the
// first tile's scores, the last tile's PV and the stores take 10-14 us per
// piece of 128 rows against ~1.8 us per tile (mla_4k: 187 / 185 / 182 us at 2 /
// 4 / 8). Fewer rows: 3-4 us against 1.4 (128 requests of ~4096 tokens, 16
// rows: 115 / 114 / 113.5 / 113 us at 0 / 2 / 4 / 8).
constexpr int kWidePieceCost = 8;

// Block sizes that are multiples of 32: a tile's rows lie in one block, so a
// wave's copies need one scalar block id (the per-lane gather of other sizes
// keeps to the 8-wave kernels, which have registers for it). Past 64 rows the
// 8-wave kernels also keep
//  - fixed splits (num_splits > 1) of at most 2048 tokens of the longest
//    sequence: twice the waves load Q and store the states, which weighs more
//    than the tiles there (64 requests of ~1024 tokens at 4 splits, 128 rows:
//    51.8 against 55.5 us; of ~4096 tokens: 124.6 against 121.3);
//  - balanced launches of at most 8 tiles in all (one request of 64 tokens:
//    18.9 against 19.4 us; of 1024: 23.9 against 22.9).
// (The phase-timing build stamps the 8-wave kernels, and runs them alone.)
#ifndef MLA_PHASE_TIMING
#define MLA_PHASE_TIMING 0
#endif
inline bool wide_blocks(const MlaArgs& a) {
  return !MLA_PHASE_TIMING && a.block_size % kTile == 0;
}
inline int64_t tile_bound(const MlaArgs& a) {  // tiles of the longest sequence
  return ((int64_t)a.max_blocks * a.block_size + kTile - 1) / kTile;
}
inline bool wide_splitkv(const MlaArgs& a) {
  return wide_blocks(a) &&
         (a.R <= 64 || a.num_splits == 1 || tile_bound(a) * kTile > 2048ll * a.num_splits);
}
inline bool wide_balanced(const MlaArgs& a) {
  return wide_blocks(a) && (a.R <= 64 || a.B * tile_bound(a) > 8);
}

hipError_t launch_wide_splitkv(const MlaArgs& a, hipStream_t stream);
hipError_t launch_wide_balanced(const MlaArgs& a, hipStream_t stream);

}  // namespace mla

// The device-side plan of the token-balanced MLA launch, computed by every
// workgroup from seq_lens (no host synchronisation, no plan launch). The work
// is a line of units, request after request: a request with tiles takes
// piece_cost units for what a piece costs besides its tiles (Q, the first
// tile's scores, the stores) and then one unit per 32-token tile. Share w of n
// is the line's units [w U / n, (w + 1) U / n): its tiles, and the requests it
// begins, weigh the same in every share.
#pragma once

#include "mla_common.hpp"

namespace mla {

__device__ __forceinline__ int live_len(const MlaArgs& a, int b) {
  return min(max(a.seq_lens[b], 0), a.max_blocks * a.block_size);
}
__device__ __forceinline__ uint64_t tiles_of(const MlaArgs& a, int b) {
  return (uint64_t)((live_len(a, b) + kTile - 1) / kTile);
}

__device__ __forceinline__ uint64_t units_of(const MlaArgs& a, int b) {
  const uint64_t t = tiles_of(a, b);
  return t ? t + (uint64_t)a.piece_cost : 0;
}

// Share w's first unit.
__device__ __forceinline__ uint64_t share_start(uint64_t U, int w, int n) {
  return (uint64_t)w * U / (uint64_t)n;
}
// The share that holds unit u: the largest w with share_start(w) <= u.
__device__ __forceinline__ int share_of(uint64_t U, uint64_t u, int n) {
  return (int)(((u + 1) * (uint64_t)n - 1) / U);
}

// Shares for U units: at most nshare, and no more than 5 sqrt(U). A share costs
// its units one after the other (~1.5 us each) and its states in the merge
// (~0.06 us per share for 128 rows), so with little work fewer shares than CUs
// are faster. One request of 4096 tokens, 128 heads (136 units): 36.8 / 31.6 /
// 28.8 / 31.0 us at 136 / 68 / 34 / 17 shares; 16 heads (132): 17.7 / 15.7 /
// 16.3 / 18.8 us. From about 2600 units on every CU has a share.
__device__ __forceinline__ int share_count(uint64_t U, int nshare) {
  uint64_t n = (uint64_t)(5.f * sqrtf((float)U)) + 1;
  n = n < U ? n : U;
  return (int)(n < (uint64_t)nshare ? n : (uint64_t)nshare);
}

// Values every lane holds alike, handed to the compiler as scalars.
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ uint64_t uniform(uint64_t x) {
  return (uint64_t)(uint32_t)uniform((int)x) | ((uint64_t)(uint32_t)uniform((int)(x >> 32)) << 32);
}

// Where a share's tiles begin: token ts of request b, with `units` units of the
// share from that tile on (no tile at all if units <= 0).
struct SharePlan {
  int b, ts;
  int64_t units;
};

// Plan of share w for a workgroup of NT threads (every thread calls it; it
// joins workgroup barriers): units summed over NT chunks of the batch, an
// inclusive scan of the chunk sums in `part` (NT words of LDS; within the
// waves by shuffles, then across them), the share's bounds, and its first
// request by bisection of the chunks and a walk within one. With `write_pre`
// the requests' first units go to a.pre (pre[0 .. B - 1], pre[B] = U,
// pre[B + 1] = n) for the merge.
template <int NT>
__device__ __forceinline__ SharePlan plan_share(const MlaArgs& a, int w, uint64_t* part,
                                                bool write_pre) {
  constexpr int NW = NT / 64;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int per = (a.B + NT - 1) / NT;
  const int b0 = min(tid * per, a.B), b1 = min(b0 + per, a.B);
  uint64_t sum = 0;
  for (int b = b0; b < b1; ++b) sum += units_of(a, b);
  uint64_t x = sum;  // inclusive scan within the wave
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t y = __shfl_up((unsigned long long)x, o, 64);
    if (lane >= o) x += y;
  }
  part[tid] = x;
  __syncthreads();
  uint64_t before = 0, U = 0;  // the waves before this one; all of them
#pragma unroll
  for (int k = 0; k < NW; ++k) {
    const uint64_t t = part[64 * k + 63];
    before += k < wv ? t : 0;
    U += t;
  }
  x += before;
  U = uniform(U);
  __syncthreads();
  part[tid] = x;
  __syncthreads();
  const int n = share_count(U, a.nshare);
  if (write_pre) {
    uint64_t run = x - sum;
    for (int b = b0; b < b1; ++b) {
      a.pre[b] = run;
      run += units_of(a, b);
    }
    if (tid == 0) {
      a.pre[a.B] = U;
      a.pre[a.B + 1] = (uint64_t)n;
    }
  }
  SharePlan p{0, 0, 0};
  if (w >= n) return p;
  const uint64_t u0 = share_start(U, w, n), u1 = share_start(U, w + 1, n);
  int lo = 0, hi = NT - 1;  // the first chunk that ends past u0
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (part[mid] > u0) hi = mid; else lo = mid + 1;
  }
  lo = uniform(lo);
  uint64_t p0 = lo > 0 ? uniform(part[lo - 1]) : 0;  // request p.b's first unit
  p.b = lo * per;
  for (uint64_t nu = units_of(a, p.b); p0 + nu <= u0; nu = units_of(a, p.b)) {
    p0 += nu;
    ++p.b;
  }
  p.b = uniform(p.b);
  const uint64_t first = uniform(p0) + (uint64_t)a.piece_cost;  // its first tile's unit
  p.ts = u0 > first ? (int)(u0 - first) * kTile : 0;
  p.units = (int64_t)u1 - (int64_t)(u0 > first ? u0 : first);
  return p;
}

// A piece of a share: `tiles` tiles of request b, tokens [start, end) of its S.
struct Piece {
  int b, S, start, end, tiles;
};

// The piece at token ts of request b, or (ts == 0) of the next request with
// tokens, of a share with units > 0 units from there on.
__device__ __forceinline__ Piece piece_at(const MlaArgs& a, int b, int ts, int64_t units) {
  // The lengths are read-only for the launch; through the constant address
  // space the uniform loads are scalar.
  const __attribute__((address_space(4))) int* lens =
      (const __attribute__((address_space(4))) int*)a.seq_lens;
  const int s_cap = a.max_blocks * a.block_size;
  int S = min(lens[b], s_cap);
  while (S <= ts) S = min(lens[++b], s_cap);
  const int in_request = (S - ts + kTile - 1) / kTile;
  Piece p;
  p.b = b;
  p.S = S;
  p.start = ts;
  p.tiles = (int)(units < in_request ? units : in_request);
  p.end = p.tiles == in_request ? S : ts + p.tiles * kTile;
  return p;
}

// Moves on from piece p of a share with `units` units left: the next piece, or
// false at the share's end.
__device__ __forceinline__ bool next_piece(const MlaArgs& a, Piece& p, int64_t& units) {
  units -= p.tiles + a.piece_cost;
  if (units <= 0) return false;
  p = piece_at(a, p.b + 1, 0, units);
  return true;
}

}  // namespace mla

// The device-side plan of the token-balanced MLA launch, computed by every
// workgroup from seq_lens (no host synchronisation, no plan launch). The work
// is a line of units, request after request: a request with tiles takes
// piece_cost units for what a piece costs besides its tiles (Q, the first
// tile's scores, the stores) and then one unit per 32-token tile. Share w of n
// is the line's units [w U / n, (w + 1) U / n): its tiles, and the requests it
// begins, weigh the same in every share. (Even batches: no piece_cost units, see
// kEvenTiles.)
#pragma once

#include "mla_common.hpp"

namespace mla {

__device__ __forceinline__ int live_len(const MlaArgs& a, int b) {
  return min(max(a.seq_lens[b], 0), a.max_blocks * a.block_size);
}
// The lengths are read-only for the launch; through the constant address space
// the loads of uniform ones are scalar.
__device__ __forceinline__ const __attribute__((address_space(4))) int* scalar_lens(
    const MlaArgs& a) {
  return (const __attribute__((address_space(4))) int*)a.seq_lens;
}
__device__ __forceinline__ int scalar_live_len(const MlaArgs& a, int b) {
  return min(max(scalar_lens(a)[b], 0), a.max_blocks * a.block_size);
}
__device__ __forceinline__ uint64_t tiles_of(const MlaArgs& a, int b) {
  return (uint64_t)((live_len(a, b) + kTile - 1) / kTile);
}

__device__ __forceinline__ uint64_t units_of(const MlaArgs& a, int b) {
  const uint64_t t = tiles_of(a, b);
  return t ? t + (uint64_t)a.piece_cost : 0;
}

// x / n. (A 64-bit division is a loop of its own, the 32-bit one some 20
// instructions; U n stays below 2^32 up to 500 million tokens on 256 CUs.)
__device__ __forceinline__ uint64_t div_by(uint64_t x, uint64_t n) {
  if (__builtin_amdgcn_ballot_w64(((x | n) >> 32) != 0) == 0) return (uint32_t)x / (uint32_t)n;
  return x / n;
}
// Share w's first unit.
__device__ __forceinline__ uint64_t share_start(uint64_t U, int w, int n) {
  return div_by((uint64_t)w * U, (uint64_t)n);
}
// The share that holds unit u: the largest w with share_start(w) <= u.
__device__ __forceinline__ int share_of(uint64_t U, uint64_t u, int n) {
  return (int)div_by((u + 1) * (uint64_t)n - 1, U);
}

// Shares for U units of B requests: at most nshare, and no more than 5 sqrt(U)
// or one per request. A share costs its units one after the other and its states
// in the merge, so with little work fewer shares than CUs can be faster. Balanced
// launch (us) with at most 2.5 / 5 / 10 sqrt(U) shares and one per CU, 16 heads:
//   1 request of 4096 tokens    16.6   15.6   17.1   17.2
//   1 of 1000                   14.2   13.6   13.1   13.1
//   1 of 16384                  21.1   20.7   24.6   24.4
//   3 of ~16384, 32 heads       29.5   28.1   30.4   30.5
//   16 of ~500                  18.5   16.4   16.1   16.6
// (At more heads the row groups often leave fewer shares than that: one request
// of 1000 tokens, 128 heads, 15.6 / 16.6 / 16.6 / 16.6.) As many shares as
// requests cost no merge: 256 requests of 32 tokens, 16 heads, 14.5 us in 240
// shares, 10.4 in 256.
__host__ __device__ inline int share_count(uint64_t U, int B, int nshare) {
  uint64_t n = (uint64_t)(5.f * sqrtf((float)U)) + 1;
  n = n > (uint64_t)B ? n : (uint64_t)B;
  n = n < U ? n : U;
  return (int)(n < (uint64_t)nshare ? n : (uint64_t)nshare);
}

// Values every lane holds alike, handed to the compiler as scalars.
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ uint64_t uniform(uint64_t x) {
  return (uint64_t)(uint32_t)uniform((int)x) | ((uint64_t)(uint32_t)uniform((int)(x >> 32)) << 32);
}

// Lane l gets the sum of x over lanes 0 .. l (gfx9 row_shr and row_bcast).
template <int kCtrl, int kRows>
__device__ __forceinline__ uint64_t dpp_u64(uint64_t x) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)x, kCtrl, kRows, 0xF,
                                                            false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(x >> 32), kCtrl, kRows, 0xF,
                                                            false);
  return (uint64_t)lo | ((uint64_t)hi << 32);
}
__device__ __forceinline__ uint64_t wave_scan(uint64_t x) {
  x += dpp_u64<0x111, 0xF>(x);  // row_shr:1, 2, 4, 8 (lanes shifted in: 0)
  x += dpp_u64<0x112, 0xF>(x);
  x += dpp_u64<0x114, 0xF>(x);
  x += dpp_u64<0x118, 0xF>(x);
  x += dpp_u64<0x142, 0xA>(x);  // row_bcast:15 into rows 1 and 3
  x += dpp_u64<0x143, 0xC>(x);  // row_bcast:31 into rows 2 and 3
  return x;
}

// Where a share's tiles begin: token ts of request b (of S tokens), with
// `units` units of the share from that tile on (no tile at all if units <= 0).
struct SharePlan {
  int b, S, ts;
  int64_t units;
};

// An even batch, of as many tiles in every request and n a multiple of B, is cut
// without the weight: every share then holds one piece, and charged for it the
// shares that begin a request get fewer tiles than they could. From this many
// tiles per share on (shorter shares gain nothing). Balanced launch, with the
// weight -> without (and the 8-wave kernels, which know none), 128 heads: 64
// requests of 4096 tokens 98.7 -> 96.6 us (96.5), 128 of 2048 101.2 -> 98.4
// (98.5), 128 of 4096 165.3 -> 162.0 (165.7); 16 heads, 128 of 4096, 102.9 ->
// 100.8 (124.7). All other calls pay up to 0.1 us for the looking.
constexpr int kEvenTiles = 16;

// Plan of share w for a workgroup of NT threads (every thread calls it; it
// joins workgroup barriers): units summed over NT chunks of the batch, an
// inclusive scan of the chunk sums within the waves, across them through `lds`
// (NT / 32 + 2 words), the share's bounds, and its first request, found by the
// thread whose chunk holds the share's first unit. `capped` asks for
// share_count's shares instead of a.nshare, and for even batches to be cut
// without the weight. With `write_pre` the requests' first units go to a.pre for
// the merge (pre[0 .. B - 1], pre[B] = U, pre[B + 1] = n and the weight in the
// high half).
//
// A chain of latencies that every workgroup pays before its first load: kept
// short by scanning in registers, two barriers, 32-bit divisions and no load
// after the lengths (one request of 4096 tokens: 15.9 -> 15.2 us with 16 heads,
// 20.1 -> 19.3 with 128, against a scan by shuffles and a bisection in the
// LDS). The chunk is walked by its whole wave: a branch that one lane takes
// alone made the compiler spill in the 128-row kernel.
template <int NT>
__device__ __forceinline__ SharePlan plan_share(const MlaArgs& a, int w, uint64_t* lds,
                                                bool capped, bool write_pre) {
  constexpr int NW = NT / 64;
  const int tid = threadIdx.x, wv = tid >> 6;
  const int per = (a.B + NT - 1) / NT;
  const int b0 = min(tid * per, a.B), b1 = min(b0 + per, a.B);
  uint64_t sum = 0;
  for (int b = b0; b < b1; ++b) sum += units_of(a, b);
  uint64_t x = wave_scan(sum);
  if ((tid & 63) == 63) lds[wv] = x;
  __syncthreads();
  uint64_t before = 0, U = 0;  // the waves before this one; all of them
#pragma unroll
  for (int k = 0; k < NW; ++k) {
    const uint64_t t = lds[k];
    before += k < wv ? t : 0;
    U += t;
  }
  x += before - sum;  // the chunk's first unit
  U = uniform(U);
  const int n = capped ? share_count(U, a.B, a.nshare)
                       : (int)(U < (uint64_t)a.nshare ? U : (uint64_t)a.nshare);
  if (capped && __builtin_expect(U >= (uint64_t)kEvenTiles * (uint32_t)n, 0) && n % a.B == 0) {
    // An even batch: t tiles in every request (the first one, the last one and
    // the sum are looked at before every one is), k whole shares for each.
    const int t = (scalar_live_len(a, 0) + kTile - 1) / kTile;
    const uint64_t T = (uint64_t)a.B * (uint32_t)t;
    if (t > 0 && U == T + (uint64_t)a.B * (uint32_t)a.piece_cost &&
        (scalar_live_len(a, a.B - 1) + kTile - 1) / kTile == t &&
        T >= (uint64_t)kEvenTiles * (uint32_t)n) {
      bool even = true;
      for (int b = b0; b < b1; ++b) even = even && tiles_of(a, b) == (uint64_t)t;
      const bool wave_even = __builtin_amdgcn_ballot_w64(!even) == 0;
      if ((tid & 63) == 0) lds[NW + 2 + wv] = wave_even;
      __syncthreads();
      uint64_t all = 1;
#pragma unroll
      for (int k = 0; k < NW; ++k) all &= lds[NW + 2 + k];
      if (uniform((int)all) != 0) {
        if (write_pre) {
          for (int b = b0; b < b1; ++b) a.pre[b] = (uint64_t)b * (uint32_t)t;
          if (tid == 0) {
            a.pre[a.B] = T;
            a.pre[a.B + 1] = (uint64_t)(uint32_t)n;
          }
        }
        // Share w: piece i of the k of request w / k.
        SharePlan p{0, 0, 0, 0};
        if (w >= n) return p;
        const int k = n / a.B, i = w % k;
        const int t0 = (int)div_by((uint64_t)i * (uint32_t)t, k);
        p.b = w / k;
        p.S = scalar_live_len(a, p.b);
        p.ts = t0 * kTile;
        p.units = (int)div_by((uint64_t)(i + 1) * (uint32_t)t, k) - t0;
        return p;
      }
    }
  }
  if (write_pre) {
    uint64_t run = x;
    for (int b = b0; b < b1; ++b) {
      a.pre[b] = run;
      run += units_of(a, b);
    }
    if (tid == 0) {
      a.pre[a.B] = U;
      a.pre[a.B + 1] = (uint64_t)(uint32_t)n | ((uint64_t)(uint32_t)a.piece_cost << 32);
    }
  }
  SharePlan p{0, 0, 0, 0};
  if (w >= n) return p;
  const uint64_t u0 = uniform(share_start(U, w, n)), u1 = uniform(share_start(U, w + 1, n));
  // One thread's chunk holds u0 < U; its wave walks the chunk together.
  const uint64_t owner = __builtin_amdgcn_ballot_w64(x <= u0 && u0 < x + sum);
  if (owner != 0) {
    const int l = __builtin_ctzll(owner);
    uint64_t p0 = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, l) |
                  ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(x >> 32), l) << 32);
    int b = uniform((64 * wv + l) * per);
    for (uint64_t nu = uniform(units_of(a, b)); p0 + nu <= u0; nu = uniform(units_of(a, b))) {
      p0 += nu;
      ++b;
    }
    lds[NW] = p0;
    lds[NW + 1] = (uint64_t)(uint32_t)b | ((uint64_t)(uint32_t)live_len(a, b) << 32);
  }
  __syncthreads();
  const uint64_t b_and_s = uniform(lds[NW + 1]);
  p.b = (int)(uint32_t)b_and_s;
  p.S = (int)(b_and_s >> 32);
  const uint64_t first = uniform(lds[NW]) + (uint64_t)a.piece_cost;  // its first tile's unit
  p.ts = u0 > first ? (int)(u0 - first) * kTile : 0;
  p.units = (int64_t)u1 - (int64_t)(u0 > first ? u0 : first);
  return p;
}

// A piece of a share: `tiles` tiles of request b, tokens [start, end) of its S.
struct Piece {
  int b, S, start, end, tiles;
};

// The piece at token ts < S of request b, of a share with units > 0 units from
// there on.
__device__ __forceinline__ Piece piece_of(int b, int S, int ts, int64_t units) {
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
  const auto* lens = scalar_lens(a);
  int b = p.b + 1;
  while (lens[b] <= 0) ++b;
  p = piece_of(b, min(lens[b], a.max_blocks * a.block_size), 0, units);
  return true;
}

}  // namespace mla

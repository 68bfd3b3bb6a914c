// MLA absorbed-path paged decode on one wave per SIMD, for block sizes that
// keep 8 aligned tokens inside one cache block (multiples of 8).
//
// A workgroup of 4 waves owns M x RW query rows of a request (RW rows for
// each of M row sets) and walks the tiles of its pieces. Every tile is copied
// HBM -> LDS once (each wave copies one of its 4 row blocks) into a ring of 4
// slots. Wave w serves row set w % M:
//   QK^T   S^T[32 tok x RW rows] = K[32 tok x 576] . Q^T, Q^T in registers;
//   softmax on the C layout, a lane holding one row's scores: the
//          probabilities are the P^T operand of PV without leaving the
//          registers (the tokens of PV's k-slots are permuted to match, in P^T
//          and in V alike);
//   PV     O^T[dims x RW rows] += V^T[dims x 32 tok] . P^T[32 tok x RW rows],
//          over the wave's part w / M of the 512 dims (all of them for M = 4).
// So the waves share tiles and nothing else: one barrier per tile, which hands
// over the next tile and a free slot. RW = 32 with M = 4 takes 128 rows; RW =
// 16 takes 16, 32 or 64 rows (M = 1, 2, 4; with M < 4 the row set's 4 / M
// waves each score the whole tile and share the dims).
//
// What bounds it. 128 rows: the matrix units, through the power limit. One
// wave per SIMD holds 512 registers: Q^T of 32 rows takes 144, their 512 dims
// of output 256 accumulators (AGPRs), so each operand read from the LDS feeds
// 32 rows (v_mfma_f32_32x32x16_bf16; 272 KiB of LDS reads per tile). A wave's
// own VALU and LDS instructions run under its MFMAs as long as at most about
// five issue per 32-cycle MFMA (measured: 32x32x16 with 0 / 5 / 8 FMAs between
// 33.5 / 37.0 / 50.8 cycles each), so the softmax, the copies and the operand
// reads are dealt out evenly between the MFMAs by hand, fenced with scheduling
// barriers: tile s's exponentials and the copies of tile s + 3 between the
// QK^T MFMAs of tile s + 1, tile s + 1's exponents between the PV MFMAs of tile
// s. Fewer rows: HBM.
//
// The copies run ahead across the pieces of a share (the next piece's first
// tiles land while the last piece ends).
#include "gqa_device.hpp"
#include "mla_common.hpp"
#include "mla_plan.hpp"
#include "mla_wide.hpp"

#include <type_traits>

namespace mla {
namespace {

constexpr int kWWaves = 4;
constexpr int kWThreads = 64 * kWWaves;
constexpr int kWDepth = 4;            // ring slots
constexpr int kWCopies = kColBlocks;  // copies of a wave per tile: row block w
constexpr int kWRing = kWDepth * kTileBytes;
constexpr int kWLds = kWRing + 32;  // and the votes of two pieces
constexpr int kWSteps = 36;         // QK^T MFMAs per tile, either shape
// Operand reads run ahead of their MFMA through rings of registers.
constexpr int kWKRing = 6;
constexpr int kWVRing = 5;
// A row's exponents are taken relative to a reference set by its first live
// tile; a later score this much above it sends the piece through once more,
// against the rows' true maxima.
constexpr float kWSlack = 32.f;

typedef float f32x16_t __attribute__((ext_vector_type(16)));

// Two floats as bf16 (round to nearest even), lo in the low half.
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t,
                            __builtin_convertvector((f32x2_t){lo, hi}, gqa::bf16x2_t));
}

// The two matrix shapes. Lane l serves row l % RW; kTokOff(e) + 4 (l / RW) is
// the token of its score e in the tile. swz(t) is the position XOR of token
// t's 16-byte chunks in a column block; each makes its shape's K (ds_read_b128)
// and V (ds_read_b64_tr_b16) reads free of bank conflicts.
template <int RW>
struct Shape;

// c = A B and c += A B with c in VGPRs: left to itself the compiler puts every
// MFMA result in an AGPR, and the PV accumulators of 32 rows fill all of those.
// The compiler does not know these instructions' latency: their results are
// first read behind several other MFMAs (or behind s_nops).
template <>
struct Shape<32> {
  typedef f32x16_t acc_t;
  static constexpr int kEl = 16;        // scores of a lane per tile
  static constexpr int kDimsPerMfma = 32;
  static constexpr int kPvSteps = 2;    // PV k-steps of 16 tokens
  static constexpr int kMaxTok = 27;    // largest kTokOff
  static constexpr int kChains = 2;     // QK^T accumulators: even and odd k-steps
  __device__ static constexpr int tok_off(int e) { return 8 * (e >> 2) + (e & 3); }
  __device__ static constexpr int chain(int i) { return i & 1; }
  __device__ static int q_dim(int i) { return 16 * i; }  // k-step i's dims + 8 (l / 32)
  static constexpr int kQ = 36;                          // Q^T registers of 16 bytes
  __device__ static constexpr int q_of(int i) { return i; }
  __device__ static int swz(int t) { return 4 * ((t >> 1) & 1) + ((t >> 3) & 3); }
  __device__ static uint32_t k_off(int l) {  // token l % 32, chunk l / 32
    const int t = l & 31;
    return (uint32_t)((t >> 3) * kRowBlockBytes + (t & 7) * 128 + 16 * ((l >> 5) ^ swz(t)));
  }
  static constexpr int kKAddr = 4;
  __device__ static constexpr uint32_t k_xor(int a) { return 32u * a; }
  __device__ static constexpr int k_addr(int i) { return i & 3; }
  __device__ static constexpr uint32_t k_imm(int i) { return 1024u * (i >> 2); }
  __device__ static uint32_t v_off(int l) {
    const int x = l & 15, u = (l >> 4) & 1, r = 4 * (l >> 5) + (x >> 2);
    return (uint32_t)(r * 128 + 16 * ((2 * u + ((x & 3) >> 1)) ^ (4 * ((r >> 1) & 1))) +
                      8 * (x & 1));
  }
  // V^T of 32 dims (block nb) and the 16 tokens of k-step t.
  __device__ static bf16x8_t read_v(uint32_t T, int nb, int t) {
    const uint32_t off = 1024u * (nb >> 1), x = 64u * (nb & 1);
    const bf16x4_t v0 = lds_load_tr((T ^ (x + 32u * t)) + off + (2 * t) * kRowBlockBytes);
    const bf16x4_t v1 = lds_load_tr((T ^ (x + 32u * t + 16u)) + off + (2 * t + 1) * kRowBlockBytes);
    return bf16x8_t{v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
  }
  __device__ static void qk0(acc_t& c, bf16x8_t A, bf16x8_t B) {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=v"(c) : "v"(A), "v"(B));
  }
  __device__ static void qk(acc_t& c, bf16x8_t A, bf16x8_t B) {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(A), "v"(B));
  }
  __device__ static acc_t pv(bf16x8_t A, bf16x8_t B, acc_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, B, c, 0, 0, 0);
  }
  __device__ static float exponent(const acc_t (&c)[2], int e, float scale, float nbase) {
    return fmaf(c[0][e], scale, fmaf(c[1][e], scale, nbase));
  }
  // Over the lanes of one row.
  __device__ static float row_max(float x) {
    float a, b;
    gqa::xor32_pair(x, a, b);
    return fmaxf(a, b);
  }
  __device__ static float row_sum(float x) { return gqa::xor32_sum(x); }
  // 16-byte unit of a 64-dim chunk that 4-dim group x (block x / 4 of the
  // chunk, group x % 4 of its accumulator) of lane l fills.
  static constexpr int kGroups = 8;
  __device__ static int unit(int x, int l) { return 2 * x + (l >> 5); }
  __device__ static constexpr int group_block(int x) { return x / 4; }
  __device__ static constexpr int group_reg(int x) { return 4 * (x % 4); }
};

template <>
struct Shape<16> {
  typedef f32x4_t acc_t;
  static constexpr int kEl = 8;
  static constexpr int kDimsPerMfma = 16;
  static constexpr int kPvSteps = 1;  // one k-step of 32 tokens
  static constexpr int kMaxTok = 19;
  // Token groups of 16, and for each even and odd k-steps (a single chain of
  // 16x16x32 MFMAs would wait for itself).
  static constexpr int kChains = 4;
  __device__ static constexpr int tok_off(int e) { return 16 * (e >> 2) + (e & 3); }
  __device__ static constexpr int chain(int i) { return i & 3; }
  __device__ static int q_dim(int i) { return 32 * i; }  // + 8 (l / 16)
  static constexpr int kQ = 18;
  __device__ static constexpr int q_of(int i) { return i >> 1; }
  __device__ static int swz(int t) { return t & 6; }
  __device__ static uint32_t k_off(int l) {  // token l % 16, chunk l / 16
    const int t = l & 15;
    return (uint32_t)((t >> 3) * kRowBlockBytes + (t & 7) * 128 + 16 * ((l >> 4) ^ swz(t)));
  }
  static constexpr int kKAddr = 2;
  __device__ static constexpr uint32_t k_xor(int a) { return 64u * a; }
  __device__ static constexpr int k_addr(int i) { return (i >> 1) & 1; }
  __device__ static constexpr uint32_t k_imm(int i) {  // k-step i / 2, token group i % 2
    return 1024u * (i >> 2) + 2u * kRowBlockBytes * (i & 1);
  }
  __device__ static uint32_t v_off(int l) {
    const int x = l & 15, g = l >> 4, r = 4 * (g & 1) + (x >> 2);
    return (uint32_t)((g >> 1) * kRowBlockBytes + r * 128 + 16 * (((x & 3) >> 1) ^ (r & 6)) +
                      8 * (x & 1));
  }
  __device__ static bf16x8_t read_v(uint32_t T, int nb, int) {
    const uint32_t a = (T ^ (32u * (nb & 3))) + 1024u * (nb >> 2);
    const bf16x4_t v0 = lds_load_tr(a), v1 = lds_load_tr(a + 2 * kRowBlockBytes);
    return bf16x8_t{v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
  }
  __device__ static void qk0(acc_t& c, bf16x8_t A, bf16x8_t B) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=v"(c) : "v"(A), "v"(B));
  }
  __device__ static void qk(acc_t& c, bf16x8_t A, bf16x8_t B) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(A), "v"(B));
  }
  __device__ static acc_t pv(bf16x8_t A, bf16x8_t B, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, B, c, 0, 0, 0);
  }
  __device__ static float exponent(const acc_t (&c)[4], int e, float scale, float nbase) {
    return fmaf(c[e >> 2][e & 3], scale, fmaf(c[2 + (e >> 2)][e & 3], scale, nbase));
  }
  __device__ static float row_max(float x) { return gqa::xor32_max(gqa::xor16_max(x)); }
  __device__ static float row_sum(float x) { return gqa::xor32_sum(gqa::xor16_sum(x)); }
  static constexpr int kGroups = 4;
  __device__ static int unit(int x, int l) { return 4 * x + (l >> 4); }
  __device__ static constexpr int group_block(int x) { return x; }
  __device__ static constexpr int group_reg(int) { return 0; }
};

// A split without tokens: the neutral state, or out = 0 and lse = -inf.
__device__ __forceinline__ void empty_piece(const MlaArgs& a, int b, int row0, int nrows,
                                            const PieceOut& po) {
  const int rows = min(nrows, a.R - row0);
  for (int i = threadIdx.x; i < rows * (kDV / 4); i += kWThreads) {
    const int row = row0 + i / (kDV / 4), x = i % (kDV / 4);
    const size_t br = (size_t)b * a.R + row, sx = po.st_base + (size_t)row * po.st_stride;
    if (po.direct)
      reinterpret_cast<uint2*>(a.out + br * kDV)[x] = make_uint2(0, 0);
    else
      reinterpret_cast<float4*>(a.ws_acc + sx * kDV)[x] = make_float4(0, 0, 0, 0);
    if (x != 0) continue;
    if (po.direct) {
      const int qi = row / a.h_q, hq = row - qi * a.h_q;
      if (a.lse) a.lse[((size_t)b * a.h_q + hq) * a.s_q + qi] = kNegInf;
    } else {
      a.ws_m[sx] = kNegInf;
      a.ws_l[sx] = 0.f;
    }
  }
}

// Runs the pieces of a share: `p` and, while next_piece finds more of the
// share's `units`, those after it, for row group rg. out_of(p, first) is where
// a piece's results go.
template <int RW, int M, typename OutOf>
__device__ __forceinline__ void wide_run(const MlaArgs& a, uint8_t* smem, int rg, Piece p,
                                         int64_t units, OutOf&& out_of) {
  typedef Shape<RW> Sh;
  typedef typename Sh::acc_t acc_t;
  constexpr int kParts = kWWaves / M;                            // dim parts
  constexpr int kBlocks = kDV / Sh::kDimsPerMfma / kParts;       // PV dim blocks of a wave
  constexpr int kPv = kBlocks * Sh::kPvSteps;                    // PV MFMAs of a tile
  static_assert(kPv >= 8 && kPv >= kWVRing + 1, "the exponents are dealt out over the PV MFMAs");
  typedef __attribute__((address_space(3))) uint8_t lds_u8;
  uint32_t tid = threadIdx.x;
  refresh(tid);
  const int lane = (int)(tid & 63);
  const int w = __builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const int part = w / M;
  const uint32_t smem_lds = (uint32_t)(uintptr_t)(lds_u8*)smem;
  // (Lane values that the tile loop does not need are computed again from tid
  // where they are used: nothing but the loop's own values is held through it.)
  auto fresh_lane = [&]() -> int {
    uint32_t t = tid;
    refresh(t);
    return (int)(t & 63);
  };
  const int row0 = (rg * M + w % M) * RW;
  // Lanes past the last row score it again, bit for bit.
  auto query_row = [&](int l) -> int { return min(row0 + l % RW, a.R - 1); };

  // This wave's copies fill row block w of a tile, lane l row l / 8's chunk.
  auto copy_row = [&]() -> int { return (int)((tid >> 3) & 7); };
  uint32_t ro = (uint32_t)((lane >> 3) * kD +
                           8 * ((lane & 7) ^ Sh::swz(8 * w + (lane >> 3)))) * 2u;
  uint32_t qoff = Sh::k_off(lane);
  uint32_t voff = Sh::v_off(lane);

  uint4 qf[Sh::kQ];
  auto load_q = [&](int b) {
    const int l = fresh_lane();
    const uint16_t* src = a.q + ((size_t)b * a.R + query_row(l)) * kD + 8 * (l / RW);
#pragma unroll
    for (int i = 0; i < Sh::kQ; ++i)
      qf[i] = *reinterpret_cast<const uint4*>(src + Sh::q_dim(i));
  };

  // The copies run through the share's tiles ahead of the pieces that use
  // them, across piece boundaries: the cursor is at token c_ts of piece c. At
  // the share's end they repeat one row (a copy count that does not depend on
  // the tile keeps the loop free of branches).
  Piece c = p;
  int64_t c_units = units;
  int c_ts = p.start;
  bool c_live = true;
  uint32_t c_slot = 0;
  const int bs = a.block_size;
  // The first token this wave copies: of its row block, or the tile's first one
  // if the row block lies past the piece's end.
  auto cursor_token = [&]() -> int {
    const int t = c_ts + 8 * w;
    return t < c.end ? t : c_ts;
  };
  auto cursor_block = [&]() -> int {
    // The table is read-only for the launch; through the constant address
    // space the uniform block-id loads are scalar.
    return ((const __attribute__((address_space(4))) int*)(a.block_table + (size_t)c.b *
                                                                             a.max_blocks))
        [gqa::fastdiv((uint32_t)cursor_token(), a.bs_div)];
  };
  auto advance = [&]() {
    c_slot = c_slot + 1 < kWDepth ? c_slot + 1 : 0;
    if (c_ts + kTile < c.end) {
      c_ts += kTile;
    } else if (c_live) {
      c_live = next_piece(a, c, c_units);
      if (c_live) c_ts = c.start;
    }
  };
  struct Source {  // where this wave's copies of the cursor's tile read
    const uint16_t* base;
    uint32_t voff;
    uint32_t slot;
  };
  auto source = [&](int id) -> Source {
    Source s;
    s.slot = smem_lds + c_slot * kTileBytes + (uint32_t)w * kRowBlockBytes;
    const int t = cursor_token();
    const uint32_t lb = gqa::fastdiv((uint32_t)t, a.bs_div);
    s.base = a.kv + ((size_t)id * bs + (t - (int)lb * bs)) * kD;
    // Rows past the piece's end read that token's row (masked later).
    const int valid = c_live ? c.end - c_ts - 8 * w : 0;
    s.voff = copy_row() < valid ? ro : (ro & 0x70u);
    return s;
  };
  auto copy = [&](const Source& s, int i) {
    load_to_lds(s.base + 64 * i, s.voff, __builtin_amdgcn_readfirstlane(s.slot + 1024u * i));
  };
  auto stage = [&]() {
    const Source s = source(cursor_block());
#pragma unroll
    for (int i = 0; i < kWCopies; ++i) copy(s, i);
    advance();
  };

  acc_t o[kBlocks];
  acc_t c4[Sh::kChains];  // QK^T accumulators
  float e[Sh::kEl];       // the exponents of the tile whose probabilities come next
  float lsum = 0.f;      // the row's probabilities, before their rounding to bf16
  float lpv = 0.f;       // and as PV multiplies them
  float nbase = 0.f;     // less the row's reference (log2 units); 0 until its first live tile
  // Largest exponent of this lane's tokens, relative to the reference, and at
  // least 0 (the tile that set it); -inf until the row's first live tile.
  float mrel = kNegInf;
  int d = 0;             // the lane's score i of the tile is live iff tok_off(i) < d

  uint32_t g0 = 0;  // ring slot of the piece's first tile
  auto slot_of = [&](int s) -> uint32_t {
    return smem_lds + ((g0 + (uint32_t)s) % kWDepth) * kTileBytes;
  };
  uint32_t ka[Sh::kKAddr];
  auto set_ka = [&](int s) {
#pragma unroll
    for (int i = 0; i < Sh::kKAddr; ++i) ka[i] = (slot_of(s) + qoff) ^ Sh::k_xor(i);
  };
  u32x4_t kr[kWKRing];
  bf16x8_t vr[kWVRing];
  uint32_t pw[Sh::kEl / 2];  // the tile's probabilities, packed
  auto read_k = [&](int i) {
    kr[i % kWKRing] = lds_load16(ka[Sh::k_addr(i)] + Sh::k_imm(i));
  };
  auto read_v = [&](uint32_t T, int i) {
    vr[i % kWVRing] = Sh::read_v(T, i % kBlocks, i / kBlocks);
  };
  auto qk_mfma = [&](int i) {
    const bf16x8_t kv = as_bf16x8(kr[i % kWKRing]), qv = as_bf16x8(qf[Sh::q_of(i)]);
    if (i < Sh::kChains)
      Sh::qk0(c4[Sh::chain(i)], kv, qv);
    else
      Sh::qk(c4[Sh::chain(i)], kv, qv);
  };
  auto pv_mfma = [&](int i) {
    const int nb = i % kBlocks, t = i / kBlocks;
    o[nb] = Sh::pv(vr[i % kWVRing],
                   as_bf16x8(make_uint4(pw[4 * t], pw[4 * t + 1], pw[4 * t + 2], pw[4 * t + 3])),
                   o[nb]);
  };
  auto settle = [&](int i) { e[i] = Sh::exponent(c4, i, a.scale_log2e, nbase); };
  // PV takes the probabilities rounded to bf16. Its normaliser sums the rounded
  // ones too, so that an output is a weighted mean of its value rows (with the
  // unrounded sum a constant value column of 16 tokens came back up to 1e-3
  // off); lse takes the sum before the rounding (against float64 5e-7 rms; from
  // the rounded ones 2e-5 to 6e-5).
  auto pack_probs = [&](int k, float x, float y) {
    pw[k] = pack_bf16(x, y);
    lsum += x + y;
  };
  auto sum_packed = [&]() {
    asm volatile("" : "+v"(lpv));  // (kept where it is called)
#pragma unroll
    for (int k = 0; k < Sh::kEl / 2; ++k) lpv = gqa::dot2_bf16(pw[k], 0x3F803F80u, lpv);
    asm volatile("" : "+v"(lpv));
  };
  auto max_of = [&]() {
    float m = fmaxf(e[0], e[1]);
#pragma unroll
    for (int i = 2; i < Sh::kEl; i += 2) m = fmaxf(fmaxf(m, e[i]), e[i + 1]);
    return m;
  };
  // A tile with masked tokens, or a row's first live tile (its maximum becomes
  // the row's reference): rare, behind a uniform branch.
  auto check_tile = [&](float mx) {
    if (__builtin_amdgcn_ballot_w64(d <= Sh::kMaxTok || mrel == kNegInf) != 0) {
#pragma unroll
      for (int i = 0; i < Sh::kEl; ++i) e[i] = Sh::tok_off(i) < d ? e[i] : kNegInf;
      const float m = Sh::row_max(max_of());
      const float delta = mrel == kNegInf && m != kNegInf ? m : 0.f;
      mrel = m != kNegInf ? fmaxf(mrel, 0.f) : mrel;
      nbase -= delta;
#pragma unroll
      for (int i = 0; i < Sh::kEl; ++i) e[i] -= delta;
      mx = max_of();
    }
    mrel = fmaxf(mrel, mx);
  };

  int* const votes = reinterpret_cast<int*>(smem + kWRing);
  uint32_t parity = 0;
  bool again = false;  // the piece runs a second time, against its rows' true maxima
  bool first = true;   // the share's first piece
  int id_next = 0;
  auto start = [&]() {  // queries and first tiles of piece p
    load_q(p.b);
    stage();
    stage();
    stage();
    id_next = cursor_block();
    publish_barrier<kWCopies>();  // Q and tiles 0 and 1 landed, tile 2 in flight
  };

  start();
  for (;;) {
    const int ntiles = p.tiles;
    {
      const int l = fresh_lane();
      const int end = a.causal ? p.S - (a.s_q - 1 - query_row(l) / a.h_q) : p.S;
      d = min(p.end, end) - 4 * (l / RW) - p.start;
    }
    lsum = lpv = 0.f;
    if (!again) {
      mrel = kNegInf;
      nbase = 0.f;
    }
#pragma unroll
    for (int nb = 0; nb < kBlocks; ++nb)
#pragma unroll
      for (int i = 0; i < (int)(sizeof(acc_t) / 4); ++i) o[nb][i] = 0.f;
    set_ka(0);
#pragma unroll
    for (int i = 0; i < kWKRing - 1; ++i) read_k(i);
#pragma unroll
    for (int i = 0; i < kWSteps; ++i) {
      if (i + kWKRing - 1 < kWSteps) read_k(i + kWKRing - 1);
      __builtin_amdgcn_sched_barrier(0);
      qk_mfma(i);
      __builtin_amdgcn_sched_barrier(0);
    }
    // (Tied to the accumulators: the exponents below cannot move before it.)
#pragma unroll
    for (int i = 0; i < Sh::kChains; ++i) asm volatile("s_nop 15" : "+v"(c4[i]));
    asm volatile("s_nop 15" : "+v"(c4[0]));
#pragma unroll
    for (int i = 0; i < Sh::kEl; ++i) settle(i);
    check_tile(max_of());
    set_ka(1);
#pragma unroll
    for (int i = 0; i < kWKRing - 1; ++i) read_k(i);
    for (int s = 0; s + 1 < ntiles; ++s) {
      refresh(ro);
      refresh(qoff);
      refresh(voff);
      // QK^T of tile s + 1; the probabilities of tile s and the copies of tile
      // s + 3 between its MFMAs.
      const Source src = source(id_next);
      const uint32_t T = slot_of(s) + voff + 1024u * (uint32_t)(part * (kColBlocks - 1) / kParts);
      float x0 = 0.f, x1 = 0.f;
#pragma unroll
      for (int i = 0; i < kWSteps; ++i) {
        if (i + kWKRing - 1 < kWSteps)
          read_k(i + kWKRing - 1);
        else if (i - (kWSteps - kWKRing + 1) < kWVRing - 1)
          read_v(T, i - (kWSteps - kWKRing + 1));
        __builtin_amdgcn_sched_barrier(0);
        qk_mfma(i);
        if (i % 4 == 0) copy(src, i / 4);
        if (i / 4 < Sh::kEl / 2) {
          const int k = i / 4;
          if (i % 4 == 1) x0 = exp2_fast(e[2 * k]);
          if (i % 4 == 2) x1 = exp2_fast(e[2 * k + 1]);
          if (i % 4 == 3) pack_probs(k, x0, x1);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // PV of tile s; the exponents of tile s + 1 between its MFMAs.
      d -= kTile;
      float mx = kNegInf;
#pragma unroll
      for (int i = 0; i < kPv; ++i) {
        if (i + kWVRing - 1 < kPv) read_v(T, i + kWVRing - 1);
        if (i == kPv - kWVRing + 2) {
          // Every V operand of tile s has been read: its slot is free after
          // this barrier, which also publishes tile s + 2 (tile s + 3 stays in
          // flight).
          advance();
          id_next = cursor_block();
          publish_barrier<kWCopies>();
          set_ka(s + 2);
#pragma unroll
          for (int k = 0; k < kWKRing - 1; ++k) read_k(k);
          // Summed here because the MFMAs wait for these reads anyway (128
          // heads, 128 requests of ~4096 tokens / the same with s_q = 2 / of
          // ~16384 with s_q = 2: 171 / 300 / 1046 us with the 8 instructions
          // between the QK^T MFMAs, 169 / 292 / 992 here, 169 / 290 / 994
          // without them).
          __builtin_amdgcn_sched_barrier(0);
          sum_packed();
        }
        __builtin_amdgcn_sched_barrier(0);
        pv_mfma(i);
        // The exponents start three MFMAs in (the QK^T results have settled by
        // then) and take one slot each, two each where there are few slots.
        constexpr int kPerSlot = kPv >= Sh::kEl + 8 ? 1 : 2;
        constexpr int kLast = 3 + Sh::kEl / kPerSlot;
        if (i >= 3 && i < kLast) {
#pragma unroll
          for (int k = 0; k < kPerSlot; ++k) settle(kPerSlot * (i - 3) + k);
        }
        if constexpr (kPv >= kLast + 5) {  // the maximum over four slots
          constexpr int kQuarter = Sh::kEl / 4;
          if (i > kLast && i <= kLast + 4) {
#pragma unroll
            for (int k = 0; k < kQuarter; ++k)
              mx = fmaxf(mx, e[kQuarter * (i - kLast - 1) + k]);
          }
          __builtin_amdgcn_sched_barrier(0);
          if (i == kLast + 4) check_tile(mx);
        } else {
          __builtin_amdgcn_sched_barrier(0);
          if (i == kPv - 1) check_tile(max_of());
        }
      }
    }
    // The last tile's probabilities and PV, with the copies of the next piece's
    // tile 2 (tiles 0 and 1 are on their way).
    const bool beaten = !again && __builtin_amdgcn_ballot_w64(mrel > kWSlack) != 0;
    if (fresh_lane() == 0) votes[4 * parity + w] = beaten;
    Piece np = p;
    int64_t n_units = units;
    const bool more = next_piece(a, np, n_units);
    {
      const Source src = source(id_next);
      const uint32_t T =
          slot_of(ntiles - 1) + voff + 1024u * (uint32_t)(part * (kColBlocks - 1) / kParts);
#pragma unroll
      for (int k = 0; k < Sh::kEl / 2; ++k)
        pack_probs(k, exp2_fast(e[2 * k]), exp2_fast(e[2 * k + 1]));
#pragma unroll
      for (int i = 0; i < kWVRing - 1; ++i) read_v(T, i);
      __builtin_amdgcn_sched_barrier(0);
      sum_packed();
#pragma unroll
      for (int i = 0; i < kPv; ++i) {
        if (i + kWVRing - 1 < kPv) read_v(T, i + kWVRing - 1);
        __builtin_amdgcn_sched_barrier(0);
        pv_mfma(i);
        if constexpr (kPv >= 3 * kWCopies) {
          if (i % 3 == 0 && i / 3 < kWCopies) copy(src, i / 3);
        } else {
          if (i < kWCopies) copy(src, i);
          if (i == kPv - 1) {
#pragma unroll
            for (int k = kPv; k < kWCopies; ++k) copy(src, k);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      advance();
      id_next = cursor_block();
      publish_barrier<kWCopies>();
    }
    g0 = (g0 + (uint32_t)ntiles) % kWDepth;
    const int4 v = *reinterpret_cast<const int4*>(votes + 4 * parity);
    parity ^= 1;
    if (__builtin_amdgcn_readfirstlane(v.x | v.y | v.z | v.w) != 0) {
      // Some row's later tile beat its reference by more than kWSlack: the
      // piece runs again, the copies start over at its first tile.
      nbase -= fmaxf(Sh::row_max(mrel), 0.f);
      again = true;
      publish_barrier<0>();
      c = p;
      c_units = units;
      c_ts = p.start;
      c_live = true;
      c_slot = g0 = 0;
      start();
      continue;
    }
    again = false;

    // Results, 64 dims at a time through the wave's row block of the free ring
    // slot (the one its next copies fill): lanes hold 4 dims of one row each,
    // the stores take 256 bytes (128 of out) of 4 rows each. Storing the
    // accumulators as they lie, 16 bytes of 32 rows per instruction, took 10.5
    // us per piece of 128 rows, this 5.5.
    const PieceOut po = out_of(p, first);
    const bool direct = uniform((int)po.direct) != 0;
    if (row0 < a.R) {
      const float L = Sh::row_sum(lsum), Lpv = Sh::row_sum(lpv);
      const float inv = L > 0.f ? 1.f / Lpv : 0.f;
      const int l = fresh_lane();
      const int row = row0 + l % RW;
      if (row < a.R && l < RW && part == 0) {
        // lse; or a state's m (natural-log units), for a sum of Lpv, what its
        // rows are a weighted sum by: m + ln Lpv is the piece's lse. (Rows scaled
        // to a sum of L instead cost 0.1 to 0.2 us of a call.)
        const float x = L > 0.f ? logf(direct ? L : L * inv) - nbase * kLn2 : kNegInf;
        if (!direct) {
          const size_t sx = po.st_base + (size_t)row * po.st_stride;
          a.ws_m[sx] = x;
          a.ws_l[sx] = Lpv;
        } else if (a.lse) {
          const int qi = row / a.h_q, hq = row - qi * a.h_q;
          a.lse[((size_t)p.b * a.h_q + hq) * a.s_q + qi] = x;
        }
      }
      const uint32_t buf =
          smem_lds + (g0 + kWDepth - 1) % kWDepth * kTileBytes + (uint32_t)w * kRowBlockBytes;
      const uint32_t dst = buf + (uint32_t)(l % RW) * 256;
      // This lane's rows 4 i + l / 16: what it reads back and stores. (Past the
      // last row: the last row's values once more.)
      float iv[RW / 4];
      uint32_t off[RW / 4];
#pragma unroll
      for (int i = 0; i < RW / 4; ++i) {
        const int r = 4 * i + (l >> 4);
        iv[i] = __shfl(inv, r, 64);
        off[i] = (uint32_t)min(r, a.R - 1 - row0);
      }
      const int dim0 = part * (kDV / kParts) + 4 * (l & 15);
      uint16_t* const out0 = a.out + ((size_t)p.b * a.R + row0) * kDV + dim0;
      float* const acc0 = a.ws_acc + (po.st_base + (size_t)row0 * po.st_stride) * kDV + dim0;
      const uint32_t pitch = (uint32_t)po.st_stride * kDV;
      constexpr int kChunkBlocks = 64 / Sh::kDimsPerMfma;
#pragma unroll
      for (int k = 0; k < kBlocks / kChunkBlocks; ++k) {
        wave_lds_sync();
#pragma unroll
        for (int x = 0; x < Sh::kGroups; ++x) {
          const acc_t& v = o[kChunkBlocks * k + Sh::group_block(x)];
          const int q = Sh::group_reg(x);
          lds_store16(dst + 16u * (uint32_t)(Sh::unit(x, l) ^ (l & 15)),
                      u32x4_t{__float_as_uint(v[q]), __float_as_uint(v[q + 1]),
                              __float_as_uint(v[q + 2]), __float_as_uint(v[q + 3])});
        }
        wave_lds_sync();
        u32x4_t v[RW / 4];
#pragma unroll
        for (int i = 0; i < RW / 4; ++i) {
          const int r = 4 * i + (l >> 4);
          v[i] = lds_load16(buf + (uint32_t)r * 256 + 16u * (uint32_t)((l ^ r) & 15));
        }
        if (direct) {
#pragma unroll
          for (int i = 0; i < RW / 4; ++i)
            *reinterpret_cast<uint2*>(out0 + off[i] * kDV + 64 * k) =
                make_uint2(pack_bf16(__uint_as_float(v[i].x) * iv[i], __uint_as_float(v[i].y) * iv[i]),
                           pack_bf16(__uint_as_float(v[i].z) * iv[i], __uint_as_float(v[i].w) * iv[i]));
        } else {
#pragma unroll
          for (int i = 0; i < RW / 4; ++i)
            *reinterpret_cast<u32x4_t*>(acc0 + off[i] * pitch + 64 * k) = v[i];
        }
      }
    }
    wave_lds_sync();
    if (!more) break;
    first = false;
    p = np;
    units = n_units;
    load_q(p.b);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // no copy outlives the workgroup
}

// Fixed splits: workgroup (rg, b, split).
template <int RW, int M>
__global__ __launch_bounds__(kWThreads, 1) void mla_wide_kernel(const MlaArgs a) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kWLds];
  const int rg = blockIdx.x, b = blockIdx.y, split = blockIdx.z;
  const int S = live_len(a, b);
  const int ns = a.num_splits;
  const int chunk = ((S + ns - 1) / ns + (kTile - 1)) & ~(kTile - 1);
  const int start = min(split * chunk, S), end = min(S, start + chunk);
  PieceOut po;
  po.direct = ns == 1;
  po.st_base = (size_t)b * a.R * ns + split;
  po.st_stride = ns;
  if (start >= end) {
    empty_piece(a, b, rg * M * RW, M * RW, po);
    return;
  }
  const Piece p{b, S, start, end, (end - start + kTile - 1) / kTile};
  wide_run<RW, M>(a, smem, rg, p, p.tiles, [&](const Piece&, bool) { return po; });
}

// Token-balanced: workgroup (w, rg), share w of row group rg.
template <int RW, int M>
__global__ __launch_bounds__(kWThreads, 1) void mla_wide_balanced_kernel(const MlaArgs a) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kWLds];
  const int w = blockIdx.x, rg = blockIdx.y;
  const SharePlan sp = plan_share<kWThreads>(a, w, reinterpret_cast<uint64_t*>(smem), true,
                                             w == 0 && rg == 0);
  if (sp.units <= 0) return;
  __syncthreads();
  wide_run<RW, M>(a, smem, rg, piece_of(sp.b, sp.S, sp.ts, sp.units), sp.units,
                  [&](const Piece& p, bool first) {
                    PieceOut po;
                    po.direct = p.start == 0 && p.end == p.S;
                    po.st_base = (size_t)(2 * w + (first ? 0 : 1)) * a.R;
                    po.st_stride = 1;
                    return po;
                  });
}

}  // namespace

hipError_t launch_wide_splitkv(const MlaArgs& a, int rows, hipStream_t stream) {
  const dim3 grid(row_groups(a.R, rows), a.B, a.num_splits);
  switch (rows) {
    case 16:
      hipLaunchKernelGGL((mla_wide_kernel<16, 1>), grid, dim3(kWThreads), 0, stream, a);
      break;
    case 32:
      hipLaunchKernelGGL((mla_wide_kernel<16, 2>), grid, dim3(kWThreads), 0, stream, a);
      break;
    case 64:
      hipLaunchKernelGGL((mla_wide_kernel<16, 4>), grid, dim3(kWThreads), 0, stream, a);
      break;
    default:
      hipLaunchKernelGGL((mla_wide_kernel<32, 4>), grid, dim3(kWThreads), 0, stream, a);
  }
  return hipGetLastError();
}

hipError_t launch_wide_balanced(const MlaArgs& a, int rows, hipStream_t stream) {
  const dim3 grid(a.nshare, row_groups(a.R, rows));
  switch (rows) {
    case 16:
      hipLaunchKernelGGL((mla_wide_balanced_kernel<16, 1>), grid, dim3(kWThreads), 0, stream, a);
      break;
    case 32:
      hipLaunchKernelGGL((mla_wide_balanced_kernel<16, 2>), grid, dim3(kWThreads), 0, stream, a);
      break;
    case 64:
      hipLaunchKernelGGL((mla_wide_balanced_kernel<16, 4>), grid, dim3(kWThreads), 0, stream, a);
      break;
    default:
      hipLaunchKernelGGL((mla_wide_balanced_kernel<32, 4>), grid, dim3(kWThreads), 0, stream, a);
  }
  return hipGetLastError();
}

}  // namespace mla

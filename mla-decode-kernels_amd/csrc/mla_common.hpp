// What the MLA decode kernels share (mla_decode.hip, mla_decode_wide.hip): sizes,
// launch arguments, LDS access by address, HBM -> LDS copies.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gqa_device.hpp"
#include "mla_decode.h"

namespace mla {

using gqa::exp2_fast;
using gqa::f32_to_bf16_bits;
using gqa::FastDiv;
using gqa::kLn2;
using gqa::kLog2e;
using gqa::kNegInf;

constexpr int kD = MLA_DECODE_HEAD_DIM;     // 576
constexpr int kDV = MLA_DECODE_HEAD_DIM_V;  // 512
constexpr int kTile = 32;                   // tokens per tile
// A tile in the LDS: 4 row blocks of 8 tokens, each 9 column blocks of 64 dims
// (8 rows x 128 bytes = 1 KiB, what one copy instruction fills).
constexpr int kColBlocks = kD / 64;
constexpr int kRowBlockBytes = kColBlocks * 1024;
constexpr int kTileBytes = 4 * kRowBlockBytes;  // 36 KiB

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) bf16x4_t lds_bf16x4_t;

struct MlaArgs {
  const uint16_t* q;
  const uint16_t* kv;
  const int* block_table;
  const int* seq_lens;
  uint16_t* out;
  float* lse;
  float* ws_acc;  // [B, R, ns, 512]
  float* ws_m;    // [B, R, ns] natural-log units
  float* ws_l;
  uint64_t* pre;        // balanced launch: unit prefix sums [B + 2] (written by the split kernel)
  int B, s_q, h_q, R, block_size, max_blocks, num_splits, causal, nshare;
  int piece_cost;       // balanced launch: what a piece weighs besides its tiles, in tiles
  FastDiv bs_div;
  float scale_log2e;
};

__device__ __forceinline__ bf16x8_t as_bf16x8(const uint4& u) {
  return __builtin_bit_cast(bf16x8_t, u);
}

// Direct HBM -> LDS copies of 16 bytes per lane (global_load_lds_dwordx4):
// lane x's bytes land at LDS byte address lds + 16 x; lds must be
// wave-uniform. They are issued through inline assembly so that the compiler
// does not tie its LDS reads of the other ring slots to these loads'
// completion (it would wait for every load in flight before each read);
// completion is awaited explicitly with s_waitcnt vmcnt before the barrier
// that publishes a tile. The first form addresses base + voff (a uniform
// 64-bit base, a 32-bit per-lane offset); the second a per-lane address.
// On gfx9-family GPUs an LDS-DMA instruction needs one wait state after an
// SALU write of M0; the compiler inserts it for its own LDS-DMA code but does
// not look inside inline assembly, hence the s_nop (measured cost: up to ~3 %
// on the matrix-bound s_q = 2 workloads).
// M0 is a register the compiler reserves (hipcc notes the clobber as such and
// will not restore it): these kernels rely on the compiler emitting no M0 use
// of its own, which tests/test_mla_codegen.py checks on the generated code,
// together with the spill-free and wait-free tile loops.
__device__ __forceinline__ void load_to_lds(const uint16_t* base, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt"
               :
               : "v"(voff), "s"(base), "s"(lds)
               : "memory", "m0");
}
__device__ __forceinline__ void load_to_lds(const uint16_t* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt"
               :
               : "v"(src), "s"(lds)
               : "memory", "m0");
}

// Waits until at most kInFlight of this wave's direct loads are outstanding
// (they complete in issue order) and its LDS writes are done, then joins the
// workgroup barrier; LDS reads and writes are not moved across it.
template <int kInFlight>
__device__ __forceinline__ void publish_barrier() {
  static_assert(kInFlight >= 0 && kInFlight < 64, "vmcnt holds 6 bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(kInFlight) : "memory");
}

// Where a piece's results go: normalised rows to out and lse (direct), or
// unnormalised states, row r of the piece's request at index
// st_base + r * st_stride of ws_acc (x 512), ws_m and ws_l.
struct PieceOut {
  bool direct;
  size_t st_base;
  int st_stride;
};

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) u32x4_t lds_u32x4_t;
typedef __attribute__((address_space(3))) u32x2_t lds_u32x2_t;

// LDS accesses by 32-bit LDS byte address.
__device__ __forceinline__ u32x4_t lds_load16(uint32_t addr) {
  return *(const lds_u32x4_t*)(uintptr_t)addr;
}
__device__ __forceinline__ void lds_store8(uint32_t addr, u32x2_t v) {
  *(lds_u32x2_t*)(uintptr_t)addr = v;
}
__device__ __forceinline__ void lds_store16(uint32_t addr, u32x4_t v) {
  *(lds_u32x4_t*)(uintptr_t)addr = v;
}
// Hands LDS data from some lanes of a wave to others: waits for the wave's LDS
// operations (vmcnt untouched) and keeps memory accesses from moving across.
__device__ __forceinline__ void wave_lds_sync() {
  asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
  __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ bf16x4_t lds_load_tr(uint32_t addr) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4_t*)(uintptr_t)addr);
}
__device__ __forceinline__ bf16x8_t as_bf16x8(const u32x4_t& u) {
  return __builtin_bit_cast(bf16x8_t, u);
}

// Hands x back through an empty asm statement, so that the compiler treats it
// as a new value: applied to the lane's operand offsets at the top of every
// interval, it keeps values derived from them (offset ^ constant, one per
// matrix step) from being hoisted out of the tile loop, where they would
// outgrow the register budget of two waves per SIMD.
__device__ __forceinline__ void refresh(uint32_t& x) { asm volatile("" : "+v"(x)); }

}  // namespace mla

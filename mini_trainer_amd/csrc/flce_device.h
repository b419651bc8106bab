// Device-side building blocks of the fused linear + cross-entropy kernels
// (gfx950 / CDNA4 only).
//
// LDS tile layout (operand rows contiguous along K)
//   A tile holds rows x 128 bytes of K.  A row is 8 chunks of 16 bytes.
//   Rows r and r + 8 of a 16-row group share one 256-byte line (halves 0/1);
//   the chunk index is XOR-swizzled with (r & 7).  With this layout the
//   16-lane groups of an MFMA operand read (16 consecutive rows, one chunk)
//   and the 8-lane / 16-lane groups of the LDS DMA that fills it touch
//   distinct 16-byte slots of a 256-byte window, so neither 32- nor 64-bank
//   LDS organisations see conflicts.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mtf {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

typedef __attribute__((address_space(3))) void lds_void_t;

__device__ __forceinline__ uint32_t lane_id() { return threadIdx.x & 63u; }
__device__ __forceinline__ uint32_t wave_id() {
  return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr float kNegBig = -1.0e30f;  // "minus infinity" that keeps exp2(a - b) finite

// Byte offset of (row, logical 16-byte chunk) inside one tile.
__device__ __forceinline__ uint32_t tile_off(uint32_t row, uint32_t chunk) {
  return ((row >> 4) << 11) | ((row & 7u) << 8) | (((row >> 3) & 1u) << 7) |
         (((chunk ^ row) & 7u) << 4);
}

__device__ __forceinline__ u32x4_t lds_read16(const char* lds, uint32_t off) {
  return *reinterpret_cast<const u32x4_t*>(lds + off);
}
__device__ __forceinline__ void lds_write16(char* lds, uint32_t off, u32x4_t v) {
  *reinterpret_cast<u32x4_t*>(lds + off) = v;
}

// One 16-byte chunk of bf16 A and B per lane -> 16x16 fp32 fragment update.
__device__ __forceinline__ f32x4_t mma_chunk(u32x4_t a, u32x4_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                  __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

// Two fp32 -> packed bf16 pair (v_cvt_pk_bf16_f32: round to nearest even).
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t));
}

// Values of (lo, hi) after a round trip through bf16.
__device__ __forceinline__ void round_pair(float& lo, float& hi) {
  const uint32_t p = pack_bf16x2(lo, hi);
  lo = __builtin_bit_cast(float, p << 16);
  hi = __builtin_bit_cast(float, p & 0xffff0000u);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fast_log2(float x) { return __builtin_amdgcn_logf(x); }

// tanh(x) from exp2: 1 - 2 / (exp(2|x|) + 1), sign restored.  The quotient is
// the reciprocal instruction (1 ulp) and one Newton step (rounded like a
// division but for its last bit) instead of the division's ten instructions:
// softcapped forward -3.5%, recompute -6%, the in-place pass over kept logits
// -16% (121 -> 101 us for 2400 x 50257).  |x| is capped where tanh is 1 in fp32,
// so that the step never sees an infinity.  NaN stays NaN.
__device__ __forceinline__ float tanh_approx(float x) {
  const float ax = fabsf(x);
  const float d = fast_exp2((ax > 20.f ? 20.f : ax) * (2.0f * kLog2e)) + 1.0f;
  float r = __builtin_amdgcn_rcpf(d);
  r = fmaf(fmaf(-d, r, 1.0f), r, r);
  return copysignf(fmaf(-2.0f, r, 1.0f), x);
}

// Online log-sum-exp state merge in the log2 domain: (m, d) represents
// d * 2^m.
__device__ __forceinline__ void lse_merge(float& m, float& d, float m2, float d2) {
  float mn = fmaxf(m, m2);
  d = d * fast_exp2(m - mn) + d2 * fast_exp2(m2 - mn);
  m = mn;
}

// Workgroup id -> logical tile id such that the workgroups resident on one
// XCD (hardware dispatches id i to XCD i % 8) get a contiguous logical range.
// A bijection of [0, nwg) for any nwg: XCD x < nwg % 8 owns one id more than
// the others, and the ranges are laid out XCD after XCD.
__device__ __forceinline__ uint32_t xcd_remap(uint32_t bid, uint32_t nwg) {
  const uint32_t kXcd = 8;
  const uint32_t q = nwg / kXcd, r = nwg % kXcd;
  const uint32_t x = bid % kXcd, i = bid / kXcd;
  return x < r ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
}

// Logical tile id -> (tile_m, tile_n) walking groups of `group_m` tile rows
// column by column, so concurrently running tiles share operand panels.
__device__ __forceinline__ void grouped_tile(uint32_t lid, uint32_t tiles_m, uint32_t tiles_n,
                                             uint32_t group_m, uint32_t& tm, uint32_t& tn) {
  uint32_t per_group = group_m * tiles_n;
  uint32_t g = lid / per_group;
  uint32_t first_m = g * group_m;
  uint32_t gm = tiles_m - first_m < group_m ? tiles_m - first_m : group_m;
  uint32_t in = lid - g * per_group;
  tm = first_m + in % gm;
  tn = in / gm;
  // lid is uniform (a workgroup's tile index), but the divisions above run
  // in vector registers and the compiler does not always prove the results
  // uniform; a pointer or buffer resource built from them then becomes a
  // per-lane waterfall loop around every memory instruction that uses it.
  tm = __builtin_amdgcn_readfirstlane(tm);
  tn = __builtin_amdgcn_readfirstlane(tn);
}

}  // namespace mtf

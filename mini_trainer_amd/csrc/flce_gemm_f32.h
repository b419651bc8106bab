// Operands and MFMA main loop of the fp32 GEMM-shaped kernels (gfx950).
//
// Bound: the fp32 matrix rate (v_mfma_f32_16x16x4_f32, 64 flop per cycle and
// SIMD: 157 TFLOP/s on 256 CUs at 2.4 GHz; a large library product reaches
// 151).  A 128 x 128 output tile is multiplied by 4 waves of 64 x 64 (64
// accumulators each), K advances in stages of 32 fp32 (128 bytes per operand
// row), double-buffered in 64 KiB of LDS, so two workgroups share a CU: a
// stage is 4096 MFMA cycles per wave, and the second workgroup's MFMAs cover
// the first one's barrier, LDS reads and epilogue.  The tile is half as wide
// as the bf16 kernels' because an fp32 MFMA does a sixteenth of the work per
// cycle: operand traffic does not bound it, while small tiles waste less on
// a hidden size that is not a multiple of 256 and split evenly over the CUs.
//
// LDS tile formats (per operand and stage, 16 KiB):
//   KC  rows contiguous along K: tile_off(row, chunk) of flce_device.h; lane l
//       reads, for K half kk and fragment f, the 16-byte chunk kk * 4 + l / 16
//       of row f * 16 + l % 16: elements e = 0..3 are K = 16 kk + 4 (l / 16) + e.
//   TR  operand stored K-major (row = K entry): 32 K rows of 128 columns, 512
//       bytes each, as they lie in memory.  Lane l reads, for K half kk and
//       element e, columns 4 (l % 16) .. + 3 of K row 16 kk + 4 (l / 16) + e:
//       column j of the four belongs to fragment j, whose index i along the
//       tile is column 4 i + j.  No transpose is needed, only this column
//       order in the epilogue.  16 lanes read 256 contiguous bytes.
// MFMA (kk, e) pairs K entry 16 kk + 4 (l / 16) + e of both operands.
//
// Accumulator layout (the B fragment is the MFMA's first operand), lane l,
// element r of fragment (fm, fn), relative to the wave's 64 x 64 block:
//   row (A)  KC: 16 fm + l % 16          TR: 4 (l % 16) + fm
//   col (B)  KC: 16 fn + 4 (l / 16) + r  TR: 16 (l / 16) + 4 r + fn
#pragma once

#include "flce_device.h"

namespace mtf {

constexpr int kThreadsF = 256;
constexpr int kTileF = 128;               // output tile rows and columns
constexpr int kBKF = 32;                  // K elements per stage
constexpr int kOperandF = kTileF * 128;   // one operand, one stage: 16 KiB
constexpr int kStageF = 2 * kOperandF;    // A + B
constexpr int kLdsF = 2 * kStageF;        // double buffered: 64 KiB
constexpr int kNIF = 4;                   // 1 KiB DMA instructions per wave and operand

#define MT_F32_KERNEL __global__ __launch_bounds__(256, 2)

// Operand whose rows are contiguous along K (rows gathered by address).
struct KcF {
  static constexpr bool kTr = false;
  const char* p[kNIF];
  uint32_t frag[2];
  uint32_t tail_bad;  // bit i: DMA i's chunk lies past K in the last stage

  __device__ __forceinline__ static uint32_t row_of(uint32_t i) {
    const uint32_t l = lane_id(), q = wave_id() * kNIF + i;
    return (q >> 1) * 16 + ((l >> 3) & 1u) * 8 + (q & 1u) * 4 + (l >> 4);
  }
  __device__ __forceinline__ static uint32_t chunk_of(uint32_t i) {
    const uint32_t l = lane_id(), q = wave_id() * kNIF + i;
    return (l & 7u) ^ ((q & 1u) * 4 + (l >> 4));
  }
  // row_ptr(r): address of K element 0 of tile row r; wave0: first tile row of
  // this wave's block
  template <class RowPtr>
  __device__ __forceinline__ void init(RowPtr row_ptr, uint32_t wave0) {
#pragma unroll
    for (uint32_t i = 0; i < kNIF; ++i) p[i] = row_ptr(row_of(i)) + chunk_of(i) * 16u;
    const uint32_t l = lane_id();
#pragma unroll
    for (uint32_t kk = 0; kk < 2; ++kk) frag[kk] = tile_off(wave0 + (l & 15u), kk * 4 + (l >> 4));
    tail_bad = 0;
  }
  // c_lim: 16-byte chunks (of 8) of the last K stage that lie below K
  __device__ __forceinline__ void set_tail(uint32_t c_lim) {
    uint32_t m = 0;
#pragma unroll
    for (uint32_t i = 0; i < kNIF; ++i) m |= (chunk_of(i) >= c_lim ? 1u : 0u) << i;
    tail_bad = m;
  }
  // tail (the last, partial stage): chunks past K re-read chunk 0 of their row
  // (in bounds); the fragments that hold them are zeroed after the LDS read
  __device__ __forceinline__ void issue(char* tile, int kt, bool tail) const {
    const int64_t koff = (int64_t)kt * 128;
#pragma unroll
    for (uint32_t i = 0; i < kNIF; ++i) {
      const char* src = tail && ((tail_bad >> i) & 1u) ? p[i] - chunk_of(i) * 16u : p[i] + koff;
      __builtin_amdgcn_global_load_lds(src, (lds_void_t*)(tile + (wave_id() * kNIF + i) * 1024u),
                                       16, 0, 0);
    }
  }
  __device__ __forceinline__ f32x4_t read(const char* tile, int kk, int f) const {
    return __builtin_bit_cast(f32x4_t, lds_read16(tile, frag[kk] + (uint32_t)f * 2048u));
  }
};

// Operand stored K-major: row-major [K, 128-column tile].
struct TrF {
  static constexpr bool kTr = true;
  const char* base;   // K row 0, tile column 0, plus this lane's column offset
  int64_t ld_b;
  int32_t k_limit;    // K rows at or past it read row k_limit - 1 (their products
                      // meet zeros or are discarded)
  uint32_t frag;

  // m_valid: tile columns that exist (a multiple of 4; the others read column
  // 0 and are discarded by the epilogue)
  __device__ __forceinline__ void init(const char* base_, int64_t ld_b_, int32_t k_limit_,
                                       int32_t m_valid, uint32_t wave0) {
    const uint32_t l = lane_id();
    const int32_t m0 = (int32_t)(l & 31u) * 4;
    base = base_ + (m0 < m_valid ? m0 * 4 : 0);
    ld_b = ld_b_;
    k_limit = k_limit_;
    frag = (l >> 4) * 4u * 512u + wave0 * 4u + (l & 15u) * 16u;
  }
  __device__ __forceinline__ void issue(char* tile, int kt, bool) const {
    const uint32_t l = lane_id();
#pragma unroll
    for (uint32_t i = 0; i < kNIF; ++i) {
      const uint32_t q = wave_id() * kNIF + i;
      int32_t k = kt * kBKF + (int32_t)(2u * q + (l >> 5));
      k = k < k_limit ? k : k_limit - 1;
      __builtin_amdgcn_global_load_lds(base + (int64_t)k * ld_b, (lds_void_t*)(tile + q * 1024u), 16,
                                       0, 0);
    }
  }
  // element e = f of K half kk: one value for each of the four fragments
  __device__ __forceinline__ f32x4_t read(const char* tile, int kk, int f) const {
    return __builtin_bit_cast(
        f32x4_t, lds_read16(tile, frag + (uint32_t)(kk * 16 + f) * 512u));
  }
};

// Element e of fragment f from an operand's four registers of one K half.
template <class Op>
__device__ __forceinline__ float f32_elem(const f32x4_t (&r)[4], int f, int e) {
  return Op::kTr ? r[e][f] : r[f][e];
}

// acc = sum over KT stages of A_tile * B_tile^T.  c_lim < 8 (both operands
// KcF): the last stage holds only c_lim of its 8 chunks below K.  Ends with
// every wave past its last LDS read.
// kLong (dX, dW: K is a vocabulary block or the counted tokens): the sum is
// kept in two levels, runs of kFoldF stages (256 K entries) added up
// separately, so that its rounding error grows with the square root of the run
// and of the number of runs, not of K (dX over 35k columns in one run: 1.4e-6
// of its norm off the 64-bit result, in runs of 256: 4e-7).
constexpr int kFoldF = 8;
template <bool kKTail, bool kLong, class A, class B>
__device__ __forceinline__ void mainloop_f32(char* lds, f32x4_t (&acc)[4][4], const A& a, const B& b,
                                             int KT, uint32_t c_lim = 8) {
#pragma unroll
  for (int fm = 0; fm < 4; ++fm)
#pragma unroll
    for (int fn = 0; fn < 4; ++fn) acc[fm][fn] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (KT <= 0) return;
  f32x4_t total[4][4];
  if constexpr (kLong) {
#pragma unroll
    for (int fm = 0; fm < 4; ++fm)
#pragma unroll
      for (int fn = 0; fn < 4; ++fn) total[fm][fn] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  a.issue(lds, 0, kKTail && KT == 1);
  b.issue(lds + kOperandF, 0, kKTail && KT == 1);
  __syncthreads();
  for (int kt = 0; kt < KT; ++kt) {
    char* cur = lds + (kt & 1) * kStageF;
    char* nxt = lds + ((kt + 1) & 1) * kStageF;
    if (kt + 1 < KT) {
      a.issue(nxt, kt + 1, kKTail && kt + 1 == KT - 1);
      b.issue(nxt + kOperandF, kt + 1, kKTail && kt + 1 == KT - 1);
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      f32x4_t fa[4], fb[4];
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        fa[f] = a.read(cur, kk, f);
        fb[f] = b.read(cur + kOperandF, kk, f);
      }
      if (kKTail && kt == KT - 1 && (uint32_t)kk * 4u + (lane_id() >> 4) >= c_lim) {
#pragma unroll
        for (int f = 0; f < 4; ++f) {
          fa[f] = f32x4_t{0.f, 0.f, 0.f, 0.f};
          fb[f] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
      }
      // sixteen independent accumulators between two MFMAs on the same one
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int fm = 0; fm < 4; ++fm)
#pragma unroll
          for (int fn = 0; fn < 4; ++fn)
            acc[fm][fn] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                f32_elem<B>(fb, fn, e), f32_elem<A>(fa, fm, e), acc[fm][fn], 0, 0, 0);
    }
    __syncthreads();
    if (kLong && (kt % kFoldF == kFoldF - 1 || kt == KT - 1)) {
#pragma unroll
      for (int fm = 0; fm < 4; ++fm)
#pragma unroll
        for (int fn = 0; fn < 4; ++fn) {
          total[fm][fn] += acc[fm][fn];
          acc[fm][fn] = kt == KT - 1 ? total[fm][fn] : f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
    }
  }
}

}  // namespace mtf

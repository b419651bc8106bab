// fp32 kernels of the fused LM-head linear + per-token cross-entropy: 128 x
// 128 output tiles on the main loop of flce_gemm_f32.h, two workgroups per CU.
// Arguments and arithmetic as the bf16 kernels' (flce_kernels_bf16.h), with
// logits and G kept in fp32.
#pragma once

#include "flce_gemm_f32.h"
#include "flce_kernels.h"

namespace mtf {

// Wave (wm, wn) of the 2 x 2 wave grid and this lane's place in its block.
struct CoordsF {
  uint32_t lane, wm, wn;
  __device__ __forceinline__ CoordsF() {
    lane = lane_id();
    const uint32_t w = wave_id();
    wm = w >> 1;
    wn = w & 1u;
  }
  // tile-local row of fragment fm (A a KcF operand)
  __device__ __forceinline__ int row(int fm) const { return wm * 64 + fm * 16 + (lane & 15u); }
  // tile-local row of fragment fm (A a TrF operand)
  __device__ __forceinline__ int row_tr(int fm) const { return wm * 64 + 4 * (lane & 15u) + fm; }
  // tile-local column of element 0 of fragment fn (B a KcF operand)
  __device__ __forceinline__ int col(int fn) const { return wn * 64 + fn * 16 + 4 * (lane >> 4); }
  // tile-local column of fragment 0, element r (B a TrF operand)
  __device__ __forceinline__ int col_tr(int r) const { return wn * 64 + 16 * (lane >> 4) + 4 * r; }
};

// K stages of `k` entries and the 16-byte chunks of the last one below k.
__device__ __forceinline__ int stages_f32(int32_t k, uint32_t& c_lim) {
  const int KT = (k + kBKF - 1) / kBKF;
  c_lim = (uint32_t)(k - (KT - 1) * kBKF) / 4u;
  return KT;
}

// ---------------------------------------------------------------------------
// Forward: workgroup (tm, ts) multiplies row tile tm with the vocabulary tiles
// of split ts, keeping each row's running (max, sum) in registers; no logits
// are written.  kKTail: H is not a multiple of 32.
// ---------------------------------------------------------------------------
template <bool kCap>
__device__ __forceinline__ void fwd_tile_f32(const f32x4_t (&acc)[4][4], float (&m2)[4],
                                             float (&d)[4], const int32_t (&lbl)[4],
                                             const int32_t (&rglob)[4], int32_t vrow0,
                                             const CoordsF& ec, const FwdArgs& a) {
  const int32_t ncol0 = vrow0 + ec.col(0);
  const float cap = a.softcap, inv_cap = kCap ? 1.0f / a.softcap : 0.f;
#pragma unroll
  for (int fm = 0; fm < 4; ++fm) {
    const int32_t rel = lbl[fm] - ncol0;  // the lane holds columns 16 fn + 0..3 from ncol0
    float v[4][4];
    float tmax = -INFINITY, hit = 0.f;
#pragma unroll
    for (int fn = 0; fn < 4; ++fn)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float x = acc[fm][fn][r];
        if (kCap) x = cap * tanh_approx(x * inv_cap);
        x = ncol0 + fn * 16 + r < a.V ? x : -INFINITY;
        hit = rel == fn * 16 + r ? x : hit;
        v[fn][r] = x;
        tmax = fmaxf(tmax, x);
      }
    const float mn = fmaxf(m2[fm], tmax * kLog2e);
    float s = 0.f;
#pragma unroll
    for (int fn = 0; fn < 4; ++fn)
#pragma unroll
      for (int r = 0; r < 4; ++r) s += fast_exp2(fmaf(v[fn][r], kLog2e, -mn));
    d[fm] = fmaf(d[fm], fast_exp2(m2[fm] - mn), s);
    m2[fm] = mn;
    if (lane_holds<4>(rel) && rglob[fm] < a.N) a.xy[rglob[fm]] = hit;
  }
}

template <bool kKTail>
MT_F32_KERNEL void fwd_f32_kernel(FwdArgs a) {
  __shared__ __attribute__((aligned(1024))) char lds[kLdsF];
  uint32_t tm, ts;
  grouped_tile(xcd_remap(blockIdx.x, gridDim.x), a.tiles_m, a.splits, 8, tm, ts);
  const CoordsF ec;
  const int32_t row0 = (int32_t)tm * kTileF;
  uint32_t c_lim;
  const int KT = stages_f32(a.H, c_lim);
  KcF A, B;
  A.init([&](uint32_t r) __attribute__((always_inline)) {
    int32_t rr = row0 + (int32_t)r;
    rr = rr < a.N ? rr : a.N - 1;
    return a.X + (int64_t)a.row_index[rr] * a.ldx_b;
  }, ec.wm * 64);
  if constexpr (kKTail) A.set_tail(c_lim);
  int32_t lbl[4], rglob[4];
  float m2[4], d[4];
#pragma unroll
  for (int fm = 0; fm < 4; ++fm) {
    rglob[fm] = row0 + ec.row(fm);
    lbl[fm] = rglob[fm] < a.N ? a.row_label[rglob[fm]] : -1;
    m2[fm] = kNegBig;
    d[fm] = 0.f;
  }
  const int vt0 = (int)ts * a.vt_per_split, vt1 = min(vt0 + a.vt_per_split, a.vt_total);
  for (int vt = vt0; vt < vt1; ++vt) {
    const int32_t vrow0 = vt * kTileF;
    B.init([&](uint32_t r) __attribute__((always_inline)) {
      int32_t v = vrow0 + (int32_t)r;
      v = v < a.V ? v : a.V - 1;
      return a.W + (int64_t)v * a.ldw_b;
    }, ec.wn * 64);
    if constexpr (kKTail) B.set_tail(c_lim);
    f32x4_t acc[4][4];
    mainloop_f32<kKTail, false>(lds, acc, A, B, KT, c_lim);
    if (a.softcap > 0.f) fwd_tile_f32<true>(acc, m2, d, lbl, rglob, vrow0, ec, a);
    else fwd_tile_f32<false>(acc, m2, d, lbl, rglob, vrow0, ec, a);
  }
  // the four lanes, then the two waves that share a row
#pragma unroll
  for (int fm = 0; fm < 4; ++fm) {
    lse_merge(m2[fm], d[fm], xor16(m2[fm]), xor16(d[fm]));
    lse_merge(m2[fm], d[fm], xor32(m2[fm]), xor32(d[fm]));
  }
  float* red = reinterpret_cast<float*>(lds);  // [128 rows][2]
  __syncthreads();
  if (ec.wn == 1 && (ec.lane >> 4) == 0) {
#pragma unroll
    for (int fm = 0; fm < 4; ++fm) {
      red[ec.row(fm) * 2] = m2[fm];
      red[ec.row(fm) * 2 + 1] = d[fm];
    }
  }
  __syncthreads();
  if (ec.wn == 0 && (ec.lane >> 4) == 0) {
#pragma unroll
    for (int fm = 0; fm < 4; ++fm) {
      lse_merge(m2[fm], d[fm], red[ec.row(fm) * 2], red[ec.row(fm) * 2 + 1]);
      if (rglob[fm] < a.N) {
        const int64_t o = ((int64_t)rglob[fm] * a.splits + ts) * 2;
        a.part[o + 0] = m2[fm];
        a.part[o + 1] = d[fm];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Backward, step 1: G = g (softmax - onehot) of one block, fp32.
// ---------------------------------------------------------------------------
template <bool kCap>
__device__ __forceinline__ void recompute_epilogue_f32(const f32x4_t (&acc)[4][4],
                                                       const RecompArgs& a, const CoordsF& ec,
                                                       int32_t row0, int32_t col0) {
  const float cap = a.softcap, inv_cap = kCap ? 1.0f / a.softcap : 0.f;
  const int32_t ncol0 = col0 + ec.col(0);  // block-local column of fn = 0, r = 0
#pragma unroll
  for (int fm = 0; fm < 4; ++fm) {
    const int32_t rowl = row0 + ec.row(fm);
    const bool rv = rowl < a.Cn;
    const int32_t rr = rv ? rowl : 0;
    const float lse2 = a.lse[rr] * kLog2e;
    const float g = rv ? a.grad[(int64_t)a.row_index[rr] * a.gstride] : 0.f;
    const int32_t rel = rv ? a.row_label[rr] - a.v0 - ncol0 : -1;
    char* grow = a.G + (int64_t)rowl * a.ldg_b;
#pragma unroll
    for (int fn = 0; fn < 4; ++fn) {
      f32x4_t o;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float x = acc[fm][fn][r];
        float dcap = 1.f;
        if (kCap) {
          const float t = tanh_approx(x * inv_cap);
          x = cap * t;
          dcap = 1.f - t * t;
        }
        float p = fast_exp2(fmaf(x, kLog2e, -lse2));
        p -= rel == fn * 16 + r ? 1.f : 0.f;
        const bool ok = rv && ncol0 + fn * 16 + r < a.cv;
        o[r] = ok ? p * g * dcap : 0.f;
      }
      *reinterpret_cast<f32x4_t*>(grow + (int64_t)(ncol0 + fn * 16) * 4) = o;
    }
  }
}

template <bool kKTail>
MT_F32_KERNEL void recompute_f32_kernel(RecompArgs a) {
  __shared__ __attribute__((aligned(1024))) char lds[kLdsF];
  uint32_t tm, tn;
  grouped_tile(xcd_remap(blockIdx.x, gridDim.x), a.tiles_m, a.tiles_n, 8, tm, tn);
  const CoordsF ec;
  const int32_t row0 = (int32_t)tm * kTileF, vloc0 = (int32_t)tn * kTileF;
  uint32_t c_lim;
  const int KT = stages_f32(a.H, c_lim);
  KcF A, B;
  A.init([&](uint32_t r) __attribute__((always_inline)) {
    int32_t rr = row0 + (int32_t)r;
    rr = rr < a.Cn ? rr : a.Cn - 1;
    return a.X + (int64_t)a.row_index[rr] * a.ldx_b;
  }, ec.wm * 64);
  B.init([&](uint32_t r) __attribute__((always_inline)) {
    int32_t v = vloc0 + (int32_t)r;
    v = v < a.cv ? v : a.cv - 1;  // rows past the block repeat its last one
    return a.W + (int64_t)v * a.ldw_b;
  }, ec.wn * 64);
  if constexpr (kKTail) {
    A.set_tail(c_lim);
    B.set_tail(c_lim);
  }
  f32x4_t acc[4][4];
  mainloop_f32<kKTail, false>(lds, acc, A, B, KT, c_lim);
  if (a.softcap > 0.f) recompute_epilogue_f32<true>(acc, a, ec, row0, vloc0);
  else recompute_epilogue_f32<false>(acc, a, ec, row0, vloc0);
}

// ---------------------------------------------------------------------------
// Backward, steps 2 and 3 in one launch: workgroups [0, dx_blocks) form dX
// (its items are the longer ones, so they go first), the rest dW.
//
// dX has only rows / 128 x H / 128 output tiles, each contracting a whole
// vocabulary block, so each tile is split over K into nsplit slices of kslice
// entries; slice z adds into its own fp32 plane (accbuf + z split_stride),
// and dx_sum_f32_kernel sums the planes in slice order once the last block
// is done (no atomics: the same result every time).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void dx_f32_item(char* lds, const DxArgs& a, uint32_t b, uint32_t nb) {
  const uint32_t ns = (uint32_t)a.nsplit, z = b % ns;
  uint32_t tm, tn;
  grouped_tile(xcd_remap(b / ns, nb / ns), a.tiles_m, a.tiles_n, 8, tm, tn);
  const CoordsF ec;
  const int32_t row0 = (int32_t)tm * kTileF, h0 = (int32_t)tn * kTileF;
  const int32_t k0 = (int32_t)z * a.kslice, kv = min(a.kslice, a.kv - k0);
  KcF A;
  TrF B;
  A.init([&](uint32_t r) __attribute__((always_inline)) {
    return a.G + (int64_t)(row0 + (int32_t)r) * a.ldg_b + (int64_t)k0 * 4;
  }, ec.wm * 64);
  B.init(a.W + (int64_t)k0 * a.ldw_b + (int64_t)h0 * 4, a.ldw_b, a.V - a.v0 - k0, a.H - h0,
         ec.wn * 64);
  f32x4_t acc[4][4];
  mainloop_f32<false, true>(lds, acc, A, B, (kv + kBKF - 1) / kBKF);
  float* plane = a.accbuf + (int64_t)z * a.split_stride;
#pragma unroll
  for (int fm = 0; fm < 4; ++fm) {
    const int32_t rowl = row0 + ec.row(fm);
    if (rowl >= a.Cn) continue;
    float* arow = plane + (int64_t)rowl * a.ld_acc;
    float* xrow = reinterpret_cast<float*>(a.dX + (int64_t)a.row_index[rowl] * a.lddx_b);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int32_t h = h0 + ec.col_tr(r);
      if (h >= a.H) continue;
      f32x4_t v = {acc[fm][0][r], acc[fm][1][r], acc[fm][2][r], acc[fm][3][r]};
      if (a.mode == kDxAdd || a.mode == kDxAddEmit) v += *reinterpret_cast<const f32x4_t*>(arow + h);
      *reinterpret_cast<f32x4_t*>((a.mode >= kDxAddEmit ? xrow : arow) + h) = v;
    }
  }
}

__device__ __forceinline__ void dw_f32_item(char* lds, const DwArgs& a, uint32_t b, uint32_t nb) {
  uint32_t tm, tn;
  grouped_tile(xcd_remap(b, nb), a.tiles_m, a.tiles_n, 8, tm, tn);
  const CoordsF ec;
  const int32_t m0 = (int32_t)tm * kTileF, h0 = (int32_t)tn * kTileF;
  TrF A;
  KcF B;
  A.init(a.G + (int64_t)m0 * 4, a.ldg_b, a.g_rows, a.g_cols - m0, ec.wm * 64);
  B.init([&](uint32_t r) __attribute__((always_inline)) {
    int32_t h = h0 + (int32_t)r;
    h = h < a.H ? h : a.H - 1;
    return a.XcT + (int64_t)h * a.ldxt_b;
  }, ec.wn * 64);
  f32x4_t acc[4][4];
  mainloop_f32<false, true>(lds, acc, A, B, (a.kt_rows + kBKF - 1) / kBKF);
#pragma unroll
  for (int fm = 0; fm < 4; ++fm) {
    const int32_t vl = m0 + ec.row_tr(fm);
    if (vl >= a.cv) continue;
    float* wrow = a.dW + (int64_t)(a.v0 + vl) * a.lddw;
#pragma unroll
    for (int fn = 0; fn < 4; ++fn) {
      const int32_t h = h0 + ec.col(fn);
      if (h >= a.H) continue;
      f32x4_t v = acc[fm][fn];
      if (a.accumulate) v += *reinterpret_cast<const f32x4_t*>(wrow + h);
      *reinterpret_cast<f32x4_t*>(wrow + h) = v;
    }
  }
}

MT_F32_KERNEL void dx_dw_f32_kernel(DxArgs x, DwArgs w, uint32_t dx_blocks) {
  __shared__ __attribute__((aligned(1024))) char lds[kLdsF];
  if (blockIdx.x < dx_blocks) dx_f32_item(lds, x, blockIdx.x, dx_blocks);
  else dw_f32_item(lds, w, blockIdx.x - dx_blocks, gridDim.x - dx_blocks);
}

// dX rows of a row block from the nsplit planes of dx_dw_f32_kernel: row t <
// cn, four columns per thread.
__global__ __launch_bounds__(256) void dx_sum_f32_kernel(const float* part, int64_t stride,
                                                         int32_t nsplit, int32_t cn, int32_t H,
                                                         const int32_t* row_index, char* dX,
                                                         int64_t lddx_b) {
  const int64_t nv = H / 4, i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t t = i / nv, h = (i - t * nv) * 4;
  if (t >= cn) return;
  const float* p = part + t * H + h;
  f32x4_t v = *reinterpret_cast<const f32x4_t*>(p);
  for (int32_t z = 1; z < nsplit; ++z) v += *reinterpret_cast<const f32x4_t*>(p + z * stride);
  *reinterpret_cast<f32x4_t*>(dX + (int64_t)row_index[t] * lddx_b + h * 4) = v;
}

}  // namespace mtf

// Kernels of the fused LM-head linear + per-token cross-entropy path.
//
//   argument structures of the GEMM-shaped kernels (flce_kernels_bf16.h,
//   flce_kernels_f32.h) and what both share of their epilogues
//   fwd_finalize     merge of the per-split (max, sum) partials -> lse, loss
//   small kernels    valid-row compaction, gather-transpose of X rows,
//                    zeroing of ignored rows, per-sample segment sums.
#pragma once

#include "flce_device.h"

namespace mtf {

// Output coordinates of this lane's accumulators for a wave tile of
// 128 rows x (NFN * 16) columns, WC waves across the tile's columns (tile
// width NFN * 16 * WC: 8 x 16 x 2 for the bf16 kernels).
template <int NFN, int WC = 2>
struct EpiCoordsT {
  static constexpr int kNF = NFN;
  static constexpr int kWC = WC;
  static constexpr int kTileN = NFN * 16 * WC;
  uint32_t lane, wm, wn;
  __device__ __forceinline__ EpiCoordsT() {
    lane = lane_id();
    uint32_t w = wave_id();
    wm = w / WC;
    wn = w % WC;
  }
  // Tile-local output row of fragment row fm held by this lane.
  __device__ __forceinline__ int row(int fm) const { return wm * 128 + fm * 16 + (lane & 15u); }
  // Tile-local output column of element 0 of fragment column fn.
  __device__ __forceinline__ int col(int fn) const {
    return wn * (NFN * 16) + fn * 16 + 4 * (lane >> 4);
  }
};

// Is column offset `rel` (label column minus this lane's column of fn = 0,
// r = 0) one of the NFN * 4 columns this lane holds?
template <int NFN>
__device__ __forceinline__ bool lane_holds(int rel) {
  return rel >= 0 && rel < NFN * 16 && (rel & 12) == 0;
}

// ===========================================================================
// Forward
// ===========================================================================
struct FwdArgs {
  const char* X;
  const char* W;  // vocabulary row vcol0 of the weight
  int64_t ldx_b, ldw_b;
  int32_t H, V, N;  // V: vocabulary rows from W on (this launch's block)
  int32_t vcol0;    // global vocabulary index of W's row 0 (a multiple of 256)
  uint32_t x_range, w_range, s_range;  // bytes addressable from X, W, S
  const int32_t* row_index;
  const int32_t* row_label;
  float softcap;
  int32_t tiles_m, splits, vt_total, vt_per_split;
  float* part;  // [N][splits][2] = (max in log2 units, scaled sum)
  float* xy;    // [N] label logit
  char* S;      // bf16 logits or exponentials [>= tiles_m * 256][lds_b / 2] (fused path only)
  int64_t lds_b;
  const int32_t* run_if = nullptr;  // non-null: the kernel does nothing unless *run_if != 0
  int32_t* guard_reset = nullptr;   // non-null: set to 0 by the launch (read only after it)
};

// x of lane l ^ 16 and of lane l ^ 32, from one lane swap and a select
// (v_permlane16_swap / v_permlane32_swap with x as both operands hand back
// rows (0, 0, 2, 2) and (1, 1, 3, 3) of 16 lanes, or halves (lo, lo) and
// (hi, hi)) instead of an LDS permute and its wait.
__device__ __forceinline__ float xor16(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return __builtin_bit_cast(float, (lane_id() & 16u) ? p[0] : p[1]);
}
__device__ __forceinline__ float xor32(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const auto p = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, (lane_id() & 32u) ? p[0] : p[1]);
}

// Merge the four lanes that share a row, then the WC waves (wn = 0 .. WC - 1)
// that share the row through LDS, and write this split's (max, sum) partial
// of every row.
template <int NFN, int WC>
__device__ __forceinline__ void fwd_final_merge(char* lds, float (&m2)[8], float (&d)[8],
                                                const int32_t (&rglob)[8], uint32_t ts,
                                                const EpiCoordsT<NFN, WC>& ec, const FwdArgs& a) {
#pragma unroll
  for (int fm = 0; fm < 8; ++fm) {
    lse_merge(m2[fm], d[fm], xor16(m2[fm]), xor16(d[fm]));
    lse_merge(m2[fm], d[fm], xor32(m2[fm]), xor32(d[fm]));
  }
  float* red = reinterpret_cast<float*>(lds);  // [WC - 1][256 rows][2]
  __syncthreads();
  if (ec.wn != 0 && (ec.lane >> 4) == 0) {
#pragma unroll
    for (int fm = 0; fm < 8; ++fm) {
      float* r = red + ((ec.wn - 1) * 256 + ec.row(fm)) * 2;
      r[0] = m2[fm];
      r[1] = d[fm];
    }
  }
  __syncthreads();
  if (ec.wn == 0 && (ec.lane >> 4) == 0) {
#pragma unroll
    for (int fm = 0; fm < 8; ++fm) {
#pragma unroll
      for (int w = 0; w < WC - 1; ++w) {
        const float* r = red + (w * 256 + ec.row(fm)) * 2;
        lse_merge(m2[fm], d[fm], r[0], r[1]);
      }
      if (rglob[fm] < a.N) {
        int64_t o = ((int64_t)rglob[fm] * a.splits + ts) * 2;
        a.part[o + 0] = m2[fm];
        a.part[o + 1] = d[fm];
      }
    }
  }
}

// lse and loss of each valid row from its `splits` (max, sum) partials: one
// wave per row, lanes merge strided partials, then a fixed shuffle tree
// (deterministic order).
// guard (non-null): set to 1 when some row's largest logit lies outside
// [kGuardLo, kGuardHi], the range in which the fused path keeps exp(logit)
// itself in bf16 (see fused_grad_kernel): at a row maximum of -48 the
// terms within 39 of it (relative weight e^-39 and more) stay normal numbers
// (e^-87 is about the smallest), and at +48, lse <= 48 + ln V keeps the row
// factor g exp(-lse) a normal fp32 number for g down to 1e-10 at V = 2^20.
constexpr float kGuardLo = -48.f, kGuardHi = 48.f;
// Rows N .. N + n_ignored of row_index (the last row block's caller passes the
// ignored rows that follow the counted ones) get loss +0.0, by the grid's last
// workgroups.
__global__ __launch_bounds__(256) void fwd_finalize_kernel(const float* part, const float* xy,
                                                           int32_t N, int32_t splits,
                                                           const int32_t* row_index, float* loss,
                                                           float* lse, int32_t* guard,
                                                           int32_t n_ignored = 0) {
  const uint32_t row_blocks = ((uint32_t)N + 3u) / 4u;
  if (blockIdx.x >= row_blocks) {
    const int32_t i = (int32_t)((blockIdx.x - row_blocks) * 256u + threadIdx.x);
    if (i < n_ignored) loss[row_index[N + i]] = 0.0f;
    return;
  }
  const int32_t r = (int32_t)(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (r >= N) return;  // uniform per wave
  const int lane = (int)(threadIdx.x & 63u);
  const float* pr = part + (int64_t)r * splits * 2;
  float m = kNegBig, d = 0.f;
  for (int s = lane; s < splits; s += 64) lse_merge(m, d, pr[2 * s], pr[2 * s + 1]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) lse_merge(m, d, __shfl_xor(m, off), __shfl_xor(d, off));
  if (lane == 0) {
    const float L = (m + fast_log2(d)) * kLn2;
    lse[r] = L;
    loss[row_index[r]] = L - xy[r];
    const float mx = m * kLn2;
    if (guard && !(mx >= kGuardLo && mx <= kGuardHi)) atomicOr(guard, 1);
  }
}

// ===========================================================================
// Backward, step 1: G = g * (softmax(logits) - onehot) for one block.
// ===========================================================================
struct RecompArgs {
  const char* X;
  const char* W;  // vocabulary row v0 of the weight (the block's first row)
  int64_t ldx_b, ldw_b;
  int32_t H, V;
  uint32_t x_range, w_range, g_range;  // bytes addressable from X, W, G
  const int32_t* row_index;  // offset to the block's first valid row
  const int32_t* row_label;
  const float* lse;
  int32_t Cn;  // valid rows in the block
  const float* grad;
  int64_t gstride;
  float softcap;
  int32_t v0, cv;  // vocabulary range [v0, v0 + cv)
  char* G;         // [tiles_m * 256][>= tiles_n * 256], row pitch ldg_b
  int64_t ldg_b;
  int32_t tiles_m, tiles_n;
  uint32_t* zero_words = nullptr;  // cleared by the launch (dW's work queue, read after it)
  // non-null (bf16): the launch computes nothing unless *run_if != 0 (the
  // first vocabulary block, whose G a forward kept as exponentials, when
  // those left their range); zero_words is cleared either way
  const int32_t* run_if = nullptr;
};

// The first vocabulary block's G from the exponentials E = exp(z) that
// mt_flce_forward_keep left in the G block (columns [0, cols), softcap off):
// G = g (E exp(-lse) - onehot), in place, one workgroup per row of the block
// (rows >= cn become 0).  Nothing when *skip_if != 0: some row's largest
// logit left the range in which E holds its terms, and the block is
// recomputed instead (recompute_bf16_kernel with run_if = the same word).
// HBM-bound: one 16-byte read and one 16-byte write per 8 entries.
__global__ __launch_bounds__(256) void exp_to_grad_kernel(char* G, int64_t ldg_b, int32_t cols,
                                                          int32_t cn, const float* lse,
                                                          const float* grad, int64_t gstride,
                                                          const int32_t* row_index,
                                                          const int32_t* row_label,
                                                          const int32_t* skip_if) {
  if (*skip_if != 0) return;
  const int32_t row = (int32_t)blockIdx.x;
  const bool rv = row < cn;
  float s = 0.f, g = 0.f;
  int32_t y = -1;
  if (rv) {
    g = grad[(int64_t)row_index[row] * gstride];
    s = g * fast_exp2(-lse[row] * kLog2e);
    y = row_label[row];
  }
  char* p = G + (int64_t)row * ldg_b;
  for (int32_t c = (int32_t)threadIdx.x * 8; c < cols; c += 256 * 8) {
    u32x4_t v = *reinterpret_cast<const u32x4_t*>(p + (int64_t)c * 2);
    u32x4_t o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float e0 = __builtin_bit_cast(float, v[j] << 16);
      const float e1 = __builtin_bit_cast(float, v[j] & 0xffff0000u);
      const int32_t c0 = c + 2 * j;
      const float g0 = fmaf(s, e0, c0 == y ? -g : 0.f);
      const float g1 = fmaf(s, e1, c0 + 1 == y ? -g : 0.f);
      o[j] = rv ? pack_bf16x2(g0, g1) : 0u;
    }
    *reinterpret_cast<u32x4_t*>(p + (int64_t)c * 2) = o;
  }
}

// ===========================================================================
// Backward, step 2: dX rows of the block (+)= G . W[v0 : v0 + cv]
// ===========================================================================
enum DxMode : int32_t { kDxStore = 0, kDxAdd = 1, kDxAddEmit = 2, kDxEmit = 3 };
// bf16 only: kDxStore / kDxAdd / kDxAddEmit with the fp32 accumulator held as
// 256 x 256 tiles (accbuf + (tm * tiles_n + tn) * 65536 floats, each in the
// order of the wave's accumulators: one contiguous KiB per load and store)
constexpr int32_t kDxTiledAcc = 4;

struct DxArgs {
  const char* G;
  int64_t ldg_b;
  const char* W;  // vocabulary row v0 of the weight (the block's first row)
  int64_t ldw_b;
  uint32_t g_range, w_range;  // bytes addressable from G, W
  int32_t V, v0, kv;  // K = vocabulary entries v0 .. v0 + kv
  int32_t H, Cn;
  float* accbuf;  // fp32 [>= Cn][ld_acc] (modes >= kDxTiledAcc: tiles_m x tiles_n tiles)
  int64_t ld_acc;
  int32_t mode;
  char* dX;
  int64_t lddx_b;
  const int32_t* row_index;  // offset to the block's first valid row
  int32_t tiles_m, tiles_n;
  const float* row_scale = nullptr;  // non-null (bf16 kDxEmit): dX row r times row_scale[r]
  // split over K (bf16): nsplit slices of kslice vocabulary entries, slice z
  // stored (kDxStore) at accbuf + z * split_stride; the grid is
  // tiles_m * tiles_n * nsplit (dx_split_reduce_kernel sums the slices)
  int32_t nsplit = 1, kslice = 0;
  int64_t split_stride = 0;
  // non-null (bf16 kDxEmit without row_scale, kDxTiledAcc + kDxAddEmit): every
  // dX row times *out_scale
  const float* out_scale = nullptr;
  // dX beside a work-queue dW in one launch (dx_dw_bf16_kernel), XCD-
  // partitioned: xcds > 0 gives dX whole XCDs -- workgroup b (on XCD b % 8)
  // takes logical tile (b % 8) per_xcd + b / 8 when b % 8 < xcds and
  // b / 8 < per_xcd -- and every other workgroup is a dW worker, so that dX
  // and dW never share an XCD's L2 while dX runs; 0: workgroups [0, tiles)
  // are dX's (xcd_remap order)
  int32_t xcds = 0, per_xcd = 0;
};

// dX of a K-split chunk: row t < cn, columns h .. h + 3 of the sum of the
// nsplit fp32 slices (in slice order), times scale[t * scale_stride] (null: 1),
// to bf16 at dX row row_index[t].  One thread per 4 columns.
__global__ __launch_bounds__(256) void dx_split_reduce_kernel(const float* part, int64_t stride,
                                                              int32_t nsplit, int64_t ld, int32_t cn,
                                                              int32_t H, const float* scale,
                                                              int64_t scale_stride,
                                                              const int32_t* row_index, char* dX,
                                                              int64_t lddx_b) {
  const int32_t t = (int32_t)blockIdx.y;
  const int32_t h = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (t >= cn || h >= H) return;
  const float* p = part + (int64_t)t * ld + h;
  f32x4_t v = *reinterpret_cast<const f32x4_t*>(p);
  for (int32_t z = 1; z < nsplit; ++z) v += *reinterpret_cast<const f32x4_t*>(p + z * stride);
  if (scale) v *= scale[t * scale_stride];
  u32x2_t o;
  o[0] = pack_bf16x2(v[0], v[1]);
  o[1] = pack_bf16x2(v[2], v[3]);
  *reinterpret_cast<u32x2_t*>(dX + (int64_t)row_index[t] * lddx_b + (int64_t)h * 2) = o;
}

// ===========================================================================
// Backward, step 3: dW[v0 : v0 + cv] (+)= G^T . X_block
// ===========================================================================
constexpr int kQueueWords = 8;
struct DwArgs {
  const char* G;  // [K = tokens][vocab], row pitch ldg_b
  int64_t ldg_b;
  int32_t g_rows;  // rows of G that exist (>= K rounded up to the K slab)
  int32_t g_cols;  // columns of G that exist
  const char* XcT;  // [H][K] gathered + transposed X rows of the block
  int64_t ldxt_b;
  uint32_t g_range, xt_range;  // bytes addressable from G, XcT
  int32_t kt_rows;  // K extent (valid rows of the block)
  int32_t H, cv, v0;
  float* dW;
  int64_t lddw;
  int32_t accumulate;
  int32_t tiles_m, tiles_n;
  // non-null: persistent schedule over a work queue (dw_bf16_kernel<true>):
  // kQueueWords counters, zero at launch, one per XCD's share of the tiles
  uint32_t* queue = nullptr;
  // tiled (bf16): dW in the library's tile order instead of rows of pitch
  // lddw, over two buffers: tile (tm, tn) at floats tile_pad + (tm tiles_n
  // + tn) 65536 from dW for tm < lo_rows, else at ((tm - lo_rows) tiles_n +
  // tn) 65536 from dW_hi; tm counted from vocabulary row 0 (the block's tile
  // rows start at v0 / 256, v0 a multiple of 256), wave w's fragment (fm,
  // fn) at ((w 64 + fm 8 + fn) 64 + lane) 4 within the tile
  int32_t tiled = 0;
  int64_t tile_pad = 0;
  float* dW_hi = nullptr;
  int32_t lo_rows = 0;
  // narrow (bf16, a dW every tile completes in one pass): dW is bf16 rows of
  // pitch lddw elements, each tile narrowed in its epilogue (kDwNarrow), times
  // *out_scale when that is non-null
  int32_t narrow = 0;
  const float* out_scale = nullptr;
};

// Where a bf16 dW kernel puts its tiles (template argument kOut): fp32 rows
// of pitch lddw, fp32 tiles (DwArgs::tiled), or -- for a dW that every tile
// completes in one pass (one row block, nothing added into) -- bf16 rows of
// pitch lddw (elements) at dW, narrowed in the epilogue.
constexpr int kDwRows = 0, kDwTiles = 1, kDwNarrow = 2;

// ===========================================================================
// Small kernels
// ===========================================================================

// XcT[h][t] = X[row_index[t]][h] for t < Cn, 0 for Cn <= t < t_pad.
// 64 x 64 element tiles; 16-byte loads along h, 16-byte stores along t.
// scale (bf16 only): row t is multiplied by scale(t) in fp32 and rounded to
// bf16 (the fused path's per-row factor of G, see fused_grad_kernel); kScale
// false: not at all.
template <typename T, bool kScale, class Scale>
__device__ __forceinline__ void gather_t_tile(T (&tile)[64][64 + 1], int32_t t0, int32_t hb,
                                              const char* X, int64_t ldx_b, const int32_t* row_index,
                                              int32_t Cn, int32_t H, char* XcT, int64_t ldxt_b,
                                              Scale scale) {
  constexpr int E = sizeof(T);
  constexpr int PER = 16 / E;  // elements per 16-byte vector
  // load 64 rows (t) x 64 h
  for (int v = threadIdx.x; v < 64 * 64 / PER; v += 256) {
    const int tr = v / (64 / PER), hc = (v % (64 / PER)) * PER;
    const int32_t t = t0 + tr;
    u32x4_t val = {0u, 0u, 0u, 0u};
    if (t < Cn && hb + hc < H)
      val = *reinterpret_cast<const u32x4_t*>(X + (int64_t)row_index[t] * ldx_b +
                                              (int64_t)(hb + hc) * E);
    if constexpr (kScale) {
      if (t < Cn) {
        const float sc = scale(t);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          val[j] = pack_bf16x2(__builtin_bit_cast(float, val[j] << 16) * sc,
                               __builtin_bit_cast(float, val[j] & 0xffff0000u) * sc);
      }
    }
    const T* e = reinterpret_cast<const T*>(&val);
#pragma unroll
    for (int j = 0; j < PER; ++j) tile[tr][hc + j] = e[j];
  }
  __syncthreads();
  for (int v = threadIdx.x; v < 64 * 64 / PER; v += 256) {
    const int hr = v / (64 / PER), tc = (v % (64 / PER)) * PER;
    if (hb + hr >= H) continue;
    u32x4_t val;
    T* e = reinterpret_cast<T*>(&val);
#pragma unroll
    for (int j = 0; j < PER; ++j) e[j] = tile[tc + j][hr];
    *reinterpret_cast<u32x4_t*>(XcT + (int64_t)(hb + hr) * ldxt_b + (int64_t)(t0 + tc) * E) = val;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void gather_t_kernel(const char* X, int64_t ldx_b,
                                                       const int32_t* row_index, int32_t Cn,
                                                       int32_t H, char* XcT, int64_t ldxt_b) {
  __shared__ T tile[64][64 + 1];
  gather_t_tile<T, false>(tile, blockIdx.x * 64, blockIdx.y * 64, X, ldx_b, row_index, Cn, H, XcT,
                          ldxt_b, 0);
}

// Zero `nrows` rows (ids from rows[]) of a row-major matrix, row_bytes each
// (a multiple of 16).
__global__ __launch_bounds__(256) void zero_rows_kernel(char* base, int64_t ld_b,
                                                        const int32_t* rows, int64_t nrows,
                                                        int64_t row_bytes) {
  const int64_t nvec = row_bytes / 16;
  for (int64_t r = blockIdx.x; r < nrows; r += gridDim.x) {
    char* p = base + (int64_t)rows[r] * ld_b;
    for (int64_t v = threadIdx.x; v < nvec; v += blockDim.x)
      reinterpret_cast<u32x4_t*>(p)[v] = u32x4_t{0u, 0u, 0u, 0u};
  }
}

// Zero a dense [rows][cols] fp32 matrix with leading dimension ld.
__global__ __launch_bounds__(256) void zero_matrix_f32_kernel(float* p, int64_t rows, int64_t cols,
                                                              int64_t ld) {
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x)
    for (int64_t c = threadIdx.x; c < cols; c += blockDim.x) p[r * ld + c] = 0.f;
}

__global__ void set_i32_kernel(int32_t* p, int32_t v) { *p = v; }

// loss[rows[i]] = +0.0 for i < n.
__global__ __launch_bounds__(256) void zero_scatter_f32_kernel(float* loss, const int32_t* rows,
                                                               int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    loss[rows[i]] = 0.0f;
}

// Valid-row compaction, one workgroup of 1024 threads per `span` labels (a
// multiple of 4096).
//   row_index[0 .. N)    positions t with a valid label, ascending
//   row_index[N .. T)    every other position (descending from the end)
//   row_label[0 .. N)    their labels
//   counts = {N, #labels outside [0, V), first such t or -1, 0}
// Each workgroup counts the labels before its own by itself (they come from L2;
// independent loads), so no workgroup waits for another and no scratch is
// needed; the last one writes counts.  Bound by latency: one workgroup walking
// all labels, a scan and two barriers per 4096, took 58 us for 53k labels.  The
// labels read again grow with the workgroups (1/2 T each on average), so there
// are at most kPrepBlocks, which from 2^20 labels on take longer spans: 16.8M
// labels 13.0 ms in one workgroup, 34 ms at 4096 apiece, 2.7 ms in 256; 53k
// labels 41 us in one, 13 us at 4096 apiece.
constexpr int kPrepItems = 4, kPrepLabels = 1024 * kPrepItems, kPrepBlocks = 256;
__global__ __launch_bounds__(1024) void prepare_kernel(const int64_t* labels, int64_t T, int64_t V,
                                                       int64_t ignore, int shift, int64_t span,
                                                       int32_t* row_index, int32_t* row_label,
                                                       int32_t* counts) {
  __shared__ int32_t wsum_v[16], wpre_v[16], wbad[16], wfirst[16];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int64_t start = (int64_t)blockIdx.x * span, end = min(start + span, T);
  auto label = [&](int64_t t) __attribute__((always_inline)) {
    return shift ? (t + 1 < T ? labels[t + 1] : ignore) : labels[t];
  };
  // 0 ignored, 1 valid, 2 out of range
  auto kind = [&](int64_t lab) __attribute__((always_inline)) {
    return lab == ignore ? 0 : (lab < 0 || lab >= V ? 2 : 1);
  };
  int32_t pre_v = 0, bad = 0, first = INT32_MAX;
  auto see_bad = [&](int k, int64_t t) __attribute__((always_inline)) {
    if (k == 2) {
      ++bad;
      first = min(first, (int32_t)t);
    }
  };
  for (int64_t t0 = tid; t0 < start; t0 += 1024 * 8) {
    int64_t lab[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) lab[j] = t0 + j * 1024 < start ? label(t0 + j * 1024) : ignore;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = kind(lab[j]);
      pre_v += k == 1;
      see_bad(k, t0 + j * 1024);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) pre_v += __shfl_xor(pre_v, o);
  if (lane == 63) wpre_v[wid] = pre_v;
  int32_t base = 0;  // valid before the labels at hand
  for (int64_t c0 = start; c0 < end || c0 == start; c0 += kPrepLabels) {
    int32_t y[kPrepItems];
    uint32_t vmask = 0, mmask = 0;
#pragma unroll
    for (int j = 0; j < kPrepItems; ++j) {
      const int64_t t = c0 + tid * kPrepItems + j;
      y[j] = 0;
      if (t >= end) continue;
      const int64_t lab = label(t);
      const int k = kind(lab);
      see_bad(k, t);
      if (k == 1) {
        vmask |= 1u << j;
        y[j] = (int32_t)lab;
      } else {
        mmask |= 1u << j;
      }
    }
    const int cv = __builtin_popcount(vmask);
    int sv = cv;  // inclusive wave scan of these 4096 labels' valid ones
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int up = __shfl_up(sv, o);
      if (lane >= o) sv += up;
    }
    if (c0 != start) __syncthreads();  // (the sums of the labels before have been read)
    if (lane == 63) wsum_v[wid] = sv;
    __syncthreads();
    int32_t before = 0, own = 0;  // valid before this wave's labels, and in all
    for (int w = 0; w < 16; ++w) {
      if (w < wid) before += wsum_v[w];
      own += wsum_v[w];
      if (c0 == start) base += wpre_v[w];
    }
    int32_t ov = base + before + sv - cv;
    int32_t om = (int32_t)(c0 + (int64_t)tid * kPrepItems) - ov;  // others before this thread's labels
#pragma unroll
    for (int j = 0; j < kPrepItems; ++j) {
      const int32_t t = (int32_t)(c0 + tid * kPrepItems + j);
      if (vmask & (1u << j)) {
        row_index[ov] = t;
        row_label[ov] = y[j];
        ++ov;
      } else if (mmask & (1u << j)) {
        row_index[T - 1 - om] = t;
        ++om;
      }
    }
    base += own;
  }
  if (blockIdx.x != gridDim.x - 1) return;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    bad += __shfl_xor(bad, o);
    first = min(first, __shfl_xor(first, o));
  }
  if (lane == 63) {
    wbad[wid] = bad;
    wfirst[wid] = first;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 16; ++w) {
      bad += wbad[w];
      first = min(first, wfirst[w]);
    }
    counts[0] = base;
    counts[1] = bad;
    counts[2] = bad ? first : -1;
    counts[3] = 0;
  }
}

// status = 1 if cu_seqlens is not a valid partition of [0, T).
__global__ __launch_bounds__(256) void segment_check_kernel(const int32_t* cu, int64_t S, int64_t T,
                                                            int32_t* status) {
  __shared__ int32_t bad;
  if (threadIdx.x == 0) bad = (cu[0] != 0 || (int64_t)cu[S] != T) ? 1 : 0;
  __syncthreads();
  for (int64_t s = threadIdx.x; s < S; s += blockDim.x)
    if (cu[s + 1] < cu[s]) atomicOr(&bad, 1);
  __syncthreads();
  if (threadIdx.x == 0) *status = bad;
}

// One workgroup per sample: fixed-order tree sum of loss and count of valid
// targets over [cu[s], cu[s+1]).  With shift, the target of position t is
// labels[t + 1] (ignore_index at t = T - 1), as the causal shift forms it.
__global__ __launch_bounds__(256) void segment_sum_kernel(const float* loss, const int64_t* target,
                                                          int64_t T, int64_t ignore, int shift,
                                                          const int32_t* cu,
                                                          const int32_t* status, float* seg_loss,
                                                          int32_t* seg_count) {
  __shared__ float sl[256];
  __shared__ int32_t sc[256];
  const int64_t s = blockIdx.x;
  float acc = 0.f;
  int32_t cnt = 0;
  if (*status == 0) {
    for (int64_t t = cu[s] + threadIdx.x; t < cu[s + 1]; t += 256) {
      acc += loss[t];
      const int64_t src = t + (shift ? 1 : 0);
      cnt += (src < T && target[src] != ignore) ? 1 : 0;
    }
  }
  sl[threadIdx.x] = acc;
  sc[threadIdx.x] = cnt;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      sl[threadIdx.x] += sl[threadIdx.x + o];
      sc[threadIdx.x] += sc[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    seg_loss[s] = sl[0];
    seg_count[s] = sc[0];
  }
}

// ===========================================================================
// Gradients formed for a unit upstream gradient, rescaled once the real one
// is known: the reference's fused loss computes dX and dW in its forward and
// multiplies them by the scalar grad_output in its backward.  The scale is
// read from device memory (no host sync).  Rows are a grid-stride loop, 16
// bytes per thread and access; a column tail that is not a whole vector
// goes element by element.
// ===========================================================================

// dst[r, c] = scale * src[r, c] for an fp32 matrix; dst fp32 (may be src:
// every element is read and written by the same thread) or bf16 (round to
// nearest even).
template <bool kOutBf16>
__global__ __launch_bounds__(256) void scale_rows_f32_kernel(const float* src, int64_t ld_src,
                                                             void* dst, int64_t ld_dst,
                                                             int64_t rows, int64_t cols,
                                                             const float* scale) {
  const float c = *scale;
  const int64_t nv = cols / 4;
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    const float* s = src + r * ld_src;
    for (int64_t v = threadIdx.x; v < nv; v += blockDim.x) {
      const f32x4_t x = reinterpret_cast<const f32x4_t*>(s)[v];
      const float y0 = x[0] * c, y1 = x[1] * c, y2 = x[2] * c, y3 = x[3] * c;
      if (kOutBf16) {
        u32x2_t o;
        o[0] = pack_bf16x2(y0, y1);
        o[1] = pack_bf16x2(y2, y3);
        reinterpret_cast<u32x2_t*>(static_cast<char*>(dst) + r * ld_dst * 2)[v] = o;
      } else {
        reinterpret_cast<f32x4_t*>(static_cast<float*>(dst) + r * ld_dst)[v] =
            f32x4_t{y0, y1, y2, y3};
      }
    }
    for (int64_t k = nv * 4 + threadIdx.x; k < cols; k += blockDim.x) {
      const float y = s[k] * c;
      if (kOutBf16)
        reinterpret_cast<__bf16*>(static_cast<char*>(dst) + r * ld_dst * 2)[k] = (__bf16)y;
      else
        (static_cast<float*>(dst) + r * ld_dst)[k] = y;
    }
  }
}

// In place: p[r, c] = bf16(scale * p[r, c]) for a bf16 matrix of row pitch
// ld_b bytes.
__global__ __launch_bounds__(256) void scale_rows_bf16_kernel(char* p, int64_t ld_b, int64_t rows,
                                                              int64_t cols, const float* scale) {
  const float c = *scale;
  const int64_t nv = cols / 8;
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    u32x4_t* row = reinterpret_cast<u32x4_t*>(p + r * ld_b);
    for (int64_t v = threadIdx.x; v < nv; v += blockDim.x) {
      u32x4_t w = row[v];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float lo = __builtin_bit_cast(float, w[j] << 16) * c;
        const float hi = __builtin_bit_cast(float, w[j] & 0xffff0000u) * c;
        w[j] = pack_bf16x2(lo, hi);
      }
      row[v] = w;
    }
    __bf16* e = reinterpret_cast<__bf16*>(p + r * ld_b);
    for (int64_t k = nv * 8 + threadIdx.x; k < cols; k += blockDim.x)
      e[k] = (__bf16)((float)e[k] * c);
  }
}

// In-place narrowing: bf16 row r = scale * fp32 row r, written to the first
// bytes of the same allocation (bf16 row r at element offset r * ld in bf16
// units, i.e. bytes [2 r ld, 2 r ld + 2 cols)), so the weight gradient in the
// weight's dtype needs no second buffer.  bf16 row r overlaps fp32 row
// floor(r / 2) only, so one launch per phase of rows -- {0}, {1}, [2, 4),
// [4, 8), ... -- overwrites only rows an earlier phase has consumed; within a
// row (row 0 overlaps itself) the workgroup reads the whole row before any of
// it is written.  kPer 16-byte vectors per thread cover cols <= 1024 kPer.
template <int kPer>
__global__ __launch_bounds__(256) void narrow_rows_inplace_kernel(float* base, int64_t ld,
                                                                  int64_t r0, int64_t r1,
                                                                  int64_t cols,
                                                                  const float* scale) {
  const float c = *scale;
  const int64_t nv = cols / 4, nt = cols - nv * 4;
  for (int64_t r = r0 + blockIdx.x; r < r1; r += gridDim.x) {
    const float* src = base + r * ld;
    f32x4_t v[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int64_t idx = threadIdx.x + (int64_t)i * 256;
      v[i] = idx < nv ? reinterpret_cast<const f32x4_t*>(src)[idx] : f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    const float t = (int64_t)threadIdx.x < nt ? src[nv * 4 + threadIdx.x] : 0.f;
    __syncthreads();
    char* dst = reinterpret_cast<char*>(base) + r * ld * 2;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int64_t idx = threadIdx.x + (int64_t)i * 256;
      if (idx < nv) {
        u32x2_t o;
        o[0] = pack_bf16x2(v[i][0] * c, v[i][1] * c);
        o[1] = pack_bf16x2(v[i][2] * c, v[i][3] * c);
        reinterpret_cast<u32x2_t*>(dst)[idx] = o;
      }
    }
    if ((int64_t)threadIdx.x < nt)
      reinterpret_cast<__bf16*>(dst)[nv * 4 + threadIdx.x] = (__bf16)(t * c);
    __syncthreads();
  }
}

// ===========================================================================
// Cross-entropy over materialised logits [T, V] (reduction 'none').
// One workgroup of 256 threads per row; 16-byte loads along V.
// ===========================================================================
template <typename T>
__device__ __forceinline__ void load_vec(const char* p, float (&x)[16 / sizeof(T)]);
template <>
__device__ __forceinline__ void load_vec<float>(const char* p, float (&x)[4]) {
  f32x4_t v = *reinterpret_cast<const f32x4_t*>(p);
  x[0] = v[0];
  x[1] = v[1];
  x[2] = v[2];
  x[3] = v[3];
}
template <>
__device__ __forceinline__ void load_vec<__bf16>(const char* p, float (&x)[8]) {
  u32x4_t v = *reinterpret_cast<const u32x4_t*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = v[i];
    x[2 * i] = __builtin_bit_cast(float, w << 16);
    x[2 * i + 1] = __builtin_bit_cast(float, w & 0xffff0000u);
  }
}
template <typename T>
__device__ __forceinline__ float load_one(const char* p) {
  if constexpr (sizeof(T) == 4) {
    return *reinterpret_cast<const float*>(p);
  } else {
    return __builtin_bit_cast(float, (uint32_t)*reinterpret_cast<const uint16_t*>(p) << 16);
  }
}

// 16 bytes of T from floats (bf16: rounded to nearest even).
template <typename T>
__device__ __forceinline__ void store_vec(char* p, const float (&x)[16 / sizeof(T)]) {
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<f32x4_t*>(p) = f32x4_t{x[0], x[1], x[2], x[3]};
  } else {
    u32x4_t v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = pack_bf16x2(x[2 * i], x[2 * i + 1]);
    *reinterpret_cast<u32x4_t*>(p) = v;
  }
}

// The same past the caches (data read once, larger than they hold).
template <typename T>
__device__ __forceinline__ void load_vec_nt(const char* p, float (&x)[16 / sizeof(T)]) {
  const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
  if constexpr (sizeof(T) == 4) {
    const f32x4_t f = __builtin_bit_cast(f32x4_t, v);
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = f[i];
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t w = v[i];
      x[2 * i] = __builtin_bit_cast(float, w << 16);
      x[2 * i + 1] = __builtin_bit_cast(float, w & 0xffff0000u);
    }
  }
}

// *status = 1 (the caller has cleared it) if some target is neither ignore
// nor in [0, V).
__global__ __launch_bounds__(256) void ce_check_kernel(const int64_t* target, int64_t T, int64_t V,
                                                       int64_t ignore, int32_t* status) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= T) return;
  const int64_t y = target[t];
  if (y != ignore && (y < 0 || y >= V)) *status = 1;
}

// Block-wide merge of per-thread (m, d) states; result valid in all threads.
__device__ __forceinline__ void block_lse_merge(float& m, float& d, float* sm) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) lse_merge(m, d, __shfl_xor(m, o), __shfl_xor(d, o));
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    sm[2 * w] = m;
    sm[2 * w + 1] = d;
  }
  __syncthreads();
  m = kNegBig;
  d = 0.f;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) lse_merge(m, d, sm[2 * i], sm[2 * i + 1]);
}

// HBM-bound: the logits of the counted rows are read once.  kNt: with loads
// past the caches, for logits larger than the 256 MB Infinity Cache (2048 x
// 151936 fp32 150 -> 137 us, 4096 x 128256 bf16 182 -> 160 us: 6.6 TB/s); smaller
// ones may lie in it (1000 x 32003 bf16 12.9 against 13.6 us) and the backward
// reads them again.  status null: the targets have been checked
// (ce_check_kernel).
template <typename T, bool kNt>
__global__ __launch_bounds__(256) void ce_forward_kernel(const char* logits, int64_t V, int64_t ld_b,
                                                         const int64_t* target, int64_t ignore,
                                                         float* loss, float* lse, int32_t* status) {
  constexpr int E = sizeof(T), VEC = 16 / E;
  __shared__ float sm[16];
  const int64_t t = blockIdx.x;
  const int64_t y = target[t];
  if (y == ignore) {
    if (threadIdx.x == 0) {
      loss[t] = 0.0f;
      lse[t] = 0.0f;
    }
    return;
  }
  if (y < 0 || y >= V) {
    if (threadIdx.x == 0) {
      if (status) atomicOr(status, 1);
      loss[t] = 0.0f;
      lse[t] = 0.0f;
    }
    return;
  }
  const char* row = logits + t * ld_b;
  float m = kNegBig, d = 0.f;
  // scalar head up to 16-byte alignment, 16-byte vectors, scalar tail
  const int64_t mis = (int64_t)(reinterpret_cast<uintptr_t>(row) & 15u) / E;
  const int64_t head = mis ? min<int64_t>(VEC - mis, V) : 0;
  const int64_t nvec = (V - head) / VEC;
  const char* vrow = row + head * E;
  auto merge_vec = [&](const float (&x)[VEC]) __attribute__((always_inline)) {
    float mx = x[0];
#pragma unroll
    for (int j = 1; j < VEC; ++j) mx = fmaxf(mx, x[j]);
    const float mn = fmaxf(m, mx * kLog2e);
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < VEC; ++j) s += fast_exp2(fmaf(x[j], kLog2e, -mn));
    d = fmaf(d, fast_exp2(m - mn), s);
    m = mn;
  };
  // four 16-byte loads in flight per thread
  int64_t i = threadIdx.x;
  for (; i + 3 * 256 < nvec; i += 4 * 256) {
    float x[4][VEC];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if constexpr (kNt) load_vec_nt<T>(vrow + (i + k * 256) * 16, x[k]);
      else load_vec<T>(vrow + (i + k * 256) * 16, x[k]);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) merge_vec(x[k]);
  }
  for (; i < nvec; i += 256) {
    float x[VEC];
    load_vec<T>(vrow + i * 16, x);
    merge_vec(x);
  }
  for (int64_t v = threadIdx.x; v < head; v += 256) lse_merge(m, d, load_one<T>(row + v * E) * kLog2e, 1.0f);
  for (int64_t v = head + nvec * VEC + threadIdx.x; v < V; v += 256)
    lse_merge(m, d, load_one<T>(row + v * E) * kLog2e, 1.0f);
  block_lse_merge(m, d, sm);
  if (threadIdx.x == 0) {
    const float L = (m + fast_log2(d)) * kLn2;
    lse[t] = L;
    loss[t] = L - load_one<T>(row + y * E);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void ce_backward_kernel(const char* logits, int64_t V, int64_t ld_b,
                                                          const int64_t* target, int64_t ignore,
                                                          const float* lse, const float* grad,
                                                          int64_t gstride, char* dlogits,
                                                          int64_t ldd_b) {
  constexpr int E = sizeof(T);
  const int64_t t = blockIdx.x;
  const int64_t y = target[t];
  const bool valid = y != ignore && y >= 0 && y < V;
  const float g = valid ? grad[t * gstride] : 0.f;
  const float l2 = valid ? lse[t] * kLog2e : 0.f;
  const char* row = logits + t * ld_b;
  char* drow = dlogits + t * ldd_b;
  constexpr int VEC = 16 / E;
  if (((reinterpret_cast<uintptr_t>(row) ^ reinterpret_cast<uintptr_t>(drow)) & 15u) == 0) {
    // logits and gradient row alike within 16 bytes (the usual case: the same
    // pitch, also an odd one): up to VEC - 1 elements one by one to the next
    // 16-byte boundary, whole vectors with four loads in flight per thread,
    // then the rest of the row.  (An odd row went two elements at a time: 1000 x
    // 32003 bf16, 30% of the rows ignored, 46 us, now 19 us, call after call.)
    const int64_t mis = (int64_t)(reinterpret_cast<uintptr_t>(row) & 15u) / E;
    const int64_t head = mis ? min<int64_t>(VEC - mis, V) : 0;
    const int64_t nvec = (V - head) / VEC;
    const char* vrow = row + head * E;
    char* vdrow = drow + head * E;
    auto grad_vec = [&](float (&x)[VEC], int64_t c0) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        const float p = fast_exp2(fmaf(x[j], kLog2e, -l2));
        x[j] = valid ? g * (p - (c0 + j == y ? 1.f : 0.f)) : 0.f;
      }
    };
    auto grad_one = [&](int64_t c) __attribute__((always_inline)) {
      float r = 0.f;
      if (valid) r = g * (fast_exp2(fmaf(load_one<T>(row + c * E), kLog2e, -l2)) - (c == y ? 1.f : 0.f));
      if constexpr (E == 4)
        reinterpret_cast<float*>(drow)[c] = r;
      else
        *reinterpret_cast<uint16_t*>(drow + c * 2) = (uint16_t)(pack_bf16x2(r, 0.f) & 0xffffu);
    };
    int64_t i = threadIdx.x;
    for (; i + 3 * 256 < nvec; i += 4 * 256) {
      float x[4][VEC];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (valid) load_vec<T>(vrow + (i + k * 256) * 16, x[k]);
        else
#pragma unroll
          for (int j = 0; j < VEC; ++j) x[k][j] = 0.f;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        grad_vec(x[k], head + (i + k * 256) * VEC);
        store_vec<T>(vdrow + (i + k * 256) * 16, x[k]);
      }
    }
    for (; i < nvec; i += 256) {
      float x[VEC];
      if (valid) load_vec<T>(vrow + i * 16, x);
      else
#pragma unroll
        for (int j = 0; j < VEC; ++j) x[j] = 0.f;
      grad_vec(x, head + i * VEC);
      store_vec<T>(vdrow + i * 16, x);
    }
    if ((int64_t)threadIdx.x < head) grad_one(threadIdx.x);
    for (int64_t c = head + nvec * VEC + threadIdx.x; c < V; c += 256) grad_one(c);
    return;
  }
  // any alignment: pairs of elements so bf16 rows are written 4 bytes at a time
  for (int64_t v = 2 * threadIdx.x; v < V; v += 512) {
    float o[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t c = v + j;
      float r = 0.f;
      if (valid && c < V) {
        const float p = fast_exp2(fmaf(load_one<T>(row + c * E), kLog2e, -l2));
        r = g * (p - (c == y ? 1.f : 0.f));
      }
      o[j] = r;
    }
    if constexpr (E == 4) {
      reinterpret_cast<float*>(drow)[v] = o[0];
      if (v + 1 < V) reinterpret_cast<float*>(drow)[v + 1] = o[1];
    } else {
      const uint32_t pk = pack_bf16x2(o[0], o[1]);
      char* p = drow + v * 2;
      if (v + 1 < V && (reinterpret_cast<uintptr_t>(p) & 3u) == 0) {
        *reinterpret_cast<uint32_t*>(p) = pk;
      } else {
        *reinterpret_cast<uint16_t*>(p) = (uint16_t)(pk & 0xffffu);
        if (v + 1 < V) *reinterpret_cast<uint16_t*>(p + 2) = (uint16_t)(pk >> 16);
      }
    }
  }
}

}  // namespace mtf

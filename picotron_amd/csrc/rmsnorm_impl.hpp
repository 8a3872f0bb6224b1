// RMSNorm forward and backward kernels for gfx950.  Templates only: the per-storage-type
// launchers are instantiated in rmsnorm_{fwd,bwd}_{f32,f16,bf16}.hip (compiled in
// parallel) and called from the C ABI in rmsnorm.hip.
//
// Reference semantics (AndyMLAndAI/picotron):
//   forward  src/picotron/nn/triton_kernels/rmsnorm.py:49-60   r = rsqrt(mean(x^2) + eps),
//            y = (x * r) * w in fp32, stored in x's type
//   backward src/picotron/nn/triton_kernels/rmsnorm.py:110-134
//            wg = g * w; dm = mean(wg * x); dx = r * (wg - (x * r^2) * dm);
//            dW = sum_rows((g * x) * r)
//
// Layout: rows are `cols` contiguous elements, consecutive rows `*_row_stride` apart.
// A row is owned by WPR waves (64*WPR lanes), or by 16 lanes of a wave that holds four rows
// (WPR 0).  Lane `rl` of the row holds the 16-byte vectors rl, rl + LANES, ... (VPL of them),
// so each wave instruction moves 1 KiB of memory, and the whole row stays in registers (packed
// in its storage type) between the reduction and the elementwise pass: x and dy are read from
// HBM once.
//
// ALIGNED rows are whole 16-byte vectors on 16-byte boundaries.  Other rows -- any hidden size,
// stride and base -- take the same vectors from the row's first element at whatever address that
// is (global accesses of the element's alignment, which gfx950 serves unaligned), and the
// hidden size's remainder of fewer than VEC elements one per lane.  [16383, 1370] bf16: forward
// 18 us (the bytes at copy speed: 14), backward 31, against 62 and 72 for element-wide accesses
// of the same lanes (each wave instruction then moves 128 bytes spread over a kilobyte).
//
// Backward weight gradient: each block accumulates sum((g*x)*r) for its rows in fp32
// registers, combines its row slots in LDS in slot order, and writes one fp32 partial
// row to the workspace; a second kernel sums the partial rows in a fixed order.  No
// atomics, so dW is bitwise reproducible for a given (rows, cols).
#pragma once

#include <cstdlib>
#include <string>
#include <type_traits>

#include "pt_common.hpp"

namespace pt {
namespace rmsnorm {

// Waves per block: the backward uses 8 (one weight-gradient partial per 8 waves) and the
// forward 4, or in both cases as many as a row spans when that is more.
constexpr int kBwdWaves = 8;
constexpr int kFwdWaves = 4;
// Cache policy of the row loads (x, dy): nontemporal, the measured optimum on MI355X for data
// read once per kernel.  The row stores: RowStore.
constexpr bool kLoadNT = true;

// ------------------------------------------------------------------ device helpers

// 32 bytes that a lane without a vector of its own reads instead, where a row may be shorter than
// one vector (its value is never used).
static __device__ __align__(16) unsigned int kPad[8];

// True if vector k of lane rl lies wholly inside the row.  For rows of whole vectors the test is
// the one of their loads, so that the compiler keeps one mask for both.
template <typename T, int LANES, bool ALIGNED>
__device__ __forceinline__ bool in_row(int rl, int k, int cols) {
  const int e = (rl + k * LANES) * Elem<T>::VEC;
  return ALIGNED ? e < cols : e + Elem<T>::VEC <= cols;
}

// The remainder element of this lane (rows that are not whole vectors): its column, or -1.
template <typename T>
__device__ __forceinline__ int tail_col(int rl, int cols) {
  const int tail = cols % Elem<T>::VEC;
  return rl < tail ? cols - tail + rl : -1;
}

// A lane's weights kept as loaded and converted to fp32 at each use, which halves their
// registers for 16-bit weights: 16-byte words, branch-free (a vector past the row end loads
// something else; its products are never stored or summed), so that the loads issue back to back
// and their one wait comes at first use.  WT == void: a runtime weight type, loaded by elements
// into fp32, zero past the row end.
template <typename T, typename WT, int VPL, int LANES, bool ALIGNED>
struct LaneWeights {
  static constexpr int N = Elem<T>::VEC;
  static constexpr int kPer = 16 / static_cast<int>(sizeof(WT));  // weights per 16-byte word
  static constexpr int kWords = N / kPer;
  static_assert(kWords * kPer == N, "weights of one vector fill whole 16-byte words");
  union Word {
    u32x4 raw;
    WT e[kPer];
  };
  Word wd[VPL][kWords];
  float tail;
  __device__ __forceinline__ void load(const void* w, int, int rl, int cols) {
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int e = (rl + k * LANES) * N;
      const WT* p = reinterpret_cast<const WT*>(w);
      if constexpr (ALIGNED) {
        p += e < cols ? e : 0;
      } else {
        p = in_row<T, LANES, ALIGNED>(rl, k, cols) ? p + e : reinterpret_cast<const WT*>(kPad);
      }
#pragma unroll
      for (int l = 0; l < kWords; ++l) wd[k][l].raw = load_vec<WT, ALIGNED, false>(p + l * kPer);
    }
    if constexpr (!ALIGNED) {
      const int c = tail_col<T>(rl, cols);
      tail = static_cast<float>(reinterpret_cast<const WT*>(w)[c < 0 ? 0 : c]);
    }
  }
  __device__ __forceinline__ float at(int k, int i) const {
    return static_cast<float>(wd[k][i / kPer].e[i % kPer]);
  }
};

template <typename T, int VPL, int LANES, bool ALIGNED>
struct LaneWeights<T, void, VPL, LANES, ALIGNED> {
  static constexpr int N = Elem<T>::VEC;
  float f[VPL][N];
  float tail;
  __device__ __forceinline__ void load(const void* w, int wdt, int rl, int cols) {
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const bool in = in_row<T, LANES, ALIGNED>(rl, k, cols);
#pragma unroll
      for (int i = 0; i < N; ++i) f[k][i] = in ? load_any(w, (rl + k * LANES) * N + i, wdt) : 0.0f;
    }
    const int c = tail_col<T>(rl, cols);
    tail = load_any(w, c < 0 ? 0 : c, wdt);
  }
  __device__ __forceinline__ float at(int k, int i) const { return f[k][i]; }
};

// The 16-byte vectors of one row held by a lane, packed in the storage type, and its remainder
// element (rows that are not whole vectors).
template <typename T, int VPL>
struct RowRegs {
  Vec16<T> v[VPL];
  T tail;

  __device__ __forceinline__ float at(int k, int i) const { return Elem<T>::to_f32(v[k].e[i]); }

  // Tells the compiler the packed words may have changed, so fp32 values converted
  // before this point are not kept alive past it (they are re-derived from the packed
  // words instead).  Keeps the row at 2 bytes/element of registers across the
  // reduction for 16-bit types.
  __device__ __forceinline__ void opaque() {
#pragma unroll
    for (int k = 0; k < VPL; ++k) asm volatile("" : "+v"(v[k].raw));
  }
};

// Stand-in for an absent row buffer (template variants without a residual stream).
struct NoRegs {
  __device__ __forceinline__ void opaque() {}
};

// Residual stream of the fused add + norm (decoder block: h = x + res, then norm(h)).
template <typename T>
struct ResidualIn {
  const T* res;
  int64_t res_stride;
  T* h;
  int64_t h_stride;
};

// Incoming gradient of h added to the norm's input gradient (h also feeds the block's
// final residual add): dh = norm_backward(dy) + dh_in.
template <typename T>
struct ResidualGrad {
  const T* dh_in;
  int64_t dh_in_stride;
};

// Loads the lane's part of a row, branch-free and unmasked: a lane whose vector (or remainder
// element) lies past the row end loads something else instead -- the row's first vector, or
// kPad where the row may hold none -- and the caller ignores it (in_row(), tail_col()).  Nothing
// may consume the loaded registers here: loads under divergent branches, or a select right after
// them, make the compiler wait for the data at load time and so drain the next row's prefetch.
template <typename T, int VPL, int LANES, bool ALIGNED, bool NT>
__device__ __forceinline__ void load_row(const T* __restrict__ row, int rl, int cols,
                                         RowRegs<T, VPL>& r) {
#pragma unroll
  for (int k = 0; k < VPL; ++k) {
    const int e = (rl + k * LANES) * Elem<T>::VEC;
    if constexpr (ALIGNED) {
      r.v[k].raw = load16<NT>(row + (e < cols ? e : 0));
    } else {
      const T* p = in_row<T, LANES, ALIGNED>(rl, k, cols) ? row + e : reinterpret_cast<const T*>(kPad);
      r.v[k].raw = load_vec<T, false, NT>(p);
    }
  }
  if constexpr (!ALIGNED) {
    const int c = tail_col<T>(rl, cols);
    r.tail = row[c < 0 ? 0 : c];
  }
}

// Stores of one row's vectors.  Aligned rows: buffer stores with cache policy POLICY through a
// resource over the row, whose base is wave-uniform (all lanes of a wave work on the same row);
// the resource's range check drops vectors past the row end, so the stores need no branch.
// Other rows: nontemporal global stores of the vectors inside the row and of the remainder
// elements (the ends of neighbouring rows share lines, which L2 then merges).
// The forward's stores are write-through (kWriteThrough: 43.9 against 44.3 us per launch at
// [16384, 4096] bf16), the backward's nontemporal (kNonTemporal: 71.9 against 72.2 us: with
// two read streams beside it, write-through costs more than it saves).
template <typename T, int LANES, bool ALIGNED, int POLICY>
struct RowStore {
  T* row;
  int cols;
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ RowStore(T* r, int c) : row(r), cols(c) {
    if constexpr (ALIGNED) rsrc = uniform_buffer(r, c * static_cast<int>(sizeof(T)));
  }
  __device__ __forceinline__ void store(int rl, int k, const float (&o)[Elem<T>::VEC]) const {
    constexpr int V = Elem<T>::VEC;
    const int e = (rl + k * LANES) * V;
    Vec16<T> v;
#pragma unroll
    for (int i = 0; i < V; ++i) v.e[i] = Elem<T>::from_f32(o[i]);
    if constexpr (ALIGNED) {
      __builtin_amdgcn_raw_buffer_store_b128(v.raw, rsrc, e * static_cast<int>(sizeof(T)), 0,
                                             POLICY);
    } else if (in_row<T, LANES, ALIGNED>(rl, k, cols)) {
      store_vec<T, false, true>(row + e, v.raw);
    }
  }
  __device__ __forceinline__ void store_tail(int rl, float o) const {
    const int c = tail_col<T>(rl, cols);
    if (c >= 0) row[c] = Elem<T>::from_f32(o);
  }
};

// Sum over the WPR waves (or, for WPR 0, the 16 lanes) that share a row.  `red` holds 2*WAVES
// floats; `buf` alternates between consecutive calls so one barrier per row suffices (a wave cannot overwrite a
// buffer before every wave has passed the barrier of the call in between).  Waves sum the
// partials of their row in wave order, so every wave of a row gets the same value.
template <int WPR, int WAVES>
__device__ __forceinline__ float row_sum(float v, float* red, int wave, int lane, int buf) {
  if constexpr (WPR == 0) return row16_sum(v);
  v = wave_sum(v);
  if constexpr (WPR > 1) {
    float* b = red + buf * WAVES;
    if (lane == 0) b[wave] = v;
    __syncthreads();
    const int first = (wave / WPR) * WPR;
    float t = 0.0f;
#pragma unroll
    for (int i = 0; i < WPR; ++i) t += b[first + i];
    v = t;
  }
  return v;
}

// Lanes of a row and row slots of a workgroup of `waves` waves.
constexpr __host__ __device__ int row_lanes(int wpr) { return wpr == 0 ? 16 : 64 * wpr; }
constexpr __host__ __device__ int row_slots(int wpr, int waves) { return waves * 64 / row_lanes(wpr); }

// ------------------------------------------------------------------ forward
//
// Row groups: a block has row_slots(WPR, WAVES) row slots; at step `it` block b works on the group of
// rows starting at (it * gridDim.x + b) * slots, so at any moment all blocks work on one
// compact window of rows (DRAM-friendly, like a non-persistent grid).  With a grid that
// covers every row once (the default) each wave handles one row; smaller grids loop, and
// the next row is then loaded into the second register buffer before the current one is
// reduced (PERSIST).  Weights are loaded once per wave, kept packed.  Without PERSIST the
// kernel holds one row buffer only: fewer registers, more waves in flight per CU.

// ADD: the fused residual add.  h = x + res is computed in fp32, rounded to the storage
// type and written; the norm is taken of the rounded h, as the unfused graph normalises the
// stored sum.

template <typename T, typename WT, int VPL, int WPR, int WAVES, bool ALIGNED, bool LOAD_NT,
          bool PERSIST, bool ADD>
__global__ __launch_bounds__(WAVES * 64) void rmsnorm_fwd_kernel(
    const T* __restrict__ x, int64_t xs, const void* __restrict__ w, int wdt, T* __restrict__ y,
    int64_t ys, float* __restrict__ rstd, int64_t rows, int cols, float eps, int iters,
    ResidualIn<T> rin) {
  static_assert(WPR == 0 ? !ALIGNED : WAVES % WPR == 0, "row slots must tile the block");
  constexpr int V = Elem<T>::VEC;
  constexpr int RPB = row_slots(WPR, WAVES);
  constexpr int LANES = row_lanes(WPR);
  __shared__ float red[2 * WAVES];

  const int wave = threadIdx.x / 64;
  const int lane = threadIdx.x % 64;
  const int slot = threadIdx.x / LANES;
  const int rl = threadIdx.x % LANES;
  // iters = ceil(rows / group_stride), computed on the host: the same for every wave.
  const int64_t group_stride = static_cast<int64_t>(gridDim.x) * RPB;
  const int64_t r1 = rows;
  const float inv_cols = 1.0f / static_cast<float>(cols);
  const bool has_tail = !ALIGNED && tail_col<T>(rl, cols) >= 0;

  LaneWeights<T, WT, VPL, LANES, ALIGNED> wv;
  wv.load(w, wdt, rl, cols);
  // Long rows (eight vectors per lane, or four of several waves): every weight before the row.  Left alone,
  // the compiler issues the first vectors' weights behind the row's loads, and the first store waits for
  // them: [16384, 4096] fp32 88.4 us against 86.0, [2048, 4096] 13.8 against 13.2, [512, 8192] 8.1 against
  // 7.2; bf16 [512, 16384] 8.2 against 7.8, [512, 12288] 6.8 against 6.5.  (Shorter rows, [512, 2048] bf16 2.6
  // against 2.95, and the residual form gain and lose by it in turn.)
  if constexpr (!ADD && (VPL == 8 || (VPL == 4 && WPR > 1))) __builtin_amdgcn_sched_barrier(0);

  using ResRegs = std::conditional_t<ADD, RowRegs<T, VPL>, NoRegs>;
  struct Row {
    RowRegs<T, VPL> x;
    ResRegs res;
  };
  auto process = [&](Row& rw, int64_t row, int buf) {
    RowRegs<T, VPL>& xr = rw.x;
    const bool active = row < r1;
    if constexpr (ADD) {
      const RowStore<T, LANES, ALIGNED, kWriteThrough> hs(rin.h + row * rin.h_stride, cols);
#pragma unroll
      for (int k = 0; k < VPL; ++k) {
        float o[V];
#pragma unroll
        for (int i = 0; i < V; ++i) {
          xr.v[k].e[i] = Elem<T>::from_f32(xr.at(k, i) + rw.res.at(k, i));
          o[i] = xr.at(k, i);
        }
        if (active) hs.store(rl, k, o);
      }
      if constexpr (!ALIGNED) {
        xr.tail = Elem<T>::from_f32(Elem<T>::to_f32(xr.tail) + Elem<T>::to_f32(rw.res.tail));
        if (active) hs.store_tail(rl, Elem<T>::to_f32(xr.tail));
      }
    }
    // Rows that two kernels take by their count (short_row_fwd, fwd_vpl_cap_for) get the same bits from
    // both: 16 lanes sum each 16 vectors of their row apart and add the sums in order, as one wave
    // does (wave_sum), and one wave sums every other 64 vectors apart, as two waves do (row_sum).
    constexpr int kParts =
        WPR == 0 ? VPL : (ALIGNED && WPR == 1 && VPL == 8 && sizeof(T) == 4 ? 2 : 1);
    float ss[kParts] = {};
    if (active) {
#pragma unroll
      for (int k = 0; k < VPL; ++k) {
        float part = 0.0f;
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const float f = xr.at(k, i);
          part += f * f;
        }
        ss[k % kParts] += in_row<T, LANES, ALIGNED>(rl, k, cols) ? part : 0.0f;
      }
      if constexpr (!ALIGNED) {
        const float f = Elem<T>::to_f32(xr.tail);
        ss[0] += has_tail ? f * f : 0.0f;
      }
    }
    xr.opaque();
    float sum = row_sum<WPR, WAVES>(ss[0], red, wave, lane, buf);
#pragma unroll
    for (int p = 1; p < kParts; ++p) sum += row_sum<WPR, WAVES>(ss[p], red, wave, lane, buf);
    if (!active) return;
    const float r = 1.0f / sqrtf(sum * inv_cols + eps);
    if (rl == 0) rstd[row] = r;
    const RowStore<T, LANES, ALIGNED, kWriteThrough> yst(y + row * ys, cols);
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      float o[V];
#pragma unroll
      for (int i = 0; i < V; ++i) o[i] = (xr.at(k, i) * r) * wv.at(k, i);
      yst.store(rl, k, o);
    }
    if constexpr (!ALIGNED) yst.store_tail(rl, (Elem<T>::to_f32(xr.tail) * r) * wv.tail);
  };

  // Rows past the end are clamped to the last row for loading (keeping the loads
  // unconditional) and skipped by process().
  auto load = [&](Row& rw, int64_t row) {
    const int64_t lr = row < r1 ? row : r1 - 1;
    load_row<T, VPL, LANES, ALIGNED, LOAD_NT>(x + lr * xs, rl, cols, rw.x);
    if constexpr (ADD)
      load_row<T, VPL, LANES, ALIGNED, LOAD_NT>(rin.res + lr * rin.res_stride, rl, cols, rw.res);
  };
  int64_t ra = static_cast<int64_t>(blockIdx.x) * RPB + slot;
  if constexpr (!PERSIST) {
    Row a;
    load(a, ra);
    process(a, ra, 0);
  } else {
    // Unconditional prefetches inside the loop, the last one or two rows peeled (as in the
    // backward: a prefetch under a branch makes the compiler wait for it at the join).
    Row a, b;
    load(a, ra);
    int it = 0;
    for (; it + 2 < iters; it += 2) {
      const int64_t rb = ra + group_stride;
      load(b, rb);
      process(a, ra, 0);
      const int64_t rc = rb + group_stride;
      load(a, rc);
      process(b, rb, 1);
      ra = rc;
    }
    if (it + 1 < iters) {
      const int64_t rb = ra + group_stride;
      load(b, rb);
      process(a, ra, 0);
      process(b, rb, 1);
    } else {
      process(a, ra, 0);
    }
  }
}

// ------------------------------------------------------------------ weight-gradient sum
//
// dW[c] = sum_p partial[p][c] in a fixed order, cast to the weight type: 256 threads cover
// kFinishCols columns with kFinishGroups groups of 32 lanes; group g sums p = g, g+8, ... in
// increasing p (up to 64 loads in flight per lane: one round trip at 512 partials), then the
// groups are added in group order (rmsnorm_dw_finish_kernel).
constexpr int kFinishCols = 32;
constexpr int kFinishGroups = 8;

__device__ __forceinline__ float column_group_sum(const float* __restrict__ partial,
                                                  int64_t nparts, int cols, int c, int grp) {
  constexpr int kUnroll = 64;
  const float* p = partial + c;
  float s = 0.0f;
  int64_t i = grp;
  for (; i + static_cast<int64_t>(kFinishGroups) * (kUnroll - 1) < nparts;
       i += static_cast<int64_t>(kFinishGroups) * kUnroll) {
    float v[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) v[u] = p[(i + u * kFinishGroups) * cols];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) s += v[u];
  }
  // The remainder (fewer than kUnroll partials per group) in batches of 16 independent loads: whole
  // ones, then one filled up with the group's last partial, counted as 0 -- a few round trips rather than
  // one per partial.  Whole batches without clamps, and the clamp as a running offset: a multiplied and
  // selected index for each load costs 0.4 to 0.9 us per call ([16, 2048] and [512, 1024] fp32).
  constexpr int kRest = 16;
  const int64_t step = static_cast<int64_t>(kFinishGroups) * cols;
  for (; i + static_cast<int64_t>(kFinishGroups) * (kRest - 1) < nparts;
       i += static_cast<int64_t>(kFinishGroups) * kRest) {
    const float* q = p + i * cols;
    float v[kRest];
#pragma unroll
    for (int u = 0; u < kRest; ++u) v[u] = q[u * step];
#pragma unroll
    for (int u = 0; u < kRest; ++u) s += v[u];
  }
  if (i < nparts) {
    const int left = static_cast<int>((nparts - 1 - i) / kFinishGroups) + 1;
    const float* q = p + i * cols;
    float v[kRest];
#pragma unroll
    for (int u = 0; u < kRest; ++u) {
      if (u > 0) q += u < left ? step : 0;
      v[u] = *q;
    }
#pragma unroll
    for (int u = 0; u < kRest; ++u) s += u < left ? v[u] : 0.0f;
  }
  return s;
}

__global__ __launch_bounds__(256) void rmsnorm_dw_finish_kernel(const float* __restrict__ partial,
                                                                int64_t nparts, int cols,
                                                                void* __restrict__ dw, int wdt);

// ------------------------------------------------------------------ backward
//
// Persistent blocks walking the same interleaved row groups as the forward (step `it`:
// rows (it * gridDim.x + b) * slots + slot), with the next row double-buffered in
// registers.  Per row: dot = sum((g*w)*x) over the row (fp32, wave + LDS reduction),
// dx = r*((g*w) - (x*r^2)*dm) written from the registers, and sum((g*x)*r) accumulated
// per lane in fp32.  Spreading a row over WPR waves divides that accumulator (and the row
// registers) by WPR.  At the end the row slots are combined in LDS in slot order and the
// block writes one fp32 partial row; the partial count (the grid) is fixed for a given
// shape and tuning, so the weight gradient is reproducible.

// ADD: dx = norm_backward(dy) + dh_in, summed in fp32 and rounded once (the fused residual
// add's backward; dx may alias dh_in, each element being read before it is written by the
// same lane).

template <typename T, typename WT, int VPL, int WPR, int WAVES, bool ALIGNED, bool LOAD_NT,
          bool ADD>
__global__ __launch_bounds__(WAVES * 64) void rmsnorm_bwd_kernel(
    const T* __restrict__ dy, int64_t dys, const T* __restrict__ x, int64_t xs,
    const void* __restrict__ w, int wdt, const float* __restrict__ rstd, T* dx,
    int64_t dxs, float* __restrict__ partial, int64_t rows, int cols, int iters,
    ResidualGrad<T> rg) {
  static_assert(WPR == 0 ? !ALIGNED : WAVES % WPR == 0, "row slots must tile the block");
  constexpr int V = Elem<T>::VEC;
  constexpr int RPB = row_slots(WPR, WAVES);
  constexpr int LANES = row_lanes(WPR);
  __shared__ float red[2 * WAVES];
  extern __shared__ float lds_dw[];  // [cols] when RPB > 1 and partial != nullptr

  const int wave = threadIdx.x / 64;
  const int lane = threadIdx.x % 64;
  const int slot = threadIdx.x / LANES;
  const int rl = threadIdx.x % LANES;
  // iters = ceil(rows / group_stride), computed on the host: the same for every wave.
  const int64_t group_stride = static_cast<int64_t>(gridDim.x) * RPB;
  const int64_t r1 = rows;
  const bool want_dw = partial != nullptr;
  const float inv_cols = 1.0f / static_cast<float>(cols);
  const bool has_tail = !ALIGNED && tail_col<T>(rl, cols) >= 0;

  float wv[VPL][V], wtail = 0.0f;
  {
    LaneWeights<T, WT, VPL, LANES, ALIGNED> lw;
    lw.load(w, wdt, rl, cols);
#pragma unroll
    for (int k = 0; k < VPL; ++k)
#pragma unroll
      for (int i = 0; i < V; ++i) wv[k][i] = lw.at(k, i);
    if constexpr (!ALIGNED) wtail = lw.tail;
  }
  float acc[VPL][V], acc_tail = 0.0f;
#pragma unroll
  for (int k = 0; k < VPL; ++k)
#pragma unroll
    for (int i = 0; i < V; ++i) acc[k][i] = 0.0f;

  using ResRegs = std::conditional_t<ADD, RowRegs<T, VPL>, NoRegs>;
  struct Buf {
    RowRegs<T, VPL> g, x;
    ResRegs d;
    float r;
  };
  // Rows past the end are clamped to the last row for loading (keeping the loads
  // unconditional) and skipped by process().
  auto load = [&](Buf& bf, int64_t row) {
    const int64_t lr = row < r1 ? row : r1 - 1;
    load_row<T, VPL, LANES, ALIGNED, LOAD_NT>(dy + lr * dys, rl, cols, bf.g);
    load_row<T, VPL, LANES, ALIGNED, LOAD_NT>(x + lr * xs, rl, cols, bf.x);
    if constexpr (ADD)
      load_row<T, VPL, LANES, ALIGNED, LOAD_NT>(rg.dh_in + lr * rg.dh_in_stride, rl, cols, bf.d);
    bf.r = rstd[lr];
  };
  auto process = [&](Buf& bf, int64_t row, int buf) {
    const bool active = row < r1;
    float dot = 0.0f;
    if (active) {
#pragma unroll
      for (int k = 0; k < VPL; ++k) {
        float part = 0.0f;
#pragma unroll
        for (int i = 0; i < V; ++i) part += (bf.g.at(k, i) * wv[k][i]) * bf.x.at(k, i);
        dot += in_row<T, LANES, ALIGNED>(rl, k, cols) ? part : 0.0f;
      }
      if constexpr (!ALIGNED) {
        const float part = (Elem<T>::to_f32(bf.g.tail) * wtail) * Elem<T>::to_f32(bf.x.tail);
        dot += has_tail ? part : 0.0f;
      }
    }
    bf.g.opaque();
    bf.x.opaque();
    bf.d.opaque();
    dot = row_sum<WPR, WAVES>(dot, red, wave, lane, buf);
    if (!active) return;
    const float r = bf.r;
    const float dm = dot * inv_cols;
    const float r2 = r * r;
    if (dx != nullptr) {
      const RowStore<T, LANES, ALIGNED, kNonTemporal> dxst(dx + row * dxs, cols);
#pragma unroll
      for (int k = 0; k < VPL; ++k) {
        float o[V];
#pragma unroll
        for (int i = 0; i < V; ++i) {
          o[i] = r * (bf.g.at(k, i) * wv[k][i] - (bf.x.at(k, i) * r2) * dm);
          if constexpr (ADD) o[i] += bf.d.at(k, i);
        }
        dxst.store(rl, k, o);
      }
      if constexpr (!ALIGNED) {
        float o = r * (Elem<T>::to_f32(bf.g.tail) * wtail - (Elem<T>::to_f32(bf.x.tail) * r2) * dm);
        if constexpr (ADD) o += Elem<T>::to_f32(bf.d.tail);
        dxst.store_tail(rl, o);
      }
    }
    if (want_dw) {
#pragma unroll
      for (int k = 0; k < VPL; ++k)
#pragma unroll
        for (int i = 0; i < V; ++i) acc[k][i] += (bf.g.at(k, i) * bf.x.at(k, i)) * r;
      if constexpr (!ALIGNED)
        acc_tail += (Elem<T>::to_f32(bf.g.tail) * Elem<T>::to_f32(bf.x.tail)) * r;
    }
  };

  // The next row is double-buffered in registers.  The loop body issues its two prefetches
  // unconditionally (both rows are within the block's iterations), so the wait for the row
  // being reduced counts only that row's loads: a prefetch under a branch would make the
  // compiler wait for everything at the join.  The last one or two rows are peeled.
  int64_t ra = static_cast<int64_t>(blockIdx.x) * RPB + slot;
  Buf a, b;
  load(a, ra);
  int it = 0;
  for (; it + 2 < iters; it += 2) {
    const int64_t rb = ra + group_stride;
    load(b, rb);
    process(a, ra, 0);
    const int64_t rc = rb + group_stride;
    load(a, rc);
    process(b, rb, 1);
    ra = rc;
  }
  if (it + 1 < iters) {
    const int64_t rb = ra + group_stride;
    load(b, rb);
    process(a, ra, 0);
    process(b, rb, 1);
  } else {
    process(a, ra, 0);
  }
  if (!want_dw) return;

  float* prow = partial + static_cast<int64_t>(blockIdx.x) * cols;
  if constexpr (WPR == 0) {
    // A wave's four rows hold the same columns: lanes 0-15 get their sum.
#pragma unroll
    for (int k = 0; k < VPL; ++k)
#pragma unroll
      for (int i = 0; i < V; ++i) acc[k][i] = quarters_sum(acc[k][i]);
    acc_tail = quarters_sum(acc_tail);
  }
  const int tail_c = ALIGNED ? -1 : tail_col<T>(rl, cols);
  if constexpr (RPB == 1) {
    // The block's single row slot: each lane owns distinct columns.
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int e = (rl + k * LANES) * V;
#pragma unroll
      for (int i = 0; i < V; ++i)
        if (in_row<T, LANES, ALIGNED>(rl, k, cols)) prow[e + i] = acc[k][i];
    }
    if (tail_c >= 0) prow[tail_c] = acc_tail;
  } else {
    // Row slots (for WPR 0, the waves) hold the same columns: combine them in LDS in slot order.
    constexpr int kSums = WPR == 0 ? WAVES : RPB;
    const int mine = WPR == 0 ? (lane < 16 ? wave : -1) : slot;
    for (int s = 0; s < kSums; ++s) {
      if (mine == s) {
#pragma unroll
        for (int k = 0; k < VPL; ++k) {
          const int e = (rl + k * LANES) * V;
#pragma unroll
          for (int i = 0; i < V; ++i) {
            if (in_row<T, LANES, ALIGNED>(rl, k, cols))
              lds_dw[e + i] = (s == 0) ? acc[k][i] : lds_dw[e + i] + acc[k][i];
          }
        }
        if (tail_c >= 0) lds_dw[tail_c] = (s == 0) ? acc_tail : lds_dw[tail_c] + acc_tail;
      }
      __syncthreads();
    }
    for (int c = threadIdx.x; c < cols; c += WAVES * 64) prow[c] = lds_dw[c];
  }
}

// ------------------------------------------------------------------ host-side shapes

struct Shape {
  int vpl = 0;  // 16-byte vectors per lane
  int wpr = 0;  // waves per row
};

// Launch tuning.  Defaults were chosen by measurement on MI355X; the environment can
// override them (PT_RMSNORM_FWD_VPL_CAP, PT_RMSNORM_BWD_VPL_CAP, PT_RMSNORM_FWD_BLOCKS_PER_CU,
// PT_RMSNORM_BWD_PARTIALS, PT_RMSNORM_FWD_OCCUPANCY, PT_RMSNORM_BWD_OCCUPANCY), read once
// per process.  The backward partial count fixes the
// weight-gradient summation order, so dW is reproducible for a given setting.
struct Tuning {
  int fwd_vpl_cap = 0;  // 0: by element size (fwd_vpl_cap_for)
  int bwd_vpl_cap = 0;  // 0: by row length (bwd_vpl_cap_for)
  int64_t fwd_blocks_per_cu = 0;  // 0: no cap (one row per row slot)
  int64_t bwd_partials = 0;  // 0: by the bytes of a row (bwd_partials_for)
  int fwd_occupancy = 0;  // resident forward workgroups per CU (0: no limit)
  int bwd_occupancy = 0;  // resident backward workgroups per CU (0: no limit)
};

// Backward vectors per lane: one for rows of at most 256 16-byte vectors (bf16 hidden
// <= 2048; measured 960: 40.7 -> 34.1 us, 2048: 64.2 -> 62.1 us per fwd+bwd layer at 16384
// rows), two above (4096: 116.0 against 117.8 with one), unless the environment sets it.
inline int bwd_vpl_cap_for(int tuned, int64_t cols, int vec) {
  if (tuned > 0) return tuned;
  return (cols + vec - 1) / vec <= 256 ? 1 : 2;
}

// Forward vectors per lane: 32 elements per lane, four 16-byte vectors of a 16-bit type and
// eight of fp32 (two waves per 4096-wide row either way); measured at [16384, 4096], 4 layers:
// bf16 0.4628-0.4639 ms per step against 0.4660-0.4684 with two and 0.4747-0.4763 with eight,
// fp32 0.8769-0.8777 ms against 0.8868-0.8871 with four.
// Aligned fp32 rows of 257-512 vectors hold four per lane of two waves instead of eight of one
// (the general kernels lose by it: [16384, 1370] 66.0 -> 67.9 with the add) where the rows leave CUs
// with little to do or fill all of them several times; in between one wave per row spreads evenly
// over the CUs, and the two waves' barrier only costs.  us, one wave against two, 2048 columns:
// plain / with the residual add 64 rows 2.7 2.5 / 3.9 3.2, 512 3.9 3.6 / 6.0 5.0, 1024 4.4 4.9 / 7.8 7.4,
// 2048 7.1 7.9 / 12.6 13.4, 3072 9.7 10.5 / 18.6 18.7, 4096 13.5 13.3 / 24.4 24.0, 16384 44.9 43.8 /
// 89.1 87.2; 1280 columns 512 3.4 3.1, 1024 3.9 4.0, 3072 7.1 8.0, 4096 9.9 9.5.
inline int fwd_vpl_cap_for(int tuned, int64_t rows, int64_t cols, int vec) {
  if (tuned > 0) return tuned;
  const int64_t nvec = (cols + vec - 1) / vec;
  const bool two_waves = rows < 1024 || rows >= 4096;
  return vec == 4 && nvec > 256 && nvec <= 512 && two_waves ? 4 : 32 / vec;
}

inline int64_t env_positive(const char* name, int64_t fallback) {
  const char* v = std::getenv(name);
  if (v == nullptr || *v == '\0') return fallback;
  char* end = nullptr;
  const long long x = std::strtoll(v, &end, 10);
  return (end != v && x > 0) ? static_cast<int64_t>(x) : fallback;
}

inline const Tuning& tuning() {
  static const Tuning t = [] {
    Tuning d;
    d.fwd_vpl_cap = static_cast<int>(env_positive("PT_RMSNORM_FWD_VPL_CAP", d.fwd_vpl_cap));
    d.bwd_vpl_cap = static_cast<int>(env_positive("PT_RMSNORM_BWD_VPL_CAP", d.bwd_vpl_cap));
    d.fwd_blocks_per_cu = env_positive("PT_RMSNORM_FWD_BLOCKS_PER_CU", d.fwd_blocks_per_cu);
    d.bwd_partials = env_positive("PT_RMSNORM_BWD_PARTIALS", d.bwd_partials);
    d.fwd_occupancy = static_cast<int>(env_int("PT_RMSNORM_FWD_OCCUPANCY", d.fwd_occupancy));
    d.bwd_occupancy = static_cast<int>(env_int("PT_RMSNORM_BWD_OCCUPANCY", d.bwd_occupancy));
    return d;
  }();
  return t;
}

inline int pow2_at_least(int64_t n) {
  int v = 1;
  while (v < n) v *= 2;
  return v;
}

// Smallest waves-per-row in {1, 2, 4, 8, 16} whose vectors-per-lane fit under `cap`
// (VPL a power of two); past that, 16 waves per row with up to 16 vectors per lane.
inline bool choose_shape(int64_t cols, int vec, int cap, Shape* s) {
  const int64_t nvec = (cols + vec - 1) / vec;
  for (int wpr = 1; wpr <= 16; wpr *= 2) {
    const int64_t per_lane = (nvec + 64 * wpr - 1) / (64 * wpr);
    if (per_lane <= cap) {
      *s = {pow2_at_least(per_lane), wpr};
      return true;
    }
  }
  const int64_t per_lane = (nvec + 1023) / 1024;
  if (per_lane > 16) return false;
  *s = {pow2_at_least(per_lane), 16};
  return true;
}

// The general kernels take rows that are not whole aligned vectors, weights of another 16-bit
// type, and short rows of any alignment: up to kQuarterVecs vectors a row has 16 lanes (four rows
// to a wave, so one reduction and one wave for four).  Measured per launch, one wave per row
// against four rows per wave: [131072, 64] bf16 forward 25.5 -> 9.2 us, backward 37.4 -> 17.3;
// [131072, 128] bf16 29.6 -> 12.9 and 40.4 -> 22.5; [131072, 128] fp32 (32 vectors) 36.5 -> 21.7
// and 38.2 -> 37.4; at 40 vectors (fp32 160) the backward loses, 15.7 -> 20.9 with the forward equal.
constexpr int64_t kQuarterVecs = 32;

// Aligned rows that the general kernels take too.
inline bool short_row(int64_t cols, int vec) { return (cols + vec - 1) / vec <= kQuarterVecs; }

// The forward's: a few rows of nearly 32 vectors are as many waves too few that way, and stay with one
// wave each.  us, four rows per wave against one: [2048, 256] bf16 2.6 2.3, with the residual add
// 3.1 2.8, [512, 256] 2.1 2.1 and 2.6 2.3, [2048, 128] fp32 2.5 2.2 and 2.8 2.7; [4096, 256] bf16 2.7 2.8
// and 3.3 3.8, [4096, 128] fp32 2.6 2.5 and 3.0 3.7, [8192, 256] bf16 3.2 3.9.  At 25 vectors four per
// wave win at every count ([512, 200] bf16 2.2 2.4, [2048, 100] fp32 2.6 2.7).
inline bool short_row_fwd(int64_t rows, int64_t cols, int vec, bool fused) {
  const int64_t nvec = (cols + vec - 1) / vec;
  return short_row(cols, vec) && (nvec <= 28 || rows > (fused ? 2048 : 4096));
}

inline Shape general_shape(int64_t cols, int vec, bool backward) {
  const int64_t nvec = (cols + vec - 1) / vec;
  if (nvec <= kQuarterVecs) return {pow2_at_least((nvec + 15) / 16), 0};
  Shape s;
  (void)choose_shape(cols, vec, backward ? bwd_vpl_cap_for(0, cols, vec) : 32 / vec, &s);
  return s;
}

// Calls f.template run<VPL, WPR>() for a runtime shape and returns true, or returns false
// if that shape is not instantiated.  FULL: aligned rows, every shape that a tuning variable can
// ask for; otherwise those that choose_shape gives for the default caps.
template <bool FULL, typename F>
bool dispatch_shape(const Shape& s, const F& f) {
#define PT_RMS_CASE(V, W)            \
  if (s.vpl == V && s.wpr == W) {    \
    f.template run<V, W>();          \
    return true;                     \
  }
  if constexpr (FULL) {
    PT_RMS_CASE(1, 1) PT_RMS_CASE(2, 1) PT_RMS_CASE(4, 1) PT_RMS_CASE(8, 1)
    PT_RMS_CASE(1, 2) PT_RMS_CASE(2, 2) PT_RMS_CASE(4, 2) PT_RMS_CASE(8, 2)
    PT_RMS_CASE(1, 4) PT_RMS_CASE(2, 4) PT_RMS_CASE(4, 4) PT_RMS_CASE(8, 4)
    PT_RMS_CASE(1, 8) PT_RMS_CASE(2, 8) PT_RMS_CASE(4, 8) PT_RMS_CASE(8, 8)
    PT_RMS_CASE(1, 16) PT_RMS_CASE(2, 16) PT_RMS_CASE(4, 16) PT_RMS_CASE(8, 16)
    PT_RMS_CASE(16, 16)
  } else {
    PT_RMS_CASE(1, 0) PT_RMS_CASE(2, 0) PT_RMS_CASE(1, 1)
    if constexpr (F::kBackward) {
      PT_RMS_CASE(1, 2) PT_RMS_CASE(1, 4) PT_RMS_CASE(2, 4)
      PT_RMS_CASE(2, 8) PT_RMS_CASE(2, 16) PT_RMS_CASE(4, 16)
    } else if constexpr (F::kVec == 8) {
      PT_RMS_CASE(2, 1) PT_RMS_CASE(4, 1) PT_RMS_CASE(4, 2) PT_RMS_CASE(4, 4) PT_RMS_CASE(4, 8)
      PT_RMS_CASE(4, 16)
    } else {
      PT_RMS_CASE(2, 1) PT_RMS_CASE(4, 1) PT_RMS_CASE(8, 1) PT_RMS_CASE(8, 2) PT_RMS_CASE(8, 4)
      PT_RMS_CASE(8, 8)
    }
    PT_RMS_CASE(8, 16) PT_RMS_CASE(16, 16)
  }
#undef PT_RMS_CASE
  return false;
}

inline int bwd_waves(const Shape& s) { return s.wpr > kBwdWaves ? s.wpr : kBwdWaves; }

// Most weight-gradient partial rows (workgroups) of the backward.
constexpr int64_t kMostPartials = 512;

// One workgroup per CU keeps HBM busy when its rows are long enough, two streams of the current
// and the next row group in flight, and half as many partial rows are then written and summed.
// us of the whole call with 512 against 256 workgroups (plain, residual form): bf16 4096 columns 2048 rows
// 16.6 15.7 and 19.3 18.0, 16384 rows 71.8 69.0 and 95.8 92.4; 8192 columns 512 rows 15.8 11.5 and
// 17.1 12.4, 16384 rows 139.4 132.8 and 180.7 175.0; fp32 1024 columns 2048 rows 10.0 9.4 and 11.1 10.5,
// 16384 rows 37.0 36.0 and 49.2 47.3; 4096 columns 16384 rows 132.9 128.6 and 183.6 178.5.  Shorter rows
// lose ([16384, 2048] bf16 38.2 41.2), and so do many rows that fill two vectors of each of 16 waves'
// lanes: 16384 rows of 16384 bf16 271.2 277.6 and 373.2 387.4, of 8192 fp32 271.7 277.4 and 376.3 377.4
// (8192 rows 143.8 138.0 and 193.6 192.6, and 136.6 135.6 and 187.1 190.6); fp32 rows beyond that
// also (16384 columns 547.8 567.5 and 933.1 927.5), bf16 ones not (32768: 1439 1416).
// 384 leave half of the CUs with two workgroups and are slower than both.
// The residual form takes the plain one's count, so that their weight gradients are the same bits.
inline int64_t bwd_partials_for(int64_t rows, int64_t cols, int esize) {
  if (tuning().bwd_partials > 0) return tuning().bwd_partials;
  const int64_t bytes = cols * esize;
  if (bytes < (esize == 4 ? 4096 : 8192)) return kMostPartials;
  const bool full = bytes > 24576 && (bytes <= 32768 || esize == 4);
  return full && rows >= 16384 ? kMostPartials : kMostPartials / 2;
}

// The most that bwd_partials_for gives, for sizing workspaces.
inline int64_t most_partials() {
  return tuning().bwd_partials > 0 ? tuning().bwd_partials : kMostPartials;
}

// Backward grid = number of weight-gradient partial rows, at most `partials`.
inline int64_t bwd_blocks(int64_t rows, const Shape& s, int64_t partials) {
  const int64_t slots = row_slots(s.wpr, bwd_waves(s));
  int64_t b = (rows + slots - 1) / slots;
  if (b > partials) b = partials;
  return b < 1 ? 1 : b;
}

// Partial rows that a workspace has to hold, whatever the grid: the figure of the workspace
// query, of the workspace check and of pt_rmsnorm_bwd_noalloc's size limit.  Whole aligned vectors
// (`vectors`): the most workgroups of their shape; other rows: one per two rows up to 2048
// vectors a row, one per row above.  The grid never exceeds it.
inline int64_t bwd_partial_bound(int64_t rows, int64_t cols, int vec, bool vectors, const Shape& s) {
  if (vectors) return bwd_blocks(rows, s, most_partials());
  const int64_t b = (cols + vec - 1) / vec <= 2048 ? (rows + 1) / 2 : rows;
  return b < 1 ? 1 : (b < most_partials() ? b : most_partials());
}

inline int fwd_waves(const Shape& s) { return s.wpr > kFwdWaves ? s.wpr : kFwdWaves; }

// Forward grid: one row per row slot (non-persistent, measured fastest), optionally capped
// at PT_RMSNORM_FWD_BLOCKS_PER_CU blocks per CU (aligned rows; the general kernels do not loop).
inline int64_t fwd_blocks(int64_t rows, const Shape& s, int ncu, bool aligned) {
  const int64_t slots = row_slots(s.wpr, fwd_waves(s));
  int64_t b = (rows + slots - 1) / slots;
  const int64_t per_cu = aligned ? tuning().fwd_blocks_per_cu : 0;
  if (per_cu > 0 && b > static_cast<int64_t>(ncu) * per_cu) b = static_cast<int64_t>(ncu) * per_cu;
  return b < 1 ? 1 : b;
}

// Row-group steps of a grid of `blocks` blocks with `slots` row slots each.
inline int row_iters(int64_t rows, int64_t blocks, int slots) {
  const int64_t stride = blocks * slots;
  return static_cast<int>((rows + stride - 1) / stride);
}

struct FwdArgs {
  const void* x;
  int64_t xs;
  const void* w;
  int wdt;
  void* y;
  int64_t ys;
  float* rstd;
  int64_t rows;
  int cols;
  float eps;
  int xdt;
  bool aligned;
  Shape shape;
  int64_t blocks;
  hipStream_t st;
  // fused residual add (res == nullptr: plain norm)
  const void* res = nullptr;
  int64_t res_s = 0;
  void* h = nullptr;
  int64_t h_s = 0;
};

struct BwdArgs {
  const void* dy;
  int64_t dys;
  const void* x;
  int64_t xs;
  const void* w;
  int wdt;
  const float* rstd;
  void* dx;
  int64_t dxs;
  float* partial;
  int64_t blocks;
  int64_t rows;
  int cols;
  int xdt;
  bool aligned;
  Shape shape;
  hipStream_t st;
  // incoming gradient of h for the fused residual add (nullptr: plain norm backward)
  const void* dh_in = nullptr;
  int64_t dh_in_s = 0;
};

template <typename T, typename WT, bool ALIGNED>
struct FwdLaunch {
  static constexpr bool kBackward = false;
  static constexpr int kVec = Elem<T>::VEC;
  const FwdArgs& a;
  template <int VPL, int WPR, bool PERSIST, bool ADD>
  void go(int iters) const {
    constexpr int WAVES = WPR > kFwdWaves ? WPR : kFwdWaves;
    const ResidualIn<T> rin{static_cast<const T*>(a.res), a.res_s, static_cast<T*>(a.h), a.h_s};
    const auto kernel =
        rmsnorm_fwd_kernel<T, WT, VPL, WPR, WAVES, ALIGNED, kLoadNT, PERSIST, ADD>;
    size_t lds = occupancy_lds(tuning().fwd_occupancy, 0);
    if (allow_dynamic_lds(reinterpret_cast<const void*>(kernel), lds) != PT_OK) lds = 0;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(a.blocks)), dim3(WAVES * 64), lds, a.st,
                       static_cast<const T*>(a.x), a.xs, a.w, a.wdt, static_cast<T*>(a.y), a.ys,
                       a.rstd, a.rows, a.cols, a.eps, iters, rin);
  }
  template <int VPL, int WPR>
  void run() const {
    constexpr int WAVES = WPR > kFwdWaves ? WPR : kFwdWaves;
    const int iters = row_iters(a.rows, a.blocks, row_slots(WPR, WAVES));
    if constexpr (ALIGNED) {
      if (iters > 1) {
        if (a.res != nullptr) {
          go<VPL, WPR, true, true>(iters);
        } else {
          go<VPL, WPR, true, false>(iters);
        }
        return;
      }
    }
    if (a.res != nullptr) {
      go<VPL, WPR, false, true>(iters);
    } else {
      go<VPL, WPR, false, false>(iters);
    }
  }
};

template <typename T, typename WT, bool ALIGNED>
struct BwdLaunch {
  static constexpr bool kBackward = true;
  static constexpr int kVec = Elem<T>::VEC;
  const BwdArgs& a;
  template <bool ADD, int VPL, int WPR, int WAVES>
  void go(size_t need, size_t lds, int iters) const {
    const auto kernel = rmsnorm_bwd_kernel<T, WT, VPL, WPR, WAVES, ALIGNED, kLoadNT, ADD>;
    if (allow_dynamic_lds(reinterpret_cast<const void*>(kernel), lds) != PT_OK) lds = need;
    const ResidualGrad<T> rg{static_cast<const T*>(a.dh_in), a.dh_in_s};
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(a.blocks)), dim3(WAVES * 64), lds, a.st,
                       static_cast<const T*>(a.dy), a.dys, static_cast<const T*>(a.x), a.xs, a.w,
                       a.wdt, a.rstd, static_cast<T*>(a.dx), a.dxs, a.partial, a.rows, a.cols,
                       iters, rg);
  }
  template <int VPL, int WPR>
  void run() const {
    constexpr int WAVES = WPR > kBwdWaves ? WPR : kBwdWaves;
    constexpr int RPB = row_slots(WPR, WAVES);
    const size_t need =
        (RPB > 1 && a.partial != nullptr) ? static_cast<size_t>(a.cols) * sizeof(float) : 0;
    const size_t share = occupancy_lds(tuning().bwd_occupancy, 0);
    const size_t lds = share > need ? share : need;
    const int iters = row_iters(a.rows, a.blocks, RPB);
    if (a.dh_in != nullptr) {
      go<true, VPL, WPR, WAVES>(need, lds, iters);
    } else {
      go<false, VPL, WPR, WAVES>(need, lds, iters);
    }
  }
};

// True when the aligned kernels have an instance for the weight type (x's type or fp32).
inline bool vector_weight(int xdt, int wdt) { return wdt == xdt || wdt == PT_FLOAT32; }

// Per-storage-type launchers; false if no kernel matched the shape (a bug, reported by
// the caller as an error rather than silently skipping the launch).
template <typename T>
bool launch_fwd(const FwdArgs& a) {
  if (a.aligned && a.wdt == a.xdt) return dispatch_shape<true>(a.shape, FwdLaunch<T, T, true>{a});
  if (a.aligned && a.wdt == PT_FLOAT32)
    return dispatch_shape<true>(a.shape, FwdLaunch<T, float, true>{a});
  if (a.wdt == a.xdt) return dispatch_shape<false>(a.shape, FwdLaunch<T, T, false>{a});
  if (a.wdt == PT_FLOAT32) return dispatch_shape<false>(a.shape, FwdLaunch<T, float, false>{a});
  return dispatch_shape<false>(a.shape, FwdLaunch<T, void, false>{a});
}

template <typename T>
bool launch_bwd(const BwdArgs& a) {
  if (a.aligned && a.wdt == a.xdt) return dispatch_shape<true>(a.shape, BwdLaunch<T, T, true>{a});
  if (a.aligned && a.wdt == PT_FLOAT32)
    return dispatch_shape<true>(a.shape, BwdLaunch<T, float, true>{a});
  if (a.wdt == a.xdt) return dispatch_shape<false>(a.shape, BwdLaunch<T, T, false>{a});
  if (a.wdt == PT_FLOAT32) return dispatch_shape<false>(a.shape, BwdLaunch<T, float, false>{a});
  return dispatch_shape<false>(a.shape, BwdLaunch<T, void, false>{a});
}

extern template bool launch_fwd<float>(const FwdArgs&);
extern template bool launch_fwd<_Float16>(const FwdArgs&);
extern template bool launch_fwd<__bf16>(const FwdArgs&);
extern template bool launch_bwd<float>(const BwdArgs&);
extern template bool launch_bwd<_Float16>(const BwdArgs&);
extern template bool launch_bwd<__bf16>(const BwdArgs&);

}  // namespace rmsnorm
}  // namespace pt

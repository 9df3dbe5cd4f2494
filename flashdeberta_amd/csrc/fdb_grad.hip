// The products of a layer's training backward, 16-bit types: the gradients of what the projections read (fdb_dgrad) and of their weights
// and biases (fdb_wgrad).  Tokens and position tables go through the same weights, so both of their products are one launch
// each:
//   d hidden = d qkv . W and d rel = d pos . W[q, k], tiles of one grid;
//   d W = d qkv^T . hidden + [d pos^T . rel] on the rows of q and k, one contraction over tokens and table rows, and d b, the column sums of
//   d qkv and d pos, from the tiles as they pass (a product with ones).
// 8 x 512 tokens, 12 heads, bf16, against a library product each (the second weight product onto the first one's rounded result) and two
// launches for the column sums: 35.9 -> 21.1 us and 52.9 -> 29; 1000 tokens 23.9 -> 14.5 and 33.5 -> 23.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>

#include "fdb_device.h"
#include "fdb_kernels.h"
#include "../../include/fdb.h"

using namespace fdb;

namespace {

// LDS rows are 128 bytes, slot (row, s) = chunk s ^ swz16(row), as in fdb_gemm.hip.  An operand whose contraction runs down its rows is staged in
// panels of 64 rows (one stage of the contraction) by 64 columns and read transposed.
constexpr int kDepth = 64, kRow = 128, kPanel = kDepth * kRow;

// This lane's part of the address of a transposed operand: 16 columns from 16 * f on, contraction 8 * kg + 4 * h + 0..3 of the 32 at
// hand; f, h and the 32 are left to the instruction's offset where they do not touch the swizzle.
__device__ __forceinline__ uint32_t tr_lane(int lane, int f, int h) {
  const int s16 = lane & 15, row = 8 * (lane >> 4) + 4 * h + (s16 >> 2);
  return (uint32_t)(row * kRow + (((2 * (f & 3) + ((s16 >> 1) & 1)) ^ swz16(row)) * 16) + (s16 & 1) * 8);
}
template <class QT>
__device__ __forceinline__ typename QT::frag tr_frag(uint32_t lo, uint32_t hi, int offset) {   // the offset travels in the instructions
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)((LDS_AS char*)(uintptr_t)lo + offset));
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)((LDS_AS char*)(uintptr_t)hi + offset));
  return __builtin_bit_cast(typename QT::frag, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}
__device__ __forceinline__ void meet() {   // a barrier that leaves loads under way
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// ---- out = x . w: rows of x contiguous along the contraction, w [depth, cols] with the contraction down its rows ---------------------
struct DgradParams {
  const char *x[2], *w;
  char* out[2];
  int32_t rows[2], depth[2], tiles[2], cols, tiles_n;
};
template <int ROWS, int WM_, int WN_, int STAGES_, int PER_CU_>
struct DShape {
  static constexpr int TM = ROWS, TN = 128, WM = WM_, WN = WN_, NW = WM * WN, STAGES = STAGES_, PER_CU = PER_CU_, FM = TM / WM / 16, FN = TN / WN / 16, PITCH = TN * 2 + 16;
  static constexpr int STAGE = TM * kRow + TN / 64 * kPanel, LOADS = STAGE / 1024 / NW, XLOADS = TM / 8 / NW;
  static constexpr int LDS = STAGES * STAGE;
  static_assert(TM * PITCH <= LDS && PER_CU * LDS <= 160 * 1024, "LDS budget");
};

template <class QT, class S>
__global__ __launch_bounds__(64 * S::NW, S::PER_CU * S::NW / 4) void fdb_dgrad_kernel(const DgradParams p) {
  using frag = typename QT::frag;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 15, kg = lane >> 4;
  const int wm = wave / S::WN, wn = wave % S::WN;
  // every XCD takes a run of tiles
  const int all = p.tiles[0] + p.tiles[1], n = blockIdx.x, xcd = n & 7, each = all >> 3, more = all & 7;
  int tile = xcd * each + min(xcd, more) + (n >> 3);
  const int which = tile >= p.tiles[0] ? 1 : 0;
  tile -= which ? p.tiles[0] : 0;
  const int tm = tile / p.tiles_n, m0 = tm * S::TM, n0 = (tile - tm * p.tiles_n) * S::TN;
  const int rows = p.rows[which], depth = p.depth[which], cols = p.cols;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LDS_AS char*)smem;
  const char* x_at = p.x[which] + (int64_t)m0 * depth * 2;   // of the stage that is fetched next
  const char* w_at = p.w;
  const int64_t w_step = (int64_t)kDepth * cols * 2;
  uint32_t off[S::LOADS];   // rows of x past the end re-read the last one, panels past the last column the last panel
#pragma unroll
  for (int j = 0; j < S::LOADS; ++j) {
    const int c = wave + S::NW * j;
    if (j < S::XLOADS) {
      const int row = 8 * c + (lane >> 3);
      off[j] = (uint32_t)(min(m0 + row, rows - 1) - m0) * (uint32_t)(depth * 2) + (uint32_t)(((lane & 7) ^ swz16(row)) * 16);
    } else {
      const int w = c - S::TM / 8, row = 8 * (w & 7) + (lane >> 3);
      off[j] = (uint32_t)row * (uint32_t)(cols * 2) + (uint32_t)(min(n0 + 64 * (w >> 3), cols - 64) * 2) + (uint32_t)(((lane & 7) ^ swz16(row)) * 16);
    }
  }
  auto fill = [&](int buf) __attribute__((always_inline)) {
    const uint32_t dst = lds0 + (uint32_t)buf * S::STAGE + (uint32_t)wave * 1024u;
#pragma unroll
    for (int j = 0; j < S::LOADS; ++j) dma16sn(j < S::XLOADS ? x_at : w_at, off[j], dst + j * S::NW * 1024u);
    x_at += kRow;
    w_at += w_step;
  };
  f32x4 acc[S::FM][S::FN];
#pragma unroll
  for (int i = 0; i < S::FM; ++i)
#pragma unroll
    for (int j = 0; j < S::FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = depth / kDepth;
#pragma unroll
  for (int t = 0; t < S::STAGES - 1; ++t)
    if (t < steps) fill(t);
  const uint32_t xrow = lds0 + (uint32_t)((wm * 16 * S::FM + r) * kRow), f = (uint32_t)swz16(r);
  uint32_t wlane[S::FN][2];
#pragma unroll
  for (int j = 0; j < S::FN; ++j)
#pragma unroll
    for (int h = 0; h < 2; ++h) wlane[j][h] = lds0 + S::TM * kRow + (uint32_t)((wn * S::FN + j) >> 2) * kPanel + tr_lane(lane, wn * S::FN + j, h);
  int buf = 0;
#pragma unroll 1
  for (int t = 0; t < steps; ++t) {
    if (t + S::STAGES - 1 <= steps) wait_vmcnt<(S::STAGES - 2) * S::LOADS>();
    else wait_vmcnt<0>();
    meet();
    if (t + S::STAGES - 1 < steps) fill(buf == 0 ? S::STAGES - 1 : buf - 1);
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t at = (uint32_t)buf * S::STAGE;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      frag xf[S::FM], wf[S::FN];
#pragma unroll
      for (int i = 0; i < S::FM; ++i) xf[i] = *(LDS_AS const frag*)((LDS_AS const char*)(uintptr_t)(at + xrow + ((uint32_t)(4 * s + kg) ^ f) * 16) + i * 16 * kRow);
#pragma unroll
      for (int j = 0; j < S::FN; ++j) wf[j] = tr_frag<QT>(at + wlane[j][0], at + wlane[j][1], s * 32 * kRow);
#pragma unroll
      for (int i = 0; i < S::FM; ++i)
#pragma unroll
        for (int j = 0; j < S::FN; ++j) acc[i][j] = mma16(wf[j], xf[i], acc[i][j]);
    }
    buf = buf == S::STAGES - 1 ? 0 : buf + 1;
  }
  __syncthreads();   // the staged tiles have been read: their memory takes the result
#pragma unroll
  for (int i = 0; i < S::FM; ++i)
#pragma unroll
    for (int j = 0; j < S::FN; ++j)
      QT::store4(smem + ((wm * S::FM + i) * 16 + r) * S::PITCH + ((wn * S::FN + j) * 16 + 4 * kg) * 2, acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
  __syncthreads();
  constexpr int CH = S::TN / 8;
  for (int c = tid; c < S::TM * CH; c += 64 * S::NW) {
    const int row = c / CH, col = (c - row * CH) * 8;
    if (m0 + row < rows && n0 + col < cols) *(frag*)(p.out[which] + ((int64_t)(m0 + row) * cols + n0 + col) * 2) = *(const frag*)(smem + row * S::PITCH + col * 2);
  }
}

// ---- part = x^T . y over a share of the rows ------------------------------------------------------------------------------------------
struct WgradParams {
  const char *x[2], *y[2];
  float *parts, *bias_parts;   // [shares][x_cols][y_cols], [shares][x_cols]
  int32_t rows[2], x_cols[2], y_cols, tiles_n, tiles, shares;
};
// 128 x 128 outputs by four waves, two stages, two workgroups per CU, of which one multiplies while the other waits at its barrier.  8 x 512
// tokens, 12 heads, with the fold, best number of shares: 31.2 us (29.0 since rows past the last one are zeroed in the LDS); 128 x 192 by eight waves, three stages, alone on its CU 36.0, 128 x 64
// 36.6, 64 x 192 33.5, 128 x 256 34.4, 128 x 128 by eight waves 38.4 and 44.0.
struct WShape {
  static constexpr int TM = 128, TN = 128, WN = 2, STAGES = 2, PER_CU = 2, NW = 4, FM = 4, FN = 4;
  static constexpr int STAGE = (TM + TN) / 64 * kPanel, LOADS = STAGE / 1024 / NW, XLOADS = TM / 64 * 8 / NW, PITCH = TN * 4 + 16;
  static constexpr int LDS = STAGES * STAGE > TM * PITCH ? STAGES * STAGE : TM * PITCH;
  static_assert(PER_CU * LDS <= 160 * 1024, "two workgroups per CU");
};

template <class QT>
__global__ __launch_bounds__(64 * WShape::NW, 2) void fdb_wgrad_kernel(const WgradParams p) {
  using S = WShape;
  using frag = typename QT::frag;
  using elem = typename QT::scratch_t;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 15, kg = lane >> 4;
  const int wm = wave / S::WN, wn = wave % S::WN;
  // every XCD takes a run of tiles of one share, or of two neighbouring ones: their rows pass through one L2
  const int all = p.tiles * p.shares, n = blockIdx.x, xcd = n & 7, each = all >> 3, more = all & 7;
  const int place = xcd * each + min(xcd, more) + (n >> 3);
  const int share = place / p.tiles, tile = place - share * p.tiles;
  const int tm = tile / p.tiles_n, m0 = tm * S::TM, n0 = (tile - tm * p.tiles_n) * S::TN;
  // stages of the first pair of matrices, then of the second where this tile's columns are in it (the second has 128 * heads columns)
  const int first = (p.rows[0] + kDepth - 1) / kDepth, second = m0 < p.x_cols[1] ? (p.rows[1] + kDepth - 1) / kDepth : 0;
  const int t0 = (int)((uint32_t)((first + second) * share) / (uint32_t)p.shares), t1 = (int)((uint32_t)((first + second) * (share + 1)) / (uint32_t)p.shares);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LDS_AS char*)smem;
  uint32_t off[2][S::LOADS];   // from the stage's first row, with the swizzle; panels past the last column re-read the last panel
#pragma unroll
  for (int j = 0; j < S::LOADS; ++j) {
    const int c = wave + S::NW * j, row = 8 * (c & 7) + (lane >> 3);
    const uint32_t chunk = (uint32_t)(((lane & 7) ^ swz16(row)) * 16);
#pragma unroll
    for (int w = 0; w < 2; ++w)
      off[w][j] = (uint32_t)row * (uint32_t)((j < S::XLOADS ? p.x_cols[w] : p.y_cols) * 2) + chunk +
                  (uint32_t)(j < S::XLOADS ? min(m0 + 64 * (c >> 3), p.x_cols[w] - 64) : min(n0 + 64 * ((c >> 3) - S::TM / 64), p.y_cols - 64)) * 2u;
  }
  // What the stage that is fetched next starts from; in registers, both matrices' (an argument picked by a condition becomes a load that
  // every stage waits for).
  const int rows0 = p.rows[0], rows1 = p.rows[1];
  const int64_t x_pitch0 = (int64_t)p.x_cols[0] * 2, x_pitch1 = (int64_t)p.x_cols[1] * 2, y_pitch = (int64_t)p.y_cols * 2;
  const char *x1 = p.x[1], *y1 = p.y[1];
  const bool late = t0 >= first;
  const int64_t k0 = (int64_t)(late ? t0 - first : t0) * kDepth;
  const char *x_at = p.x[0] + k0 * x_pitch0, *y_at = p.y[0] + k0 * y_pitch;
  int64_t x_pitch = x_pitch0;
  int left = rows0 - (int)k0, fetched = t0;
  uint32_t at[S::LOADS];
#pragma unroll
  for (int j = 0; j < S::LOADS; ++j) at[j] = off[0][j];
  auto go_on = [&](int64_t k) __attribute__((always_inline)) {
    x_at = x1 + k * x_pitch1, y_at = y1 + k * y_pitch, x_pitch = x_pitch1, left = rows1 - (int)k;
#pragma unroll
    for (int j = 0; j < S::XLOADS; ++j) at[j] = off[1][j];
  };
  if (late) go_on(k0);
  auto fill = [&](int buf) __attribute__((always_inline)) {
    const uint32_t dst = lds0 + (uint32_t)buf * S::STAGE + (uint32_t)wave * 1024u;
    if (left >= kDepth) {
#pragma unroll
      for (int j = 0; j < S::LOADS; ++j) dma16sn(j < S::XLOADS ? x_at : y_at, at[j], dst + j * S::NW * 1024u);
    } else {   // rows past the last one re-read it
#pragma unroll
      for (int j = 0; j < S::LOADS; ++j) {
        const int past = max(8 * ((wave + S::NW * j) & 7) + (lane >> 3) - (left - 1), 0);
        dma16sn(j < S::XLOADS ? x_at : y_at, at[j] - (uint32_t)past * (uint32_t)(j < S::XLOADS ? x_pitch : y_pitch), dst + j * S::NW * 1024u);
      }
    }
    x_at += kDepth * x_pitch, y_at += kDepth * y_pitch, left -= kDepth;
    if (++fetched == first) go_on(0);
  };
  f32x4 acc[S::FM][S::FN], sums[S::FM];
#pragma unroll
  for (int i = 0; i < S::FM; ++i) {
    sums[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < S::FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const bool for_bias = n0 == 0 && wn == 0;   // the column sums: the product with ones, by one wave of each row block
  const elem one = (elem)1.f;
  const frag ones = {one, one, one, one, one, one, one, one};
  uint32_t xlane[S::FM][2], ylane[S::FN][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int i = 0; i < S::FM; ++i) xlane[i][h] = lds0 + (uint32_t)((wm * S::FM + i) >> 2) * kPanel + tr_lane(lane, wm * S::FM + i, h);
#pragma unroll
    for (int j = 0; j < S::FN; ++j) ylane[j][h] = lds0 + (uint32_t)(S::TM / 64 + ((wn * S::FN + j) >> 2)) * kPanel + tr_lane(lane, wn * S::FN + j, h);
  }
  auto multiply = [&](uint32_t at) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      frag xf[S::FM], yf[S::FN];
#pragma unroll
      for (int i = 0; i < S::FM; ++i) xf[i] = tr_frag<QT>(at + xlane[i][0], at + xlane[i][1], s * 32 * kRow);
#pragma unroll
      for (int j = 0; j < S::FN; ++j) yf[j] = tr_frag<QT>(at + ylane[j][0], at + ylane[j][1], s * 32 * kRow);
#pragma unroll
      for (int i = 0; i < S::FM; ++i)
#pragma unroll
        for (int j = 0; j < S::FN; ++j) acc[i][j] = mma16(yf[j], xf[i], acc[i][j]);
      if (for_bias) {
#pragma unroll
        for (int i = 0; i < S::FM; ++i) sums[i] = mma16(ones, xf[i], sums[i]);
      }
    }
  };
#pragma unroll
  for (int t = 0; t < S::STAGES - 1; ++t)
    if (t0 + t < t1) fill(t);
  int buf = 0;
#pragma unroll 1
  for (int t = t0; t < t1; ++t) {
    if (t + S::STAGES - 1 <= t1) wait_vmcnt<(S::STAGES - 2) * S::LOADS>();
    else wait_vmcnt<0>();
    meet();
    if (t + S::STAGES - 1 < t1) fill(buf == 0 ? S::STAGES - 1 : buf - 1);
    __builtin_amdgcn_sched_barrier(0);
    const int real = t < first ? rows0 - t * kDepth : rows1 - (t - first) * kDepth;
    if (real < kDepth) {   // rows past the last one: zeros on both sides, whatever the row they re-read holds
      for (int c = tid; c < (S::TM + S::TN) / 64 * kDepth * 8; c += 64 * S::NW)
        if (((c >> 3) & (kDepth - 1)) >= real) *(u32x4*)(smem + buf * S::STAGE + c * 16) = u32x4{0u, 0u, 0u, 0u};
      __syncthreads();
    }
    multiply((uint32_t)buf * S::STAGE);
    buf = buf == S::STAGES - 1 ? 0 : buf + 1;
  }
  // the result by way of the LDS, in whole rows of the tile
  const int64_t x_cols = p.x_cols[0];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < S::FM; ++i) {
    const int m = (wm * S::FM + i) * 16 + r;
#pragma unroll
    for (int j = 0; j < S::FN; ++j) *(f32x4*)(smem + m * S::PITCH + ((wn * S::FN + j) * 16 + 4 * kg) * 4) = acc[i][j];
    if (for_bias && kg == 0 && m0 + m < x_cols) p.bias_parts[share * x_cols + m0 + m] = sums[i][0];
  }
  __syncthreads();
  constexpr int CH = S::TN / 4;
  for (int c = tid; c < S::TM * CH; c += 64 * S::NW) {
    const int m = c / CH, col = (c - m * CH) * 4;
    if (m0 + m < x_cols && n0 + col < p.y_cols) *(f32x4*)(p.parts + ((int64_t)share * x_cols + m0 + m) * p.y_cols + n0 + col) = *(const f32x4*)(smem + m * S::PITCH + col * 4);
  }
}

// The shares' sums, rounded once: eight entries of d W a thread, then those of d b.
template <class QT>
__global__ __launch_bounds__(256) void fdb_wgrad_fold_kernel(const float* __restrict__ parts, const float* __restrict__ bias_parts, char* __restrict__ dw, char* __restrict__ db,
                                                             int64_t entries, int32_t biases, int32_t shares) {
  int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
  const bool bias = at >= entries;
  const float* from = bias ? bias_parts : parts;
  const int64_t n = bias ? biases : entries;
  at -= bias ? entries : 0;
  if (at >= n) return;
  f32x8 sum = *(const f32x8*)(from + at);
  for (int s = 1; s < shares; ++s) sum += *(const f32x8*)(from + s * n + at);
  *(typename QT::frag*)((bias ? db : dw) + at * 2) = QT::from_f32(sum);
}

int tiles_of(int64_t n, int t) { return (int)((n + t - 1) / t); }

template <class QT, class S>
int launch_dgrad(DgradParams p, hipStream_t stream) {
  auto kern = fdb_dgrad_kernel<QT, S>;
  static std::atomic<uint64_t> lds_set{0};
  const hipError_t e = fdb_set_lds_once((const void*)kern, S::LDS, lds_set);
  if (e != hipSuccess) return (int)e;
  p.tiles_n = tiles_of(p.cols, S::TN);
  for (int i = 0; i < 2; ++i) p.tiles[i] = p.rows[i] > 0 ? tiles_of(p.rows[i], S::TM) * p.tiles_n : 0;
  hipLaunchKernelGGL(kern, dim3(p.tiles[0] + p.tiles[1]), dim3(64 * S::NW), S::LDS, stream, p);
  return (int)hipGetLastError();
}
// Eight waves a tile where it has its CU to itself: a stage is 0.35 us of latency and barrier for such a workgroup, and half of it for two that share one; four
// waves a tile where two share a CU, the matrix cores are busy and a wave's operands serve more products.  Whole launches, replayed, bf16, 512 table rows, us:
//   tiles of 64 (128) rows      64 x 8 waves   64 x 4   128 x 8, four stages   128 x 8, two a CU   128 x 4
//   12 heads,  1024 tokens  144 (72)   19.1*   21.2   24.4    29.0    29.2      16 heads, 1600   264 (136)  29.4   28.1*  30.1   36.4   36.8
//              2500         288 (144)  24.3    23.8*  24.8    28.9    29.2      24 heads, 1024   288 (144)  43.9   36.9*  40.8   51.2   51.8
//              3000         330 (168)  26.6    26.9   24.9*   29.1    29.4      16 heads, 2048   320 (160)  33.3   30.4   30.2*  36.4   36.9
//              4096         432 (216)  27.2    27.0   25.2*   29.7    30.1      24 heads, 2048   480 (240)  52.8   50.4   42.7*  51.6   52.3
//              6144         624 (312)  38.1    40.0   43.3    32.2*   33.8      16 heads, 5000   696 (352)  49.8   51.9   54.6   41.9*  42.6
//              8192         816 (408)  45.0    43.5   43.6    35.8    36.1*     24 heads, 3500   756 (384)  75.4   75.3   77.1   63.3   61.1*
//              20000       1926 (966)  88.2    85.5   83.2    73.2    70.3*     16 heads, 7000   944 (472)  62.4   59.3   55.3   49.7   48.2*
//              16384       1584 (792)  78.6    79.3   81.7    65.0    64.1*     24 heads, 8192  1632 (816)   165    159    151    128    118*
// Waves that lie across the 128 columns (2 x 4) where x is the shorter side, along the rows where it is not (the other way round: 16.8 and 22.0 us).
template <class QT>
int launch_dgrad_rows(const DgradParams& p, hipStream_t stream) {
  const int64_t cus = fdb_cu_count();
  auto tiles = [&](int rows) { return (int64_t)(tiles_of(p.rows[0], rows) + tiles_of(p.rows[1], rows)) * tiles_of(p.cols, 128); };
  if (tiles(64) <= cus) return launch_dgrad<QT, DShape<64, 2, 4, 3, 2>>(p, stream);
  if (tiles(64) * 8 <= cus * 9) return launch_dgrad<QT, DShape<64, 2, 2, 3, 2>>(p, stream);   // few CUs have two
  if (tiles(128) <= cus) return launch_dgrad<QT, DShape<128, 4, 2, 4, 1>>(p, stream);
  if (tiles(128) * 2 < cus * 3) return launch_dgrad<QT, DShape<128, 4, 2, 2, 2>>(p, stream);   // most CUs have one
  return launch_dgrad<QT, DShape<128, 2, 2, 2, 2>>(p, stream);
}

template <class QT>
int launch_wgrad(WgradParams p, void* dw, void* db, hipStream_t stream) {
  using S = WShape;
  auto kern = fdb_wgrad_kernel<QT>;
  static std::atomic<uint64_t> lds_set{0};
  const hipError_t e = fdb_set_lds_once((const void*)kern, S::LDS, lds_set);
  if (e != hipSuccess) return (int)e;
  p.tiles_n = tiles_of(p.y_cols, S::TN);
  p.tiles = tiles_of(p.x_cols[0], S::TM) * p.tiles_n;
  hipLaunchKernelGGL(kern, dim3(p.tiles * p.shares), dim3(64 * S::NW), S::LDS, stream, p);
  const int64_t entries = (int64_t)p.x_cols[0] * p.y_cols;
  hipLaunchKernelGGL(fdb_wgrad_fold_kernel<QT>, dim3((unsigned)((entries + p.x_cols[0] + 2047) / 2048)), dim3(256), 0, stream, p.parts, p.bias_parts, (char*)dw, (char*)db,
                     entries, p.x_cols[0], p.shares);
  return (int)hipGetLastError();
}

}  // namespace

// Shares of the contraction: as many as have a place of their own on the chip, each with six stages at least (a share's partial result
// costs as much as three).  12 heads, 1 / 2 / 3 / 4 / 5 shares: 4096 tokens 71.9 42.0 35.7 31.2* 41.4 us, 1000 tokens 30.6 23.0 22.9 23.3* 27.7, 300 tokens
// 21.3 19.0* 20.3 22.5 24.3; 16 heads, 4096 tokens 73.9 47.0* 59.6 54.7 52.7.  A library product each and the column sums: 52.9, 33.5, -, 60.7.
int fdb_wgrad_shares(int64_t rows, int64_t x_cols, int64_t y_cols) {
  const int64_t tiles = (int64_t)tiles_of(x_cols, WShape::TM) * tiles_of(y_cols, WShape::TN), stages = tiles_of(rows, kDepth);
  return (int)std::max<int64_t>(1, std::min<int64_t>({2 * fdb_cu_count() / tiles, stages / 6, 16}));
}

// Where one launch beats a library product each: unless a second round of workgroups, or the last of more, is mostly empty.  Tiles, this and the library
// (torch.mm of each), us: 16 heads 512 50.3 and 61 | 544 75.2 and 64.3 | 664 75.8 and 71.5 | 912 87.0 and 87.5 | 1056 115 and 94.3 | 1288 123 and 127;
// 12 heads 498 39.5 and 50.1 | 600 58.9 and 55.2 | 792 64.1 and 66.5 | 966 70.3 and 72.5; 24 heads 528 108 and 87 | 816 118 and 116 | 996 132 and 129 |
// 1200 171 and 175 | 1368 183 and 191.  (600 tiles at 16 heads, 75.6 and 84, and 1584 at 24, 230 and 214, fall on the wrong side.)
extern "C" int32_t fdb_dgrad_serves(int64_t rows0, int64_t rows1, int64_t cols) {
  const int64_t tiles = (tiles_of(rows0, 128) + tiles_of(rows1, 128)) * (int64_t)tiles_of(cols, 128), places = 2 * fdb_cu_count(), rounds = (tiles + places - 1) / places;
  return 4 * tiles >= 3 * places * rounds || rounds == 1;
}

int fdb_launch_dgrad(const void* x0, int32_t rows0, int32_t depth0, const void* x1, int32_t rows1, int32_t depth1, const void* w, int32_t cols, void* out0,
                     void* out1, int dtype, void* stream) {
  const DgradParams p{{(const char*)x0, (const char*)x1}, (const char*)w, {(char*)out0, (char*)out1}, {rows0, rows1}, {depth0, depth1}, {0, 0}, cols, 0};
  return dtype == FDB_BF16 ? launch_dgrad_rows<Bf16Tr>(p, (hipStream_t)stream) : launch_dgrad_rows<F16Tr>(p, (hipStream_t)stream);
}

int fdb_launch_wgrad(const void* x0, const void* y0, int32_t rows0, int32_t x_cols0, const void* x1, const void* y1, int32_t rows1, int32_t x_cols1, int32_t y_cols,
                     void* dw, void* db, float* ws, int32_t shares, int dtype, void* stream) {
  const WgradParams p{{(const char*)x0, (const char*)x1}, {(const char*)y0, (const char*)y1}, ws, ws + (int64_t)shares * x_cols0 * y_cols, {rows0, rows1}, {x_cols0, x_cols1},
                      y_cols, 0, 0, shares};
  return dtype == FDB_BF16 ? launch_wgrad<Bf16Tr>(p, dw, db, (hipStream_t)stream) : launch_wgrad<F16Tr>(p, dw, db, (hipStream_t)stream);
}

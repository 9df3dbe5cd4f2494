// A whole attention layer of short texts in one launch: the three projections and the attention of one head of one sequence by one workgroup, for
// sequences of up to 32 tokens, head_dim 64, 16-bit types, both position terms.
//
// At these sizes a layer is latency.  As two launches, 1 x 24 at 12 heads is 4.5 us for the projections, a gap, and 6.5 us for a near launch whose one step
// of work takes 1.9.  Here a workgroup streams its head's 192 rows of the joined weights (295 KB at a depth of 768) and its sequence's rows through
// four LDS stages, as fdb_gemm.hip's tiles do, leaves q, k and v rounded to the type in LDS, where the attention's operands are read from, and one
// wave does the one 32 x 32 block there is: fdb_near.hip's products and skews, with all scores in hand and so without a running soft-max.  The 64
// rows of either table that the block's relative positions name are on their way while the projections are made.
//
// What bounds it: the weights on their way into one CU's LDS, then one wave's chain of products, exponentials and LDS trips; and the host.  Pass of a layer,
// two launches -> one, us (12 heads, depth 768, bf16, passes back to back): 1 x 24 13.8 -> 9.1, 4 x 24 14.2 -> 9.1, 16 x 32 14.9 -> 9.5, 21 x 32 15.2 -> 9.5.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <utility>

#include "fdb_device.h"
#include "fdb_kernels.h"
#include "../../include/fdb.h"

using namespace fdb;

namespace {

constexpr int kThreads = 256, kDepth = 64, kStages = 4;
constexpr int kRow = 128;                                        // bytes of a row of a stage, of a head's q, k or v and of a table
constexpr int kRows = 32, kCols = 192;                           // rows of the sequence, columns q | k | v of the head
constexpr int kStage = (kRows + kCols) * kRow, kLoads = (kRows + kCols) / 8 / 4;
constexpr int kPitch = 68;                                       // 16-bit elements of a scratch row: 64 columns
constexpr int kOffE = kStages * kStage, kOffScr = kOffE + 2 * 64 * kRow, kLds = kOffScr + 32 * kPitch * 2;
static_assert((kRows + kCols) % 32 == 0 && 3 * kRows * kRow <= kStage && kLds <= 160 * 1024, "whole loads for four waves; q, k and v in the place of a stage");

struct SmallParams {
  const char *x, *w, *bias, *pk, *pq;
  char* out;
  const int32_t *start, *length;
  const int16_t* lut;
  int64_t ldx, ldw, pk_sh, pk_sr, pq_sh, pq_sr;   // elements
  int32_t B, L, H, K, R;
  float scale_log2;
};

__device__ __forceinline__ int ring_f(int row) { return 4 * ((row >> 1) & 1) | ((row >> 2) & 3); }   // see fdb_near.hip

template <int OFFSET>
__device__ __forceinline__ float swizzle(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, x), OFFSET));
}
template <int ROT0, int... V>
__device__ __forceinline__ void rotate16(const float (&xs)[16], float (&px)[16], std::integer_sequence<int, V...>) {
  ((px[V] = swizzle<(0xC000 | (((ROT0 - (8 * (V >> 2) + 3 - (V & 3))) & 31) << 5))>(xs[V])), ...);
}

template <class QT>
__global__ __launch_bounds__(kThreads, 1) void fdb_small_kernel(const SmallParams p) {
  using frag = typename QT::frag;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LDS_AS char*)smem;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  // the sequences of a head one after the other on one XCD, whose L2 then holds that head's weights
  const int n = (int)blockIdx.x, all = (int)gridDim.x, xcd = n & 7, item = xcd * (all >> 3) + min(xcd, all & 7) + (n >> 3);
  const int h = __builtin_amdgcn_readfirstlane(item / p.B), b = item - h * p.B;
  const int tok0 = p.start ? min(max(p.start[b], 0), p.L) : 0;
  const int sl = p.length ? p.length[b] : p.L;   // negative: a mask the caller could not express, NaN throughout
  const int Lb = min(max(sl, 0), p.L - tok0);
  const int64_t o_row = (int64_t)p.H * 64;       // elements
  char* ob = p.out + ((int64_t)b * p.L * o_row + (int64_t)h * 64) * 2;
  if (Lb < p.L) fill_pad_rows<kRow>(ob, o_row * 2, 0, p.L, tok0, Lb, sl < 0 ? QT::NAN_WORD : 0u, tid);
  if (Lb == 0) return;

  // ---- the projections: [32 x 192] outputs of a contraction over depth, stages of 64 ---------------------------------------------------------
  const char* pkb = p.pk + (int64_t)h * p.pk_sh * 2;
  const char* pqb = p.pq + (int64_t)h * p.pq_sh * 2;
  const int srow = lane >> 3, slot = lane & 7;
  int delta[2];   // table row e holds relative position e - 32
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = 8 * (wave + 4 * j) + srow - 32;
    delta[j] = (int)((const uint16_t*)p.lut)[max(-p.R, min(p.R, r)) + p.R];
  }
  const char* xb = p.x + ((int64_t)b * p.L + tok0) * p.ldx * 2;
  const char* wb = p.w + (int64_t)h * 64 * p.ldw * 2;
  uint64_t from[kLoads];
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const int c = wave + 4 * j, row = 8 * c + srow, col = row - kRows;   // rows past the end re-read the last one
    const uint64_t chunk = (uint64_t)((slot ^ swz16(row)) * 16);
    const char* at = c < kRows / 8 ? xb + (uint64_t)(uint32_t)min(row, Lb - 1) * (uint64_t)(p.ldx * 2) : wb + ((uint64_t)(uint32_t)((col >> 6) * p.H * 64 + (col & 63))) * (uint64_t)(p.ldw * 2);
    from[j] = (uint64_t)(uintptr_t)at + chunk;
  }
  auto fill = [&](int t) __attribute__((always_inline)) {
    const uint32_t dst = lds0 + (uint32_t)(t & (kStages - 1)) * kStage + (uint32_t)wave * 1024u;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) dma16n((const void*)(uintptr_t)(from[j] + (uint64_t)(uint32_t)t * kRow), dst + j * 4096u);
  };
  const int steps = p.K / kDepth;
#pragma unroll
  for (int t = 0; t < kStages - 1; ++t)
    if (t < steps) fill(t);
  // (taken here: the compiler does not count the direct loads)
  asm volatile("" : "+v"(delta[0]), "+v"(delta[1]));
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t row = (uint32_t)(8 * (wave + 4 * j) + srow), chunk = (uint32_t)((slot ^ ring_f((int)row)) * 16), dst = lds0 + kOffE + (uint32_t)(wave + 4 * j) * 1024u;
    dma16sn(pkb, __umul24((uint32_t)delta[j], (uint32_t)(p.pk_sr * 2)) + chunk, dst);
    dma16sn(pqb, __umul24((uint32_t)delta[j], (uint32_t)(p.pq_sr * 2)) + chunk, dst + 64 * kRow);
  }
  const int r16 = lane & 15, kg = lane >> 4;
  f32x4 acc[2][3];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t xrow = (uint32_t)(r16 * kRow), wrow = (uint32_t)((kRows + wave * 48 + r16) * kRow), f = (uint32_t)swz16(r16);
#pragma unroll 1
  for (int t = 0; t < steps; ++t) {
    // this wave's loads of stage t have landed, those of the two after it may still fly (and the tables' rows with them)
    if (t + kStages - 1 <= steps) wait_vmcnt<(kStages - 2) * kLoads>();
    else wait_vmcnt<0>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();   // ... and everybody's; everybody has read stage t - 1
    asm volatile("" ::: "memory");
    if (t + kStages - 1 < steps) fill(t + kStages - 1);
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t at = lds0 + (uint32_t)(t & (kStages - 1)) * kStage;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      frag xf[2], wf[3];
      const uint32_t sl16 = ((uint32_t)(4 * s + kg) ^ f) * 16;
#pragma unroll
      for (int j = 0; j < 3; ++j) wf[j] = *(LDS_AS const frag*)(uintptr_t)(at + wrow + sl16 + j * 16 * kRow);
#pragma unroll
      for (int i = 0; i < 2; ++i) xf[i] = *(LDS_AS const frag*)(uintptr_t)(at + xrow + sl16 + i * 16 * kRow);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) acc[i][j] = mma16(wf[j], xf[i], acc[i][j]);
    }
  }
  f32x4 bias[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int col = wave * 48 + j * 16 + 4 * kg;
    bias[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (p.bias) bias[j] = QT::load4(p.bias + ((int64_t)(col >> 6) * p.H * 64 + h * 64 + (col & 63)) * 2);
  }
  wait_vmcnt<0>();
  __syncthreads();   // the stages have been read, the tables' rows are there
  // q, k and v as the attention reads them: rows of 128 bytes, slot (row, s) = chunk s ^ ring_f(row), k's rows with the low two bits inverted
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int col = wave * 48 + j * 16 + 4 * kg, what = col >> 6, c = col & 63, row = (i * 16 + r16) ^ (what == 1 ? 3 : 0);
      const f32x4 y = acc[i][j] + bias[j];
      QT::store4(smem + what * (kRows * kRow) + row * kRow + (((c >> 3) ^ ring_f(row)) * 16) + ((c >> 2) & 1) * 8, y[0], y[1], y[2], y[3]);
    }
  __syncthreads();
  if (wave != 0) return;

  // ---- the attention of the one block ------------------------------------------------------------------------------------------------------------
  const int li = lane & 31, g = lane >> 5;
  auto rows_of = [&](uint32_t base, frag (&o)[4]) __attribute__((always_inline)) {   // row li, contraction elements 16 x + 8 g + 0 .. 7
#pragma unroll
    for (int x = 0; x < 4; ++x) o[x] = *(LDS_AS const frag*)(uintptr_t)(base + li * kRow + (((g ^ ring_f(li)) * 16) ^ (32 * x)));
  };
  frag qf[4], kf[4], e[4][4];   // e: E_K's rows of block 0, block 1, E_Q's
  rows_of(lds0, qf);
  rows_of(lds0 + kRows * kRow, kf);
#pragma unroll
  for (int t = 0; t < 4; ++t) rows_of(lds0 + kOffE + t * 32 * kRow, e[t]);
#pragma unroll
  for (int x = 0; x < 4; ++x) qf[x] = QT::from_f32(QT::to_f32(qf[x]) * p.scale_log2);   // the soft-max scale, in base 2
  f32x16 zero, c[2], pr[2], s;
#pragma unroll
  for (int v = 0; v < 16; ++v) zero[v] = 0.f;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    c[0] = QT::mma(e[0][x], qf[x], x == 0 ? zero : c[0]);
    c[1] = QT::mma(e[1][x], qf[x], x == 0 ? zero : c[1]);
  }
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    pr[0] = QT::mma(kf[x], e[2][x], x == 0 ? zero : pr[0]);
    pr[1] = QT::mma(kf[x], e[3][x], x == 0 ? zero : pr[1]);
    s = QT::mma(kf[x], qf[x], x == 0 ? zero : s);
  }
  // C[li][column 32 bk + m] through the scratch; element (jj, li) wants column li + 32 - jj, and register 4 q + t is key jj = 8 q + 4 g + 3 - t
  typename QT::scratch_t* row = (typename QT::scratch_t*)(smem + kOffScr) + li * kPitch;
#pragma unroll
  for (int bk = 0; bk < 2; ++bk)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *(typename QT::scratch4*)(row + 32 * bk + 8 * q + 4 * g) = QT::pack4(f32x4{c[bk][4 * q], c[bk][4 * q + 1], c[bk][4 * q + 2], c[bk][4 * q + 3]});
  wave_lds_fence();
  float xs[16], px[16];
#pragma unroll
  for (int v = 0; v < 16; ++v) xs[v] = (li + 4 * g < 32 - (8 * (v >> 2) + 3 - (v & 3))) ? pr[1][v] : pr[0][v];
  if (g == 0)
    rotate16<32>(xs, px, std::make_integer_sequence<int, 16>{});
  else
    rotate16<28>(xs, px, std::make_integer_sequence<int, 16>{});
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int v = 4 * q + t;
      s[v] = __builtin_fmaf(px[v], p.scale_log2, s[v] + (float)row[li + 29 - 8 * q - 4 * g + t]);
      if (8 * q + 4 * g + 3 - t >= Lb) s[v] = -INFINITY;
    }
  float mx = s[0];
#pragma unroll
  for (int v = 1; v < 16; ++v) mx = fmaxf(mx, s[v]);
  mx = wave_half_max(mx);
  const float m = mx > -INFINITY ? mx : 0.f;
  frag pf[2];
  float l = 0.f;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    f32x8 pv;
#pragma unroll
    for (int t = 0; t < 8; ++t) pv[t] = __builtin_amdgcn_exp2f(s[8 * k + (t ^ 3)] - m);   // the V^T operand takes the keys in ascending order
    pf[k] = QT::from_f32(pv);
    l = sum8(pv, l);
  }
  l = wave_half_sum(l);
  f32x16 o[2] = {zero, zero};
  const int s16 = lane & 15, grp = lane >> 4, slotl = (2 * (grp & 1) + ((s16 & 3) >> 1)) ^ (4 * ((s16 >> 3) & 1)) ^ (grp >> 1);
  const uint32_t vlane = lds0 + 2 * kRows * kRow, vat = (uint32_t)((4 * (grp >> 1) + (s16 >> 2)) * kRow + slotl * 16 + (s16 & 1) * 8);
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(uintptr_t)(vlane + (vat ^ (64 * d)) + 2048 * k));
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(uintptr_t)(vlane + (vat ^ (64 * d) ^ 32) + 2048 * k + 1024));
      o[d] = QT::mma(__builtin_bit_cast(frag, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)), pf[k], o[d]);
    }
  if (li >= Lb) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  char* orow = ob + (int64_t)(tok0 + li) * o_row * 2;
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      QT::store4(orow + (32 * d + 8 * q + 4 * g) * 2, o[d][4 * q] * inv, o[d][4 * q + 1] * inv, o[d][4 * q + 2] * inv, o[d][4 * q + 3] * inv);
}

template <class QT>
int launch(const SmallParams& p, hipStream_t stream) {
  auto kern = fdb_small_kernel<QT>;
  static std::atomic<uint64_t> lds_set{0};
  const hipError_t e = fdb_set_lds_once((const void*)kern, kLds, lds_set);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.B * p.H)), dim3(kThreads), kLds, stream, p);
  return (int)hipGetLastError();
}

}  // namespace

// One workgroup fills a CU (132 KB of LDS), so a round of them is where it is faster: 24 x 32 at 12 heads, 288 workgroups, 16.1 us as two launches and
// 17.1 here, 48 x 32 24.5 and 25.1.
extern "C" int32_t fdb_layer_small_serves(int64_t batch, int64_t seqlen, int64_t heads, int64_t depth) {
  return batch >= 1 && heads >= 1 && seqlen >= 1 && seqlen <= kRows && depth >= kDepth && depth % kDepth == 0 && batch <= (1 << 16) && heads <= (1 << 16) &&
         batch * heads <= fdb_cu_count();
}

int fdb_launch_small(const void* x, const void* w, const void* bias, const void* pos_key, const void* pos_query, void* out, const int32_t* start, const int32_t* length,
                     const int16_t* lut, int32_t batch, int32_t seqlen, int32_t heads, int32_t depth, int64_t ldx, int64_t ldw, int64_t pk_sh, int64_t pk_sr, int64_t pq_sh,
                     int64_t pq_sr, int32_t radius, float sm_scale, int dtype, void* stream) {
  const SmallParams p{(const char*)x, (const char*)w, (const char*)bias, (const char*)pos_key, (const char*)pos_query, (char*)out, start, length, lut, ldx, ldw, pk_sh, pk_sr,
                      pq_sh, pq_sr, batch, seqlen, heads, depth, radius, sm_scale * 1.4426950408889634f};
  return dtype == FDB_BF16 ? launch<Bf16Tr>(p, (hipStream_t)stream) : launch<F16Tr>(p, (hipStream_t)stream);
}

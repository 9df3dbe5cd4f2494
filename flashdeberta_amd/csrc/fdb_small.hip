// A whole attention layer of short texts in one launch: the three projections and the attention of one head of one sequence by one workgroup, for
// sequences of up to 128 tokens, head_dim 64, 16-bit types, both position terms.
//
// At these sizes a layer is latency.  As two launches, 1 x 24 at 12 heads is 4.5 us for the projections, a gap, and 6.5 us for a near launch whose one step
// of work takes 1.9.  Here a workgroup streams its head's 192 rows of the joined weights (295 KB at a depth of 768) and its sequence's rows through
// LDS stages, as fdb_gemm.hip's tiles do, leaves q, k and v rounded to the type in LDS, where the attention's operands are read from, and does the
// attention by blocks of 32 x 32: fdb_near.hip's products and skews, with all scores of a row in registers and so without a running soft-max; two waves share the
// keys of a query block where there are two or more.  The rows of either table that the blocks' relative positions name are on their way while
// the projections are made.
//
// What bounds it: the weights on their way into one CU's LDS (1 x 24: 3.8 of 8.1 us; four stages of 28 KB on their way at a time, about what a latency of 1.1 us lets
// through; five stages instead of four, where they fit, 9.3 -> 9.1 us a pass), then one wave's chain of products, exponentials and LDS trips (1.6); and the host.
// Pass of a layer, two launches -> one, us (12 heads, depth 768, bf16, passes back to back):
//   1 x 24 13.8 -> 9.1   4 x 24 14.2 -> 9.1   16 x 32 14.9 -> 9.5   21 x 32 15.3 -> 9.9     1 x 48 14.4 -> 11.2   8 x 64 15.6 -> 11.4   21 x 64 18.7 -> 12.8
//   8 x 128 20.3 -> 17.7   21 x 100 24.4 -> 18.4.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <utility>

#include "fdb_device.h"
#include "fdb_kernels.h"
#include "../../include/fdb.h"

using namespace fdb;

namespace {

constexpr int kDepth = 64, kRow = 128, kCols = 192;              // depth of a stage; bytes of a row of it, of a head's q, k or v and of a table; q | k | v
constexpr int kPitch = 68;                                       // 16-bit elements of a scratch row: 64 columns
constexpr int kScr = 32 * kPitch * 2;

// NB blocks of 32 tokens.  PARTS waves share the keys of a query block.
template <int NB>
struct Small {
  static constexpr int ROWS = 32 * NB, NW = NB == 1 ? 4 : 8, WM = NB == 1 ? 1 : 2, FM = ROWS / (16 * WM), FN = 3;
  static constexpr int STAGES = NB == 1 ? 5 : NB == 2 ? 4 : 3, STAGE = (ROWS + kCols) * kRow, LOADS = (ROWS + kCols) / 8 / NW;
  static constexpr int TABLE = 2 * ROWS * kRow, TABLE_LOADS = 2 * ROWS / 8 / NW;   // rows -ROWS .. ROWS - 1 of a table
  static constexpr bool LATE = NB == 4;   // no room for the second table beside the stages: it takes the place of one of the last
  static constexpr int PARTS = NB == 1 ? 1 : 2, BLOCKS = NB / PARTS;
  static constexpr int OFF_E = STAGES * STAGE, E_BYTES = LATE ? TABLE + kScr : 2 * TABLE, LDS = OFF_E + E_BYTES;
  static constexpr int MERGE = 34 * 64 * 4;   // a wave's partial result
  static constexpr int V_SCR = LATE ? (STAGE - ROWS * kRow) / kScr : NB * PARTS;   // waves whose scratch follows v
  static_assert((ROWS + kCols) % (8 * NW) == 0 && LDS <= 160 * 1024 && NB * MERGE <= E_BYTES, "whole loads, LDS");
  static_assert(LATE ? V_SCR + 3 >= NB * PARTS && 2 * ROWS * kRow + kScr <= STAGE && TABLE + kScr <= STAGE : 3 * ROWS * kRow + V_SCR * kScr <= STAGES * STAGE,
                "LATE: q and k, or v, or a table in a stage's place, and a scratch behind each");
};

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

template <class QT, int NB>
__global__ __launch_bounds__(64 * Small<NB>::NW, Small<NB>::NW / 4) void fdb_small_kernel(const SmallParams p) {
  using S = Small<NB>;
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
  if (Lb < p.L && tid < 256) fill_pad_rows<kRow>(ob, o_row * 2, 0, p.L, tok0, Lb, sl < 0 ? QT::NAN_WORD : 0u, tid);
  if (Lb == 0) return;

  // ---- the projections: [ROWS x 192] outputs of a contraction over depth, stages of 64 --------------------------------------------------------
  const char* pkb = p.pk + (int64_t)h * p.pk_sh * 2;
  const char* pqb = p.pq + (int64_t)h * p.pq_sh * 2;
  const int srow = lane >> 3, slot = lane & 7;
  int delta[S::TABLE_LOADS];   // table row e holds relative position e - ROWS
#pragma unroll
  for (int j = 0; j < S::TABLE_LOADS; ++j) {
    const int r = 8 * (wave + S::NW * j) + srow - S::ROWS;
    delta[j] = (int)((const uint16_t*)p.lut)[max(-p.R, min(p.R, r)) + p.R];
  }
  const int r16 = lane & 15, kg = lane >> 4, wm = wave / 4, wn = wave % 4;
  f32x4 bias[S::FN];
#pragma unroll
  for (int j = 0; j < S::FN; ++j) {
    const int col = wn * 48 + j * 16 + 4 * kg;
    bias[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (p.bias) bias[j] = QT::load4(p.bias + ((int64_t)(col >> 6) * p.H * 64 + h * 64 + (col & 63)) * 2);
  }
  const char* xb = p.x + ((int64_t)b * p.L + tok0) * p.ldx * 2;
  const char* wb = p.w + (int64_t)h * 64 * p.ldw * 2;
  uint32_t off[S::LOADS];
#pragma unroll
  for (int j = 0; j < S::LOADS; ++j) {
    const int c = wave + S::NW * j, row = 8 * c + srow, col = row - S::ROWS;   // rows past the end re-read the last one
    const uint32_t place = c < S::ROWS / 8 ? (uint32_t)min(row, Lb - 1) * (uint32_t)(p.ldx * 2) : (uint32_t)((col >> 6) * p.H * 64 + (col & 63)) * (uint32_t)(p.ldw * 2);
    off[j] = place + (uint32_t)((slot ^ swz16(row)) * 16);
  }
  int into = 0;   // the buffer the next stage goes to
  auto load = [&](int t, uint32_t dst, int j) __attribute__((always_inline)) {
    dma16sn((wave + S::NW * j < S::ROWS / 8 ? xb : wb) + (uint64_t)(uint32_t)t * kRow, off[j], dst + (uint32_t)wave * 1024u + j * S::NW * 1024u);
  };
  auto next_buffer = [&]() __attribute__((always_inline)) {
    const uint32_t dst = lds0 + (uint32_t)into * S::STAGE;
    into = into == S::STAGES - 1 ? 0 : into + 1;
    return dst;
  };
  auto table_dma = [&](const char* table, int64_t stride, uint32_t to) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < S::TABLE_LOADS; ++j) {
      const int c = wave + S::NW * j;
      dma16sn(table, __umul24((uint32_t)delta[j], (uint32_t)(stride * 2)) + (uint32_t)((slot ^ ring_f(8 * c + srow)) * 16), to + (uint32_t)c * 1024u);
    }
  };
  const int steps = p.K / kDepth;
#pragma unroll
  for (int t = 0; t < S::STAGES - 1; ++t) {
    const uint32_t dst = next_buffer();
    if (t < steps) {
#pragma unroll
      for (int j = 0; j < S::LOADS; ++j) load(t, dst, j);
    }
  }
  // (taken here: the compiler does not count the direct loads)
#pragma unroll
  for (int j = 0; j < S::TABLE_LOADS; ++j) asm volatile("" : "+v"(delta[j]));
#pragma unroll
  for (int j = 0; j < S::FN; ++j) asm volatile("" : "+v"(bias[j]));
  uint32_t ek = lds0 + S::OFF_E, eq = ek + S::TABLE;
  table_dma(pkb, p.pk_sr, ek);
  if constexpr (!S::LATE) table_dma(pqb, p.pq_sr, eq);
  f32x4 acc[S::FM][S::FN];
#pragma unroll
  for (int i = 0; i < S::FM; ++i)
#pragma unroll
    for (int j = 0; j < S::FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t xrow = (uint32_t)((wm * S::FM * 16 + r16) * kRow), wrow = (uint32_t)((S::ROWS + wn * 48 + r16) * kRow), f = (uint32_t)swz16(r16);
  int buf = 0;
#pragma unroll 1
  for (int t = 0; t < steps; ++t) {
    // this wave's loads of stage t have landed, those of the stages after it may still fly (and the tables' rows with them)
    if (t + S::STAGES - 1 <= steps) wait_vmcnt<(S::STAGES - 2) * S::LOADS>();
    else wait_vmcnt<0>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();   // ... and everybody's; everybody has read stage t - 1
    asm volatile("" ::: "memory");
    const uint32_t at = lds0 + (uint32_t)buf * S::STAGE;
    frag xf[2][S::FM], wf[2][S::FN];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const uint32_t sl16 = ((uint32_t)(4 * s + kg) ^ f) * 16;
#pragma unroll
      for (int j = 0; j < S::FN; ++j) wf[s][j] = *(LDS_AS const frag*)(uintptr_t)(at + wrow + sl16 + j * 16 * kRow);
#pragma unroll
      for (int i = 0; i < S::FM; ++i) xf[s][i] = *(LDS_AS const frag*)(uintptr_t)(at + xrow + sl16 + i * 16 * kRow);
    }
    __builtin_amdgcn_sched_barrier(0);
    // A load holds its wave until the CU's memory pipeline takes it: the products run meanwhile
    const bool more = t + S::STAGES - 1 < steps;
    uint32_t dst = 0;
    if (more) {
      dst = next_buffer();
    } else if (S::LATE && t == max(steps - 2, 0)) {   // the first buffer that no stage wants
      eq = lds0 + (uint32_t)into * S::STAGE;
      table_dma(pqb, p.pq_sr, eq);
    }
    constexpr int PRODUCTS = 2 * S::FM * S::FN, EACH = PRODUCTS / S::LOADS;
#pragma unroll
    for (int n = 0; n < PRODUCTS; ++n) {
      if (n % EACH == 0 && n / EACH < S::LOADS) {
        __builtin_amdgcn_sched_barrier(0);
        if (more) load(t + S::STAGES - 1, dst, n / EACH);
        __builtin_amdgcn_sched_barrier(0);
      }
      const int s = n / (S::FM * S::FN), i = n / S::FN % S::FM, j = n % S::FN;
      acc[i][j] = mma16(wf[s][j], xf[s][i], acc[i][j]);
    }
    buf = buf == S::STAGES - 1 ? 0 : buf + 1;
  }
  wait_vmcnt<0>();
  __syncthreads();   // the stages have been read, the tables' rows are there
  // q, k and v as the attention reads them: rows of 128 bytes, slot (row, s) = chunk s ^ ring_f(row), k's rows with the low two bits inverted.  They and the
  // scratch lie where the stages were (LATE: in the two buffers that hold no table).
  uint32_t qk = lds0, vs = lds0 + 2 * S::ROWS * kRow;
  if constexpr (S::LATE) {
    const uint32_t x = (eq - lds0) / S::STAGE;
    qk = lds0 + (x == 2 ? 0 : x + 1) * S::STAGE, vs = lds0 + (x == 0 ? 2 : x - 1) * S::STAGE;
  }
#pragma unroll
  for (int j = 0; j < S::FN; ++j)
#pragma unroll
    for (int i = 0; i < S::FM; ++i) {
      const int col = wn * 48 + j * 16 + 4 * kg, what = col >> 6, c = col & 63, row = (wm * S::FM * 16 + i * 16 + r16) ^ (what == 1 ? 3 : 0);
      const f32x4 y = acc[i][j] + bias[j];
      const uint32_t at = (what == 2 ? vs : qk + (uint32_t)what * (S::ROWS * kRow)) + (uint32_t)(row * kRow + (((c >> 3) ^ ring_f(row)) * 16) + ((c >> 2) & 1) * 8);
      *(LDS_AS typename QT::scratch4*)(uintptr_t)at = QT::pack4(y);
    }
  __syncthreads();

  // ---- the attention: wave (query block, part), BLOCKS key blocks each ------------------------------------------------------------------------------
  const int qb = wave % NB, part = wave / NB, li = lane & 31, g = lane >> 5;
  const bool works = part < S::PARTS && 32 * qb < Lb;
  f32x16 zero, o[2];
#pragma unroll
  for (int v = 0; v < 16; ++v) zero[v] = o[0][v] = o[1][v] = 0.f;
  float m = -INFINITY, l = 0.f;   // of the scores; the sum of exp2(score - m)
  if (works) {
    auto rows_of = [&](uint32_t base, frag (&r)[4]) __attribute__((always_inline)) {   // row li, contraction elements 16 x + 8 g + 0 .. 7
#pragma unroll
      for (int x = 0; x < 4; ++x) r[x] = *(LDS_AS const frag*)(uintptr_t)(base + li * kRow + (((g ^ ring_f(li)) * 16) ^ (32 * x)));
    };
    frag qf[4];
    rows_of(qk + qb * 32 * kRow, qf);
#pragma unroll
    for (int x = 0; x < 4; ++x) qf[x] = QT::from_f32(QT::to_f32(qf[x]) * p.scale_log2);   // the soft-max scale, in base 2
    const uint32_t scr = (wave < S::V_SCR ? vs + S::ROWS * kRow + (uint32_t)(wave * kScr)
                                          : wave == S::V_SCR ? ek + S::TABLE : wave == S::V_SCR + 1 ? qk + 2 * S::ROWS * kRow : eq + S::TABLE) + (uint32_t)(li * (kPitch * 2));
    f32x16 s[S::BLOCKS];
#pragma unroll
    for (int n = 0; n < S::BLOCKS; ++n) {
      const int kb = part * S::BLOCKS + n;
      if (32 * kb >= Lb) {
#pragma unroll
        for (int v = 0; v < 16; ++v) s[n][v] = -INFINITY;
        continue;
      }
      frag kf[4], e[4][4];   // e: E_K's rows of block 0 (relative positions below the blocks' distance) and block 1, E_Q's
      rows_of(qk + (S::ROWS + kb * 32) * kRow, kf);
      const uint32_t lower = (uint32_t)((qb - kb + NB - 1) * 32 * kRow);
#pragma unroll
      for (int t = 0; t < 4; ++t) rows_of((t < 2 ? ek : eq) + lower + (t & 1) * 32 * kRow, e[t]);
      f32x16 c[2], pr[2];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        c[0] = QT::mma(e[0][x], qf[x], x == 0 ? zero : c[0]);
        c[1] = QT::mma(e[1][x], qf[x], x == 0 ? zero : c[1]);
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        pr[0] = QT::mma(kf[x], e[2][x], x == 0 ? zero : pr[0]);
        pr[1] = QT::mma(kf[x], e[3][x], x == 0 ? zero : pr[1]);
        s[n] = QT::mma(kf[x], qf[x], x == 0 ? zero : s[n]);
      }
      // C[li][column 32 bk + m] through the scratch; element (jj, li) wants column li + 32 - jj, and register 4 q + t is key jj = 8 q + 4 g + 3 - t
      wave_lds_fence();
#pragma unroll
      for (int bk = 0; bk < 2; ++bk)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *(LDS_AS typename QT::scratch4*)(uintptr_t)(scr + 2 * (32 * bk + 8 * q + 4 * g)) = QT::pack4(f32x4{c[bk][4 * q], c[bk][4 * q + 1], c[bk][4 * q + 2], c[bk][4 * q + 3]});
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
          const float cv = (float)*(LDS_AS const typename QT::scratch_t*)(uintptr_t)(scr + 2 * (li + 29 - 8 * q - 4 * g + t));
          s[n][v] = __builtin_fmaf(px[v], p.scale_log2, s[n][v] + cv);
          if (32 * kb + 8 * q + 4 * g + 3 - t >= Lb) s[n][v] = -INFINITY;
        }
    }
#pragma unroll
    for (int n = 0; n < S::BLOCKS; ++n)
#pragma unroll
      for (int v = 0; v < 16; ++v) m = fmaxf(m, s[n][v]);
    m = wave_half_max(m);
    const float from_m = m > -INFINITY ? m : 0.f;
    const int s16 = lane & 15, grp = lane >> 4, slotl = (2 * (grp & 1) + ((s16 & 3) >> 1)) ^ (4 * ((s16 >> 3) & 1)) ^ (grp >> 1);
    const uint32_t vat = (uint32_t)((4 * (grp >> 1) + (s16 >> 2)) * kRow + slotl * 16 + (s16 & 1) * 8);
#pragma unroll
    for (int n = 0; n < S::BLOCKS; ++n) {
      const uint32_t vb = vs + (uint32_t)((part * S::BLOCKS + n) * 32 * kRow);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        f32x8 pv;
#pragma unroll
        for (int t = 0; t < 8; ++t) pv[t] = __builtin_amdgcn_exp2f(s[n][8 * k + (t ^ 3)] - from_m);   // the V^T operand takes the keys in ascending order
        const frag pf = QT::from_f32(pv);
        l = sum8(pv, l);
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(uintptr_t)(vb + (vat ^ (64 * d)) + 2048 * k));
          const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(uintptr_t)(vb + (vat ^ (64 * d) ^ 32) + 2048 * k + 1024));
          o[d] = QT::mma(__builtin_bit_cast(frag, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)), pf, o[d]);
        }
      }
    }
    l = wave_half_sum(l);
  }
  if constexpr (S::PARTS > 1) {
    // the second part's sums, in the place of the tables' rows, to the first part's wave
    __syncthreads();
    const uint32_t at = ek + (uint32_t)(qb * S::MERGE + lane * 4);
    if (works && part == 1) {
#pragma unroll
      for (int v = 0; v < 32; ++v) *(LDS_AS float*)(uintptr_t)(at + v * 256) = o[v >> 4][v & 15];
      *(LDS_AS float*)(uintptr_t)(at + 32 * 256) = m;
      *(LDS_AS float*)(uintptr_t)(at + 33 * 256) = l;
    }
    __syncthreads();
    if (!works || part != 0) return;
    const float m1 = *(LDS_AS const float*)(uintptr_t)(at + 32 * 256), l1 = *(LDS_AS const float*)(uintptr_t)(at + 33 * 256), top = fmaxf(m, m1);
    const float w0 = m > -INFINITY ? __builtin_amdgcn_exp2f(m - top) : 0.f, w1 = m1 > -INFINITY ? __builtin_amdgcn_exp2f(m1 - top) : 0.f;
    l = w0 * l + w1 * l1;
#pragma unroll
    for (int v = 0; v < 32; ++v) o[v >> 4][v & 15] = w0 * o[v >> 4][v & 15] + w1 * *(LDS_AS const float*)(uintptr_t)(at + v * 256);
  }
  const int i = 32 * qb + li;
  if (!works || i >= Lb) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  char* orow = ob + (int64_t)(tok0 + i) * o_row * 2;
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      QT::store4(orow + (32 * d + 8 * q + 4 * g) * 2, o[d][4 * q] * inv, o[d][4 * q + 1] * inv, o[d][4 * q + 2] * inv, o[d][4 * q + 3] * inv);
}

template <class QT, int NB>
int launch_blocks(const SmallParams& p, hipStream_t stream) {
  auto kern = fdb_small_kernel<QT, NB>;
  static std::atomic<uint64_t> lds_set{0};
  const hipError_t e = fdb_set_lds_once((const void*)kern, Small<NB>::LDS, lds_set);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.B * p.H)), dim3(64 * Small<NB>::NW), Small<NB>::LDS, stream, p);
  return (int)hipGetLastError();
}
template <class QT>
int launch(const SmallParams& p, hipStream_t stream) {
  return p.L <= 32 ? launch_blocks<QT, 1>(p, stream) : p.L <= 64 ? launch_blocks<QT, 2>(p, stream) : launch_blocks<QT, 4>(p, stream);
}

}  // namespace

// One workgroup fills a CU (160 KB of LDS), so a round of them is where it is faster: 24 x 32 at 12 heads, 288 workgroups, 16.1 us as two launches and
// 17.1 here, 48 x 32 24.5 and 25.1; 32 x 64 22.4 and 22.7.  Beyond 64 tokens the workgroup's own time, which grows with the depth, is that of two launches
// for few rows, whose time grows with the batch: at 12 heads 1 x 100 15.6 and 17.2, 3 x 128 17.4 and 17.5, 4 x 100 17.7 and 17.3, 12 x 128 23.4 and 18.0.  Other widths, a
// layer replayed one by one (its start of about 18 us included), two launches and one:
//   6 heads, depth 384     1 x 80  32.7 and 32.8   2 x 100 34.4 and 34.1   2 x 128 34.4 and 34.3   16 x 128 38.4 and 34.5   40 x 128 46.6 and 39.1
//   16 heads, depth 1024   1 x 80  49.4 and 47.3   1 x 100 51.2 and 48.3   4 x 128 53.5 and 51.1   8 x 100 54.3 and 51.6   16 x 128 58.3 and 51.8   1 x 48 45.4 and 41.0
//   24 heads, depth 1536   1 x 80  55.1 and 60.7   2 x 100 61.4 and 61.5   4 x 100 64.8 and 60.7   8 x 100 68.5 and 61.9   10 x 128 69.9 and 61.6   1 x 48 53.1 and 52.8
// (so at 16 heads the line is on the safe side by up to 5 %).
extern "C" int32_t fdb_layer_small_serves(int64_t batch, int64_t seqlen, int64_t heads, int64_t depth) {
  return batch >= 1 && heads >= 1 && seqlen >= 1 && seqlen <= 128 && depth >= kDepth && depth % kDepth == 0 && batch <= (1 << 16) && heads <= (1 << 16) &&
         batch * heads <= fdb_cu_count() && (seqlen <= 64 || 2 * batch * seqlen > depth);
}

int fdb_launch_small(const void* x, const void* w, const void* bias, const void* pos_key, const void* pos_query, void* out, const int32_t* start, const int32_t* length,
                     const int16_t* lut, int32_t batch, int32_t seqlen, int32_t heads, int32_t depth, int64_t ldx, int64_t ldw, int64_t pk_sh, int64_t pk_sr, int64_t pq_sh,
                     int64_t pq_sr, int32_t radius, float sm_scale, int dtype, void* stream) {
  const SmallParams p{(const char*)x, (const char*)w, (const char*)bias, (const char*)pos_key, (const char*)pos_query, (char*)out, start, length, lut, ldx, ldw, pk_sh, pk_sr,
                      pq_sh, pq_sr, batch, seqlen, heads, depth, radius, sm_scale * 1.4426950408889634f};
  return dtype == FDB_BF16 ? launch<Bf16Tr>(p, (hipStream_t)stream) : launch<F16Tr>(p, (hipStream_t)stream);
}

// Backward of the disentangled attention for gfx950, head_dim 64, 16-bit types, both position terms: dQ, dK, dV and the
// gradients of the two tables, without position-score tensors in memory.  (fdb_bwd.hip, which gathers the scores from tensors
// and returns their gradients as tensors, serves the other types, head_dims and term sets.)
// Counterpart of src/flashdeberta/ops/flash_attention.py:490-1086 and of the autograd backward of model.py:189-192.
//
// Two roles of one kernel, as one launch or one after the other, then two small launches for the tables:
//   role dQ    : lane side X = queries (4 waves x 32 rows, one row per lane and its partner lane ^ 32), loop side Y = keys
//   role dK/dV : X = keys, Y = queries
// With x a lane row, y a loop row and r' = x - y (the relative position i - j in the dQ role, j - i in the other) both roles see
// one geometry, and a 32-row step of the loop is one of three kinds, as in the forward:
//   far   every |r'| >= R: the term of the lane row is a constant of the row, the term of the loop row is folded into the lane
//         side's operand (x + the saturated table row); the score gradients' sums over the step are all the tables get;
//   near  the 63 relative positions of a wave's 32 x 32 block are two blocks of 32 table rows, contracted from LDS rings of
//         expanded tables E[r'] = table[delta(r')]; the skews are the near forward's (fdb_near.hip): the lane row's product
//         through a per-wave scratch, the loop row's by rotations of half-waves.
// What the backward adds is the way back through the tables.  The scratch entry (x, r') holds the lane row's score of exactly one
// element (x, y), so once the element's score gradient is known it takes that entry's place: a block of 32 relative
// positions is complete after the two steps that meet it, and is then
//   * an MFMA operand: dX[x] += sum_r' G[x][r'] E[r'] (four MFMAs; E read transposed from the ring), and
//   * in the dQ role, stored (2 KB per wave and step, 64 contiguous bytes per row) for the tables' gradients,
//       dK_r: dE_K[r] = sum_i G[i][r] q_i,   dQ_r: dE_Q[r] = sum_i G[i][r] k_(i-r),
//     which fdb_table_grad_kernel accumulates over all tokens for its relative positions (the rows of G read back shifted
//     against each other for the second one) and fdb_table_fold_kernel sums over the positions of a table row.
// Against gathers from score tensors and score gradients collected per table row (fdb_bwd.hip), bf16, 12 heads, mean of a launch
// (a box or its warmth moves these by up to 8 %):
//   B = 8, L = 4096   dQ 1377 -> 956 us, dK/dV 1553 -> 1125 us; score products, chain and transposes 600 -> 309 us (tables)
//   B = 8, L = 512    68 + 66 -> 83 us (both as one launch); around them 90 -> 46 us (row statistics, tables)
// A near step is bound like the forward's by what its waves issue (with two waves per SIMD, one instruction per 4.5 clocks each)
// next to its 28 (dQ) or 32 MFMAs; a far step by MFMA plus VALU time.
//
// LDS: tiles 16 KB + ring of the lane side's table 24 KB (six batches: the one whose block completes in a step is read transposed
// while the next one arrives) + ring of the loop side's table 20 KB + scratch 17 KB + statistics: 77.5 KB, two workgroups per CU.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <utility>

#include "fdb_device.h"
#include "fdb_kernels.h"
#include "../../include/fdb.h"

using namespace fdb;

namespace {

constexpr int kThreads = 256;
constexpr int kStep = 32;
constexpr int kRowBytes = 128;                 // head_dim 64, 16-bit
constexpr int kTile = kStep * kRowBytes;       // 4 KB: one 32-row tile, one ring batch
constexpr int kXBatches = 6, kYBatches = 5;    // ring batches of the lane / the loop side's table
constexpr int kScrPitch = 68;                  // 16-bit elements per scratch row, see fdb_near.hip
constexpr int kScrElems = 32 * kScrPitch;
constexpr int kOffX = 4 * kTile, kOffY = kOffX + kXBatches * kTile, kOffScr = kOffY + kYBatches * kTile;
constexpr int kOffStat = kOffScr + 4 * kScrElems * 2;
constexpr int kLds = kOffStat + 2 * 2 * kStep * 4;
static_assert(kLds <= 80 * 1024, "two workgroups per CU");

// slot (row, s) of an unpadded 128-byte row holds chunk s ^ swz(row)
__device__ __forceinline__ int swz(int row) { return 4 * ((row >> 1) & 1) | ((row >> 2) & 3); }

template <int OFFSET>
__device__ __forceinline__ float swizzle_asm(float x) {
  float r;
  asm volatile("ds_swizzle_b32 %0, %1 offset:%2" : "=v"(r) : "v"(x), "n"(OFFSET));
  return r;
}
// px[v] = xs[v] of the lane (ROT0 - c(v)) places further up in this lane's half-wave (mod 32), c(v) = 8*(v/4) + 3 - v%4
template <int ROT0, int... V>
__device__ __forceinline__ void rotate16(const float (&xs)[16], float (&px)[16], std::integer_sequence<int, V...>) {
  ((px[V] = swizzle_asm<(0xC000 | (((ROT0 - (8 * (V >> 2) + 3 - (V & 3))) & 31) << 5))>(xs[V])), ...);
}
template <class QT, int OFF>
__device__ __forceinline__ float lds_elem_f32(uint32_t addr) {
  if constexpr (std::is_same<QT, Bf16Tr>::value) {
    float r;  // the load that fills the upper half of the register clears the lower half: the register is the value
    asm volatile("ds_read_u16_d16_hi %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF));
    return r;
  } else {
    return (float)*(LDS_AS const _Float16*)(uintptr_t)(addr + OFF);
  }
}
// a packed pair's low / high element to LDS
template <int OFF>
__device__ __forceinline__ void lds_put_lo(uint32_t addr, uint32_t pair) {
  asm volatile("ds_write_b16 %0, %1 offset:%2" ::"v"(addr), "v"(pair), "n"(OFF) : "memory");
}
template <int OFF>
__device__ __forceinline__ void lds_put_hi(uint32_t addr, uint32_t pair) {
  asm volatile("ds_write_b16_d16_hi %0, %1 offset:%2" ::"v"(addr), "v"(pair), "n"(OFF) : "memory");
}
__device__ __forceinline__ void lds_wait_all() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

__device__ __forceinline__ u32x4 frag_bits(bf16x8 x) { return __builtin_bit_cast(u32x4, x); }
__device__ __forceinline__ u32x4 frag_bits(f16x8 x) { return __builtin_bit_cast(u32x4, x); }

// The three kinds of steps of the 128-row tile at m0: far (r' >= R) [y_lo, s0), near [s0, s1), far (r' <= -R) [s1, y_hi), in steps.
struct Zones {
  int lo, s0, s1, hi;
};
__device__ __forceinline__ Zones zones_of(int m0, int Lb, int R, bool causal, bool dq) {
  Zones z;
  z.lo = causal && !dq ? m0 / kStep : 0;
  z.hi = ((causal && dq ? min(Lb, m0 + FDB_BM) : Lb) + kStep - 1) / kStep;
  const int lim = m0 - R - (kStep - 1);
  z.s0 = max(z.lo, min(z.hi, lim >= 0 ? lim / kStep + 1 : 0));
  z.s1 = max(z.s0, min(z.hi, (m0 + FDB_BM - 1 + R + kStep - 1) / kStep));
  return z;
}

// near steps cost twice a far one, so the tiles with the most of them start first (causal: those with the most steps)
__device__ __forceinline__ int order_of(const FdbBwdRingParams& p, bool dq) { return p.causal ? (dq ? kLastFirst : kNatural) : kMiddleFirst; }

// One workgroup of a role, the wg-th of its grid.  STATS: the row statistics are there (fdb_row_stats_kernel); otherwise the dQ role,
// launched on its own before the other, computes them on its way.
// BY_LENGTH: of a padded batch, whose place `at` is read from the table of find_places (an instantiation of its own: its registers cost the other 1 to 3 %).
template <class QT, int ROLE, bool STATS, bool BY_LENGTH>
__device__ __forceinline__ void bwd_ring(const FdbBwdRingParams& p, const int wg, const FdbPlace* at) {
  constexpr bool kDQ = ROLE == 0;
  constexpr int KS = 4, DBLKS = 2;
  using frag = typename QT::frag;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LDS_AS char*)smem;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, li = lane & 31, g = lane >> 5;
  int b, tile_x, h;
  if constexpr (BY_LENGTH) b = (int)own_sgpr((uint32_t)at->b), tile_x = (int)own_sgpr((uint32_t)at->tile), h = (int)own_sgpr((uint32_t)at->h);
  else block_map<false>(wg, p.B, p.H, p.tiles, p.groups_together, true, order_of(p, kDQ), b, tile_x, h);
  const int m0 = tile_x * FDB_BM;
  const int tok0 = BY_LENGTH ? (int)own_sgpr((uint32_t)at->tok0) : p.seq_start ? min(max(p.seq_start[b], 0), p.L) : 0;
  const int Lb = BY_LENGTH ? (int)own_sgpr((uint32_t)at->tokens) : p.seq_len ? min(max(p.seq_len[b], 0), p.L - tok0) : p.L;
  if (p.seq_start || p.seq_len) {  // rows of padding have no gradient
    auto clear = [&](char* t, int64_t sb, int64_t st, int64_t sh) {
      fill_pad_rows<kRowBytes>(t + ((int64_t)b * sb + (int64_t)h * sh) * 2, st * 2, tile_x, p.L, tok0, Lb, 0u, tid);
    };
    if (kDQ) {
      clear(p.dq, p.dq_sb, p.dq_st, p.dq_sh);
    } else {
      clear(p.dk, p.dk_sb, p.dk_st, p.dk_sh);
      clear(p.dv, p.dv_sb, p.dv_st, p.dv_sh);
    }
  }
  if (kDQ && wg == 0 && tid < 128) *(u32x4*)(p.zero_block + tid * 16) = u32x4{0u, 0u, 0u, 0u};  // what stands in for a block of G that no step met
  if (m0 >= Lb) return;
  auto base = [&](const char* ptr, int64_t sb, int64_t st, int64_t sh) { return ptr + (b * sb + (int64_t)tok0 * st + (int64_t)h * sh) * 2; };
  const char* qb = base(p.q, p.q_sb, p.q_st, p.q_sh);
  const char* kb = base(p.k, p.k_sb, p.k_st, p.k_sh);
  const char* vb = base(p.v, p.v_sb, p.v_st, p.v_sh);
  const char* gb = base(p.dout, p.g_sb, p.g_st, p.g_sh);
  const char* x1b = kDQ ? qb : kb;
  const char* x2b = kDQ ? gb : vb;
  const int64_t x1_st = kDQ ? p.q_st : p.k_st, x2_st = kDQ ? p.g_st : p.v_st;
  const char* y1b = kDQ ? kb : qb;
  const char* y2b = kDQ ? vb : gb;
  const uint32_t y1_rsb = own_sgpr((uint32_t)((kDQ ? p.k_st : p.q_st) * 2)), y2_rsb = own_sgpr((uint32_t)((kDQ ? p.v_st : p.g_st) * 2));
  const char* pkb = p.pk + (int64_t)h * p.pk_sh * 2;
  const char* pqb = p.pq + (int64_t)h * p.pq_sh * 2;
  const char* txb = kDQ ? pkb : pqb;   // the table the lane side meets, and the loop side's
  const char* tyb = kDQ ? pqb : pkb;
  const uint32_t tx_rowb = own_sgpr((uint32_t)((kDQ ? p.pk_sr : p.pq_sr) * 2)), ty_rowb = own_sgpr((uint32_t)((kDQ ? p.pq_sr : p.pk_sr) * 2));
  const uint16_t* lut = own_sgpr((const uint16_t*)p.lut);
  const int R = (int)own_sgpr((uint32_t)p.R);
  const float x_scale = p.scale_log2;

  const int xw0 = m0 + wave * 32, xr = xw0 + li;
  const bool x_ok = xr < Lb;
  const Zones z = zones_of(m0, Lb, p.R, p.causal, kDQ);
  const int n_near = z.s1 - z.s0;

  // ---- this lane's row ---------------------------------------------------------------------------------------------------
  frag x1[KS], x2[KS];
  auto load_x1 = [&](int s) __attribute__((always_inline)) { return x_ok ? QT::load(x1b + ((int64_t)xr * x1_st + 16 * s + 8 * g) * 2) : QT::zero(); };
#pragma unroll
  for (int s = 0; s < KS; ++s) x2[s] = x_ok ? QT::load(x2b + ((int64_t)xr * x2_st + 16 * s + 8 * g) * 2) : QT::zero();
  const int64_t stat_row = ((int64_t)b * p.H + h) * p.stat_len;   // row statistics by (batch row, head), local row index
  float lse_x = 0.f, del_x = 0.f;   // dQ role: -lse in base 2, -Delta
  if (kDQ && STATS) {
    if (x_ok) {
      lse_x = p.neg_lse[stat_row + xr];
      del_x = p.neg_delta[stat_row + xr];
    }
  } else if (kDQ) {
    // Delta = dO . O of this lane's row; both statistics are left for the dK/dV launch in the form it starts its products from
    const char* ob = base(p.out, p.o_sb, p.o_st, p.o_sh);
    float dot = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const f32x8 o8 = QT::to_f32(x_ok ? QT::load(ob + ((int64_t)xr * p.o_st + 16 * s + 8 * g) * 2) : QT::zero()), g8 = QT::to_f32(x2[s]);
#pragma unroll
      for (int e = 0; e < 8; ++e) dot = __builtin_fmaf(o8[e], g8[e], dot);
    }
    del_x = -wave_half_sum(dot);
    if (x_ok) lse_x = p.lse[((int64_t)b * p.L + tok0 + xr) * p.H + h] * -1.4426950408889634f;
    if (x_ok && g == 0) {
      p.neg_lse[stat_row + xr] = lse_x;
      p.neg_delta[stat_row + xr] = del_x;
    }
  }
  f32x16 acc1[DBLKS], acc2[DBLKS];  // dQ^T / dK^T and dV^T
#pragma unroll
  for (int d = 0; d < DBLKS; ++d)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc1[d][v] = acc2[d][v] = 0.f;
  float far_sum[2] = {0.f, 0.f};    // this row's score gradients over the far steps of either side
  float edge_sum[2] = {0.f, 0.f};   // ... and over the elements |r'| >= R of its near steps
  f32x16 zero;
#pragma unroll
  for (int v = 0; v < 16; ++v) zero[v] = 0.f;

  // ---- staging: tiles, ring batches ------------------------------------------------------------------------------------
  // A direct load fills 1 KB = 8 rows per wave; thread tid owns slot scc of row srow.  Tile row srow holds loop row srow ^ 3 of the
  // step (see fdb_near.hip); rows past the end re-read the last one, their scores are masked.
  const int srow = tid >> 3, scc = tid & 7;
  const uint32_t chunk_off = (uint32_t)((scc ^ swz(srow)) * 16), wave_kb = lds0 + (uint32_t)wave * 1024u;
  const uint32_t y1_lane = (uint32_t)(srow ^ 3) * y1_rsb + chunk_off, y2_lane = (uint32_t)(srow ^ 3) * y2_rsb + chunk_off;
  auto tiles_dma = [&](int s, int buf) __attribute__((always_inline)) {
    if ((s + 1) * kStep <= Lb) {
      dma16sn(y1b + (uint64_t)(uint32_t)(s * kStep) * y1_rsb, y1_lane, wave_kb + buf * kTile);
      dma16sn(y2b + (uint64_t)(uint32_t)(s * kStep) * y2_rsb, y2_lane, wave_kb + 2 * kTile + buf * kTile);
    } else {
      const uint32_t row = (uint32_t)min(s * kStep + (srow ^ 3), Lb - 1);
      dma16n(y1b + (uint64_t)row * y1_rsb + chunk_off, wave_kb + buf * kTile);
      dma16n(y2b + (uint64_t)row * y2_rsb + chunk_off, wave_kb + 2 * kTile + buf * kTile);
    }
    // the loop rows' statistics, in the order of the tile rows: the log-sum-exps in the first half-wave, the Deltas in the second
    if (!kDQ && wave == 0)
      dma4((g == 0 ? p.neg_lse : p.neg_delta) + stat_row + s * kStep + (li ^ 3), lds0 + kOffStat + (uint32_t)(buf * 2 * kStep * 4));
  };
  int r_tab = 0;
  auto batch_delta = [&]() __attribute__((always_inline)) {
    const int r = kDQ ? r_tab : -r_tab;
    const int d = (int)lut[(uint32_t)(max(-R, min(R, r)) + R)];
    r_tab -= 32;
    return d;
  };
  auto batch_dma = [&](int delta, int xslot, int yslot) __attribute__((always_inline)) {
    dma16sn(txb, __umul24((uint32_t)delta, tx_rowb) + chunk_off, wave_kb + kOffX + (uint32_t)xslot * kTile);
    dma16sn(tyb, __umul24((uint32_t)delta, ty_rowb) + chunk_off, wave_kb + kOffY + (uint32_t)yslot * kTile);
  };

  // ---- per-lane LDS addresses ----------------------------------------------------------------------------------------------
  uint32_t yl[KS], yt[4];  // row fragments and transposed operands of a tile, see fdb_near.hip
  {
    const int s16 = lane & 15, grp = lane >> 4;
    const int slotl = (2 * (grp & 1) + ((s16 & 3) >> 1)) ^ (4 * ((s16 >> 3) & 1)) ^ (grp >> 1);
    const uint32_t vlane = (4 * (grp >> 1) + (s16 >> 2)) * kRowBytes + slotl * 16 + (s16 & 1) * 8;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      yl[x] = lds0 + ((li * kRowBytes + ((g ^ swz(li)) * 16)) ^ (32 * x));
      yt[x] = lds0 + (vlane ^ (64 * (x >> 1) ^ 32 * (x & 1)));
    }
  }
  auto y_frag = [&](int x, int off) __attribute__((always_inline)) { return *(LDS_AS const frag*)(uintptr_t)(yl[x] + off); };
  auto y_trans = [&](int c, int d, int off) __attribute__((always_inline)) {
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(uintptr_t)(yt[2 * d] + off + 2048 * c));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(uintptr_t)(yt[2 * d + 1] + off + 2048 * c + 1024));
    return __builtin_bit_cast(frag, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  // probabilities and score gradients of a step from its scores (minus log-sum-exp, base 2) and dP - Delta; the entries past
  // the end of the sequence, or past the diagonal of a causal call, are zero.  One branch per step.
  auto gradients = [&](f32x16& s, f32x16& dp, int y0, bool edge) __attribute__((always_inline)) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      s[v] = __builtin_amdgcn_exp2f(s[v]);
      dp[v] *= s[v];
    }
    if (edge) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int yr = y0 + 8 * (v >> 2) + 4 * g + 3 - (v & 3);
        const bool ok = x_ok && yr < Lb && (!p.causal || (kDQ ? yr <= xr : xr <= yr));
        s[v] = ok ? s[v] : 0.f;
        dp[v] = ok ? dp[v] : 0.f;
      }
    }
  };
  // dX^T += Y1^T dS, dV^T += dO^T P: the loop rows are the accumulators' registers.  The transposed operands are asked for
  // well ahead of their use.
  struct Trans {
    frag y1[2][DBLKS], y2[kDQ ? 1 : 2][DBLKS];
  };
  auto request_trans = [&](Trans& t, int off) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int d = 0; d < DBLKS; ++d) {
        t.y1[c][d] = y_trans(c, d, off);
        if constexpr (!kDQ) t.y2[c][d] = y_trans(c, d, off + 2 * kTile);
      }
  };
  auto outputs = [&](const f32x16& pr, const frag (&dsf)[2], const Trans& t) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int d = 0; d < DBLKS; ++d) acc1[d] = QT::mma(t.y1[c][d], dsf[c], acc1[d]);
      if constexpr (!kDQ) {
        f32x8 p8;
#pragma unroll
        for (int e = 0; e < 8; ++e) p8[e] = pr[8 * c + e];
        const frag pf = QT::from_f32(p8);
#pragma unroll
        for (int d = 0; d < DBLKS; ++d) acc2[d] = QT::mma(t.y2[c][d], pf, acc2[d]);
      }
    }
  };
  auto pack = [&](const f32x16& ds, frag (&dsf)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      f32x8 d8;
#pragma unroll
      for (int e = 0; e < 8; ++e) d8[e] = ds[8 * c + e];
      dsf[c] = QT::from_f32(d8);
    }
  };
  // -Delta of the loop rows (dK/dV role: one per register) or of this lane's row
  auto start_stat = [&](int which, int buf) __attribute__((always_inline)) {
    f32x16 r;
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const f32x4 s4 = *(LDS_AS const f32x4*)(uintptr_t)(lds0 + kOffStat + (uint32_t)((buf * 2 + which) * kStep * 4) + (8 * q4 + 4 * g) * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) r[4 * q4 + e] = s4[e];
    }
    return r;
  };
  auto splat = [&](float x) __attribute__((always_inline)) {
    f32x16 r;
#pragma unroll
    for (int v = 0; v < 16; ++v) r[v] = x;
    return r;
  };
  const f32x16 del16 = splat(del_x);

  // ---- far steps ---------------------------------------------------------------------------------------------------------
  // The buffer of a step's tiles is its distance from the first near step, modulo two, in every zone.
  auto buf_of = [&](int s) __attribute__((always_inline)) { return (s - z.s0) & 1; };
  if (z.lo < z.hi) tiles_dma(z.lo, buf_of(z.lo));
  auto far_range = [&](int from, int to, int side) __attribute__((always_inline)) {
    if (from >= to) return;
    // side 0: r' >= R, side 1: r' <= -R.  The lane operand takes the loop side's table row and the soft-max scale; the lane row's
    // own score is a constant of the row.
    const int delta = p.lut[(side == 0) == kDQ ? 2 * p.R : 0];
    float a = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const f32x8 x8 = QT::to_f32(load_x1(s));
      const f32x8 tx = QT::to_f32(QT::load(txb + (int64_t)delta * tx_rowb + (16 * s + 8 * g) * 2));
#pragma unroll
      for (int e = 0; e < 8; ++e) a = __builtin_fmaf(tx[e], x8[e], a);
      x1[s] = QT::from_f32((x8 + QT::to_f32(QT::load(tyb + (int64_t)delta * ty_rowb + (16 * s + 8 * g) * 2))) * x_scale);
    }
    a = wave_half_sum(a) * x_scale;
    const float start = a + lse_x;
    const f32x16 start16 = splat(start);
#pragma unroll
    for (int s = 0; s < KS; ++s) asm volatile("" ::"v"(x1[s]));
    float sum = 0.f;
#pragma unroll 1
    for (int s = from; s < to; ++s) {
      const int buf = buf_of(s), off = buf * kTile, y0 = s * kStep;
      wait_vmcnt<0>();
      __syncthreads();
      if (s + 1 < z.hi) tiles_dma(s + 1, buf ^ 1);
      f32x16 sacc, dpacc;
      frag yf[KS], zf[KS];   // every operand of the eight products is requested before the first of them waits for one
      if constexpr (!kDQ) {
        sacc = start_stat(0, buf);
        dpacc = start_stat(1, buf);
      }
#pragma unroll
      for (int x = 0; x < KS; ++x) {
        yf[x] = y_frag(x, off);
        zf[x] = y_frag(x, off + 2 * kTile);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!kDQ) {
#pragma unroll
        for (int v = 0; v < 16; ++v) sacc[v] += start;
      }
#pragma unroll
      for (int x = 0; x < KS; ++x) {
        sacc = QT::mma(yf[x], x1[x], kDQ && x == 0 ? start16 : sacc);
        dpacc = QT::mma(zf[x], x2[x], kDQ && x == 0 ? del16 : dpacc);
      }
      Trans tr;
      request_trans(tr, off);
      __builtin_amdgcn_sched_barrier(0);
      const bool edge = xw0 + 31 >= Lb || y0 + kStep > Lb || (p.causal && (kDQ ? y0 + kStep - 1 > xw0 : xw0 + 31 > y0));
      gradients(sacc, dpacc, y0, edge);
      frag dsf[2];
      pack(dpacc, dsf);
      sum += (((dpacc[0] + dpacc[1]) + (dpacc[2] + dpacc[3])) + ((dpacc[4] + dpacc[5]) + (dpacc[6] + dpacc[7]))) +
             (((dpacc[8] + dpacc[9]) + (dpacc[10] + dpacc[11])) + ((dpacc[12] + dpacc[13]) + (dpacc[14] + dpacc[15])));
      outputs(sacc, dsf, tr);
    }
    far_sum[side] = sum;
  };
  far_range(z.lo, z.s0, 0);

  // ---- near steps ----------------------------------------------------------------------------------------------------------
  if (n_near > 0) {
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      x1[s] = QT::from_f32(QT::to_f32(load_x1(s)) * x_scale);
      asm volatile("" ::"v"(x1[s]));
    }
    const f32x16 lse16 = splat(lse_x);
    const int arow = 31 - li;
    uint32_t ra[KS];
#pragma unroll
    for (int x = 0; x < KS; ++x) ra[x] = lds0 + kOffX + (uint32_t)(arow * kRowBytes) + (uint32_t)(((g ^ swz(arow)) * 16) ^ (32 * x));
    // Transposed operand of a ring batch: contraction index c = 16 s + 8 g + e counts relative positions upwards, i.e. batch row
    // 31 - c; each source lane of the transposing read names its own row, so the reversal costs nothing.
    uint32_t et[4];
    {
      const int s16 = lane & 15, grp = lane >> 4;
#pragma unroll
      for (int x = 0; x < 4; ++x) {  // x = 2 d + half of the eight
        const int row = 15 - (8 * (grp >> 1) + 4 * (x & 1) + (s16 >> 2)), chunk = 4 * (x >> 1) + 2 * (grp & 1) + ((s16 & 3) >> 1);
        et[x] = lds0 + kOffX + (uint32_t)(row * kRowBytes + (chunk ^ swz(row)) * 16 + (s16 & 1) * 8);
      }
    }
    const uint32_t scr0 = lds0 + kOffScr + (uint32_t)wave * (kScrElems * 2) + (uint32_t)li * (kScrPitch * 2);
    const uint32_t c_wr = scr0 + 8u * g, c_dup = scr0 + (g == 0 ? 128u : 8u);
    uint32_t c_rd[2][4];
#pragma unroll
    for (int par = 0; par < 2; ++par)
#pragma unroll
      for (int q = 0; q < 4; ++q) c_rd[par][q] = scr0 + 2u * (uint32_t)((32 * par + li + 29 - 8 * q - 4 * g) & 63);
    const uint32_t g_rd = scr0 + 16u * g;
    const int xl = li + 4 * g;
    // columns 0 .. n-1 of half 0 lie in the repeated columns where this row's run of four wrapped there (n = 0 .. 3)
    const uint32_t n_dup = g == 0 ? (uint32_t)((li + 1) & 3) : 0u;
    const uint32_t dup_m0 = n_dup >= 2 ? 0xffffffffu : n_dup == 1 ? 0xffffu : 0u, dup_m1 = n_dup == 3 ? 0xffffu : 0u;
    frag ax[KS], ay[2][KS];
    auto x_read = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
      for (int x = 0; x < KS; ++x) ax[x] = *(LDS_AS const frag*)(uintptr_t)(ra[x] + (uint32_t)slot * kTile);
    };
    auto y_read = [&](int buf, int slot) __attribute__((always_inline)) {
#pragma unroll
      for (int x = 0; x < KS; ++x) ay[buf][x] = *(LDS_AS const frag*)(uintptr_t)(ra[x] + (kOffY - kOffX) + (uint32_t)slot * kTile);
    };
    typedef typename QT::scratch4 s4t;
    auto c_store = [&](const f32x16& c, int half) __attribute__((always_inline)) {
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const s4t packed = QT::pack4(f32x4{c[4 * q4], c[4 * q4 + 1], c[4 * q4 + 2], c[4 * q4 + 3]});
        *(LDS_AS s4t*)(uintptr_t)(c_wr + 64 * half + 16 * q4) = packed;
        if (half == 0 && q4 == 0) *(LDS_AS s4t*)(uintptr_t)c_dup = packed;
      }
    };
    // a completed block of score gradients: this row's 32 relative positions as the two operands of a contraction over them
    auto g_load = [&](int half, frag (&gf)[2]) __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        u32x2 lo = *(LDS_AS const u32x2*)(uintptr_t)(g_rd + 64 * half + 32 * s);
        const u32x2 hi = *(LDS_AS const u32x2*)(uintptr_t)(g_rd + 64 * half + 32 * s + 8);
        if (half == 0 && s == 0) {
          const u32x2 du = *(LDS_AS const u32x2*)(uintptr_t)(scr0 + 128);
          lo[0] = (lo[0] & ~dup_m0) | (du[0] & dup_m0);
          lo[1] = (lo[1] & ~dup_m1) | (du[1] & dup_m1);
        }
        gf[s] = __builtin_bit_cast(frag, u32x4{lo[0], lo[1], hi[0], hi[1]});
      }
    };
    // Block of relative positions rho = (xw0 / 32) - s, s the step it is the upper block of: its slot in memory
    char* g_out = nullptr;
    if (kDQ) g_out = p.g_blocks + (((int64_t)b * p.H + h) * p.g_rows + (xw0 >> 5)) * (int64_t)p.g_slots * 2048 + li * 64 + g * 16;
    auto g_use = [&](const frag (&gf)[2], int xslot, int k) __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int d = 0; d < DBLKS; ++d) {
          const uint32_t at = (uint32_t)xslot * kTile + (s == 0 ? 2048u : 0u);
          const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(uintptr_t)(et[2 * d] + at));
          const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(uintptr_t)(et[2 * d + 1] + at));
          acc1[d] = QT::mma(__builtin_bit_cast(frag, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)), gf[s], acc1[d]);
        }
        if constexpr (kDQ) *(u32x4*)(g_out + (int64_t)k * 2048 + 32 * s) = frag_bits(gf[s]);
      }
    };
    // ring slots: batch n of the lane side's table in slot n % 6, of the loop side's in n % 5.  Wave w's block bk at step k is
    // batch k + 4 - w - bk.
    int xs_new = 4 - wave, ys_new = 4 - wave, xs_dma = 5, ys_dma = 0;
    int dnext;
    r_tab = m0 + FDB_BM - 1 - z.s0 * kStep - srow;
    {
      int d0[6];
#pragma unroll
      for (int bt = 0; bt < 6; ++bt) d0[bt] = batch_delta();
#pragma unroll
      for (int bt = 0; bt < 6; ++bt) asm volatile("" : "+v"(d0[bt]));
#pragma unroll
      for (int bt = 0; bt < 5; ++bt) batch_dma(d0[bt], bt, bt);
      dnext = d0[5];
      wait_vmcnt<0>();
      __syncthreads();
      x_read(3 - wave);   // block 1 of step 0
      y_read(1, 3 - wave);
      f32x16 c1;
#pragma unroll
      for (int x = 0; x < KS; ++x) c1 = QT::mma(ax[x], x1[x], x == 0 ? zero : c1);
      // its entries beyond this row's own position belong to loop rows before the first near step: no score gradient comes to them
#pragma unroll
      for (int v = 0; v < 16; ++v) c1[v] = 8 * (v >> 2) + 4 * g + (v & 3) > li ? 0.f : c1[v];
      c_store(c1, 1);
    }
    auto step = [&](auto par_tag, int k) __attribute__((always_inline)) {
      constexpr int PAR = decltype(par_tag)::value;
      constexpr int OFF = PAR * kTile;
      const int s = z.s0 + k, y0 = s * kStep;
      wait_vmcnt<kDQ ? 2 : 0>();   // the loads of the step before; the two stores of G after them may still be on their way
      asm volatile("" : "+v"(dnext));
      __syncthreads();
      tiles_dma(s + 1, PAR ^ 1);
      batch_dma(dnext, xs_dma, ys_dma);  // batch k + 5
      __builtin_amdgcn_sched_barrier(0);
      dnext = batch_delta();
      frag yf[KS];
#pragma unroll
      for (int x = 0; x < KS; ++x) yf[x] = y_frag(x, OFF);
      x_read(xs_new);
      f32x16 sacc, cnew, pacc[2], dpacc;
      if constexpr (kDQ) sacc = lse16;
      else sacc = start_stat(0, PAR);
      y_read(PAR, ys_new);
#pragma unroll
      for (int x = 0; x < KS; ++x) {
        cnew = QT::mma(ax[x], x1[x], x == 0 ? zero : cnew);
        sacc = QT::mma(yf[x], x1[x], sacc);
      }
#pragma unroll
      for (int x = 0; x < KS; ++x) {
        pacc[1] = QT::mma(yf[x], ay[PAR ^ 1][x], x == 0 ? zero : pacc[1]);
        pacc[0] = QT::mma(yf[x], ay[PAR][x], x == 0 ? zero : pacc[0]);
      }
      float cband[16];
      c_store(cnew, PAR);
      wave_lds_fence();
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        cband[4 * q + 0] = lds_elem_f32<QT, 0>(c_rd[PAR][q]);
        cband[4 * q + 1] = lds_elem_f32<QT, 2>(c_rd[PAR][q]);
        cband[4 * q + 2] = lds_elem_f32<QT, 4>(c_rd[PAR][q]);
        cband[4 * q + 3] = lds_elem_f32<QT, 6>(c_rd[PAR][q]);
      }
      wave_lds_fence();
      float px[16];
      {
        float xs[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int c = 8 * (v >> 2) + 3 - (v & 3);
          xs[v] = (xl < 32 - c) ? pacc[1][v] : pacc[0][v];
        }
        if (g == 0)
          rotate16<32>(xs, px, std::make_integer_sequence<int, 16>{});
        else
          rotate16<28>(xs, px, std::make_integer_sequence<int, 16>{});
      }
      // dP - Delta while the band and the rotated values are on their way
      if constexpr (kDQ) dpacc = del16;
      else dpacc = start_stat(1, PAR);
#pragma unroll
      for (int x = 0; x < KS; ++x) dpacc = QT::mma(y_frag(x, OFF + 2 * kTile), x2[x], dpacc);
      __builtin_amdgcn_sched_barrier(0);
      lds_wait_all();
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        if constexpr (std::is_same<QT, Bf16Tr>::value) asm volatile("" : "+v"(cband[v]));
        asm volatile("" : "+v"(px[v]));
      }
#pragma unroll
      for (int v = 0; v < 16; ++v) sacc[v] = __builtin_fmaf(px[v], x_scale, sacc[v] + cband[v]);
      const bool edge = xw0 + 31 >= Lb || y0 + kStep > Lb || (p.causal && (kDQ ? y0 + kStep - 1 > xw0 : xw0 + 31 > y0));
      Trans tr;
      request_trans(tr, OFF);
      __builtin_amdgcn_sched_barrier(0);
      gradients(sacc, dpacc, y0, edge);
      // The saturated rows of a table's gradient come from the sums per lane row alone (far steps and these few elements),
      // the rows inside the radius from the blocks of G: where the two roles' far steps begin does not matter then.
      if (xw0 + 31 - y0 >= p.R || xw0 - y0 - 31 <= -p.R) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int r = xr - (y0 + 8 * (v >> 2) + 4 * g + 3 - (v & 3));
          edge_sum[0] += r >= p.R ? dpacc[v] : 0.f;
          edge_sum[1] += r <= -p.R ? dpacc[v] : 0.f;
        }
      }
      frag dsf[2];
      pack(dpacc, dsf);
      // the score gradients take the place of the scores they belong to
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const u32x4 w = frag_bits(dsf[c]);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const uint32_t at = c_rd[PAR][2 * c + q];
          lds_put_lo<0>(at, w[2 * q]);
          lds_put_hi<2>(at, w[2 * q]);
          lds_put_lo<4>(at, w[2 * q + 1]);
          lds_put_hi<6>(at, w[2 * q + 1]);
        }
      }
      wave_lds_fence();
      outputs(sacc, dsf, tr);
      frag gf[2];
      g_load(PAR ^ 1, gf);
      g_use(gf, xs_new == 0 ? kXBatches - 1 : xs_new - 1, k);
      xs_new = xs_new == kXBatches - 1 ? 0 : xs_new + 1;
      ys_new = ys_new == kYBatches - 1 ? 0 : ys_new + 1;
      xs_dma = xs_dma == kXBatches - 1 ? 0 : xs_dma + 1;
      ys_dma = ys_dma == kYBatches - 1 ? 0 : ys_dma + 1;
    };
    using T0 = std::integral_constant<int, 0>;
    using T1 = std::integral_constant<int, 1>;
    int k = 0;
#pragma unroll 1
    for (; k + 1 < n_near; k += 2) {
      step(T0{}, k);
      step(T1{}, k + 1);
    }
    if (k < n_near) step(T0{}, k);
    // the lower block of the last step: complete but for the loop rows that follow the near range, to which no gradient came
    {
      frag gf[2];
      const int half = (n_near - 1) & 1;
      if (half == 0) g_load(0, gf);   // never wrapped here: the columns a run wraps into are cleared below
      else g_load(1, gf);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        u32x4 w = frag_bits(gf[s]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int col = 16 * s + 8 * g + 2 * e;
          w[e] = col > li ? w[e] : col + 1 > li ? (w[e] & 0xffff0000u) : 0u;
        }
        gf[s] = __builtin_bit_cast(frag, w);
      }
      g_use(gf, xs_new == 0 ? kXBatches - 1 : xs_new - 1, n_near);
    }
  }
  far_range(z.s1, z.hi, 1);
  wait_vmcnt<0>();

  // ---- epilogue ---------------------------------------------------------------------------------------------------------------
  const float far0 = wave_half_sum(far_sum[0]), far1 = wave_half_sum(far_sum[1]);
  const float sat0 = far0 + wave_half_sum(edge_sum[0]), sat1 = far1 + wave_half_sum(edge_sum[1]);
  if (!x_ok) return;
  {
    // the far steps' way back through the table: two rows of it
    const int d0 = p.lut[kDQ ? 2 * p.R : 0], d1 = p.lut[kDQ ? 0 : 2 * p.R];
    const char* t0 = txb + (int64_t)d0 * tx_rowb;
    const char* t1 = txb + (int64_t)d1 * tx_rowb;
#pragma unroll
    for (int d = 0; d < DBLKS; ++d)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int off = (32 * d + 8 * q4 + 4 * g) * 2;
        const f32x4 r0 = QT::load4(t0 + off), r1 = QT::load4(t1 + off);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc1[d][4 * q4 + e] = (acc1[d][4 * q4 + e] + far0 * r0[e] + far1 * r1[e]) * p.sm_scale;
      }
    if (g == 0) {
      // ... and what the tables' saturated rows take from this row, [delta(+R), delta(-R)]: sums over a whole sequence and without
      // the soft-max scale, which in fp16 would leave its range long before the gradients made of them do
      float* fs = (kDQ ? p.far_q : p.far_k) + ((int64_t)b * p.H + h) * 2 * p.stat_len + xr;
      fs[0] = kDQ ? sat0 : sat1;
      fs[p.stat_len] = kDQ ? sat1 : sat0;
    }
  }
  auto write = [&](char* ptr, int64_t sb, int64_t st, int64_t sh, const f32x16 (&acc)[DBLKS]) {
    char* row = ptr + (b * sb + (int64_t)(tok0 + xr) * st + (int64_t)h * sh) * 2;
#pragma unroll
    for (int d = 0; d < DBLKS; ++d)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        QT::store4(row + (32 * d + 8 * q4 + 4 * g) * 2, acc[d][4 * q4], acc[d][4 * q4 + 1], acc[d][4 * q4 + 2], acc[d][4 * q4 + 3]);
  };
  if (kDQ) {
    write(p.dq, p.dq_sb, p.dq_st, p.dq_sh, acc1);
  } else {
    write(p.dk, p.dk_sb, p.dk_st, p.dk_sh, acc1);
    write(p.dv, p.dv_sb, p.dv_st, p.dv_sh, acc2);
  }
}

template <class QT, int ROLE, bool BY_LENGTH>
__global__ __launch_bounds__(kThreads, 2) void fdb_bwd_ring_kernel(const FdbBwdRingParams p) {
  const int wg = (int)blockIdx.x;
  bwd_ring<QT, ROLE, false, BY_LENGTH>(p, wg, BY_LENGTH ? p.places + (ROLE == 0 ? wg : (int)gridDim.x + wg) : nullptr);
}

// Both roles as one launch, the longer one's workgroups first: 2 x 288 workgroups, say, leave half of the GPU's 512 places empty
// as two launches and fill them as one.
template <class QT, bool BY_LENGTH>
__global__ __launch_bounds__(kThreads, 2) void fdb_bwd_both_kernel(const FdbBwdRingParams p) {
  const int wg = (int)blockIdx.x;
  if constexpr (BY_LENGTH) {
    const FdbPlace* at = p.places + wg;
    if (at->keys) bwd_ring<QT, 1, true, true>(p, at->n, at);
    else bwd_ring<QT, 0, true, true>(p, at->n, at);
  } else {
    const int n = (int)(gridDim.x >> 1);
    if (wg < n) bwd_ring<QT, 1, true, false>(p, wg, nullptr);
    else bwd_ring<QT, 0, true, false>(p, wg - n, nullptr);
  }
}

// The places of both roles' workgroups of a padded batch (fdb_deals_by_length), batch rows x 2 of them by this workgroup, the `at`-th of tiles * heads.  The order
// is padded_map's, or block_map's where the mask hides little.  together: one launch, the roles take turns of 32, the short texts of both end it; otherwise dQ's
// places, then the others.  Turns of 8, 16, 32 and 64 and of a tile's heads, 40 ragged batches of 128 to 2048 tokens, the mean of the backward's times: 1.009, 1.010, 1, 1.002
// and 1.005 (2 x 2048 5 % longer by 8 and 16; the training layer of 8 x 512 1 % shorter by 8 or 16, 1 % longer by 64).
// A table, because the roles have no registers to spare: with padded_map at its start the dQ role spilt 19 instead of 14 and took 705 us instead of 640 (8 x 3000).
__device__ __forceinline__ void find_places(const FdbBwdRingParams& p, int at, bool together) {
  __shared__ int first[64], tokens[64], sorted[64], row[64], dealt;
  const int tid = (int)threadIdx.x, batch = p.B, heads = p.H, all = p.tiles * heads * batch;
  if (tid < 64) {
    int tok0 = 0, mine = 0;
    if (tid < batch) {
      if (p.seq_start) tok0 = min(max(p.seq_start[tid], 0), p.L);
      mine = min(max(p.seq_len[tid], 0), p.L - tok0);
    }
    const bool deals = padded_batch_deals(mine, batch, p.L, tid);
    const int blocks = tid < batch ? (mine + 31) >> 5 : -1;
    int rank = 0;
    for (int x = 0; x < batch; ++x) {
      const int other = __builtin_amdgcn_readlane(blocks, x);
      rank += other > blocks || (other == blocks && x < tid) ? 1 : 0;
    }
    first[tid] = tok0, tokens[tid] = mine;
    if (tid < batch) sorted[rank] = blocks, row[rank] = tid;
    if (tid == 0) dealt = deals;
  }
  __syncthreads();
  const int n = at * batch + tid;
  if (tid >= batch || n >= all) return;
  auto put = [&](int slot, int b, int t, int h, bool keys) {
    p.places[slot] = FdbPlace{b, t, h, first[b], tokens[b], n, keys ? 1 : 0, 0};
  };
  if (!dealt) {
#pragma unroll
    for (int keys = 0; keys < 2; ++keys) {
      int b, t, h;
      block_place(n, batch, heads, p.tiles, p.groups_together, order_of(p, keys == 0), b, t, h);
      put(together == (keys != 0) ? n : all + n, b, t, h, keys != 0);
    }
    return;
  }
  const int unit = 32, part = n / unit, at_unit = n - part * unit, in_part = min(unit, all - part * unit);
  const int slot_keys = together ? 2 * part * unit + at_unit : all + n, slot_dq = together ? slot_keys + in_part : n;
  int real = 0;
  for (int x = 0; x < batch; ++x) real += (sorted[x] + FDB_BM / 32 - 1) / (FDB_BM / 32);
  int u = n < real * heads ? n : ~(n - real * heads);
  if (u >= 0 && !p.causal) {
    int ahead = 0, here = 0, of_class = p.tiles;
    for (;; --of_class) {   // `here` sequences of that many tiles
      for (here = 0; ahead + here < batch && sorted[ahead + here] > (of_class - 1) * (FDB_BM / 32);) ++here;
      if (u < here * of_class * heads) break;
      u -= here * of_class * heads;
      ahead += here;
    }
#pragma unroll
    for (int keys = 0; keys < 2; ++keys) {
      int x, t, h;
      block_place(u, here, heads, of_class, groups_of(of_class), order_of(p, keys == 0), x, t, h);
      put(keys ? slot_keys : slot_dq, row[ahead + x], t, h, keys != 0);
    }
    return;
  }
  const bool padding = u < 0;
  if (padding) u = ~u;
  const int pair = u / heads, h = u - pair * heads;
  u = pair;
  int t, here = padding ? batch : 0;
  for (t = padding ? 0 : p.tiles - 1;; t += padding ? 1 : -1) {
    if (padding) {
      while (here > 0 && sorted[here - 1] <= t * (FDB_BM / 32)) --here;
      if (u < batch - here) break;
      u -= batch - here;
    } else {
      while (here < batch && sorted[here] > t * (FDB_BM / 32)) ++here;
      if (u < here) break;
      u -= here;
    }
  }
  if (padding) u += here;
  // Causal: the queries of a key tile are those from its own to the end of the text, as many as the mirrored query tile has keys.  Backward, highest key tile first ->
  // mirrored (the plain order): 8 x 1024 192 -> 170 us (175), 8 x 2048 328 -> 290 (330), 4 x 4096 with 16 heads 715 -> 613 (641), 48 x 384 204 -> 210 (223).
  put(slot_keys, row[u], padding ? t : (sorted[u] - 1) / (FDB_BM / 32) - t, h, true);
  put(slot_dq, row[u], t, h, false);
}

// The row statistics by themselves: -lse in base 2 and -Delta = -(dO . O), 128 rows a workgroup, two lanes a row that add up in the dQ
// role's order, so that a batch row's gradients have the same bits whichever way it is launched.  Bound by reading dO and O.
// PLACES: with the workgroups' places, the first layer of the grid (the only one: those alone).
template <class QT, bool PLACES>
__global__ __launch_bounds__(256) void fdb_row_stats_kernel(const FdbBwdRingParams p) {
  if constexpr (PLACES)
    if (blockIdx.z == 0) {
      find_places(p, (int)(blockIdx.y * gridDim.x + blockIdx.x), gridDim.z > 1);
      return;
    }
  const int b = (int)blockIdx.z - (PLACES ? 1 : 0), h = (int)blockIdx.y, g = threadIdx.x & 1, row = (int)blockIdx.x * 128 + (int)(threadIdx.x >> 1);
  const int tok0 = p.seq_start ? min(max(p.seq_start[b], 0), p.L) : 0;
  const int Lb = p.seq_len ? min(max(p.seq_len[b], 0), p.L - tok0) : p.L;
  if (row >= Lb) return;   // a row's two lanes leave together
  const int64_t tok = (int64_t)tok0 + row;
  const char* orow = p.out + ((int64_t)b * p.o_sb + tok * p.o_st + (int64_t)h * p.o_sh + 8 * g) * 2;
  const char* grow = p.dout + ((int64_t)b * p.g_sb + tok * p.g_st + (int64_t)h * p.g_sh + 8 * g) * 2;
  typename QT::frag o[4], d[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    o[s] = QT::load(orow + 32 * s);
    d[s] = QT::load(grow + 32 * s);
  }
  const float lse = p.lse[((int64_t)b * p.L + tok) * p.H + h];
  float dot = 0.f;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const f32x8 o8 = QT::to_f32(o[s]), g8 = QT::to_f32(d[s]);
#pragma unroll
    for (int e = 0; e < 8; ++e) dot = __builtin_fmaf(o8[e], g8[e], dot);
  }
  dot += __shfl_xor(dot, 1);
  if (g == 0) {
    const int64_t at = ((int64_t)b * p.H + h) * p.stat_len + row;
    p.neg_lse[at] = lse * -1.4426950408889634f;
    p.neg_delta[at] = -dot;
  }
}

// ---- gradients of the tables ----------------------------------------------------------------------------------------------
// dE_K[r] = sum_i G[i][r] q_i and dE_Q[r] = sum_i G[i][r] k_(i-r) for blocks of 32 relative positions r = 32 rho + c, from the blocks
// [32 i x 32 c] of G the dQ launch stored.  A workgroup is four waves with four neighbouring rho of one head; it walks row blocks I
// (of its share of the batch), whose rows of q all four use, while the rows of k (row block I - 1 - rho) form a ring the waves
// read at different places.  dE_Q wants, for key row j and position c, the entry of row j + r: a diagonal through the blocks I - 1
// and I, picked element by element (sixteen 2-byte LDS reads per lane); everything else is transposing reads and MFMAs, 64 fp32
// sums per lane kept for the life of the workgroup.  Bound by the reading of G: 1 GB at B = 8, L = 4096, 12 heads.
// The last group of a head collects the saturated rows' sums per token: two rows (delta(+R), delta(-R)) of each table, weights per token.
// A wave issues about one instruction per 4.5 clocks and a row block is only eight MFMAs (a third of two waves' turn), so the loop is
// written for few instructions: it is unrolled over the four ring slots of G, which makes every LDS address a lane constant plus an
// immediate; what 32 turns need to know of G's blocks (which there are, where they lie) is worked out at once, a row block per lane, and
// is then one bit and one value read from a lane; rows are clamped in vector registers, without a branch.  190 -> 118 instructions a turn, of
// which 90 scalar ones were found to be more than half of what the waves issued (and 89 -> 16 scalar registers spilled to lanes):
// 12 heads, us, 8 x 512 padded 25.3 -> 19.4, 2 x 1501 31.8 -> 26.6, 8 x 4096 270 -> 260.  Loads run two row blocks ahead.  No faster: eight
// waves, half of them for either table, which doubles the scalar instructions (25.3 -> 26.5), and the operands asked for ahead of the next loads.
// A launch without divisions and scalar loads ahead of each sequence: 19.4 -> 17.4 and 26.6 -> 25.8.  The
// groups in rising order with the saturated rows' last: falling, with those first, the backward of 2 x 1501 takes 195 us where this takes 190.5.  What is left beside the turns (0.33 us
// for two workgroups of a CU) is the writing of the shares' sums, 25 MB of them.
constexpr int kGBlk = 2048, kGRing = 4, kKRing = 8;
constexpr int kTgOffK = kGRing * kTile, kTgOffG = kTgOffK + kKRing * kTile, kTgLds = kTgOffG + 4 * kGRing * kGBlk;
static_assert(kTgLds <= 80 * 1024, "two workgroups per CU");
static_assert(kTgOffG % (kGRing * kGBlk) == 0, "a wave's ring of G wraps by a mask of its address");

// BY_LENGTH (a padded batch of up to 64 sequences): a part takes an equal share of the row blocks that hold tokens, wherever in a sequence that
// begins and ends, instead of chunks of the batch's rows, of which one part may have twice as many with tokens as another (8 x 512, lengths of 148 to
// 512, 28 row blocks in the longest of four parts: 26.2 -> 25.3 us with what follows as it was).
template <class QT, bool BY_LENGTH>
__global__ __launch_bounds__(kThreads, 2) void fdb_table_grad_kernel(const FdbBwdRingParams p) {
  using frag = typename QT::frag;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LDS_AS char*)smem;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, li = lane & 31, g = lane >> 5;
  const int h = (int)blockIdx.x, part = (int)blockIdx.y, group = (int)blockIdx.z;  // the saturated rows last
  // this part's items: (batch row, chunk of row blocks), as many as any other's
  int it0 = part * p.tg_items, it1 = it0 + p.tg_items;
  int first = 0, len = 0, before = 0, lo = 0, hi = 0;   // BY_LENGTH: this lane's sequence and the row blocks ahead of it; this part's of all
  if constexpr (BY_LENGTH) {
    if (lane < p.B) {
      if (p.seq_start) first = min(max(p.seq_start[lane], 0), p.L);
      len = min(max(p.seq_len[lane], 0), p.L - first);
    }
    const int blocks = (len + 31) / 32;
    before = blocks;
#pragma unroll
    for (int x = 1; x < 64; x <<= 1) {
      const int other = __shfl_up(before, x);
      before += lane >= x ? other : 0;
    }
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane(before, 63), share = (total + (uint32_t)p.tg_parts - 1) / (uint32_t)p.tg_parts;
    lo = (int)min(total, share * (uint32_t)part), hi = (int)min(total, lo + share);
    it0 = __popcll(__ballot(lane < p.B && before <= lo));   // sequences that end ahead of it
    before -= blocks;
    it1 = __popcll(__ballot(lane < p.B && before < hi));
  }
  // the row blocks [I0, I1) of sequence b that are the item's
  auto item = [&](int it, int n_rows, int& I0, int& I1) __attribute__((always_inline)) {
    if constexpr (BY_LENGTH) {
      const int ahead = __builtin_amdgcn_readlane(before, it);
      I0 = max(0, lo - ahead), I1 = min(n_rows, hi - ahead);
    } else {
      I0 = (int)((uint32_t)it % (uint32_t)p.tg_chunks) * p.tg_len, I1 = min(n_rows, I0 + p.tg_len);
    }
  };
  auto seq_of = [&](int b, int& tok0, int& Lb) __attribute__((always_inline)) {
    if constexpr (BY_LENGTH) {
      tok0 = __builtin_amdgcn_readlane(first, b), Lb = __builtin_amdgcn_readlane(len, b);
    } else {
      tok0 = p.seq_start ? min(max(p.seq_start[b], 0), p.L) : 0;
      Lb = p.seq_len ? min(max(p.seq_len[b], 0), p.L - tok0) : p.L;
    }
  };
  if (group == p.tg_groups) {
    // the saturated rows: a wave takes eight rows at a time, sixteen bytes of a row per lane
    f32x8 acc[2][2];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t >> 1][t & 1] = f32x8{0, 0, 0, 0, 0, 0, 0, 0};
    const int r8 = lane >> 3, c8 = lane & 7;
    for (int it = it0; it < it1; ++it) {
      const int b = BY_LENGTH ? it : (int)((uint32_t)it / (uint32_t)p.tg_chunks);
      int tok0, Lb, I0, I1;
      seq_of(b, tok0, Lb);
      item(it, (Lb + 31) / 32, I0, I1);
      const int i1 = min(Lb, I1 * 32);
      const char* qr = p.q + ((int64_t)b * p.q_sb + (int64_t)tok0 * p.q_st + (int64_t)h * p.q_sh + 8 * c8) * 2;
      const char* kr = p.k + ((int64_t)b * p.k_sb + (int64_t)tok0 * p.k_st + (int64_t)h * p.k_sh + 8 * c8) * 2;
      const float* fq = p.far_q + ((int64_t)b * p.H + h) * 2 * p.stat_len;
      const float* fk = p.far_k + ((int64_t)b * p.H + h) * 2 * p.stat_len;
#pragma unroll 4
      for (int i = I0 * 32 + 8 * wave + r8; i < i1; i += 32) {
        const f32x8 q = QT::to_f32(QT::load(qr + (int64_t)i * p.q_st * 2)), k = QT::to_f32(QT::load(kr + (int64_t)i * p.k_st * 2));
        acc[0][0] += fq[i] * q;
        acc[0][1] += fq[p.stat_len + i] * q;
        acc[1][0] += fk[i] * k;
        acc[1][1] += fk[p.stat_len + i] * k;
      }
    }
    float* s = (float*)smem;   // [32 row classes][4][64]
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int e = 0; e < 8; ++e) s[((8 * wave + r8) * 4 + t) * 64 + 8 * c8 + e] = acc[t >> 1][t & 1][e];
    __syncthreads();
    float sum = 0.f;
    for (int r = 0; r < 32; ++r) sum += s[r * 256 + tid];   // tid = (table, side, d)
    p.far_parts[((int64_t)part * p.H + h) * 256 + tid] = sum;
    return;
  }
  const int rho = p.rho_min + 4 * group + wave;
  f32x16 ek[2], eq[2];
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int v = 0; v < 16; ++v) ek[d][v] = eq[d][v] = 0.f;
  const int srow = tid >> 3, scc = tid & 7;
  const uint32_t chunk_off = (uint32_t)((scc ^ swz(srow)) * 16), wave_kb = lds0 + (uint32_t)wave * 1024u;
  uint32_t yt[4], gt[2];
  const int s16 = lane & 15, grp = lane >> 4;
  {
    const int slotl = (2 * (grp & 1) + ((s16 & 3) >> 1)) ^ (4 * ((s16 >> 3) & 1)) ^ (grp >> 1);
    const uint32_t vlane = (4 * (grp >> 1) + (s16 >> 2)) * kRowBytes + slotl * 16 + (s16 & 1) * 8;
#pragma unroll
    for (int x = 0; x < 4; ++x) yt[x] = lds0 + (vlane ^ (64 * (x >> 1) ^ 32 * (x & 1)));
    // G: rows of 64 bytes, two halves of eight contraction rows
#pragma unroll
    for (int x = 0; x < 2; ++x) gt[x] = (uint32_t)((8 * x + 4 * (grp >> 1) + (s16 >> 2)) * 64 + (16 * (grp & 1) + 4 * (s16 & 3)) * 2);
  }
  const uint32_t g_base = lds0 + kTgOffG + (uint32_t)wave * (kGRing * kGBlk);
  auto pair = [&](uint32_t lo_at, uint32_t hi_at) __attribute__((always_inline)) {
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(uintptr_t)lo_at);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4*)(uintptr_t)hi_at);
    return __builtin_bit_cast(frag, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  const int R = (int)own_sgpr((uint32_t)p.R);
  const bool causal = p.causal != 0;
  const char* const zeros = own_sgpr((const char*)p.zero_block);
  const uint32_t q_rowb = own_sgpr((uint32_t)(p.q_st * 2)), k_rowb = own_sgpr((uint32_t)(p.k_st * 2)), g_step = own_sgpr((uint32_t)(p.g_slots * kGBlk));
  const uint32_t u_lane = g_base + (uint32_t)(li * 66 + g * 256);   // G element (row 4 g + li, column li) of ring slot 0
  for (int it = it0; it < it1; ++it) {
    const int b = BY_LENGTH ? it : (int)((uint32_t)it / (uint32_t)p.tg_chunks);
    int tok0, Lb, I0, I1;
    seq_of(b, tok0, Lb);
    const int n_rows = (Lb + 31) / 32;                       // row blocks of this sequence
    item(it, n_rows, I0, I1);
    const int rho0 = p.rho_min + 4 * group;
    if (I0 >= I1) continue;
    const bool lead = I0 == 0;                               // the key rows ahead of the first row block are this item's as well
    const int last = I1 - I0;   // one more turn than row blocks: the last block's rows of k that precede it
    const char* const q_rows = p.q + ((int64_t)b * p.q_sb + (int64_t)tok0 * p.q_st + (int64_t)h * p.q_sh) * 2 + chunk_off;
    const char* const k_rows = p.k + ((int64_t)b * p.k_sb + (int64_t)tok0 * p.k_st + (int64_t)h * p.k_sh) * 2 + chunk_off;
    // What the turns n0 .. n0 + 31 and the loads they ask for have to know of G, a row block n = n0 - 1 + lane per lane: where block (I0 + n, rho)
    // begins in its row, and which of them there are (a near step the dQ launch met, inside the sequence), go into which table's products.
    int n0 = 0;
    uint32_t g_off = 0;
    uint64_t there = 0, for_k = 0, for_q = 0;
    auto window = [&](int n) __attribute__((always_inline)) {
      n0 = n;
      const int row_block = I0 + n - 1 + lane;
      const Zones z = zones_of(max(row_block, 0) / 4 * FDB_BM, Lb, R, causal, true);
      const int at = row_block - rho - z.s0;
      const bool is = (uint32_t)row_block < (uint32_t)n_rows && at >= 0 && z.s1 > z.s0 && at <= z.s1 - z.s0;
      g_off = is ? (uint32_t)at * kGBlk : 0;
      there = __ballot(is);
      const bool mine = n - 1 + lane < last;
      for_k = there & __ballot(mine);
      for_q = there | there << 1;
      if (n == 0 && !lead) for_q &= ~2ull;
    };
    // What is fetched next: row block I of q and of G, row block I - 1 - rho0 of k (the wave w = 0 uses the newest).  Rows outside the sequence
    // are finite values that meet zeros in G.
    int q_row = I0 * 32 + srow, k_row = (I0 - 1 - rho0) * 32 + srow;
    uint64_t g_at = (uint64_t)(uintptr_t)p.g_blocks + (uint64_t)(((int64_t)b * p.H + h) * p.g_rows + I0 - 1) * g_step;
    uint32_t k_to = 0, k_from = (uint32_t)(-wave & (kKRing - 1)) * kTile;   // ring places of k: the next load's, this wave's rows
    auto rows_dma = [&](const char* rows, uint32_t rowb, int row, uint32_t dst) __attribute__((always_inline)) {
      dma16n(rows + (uint64_t)(uint32_t)max(0, min(row, Lb - 1)) * rowb, dst + wave_kb);
    };
    auto g_dma = [&](int j, uint32_t ring) __attribute__((always_inline)) {   // block n0 - 1 + j; zeros where there is none
      const uint64_t at = g_at + (uint32_t)__builtin_amdgcn_readlane(g_off, j);
      dma16sn_pair((there >> j) & 1 ? (const char*)(uintptr_t)at : zeros, lane * 16, g_base + ring * kGBlk);
      g_at += g_step;
    };
    auto fetch = [&](int j, uint32_t ring) __attribute__((always_inline)) {   // what row block n0 - 1 + j needs first, four loads per wave
      rows_dma(q_rows, q_rowb, q_row, ring * kTile);
      rows_dma(k_rows, k_rowb, k_row, kTgOffK + k_to);
      g_dma(j, ring);
      q_row += 32, k_row += 32;
      k_to = (k_to + kTile) & (kKRing * kTile - 1);
    };
    __syncthreads();   // the item before is done with the rings
    for (int w = 1; w < 4; ++w) rows_dma(k_rows, k_rowb, k_row - 32 * w, kTgOffK + (uint32_t)(kKRing - w) * kTile);
    window(0);
    g_dma(0, kGRing - 1);
    fetch(1, 0);
    fetch(2, 1);
    auto turn = [&](auto slot_tag, int j) __attribute__((always_inline)) {   // row block n = n0 - 1 + j
      constexpr int RING = decltype(slot_tag)::value, PREV = (RING + kGRing - 1) % kGRing;
      wait_vmcnt<4>();   // this row block's loads have landed, those of the next one may still fly
      __syncthreads();
      fetch(j + 2, (RING + 2) % kGRing);
      const bool now_k = (for_k >> j) & 1, now_q = (for_q >> j) & 1;
      if (now_k || now_q) {   // the operands of both tables' products are requested before the first product waits for one
        frag gk[2], gq[2], tq[2][2], tk[2][2];
        uint32_t kt[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          kt[x] = yt[x] + k_from;
          asm("" : "+v"(kt[x]));   // the constant part of the address belongs into the instruction
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          gk[c] = pair(g_base + gt[0] + RING * kGBlk + 1024 * c, g_base + gt[1] + RING * kGBlk + 1024 * c);
#pragma unroll
          for (int d = 0; d < 2; ++d) tq[c][d] = pair(yt[2 * d] + RING * kTile + 2048 * c, yt[2 * d + 1] + RING * kTile + 2048 * c + 1024);
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          s16x8 a;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            // row of G behind (key row 16 c + 8 (e/4) + 4 g + e%4, position li), counted from block I - 1 on: o0 + 4 g + li
            const int o0 = 16 * c + 8 * (e >> 2) + (e & 3);
            uint32_t at = u_lane + PREV * kGBlk + o0 * 64;
            if (RING == 0) at = (at & (kGRing * kGBlk - 1)) | g_base;   // block I lies in slot 0, block I - 1 in the last one
            a[e] = *(LDS_AS const short*)(uintptr_t)at;
          }
          gq[c] = __builtin_bit_cast(frag, a);
#pragma unroll
          for (int d = 0; d < 2; ++d) tk[c][d] = pair(kt[2 * d] + kTgOffK + 2048 * c, kt[2 * d + 1] + kTgOffK + 2048 * c + 1024);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (now_k) {
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int d = 0; d < 2; ++d) ek[d] = QT::mma(gk[c], tq[c][d], ek[d]);
        }
        if (now_q) {
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int d = 0; d < 2; ++d) eq[d] = QT::mma(gq[c], tk[c][d], eq[d]);
        }
      }
      k_from = (k_from + kTile) & (kKRing * kTile - 1);
    };
    int n = 0;
#pragma unroll 1
    for (;;) {
      if (n - n0 == 32) window(n);
      const int j = n - n0 + 1;
      if (n + 3 > last) break;
      turn(std::integral_constant<int, 0>{}, j);
      turn(std::integral_constant<int, 1>{}, j + 1);
      turn(std::integral_constant<int, 2>{}, j + 2);
      turn(std::integral_constant<int, 3>{}, j + 3);
      n += 4;
    }
    if (n <= last) turn(std::integral_constant<int, 0>{}, n - n0 + 1);
    if (n + 1 <= last) turn(std::integral_constant<int, 1>{}, n - n0 + 2);
    if (n + 2 <= last) turn(std::integral_constant<int, 2>{}, n - n0 + 3);
    wait_vmcnt<0>();
  }
  // [part][head][rho][table][position][d]
  float* out = p.e_parts + (((int64_t)part * p.H + h) * (4 * p.tg_groups) + 4 * group + wave) * (2 * 32 * 64);
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int c = 8 * (v >> 2) + 4 * g + (v & 3);
      out[c * 64 + 32 * d + li] = ek[d][v];
      out[2048 + c * 64 + 32 * d + li] = eq[d][v];
    }
}

// Row delta of a table's gradient: the sum of dE over the parts and over the relative positions inside the radius with
// delta(r) = delta (a range, since delta is monotone), the saturated rows' sums at its ends, times sm_scale.  A workgroup takes
// four rows of one head and table (blockIdx.z), a wave each, which finds its range by searches 64 entries wide (three dependent
// loads for a radius of 512).  A quarter of the lanes takes every fourth part, sixteen bytes a lane, four positions at a time: a
// row is a handful of loads in flight together, so that a launch of 12288 waves is bound by how many of them are resident.
// Four bytes a lane, a load per part: 12.7 us where this takes 8.9 (25 MB, 12 heads).
constexpr int kFoldRows = 4;

// how many of the n entries of the monotone table are below v
__device__ __forceinline__ int entries_below(const int16_t* lut, int n, int v, int lane) {
  int lo = 0;
  while (n > 64) {
    const int step = (n + 63) / 64;
    const int c = __popcll(__ballot(lane * step < n && lut[lo + min(lane * step, n - 1)] < v));   // probes below v: a prefix of them
    if (c == 0) return lo;
    lo += (c - 1) * step + 1;
    n = min(step - 1, n - (c - 1) * step - 1);
  }
  return lo + __popcll(__ballot(lane < n && lut[lo + min(lane, max(n - 1, 0))] < v));
}

template <class QT>
__global__ __launch_bounds__(256) void fdb_table_fold_kernel(const FdbBwdRingParams p) {
  const int tid = threadIdx.x, lane = tid & 63, h = blockIdx.y, table = blockIdx.z, row0 = blockIdx.x * kFoldRows;
  const int row = row0 + __builtin_amdgcn_readfirstlane(tid >> 6), entries = 2 * p.R + 1;
  const int s = lane >> 4, c = lane & 15;   // parts s, s + 4, ...; elements 4 c .. 4 c + 3 of the row
  if (row >= 2 * p.S) return;
  const int from = entries_below(p.lut, entries, row, lane);   // the row's entries of the table: [from, to)
  const int wide = __popcll(__ballot(from + lane < entries && p.lut[min(from + lane, entries - 1)] == row));
  const int to = wide < 64 ? from + wide : entries_below(p.lut, entries, row + 1, lane);
  const int r_min = 32 * p.rho_min, r_max = 32 * (p.rho_min + 4 * p.tg_groups) - 1;
  const int64_t part_len = (int64_t)p.H * (4 * p.tg_groups) * 4096;
  const float* e = p.e_parts + (int64_t)h * (4 * p.tg_groups) * 4096 + table * 2048 + 4 * c;
  const bool low = from == 0 && to > 0, high = to == entries && from < to;
  const int r0 = max(max(from - p.R, -p.R + 1), r_min), r1 = min(min(to - 1 - p.R, p.R - 1), r_max);
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  for (int r = r0; r <= r1; r += 4) {
    for (int part = s; part < p.tg_parts; part += 4) {
      f32x4 v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int x = min(r + j, r1) - r_min;
        v[j] = *(const f32x4*)(e + part * part_len + (int64_t)(x >> 5) * 4096 + (x & 31) * 64);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) sum += r + j <= r1 ? v[j] : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  if (p.has_far && (low || high)) {
    const float* f = p.far_parts + (int64_t)h * 256 + table * 128 + 4 * c;
    for (int part = s; part < p.tg_parts; part += 4) {
      const f32x4 up = *(const f32x4*)(f + (int64_t)part * p.H * 256), down = *(const f32x4*)(f + (int64_t)part * p.H * 256 + 64);
      if (high) sum += up;
      if (low) sum += down;
    }
  }
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    sum[x] += __shfl_xor(sum[x], 16);
    sum[x] += __shfl_xor(sum[x], 32);
  }
  typedef typename QT::scratch_t T;   // the gradients' rows are only element aligned: one element a lane
  T* out = (T*)(table == 0 ? p.dpk : p.dpq) + (int64_t)h * p.dp_sh + (int64_t)row * p.dp_sr + 4 * c + s;
  *out = (T)((s == 0 ? sum[0] : s == 1 ? sum[1] : s == 2 ? sum[2] : sum[3]) * p.sm_scale);
}

// Up to so many workgroups a role, the two roles are one launch (with the statistics' own launch before it): what each leaves empty at
// its end the other fills, while a launch of many rounds has little to fill and pays for the statistics.  Whole backward, 12 heads,
// two launches -> one: 1x512 (48 a role) 92 -> 65 us, 8x512 (384) 139 -> 121, 2x1501 (288) 236 -> 196, 4x2048 (768) 434 -> 412,
// 4x4096 (1536) 1195 -> 1178; 8x4096 (3072) would go from 2350 to 2395.
constexpr unsigned kMostTogether = 2048;

template <class QT, bool BY_LENGTH>
int launch_all(const FdbBwdRingParams& p, hipStream_t stream) {
  auto dq = fdb_bwd_ring_kernel<QT, 0, BY_LENGTH>;
  auto dkv = fdb_bwd_ring_kernel<QT, 1, BY_LENGTH>;
  auto tg = fdb_table_grad_kernel<QT, BY_LENGTH>;
  auto both = fdb_bwd_both_kernel<QT, BY_LENGTH>;
  static std::atomic<uint64_t> set0{0}, set1{0}, set2{0}, set3{0};
  hipError_t e = fdb_set_lds_once((const void*)dq, kLds, set0);
  if (e == hipSuccess) e = fdb_set_lds_once((const void*)dkv, kLds, set1);
  if (e == hipSuccess) e = fdb_set_lds_once((const void*)tg, kTgLds, set2);
  if (e == hipSuccess) e = fdb_set_lds_once((const void*)both, kLds, set3);
  if (e != hipSuccess) return (int)e;
  const unsigned grid = (unsigned)p.tiles * (unsigned)p.H * (unsigned)p.B;
  if (grid <= kMostTogether) {
    hipLaunchKernelGGL((fdb_row_stats_kernel<QT, BY_LENGTH>), dim3((unsigned)p.tiles, (unsigned)p.H, (unsigned)p.B + (BY_LENGTH ? 1 : 0)), dim3(256), 0, stream, p);
    hipLaunchKernelGGL(both, dim3(2 * grid), dim3(kThreads), kLds, stream, p);
  } else {
    if (BY_LENGTH) hipLaunchKernelGGL((fdb_row_stats_kernel<QT, true>), dim3((unsigned)p.tiles, (unsigned)p.H), dim3(256), 0, stream, p);
    hipLaunchKernelGGL(dq, dim3(grid), dim3(kThreads), kLds, stream, p);
    hipLaunchKernelGGL(dkv, dim3(grid), dim3(kThreads), kLds, stream, p);
  }
  hipLaunchKernelGGL(tg, dim3((unsigned)p.H, (unsigned)p.tg_parts, (unsigned)(p.tg_groups + (p.has_far ? 1 : 0))), dim3(kThreads), kTgLds, stream, p);
  hipLaunchKernelGGL(fdb_table_fold_kernel<QT>, dim3((unsigned)((2 * p.S + kFoldRows - 1) / kFoldRows), (unsigned)p.H, 2), dim3(256), 0, stream, p);
  return (int)hipGetLastError();
}

}  // namespace

int fdb_launch_bwd_ring(const FdbBwdRingParams& p, int dtype, void* stream) {
  switch (dtype) {
    case FDB_BF16: return p.by_length ? launch_all<Bf16Tr, true>(p, (hipStream_t)stream) : launch_all<Bf16Tr, false>(p, (hipStream_t)stream);
    case FDB_F16: return p.by_length ? launch_all<F16Tr, true>(p, (hipStream_t)stream) : launch_all<F16Tr, false>(p, (hipStream_t)stream);
    default: return FDB_ERR_DTYPE;
  }
}

// Disentangled-attention forward in fp32 at head_dim 64 with position terms: every key tile of a query tile in one launch, in steps of 32 keys.
//
// The position products are formed as in the 16-bit near kernel (fdb_near.hip): a wave owns 32 query rows (the columns of the MFMAs), the
// expanded tables E_K[r] = K_r[delta(r)] and E_Q[r] = Q_r[delta(r)] slide through two LDS rings of five batches of 32 relative positions,
// C[r][i] = q_i . E_K[r] is contracted once per block and skewed through a per-wave scratch whose other half still holds the block of the step
// before, P[j][r] = k_j . E_Q[r] is skewed by moving its columns between lanes.  Scratch, lanes and sums are all fp32.
//
// What is different is the balance.  An fp32 MFMA (32x32x2) takes 64 clocks for an eighth of the contraction of a 16-bit one: a near step is 160 of
// them, 10240 clocks, next to which some 300 other instructions are little.  So one workgroup per CU (rows of 256 bytes: 146 KB of LDS) and one
// wave per SIMD do, if the instructions between the products are issued while MFMAs run: the content product comes last of the
// four score products, and between its 32 MFMAs a step hands C through the scratch and P from lane to lane and fetches V.
//
// What bounds it: the fp32 matrix cores (8 x 512, 16 heads: 32 steps of a workgroup in 187 us, 83 % of it products).  The kernel this took the place of
// gathered the table rows of every block from global memory, 32 cache lines an instruction, and contracted C's shared block twice.  Whole calls, replayed
// (packed ones: one after the other), us, before -> here, 12 heads unless stated; 512 and 64 are the tables' reach:
//                           both terms                                           c2p alone                      p2c alone
//                           fixed          causal         packed                 fixed          causal          fixed          causal
//   1 x 48,  512            23.7 -> 21.5   23.4 -> 21.7   20.6 -> 19.0           18.0 -> 16.8   18.0 -> 17.1    17.9 -> 17.9   17.9 -> 18.1
//   1 x 300, 512            56.5 -> 42.9   78.3 -> 64.2   54.6 -> 40.4           41.5 -> 31.9   54.1 -> 43.0    42.2 -> 36.1   55.2 -> 52.5
//   1 x 512, 512            45.0 -> 39.9   121  -> 97.6   43.4 -> 38.6           34.7 -> 31.0   82.7 -> 64.4    35.1 -> 34.2   84.6 -> 80.1
//   3 x 777, 512            191  -> 147    160  -> 130    216  -> 171            129  -> 95.1   113  -> 88.4    132  -> 120    115  -> 108
//   8 x 512, 512, 16 heads  244  -> 192    190  -> 149    368  -> 276            164  -> 124    130  -> 98.5    168  -> 156    130  -> 122
//   64 x 64, 512            59.9 -> 56.0   61.8 -> 57.7   88.7 -> 65.8           46.5 -> 41.7   48.0 -> 43.1    45.3 -> 45.0   47.1 -> 46.4
//   2 x 2048, 512           580  -> 492    401  -> 342    613  -> 509            436  -> 369    304  -> 259     443  -> 428    310  -> 298
//   4 x 4096, 512           2725 -> 2425   1660 -> 1485   2 x 8192, 512  4430 -> 4140   2710 -> 2530
//   2 x 2048, 64            375  -> 357    269  -> 255    4 x 4096, 64   1960 -> 1920   1260 -> 1220   2 x 8192, 64  3650 -> 3620   2300 -> 2260
// Errors against 64 bits are no larger (of the output's norm, before and here: 1 x 512 3.66e-7 and 3.61e-7, 1 x 2048 5.35e-7 and 5.16e-7, 1 x 4096 with a
// reach of 64 7.19e-7 and 6.88e-7).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "fdb_device.h"
#include "fdb_kernels.h"
#include "../../include/fdb.h"

using namespace fdb;

namespace {

constexpr int kStep = 32, kBatches = 5, kRow = 256;              // keys of a step; ring batches of 32 rows; bytes of a row
constexpr int kTile = 32 * kRow;                                 // 32 rows
constexpr int kPitch = 68;                                       // floats per row of a wave's scratch: two blocks of 32 columns, columns 0..3 once more
constexpr int lds_bytes(bool c2p, bool p2c) { return 4 * kTile + (c2p ? kBatches * kTile + 4 * 32 * kPitch * 4 : 0) + (p2c ? kBatches * kTile : 0); }

// Rows of sixteen 16-byte chunks.  Slot (row, s) of K and of the rings holds chunk s ^ (row % 16): sixteen consecutive rows' same chunk lies in
// sixteen bank groups.  V is read 4 bytes a lane, 32 columns of a row by half a wave and of the row four further on by the other half:
// its slots differ in the half of the row they lie in.
__device__ __forceinline__ int row_f(int row) { return row & 15; }
__device__ __forceinline__ int v_f(int row) { return 8 * ((row >> 2) & 1); }

struct Operand {   // 32 rows x 64: lane (li, g) holds chunks 2x + g of row li, element e of chunk x is contraction index 8x + 4g + e
  f32x4 a[8];
};
__device__ __forceinline__ f32x16 mma1(const Operand& a, const Operand& b, int n, f32x16 c) {   // the n-th of 32 steps of the contraction
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a.a[n >> 2][n & 3], b.a[n >> 2][n & 3], c, 0, 0, 0);
}

template <bool C2P, bool P2C>
__global__ __launch_bounds__(256, 1) void fdb_near_f32_kernel(const FdbKParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  read_arguments(p);
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, li = lane & 31, g = lane >> 5;
  int b, tile, h, tok0, sl;   // tile: the query tile of sequence b, or the entry of a packed call's work-list
  place_of((int)blockIdx.x, p, p.tiles_per_seq, p.cu == nullptr, kNatural, lane, b, tile, h, tok0, sl);
  int m0, Lb;
  int64_t qo, ko, vo, oo;
  if (p.cu) {
    if (!packed_place(p, tile, lane, b, m0, tok0, Lb)) return;
    qo = ko = vo = oo = 0;
  } else {
    m0 = tile * FDB_BM;
    Lb = min(max(sl, 0), p.L - tok0);
    if (p.fill_pad && blockIdx.y == 0)
      fill_pad_rows<kRow>(p.out + ((int64_t)b * p.o_sb + (int64_t)h * p.o_sh) * 4, p.o_st * 4, tile, p.L, tok0, Lb,
                          sl < 0 ? F32Tr::NAN_WORD : 0u, tid, p.lse && h == 0 ? p.lse + (int64_t)b * p.L * p.H : nullptr, p.H);
    if (m0 >= Lb) return;
    qo = b * p.q_sb; ko = b * p.k_sb; vo = b * p.v_sb; oo = b * p.o_sb;
  }
  const char* qb = p.q + (qo + (int64_t)tok0 * p.q_st + (int64_t)h * p.q_sh) * 4;
  const char* kb = p.k + (ko + (int64_t)tok0 * p.k_st + (int64_t)h * p.k_sh) * 4;
  const char* vb = p.v + (vo + (int64_t)tok0 * p.v_st + (int64_t)h * p.v_sh) * 4;
  char* ob = p.out + (oo + (int64_t)tok0 * p.o_st + (int64_t)h * p.o_sh) * 4;
  const char* pkb = C2P ? p.pk + (int64_t)h * p.pk_sh * 4 : nullptr;
  const char* pqb = P2C ? p.pq + (int64_t)h * p.pq_sh * 4 : nullptr;
  const uint32_t k_rsb = (uint32_t)(p.k_st * 4), v_rsb = (uint32_t)(p.v_st * 4);  // the host checks that they fit
  const float x_scale = p.scale_log2;

  const int iw0 = m0 + wave * 32, i = iw0 + li;
  auto load_row = [&](const char* row) __attribute__((always_inline)) {
    Operand o;
#pragma unroll
    for (int x = 0; x < 8; ++x) o.a[x] = *(const f32x4*)(row + (2 * x + g) * 16);
    return o;
  };
  Operand qf;
  if (i < Lb) {
    qf = load_row(qb + (int64_t)i * p.q_st * 4);
  } else {
#pragma unroll
    for (int x = 0; x < 8; ++x) qf.a[x] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // ---- the steps: [0, s0) far left of the query tile (every r >= R), [s0, s1) near, [s1, end) far right (every r <= -R) ----------------
  int j_end = Lb;
  if (p.causal) j_end = min(Lb, m0 + FDB_BM);
  const int end = (j_end + kStep - 1) / kStep;
  const int lim = m0 - (kStep - 1) - p.R;
  int s0 = lim >= 0 ? min(end, lim / kStep + 1) : 0;
  int s1 = max(s0, min(end, (m0 + FDB_BM - 1 + p.R + kStep - 1) / kStep));
  int all0 = 0, all1 = end;
  const int part = p.key_parts > 1 ? (int)blockIdx.y : 0;
  if (p.key_parts > 1) {   // this workgroup's share
    all0 = share_begins(end, part, p.key_parts);
    all1 = share_begins(end, part + 1, p.key_parts);
  }
  s0 = min(max(s0, all0), all1);
  s1 = max(s0, min(s1, all1));
  const int n_steps = s1 - s0, n_left = s0 - all0, n_right = all1 - s1, n_far = n_left + n_right;
  // far steps first, as t = -n_far .. -1, so that the near steps' operands are not held through them
  auto far_step_at = [&](int t) __attribute__((always_inline)) { return t < -n_right ? s0 + n_right + t : t < 0 ? all1 + t : s0; };
  // Relative positions at near step k: u = r_hi0 - r counts downwards from the first step's largest r; batch = u / 32, slot = batch mod 5.
  // Wave w's block bk is batch k + 4 - w - bk, MFMA row m its row 31 - m: r = iw0 - 32 s - 32 + 32 bk + m.
  const int r_hi0 = m0 + FDB_BM - 1 - s0 * kStep;

  // ---- staging: a direct load fills four rows; two per wave for 32 ---------------------------------------------------------------
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LDS_AS char*)smem;
  const uint32_t Ks = lds0, Vs = Ks + 2 * kTile, EK = Vs + 2 * kTile, EQ = EK + (C2P ? kBatches * kTile : 0), scr = EQ + (P2C ? kBatches * kTile : 0);
  int srow[2];
  uint32_t k_chunk[2], v_chunk[2];
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    srow[n] = 4 * (wave + 4 * n) + (lane >> 4);
    k_chunk[n] = (uint32_t)(((lane & 15) ^ row_f(srow[n])) * 16);
    v_chunk[n] = (uint32_t)(((lane & 15) ^ v_f(srow[n])) * 16);
  }
  auto kv_dma = [&](int s, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < 2; ++n) {   // rows past the end re-read the last one, their scores are masked
      const uint64_t row = (uint64_t)(uint32_t)min(s * kStep + srow[n], Lb - 1);
      const uint32_t at = buf * kTile + (wave + 4 * n) * 1024u;
      dma16n(kb + row * k_rsb + k_chunk[n], Ks + at);
      dma16n(vb + row * v_rsb + v_chunk[n], Vs + at);
    }
  };
  const uint32_t pk_rowb = (uint32_t)(p.pk_sr * 4), pq_rowb = (uint32_t)(p.pq_sr * 4);
  int r_tab = r_hi0;
  auto batch_delta = [&](int (&d)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < 2; ++n) d[n] = (int)((const uint16_t*)p.lut)[max(-p.R, min(p.R, r_tab - srow[n])) + p.R];
    r_tab -= 32;
  };
  auto batch_dma = [&](const int (&d)[2], int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const uint32_t at = slot * kTile + (wave + 4 * n) * 1024u;
      if constexpr (C2P) dma16sn(pkb, __umul24((uint32_t)d[n], pk_rowb) + k_chunk[n], EK + at);
      if constexpr (P2C) dma16sn(pqb, __umul24((uint32_t)d[n], pq_rowb) + k_chunk[n], EQ + at);
    }
  };

  // ---- the first step's loads, ahead of everything that can be worked out while they are on their way ------------------------------
  int dnext[2] = {0, 0};
  if (n_steps + n_far > 0) {
    kv_dma(far_step_at(-n_far), n_far & 1);
    if (n_steps > 0) {
      int d0[6][2];
#pragma unroll
      for (int bt = 0; bt < 6; ++bt) batch_delta(d0[bt]);
#pragma unroll
      for (int bt = 0; bt < 6; ++bt) asm volatile("" : "+v"(d0[bt][0]), "+v"(d0[bt][1]));
#pragma unroll
      for (int bt = 0; bt < 5; ++bt) batch_dma(d0[bt], bt);
      dnext[0] = d0[5][0], dnext[1] = d0[5][1];
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- per-lane constants ---------------------------------------------------------------------------------------------------------
  const int arow = 31 - li;
  const uint32_t k_lane = (uint32_t)(li * kRow + ((g ^ row_f(li)) * 16)), e_lane = (uint32_t)(arow * kRow + ((g ^ row_f(arow)) * 16));
  auto lds_rows = [&](uint32_t base, uint32_t at) __attribute__((always_inline)) {
    Operand o;
#pragma unroll
    for (int x = 0; x < 8; ++x) o.a[x] = *(LDS_AS const f32x4*)(uintptr_t)(base + (at ^ (32 * x)));
    return o;
  };
  // V[8 q + 4 g + e][32 d + li], element v = 4 q + e of block d: chunk 8 d + li / 4 of a row whose slots are swapped by halves where its bit 2 is set
  const uint32_t v_lane = (uint32_t)(4 * g * kRow + (((li >> 2) ^ (8 * g)) * 16) + (li & 3) * 4);
  auto v_row = [](int v) { return (uint32_t)((8 * (v >> 2) + (v & 3)) * kRow); };
  auto v_elem = [&](int par, int d, int v) __attribute__((always_inline)) {
    return *(LDS_AS const float*)(uintptr_t)(Vs + par * kTile + (v_lane ^ (128 * d)) + v_row(v));
  };
  // Scratch: row li = this lane's query; the block a step contracts goes to the half of the step's parity, element (jj, li) wants column
  // (32 par + li + 32 - jj) mod 64.  The four of jj = 8 q + 4 g + 0 .. 3 are the run that ends there for jj = 8 q + 4 g; columns 64 .. 67 repeat 0 .. 3.
  const uint32_t scr_row = scr + (uint32_t)((wave * 32 + li) * kPitch * 4);
  uint32_t c_rd[2][4];
#pragma unroll
  for (int par = 0; par < 2; ++par)
#pragma unroll
    for (int q = 0; q < 4; ++q) c_rd[par][q] = scr_row + 4u * (uint32_t)((32 * par + li + 29 - 8 * q - 4 * g) & 63);
  auto c_store = [&](const f32x16& c, int half, int q) __attribute__((always_inline)) {
    const f32x4 x = {c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]};
    *(LDS_AS f32x4*)(uintptr_t)(scr_row + (32 * half + 8 * q + 4 * g) * 4) = x;
    if (half == 0 && q == 0) *(LDS_AS f32x4*)(uintptr_t)(scr_row + (g == 0 ? 64 : 4) * 4) = x;   // (columns 4 .. 7 once more as they are)
  };
  // P: register v of lane n holds P[jj][32 bk + n], jj = c + 4 g, c = 8 (v / 4) + v % 4; the element of query li is in lane (li - jj) mod 32 of the
  // same half, in block 1 if li >= jj.  A lane's one reader wants block 1 from it if n + jj < 32.
  const int xl = li + 4 * g;
  uint32_t p_from[16];
#pragma unroll
  for (int v = 0; v < 16; ++v) p_from[v] = 4u * (uint32_t)(((xl - 8 * g - (8 * (v >> 2) + (v & 3))) & 31) + 32 * g);

  f32x16 zero, o_acc[2];
#pragma unroll
  for (int v = 0; v < 16; ++v) zero[v] = o_acc[0][v] = o_acc[1][v] = 0.f;
  float m_run = -INFINITY, l_run = 0.f, row_add = 0.f;

  int slot_rd = 4 - wave, slot_dma = 0;
  Operand aq[2];   // E_Q's rows of the new block and of the one before, by the step's parity
  Operand qx;      // the query of the far steps at hand, with Q_r's row
  auto side_begins = [&](int side) __attribute__((always_inline)) {   // 0: left of the near steps, delta(R); 1: right of them, delta(-R)
    const int delta = p.lut[side == 0 ? 2 * p.R : 0];
    qx = qf;
    if constexpr (C2P) {
      const Operand e = load_row(pkb + (int64_t)delta * p.pk_sr * 4);
      float acc = 0.f;
#pragma unroll
      for (int n = 0; n < 32; ++n) acc = __builtin_fmaf(e.a[n >> 2][n & 3], qf.a[n >> 2][n & 3], acc);
      row_add = wave_half_sum(acc);
    }
    if constexpr (P2C) {
      const Operand e = load_row(pqb + (int64_t)delta * p.pq_sr * 4);
#pragma unroll
      for (int x = 0; x < 8; ++x)
#pragma unroll
        for (int n = 0; n < 4; ++n) qx.a[x][n] = __builtin_fmaf(e.a[x][n], x_scale, qf.a[x][n]);
    }
  };

  // mask, online soft-max in base 2, O^T += V^T P^T: the scores of the keys from j0 on, to which `add` is still to be added, and their values.
  // BY_SUM: a far step, whose products wait for its soft-max.  Its probabilities are formed against the reference point as it is, and their sum says whether
  // that is high enough (a sum bounds its largest term); the maximum is looked for only where it is not.  A near step's maximum is found while its last
  // products run.
  auto absorb = [&](auto by_sum, f32x16& sacc, const float (&vr)[2][16], int j0, float add) __attribute__((always_inline)) {
    constexpr bool BY_SUM = decltype(by_sum)::value;
    if (j0 + kStep > Lb || (p.causal && j0 + kStep - 1 > m0)) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int j = j0 + 8 * (v >> 2) + 4 * g + (v & 3);
        if (j >= Lb || (p.causal && j > i)) sacc[v] = -INFINITY;
      }
    }
    auto row_max = [&]() __attribute__((always_inline)) {
      float mx = sacc[0];
#pragma unroll
      for (int v = 1; v < 16; ++v) mx = fmaxf(mx, sacc[v]);
      return wave_half_max(mx) + add;
    };
    auto refer_to = [&](float m_new) __attribute__((always_inline)) {
      const float alpha = m_run == m_new ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int v = 0; v < 16; ++v) o_acc[d][v] *= alpha;
    };
    f32x8 pv[2];
    auto probs = [&]() __attribute__((always_inline)) {
      const float off = add - (m_run == -INFINITY ? 0.f : m_run);   // -inf: the row has met no key it sees (shares, the ends of a sequence)
#pragma unroll
      for (int v = 0; v < 16; ++v) pv[v >> 3][v & 7] = __builtin_amdgcn_exp2f(sacc[v] + off);
    };
    if constexpr (BY_SUM) {
      probs();
      float sum = sum8(pv[1], sum8(pv[0], 0.f));
      const bool moves = m_run == -INFINITY || !(sum <= 256.f);   // 2^kLazyTau; also a sum that overflows
      if (__any(moves)) {
        const float m_new = fmaxf(m_run, row_max());
        refer_to(wave_half_max(moves ? 1.f : 0.f) > 0.f ? m_new : m_run);   // a row's two lanes together
        probs();
        sum = sum8(pv[1], sum8(pv[0], 0.f));
      }
      l_run += sum;
    } else {
      const float mx = row_max();
      if (__any(mx > m_run + kLazyTau)) refer_to(mx > m_run + kLazyTau ? mx : m_run);
      probs();
      l_run = sum8(pv[1], sum8(pv[0], l_run));
    }
#pragma unroll
    for (int v = 0; v < 16; ++v)
#pragma unroll
      for (int d = 0; d < 2; ++d) o_acc[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[d][v], pv[v >> 3][v & 7], o_acc[d], 0, 0, 0);
  };

  // A far step's K is in registers when it begins and its V when its scores are done, so the barrier that the next step's loads need comes
  // there, and the next K is read and what follows it is loaded while this step's soft-max and products run.  The buffer is an address here and no
  // constant: two forms of the step in one loop cost 64 moves of the sums between them.  With a step's barrier and reads ahead of its products and a maximum
  // ahead of its exponentials, far steps lost to the kernel before them: 2 x 8192 with a reach of 64 3650 us there, 3970 so, 3780 without the former, 3620 without both.
  Operand kf_far;
  auto far_begins = [&](int t) __attribute__((always_inline)) {   // step t's K and V are there; those of t + 1 are asked for
    wait_vmcnt<0>();
    __syncthreads();
    kv_dma(far_step_at(t + 1), (t & 1) ^ 1);
    kf_far = lds_rows(Ks + (t & 1) * kTile, k_lane);
  };
  auto far_step = [&](int t) __attribute__((always_inline)) {
    f32x16 sacc;
    float vr[2][16];
    uint32_t v_at[2];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      v_at[d] = Vs + (t & 1) * kTile + (v_lane ^ (128 * d));
      asm("" : "+v"(v_at[d]));   // the constant part of the address belongs into the instruction
    }
#pragma unroll
    for (int n = 0; n < 32; ++n) {
      sacc = mma1(kf_far, qx, n, n == 0 ? zero : sacc);
      vr[n >> 4][n & 15] = *(LDS_AS const float*)(uintptr_t)(v_at[n >> 4] + v_row(n & 15));
    }
    far_begins(t + 1);   // (after the last one, too: the first near step's, and once more in the other buffer, which that step's loads take over)
    absorb(std::true_type{}, sacc, vr, far_step_at(t) * kStep, row_add);
  };
  auto step = [&](auto par_tag, int k) __attribute__((always_inline)) {
    constexpr int PAR = decltype(par_tag)::value;
    const int s = s0 + k, j0 = s * kStep;
    wait_vmcnt<0>();   // this wave's direct loads of the step before, and the table values
    asm volatile("" : "+v"(dnext[0]), "+v"(dnext[1]));   // (taken here: the compiler does not count the direct loads)
    __syncthreads();   // ... and everybody's; every wave is done with what this step's loads overwrite
    kv_dma(s + 1, PAR ^ 1);   // past the last step, too: rows and table indices are clamped, nobody reads it
    batch_dma(dnext, slot_dma);   // batch k + 5 in place of batch k
    __builtin_amdgcn_sched_barrier(0);
    batch_delta(dnext);           // of batch k + 6
    const Operand kf = lds_rows(Ks + PAR * kTile, k_lane);
    f32x16 sacc, cnew, p0, p1;
    float px[16], cb[16], vr[2][16];
    Operand ac;
    if constexpr (C2P) ac = lds_rows(EK + slot_rd * kTile, e_lane);
    if constexpr (P2C) {
      aq[PAR] = lds_rows(EQ + slot_rd * kTile, e_lane);
#pragma unroll
      for (int n = 0; n < 32; ++n) p1 = mma1(kf, aq[PAR ^ 1], n, n == 0 ? zero : p1);
    }
    if constexpr (C2P) {
#pragma unroll
      for (int n = 0; n < 32; ++n) cnew = mma1(ac, qf, n, n == 0 ? zero : cnew);
    }
    if constexpr (P2C) {
#pragma unroll
      for (int n = 0; n < 32; ++n) {
        p0 = mma1(kf, aq[PAR], n, n == 0 ? zero : p0);
        if constexpr (C2P) {
          if (n >= 8 && n < 12) c_store(cnew, PAR, n - 8);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (C2P) {
      if constexpr (!P2C) {
#pragma unroll
        for (int q = 0; q < 4; ++q) c_store(cnew, PAR, q);
      }
      wave_lds_fence();   // the LDS unit runs one wave's operations in order; this keeps the compiler from moving them
    }
#pragma unroll
    for (int n = 0; n < 32; ++n) {
      sacc = mma1(kf, qf, n, n == 0 ? zero : sacc);
      if constexpr (C2P) {
        if (n < 8) {
#pragma unroll
          for (int e = 2 * (n & 1); e < 2 * (n & 1) + 2; ++e) cb[4 * (n >> 1) + e] = *(LDS_AS const float*)(uintptr_t)(c_rd[PAR][n >> 1] + 4 * (3 - e));
        }
      }
      if constexpr (P2C) {
        if (n >= 2 && n < 18) {
          const int v = n - 2, c = 8 * (v >> 2) + (v & 3);
          px[v] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((int)p_from[v], __builtin_bit_cast(int, xl < 32 - c ? p1[v] : p0[v])));
        }
      }
      vr[n >> 4][n & 15] = v_elem(PAR, n >> 4, n & 15);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      if constexpr (C2P) sacc[v] += cb[v];
      if constexpr (P2C) sacc[v] = __builtin_fmaf(px[v], x_scale, sacc[v]);
    }
    absorb(std::false_type{}, sacc, vr, j0, 0.f);
    slot_rd = slot_rd == kBatches - 1 ? 0 : slot_rd + 1;
    slot_dma = slot_dma == kBatches - 1 ? 0 : slot_dma + 1;
  };

  if (n_steps + n_far > 0) {
#pragma unroll
    for (int x = 0; x < 8; ++x) qf.a[x] *= x_scale;   // the soft-max scale, in base 2
    using T0 = std::integral_constant<int, 0>;
    using T1 = std::integral_constant<int, 1>;
    if (n_far > 0) {
      far_begins(-n_far);
#pragma unroll 1
      for (int side = n_left > 0 ? 0 : 1, t = -n_far; t < 0; ++side) {   // K and V through the two buffers so that the first near step finds its own in buffer 0
        side_begins(side);
        const int last = side == 0 ? -n_right : 0;
#pragma unroll 1
        for (; t < last; ++t) far_step(t);
      }
    }
    if (n_steps > 0) {
      wait_vmcnt<0>();
      __syncthreads();   // the first batches are there
      if constexpr (P2C) aq[1] = lds_rows(EQ + (3 - wave) * kTile, e_lane);   // block 1 of the first step
      if constexpr (C2P) {
        const Operand ac = lds_rows(EK + (3 - wave) * kTile, e_lane);
        f32x16 c1;
#pragma unroll
        for (int n = 0; n < 32; ++n) c1 = mma1(ac, qf, n, n == 0 ? zero : c1);
#pragma unroll
        for (int q = 0; q < 4; ++q) c_store(c1, 1, q);
      }
      int k = 0;
#pragma unroll 1
      for (; k + 1 < n_steps; k += 2) {
        step(T0{}, k);
        step(T1{}, k + 1);
      }
      if (k < n_steps) step(T0{}, k);
    }
    wait_vmcnt<0>();  // the last step's direct loads: none may still be writing LDS when the workgroup ends
  }

  // ---- epilogue: normalise, store ----------------------------------------------------------------------------------------------------
  const float l_tot = wave_half_sum(l_run);
  if (i < Lb) {
    const int64_t tok = p.cu ? (int64_t)tok0 + i : (int64_t)b * p.L + tok0 + i;
    char* orow = ob + (int64_t)i * p.o_st * 4;
    float* lse_row = p.lse;
    // a row whose every score is -inf has no soft-max: NaN, unless another share may have met a score that is not
    float inv = l_tot > 0.f ? 1.f / l_tot : __builtin_nanf(""), lse = l_tot > 0.f ? (m_run + __builtin_amdgcn_logf(l_tot)) * 0.6931471805599453f : __builtin_nanf("");
    if (p.key_parts > 1) {  // every share's partial result goes to its workspace slot
      orow = ws_slot_out(p, part, kRow) + (tok * p.H + h) * kRow;
      lse_row = ws_slot_lse(p, part, kRow);
      if (l_tot == 0.f) inv = 0.f, lse = -INFINITY;
    }
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        F32Tr::store4(orow + (32 * d + 8 * q + 4 * g) * 4, o_acc[d][4 * q] * inv, o_acc[d][4 * q + 1] * inv, o_acc[d][4 * q + 2] * inv, o_acc[d][4 * q + 3] * inv);
    if (lse_row && g == 0) lse_row[tok * p.H + h] = lse;
  }
}

template <bool C2P, bool P2C>
int launch(const FdbKParams& p, int grid_x, hipStream_t stream) {
  auto kern = fdb_near_f32_kernel<C2P, P2C>;
  constexpr int lds = lds_bytes(C2P, P2C);
  static_assert(lds <= 160 * 1024, "LDS budget");
  static std::atomic<uint64_t> lds_set{0};
  const hipError_t e = fdb_set_lds_once((const void*)kern, lds, lds_set);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid_x * p.H, p.key_parts > 1 ? (unsigned)p.key_parts : 1u), dim3(256), lds, stream, p);
  return (int)hipGetLastError();
}

}  // namespace

int fdb_launch_near_f32(const FdbKParams& p, int grid_x, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (p.pk && p.pq) return launch<true, true>(p, grid_x, stream);
  if (p.pk) return launch<true, false>(p, grid_x, stream);
  if (p.pq) return launch<false, true>(p, grid_x, stream);
  return FDB_ERR_UNSUPPORTED;
}

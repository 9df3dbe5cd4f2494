// How a near launch ends (fdb_near.hip, fdb_fp8.hip): a query row's sums over the near keys, merged with the far launch's partial results where there are
// some, normalised and stored; head_dim 64, 16-bit output.
#pragma once
#include "fdb_device.h"
#include "fdb_kernels.h"
#include "../../include/fdb.h"

namespace fdb {

// The row at orow (token tok, head h) from this lane's half of it, o_acc[d][4 q + e] = element 32 d + 8 q + 4 g + e relative to the reference point
// m_run, and the row's sum l_tot.  far_parts partial results: the first in out / lse, the others in the workspace (rows normalised over their keys,
// log-sum-exp -inf where a row had none).  It is what a workgroup does alone at its end, bound by its chain of loads, waits and tests: 32 x 128
// 29.6 -> 29.2 us for a layer, 64 packed sequences 322 -> 319.5, 1 x 4096 with 16 heads 121.3 -> 120.4; no difference where the clock is the limit.
template <class VT>
__device__ __forceinline__ void near_row_out(const FdbKParams& p, char* orow, int64_t tok, int h, int g, const f32x16 (&o_acc)[2], float m_run, float l_tot,
                                             int far_parts) {
  float denom = l_tot, m_out = m_run;
  if (far_parts == 0) {
    const float inv = denom > 0.f ? 1.f / denom : 0.f;
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        VT::store4(orow + (32 * d + 8 * q4 + 4 * g) * 2, o_acc[d][4 * q4] * inv, o_acc[d][4 * q4 + 1] * inv, o_acc[d][4 * q4 + 2] * inv,
                   o_acc[d][4 * q4 + 3] * inv);
  } else {
    // A part's eight pieces of the row are asked for together, the first part's along with the log-sum-exps of all: one memory latency where a load,
    // its wait and its sum one after the other were eight (and a test per piece and part; 5 us of a workgroup's life, 1.3 without a far part).
    using piece = typename VT::scratch4;
    piece far4[2][4];
    auto ask = [&](int s) __attribute__((always_inline)) {
      const char* row = s == 0 ? orow : far_part_out(p, s, 64 * 2) + (tok * p.H + h) * (64 * 2);
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) far4[d][q4] = *(const piece*)(row + (32 * d + 8 * q4 + 4 * g) * 2);
    };
    ask(0);
    float w_far[FDB_MAX_FAR_PARTS];   // log-sum-exp in base 2 until the maximum is known
#pragma unroll
    for (int s = 0; s < FDB_MAX_FAR_PARTS; ++s) {
      w_far[s] = -INFINITY;
      if (s < far_parts) w_far[s] = (s == 0 ? p.lse : far_part_lse(p, s, 64 * 2))[tok * p.H + h] * 1.4426950408889634f;
    }
    m_out = m_run + __builtin_amdgcn_logf(l_tot);
#pragma unroll
    for (int s = 0; s < FDB_MAX_FAR_PARTS; ++s) m_out = fmaxf(m_out, w_far[s]);
    const float w_near = __builtin_amdgcn_exp2f(m_run - m_out);
    denom = w_near * l_tot;
#pragma unroll
    for (int s = 0; s < FDB_MAX_FAR_PARTS; ++s) {
      w_far[s] = w_far[s] != -INFINITY ? __builtin_amdgcn_exp2f(w_far[s] - m_out) : 0.f;
      denom += w_far[s];
    }
    const float inv = denom > 0.f ? 1.f / denom : 0.f;
    f32x4 f[2][4];
#pragma unroll
    for (int s = 0; s < FDB_MAX_FAR_PARTS; ++s) {
      if (s >= far_parts) break;
      if (s > 0) ask(s);
      const float sf = w_far[s] * inv;
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const f32x4 x = __builtin_convertvector(far4[d][q4], f32x4) * sf;
          f[d][q4] = s == 0 ? x : f[d][q4] + x;
        }
    }
    const float sn = w_near * inv;
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        VT::store4(orow + (32 * d + 8 * q4 + 4 * g) * 2, o_acc[d][4 * q4] * sn + f[d][q4][0], o_acc[d][4 * q4 + 1] * sn + f[d][q4][1],
                   o_acc[d][4 * q4 + 2] * sn + f[d][q4][2], o_acc[d][4 * q4 + 3] * sn + f[d][q4][3]);
  }
  if (p.lse && g == 0) p.lse[tok * p.H + h] = (m_out + __builtin_amdgcn_logf(denom)) * 0.6931471805599453f;
}

}  // namespace fdb

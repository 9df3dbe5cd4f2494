// The linear layer in front of the attention for a batch of few rows, 16-bit types.
//
// A product of a few rows is latency, and a call of that library costs the host 8 us where a
// launch costs 2.5.  Up to 32 rows fdb_linear_kernel streams the weights: one workgroup per 16 output columns, eight or
// sixteen waves that share the contraction, so that even a [768 x 768] weight is on its way through 48 x 8 waves at once, each
// with four steps' loads in flight.  In a replayed graph, [24 x 768] . [768 x 2304]: 4.0 us against hipBLASLt's 4.8.
// Beyond that fdb_gemm.hip's tiles, for the sizes they take (columns and output rows by eights, or by fours where the streaming makes more
// than one round): [64 / 200 x 768] . [768 x 2304] 5.3 / 5.6 us.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fdb_device.h"
#include "fdb_kernels.h"
#include "../../include/fdb.h"

using namespace fdb;

namespace {

constexpr int kLinCols = 16;

// out [M, N] = x [M, K] . w [N, K]^T + bias.  Contraction steps of 32 go round the waves; MT row blocks of 16 per
// workgroup share every weight fragment.  A lane reads 16 bytes of a row, four lanes 64 contiguous bytes.
template <class QT, int MT, int kLinWaves>
__global__ __launch_bounds__(64 * kLinWaves) void fdb_linear_kernel(const char* __restrict__ x, const char* __restrict__ w,
                                                                    const typename QT::scratch_t* __restrict__ bias, char* __restrict__ out,
                                                                    int32_t M, int32_t N, int32_t K, int64_t ldx, int64_t ldw, int64_t ldo) {
  using frag = typename QT::frag;
  constexpr int ROWS = 16 * MT, PITCH = kLinCols + 4, DEPTH = 4;
  __shared__ float part[kLinWaves][ROWS * PITCH];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * kLinCols, m0 = blockIdx.y * ROWS;
  const char* wp = w + (int64_t)min(n0 + r, N - 1) * ldw * 2 + kg * 16;
  const char* xp[MT];
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    xp[t] = x + (int64_t)min(m0 + 16 * t + r, M - 1) * ldx * 2 + kg * 16;  // rows and columns past the end re-read the last one
    acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int steps = K / 32;
  for (int s = wave; s < steps; s += kLinWaves * DEPTH) {
    frag wf[DEPTH], xf[DEPTH][MT];
#pragma unroll
    for (int j = 0; j < DEPTH; ++j)
      if (s + kLinWaves * j < steps) {
        const int off = (s + kLinWaves * j) * 64;
        wf[j] = QT::load(wp + off);
#pragma unroll
        for (int t = 0; t < MT; ++t) xf[j][t] = QT::load(xp[t] + off);
      }
#pragma unroll
    for (int j = 0; j < DEPTH; ++j)
      if (s + kLinWaves * j < steps) {
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = mma16(xf[j][t], wf[j], acc[t]);
      }
  }
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) part[wave][(16 * t + 4 * kg + v) * PITCH + r] = acc[t][v];
  __syncthreads();
  // two neighbouring columns of a row per thread
  for (int c = tid; c < ROWS * (kLinCols / 2); c += 64 * kLinWaves) {
    const int row = c / (kLinCols / 2), col = 2 * (c % (kLinCols / 2));
    float a = 0.f, b = 0.f;
#pragma unroll
    for (int v = 0; v < kLinWaves; ++v) {
      a += part[v][row * PITCH + col];
      b += part[v][row * PITCH + col + 1];
    }
    const int m = m0 + row, n = n0 + col;
    if (m < M && n < N) {  // N is even
      if (bias) {
        a += (float)bias[n];
        b += (float)bias[n + 1];
      }
      typedef typename QT::scratch_t st2 __attribute__((ext_vector_type(2)));
      *(st2*)(out + ((int64_t)m * ldo + n) * 2) = st2{(typename QT::scratch_t)a, (typename QT::scratch_t)b};
    }
  }
}

template <class QT, int MT, int WAVES>
int launch_linear_mt(const void* x, const void* w, const void* bias, void* out, int32_t M, int32_t N, int32_t K, int64_t ldx, int64_t ldw,
                     int64_t ldo, hipStream_t stream) {
  const dim3 grid((N + kLinCols - 1) / kLinCols, (M + 16 * MT - 1) / (16 * MT)), block(64 * WAVES);
  const auto* b = (const typename QT::scratch_t*)bias;
  hipLaunchKernelGGL((fdb_linear_kernel<QT, MT, WAVES>), grid, block, 0, stream, (const char*)x, (const char*)w, b, (char*)out, M, N, K, ldx, ldw, ldo);
  return (int)hipGetLastError();
}

template <class QT>
int launch_linear(const void* x, const void* w, const void* bias, void* out, int32_t M, int32_t N, int32_t K, int64_t ldx, int64_t ldw,
                  int64_t ldo, hipStream_t stream) {
  // sixteen waves where the contraction gives each of them more than one turn of four steps
  const bool deep = K > 32 * 4 * 8;
  if (M <= 16) return deep ? launch_linear_mt<QT, 1, 16>(x, w, bias, out, M, N, K, ldx, ldw, ldo, stream)
                           : launch_linear_mt<QT, 1, 8>(x, w, bias, out, M, N, K, ldx, ldw, ldo, stream);
  return deep ? launch_linear_mt<QT, 2, 16>(x, w, bias, out, M, N, K, ldx, ldw, ldo, stream)
              : launch_linear_mt<QT, 2, 8>(x, w, bias, out, M, N, K, ldx, ldw, ldo, stream);
}

}  // namespace

int fdb_launch_linear(const void* x, const void* w, const void* bias, void* out, int32_t M, int32_t N, int32_t K, int64_t ldx, int64_t ldw,
                      int64_t ldo, int dtype, void* stream) {
  if (dtype == FDB_BF16) return launch_linear<Bf16Tr>(x, w, bias, out, M, N, K, ldx, ldw, ldo, (hipStream_t)stream);
  if (dtype == FDB_F16) return launch_linear<F16Tr>(x, w, bias, out, M, N, K, ldx, ldw, ldo, (hipStream_t)stream);
  return FDB_ERR_DTYPE;
}

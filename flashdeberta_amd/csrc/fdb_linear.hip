// The linear layer in front of the attention for a batch of few rows, 16-bit types.
//
// Products of many rows are hipBLASLt's; a product of a few rows is latency, and a call of that library costs the host 8 us where a
// launch costs 2.5.  Up to 32 rows fdb_linear_kernel streams the weights: one workgroup per 16 output columns, eight or
// sixteen waves that share the contraction, so that even a [768 x 768] weight is on its way through 48 x 8 waves at once, each
// with four steps' loads in flight.  In a replayed graph, [24 x 768] . [768 x 2304]: 4.0 us against hipBLASLt's 4.8.
// Beyond that fdb_linear_tile_kernel (64 x 64 outputs per workgroup); [64 / 256 x 768] . [768 x 2304] 6.6 / 6.9 us against
// 5.7 / 6.6, level with the library on the GPU while one round of workgroups does it, and 8 us less on the host.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "fdb_device.h"
#include "fdb_kernels.h"
#include "../../include/fdb.h"

using namespace fdb;

namespace {

constexpr int kLinCols = 16;

__device__ __forceinline__ f32x4 mma16(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x4 mma16(f16x8 a, f16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

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

// The same product tiled: 64 x 64 outputs per workgroup, for the row counts between the kernel above (whose every 64 rows
// read the weights, and whose lanes fetch the rows of x once per 16 columns) and the sizes at which hipBLASLt's larger tiles win.
// Two teams of four waves (2 x 2 blocks of 32 x 32) take alternate 64-wide steps of the contraction, each with three LDS buffers
// filled straight from global memory two steps ahead: 24 - 48 workgroups per 64 rows have to hide the latency of their own loads.
constexpr int kTileBytes = 64 * 128;                // 64 rows of 64 16-bit elements, unpadded, slot (row, s) = chunk s ^ swz(row)
constexpr int kTileBufs = 3, kTileTeams = 2;        // (four teams of two buffers, three of three: no faster)
constexpr int kTileLds = kTileTeams * kTileBufs * 2 * kTileBytes;
static_assert(kTileLds <= 160 * 1024, "LDS budget");
__device__ __forceinline__ int swz(int row) { return 4 * ((row >> 1) & 1) | ((row >> 2) & 3); }

template <class QT>
__global__ __launch_bounds__(256 * kTileTeams) void fdb_linear_tile_kernel(const char* __restrict__ x, const char* __restrict__ w,
                                                                 const typename QT::scratch_t* __restrict__ bias, char* __restrict__ out,
                                                                 int32_t M, int32_t N, int32_t K, int64_t ldx, int64_t ldw, int64_t ldo) {
  using frag = typename QT::frag;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 31, g = lane >> 5;
  const int team = wave >> 2, tw = wave & 3, wn = tw & 1, wm = tw >> 1;
  const int n0 = blockIdx.x * 64, m0 = blockIdx.y * 64;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LDS_AS char*)smem + (uint32_t)team * (kTileBufs * 2 * kTileBytes);
  // this lane's part of a step's loads: a wave instruction fills 8 rows, wave tw the groups tw and tw + 4 of either tile
  uint32_t woff[2], xoff[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int row = 8 * (tw + 4 * c) + (lane >> 3);
    const uint32_t chunk = (uint32_t)(((lane & 7) ^ swz(row)) * 16);
    woff[c] = (uint32_t)(min(n0 + row, N - 1) - n0) * (uint32_t)(ldw * 2) + chunk;  // rows past the end re-read the last one
    xoff[c] = (uint32_t)(min(m0 + row, M - 1) - m0) * (uint32_t)(ldx * 2) + chunk;
  }
  const char* wt = w + (int64_t)n0 * ldw * 2;
  const char* xt = x + (int64_t)m0 * ldx * 2;
  const int steps = K / 64, turns = (steps + kTileTeams - 1) / kTileTeams;
  auto fill = [&](int turn) __attribute__((always_inline)) {
    const int s = min(turn * kTileTeams + team, steps - 1);  // past the end: loads nobody uses, so that every turn waits alike
    const uint32_t dst = lds0 + (uint32_t)(turn % kTileBufs) * (2 * kTileBytes) + (uint32_t)tw * 1024u;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      dma16sn(wt + (int64_t)s * 128, woff[c], dst + c * 4096);
      dma16sn(xt + (int64_t)s * 128, xoff[c], dst + kTileBytes + c * 4096);
    }
  };
  f32x16 acc = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int t = 0; t < kTileBufs - 1; ++t) fill(t);
  const uint32_t wrow = (uint32_t)((32 * wn + li) * 128), xrow = (uint32_t)(kTileBytes + (32 * wm + li) * 128), f = (uint32_t)swz(li);
  for (int t = 0; t < turns; ++t) {
    wait_vmcnt<4 * (kTileBufs - 2)>();  // this wave's loads of turn t have landed (those of the turns after it may still fly)
    __syncthreads();  // ... and everybody's; the buffer of turn t - 1 is free
    const uint32_t b = lds0 + (uint32_t)(t % kTileBufs) * (2 * kTileBytes);
    frag wf[4], xf[4];  // asked for ahead of the loads below, whose issue (64 clocks each) their latency then hides behind
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t slot = ((uint32_t)(2 * k + g) ^ f) * 16;
      wf[k] = *(LDS_AS const frag*)(uintptr_t)(b + wrow + slot);
      xf[k] = *(LDS_AS const frag*)(uintptr_t)(b + xrow + slot);
    }
    __builtin_amdgcn_sched_barrier(0);
    fill(t + kTileBufs - 1);
    __builtin_amdgcn_sched_barrier(0);
    if (t * kTileTeams + team < steps) {
#pragma unroll
      for (int k = 0; k < 4; ++k) acc = QT::mma(wf[k], xf[k], acc);  // rows: output columns, columns: rows of x
    }
  }
  wait_vmcnt<0>();
  __syncthreads();
  float* other = (float*)smem + tw * 1024 + lane;  // the other teams' sums, [team][wave][register][lane]
  if (team > 0) {
#pragma unroll
    for (int v = 0; v < 16; ++v) other[(team - 1) * 4096 + 64 * v] = acc[v];
  }
  __syncthreads();
  if (team > 0) return;
#pragma unroll
  for (int t = 0; t < kTileTeams - 1; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] += other[t * 4096 + 64 * v];
  const int m = m0 + 32 * wm + li;
  if (m >= M) return;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int n = n0 + 32 * wn + 8 * q + 4 * g;
    f32x4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      r[e] = acc[4 * q + e];
      if (bias && n + e < N) r[e] += (float)bias[n + e];
    }
    if (n < N) QT::store4(out + ((int64_t)m * ldo + n) * 2, r[0], r[1], r[2], r[3]);  // N is a multiple of 4
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
int launch_linear_tile(const void* x, const void* w, const void* bias, void* out, int32_t M, int32_t N, int32_t K, int64_t ldx, int64_t ldw,
                       int64_t ldo, hipStream_t stream) {
  auto kern = fdb_linear_tile_kernel<QT>;
  static std::atomic<uint64_t> lds_set{0};
  const hipError_t e = fdb_set_lds_once((const void*)kern, kTileLds, lds_set);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kern, dim3((N + 63) / 64, (M + 63) / 64), dim3(256 * kTileTeams), kTileLds, stream, (const char*)x, (const char*)w,
                     (const typename QT::scratch_t*)bias, (char*)out, M, N, K, ldx, ldw, ldo);
  return (int)hipGetLastError();
}

template <class QT>
int launch_linear(const void* x, const void* w, const void* bias, void* out, int32_t M, int32_t N, int32_t K, int64_t ldx, int64_t ldw,
                  int64_t ldo, hipStream_t stream) {
  if (M > 32 && K % 64 == 0 && N % 4 == 0 && ldo % 4 == 0 && 64 * ldx * 2 <= INT32_MAX && 64 * ldw * 2 <= INT32_MAX)
    return launch_linear_tile<QT>(x, w, bias, out, M, N, K, ldx, ldw, ldo, stream);
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

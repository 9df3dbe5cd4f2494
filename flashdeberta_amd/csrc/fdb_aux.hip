// Small helper kernels around the fused attention: the varlen q-tile work-list built on the
// device from cu_seqlens (the reference builds it in a Python loop with one host sync per
// sequence, src/flashdeberta/ops/flash_attention_varlen.py:71-83) and the per-head absmax ->
// OCP e4m3 quantisation of the FP8 Q/K variant.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <stdint.h>

#include "fdb_device.h"
#include "fdb_kernels.h"
#include "../../include/fdb.h"

using namespace fdb;

namespace {

constexpr int kWlThreads = 1024;
constexpr int kWlSortMax = 1024;  // batches up to this size get their tiles ordered by sequence length
constexpr int kWlLanes = 16;      // threads that place a sequence together

// wl[0] = number of tiles, wl[1] = 0, then (sequence, first row) pairs: the tiles of the longest
// sequence first (ties in sequence order), so that a launch starts on the workgroups with the most
// key tiles and ends on the short ones.  Sixteen threads place a sequence: each sums the tiles of every sixteenth
// of the sequences that come before it in that order (the lengths in LDS), and writes every sixteenth of its pairs.  The launch is latency: a
// thread per sequence, which went through all lengths and wrote all pairs itself, 8.4 us where this takes 5.6 (64 sequences).
// Larger batches keep the sequence order and a prefix sum.
__global__ __launch_bounds__(kWlThreads) void fdb_worklist_kernel(const int32_t* __restrict__ cu, int32_t batch,
                                                                  int32_t* __restrict__ wl, int32_t max_tiles) {
  __shared__ int32_t part[kWlThreads];
  __shared__ int32_t lens[kWlSortMax];
  const int t = threadIdx.x;
  if (batch <= kWlSortMax) {
    for (int b = t; b < batch; b += kWlThreads) lens[b] = max(cu[b + 1] - cu[b], 0);
    __syncthreads();
    const int j = t % kWlLanes;
    for (int b = t / kWlLanes; b < batch; b += kWlThreads / kWlLanes) {   // a sequence's threads stay together
      const int len = lens[b];
      int32_t pos = 0, total = 0;
      for (int c = j; c < batch; c += kWlLanes) {
        const int lc = lens[c], tiles = (lc + FDB_BM - 1) / FDB_BM;
        total += tiles;
        if (lc > len || (lc == len && c < b)) pos += tiles;
      }
#pragma unroll
      for (int x = 1; x < kWlLanes; x <<= 1) {
        pos += __shfl_xor(pos, x);
        total += __shfl_xor(total, x);
      }
      if (b == 0 && j == 0) {
        wl[0] = min(total, max_tiles);
        wl[1] = 0;
      }
      pos += j;
      for (int m0 = j * FDB_BM; m0 < len; m0 += kWlLanes * FDB_BM, pos += kWlLanes)
        if (pos < max_tiles) {
          wl[2 + 2 * pos] = b;
          wl[3 + 2 * pos] = m0;
        }
    }
    return;
  }
  const int per = (batch + kWlThreads - 1) / kWlThreads;
  const int b_lo = min(batch, t * per), b_hi = min(batch, b_lo + per);
  int32_t cnt = 0;
  for (int b = b_lo; b < b_hi; ++b) cnt += (max(cu[b + 1] - cu[b], 0) + FDB_BM - 1) / FDB_BM;
  part[t] = cnt;
  __syncthreads();
  // exclusive scan over the threads' counts (Hillis-Steele)
  for (int off = 1; off < kWlThreads; off <<= 1) {
    int32_t add = (t >= off) ? part[t - off] : 0;
    __syncthreads();
    part[t] += add;
    __syncthreads();
  }
  int32_t pos = part[t] - cnt;
  if (t == kWlThreads - 1) {
    wl[0] = min(part[t], max_tiles);
    wl[1] = 0;
  }
  for (int b = b_lo; b < b_hi; ++b) {
    const int len = max(cu[b + 1] - cu[b], 0);
    for (int m0 = 0; m0 < len; m0 += FDB_BM, ++pos)
      if (pos < max_tiles) {
        wl[2 + 2 * pos] = b;
        wl[3 + 2 * pos] = m0;
      }
  }
}

// Column sums in two launches without atomics: every workgroup sums a share of the rows of x and of y for 512 columns (eight per
// lane, a wave a row at a time, the four waves' sums added in LDS) and leaves one row of fp32 sums; the second launch adds those.
// Bound by one read of x and y: 21 MB at [4096 x 2304] and [512 x 1536], 6.2 us (12.4 with all rows of y in one share).
constexpr int kColShare = 64;   // rows per workgroup: a share of 64 rows keeps the launch wide, 64 partial rows at 4096

template <class QT>
__global__ __launch_bounds__(256) void fdb_column_sums_kernel(const char* __restrict__ x, int64_t x_rows, int64_t x_cols, const char* __restrict__ y,
                                                              int64_t y_rows, int64_t y_cols, float* __restrict__ ws) {
  __shared__ float part[4][512];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int share = blockIdx.y;
  const int64_t col = (int64_t)blockIdx.x * 512 + 8 * lane, r0 = (int64_t)share * kColShare;
  f32x8 acc = {0, 0, 0, 0, 0, 0, 0, 0};
  auto add = [&](const char* src, int64_t rows, int64_t cols) __attribute__((always_inline)) {
    const int64_t r1 = min(rows, r0 + kColShare);
    if (col < cols) {
#pragma unroll 8
      for (int64_t r = r0 + wave; r < r1; r += 4) acc += QT::to_f32(QT::load(src + (r * cols + col) * 2));
    }
  };
  add(x, x_rows, x_cols);
  if (y) add(y, y_rows, y_cols);
#pragma unroll
  for (int e = 0; e < 8; ++e) part[wave][8 * lane + e] = acc[e];
  __syncthreads();
  for (int c = threadIdx.x; c < 512; c += 256)
    if ((int64_t)blockIdx.x * 512 + c < x_cols)
      ws[(int64_t)share * x_cols + (int64_t)blockIdx.x * 512 + c] = part[0][c] + part[1][c] + part[2][c] + part[3][c];
}

template <class QT>
__global__ __launch_bounds__(256) void fdb_column_sums_end_kernel(const float* __restrict__ ws, int64_t cols, int parts, typename QT::scratch_t* __restrict__ out) {
  // 64 columns per workgroup, the parts dealt to its four waves
  __shared__ float part[4][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t col = (int64_t)blockIdx.x * 64 + lane;
  float sum = 0.f;
  if (col < cols) {
#pragma unroll 8
    for (int s = wave; s < parts; s += 4) sum += ws[(int64_t)s * cols + col];
  }
  part[wave][lane] = sum;
  __syncthreads();
  if (wave == 0 && col < cols) out[col] = (typename QT::scratch_t)(part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane]);
}

template <class QT>
int launch_column_sums(const void* x, int64_t x_rows, int64_t x_cols, const void* y, int64_t y_rows, int64_t y_cols, void* out, float* ws,
                       hipStream_t stream) {
  const int parts = fdb_column_sum_parts(y && y_rows > x_rows ? y_rows : x_rows);
  hipLaunchKernelGGL(fdb_column_sums_kernel<QT>, dim3((unsigned)((x_cols + 511) / 512), (unsigned)parts), dim3(256), 0, stream,
                     (const char*)x, x_rows, x_cols, (const char*)y, y_rows, y_cols, ws);
  hipLaunchKernelGGL(fdb_column_sums_end_kernel<QT>, dim3((unsigned)((x_cols + 63) / 64)), dim3(256), 0, stream, ws, x_cols, parts,
                     (typename QT::scratch_t*)out);
  return (int)hipGetLastError();
}

// Bounds of a padded batch's real tokens, one workgroup per row: first and last non-zero mask element and their count.
// One pass over the mask in one launch; the same as a chain of torch reductions is ten launches of 3 us each.
template <class T>
__global__ __launch_bounds__(256) void fdb_mask_bounds_kernel(const T* __restrict__ mask, T ignore, int64_t stride_b, int64_t stride_l,
                                                              int32_t length, int32_t* __restrict__ start, int32_t* __restrict__ len) {
  const T* row = mask + (int64_t)blockIdx.x * stride_b;
  int32_t first = length, last = -1, count = 0;
  for (int32_t l = threadIdx.x; l < length; l += 256)
    if ((row[(int64_t)l * stride_l] & (T)~ignore) != 0) {
      first = min(first, l);
      last = l;
      ++count;
    }
  __shared__ int32_t part[3][4];
  for (int off = 32; off > 0; off >>= 1) {
    first = min(first, __shfl_xor(first, off));
    last = max(last, __shfl_xor(last, off));
    count += __shfl_xor(count, off);
  }
  if ((threadIdx.x & 63) == 0) {
    part[0][threadIdx.x >> 6] = first;
    part[1][threadIdx.x >> 6] = last;
    part[2][threadIdx.x >> 6] = count;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) {
      first = min(first, part[0][w]);
      last = max(last, part[1][w]);
      count += part[2][w];
    }
    start[blockIdx.x] = count > 0 ? first : 0;
    len[blockIdx.x] = count > 0 && last - first + 1 != count ? -1 : count;
  }
}

__global__ void fdb_fill_u32(uint32_t* p, int n, uint32_t v) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__device__ __forceinline__ float bf16_bits_to_f32(uint16_t b) { return __builtin_bit_cast(float, (uint32_t)b << 16); }

// grid (token blocks, heads); each thread owns 8 consecutive d of one token.  One atomic per
// workgroup: all of a head's atomics hit one address and are served one after the other (one per wave
// from 1024 workgroups per head took 560 us for 50 MB), so the launch also keeps the workgroups few.
// One or two tensors of one shape and one set of strides per launch (blockIdx.z picks the tensor; its absmax words
// follow the first tensor's).
struct QuantPair {
  const uint16_t* x[2];
  uint8_t* y[2];
  float* scale[2];
};

// The rows (token, head) of a tensor, D / 8 lanes a row, neighbouring lanes neighbouring heads of a token: what a workgroup asks for lies
// together where the heads do.  The grid is a multiple of the number of heads, so that a thread keeps its head and walks tokens by
// one step; it has `kAhead` loads of sixteen bytes under way.  Bound by one read of the tensors.  A head per workgroup, a load
// at a time, fetched 128 bytes here and there: [4 x 8192 x 12 x 64] twice, absmax 47 -> 26.5 us (3.8 TB/s); the quantiser, at 4.4 TB/s
// in and out either way, stays at 34.
template <int D>
struct RowWalk {
  static constexpr int kLanes = D / 8, kRows = 256 / kLanes, kAhead = 8;
  int h, c;        // head; first element of this lane's sixteen bytes
  int64_t t, step;  // first token, and from one to the next
  __device__ RowWalk(int heads) {
    const uint32_t u = blockIdx.x * kRows + threadIdx.x / kLanes;
    h = (int)(u % (uint32_t)heads);
    c = (int)(threadIdx.x % kLanes) * 8;
    t = u / (uint32_t)heads;
    step = (int64_t)(gridDim.x / (uint32_t)heads) * kRows;
  }
  // f(token, sixteen bytes) for every token of this thread
  template <class F>
  __device__ __forceinline__ void each(const uint16_t* __restrict__ x, int64_t st, int64_t sh, int32_t tokens, const F& f) const {
    const uint16_t* row = x + h * sh + c;
    for (int64_t first = t; first < tokens; first += kAhead * step) {
      uint4 raw[kAhead];
#pragma unroll
      for (int n = 0; n < kAhead; ++n) raw[n] = *(const uint4*)(row + min(first + n * step, (int64_t)tokens - 1) * st);
#pragma unroll
      for (int n = 0; n < kAhead; ++n)
        if (first + n * step < tokens) f(first + n * step, raw[n]);
    }
  }
};

template <int D>
__global__ __launch_bounds__(256) void fdb_absmax_kernel(const QuantPair pr, int64_t st, int64_t sh, uint32_t* __restrict__ absmax_all,
                                                         int32_t tokens, int32_t heads) {
  using W = RowWalk<D>;
  const W w(heads);
  float m = 0.f;
  w.each(pr.x[blockIdx.z], st, sh, tokens, [&](int64_t, const uint4& raw) __attribute__((always_inline)) {
    const uint32_t v[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      m = fmaxf(m, fabsf(bf16_bits_to_f32((uint16_t)(v[e] & 0xffffu))));
      m = fmaxf(m, fabsf(bf16_bits_to_f32((uint16_t)(v[e] >> 16))));
    }
  });
  for (int off = W::kLanes / 2; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  __shared__ float row_max[W::kRows];
  if (w.c == 0) row_max[threadIdx.x / W::kLanes] = m;
  __syncthreads();
  // rows `heads` apart belong to one head: one atomic each
  if (w.c == 0 && (int)threadIdx.x / W::kLanes < heads) {
    for (int r = (int)threadIdx.x / W::kLanes + heads; r < W::kRows; r += heads) m = fmaxf(m, row_max[r]);
    atomicMax(absmax_all + blockIdx.z * heads + w.h, __builtin_bit_cast(uint32_t, m));  // m >= 0: bit order = value order
  }
}

template <int D>
__global__ __launch_bounds__(256) void fdb_quant_kernel(const QuantPair pr, int64_t st, int64_t sh, int64_t yst, int64_t ysh,
                                                        const uint32_t* __restrict__ absmax_all, int32_t tokens, int32_t heads) {
  const RowWalk<D> w(heads);
  const float amax = fmaxf(__builtin_bit_cast(float, absmax_all[blockIdx.z * heads + w.h]), 1e-12f);
  const float sc = amax / 448.0f;
  if (w.t == 0 && w.c == 0) pr.scale[blockIdx.z][w.h] = sc;
  uint8_t* __restrict__ y = pr.y[blockIdx.z] + w.h * ysh + w.c;
  w.each(pr.x[blockIdx.z], st, sh, tokens, [&](int64_t t, const uint4& raw) __attribute__((always_inline)) {
    const uint32_t v[4] = {raw.x, raw.y, raw.z, raw.w};
    float f[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[2 * e] = fminf(fmaxf(bf16_bits_to_f32((uint16_t)(v[e] & 0xffffu)) / sc, -448.f), 448.f);
      f[2 * e + 1] = fminf(fmaxf(bf16_bits_to_f32((uint16_t)(v[e] >> 16)) / sc, -448.f), 448.f);
    }
    uint32_t outw[2];
    // two e4m3 bytes per conversion: low half of the word first, then the high half
    outw[0] = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], 0, false);
    outw[0] = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], outw[0], true);
    outw[1] = __builtin_amdgcn_cvt_pk_fp8_f32(f[4], f[5], 0, false);
    outw[1] = __builtin_amdgcn_cvt_pk_fp8_f32(f[6], f[7], outw[1], true);
    *(uint2*)(y + t * yst) = uint2{outw[0], outw[1]};
  });
}

// The inverse map, to bf16: x = bf16_rne(e4m3(y) * scale[h]).  Eight elements per thread.
template <int D>
__global__ __launch_bounds__(256) void fdb_dequant_kernel(const uint8_t* __restrict__ y, int64_t yst, int64_t ysh,
                                                          const float* __restrict__ scale, uint16_t* __restrict__ x,
                                                          int64_t st, int64_t sh, int32_t tokens) {
  constexpr int CPT = D / 8;
  const int h = blockIdx.y;
  const float sc = scale[h];
  for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < (int64_t)tokens * CPT;
       c += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = c / CPT;
    const int cc = (int)(c % CPT);
    const uint2 raw = *(const uint2*)(y + t * yst + h * ysh + cc * 8);
    const uint32_t w[2] = {raw.x, raw.y};
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8(w[e], false), hi = __builtin_amdgcn_cvt_pk_f32_fp8(w[e], true);
      typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
      typedef float f2 __attribute__((ext_vector_type(2)));
      o[2 * e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{lo[0] * sc, lo[1] * sc}, bf2));
      o[2 * e + 1] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{hi[0] * sc, hi[1] * sc}, bf2));
    }
    *(uint4*)(x + t * st + h * sh + cc * 8) = uint4{o[0], o[1], o[2], o[3]};
  }
}

}  // namespace

int fdb_launch_dequant(const void* y, int64_t y_st, int64_t y_sh, const float* scale, void* x, int64_t x_st, int64_t x_sh,
                       int32_t tokens, int32_t heads, int32_t head_dim, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  const int64_t chunks = (int64_t)tokens * head_dim / 8;
  int gx = (int)((chunks + 255) / 256);
  if (gx > 2048) gx = 2048;
  if (gx < 1) gx = 1;
#define FDB_DQ(DD)                                                                                              \
  hipLaunchKernelGGL(fdb_dequant_kernel<DD>, dim3(gx, heads), dim3(256), 0, stream, (const uint8_t*)y, y_st,    \
                     y_sh, scale, (uint16_t*)x, x_st, x_sh, tokens);
  switch (head_dim) {
    case 32: FDB_DQ(32) break;
    case 64: FDB_DQ(64) break;
    case 128: FDB_DQ(128) break;
    default: return -3;
  }
#undef FDB_DQ
  return (int)hipGetLastError();
}

namespace {
// Three weights and three biases under one another (blockIdx.y: which), sixteen bytes a lane, four lines a thread in flight: the two launches
// that torch's cat takes are 7.5 us for 3.5 MB, this one 3.
struct Join {
  const u32x4 *w[3], *b[3];
};
__global__ __launch_bounds__(256) void fdb_join_kernel(const Join from, u32x4* __restrict__ w, u32x4* __restrict__ b, int64_t w_len, int64_t b_len) {
  const int which = blockIdx.y;
  const u32x4* src = which == 0 ? from.w[0] : which == 1 ? from.w[1] : from.w[2];
  const int64_t at = (int64_t)blockIdx.x * 1024 + threadIdx.x;
  u32x4 v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (at + 256 * j < w_len) v[j] = src[at + 256 * j];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (at + 256 * j < w_len) w[which * w_len + at + 256 * j] = v[j];
  if (at < b_len) b[which * b_len + at] = (which == 0 ? from.b[0] : which == 1 ? from.b[1] : from.b[2])[at];
}
}  // namespace
int fdb_launch_join(const void* const w[3], const void* const b[3], void* w_out, void* b_out, int64_t w_bytes, int64_t b_bytes, void* stream) {
  Join from;
  for (int i = 0; i < 3; ++i) from.w[i] = (const u32x4*)w[i], from.b[i] = (const u32x4*)b[i];
  hipLaunchKernelGGL(fdb_join_kernel, dim3((unsigned)((w_bytes / 16 + 1023) / 1024), 3), dim3(256), 0, (hipStream_t)stream, from, (u32x4*)w_out, (u32x4*)b_out, w_bytes / 16,
                     b_bytes / 16);
  return (int)hipGetLastError();
}

int fdb_column_sum_parts(int64_t rows) { return (int)((rows + kColShare - 1) / kColShare); }

int fdb_launch_column_sums(const void* x, int64_t x_rows, int64_t x_cols, const void* y, int64_t y_rows, int64_t y_cols, void* out, float* ws,
                           int dtype, void* stream) {
  if (dtype == FDB_BF16) return launch_column_sums<fdb::Bf16Tr>(x, x_rows, x_cols, y, y_rows, y_cols, out, ws, (hipStream_t)stream);
  if (dtype == FDB_F16) return launch_column_sums<fdb::F16Tr>(x, x_rows, x_cols, y, y_rows, y_cols, out, ws, (hipStream_t)stream);
  return FDB_ERR_DTYPE;
}

int fdb_launch_mask_bounds(const void* mask, int elem_size, bool is_float, int64_t stride_b, int64_t stride_l, int32_t batch, int32_t length,
                           int32_t* start, int32_t* len, void* stream) {
#define FDB_MB(T)                                                                                                     \
  hipLaunchKernelGGL(fdb_mask_bounds_kernel<T>, dim3(batch), dim3(256), 0, (hipStream_t)stream, (const T*)mask,      \
                     is_float ? (T)((T)1 << (8 * sizeof(T) - 1)) : (T)0, stride_b, stride_l, length, start, len);
  switch (elem_size) {
    case 1: FDB_MB(uint8_t) break;
    case 2: FDB_MB(uint16_t) break;
    case 4: FDB_MB(uint32_t) break;
    case 8: FDB_MB(uint64_t) break;
    default: return FDB_ERR_DTYPE;
  }
#undef FDB_MB
  return (int)hipGetLastError();
}

int fdb_launch_worklist(const int32_t* cu, int32_t batch, int32_t* wl, int32_t max_tiles, void* stream) {
  hipLaunchKernelGGL(fdb_worklist_kernel, dim3(1), dim3(kWlThreads), 0, (hipStream_t)stream, cu, batch, wl, max_tiles);
  return (int)hipGetLastError();
}

// ---- merge of partial results -------------------------------------------------------------------------
// After a near launch whose workgroups each took a share of a query tile's steps: every partial result is
// a set of rows normalised over the keys it saw plus their log-sum-exp (-inf: none seen).  The far ones
// (when p.far_done: the first in out / lse, the others in workspace slots 0 .. far_parts-2) and the near
// ones (slots far_parts-1 ..) are combined with weights exp(lse_s - max) into out and lse.  One thread
// per eight elements of a (token, head) row; padded rows of a fixed-layout batch are left alone.
//
// What bounds these two launches is how long one thread takes: a few MB are read and written by threads that live once.  So the place of a row is found with
// 32-bit numbers instead of three 64-bit divisions a thread, and what a thread reads is asked for together, the weights of all parts and the values of up to four.
// Not of all eight that the far and near launch may leave: their values and addresses take 234 registers, two waves a SIMD instead of eight, whose second round
// cost more than one trip to memory.  us of the whole call, 12 heads: a part's values when its turn comes -> all eight ahead -> four
//   bf16, three shares  1 x 1536  43.9 (two shares) -> 38.1 -> 35.4      e4m3, two shares  2 x 1280  37.7 -> 38.2 -> 36.2
//   bf16, four shares, 4 heads  1 x 2048  27.0 -> 25.3 -> 24.3          e4m3, two shares  1 x 2048  49.0 -> 50.2 -> 48.4
//   bf16, near_splits = 4  8 x 2048  282 -> 297 -> 278                  fp32, four parts (the one-kernel mode's merge, which has four at most)  1 x 512  35.1 -> 33.8
namespace {

// Where a thread's row lies: CPR threads a row, in whole rows.
struct MergeRow {
  int64_t row, tok;   // tok * H + h
  int32_t h, b, l, cc;
};
template <int CPR>
__device__ __forceinline__ MergeRow merge_row(const FdbKParams& p) {
  MergeRow r;
  const int k = (int)threadIdx.x / CPR;
  r.cc = (int)threadIdx.x % CPR;
  const int64_t row0 = (int64_t)blockIdx.x * (256 / CPR);
  r.row = row0 + k;
  const int64_t tok0 = row0 <= INT32_MAX ? quick_div((int)row0, p.H) : row0 / p.H;
  const int h = (int)(row0 - tok0 * p.H) + k, tokens = quick_div(h, p.H);
  r.h = h - tokens * p.H;
  r.tok = tok0 + tokens;
  r.b = r.l = 0;
  if (!p.cu) {
    const int b0 = quick_div((int)tok0, p.L), l = (int)tok0 - b0 * p.L + tokens, rows = quick_div(l, p.L);   // tokens number at most INT32_MAX
    r.b = b0 + rows;
    r.l = l - rows * p.L;
  }
  return r;
}
// ... and whether it holds a token (rows outside the real tokens were written by the attention launch)
__device__ __forceinline__ bool merge_row_is_real(const FdbKParams& p, const MergeRow& r) {
  if (p.cu) return true;
  const int t0 = p.seq_start ? min(max(p.seq_start[r.b], 0), p.L) : 0;
  const int len = p.seq_len ? min(max(p.seq_len[r.b], 0), p.L - t0) : p.L;
  return r.l >= t0 && r.l < t0 + len;
}

template <class VT>
__global__ __launch_bounds__(256) void fdb_merge_kernel(const FdbKParams p) {
  constexpr int D = 64, CPR = D / 8, RB = D * 2;
  read_arguments(p);
  const MergeRow r = merge_row<CPR>(p);
  if (r.row >= p.ws_rows * p.H) return;
  char* dst = p.out + ((p.cu ? r.tok * p.o_st : (int64_t)r.b * p.o_sb + (int64_t)r.l * p.o_st) + (int64_t)r.h * p.o_sh) * 2 + r.cc * 16;
  constexpr int kMax = 2 * FDB_MAX_FAR_PARTS, kGroup = 4;
  const int n_far = p.far_done ? p.far_parts : 0, n = n_far + p.near_parts;
  // source s: far part s (s < n_far), else near part s - n_far
  auto slot_of = [&](int s) __attribute__((always_inline)) { return s < n_far ? s - 1 : p.far_parts - 1 + (s - n_far); };
  u32x4 part[kGroup];
  auto ask = [&](int first) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < kGroup; ++x) {
      const int slot = slot_of(first + x);
      if (first + x < n) part[x] = *(const u32x4*)(slot < 0 ? dst : ws_slot_out(p, slot, RB) + r.row * RB + r.cc * 16);
    }
  };
  float w[kMax], m = -INFINITY;
#pragma unroll
  for (int s = 0; s < kMax; ++s) {
    const int slot = slot_of(s);
    w[s] = -INFINITY;
    if (s < n) w[s] = (slot < 0 ? p.lse : ws_slot_lse(p, slot, RB))[r.row];
  }
  ask(0);
  if (!merge_row_is_real(p, r)) return;
#pragma unroll
  for (int s = 0; s < kMax; ++s) {
    w[s] *= 1.4426950408889634f;
    m = fmaxf(m, w[s]);
  }
  float denom = 0.f;
#pragma unroll
  for (int s = 0; s < kMax; ++s) {
    w[s] = (s < n && w[s] != -INFINITY) ? __builtin_amdgcn_exp2f(w[s] - m) : 0.f;
    denom += w[s];
  }
  const float inv = denom > 0.f ? 1.f / denom : 0.f;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int first = 0; first < kMax; first += kGroup) {
    if (first > 0) {
      if (first >= n) break;
      ask(first);
    }
#pragma unroll
    for (int x = 0; x < kGroup; ++x)
      if (first + x < n && w[first + x] > 0.f) {
        const f32x8 y = VT::to_f32(__builtin_bit_cast(typename VT::frag, part[x]));
        const float f = w[first + x] * inv;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = __builtin_fmaf(y[e], f, acc[e]);
      }
  }
  VT::store4(dst, acc[0], acc[1], acc[2], acc[3]);
  VT::store4(dst + 8, acc[4], acc[5], acc[6], acc[7]);
  if (r.cc == 0) p.lse[r.row] = denom > 0.f ? (m + __builtin_amdgcn_logf(denom)) * 0.6931471805599453f : -INFINITY;
}

}  // namespace

// The same for the one-kernel mode: p.key_parts partial results, all in the workspace, any element type and head_dim;
// one thread per four elements.
template <class VT, int D>
__global__ __launch_bounds__(256) void fdb_merge_parts_kernel(const FdbKParams p) {
  constexpr int CPR = D / 4, RB = D * VT::SZ;
  read_arguments(p);
  const MergeRow r = merge_row<CPR>(p);
  if (r.row >= p.ws_rows * p.H) return;
  char* dst = p.out + ((p.cu ? r.tok * p.o_st : (int64_t)r.b * p.o_sb + (int64_t)r.l * p.o_st) + (int64_t)r.h * p.o_sh + 4 * r.cc) * VT::SZ;
  float w[FDB_MAX_FAR_PARTS], m = -INFINITY;
  f32x4 part[FDB_MAX_FAR_PARTS];
#pragma unroll
  for (int s = 0; s < FDB_MAX_FAR_PARTS; ++s) {
    w[s] = -INFINITY;
    part[s] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (s < p.key_parts) {
      w[s] = ws_slot_lse(p, s, RB)[r.row];
      part[s] = VT::load4(ws_slot_out(p, s, RB) + r.row * RB + r.cc * 4 * VT::SZ);
    }
  }
  if (!merge_row_is_real(p, r)) return;
#pragma unroll
  for (int s = 0; s < FDB_MAX_FAR_PARTS; ++s) {
    w[s] *= 1.4426950408889634f;
    m = fmaxf(m, w[s]);
  }
  float denom = 0.f;
#pragma unroll
  for (int s = 0; s < FDB_MAX_FAR_PARTS; ++s) {
    w[s] = w[s] != -INFINITY ? __builtin_amdgcn_exp2f(w[s] - m) : 0.f;
    denom += w[s];
  }
  // a real token sees a key: none above 0 is a row of NaN, or of scores that are all -inf and have no soft-max
  const float inv = denom > 0.f ? 1.f / denom : __builtin_nanf("");
  float acc[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = denom > 0.f ? 0.f : inv;
#pragma unroll
  for (int s = 0; s < FDB_MAX_FAR_PARTS; ++s)
    if (s < p.key_parts && w[s] > 0.f) {
      const float f = w[s] * inv;
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(part[s][e], f, acc[e]);
    }
  VT::store4(dst, acc[0], acc[1], acc[2], acc[3]);
  if (r.cc == 0 && p.lse) p.lse[r.row] = denom > 0.f ? (m + __builtin_amdgcn_logf(denom)) * 0.6931471805599453f : inv;
}

template <class VT>
int launch_merge_parts_d(const FdbKParams& p, int head_dim, hipStream_t stream) {
  const int64_t threads = p.ws_rows * p.H * (head_dim / 4);
  const unsigned blocks = (unsigned)((threads + 255) / 256);
  switch (head_dim) {
    case 32: hipLaunchKernelGGL((fdb_merge_parts_kernel<VT, 32>), dim3(blocks), dim3(256), 0, stream, p); break;
    case 64: hipLaunchKernelGGL((fdb_merge_parts_kernel<VT, 64>), dim3(blocks), dim3(256), 0, stream, p); break;
    case 128: hipLaunchKernelGGL((fdb_merge_parts_kernel<VT, 128>), dim3(blocks), dim3(256), 0, stream, p); break;
    default: return FDB_ERR_HEAD_DIM;
  }
  return (int)hipGetLastError();
}

int fdb_launch_merge_parts(const FdbKParams& p, int dtype, int head_dim, void* stream) {
  if (dtype == FDB_F32) return launch_merge_parts_d<fdb::F32Tr>(p, head_dim, (hipStream_t)stream);
  if (dtype == FDB_F16) return launch_merge_parts_d<fdb::F16Tr>(p, head_dim, (hipStream_t)stream);
  if (dtype == FDB_BF16 || dtype == FDB_FP8_E4M3) return launch_merge_parts_d<fdb::Bf16Tr>(p, head_dim, (hipStream_t)stream);  // v's type
  return FDB_ERR_DTYPE;
}

int fdb_launch_merge(const FdbKParams& p, int dtype, void* stream) {
  const int64_t chunks = p.ws_rows * p.H * 8;
  const unsigned blocks = (unsigned)((chunks + 255) / 256);
  if (dtype == FDB_BF16)
    hipLaunchKernelGGL(fdb_merge_kernel<fdb::Bf16Tr>, dim3(blocks), dim3(256), 0, (hipStream_t)stream, p);
  else if (dtype == FDB_F16)
    hipLaunchKernelGGL(fdb_merge_kernel<fdb::F16Tr>, dim3(blocks), dim3(256), 0, (hipStream_t)stream, p);
  else
    return FDB_ERR_UNSUPPORTED;
  return (int)hipGetLastError();
}

int fdb_launch_quant(const void* x0, const void* x1, int64_t x_st, int64_t x_sh, void* y0, void* y1, int64_t y_st, int64_t y_sh,
                     float* scale0, float* scale1, uint32_t* absmax_ws, int32_t tokens, int32_t heads, int32_t head_dim,
                     void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  const unsigned n = x1 ? 2u : 1u;
  QuantPair pr;
  pr.x[0] = (const uint16_t*)x0; pr.x[1] = (const uint16_t*)x1;
  pr.y[0] = (uint8_t*)y0; pr.y[1] = (uint8_t*)y1;
  pr.scale[0] = scale0; pr.scale[1] = scale1;
  hipLaunchKernelGGL(fdb_fill_u32, dim3((n * heads + 255) / 256), dim3(256), 0, stream, absmax_ws, (int)(n * heads), 0u);
  // workgroups: a multiple of the heads, eight tokens a thread where there are as many, at most about 384 (absmax: an atomic per
  // head and workgroup) or 1536 (quantiser) per tensor
  const int64_t per = 8 * (int64_t)(256 / (head_dim / 8)), want = ((int64_t)tokens + per - 1) / per;
  const auto grid = [&](int most) { return (unsigned)(std::max<int64_t>(1, std::min<int64_t>(want, most / heads)) * heads); };
#define FDB_Q(DD)                                                                                                                 \
  hipLaunchKernelGGL(fdb_absmax_kernel<DD>, dim3(grid(384), 1, n), dim3(256), 0, stream, pr, x_st, x_sh, absmax_ws, tokens, heads); \
  hipLaunchKernelGGL(fdb_quant_kernel<DD>, dim3(grid(1536), 1, n), dim3(256), 0, stream, pr, x_st, x_sh, y_st, y_sh, absmax_ws,     \
                     tokens, heads);
  switch (head_dim) {
    case 32: FDB_Q(32) break;
    case 64: FDB_Q(64) break;
    case 128: FDB_Q(128) break;
    default: return -3;
  }
#undef FDB_Q
  return (int)hipGetLastError();
}

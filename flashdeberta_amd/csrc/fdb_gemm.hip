// Products of more rows than fdb_linear.hip streams, for the layers around the attention: out = epilogue(x . w^T + bias), 16-bit types.
//
// hipBLASLt does the plain product as fast; what is gained is what follows it.  An encoder layer adds the residual to two of its products
// and takes the GELU of a third, each a pass of its own over memory that is as long as a tenth of the layer.  Here these happen on the
// tile that is being written.  [4096 rows, bf16, on the GPU alone, in a replayed graph; product and pass by torch -> here]
//   768 -> 768 + residual 17.0 -> 9.0 us,  768 -> 3072 + GELU 37.8 -> 26.3,  3072 -> 768 + residual 30.6 -> 26.4;
// with 1500 rows 11.6 -> 6.5, 22.1 -> 15.5 and 21.7 -> 16.7.
//
// The sums run over the contraction in order, 32 at a time, in one accumulator, and are rounded where torch's separate passes round:
// the bits are those of torch's product, GELU and addition (where the library does not split the contraction).
//
// What bounds it (4096 x 3072 x 768, tile 256 x 192, 22.7 us without an epilogue): with the loads of its stages left out 19.1, with the products
// alone 21.2, with neither 11.9 (launch, first loads, operands, 25 MB of results): the matrix cores, whose clock falls under such operands to
// the rate of a large library product, plus a start and an end that one round of workgroups does not overlap with them.  Measured
// and no faster: operands read a stage ahead into registers, loads issued between the products instead of ahead of them, more
// stages, rows padded against a stride of whole channels.  GELU through erff instead of the table: 35 us instead of 27.7.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>

#include "fdb_device.h"
#include "fdb_kernels.h"
#include "../../include/fdb.h"

using namespace fdb;

namespace {

// GELU of a 16-bit value, rounded to its type, as torch's elementwise kernel computes it.  erff and what goes with it are some 45 vector
// instructions an element and no memory time hides them here; a bf16 has so few values that matter (2^-14 <= |x| < 8: 17 binades of 128
// and a sign) that each workgroup tabulates them while its first tiles are on their way, and looks the others up.  Values under 2^-14 are halves, where erff makes
// them nothing else, and those of 8 and more themselves or nothing; one is that small in a wave now and then, padding, whose rows are zeros throughout, made every such wave
// go through erff, and wide distributions nearly every wave: 4096 x 3072 x 768 27.3 -> 26.3 us, of values with a deviation of 3 36.9 -> 33.9; twelve layers of
// 8 x 512, padded, 1682 -> 1638 with the residual asked for ahead, too.
__device__ __forceinline__ float gelu(float x) { return x * 0.5f * (1.f + erff(x * 0.70710678118654752440f)); }
constexpr uint32_t kGeluHalves = 0x100, kGeluInf = 0x7F80, kGeluLow = (127 - 14) << 7, kGeluHigh = (127 + 3) << 7, kGeluCount = kGeluHigh - kGeluLow;   // bit patterns of bf16 magnitudes
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
constexpr int kGeluBytes = 2 * kGeluCount * 2;   // [sign][magnitude - low]

enum { kPlain = FDB_GEMM_PLAIN, kGelu = FDB_GEMM_GELU, kResidual = FDB_GEMM_RESIDUAL, kNarrow = FDB_GEMM_NARROW };   // out = y, gelu(y) or y + residual, y = x . w^T +
                                                                                   // bias rounded to the type; y by fours of columns, bias anywhere

struct GemmParams {
  const char *x, *w, *bias, *residual;
  char* out;
  int64_t ldx, ldw, ldo, ldr;   // elements
  int32_t M, N, K, tiles_n, tiles;
};

// A workgroup of WM x WN waves makes TM x TN outputs, PER_CU of them share a CU; stages of kDepth of the contraction go straight from global
// memory into one of STAGES LDS buffers, rows of 128 bytes, slot (row, s) = chunk s ^ swz16(row) (sixteen rows' same chunk: sixteen bank groups).
constexpr int kDepth = 64;

template <int TM_, int TN_, int WM_, int WN_, int STAGES_, int PER_CU_, int STAGED_ = TN_>
struct GemmShape {   // STAGED: rows of w that are fetched, TN or what makes whole loads for every wave
  static constexpr int TM = TM_, TN = TN_, STAGED = STAGED_, WM = WM_, WN = WN_, STAGES = STAGES_, PER_CU = PER_CU_;
  static constexpr int NW = WM * WN, FM = TM / (16 * WM), FN = TN / (16 * WN);
  static constexpr int ROWB = 2 * kDepth, RPI = 1024 / ROWB;   // bytes of a row, rows a wave's load fills
  static constexpr int XI = TM / RPI, WI = STAGED / RPI, LOADS = (XI + WI) / NW;
  static constexpr int STAGE = (TM + STAGED) * ROWB, PITCH = TN * 2 + 16;
  static constexpr int TILES = STAGES * STAGE > TM * PITCH ? STAGES * STAGE : TM * PITCH;
  static constexpr int lds_bytes(bool table) { return TILES + (table ? kGeluBytes : 0); }
  static_assert(PER_CU * TILES <= 160 * 1024, "LDS budget");   // a workgroup with a table may be alone with one fewer
  static_assert(TM % (16 * WM) == 0 && TN % (16 * WN) == 0 && TM % RPI == 0 && STAGED % RPI == 0 && STAGED >= TN && (XI + WI) % NW == 0, "whole fragments, whole loads");
};

// The rows of a product, tile by tile: all `count` of them as they lie.
struct AllRows {
  static constexpr bool BIAS_AHEAD = true;
  int count;
  __device__ __forceinline__ int64_t base(int m0) const { return m0; }
  __device__ __forceinline__ uint32_t from_base(int m0, int row) const { return (uint32_t)(min(m0 + row, count - 1) - m0); }  // past the end: the last one
};

template <class QT, int EPI, class S, class Rows>
__device__ __forceinline__ void make_tile(const GemmParams& p, const Rows& rows, int tm, int tn, char* smem) {
  constexpr int TM = S::TM, TN = S::TN, STAGES = S::STAGES;
  using frag = typename QT::frag;
  using elem = typename QT::scratch_t;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 15, kg = lane >> 4;
  const int wm = wave / S::WN, wn = wave % S::WN;
  const int m0 = tm * TM, n0 = tn * TN;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LDS_AS char*)smem;
  const char* xb = p.x + rows.base(m0) * p.ldx * 2;
  const char* wb = p.w + (int64_t)n0 * p.ldw * 2;
  uint32_t off[S::LOADS];
#pragma unroll
  for (int j = 0; j < S::LOADS; ++j) {
    const int c = wave + S::NW * j, row = c * S::RPI + (lane >> 3);   // rows past the end re-read the last one
    const uint32_t chunk = (uint32_t)(((lane & 7) ^ swz16(row)) * 16);
    if (c < S::XI) off[j] = rows.from_base(m0, row) * (uint32_t)(p.ldx * 2) + chunk;
    else off[j] = (uint32_t)(min(n0 + row - TM, p.N - 1) - n0) * (uint32_t)(p.ldw * 2) + chunk;
  }
  auto fill = [&](int t, int buf) __attribute__((always_inline)) {
    const uint32_t dst = lds0 + (uint32_t)buf * S::STAGE + (uint32_t)wave * 1024u;
#pragma unroll
    for (int j = 0; j < S::LOADS; ++j)
      dma16sn((wave + S::NW * j < S::XI ? xb : wb) + (int64_t)t * S::ROWB, off[j], dst + j * S::NW * 1024u);
  };
  f32x4 acc[S::FM][S::FN];
#pragma unroll
  for (int i = 0; i < S::FM; ++i)
#pragma unroll
    for (int j = 0; j < S::FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // What the end of the tile reads is asked for ahead of everything: a trip to memory that nothing covers there (4096 x 768 x 768 + residual 9.4 -> 9.0 us, 1500 rows
  // 7.0 -> 6.5).  Left as it lies in memory, so that nothing waits for it.  Not the bias of real rows, whose first loads wait for the lengths as it is: 2304 x 768,
  // 2346 real rows of 8 x 384 15.1 -> 15.3 us, 5223 of 64 x 128 24.0 -> 24.3 (8225 of 64 x 200, three rounds, 40.1 -> 39.9).
  using four = typename QT::scratch4;
  four bias[S::FN];
#pragma unroll
  for (int j = 0; j < S::FN; ++j) {
    const int col = n0 + (wn * S::FN + j) * 16 + 4 * kg;
    bias[j] = __builtin_bit_cast(four, u32x2{0, 0});
    if (EPI != kNarrow && Rows::BIAS_AHEAD && p.bias && col < p.N) bias[j] = *(const four*)(p.bias + (int64_t)col * 2);
  }
  constexpr int CW = EPI == kNarrow ? 4 : 8, CH = TN / CW, PIECES = TM * CH / (64 * S::NW);   // of the result, a thread
  // The residual where few registers hold it, and not where two workgroups share a CU: the other one covers the trip there (8192 x 768 x 3072 42.1 us, ahead 42.9, not 41.5).
  constexpr bool AHEAD = EPI == kResidual && TM * CH % (64 * S::NW) == 0 && PIECES <= 3 && S::PER_CU != 2;
  frag residual[AHEAD ? PIECES : 1];
  if constexpr (AHEAD) {
#pragma unroll
    for (int x = 0; x < PIECES; ++x) {
      const int c = tid + x * 64 * S::NW, row = c / CH, nn = n0 + (c - row * CH) * CW;
      residual[x] = QT::zero();
      if (m0 + row < rows.count && nn < p.N) residual[x] = QT::load(p.residual + ((rows.base(m0) + rows.from_base(m0, row)) * p.ldr + nn) * 2);
    }
  }
  const int steps = p.K / kDepth;
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t)
    if (t < steps) fill(t, t);
  constexpr bool TABLE = EPI == kGelu && std::is_same<QT, Bf16Tr>::value;
  if constexpr (TABLE) {
    uint16_t* table = (uint16_t*)(smem + S::TILES);
    for (uint32_t e = tid; e < kGeluCount; e += 64 * S::NW) {
      const float v = __builtin_bit_cast(float, (kGeluLow + e) << 16), t = erff(v * 0.70710678118654752440f);
      ((__bf16*)table)[e] = (__bf16)(v * 0.5f * (1.f + t));
      ((__bf16*)table)[kGeluCount + e] = (__bf16)(-v * 0.5f * (1.f - t));
    }
  }
  const uint32_t xrow = (uint32_t)((wm * S::FM * 16 + r) * S::ROWB), wrow = (uint32_t)((TM + wn * S::FN * 16 + r) * S::ROWB), f = (uint32_t)swz16(r);
  int buf = 0;
#pragma unroll 1
  for (int t = 0; t < steps; ++t) {
    // this wave's loads of stage t have landed, those of the STAGES - 2 after it may still fly
    if (t + STAGES - 1 <= steps) wait_vmcnt<(STAGES - 2) * S::LOADS>();
    else wait_vmcnt<0>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();   // ... and everybody's; everybody has read the buffer of stage t - 1
    asm volatile("" ::: "memory");
    if (t + STAGES - 1 < steps) fill(t + STAGES - 1, buf == 0 ? STAGES - 1 : buf - 1);
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t at = lds0 + (uint32_t)buf * S::STAGE;
#pragma unroll
    for (int s = 0; s < kDepth / 32; ++s) {
      frag xf[S::FM], wf[S::FN];
      const uint32_t slot = ((uint32_t)(4 * s + kg) ^ f) * 16;
#pragma unroll
      for (int j = 0; j < S::FN; ++j) wf[j] = *(LDS_AS const frag*)(uintptr_t)(at + wrow + slot + j * 16 * S::ROWB);
#pragma unroll
      for (int i = 0; i < S::FM; ++i) xf[i] = *(LDS_AS const frag*)(uintptr_t)(at + xrow + slot + i * 16 * S::ROWB);
#pragma unroll
      for (int i = 0; i < S::FM; ++i)
#pragma unroll
        for (int j = 0; j < S::FN; ++j) acc[i][j] = mma16(wf[j], xf[i], acc[i][j]);
    }
    buf = buf == STAGES - 1 ? 0 : buf + 1;
  }
  __syncthreads();   // the staged tiles have been read: their memory takes the result
#pragma unroll
  for (int j = 0; j < S::FN; ++j) {
    const int col = (wn * S::FN + j) * 16 + 4 * kg;
    f32x4 b = __builtin_convertvector(bias[j], f32x4);
    if (EPI != kNarrow && !Rows::BIAS_AHEAD && p.bias && n0 + col < p.N) b = QT::load4(p.bias + (int64_t)(n0 + col) * 2);
    if (EPI == kNarrow && p.bias && n0 + col < p.N) {
#pragma unroll
      for (int e = 0; e < 4; ++e) b[e] = (float)((const elem*)p.bias)[n0 + col + e];
    }
    char* const to = smem + (wm * S::FM * 16 + r) * S::PITCH + col * 2;
    if constexpr (TABLE) {
      // Sixteen rows' values at a time: the reads of a group are under way together, and one test a group finds what the table leaves out.
      u16x4 looked[S::FM];
      uint32_t most = 0;
#pragma unroll
      for (int i = 0; i < S::FM; ++i) {
        const u16x4 bits = __builtin_bit_cast(u16x4, QT::pack4(acc[i][j] + b));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t at = (bits[e] & 0x7FFFu) - kGeluLow;
          most = max(most, at);
          looked[i][e] = ((const uint16_t*)(smem + S::TILES))[min(at, kGeluCount - 1) + (bits[e] >> 15) * kGeluCount];
        }
      }
      bool all_looked = true;
      if (__any(most >= kGeluCount)) {   // zeros of padding, and a few in a hundred thousand ordinary values, under 2^-14: halves, while those are normal numbers
        bool others = false;
#pragma unroll
        for (int i = 0; i < S::FM; ++i) {
          const u16x4 bits = __builtin_bit_cast(u16x4, QT::pack4(acc[i][j] + b));
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t size = bits[e] & 0x7FFFu;
            others |= size != 0 && size - kGeluHalves >= kGeluHigh - kGeluHalves;
            if (size < kGeluLow) looked[i][e] = size == 0 ? bits[e] : bits[e] - 0x80;
          }
        }
        if (__builtin_expect(__any(others), 0)) {   // large ones: 1 + erff is 2 or 0
          others = false;
#pragma unroll
          for (int i = 0; i < S::FM; ++i) {
            const u16x4 bits = __builtin_bit_cast(u16x4, QT::pack4(acc[i][j] + b));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const uint32_t size = bits[e] & 0x7FFFu;
              others |= size != 0 && size - kGeluHalves >= kGeluInf - kGeluHalves;
              if (size >= kGeluHigh) looked[i][e] = bits[e] >> 15 ? 0x8000 : bits[e];
            }
          }
          all_looked = !__any(others);
        }
      }
      if (all_looked) {
#pragma unroll
        for (int i = 0; i < S::FM; ++i) *(u16x4*)(to + i * 16 * S::PITCH) = looked[i];
        continue;
      }   // denormal, infinite or not a number
    }
#pragma unroll
    for (int i = 0; i < S::FM; ++i) {
      f32x4 y = acc[i][j] + b;
      if constexpr (EPI == kGelu) {
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = gelu((float)(elem)y[e]);
      }
      QT::store4(to + i * 16 * S::PITCH, y[0], y[1], y[2], y[3]);
    }
  }
  __syncthreads();
  auto put = [&](int c, const frag* add) __attribute__((always_inline)) {   // the c-th piece of the result
    const int row = c / CH, col = (c - row * CH) * CW, m = m0 + row, nn = n0 + col;
    if (m < rows.count && nn < p.N) {
      const int64_t at = rows.base(m0) + rows.from_base(m0, row);
      if constexpr (EPI == kNarrow) {
        *(u32x2*)(p.out + (at * p.ldo + nn) * 2) = *(const u32x2*)(smem + row * S::PITCH + col * 2);
        return;
      }
      frag y = *(const frag*)(smem + row * S::PITCH + col * 2);
      if constexpr (EPI == kResidual) y = QT::from_f32(QT::to_f32(y) + QT::to_f32(add ? *add : QT::load(p.residual + (at * p.ldr + nn) * 2)));
      *(frag*)(p.out + (at * p.ldo + nn) * 2) = y;
    }
  };
  if constexpr (AHEAD) {
#pragma unroll
    for (int x = 0; x < PIECES; ++x) put(tid + x * 64 * S::NW, &residual[x]);
  } else {
    for (int c = tid; c < TM * CH; c += 64 * S::NW) put(c, nullptr);
  }
}

// Tile of the n-th of `tiles` workgroups: every XCD takes a run of tiles, whose rows of x and w then pass through one L2
__device__ __forceinline__ int tile_of(int n, int tiles) {
  const int xcd = n & 7;
  return xcd * (tiles >> 3) + min(xcd, tiles & 7) + (n >> 3);
}

template <class QT, int EPI, class S>
__global__ __launch_bounds__(64 * S::NW, S::PER_CU * S::NW / 4) void fdb_gemm_kernel(const GemmParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tile = tile_of(blockIdx.x, p.tiles), tm = tile / p.tiles_n;
  make_tile<QT, EPI, S>(p, AllRows{p.M}, tm, tile - tm * p.tiles_n, smem);
}

// The product of a padded batch's real rows alone (the lengths are on the device): nothing reads the projections of padding, a third of the
// rows where a batch is padded to its longest text.  Every wave adds up the lengths, so that the real rows count through; the workgroup takes
// the tile whose rounds are shortest for as many rows and looks up where its rows lie.  One workgroup a CU, which goes on to its tile of the next
// round itself: workgroups without a tile would cost a round of their own.  Against the library's product of all rows, 768 -> 2304, us:
//   real rows of        4096 (19.1)   8192 (32.4)   16384 (62.9)     and the layer, projections and attention: 32 x 128 34.0 -> 29.7, 64 x 128
//     all                 20.3          35.2           69.0          62.0 -> 49.0, 16 x 512 87.7 -> 71.4 (lengths between a quarter and all);
//     nine tenths         19.0          32.6           62.9          with a mask that masks nothing 37.4 -> 37.6, 62.4 -> 63.6, 92.8 -> 89.8.
//     six tenths          14.9          21.9           39.1
//     a quarter           10.4          14.2           19.7
// Reading the lengths and adding them up is 1 us of it.
constexpr int kRealSequences = 64;   // one a lane
constexpr int kRealExtra = 64 * 192;  // what a round costs besides its outputs, in outputs: 256 x 192 20.2 us, 64 x 192 10.4
struct RealParams {
  GemmParams g;
  const int32_t *start, *length;   // [batch]: the first real row of a sequence (NULL: 0) and how many (negative: none)
  int32_t batch, seqlen, cus, narrow, span;   // narrow: tiles of 160 columns across; span: half of the power of two from batch up
  int32_t clear;   // the rows of padding become zeros
};
using R64 = GemmShape<64, 192, 2, 4, 4, 1>;
using R128 = GemmShape<128, 192, 2, 4, 3, 1>;
using R192 = GemmShape<192, 192, 4, 2, 3, 1>;
using R256 = GemmShape<256, 192, 4, 2, 2, 1>;
using R256x160 = GemmShape<256, 160, 4, 2, 2, 1, 192>;
constexpr int kRealTiles = R192::TILES;   // the most of the four
constexpr int kRealBytes = kRealTiles + 256 * 4;   // and where a tile's rows lie
static_assert(R64::TILES <= kRealTiles && R128::TILES <= kRealTiles && R256::TILES <= kRealTiles && R256x160::TILES <= kRealTiles && kRealBytes <= 160 * 1024, "LDS budget");
struct RealRows {
  static constexpr bool BIAS_AHEAD = false;
  int count;
  const int32_t* at;   // LDS
  __device__ __forceinline__ int64_t base(int) const { return 0; }
  __device__ __forceinline__ uint32_t from_base(int, int row) const { return (uint32_t)at[row]; }
};

template <class QT>
__global__ __launch_bounds__(512, 2) void fdb_gemm_real_kernel(const RealParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  int32_t* at = (int32_t*)(smem + kRealTiles);
  const int tid = threadIdx.x, lane = tid & 63;
  int first = 0, len = 0;
  if (lane < p.batch) {
    first = p.start ? p.start[lane] : 0;
    len = p.length[lane];
  }
  first = min(max(first, 0), p.seqlen);
  len = min(max(len, 0), p.seqlen - first);
  int sum = len;   // of the sequences up to this one: within rows of sixteen lanes, then from row to row
  sum += __builtin_amdgcn_update_dpp(0, sum, 0x111, 0xf, 0xf, false);   // row_shr:1, 2, 4, 8
  sum += __builtin_amdgcn_update_dpp(0, sum, 0x112, 0xf, 0xf, false);
  sum += __builtin_amdgcn_update_dpp(0, sum, 0x114, 0xf, 0xf, false);
  sum += __builtin_amdgcn_update_dpp(0, sum, 0x118, 0xf, 0xf, false);
  sum += __builtin_amdgcn_update_dpp(0, sum, 0x142, 0xa, 0xf, false);   // row_bcast:15 into rows 1 and 3, :31 into rows 2 and 3
  sum += __builtin_amdgcn_update_dpp(0, sum, 0x143, 0xc, 0xf, false);
  const int count = __builtin_amdgcn_readlane(sum, 63);
  const int before = sum - len, shift = lane * p.seqlen + first - before;   // real rows ahead of the sequence; from a real row's number to its place
  int height = 256, wide = 0, tiles = 0, least = INT32_MAX;
  auto consider = [&](int h, int across, int width) __attribute__((always_inline)) {   // a round takes the time of its outputs and of 64 x 192 more
    const int t = (count + h - 1) / h * across, cost = (int)((uint32_t)(t + p.cus - 1) / (uint32_t)p.cus) * (h * width + kRealExtra);
    if (cost < least) least = cost, height = h, wide = across, tiles = t;
  };
  consider(256, p.g.tiles_n, 192);
  consider(256, p.narrow, 160);
  consider(192, p.g.tiles_n, 192);
  consider(128, p.g.tiles_n, 192);
  consider(64, p.g.tiles_n, 192);
  // Ahead of the tiles, under whose loads and products the stores drain (after them: 8 x 512 15.2 -> 16.5 us), and past the caches, since nobody
  // reads the rows: a training layer of 8 x 512 takes up to 1.5 us of 216 longer for it, 2.6 with ordinary stores.
  if (p.clear) {
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int i = blockIdx.x * 8 + wave; i < p.batch * p.seqlen; i += gridDim.x * 8) {   // a row a wave
      const int b = __builtin_amdgcn_readfirstlane(i / p.seqlen), row = i - b * p.seqlen, b_first = __builtin_amdgcn_readlane(first, b);
      if (row >= b_first && row < b_first + __builtin_amdgcn_readlane(len, b)) continue;
      for (int col = 8 * lane; col < p.g.N; col += 8 * 64) __builtin_nontemporal_store(u32x4{0, 0, 0, 0}, (u32x4*)(p.g.out + ((int64_t)i * p.g.ldo + col) * 2));
    }
  }
  for (int i = blockIdx.x; i < tiles; i += gridDim.x) {
    const int tile = tile_of(i, tiles), tm = tile / wide, tn = tile - tm * wide;
    const int m = min(tm * height + tid, count - 1);
    int b = 0;   // the last sequence with at most m rows ahead of it; empty ones share that number with the one after them
    for (int x = p.span; x > 0; x >>= 1) {
      const int ahead = __shfl(before, b + x);
      b += ahead <= m ? x : 0;   // lanes past the batch have all rows ahead of them
    }
    const int row = m + __shfl(shift, b);
    if (i != (int)blockIdx.x) __syncthreads();   // the tile before has been written
    if (tid < 256) at[tid] = row;
    __syncthreads();
    const RealRows rows{count, at};
    if (height == 64) make_tile<QT, kPlain, R64>(p.g, rows, tm, tn, smem);
    else if (height == 128) make_tile<QT, kPlain, R128>(p.g, rows, tm, tn, smem);
    else if (height == 192) make_tile<QT, kPlain, R192>(p.g, rows, tm, tn, smem);
    else if (wide == p.g.tiles_n) make_tile<QT, kPlain, R256>(p.g, rows, tm, tn, smem);
    else make_tile<QT, kPlain, R256x160>(p.g, rows, tm, tn, smem);
  }
}

template <class QT>
int launch_real(RealParams p, hipStream_t stream) {
  auto kern = fdb_gemm_real_kernel<QT>;
  static std::atomic<uint64_t> lds_set{0};
  const hipError_t e = fdb_set_lds_once((const void*)kern, kRealBytes, lds_set);
  if (e != hipSuccess) return (int)e;
  p.g.tiles_n = (p.g.N + 191) / 192;
  p.narrow = (p.g.N + 159) / 160;
  for (p.span = 0; std::max(1, 2 * p.span) < p.batch;) p.span = std::max(1, 2 * p.span);
  hipLaunchKernelGGL(kern, dim3((unsigned)p.cus), dim3(512), kRealBytes, stream, p);
  return (int)hipGetLastError();
}

template <class QT, int EPI, class S>
int launch_shape(GemmParams p, hipStream_t stream) {
  auto kern = fdb_gemm_kernel<QT, EPI, S>;
  constexpr int lds = S::lds_bytes(EPI == kGelu && std::is_same<QT, Bf16Tr>::value);
  static std::atomic<uint64_t> lds_set{0};
  const hipError_t e = fdb_set_lds_once((const void*)kern, lds, lds_set);
  if (e != hipSuccess) return (int)e;
  p.tiles_n = (p.N + S::TN - 1) / S::TN;
  p.tiles = (p.M + S::TM - 1) / S::TM * p.tiles_n;
  hipLaunchKernelGGL(kern, dim3(p.tiles), dim3(64 * S::NW), lds, stream, p);
  return (int)hipGetLastError();
}

using S32x64 = GemmShape<32, 64, 1, 4, 4, 3>;
using S64x64 = GemmShape<64, 64, 2, 2, 3, 3>;
using S64x64Eight = GemmShape<64, 64, 2, 4, 3, 3>;   // while each has a CU to itself: half the instructions of a stage in a row
using S64x192Deep = GemmShape<64, 192, 2, 4, 4, 1>;   // alone on its CU: four stages instead of a second workgroup
using S64x192 = GemmShape<64, 192, 2, 4, 2, 2>;
using S256x192 = GemmShape<256, 192, 4, 2, 2, 1>;

int64_t tiles_of(int64_t M, int64_t N, int tm, int tn) { return (M + tm - 1) / tm * ((N + tn - 1) / tn); }

// The smallest tile whose workgroups make one round of the chip; beyond that the tile that loads the least.  bf16, replayed graph, us, in the
// order of the list, * the chosen one ([M x K] . [K x N] and what follows):
//   512 x 768 x 768   5.4* 6.2 8.9 8.2 18.9      1500 x 768 x 768    7.7 7.3* 8.9 8.5 19.2      1024 x 3072 x 768  22.9 17.2 12.3* 14.3 24.3
//   4096 x 768 x 3072 44.6 32.3 26.9* 34.6 59.7  2048 x 3072 x 768  43.1 27.5 22.9 17.4* 25.2   8192 x 768 x 768  26.3 19.6 19.0 15.3* 23.1
//   3000 x 3072 x 768 61.0 39.8 32.7 27.9 26.4*  4096 x 3072 x 768  82.3 50.5 42.8 31.1 27.7*   8192 x 3072 x 768  155 97.3 81.4 58.1 53.4*
// The first by waves side by side, 1 x 4 instead of 2 x 2: 5.2 -> 5.0, [300 x 768] . [768 x 768] 5.0 -> 4.7.  The second by eight waves instead of four: 512 x 1536 x 768
// 5.8 -> 5.5, 1024 x 768 x 768 6.2 -> 5.7; beyond a tile a compute unit four are the faster: 1500 x 768 x 768 7.1 and 7.2, 512 x 2304 x 768 6.8 and 7.1.
// (64 x 96, 128 x 96, 128 x 128, 128 x 144, 128 x 192 and 256 x 256, with two to five stages, lie between these.)
template <class QT, int EPI>
int launch_gemm(const GemmParams& p, hipStream_t stream) {
  const int64_t cus = fdb_cu_count();
  if (tiles_of(p.M, p.N, 32, 64) <= cus) return launch_shape<QT, EPI, S32x64>(p, stream);
  if (tiles_of(p.M, p.N, 64, 64) <= cus) return launch_shape<QT, EPI, S64x64Eight>(p, stream);
  if (tiles_of(p.M, p.N, 64, 64) * 8 <= cus * 15) return launch_shape<QT, EPI, S64x64>(p, stream);
  if (tiles_of(p.M, p.N, 64, 192) <= cus) return launch_shape<QT, EPI, S64x192Deep>(p, stream);
  if (tiles_of(p.M, p.N, 64, 192) <= 2 * cus) return launch_shape<QT, EPI, S64x192>(p, stream);
  return launch_shape<QT, EPI, S256x192>(p, stream);
}

template <class QT>
int launch_type(const GemmParams& p, int epilogue, hipStream_t stream) {
  if (epilogue == kGelu) return launch_gemm<QT, kGelu>(p, stream);
  if (epilogue == kResidual) return launch_gemm<QT, kResidual>(p, stream);
  if (epilogue == kNarrow) return launch_gemm<QT, kNarrow>(p, stream);
  return launch_gemm<QT, kPlain>(p, stream);
}

}  // namespace

// Where this kernel is the faster one, and adds up as the library does.  Up to 32 rows the weights are streamed by many waves that share the
// contraction.  A long contraction over few tiles is split by the library ([512 x 3072] . [3072 x 768] + residual 13.5 us there, 13.9 here; 1500 rows
// 21.7 and 18.3).  A plain product has nothing to gain beyond two tiles of 64 x 192 a compute unit (4096 and 3000 rows to 2304 columns: 19.3 and 16.7 us there, 20.8
// and 19.7 here; 2048, 1024 and 512 rows 15.5, 11.2 and 8.1 there, 12.7, 9.4 and 7.1 here).
extern "C" int32_t fdb_gemm_serves(int64_t M, int64_t N, int64_t K, int32_t epilogue) {
  if (M <= 32 || N < 8 || K < kDepth || N % 8 || K % kDepth || M > (1 << 24) || N > (1 << 24)) return 0;
  if (K > 1536 && tiles_of(M, N, 64, 64) <= fdb_cu_count()) return 0;
  return epilogue != kPlain || tiles_of(M, N, 64, 192) <= 2 * fdb_cu_count();
}

int fdb_launch_gemm(const void* x, const void* w, const void* bias, const void* residual, void* out, int32_t M, int32_t N, int32_t K, int64_t ldx,
                    int64_t ldw, int64_t ldo, int64_t ldr, int epilogue, int dtype, void* stream) {
  const GemmParams p{(const char*)x, (const char*)w, (const char*)bias, (const char*)residual, (char*)out, ldx, ldw, ldo, ldr, M, N, K, 0, 0};
  return dtype == FDB_BF16 ? launch_type<Bf16Tr>(p, epilogue, (hipStream_t)stream) : launch_type<F16Tr>(p, epilogue, (hipStream_t)stream);
}

// From where the whole product is the library's: below that its tiles are small already (2048 x 768 x 2304 12.7 us, 14.4 here, half of them real 10.8).
extern "C" int32_t fdb_gemm_real_serves(int64_t batch, int64_t seqlen, int64_t N, int64_t K, int64_t ldx) {
  const int64_t M = batch * seqlen;
  if (batch < 1 || batch > kRealSequences || seqlen < 1 || N < 8 || K < kDepth || N % 8 || K % kDepth || M > (1 << 24) || N > (1 << 24)) return 0;
  return M * ldx * 2 <= INT32_MAX && tiles_of(M, N, 64, 192) > 2 * fdb_cu_count();
}

int fdb_launch_gemm_real(const void* x, const void* w, const void* bias, void* out, const int32_t* start, const int32_t* length, int32_t batch, int32_t seqlen,
                         int32_t N, int32_t K, int64_t ldx, int64_t ldw, int64_t ldo, bool clear, int dtype, void* stream) {
  RealParams p{};
  p.g = GemmParams{(const char*)x, (const char*)w, (const char*)bias, nullptr, (char*)out, ldx, ldw, ldo, 0, batch * seqlen, N, K, 0, 0};
  p.start = start, p.length = length, p.batch = batch, p.seqlen = seqlen, p.cus = fdb_cu_count(), p.clear = clear;
  return dtype == FDB_BF16 ? launch_real<Bf16Tr>(p, (hipStream_t)stream) : launch_real<F16Tr>(p, (hipStream_t)stream);
}

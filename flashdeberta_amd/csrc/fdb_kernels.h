// Internal interface between the host-side C ABI (fdb_api.cpp) and the device code
// (fdb_attn.hip, fdb_aux.hip).  Not installed; the public contract is include/fdb.h.
#pragma once
#include <stdint.h>

// Query rows per workgroup (4 waves x 32 rows) and keys per main-loop iteration.
#define FDB_BM 128
#define FDB_BN 64

// (sequence, head) groups whose query tiles are dealt together, see block_map
inline int32_t fdb_groups_together(int32_t tiles_per_seq) { return 8 * (tiles_per_seq < 96 ? 96 / tiles_per_seq : 1); }

// Whether a padded batch's workgroups may be dealt by the lengths of its sequences (padded_map, which looks at the lengths): a lane a sequence, and more
// workgroups (of all roles) than compute units; fewer have a unit each whatever the order.
inline bool fdb_deals_by_length(const int32_t* seq_len, int64_t batch, int64_t workgroups, int64_t cus) {
  return seq_len && batch > 1 && batch <= 64 && workgroups > cus;
}

struct FdbKParams {
  const char* q;
  const char* k;
  const char* v;
  const char* pk;  // K_r, NULL when the content->position term is absent
  const char* pq;  // Q_r, NULL when the position->content term is absent
  char* out;
  float* lse;
  const int32_t* cu;   // cu_seqlens or NULL
  const int32_t* wl;   // work-list (varlen only)
  const int32_t* seq_start;  // padded fixed layout: first real token / number of real tokens per row (or NULL)
  const int32_t* seq_len;
  const int16_t* lut;  // delta LUT, index r + R
  const float* qs;     // fp8 dequant scales per head (NULL otherwise)
  const float* ks;
  const float* pks;
  const float* pqs;
  int64_t q_sb, q_st, q_sh;
  int64_t k_sb, k_st, k_sh;
  int64_t v_sb, v_st, v_sh;
  int64_t o_sb, o_st, o_sh;
  int64_t pk_sh, pk_sr;
  int64_t pq_sh, pq_sr;
  int32_t B, H, L, tiles_per_seq;
  int32_t groups_together;  // fdb_groups_together(tiles_per_seq)
  int32_t by_length;        // fdb_deals_by_length
  int32_t R;        // LUT radius
  int32_t far_done;  // near launches: the far tiles' partial results (far_parts of them) are to be merged
  int32_t near_all;  // near launches: they walk every key tile, no far launch precedes them
  int32_t far_parts; // workgroups per query tile of the far-only launch, each with its share of the far tiles and a
                     // partial result of its own (the first in out / lse, the others in workspace slots 0 ..)
  int32_t near_parts; // workgroups per query tile of the near launch; above 1 each leaves the partial result of
                      // its share of the steps in workspace slot far_parts-1 + part, and fdb_launch_merge follows
  int32_t near_teams; // 16-bit near launches: teams of four waves in a workgroup, which share its steps out among them
  int32_t key_parts; // one-kernel mode: workgroups per query tile, each with an equal share of the key tiles and a
                     // partial result of its own in workspace slot `part`; fdb_launch_merge_parts follows (1: no sharing)
  int32_t ws_slots;  // partial results in the workspace: far_parts-1, plus near_parts if that is above 1; key_parts in the one-kernel mode
  char* ws;          // [ws_slots][ws_rows][H][D] elements of v's type (rows normalised over the keys seen), then
  int64_t ws_rows;   // [ws_slots][ws_rows][H] float log-sum-exps (-inf: no key seen); ws_rows = rows of the lse buffer
  int32_t causal;
  int32_t fill_pad; // padded fixed layout, first launch of a call: write the rows of out and lse outside the real tokens (zeros; NaN
                    // for batch rows whose seq_len is negative)
  float scale_log2; // sm_scale * log2(e)
};

// Backward launch (fdb_bwd.hip): fixed layout only.  Position scores and their gradients have q's element type, element
// (b, l, h, delta) at b * bias_sb + l * bias_st + h * bias_sh + delta; lse / delta are fp32 [B*L, H].
struct FdbBwdParams {
  const char* q;
  const char* k;
  const char* v;
  const char* dout;
  char* dq;
  char* dk;
  char* dv;
  const float* lse;
  float* delta;         // sum_d dO * O per row: read, or written by the dQ role when `out` is given
  const char* out;      // the forward's output or NULL
  const char* c2p;      // q_i . K_r[delta] or NULL; element type of q, like the gradient tensors below
  const char* p2c;      // k_j . Q_r[delta] or NULL
  char* d_c2p;          // element type of q; every entry of a real token's row is stored once, rows of padding are not touched
  char* d_p2c;
  const int32_t* seq_start;
  const int32_t* seq_len;
  const int16_t* lut;
  int64_t q_sb, q_st, q_sh;
  int64_t k_sb, k_st, k_sh;
  int64_t v_sb, v_st, v_sh;
  int64_t g_sb, g_st, g_sh;     // dout
  int64_t o_sb, o_st, o_sh;     // out
  int64_t dq_sb, dq_st, dq_sh;
  int64_t dk_sb, dk_st, dk_sh;
  int64_t dv_sb, dv_st, dv_sh;
  int64_t bias_sb, bias_st, bias_sh;
  int32_t B, H, L;
  int32_t S;        // att_span
  int32_t R;        // table radius
  int32_t causal;
  int32_t pairs_per_xcd;  // workgroup ids map to (tile, head, batch row) with whole (batch row, head) pairs per XCD
  int32_t store_chunks;   // score gradients leave the ring in aligned chunks of this many groups of four entries: 8, 4 or 1 (as the table's window leaves room)
  float scale_log2; // sm_scale * log2(e)
  float sm_scale;
};
int fdb_launch_bwd(const FdbBwdParams& p, int dtype, int head_dim, void* stream);

// Where a workgroup of the backward's roles works in a padded batch: the n-th of its role; the batch row's first token and its number of tokens.
struct FdbPlace {
  int32_t b, tile, h, tok0, tokens, n, keys, unused;   // keys: the dK/dV role
};

// Backward with the tables in the kernel (fdb_bwd_ring.hip): fixed layout, head_dim 64, 16-bit types, both position terms.
struct FdbBwdRingParams {
  const char* q;
  const char* k;
  const char* v;
  const char* dout;
  const char* out;
  const char* pk;       // K_r, Q_r
  const char* pq;
  char* dq;
  char* dk;
  char* dv;
  char* dpk;            // gradients of the tables, strides dp_sh, dp_sr; rows [0, 2S) are written
  char* dpq;
  const float* lse;     // [B*L, H]
  const int32_t* seq_start;
  const int32_t* seq_len;
  const int16_t* lut;
  // scratch: row statistics [B][H][stat_len], far sums [B][H][2][stat_len], G blocks [B][H][g_rows][g_slots][32 x 32] (element type
  // of q), partial table gradients [tg_parts][H][4 tg_groups][2][32][64] and
  // [tg_parts][H][2 tables][2 sides][64]
  float* neg_lse;
  float* neg_delta;
  float* far_q;
  float* far_k;
  char* g_blocks;
  char* zero_block;     // 2 KB of zeros, written by the dQ launch
  float* e_parts;
  float* far_parts;
  int64_t q_sb, q_st, q_sh;
  int64_t k_sb, k_st, k_sh;
  int64_t v_sb, v_st, v_sh;
  int64_t g_sb, g_st, g_sh;     // dout
  int64_t o_sb, o_st, o_sh;     // out
  int64_t dq_sb, dq_st, dq_sh;
  int64_t dk_sb, dk_st, dk_sh;
  int64_t dv_sb, dv_st, dv_sh;
  int64_t pk_sh, pk_sr, pq_sh, pq_sr, dp_sh, dp_sr;
  int32_t B, H, L, S, R, causal;
  int32_t stat_len, g_rows, g_slots;
  int32_t tiles, groups_together;  // query tiles of a sequence; fdb_groups_together(tiles)
  int32_t rho_min, tg_groups, tg_parts, tg_chunks, tg_len;  // blocks of 32 relative positions in groups of four; shares of the tokens; chunks of
                                                            // tg_len row blocks per batch row
  int32_t has_far;
  float scale_log2, sm_scale;
  // last: an argument among the others moves the sixteen-register loads of the rest, and the dQ role spills more
  int32_t by_length;   // fdb_deals_by_length
  int32_t tg_items;    // chunks a share takes
  FdbPlace* places;    // by_length: two for every (batch row, query tile, head)
};
int fdb_launch_bwd_ring(const FdbBwdRingParams& p, int dtype, void* stream);

// The chain through the position tables (fdb_chain.hip): contiguous tensors, head_dim 64, 2S = 512.
struct FdbChainParams {
  const char* g;       // [matrices][rows][2S] score gradients
  const char* x;       // the token rows of the other factor (q or k) of matrices [0, split): matrix stride x_sm, row stride x_sr (elements)
  const char* x2;      // ... of matrices [split, matrices), numbered from 0 again; same strides
  const char* pos;     // [matrices][2S][D] the tables
  char* dx;            // in and out: += g . pos; rows laid out like those of x, with strides dx_sm, dx_sr, for matrices [0, split)
  char* dx2;           // ... and for matrices [split, matrices)
  float* parts_out;    // [parts][matrices][2S][D] partial sums of g^T . x
  int64_t rows, x_sm, x_sr, dx_sm, dx_sr;
  int32_t matrices, split, parts, tiles_per_part;
};
int fdb_launch_chain(const FdbChainParams& p, int dtype, void* stream);

// Workspace slot `slot`: its output rows and its log-sum-exps (row_bytes = head_dim * element size).
#if defined(__HIPCC__)
// A kernel's first instruction: one argument of every 64 bytes that are not read at once anyway.  Left to itself the compiler reads the arguments where they
// are used, each new 64 bytes of them after a wait for memory of their own.  Not for kernels that have no registers to spare: those of csrc/fdb_attn.hip, where reads_arguments
// has the figures, and the e4m3 pair (near launch of 3 x 777 28.8 -> 29.2 us, of 2 x 700 25.9 -> 26.3; 64 x 128, whose starts count more, 18.9 -> 18.7),
// but for its near launch of all tiles with p2c alone (2 x 700 22.6 -> 22.3, 5 x 777 31.2 -> 30.7).
__device__ __forceinline__ void read_arguments(const FdbKParams& p) { asm volatile("" ::"s"(p.q_sb), "s"(p.o_sb)); }

__device__ __forceinline__ char* ws_slot_out(const FdbKParams& p, int slot, int row_bytes) {
  return p.ws + (int64_t)slot * p.ws_rows * p.H * row_bytes;
}
__device__ __forceinline__ float* ws_slot_lse(const FdbKParams& p, int slot, int row_bytes) {
  return (float*)(p.ws + (int64_t)p.ws_slots * p.ws_rows * p.H * row_bytes) + (int64_t)slot * p.ws_rows * p.H;
}
// far partial result `part` >= 1 sits in slot part - 1
__device__ __forceinline__ char* far_part_out(const FdbKParams& p, int part, int row_bytes) {
  return ws_slot_out(p, part - 1, row_bytes);
}
__device__ __forceinline__ float* far_part_lse(const FdbKParams& p, int part, int row_bytes) {
  return ws_slot_lse(p, part - 1, row_bytes);
}
#endif

#if defined(__HIPCC__)
// hipFuncSetAttribute(MaxDynamicSharedMemorySize) once per kernel instantiation and device instead of
// once per launch.  `done` is a per-instantiation bit mask over device ordinals (a racing first call
// merely sets the attribute twice).
#include <atomic>
inline hipError_t fdb_set_lds_once(const void* kern, int lds_bytes, std::atomic<uint64_t>& done) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
  const uint64_t bit = 1ull << dev;
  if (done.load(std::memory_order_acquire) & bit) return hipSuccess;
  const hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
  if (e == hipSuccess) done.fetch_or(bit, std::memory_order_release);
  return e;
}
#endif

// Most workgroups per query tile a far-only launch is split into.
#define FDB_MAX_FAR_PARTS 4

// Compute units of the current device (256 if it cannot be asked).
int fdb_cu_count();

// Launchers return the hipError_t of the launch as int.
// fdb_launch_attn, by mode:
//   FDB_MODE_FUSED      one kernel walks every key tile;
//   FDB_MODE_FAR_ONLY   it skips the near tiles and leaves the far tiles' partial result (normalised
//                       rows in out, their log-sum-exp in lse, -inf where a row has no far tile);
//   FDB_MODE_NEAR_RING  the near tiles only, four waves of 32 rows x 64 keys with the expanded
//                       relative-embedding rows in LDS rings, merged with the far partial when
//                       p.far_done.
// The last two exist for the 16-bit element types with head_dim <= 64 (fdb_near_supported).
enum { FDB_MODE_FUSED = 0, FDB_MODE_FAR_ONLY = 1, FDB_MODE_NEAR_RING = 2 };
int fdb_launch_attn(const FdbKParams& p, int dtype, int head_dim, int grid_x, int mode, void* stream);
bool fdb_near_supported(int dtype, int head_dim);
// fdb_launch_near32: the near tiles in 32-key steps, 66 KB of LDS so that two workgroups share a CU
// (16-bit element types, head_dim 64); merges the far partial like the ring mode.
bool fdb_near32_supported(int dtype, int head_dim);
int fdb_launch_near32(const FdbKParams& p, int dtype, int grid_x, void* stream);
// fp32 at head_dim 64 with a position term: every key tile in one launch (p.key_parts shares of them, as in the one-kernel mode).
int fdb_launch_near_f32(const FdbKParams& p, int grid_x, void* stream);
// The same pair of launches for OCP e4m3 q / k / K_r / Q_r with bf16 v (head_dim 64): e4m3 MFMA contractions over
// the whole head_dim for the three score products (fdb_fp8.hip).
bool fdb_fp8_pair_supported(int dtype, int head_dim);
int fdb_launch_far8(const FdbKParams& p, int grid_x, void* stream);
int fdb_launch_near8(const FdbKParams& p, int grid_x, void* stream);
// fdb_launch_merge: after a near launch with near_parts > 1: out / lse from the far partial results (when
// p.far_done) and the near ones (16-bit element types, head_dim 64).
int fdb_launch_merge(const FdbKParams& p, int dtype, void* stream);
// fdb_launch_merge_parts: after a one-kernel launch with key_parts > 1: out (and lse, when given) from the key_parts
// partial results in the workspace (any element type and head_dim).
int fdb_launch_merge_parts(const FdbKParams& p, int dtype, int head_dim, void* stream);
int fdb_launch_linear(const void* x, const void* w, const void* bias, void* out, int32_t M, int32_t N, int32_t K, int64_t ldx, int64_t ldw,
                      int64_t ldo, int dtype, void* stream);  // fdb_linear.hip
int fdb_launch_gemm(const void* x, const void* w, const void* bias, const void* residual, void* out, int32_t M, int32_t N, int32_t K, int64_t ldx,
                    int64_t ldw, int64_t ldo, int64_t ldr, int epilogue, int dtype, void* stream);  // fdb_gemm.hip
// The plain product where columns and output rows come by fours only, or the bias lies on any element: for fdb_linear, not an epilogue of fdb_gemm's.
enum { FDB_GEMM_NARROW = 3 };
int fdb_launch_small(const void* x, const void* w, const void* bias, const void* pos_key, const void* pos_query, void* out, const int32_t* start, const int32_t* length,
                     const int16_t* lut, int32_t batch, int32_t seqlen, int32_t heads, int32_t depth, int64_t ldx, int64_t ldw, int64_t pk_sh, int64_t pk_sr, int64_t pq_sh,
                     int64_t pq_sr, int32_t radius, float sm_scale, int dtype, void* stream);
int fdb_launch_gemm_real(const void* x, const void* w, const void* bias, void* out, const int32_t* start, const int32_t* length, int32_t batch, int32_t seqlen,
                         int32_t N, int32_t K, int64_t ldx, int64_t ldw, int64_t ldo, bool clear, int dtype, void* stream);
int fdb_launch_dgrad(const void* x0, int32_t rows0, int32_t depth0, const void* x1, int32_t rows1, int32_t depth1, const void* w, int32_t cols, void* out0,
                     void* out1, int dtype, void* stream);  // fdb_grad.hip
int fdb_wgrad_shares(int64_t rows, int64_t x_cols, int64_t y_cols);
int fdb_launch_wgrad(const void* x0, const void* y0, int32_t rows0, int32_t x_cols0, const void* x1, const void* y1, int32_t rows1, int32_t x_cols1, int32_t y_cols,
                     void* dw, void* db, float* ws, int32_t shares, int dtype, void* stream);
int fdb_launch_join(const void* const w[3], const void* const b[3], void* w_out, void* b_out, int64_t w_bytes, int64_t b_bytes, void* stream);
int fdb_column_sum_parts(int64_t rows);
int fdb_launch_column_sums(const void* x, int64_t x_rows, int64_t x_cols, const void* y, int64_t y_rows, int64_t y_cols, void* out, float* ws,
                           int dtype, void* stream);
int fdb_launch_mask_bounds(const void* mask, int elem_size, bool is_float, int64_t stride_b, int64_t stride_l, int32_t batch, int32_t length,
                           int32_t* start, int32_t* len, void* stream);
int fdb_launch_worklist(const int32_t* cu, int32_t batch, int32_t* wl, int32_t max_tiles, void* stream);
// one tensor (x1 == NULL) or two of one shape and one set of strides: fill, absmax and quantise in three launches
int fdb_launch_quant(const void* x0, const void* x1, int64_t x_st, int64_t x_sh, void* y0, void* y1, int64_t y_st, int64_t y_sh,
                     float* scale0, float* scale1, uint32_t* absmax_ws, int32_t tokens, int32_t heads, int32_t head_dim,
                     void* stream);
int fdb_launch_dequant(const void* y, int64_t y_st, int64_t y_sh, const float* scale, void* x, int64_t x_st, int64_t x_sh,
                       int32_t tokens, int32_t heads, int32_t head_dim, void* stream);

// Shared device helpers for the gfx950 speculative-decoding kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <limits.h>
#include <stdint.h>
#include <stdio.h>

#include <type_traits>

#include "../../include/sd_amd.h"

typedef __bf16 bf16_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

#define SD_WAVE 64

// Error text is per host thread; set by the launch wrappers.
void sd_set_error(const char* fmt, ...);
// True if sd_norm_linear / sd_norm_qkv_rope can hold M normalised rows of K columns in LDS.
bool sd_fused_norm_fits(int M, int K, bool layer_norm);

// Whether the fused-RMS-norm linear kernel works on two tiles a workgroup (tile 2 i and 2 i + 1 of workgroup i).
bool sd_linear_two_tiles_(int M, int n_tiles, int K, bool fp8);

// Weight ranges that the idle compute units of an attention launch read ahead of the launches
// that stream them (extra workgroups behind the attention grid): a matrix in 16-row tiles, or pairs of them, of
// tile_bytes, its first n_units work units (these, or half tiles: the 128-byte halves of every
// 256 bytes), unit u wanted by the XCD (u % consumer_grid) % 8.
struct sd_pf_range {
  const void* base;
  unsigned tile_bytes, n_units, half, consumer_grid;
};
// The range sd_linear (and its fused-norm forms) reads first for this matrix, at most max_bytes.
// fused_norm: of M rows (rms: RMSNorm).
sd_pf_range sd_linear_pf_range(const void* W, int M, int N, int K, int epi, int fp8, int fused_norm, int rms,
                               size_t max_bytes);
// Applies to the next attention launch of this host thread (then forgotten); n <= 2.
void sd_attn_prefetch_next(const sd_pf_range* r, int n);

// ---- what the kernels share whose operands come into LDS by direct loads (16 bytes a lane, no registers)
typedef __attribute__((address_space(3))) void lds_void;
constexpr unsigned kOutside = 0x80000000u;   // (buffers are smaller: reads of zero)
// (less than 4 GiB)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (unsigned)bytes, 0x00027000);
}
// Barrier of the workgroup behind this wave's LDS reads and all but the newest LEFT of its direct loads
// (__syncthreads() would wait for every load in flight in some places and for none in others: it does not count
// direct loads as LDS writes).
template <int LEFT>
__device__ __forceinline__ void meet() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LEFT) : "memory");
}
// Workgroups go round the 8 XCDs in launch order.  Each XCD takes a contiguous run of the work list, in which eight
// row blocks of one weight block are next to each other: the 32 or 64 blocks that an XCD runs at once then read
// about as many different weight blocks as row blocks, the least bytes for its L2 (all row blocks of a weight block
// next to each other: 963 TFLOP/s at 4096 rows of 14336, where 2048 rows reached 1197).
constexpr int kRowGroup = 8;
__device__ __forceinline__ int xcd_order(int id, int n) {
  const int q = n >> 3, r = n & 7, x = id & 7, i = id >> 3;
  return x * q + min(x, r) + i;
}

// Columns of a row that each of 256 threads asks for before it uses one (256 apart; the last one again for those past the row): body(U).
// A few rows are a chain of reads, each a round trip, so as many as eight; but no more than a narrow row has: of many rows each read counts, and
// those past the end cost as much as others.  us a column at a time / always eight / now: row norm of 4 rows of 2048 columns 4.5 / 3.3 / 3.4, 4096 of
// 256 5.9 / 7.5 / 5.2, 4096 of 2048 19.0 / 16.1 / 15.1; queries and keys normed and appended, 4096 of 256 9.4 / 11.6 / 8.6, 1024 of 1024 5.5 / 6.3 / 5.1, of
// 2560 (two batches, the second mostly past the end) 7.9 / 9.3 / 8.7; embedding 4096 of 256 5.0 / 5.7 / 5.0.
template <class F>
__device__ __forceinline__ void by_columns(int n, F body) {
  if (n <= 256) body(std::integral_constant<int, 1>());
  else if (n <= 512) body(std::integral_constant<int, 2>());
  else if (n <= 1024) body(std::integral_constant<int, 4>());
  else body(std::integral_constant<int, 8>());
}

// Layer-list models whose matrices are tiled: a portion of a pass with more rows than this runs on kernels for many
// rows, which sum in another order than those for few.  A portion's own rows decide, so that what shares its pass does
// not change its bits (linear layers, which have one rule for passes of up to 16 rows and one for others, aside).
constexpr int kLongPortion = 64;
// Whether row r belongs to a long portion (all lanes of a wave ask for the same row).
__device__ __forceinline__ bool sd_in_long_portion(const int32_t* entries, int n_entries, int r) {
  bool yes = false;
  for (int e = threadIdx.x & 63; e < n_entries; e += 64) {
    const int first = entries[4 * e + 1], rows = entries[4 * e + 2];
    yes |= (rows > kLongPortion) & (r >= first) & (r < first + rows);
  }
  return __any(yes);
}

// sd_decay_scan and sd_decay_scan_rows for the portions of at most max_rows rows.
int sd_decay_scan_(const float* q, const float* k, const float* v, int64_t ld, const float* decay, int per_channel,
                   float* state, const int32_t* entries, int n_entries, int max_rows, float* out, int H, int dk, int dv,
                   sd_stream_t stream);
int sd_decay_scan_rows_(const float* q, const float* k, int64_t ldqk, const float* v, int64_t ldv, const float* decay,
                        const float* k_scale, const void* skip, int w_f32, float* state, const int32_t* entries,
                        int n_entries, int max_rows, float* out, int H, int Gq, int dk, int dv, sd_stream_t stream);
// sd_decay_chunks / sd_head_decay_chunks with the long portions (chunks), the others (whole), or both.
struct sd_chunked_decay {
  const float *q, *k;
  int64_t ldqk;
  const float* v;
  int64_t ldv;
  const float* decay;
  int per;              // 0: decay [H], 1: [rows, H], 2: [rows, H*dk]
  const float* k_scale;
  const void* skip;
  int w_f32;
  float q_scale;
  float* state;
  const int32_t* entries;
  int n_entries, n_rows;
  float* out;
  int H, Gq, dk, dv;
};
int sd_decay_chunks_(const sd_chunked_decay* a, bool chunks, bool whole, void* scratch, size_t scratch_bytes,
                     sd_stream_t stream);

// sd_causal_conv_rows and sd_ssd_steps, in one launch where every entry is one row
int sd_conv_steps_(const float* x, int64_t ldx, const void* w, const void* b, int w_f32, float* conv_state, const int32_t* row_pos,
                   const int32_t* row_slot, const int32_t* entries, int n_entries, float* out, int64_t ldo, int n_rows, int C,
                   int taps, int act, const float* dt, const void* dt_bias, const void* a_log, float* step, float* decay, int H,
                   sd_stream_t stream);

// sd_postnorm_residual (one row of a each), and the router's product and choice (sd_moe_route_rows, sigmoid scores) on its result
int sd_postnorm_route_(float* x, const float* a, float sa, const float* b, float sb, const void* norm_w, int w_f32, float eps,
                       void* x_bf16, const void* w_router, float* logits, int32_t* sel_expert, float* sel_weight, int n_rows, int E,
                       int W, int top, sd_stream_t stream);

// sd_window_softmax_attention and sd_window_pool_attention without the rows of long portions (skip_long; the pooled
// blocks are in the cache already then), whose attention is sd_rows_softmax_attention's and sd_rows_pool_attention's:
// here with the long portions alone (long_only; all portions' blocks are pooled).
int sd_window_softmax_attention_(const float* q, int64_t ldq, const void* k_cache, const void* v_cache, int cache_f32,
                                 const int32_t* row_pos, const int32_t* row_slot, const int32_t* block_tables,
                                 int max_blocks, int page, int n_rows, int H, int G, int dk, int dv, int window,
                                 int keep_first, float scale, const int32_t* entries, int n_entries, bool skip_long,
                                 float* out, void* out_bf16, void* scratch, size_t scratch_bytes, sd_stream_t stream);
int sd_window_pool_attention_(const float* q, int64_t ldq, const void* k_cache, const void* v_cache, int cache_f32,
                              float* pk_cache, float* pv_cache, const int32_t* row_pos, const int32_t* row_slot,
                              const int32_t* block_tables, int max_blocks, int page, int n_rows, int H, int G, int dk,
                              int dv, int window, int pool, float scale, const float* head_bias, const int32_t* entries,
                              int n_entries, bool skip_long, float* out, void* scratch, size_t scratch_bytes,
                              sd_stream_t stream);
int sd_rows_softmax_attention_(const float* q, int64_t ldq, const void* k_cache, const void* v_cache,
                               const int32_t* block_tables, int max_blocks, int page, int n_rows, int H, int G, int dk,
                               int dv, int window, int keep_first, float scale, const int32_t* entries, int n_entries,
                               bool long_only, float* out, void* out_bf16, int64_t ldo, sd_stream_t stream);

// sd_gated_softmax_attention's tiled form (sd_seqmix_joint.hip); SD_ERR_UNSUPPORTED: sizes it does
// not take.
int sd_tiled_window_attention_(const float* q, int64_t ldq, const void* k_cache, const void* v_cache,
                               const int32_t* block_tables, int max_blocks, int page, int n_rows, int H,
                               int G, int dk, int dv, int window, int keep_first, float scale, float softcap,
                               const float* sinks, const float* dist1, const float* dist2, const float* gates,
                               int64_t ldg, const int32_t* entries, int n_entries, float* out, void* out_bf16,
                               int64_t ldo, sd_stream_t stream);

// Softmax attention of a prompt's rows on the matrix cores (sd_seqmix_attn.hip); v_cache nullptr: latent rows.
bool sd_rows_softmax_attention_fits_(int H, int G, int dk, int dv, int page, bool latent);
int sd_rows_pool_attention_(const float* q, int64_t ldq, const void* k_cache, const void* v_cache, const float* pk, const float* pv,
                            const int32_t* block_tables, int max_blocks, int n_rows, int H, int G, int window, int pool, int pslots,
                            float scale, const float* head_bias, const int32_t* entries, int n_entries, bool long_only,
                            float* out, sd_stream_t stream);

#define SD_REQUIRE(cond, code, ...)            \
  do {                                         \
    if (!(cond)) {                             \
      sd_set_error(__VA_ARGS__);               \
      return (code);                           \
    }                                          \
  } while (0)

#define SD_CHECK_LAUNCH(name)                                              \
  do {                                                                     \
    hipError_t e__ = hipGetLastError();                                    \
    if (e__ != hipSuccess) {                                               \
      sd_set_error("%s: launch failed: %s", name, hipGetErrorString(e__)); \
      return SD_ERR_HIP;                                                   \
    }                                                                      \
  } while (0)

static inline bool sd_aligned16(const void* p) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

__device__ __forceinline__ float bf16_to_f32(bf16_t v) { return (float)v; }
__device__ __forceinline__ bf16_t f32_to_bf16(float v) { return (bf16_t)v; }
// Round-trip through bf16: what a bf16 tensor op would have stored.
__device__ __forceinline__ float round_bf16(float v) { return (float)(bf16_t)v; }

// Eight e4m3 weights (two 32-bit words) as the bf16 MFMA operand: every e4m3 value is exact in
// bf16, so the f32 conversion is truncated to its upper half.
__device__ __forceinline__ bf16x8 fp8x8_to_bf16(uint32_t w0, uint32_t w1) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  const f32x2 a = __builtin_amdgcn_cvt_pk_f32_fp8(w0, false), b = __builtin_amdgcn_cvt_pk_f32_fp8(w0, true);
  const f32x2 c = __builtin_amdgcn_cvt_pk_f32_fp8(w1, false), d = __builtin_amdgcn_cvt_pk_f32_fp8(w1, true);
  auto pack = [](f32x2 v) {
    return __builtin_amdgcn_perm(__float_as_uint(v[1]), __float_as_uint(v[0]), 0x07060302u);
  };
  const u32x4 r = {pack(a), pack(b), pack(c), pack(d)};
  return __builtin_bit_cast(bf16x8, r);
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// Maximum and sum over a pair of lanes half a wave apart.
__device__ __forceinline__ float halves_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float halves_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Rotary position of frequency index i (0 <= i < D/2) of token row m of sequence b whose
// cache position is cache_pos: the cache position itself, or the multimodal one.
struct RopePos {
  const int32_t* pos;    // [3][rows] explicit positions, or null
  const int32_t* delta;  // [B] offset of all three components, or null
  int s_t, s_th;         // i < s_t: temporal, i < s_th: height, else width
  int rows;
};
__host__ inline RopePos sd_make_rope_pos(const sd_rope_positions* r, int rows) {
  RopePos o{nullptr, nullptr, 0, 0, rows};
  if (r) {
    o.pos = r->pos;
    o.delta = r->delta;
    o.s_t = r->section_t;
    o.s_th = r->section_t + r->section_h;
  }
  return o;
}
__device__ __forceinline__ int sd_rope_position(const RopePos& r, int cache_pos, int b, int m, int i) {
  if (r.pos) return r.pos[(size_t)(i < r.s_t ? 0 : (i < r.s_th ? 1 : 2)) * r.rows + m];
  return r.delta ? cache_pos + r.delta[b] : cache_pos;
}

// Slot of token t (0..15) inside a V page row: bits 2 and 3 swapped, so that
// the 8 consecutive slots a lane reads are the keys its accumulator registers
// hold after the K*Q^T MFMA.
__host__ __device__ __forceinline__ int sd_v_slot(int t) {
  return (t & 3) | (((t >> 3) & 1) << 2) | (((t >> 2) & 1) << 3);
}

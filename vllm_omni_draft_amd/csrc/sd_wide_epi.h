// What the many-row linear kernels share (sd_linear_wide.hip: 17..256 rows, sd_prompt.hip: more): how K is split
// and the epilogues, so that an output has the same bits whichever kernel summed it.
#pragma once
#include "sd_common.h"

namespace sd_wide {

constexpr int EPI_QKV_ROPE = 100;

constexpr int kWideThreads = 512;
constexpr int kWideWaves = kWideThreads / SD_WAVE;
constexpr int kTilesPerGroup = kWideWaves * 2;              // 16 tiles = 256 weight rows
// Matrices with fewer than kPairTiles tiles run with one tile per wave (8-tile groups): from
// kSmallTiles up that gives 128..255 workgroups in one pass with the epilogue inside; below,
// K is split (in shorter pieces than for the large matrices).
constexpr int kSmallTiles = 1024;
constexpr int kPairTiles = 2048;
constexpr int kChunkSteps = 4;                              // k-steps (32 columns) per LDS chunk
constexpr int kChunkCols = kChunkSteps * 32;

// K split: a function of the matrix alone (never of M), so results do not depend on the
// number of rows in the pass.
inline void plan_split(int n_tiles, int K, int& S, int& ks_per_split, int& group_tiles) {
  const int KS = K / 32;
  const bool small = n_tiles < kSmallTiles;
  group_tiles = n_tiles < kPairTiles ? kWideWaves : kTilesPerGroup;
  const int groups = (n_tiles + group_tiles - 1) / group_tiles;
  // one split (epilogue inside the kernel, no partial sums) once half the CUs have a
  // workgroup; otherwise enough splits for every CU
  int want = groups >= 128 ? 1 : 256 / groups;  // never more workgroups than CUs: one round
  const int min_steps = small ? 4 : 8;              // k-steps (32 columns) per split, at least
  const int max_s = (KS + min_steps - 1) / min_steps;
  want = want < 1 ? 1 : (want > max_s ? max_s : want);
  ks_per_split = ((KS + want - 1) / want + kChunkSteps - 1) / kChunkSteps * kChunkSteps;
  S = (KS + ks_per_split - 1) / ks_per_split;
}

inline int tiles_of(int N, int epi) { return epi == SD_EPI_SILU_MUL ? (N + 7) / 8 : (N + 15) / 16; }

__device__ __forceinline__ float silu_w(float v) { return v / (1.0f + __expf(-v)); }
__device__ __forceinline__ float gelu_tanh_w(float v) {
  const float c = 0.7978845608028654f;
  return 0.5f * v * (1.0f + tanhf(c * (v + 0.044715f * v * v * v)));
}

struct WideRope {
  const float* cs;
  int max_pos;
  bf16_t* kc;
  bf16_t* vc;
  const int32_t* block_tables;
  int max_blocks;
  const int32_t* seq_lens;
  int pos_offset, q_len, Hq, Hkv, D;
  RopePos mp;  // multimodal rotary positions (all null: the cache position)
  const int32_t* row_seq;  // a ragged pass: the block-table row of each token row (q_len 1, seq_lens per row); else null
};

struct WideEpiArgs {
  const float* part;  // [S][M][NR]
  int S, M, NR, N;
  const float* w_scale;  // fp8 weights: f32 scale per source row (indexed like bias); else null
  const float* x_scale;  // fp8 activations: f32 scale per token row; else null
  const bf16_t* bias;
  const bf16_t* residual;
  void* out;
  int64_t ldo;
  WideRope rope;
};

// Where row m of a QKV product goes: its position, and the page that holds it.
__device__ __forceinline__ int qkv_sequence(const WideRope& rp, int m) { return rp.q_len == 1 ? m : m / rp.q_len; }
__device__ __forceinline__ int qkv_position(const WideRope& rp, int m, int b) {
  return rp.seq_lens[b] + rp.pos_offset + m - b * rp.q_len;
}
__device__ __forceinline__ int qkv_page(const WideRope& rp, int b, int pos) {
  return rp.block_tables[(size_t)(rp.row_seq ? rp.row_seq[b] : b) * rp.max_blocks + (pos >> 4)];
}

// Four units (i0 .. i0 + 3 and their partners half a head on) of a rotated row: a lane's four queries, and its four keys, lie next
// to each other in memory, so they are one store of 8 bytes where the buffers' starts allow it (2 bytes at a time, 6144 x 4096 at
// 1024 rows 82.1 us, 4096 229; 8 bytes 76.3 and 206; 4608 x 3584 at 2946 rows of 8 prompts 138 and 130).
__device__ __forceinline__ void emit_qkv(const WideEpiArgs& a, int m, int tile, int r0, f32x4 lo, f32x4 hi, int b, int pos,
                                         int page) {
  const WideRope& rp = a.rope;
  const int D = rp.D, half = D / 2, tiles_per_head = D / 16;
  const int head = tile / tiles_per_head;
  const int i0 = (tile - head * tiles_per_head) * 8 + r0;
  const int slot = pos & 15;
  if (a.w_scale) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      lo[j] *= a.w_scale[head * D + i0 + j];
      hi[j] *= a.w_scale[head * D + i0 + j + half];
    }
  }
  if (a.bias) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      lo[j] += (float)a.bias[head * D + i0 + j];
      hi[j] += (float)a.bias[head * D + i0 + j + half];
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    lo[j] = round_bf16(lo[j]);
    hi[j] = round_bf16(hi[j]);
  }
  if (head < rp.Hq + rp.Hkv && rp.cs) {
    f32x4 c, sn;
    if (!rp.mp.pos && (reinterpret_cast<uintptr_t>(rp.cs) & 15) == 0) {   // (one position for all of a row)
      const float* cs = rp.cs + (size_t)min(max(sd_rope_position(rp.mp, pos, b, m, 0), 0), rp.max_pos - 1) * D + i0;
      c = *reinterpret_cast<const f32x4*>(cs);
      sn = *reinterpret_cast<const f32x4*>(cs + half);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r_pos = max(sd_rope_position(rp.mp, pos, b, m, i0 + j), 0);
        const float* cs = rp.cs + (size_t)min(r_pos, rp.max_pos - 1) * D;
        c[j] = cs[i0 + j];
        sn[j] = cs[half + i0 + j];
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float nl = lo[j] * c[j] - hi[j] * sn[j], nh = hi[j] * c[j] + lo[j] * sn[j];
      lo[j] = nl;
      hi[j] = nh;
    }
  }
  bf16x4 l, h;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    l[j] = (bf16_t)lo[j];
    h[j] = (bf16_t)hi[j];
  }
  auto four = [&](bf16_t* to, const bf16x4& v, bool aligned) __attribute__((always_inline)) {
    if (aligned) {
      *reinterpret_cast<bf16x4*>(to) = v;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) to[j] = v[j];
    }
  };
  if (head < rp.Hq) {
    bf16_t* q = reinterpret_cast<bf16_t*>(a.out) + (size_t)m * a.ldo + (size_t)head * D + i0;
    const bool aligned = (a.ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(a.out) & 7) == 0;
    four(q, l, aligned);
    four(q + half, h, aligned);
  } else if (head < rp.Hq + rp.Hkv) {
    bf16_t* kp = rp.kc + ((size_t)page * rp.Hkv + (head - rp.Hq)) * D * 16;
    const bool aligned = (reinterpret_cast<uintptr_t>(rp.kc) & 7) == 0;
    const int i2 = i0 + half;
    four(kp + ((i0 >> 3) * 16 + slot) * 8 + (i0 & 7), l, aligned);
    four(kp + ((i2 >> 3) * 16 + slot) * 8 + (i2 & 7), h, aligned);
  } else {
    bf16_t* vp = rp.vc + ((size_t)page * rp.Hkv + (head - rp.Hq - rp.Hkv)) * D * 16;
    const int sl = sd_v_slot(slot);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      vp[(i0 + j) * 16 + sl] = l[j];
      vp[(i0 + j + half) * 16 + sl] = h[j];
    }
  }
}

// Four neighbouring outputs of their sums (and residuals), and of their gate and up sums.
template <int EPI>
__device__ __forceinline__ bf16x4 four_of(const f32x4& y, const bf16x4& res) {
  bf16x4 r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (EPI == SD_EPI_STORE) r[j] = (bf16_t)y[j];
    else if (EPI == SD_EPI_RESIDUAL) r[j] = (bf16_t)(round_bf16(y[j]) + (float)res[j]);
    else if (EPI == SD_EPI_RELU) r[j] = (bf16_t)fmaxf(round_bf16(y[j]), 0.f);
    else r[j] = (bf16_t)gelu_tanh_w(round_bf16(y[j]));
  }
  return r;
}
__device__ __forceinline__ bf16x4 gated_of(const f32x4& g, const f32x4& up) {
  bf16x4 r;
#pragma unroll
  for (int j = 0; j < 4; ++j) r[j] = (bf16_t)(round_bf16(silu_w(round_bf16(g[j]))) * round_bf16(up[j]));
  return r;
}

// The epilogue of 4 consecutive tile rows r0..r0+3 of tile `tile` for token row m: lo holds
// their sums; in the paired modes hi holds the sums of rows r0+8..r0+11 (the up rows of a
// gated tile, the rotation partners of a rotary tile) and r0 is 0 or 4.
template <int EPI>
__device__ __forceinline__ void emit_unit(const WideEpiArgs& a, int m, int tile, int r0, f32x4 lo,
                                          f32x4 hi) {
  if (a.x_scale) {  // sums of products of fp8 activations: back to the row's scale first
    const float xs = a.x_scale[m];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      lo[j] *= xs;
      hi[j] *= xs;
    }
  }
  if (EPI == EPI_QKV_ROPE) {
    const WideRope& rp = a.rope;
    const int b = qkv_sequence(rp, m), pos = qkv_position(rp, m, b);
    if (pos < 0) return;
    emit_qkv(a, m, tile, r0, lo, hi, b, pos, tile / (rp.D / 16) >= rp.Hq ? qkv_page(rp, b, pos) : 0);
  } else if (EPI == SD_EPI_SILU_MUL) {
    const int n0 = tile * 8 + r0;
    if (n0 + 3 < a.N && ((a.ldo | a.N) & 3) == 0) {  // four outputs in one store
      f32x4 g = lo, up = hi;
      if (a.w_scale) {
        const f32x4 sg = *reinterpret_cast<const f32x4*>(a.w_scale + n0);
        const f32x4 su = *reinterpret_cast<const f32x4*>(a.w_scale + a.N + n0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          g[j] *= sg[j];
          up[j] *= su[j];
        }
      }
      if (a.bias) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          g[j] += (float)a.bias[n0 + j];
          up[j] += (float)a.bias[a.N + n0 + j];
        }
      }
      *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16_t*>(a.out) + (size_t)m * a.ldo + n0) = gated_of(g, up);
      return;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + j;
      if (n >= a.N) break;
      float g = lo[j], up = hi[j];
      if (a.w_scale) {
        g *= a.w_scale[n];
        up *= a.w_scale[a.N + n];
      }
      if (a.bias) {
        g += (float)a.bias[n];
        up += (float)a.bias[a.N + n];
      }
      g = round_bf16(silu_w(round_bf16(g)));
      reinterpret_cast<bf16_t*>(a.out)[(size_t)m * a.ldo + n] = (bf16_t)(g * round_bf16(up));
    }
  } else {
    const int n0 = tile * 16 + r0;
    if (n0 + 3 < a.N && (a.ldo & 3) == 0) {  // four outputs in one store
      f32x4 y = lo;
      if (a.w_scale) {
        const f32x4 sv = *reinterpret_cast<const f32x4*>(a.w_scale + n0);
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] *= sv[j];
      }
      if (a.bias) {
        const bf16x4 bv = *reinterpret_cast<const bf16x4*>(a.bias + n0);
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] += (float)bv[j];
      }
      const size_t o = (size_t)m * a.ldo + n0;
      if (EPI == SD_EPI_F32) {
        *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.out) + o) = y;
        return;
      }
      bf16x4 res = {0, 0, 0, 0};
      if (EPI == SD_EPI_RESIDUAL) res = *reinterpret_cast<const bf16x4*>(a.residual + o);
      *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16_t*>(a.out) + o) = four_of<EPI>(y, res);
      return;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + j;
      if (n >= a.N) break;
      float y = lo[j];
      if (a.w_scale) y *= a.w_scale[n];
      if (a.bias) y += (float)a.bias[n];
      const size_t o = (size_t)m * a.ldo + n;
      if (EPI == SD_EPI_F32) {
        reinterpret_cast<float*>(a.out)[o] = y;
      } else {
        bf16_t* ob = reinterpret_cast<bf16_t*>(a.out);
        if (EPI == SD_EPI_STORE) ob[o] = (bf16_t)y;
        else if (EPI == SD_EPI_RESIDUAL) ob[o] = (bf16_t)(round_bf16(y) + (float)a.residual[o]);
        else if (EPI == SD_EPI_RELU) ob[o] = (bf16_t)fmaxf(round_bf16(y), 0.f);
        else ob[o] = (bf16_t)gelu_tanh_w(round_bf16(y));
      }
    }
  }
}

}  // namespace sd_wide
using namespace sd_wide;

// sd_prompt.hip: the shapes its kernels are the better choice for (every other call goes through sd_linear_wide's in
// blocks of 256 rows; same bits), and the call.  epi: an SD_EPI_* number or EPI_QKV_ROPE with what that reads in `e`.
bool sd_rows_linear_fits_(int M, int n_tiles, int K, int64_t ldx, int S, int ks_per_split, int epi);
int sd_rows_linear_(const void* W, const void* x, int64_t ldx, int M, int K, int n_tiles, int S, int ks_per_split, int epi,
                    const sd_wide::WideEpiArgs& epi_args, float* part, sd_stream_t stream);
bool sd_rows_chain_fits_(int M, int n_tiles, int K, int64_t ldx, int S);  // (sd_prompt_linear_ takes these rows)
bool sd_prompt_linear_fits_(int M, int K, int64_t ldx);
bool sd_prompt_heads_fit_(const WideEpiArgs& e);  // (and EPI_QKV_ROPE's outputs)
int sd_prompt_linear_(const void* W, const void* x, int64_t ldx, int M, int K, int n_tiles, int epi,
                      const WideEpiArgs& e, sd_stream_t stream);
int sd_linear_wide_norm_(const void* W, const float* w_scale, const void* x, int64_t ldx, const void* bias, const void* residual,
                         void* out, int M, int N, int K, void* workspace, size_t workspace_bytes, const void* norm_w, float eps,
                         void* norm_out, sd_stream_t stream);  // (linear_wide's residual epilogue, and the rows' RMS norm)
int sd_prompt_shape_(int M, int n_tiles, int all_tiles, int K, int epi);
bool sd_prompt_relu_pair_fits_(int M, int n_tiles, int K, int64_t ldx, int gate_tile, int F);
int sd_prompt_relu_pair_(const void* W, const void* x, int64_t ldx, int M, int K, int n_tiles, int gate_tile, int F, float* y,
                         int64_t ldy, void* act, sd_stream_t stream);

// sd_linear_wide.hip: a linear layer over the rows of a prompt pass.  `e` holds what the epilogue reads (bias,
// residual, out, ldo, N; for EPI_QKV_ROPE the rope with one block-table row and position per row); w_scale: fp8
// weights; x_scales (2 x 256 floats): activations quantised per row as well.  workspace: of 256 rows.
int sd_linear_rows_(const void* W, const float* w_scale, float* x_scales, const void* x, int64_t ldx, int M, int K,
                    int n_tiles, int epi, const WideEpiArgs& e, void* workspace, size_t ws_bytes, sd_stream_t stream);

// Linear layers over more than 256 token rows (prompt passes), and over 33..256 where that is faster than sd_linear_wide's
// kernels, on the tiled bf16 weights of the other linear kernels.
//
// sd_linear_wide's kernels stream the weights past at most 256 rows held in LDS; a prompt of 1024 rows read
// every weight four times, split K over workgroups whenever a matrix had fewer than 128 groups (partial sums of
// S x rows x N floats written and read back) and left most of the matrix pipe idle (640 TFLOP/s on the split
// matrices of an 8B model without their second launch, 880 on gate/up).  With hundreds of rows the op is bound
// by the matrix pipe and by what feeds it.  Here both operands of a block pass through LDS by direct loads
// (16 bytes a lane, no registers), 64 columns a stage, two to four stages; four waves, each with its own TN x TM tiles
// of 16 x 16 in registers, so a fragment read from LDS feeds TM (or TN) MFMAs:
//   8 x 8 tiles a wave (256 x 256 a block), two stages: 64 B of LDS reads a clock against 128, one wave a SIMD, every
//     accumulator register there is; 7 x 8 and 8 x 6 where their blocks fill the chip's last round better;
//   2 x 2 to 4 x 8 (64 x 64 to 128 x 256): room for a second set of sums, and blocks for every CU of a small matrix;
//   2, 4 or 5 x 2, 4, 6 or 8 (all rows of a pass of 33..256), three stages: what is left is the weights' way from memory.
// Which of them a pass takes is what a model of their times says (kSplitShapes, kWholeShapes).
// The second set is for matrices whose K the narrower kernels split: a row's bits must not depend on how many
// rows share its pass, so the sums of a split are chained in one accumulator, and the splits' sums are added in
// index order from zero, as wide_epilogue_kernel adds them; in registers, without a second launch.
//
// What bounds a block is the way of its operands into LDS more than its MFMAs (4096 x 14336, 1024 rows, 128 x 128 blocks,
// 137 us: 84 without the loads, 135 without the products, 106 with all operands in the XCD's L2).  So a stage's direct
// loads are spread over the whole time between two barriers where a third stage leaves room for that (half of them behind
// the next stage's products: 400 -> 384 us at 4096 rows of 128 x 256), and the blocks whose stages are long enough ask
// for the lines of later stages ahead of time (prefetch: 366 -> 348 us for 256 x 256, 137 -> 124 for 128 x 128).
//
// A stage of a row is 128 bytes (8 pieces of 16); piece c of row r lies at slot c ^ (r & 7), which spreads the
// 16-row fragment reads over the banks; the source address carries the permutation, so a wave's direct load
// still covers whole 128-byte lines.  Loads past the matrix or past the last row are clamped or answered with
// zeros by the buffer's bounds; what they feed is never stored.
#include <type_traits>

#include "sd_common.h"
#include "sd_wide_epi.h"

namespace {

struct PromptArgs {
  const bf16_t* W;
  const bf16_t* x;
  int64_t ldx;
  int M, KS, n_tiles, ks_per_split;
  int n_blocks, m_blocks;  // grid = n_blocks * m_blocks (* splits: EPI_PARTIAL)
  float* part;             // EPI_PARTIAL: [splits][M][n_tiles * 16]
  int up_tiles;            // EPI_RELU_PAIR: from a gate tile to its up tile; n_tiles counts both
  WideEpiArgs epi;
};

constexpr int EPI_PARTIAL = -1;  // the sums of one split of K, for wide_epilogue_kernel
constexpr int EPI_RELU_PAIR = -2;  // bf16(relu(gate) * up) of two ranges of tiles of a stacked matrix

// Tile t of a block, from its first one
template <bool PAIR, int TN>
__device__ __forceinline__ int tile_at(int t, int up_tiles) {
  if (!PAIR) return t;
  const int i = t % TN;
  return t / TN * (TN / 2) + (i < TN / 2 ? i : i - TN / 2 + up_tiles);
}

// acc[i][j][reg] = (tile row 4 * xq + reg of tile i, token 16 j + xc), lane = 16 xq + xc: a lane holds four neighbouring outputs of a
// token.  Gated and rotary tiles hold the partners of rows 0..7 in rows 8..15, half a wave on: of two tiles the wave's halves
// change places, and each lane has both sums of four outputs of one of the two.
// A wave is alone on its SIMD here, and nothing hides what its epilogue waits for: through LDS, four tokens at a time, each trip a
// read, a residual's read, a chain of arithmetic and a store, 4096 x 4096 outputs of 4096 columns took 144 us, now 131 (with the residuals of
// sixteen tokens at a time 145: all of a wave's are asked for at once); 2946 x 3584 of 18944 363, now 348; 14336 gated outputs of 4096 columns,
// 1024 rows 194.5, now 191; 6144 x 4096 with rotation and pages, 1024 rows 74.5, now 63.6 (128 x 256 blocks; 128 x 128 70.9).
// The four lanes of a token and tile store 32 bytes (bf16), sixteen tokens at once; the L2 joins them.  f32 outputs, 64 bytes, go out as
// whole lines instead, eight tokens of two tiles at once (half lines: 2.5 % of a layer-list model's pass slower).
struct TileSums {
  f32x4 lo, hi;
};
__device__ __forceinline__ TileSums split_halves(const f32x4& even, const f32x4& odd) {
  TileSums s;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(even[e]), __float_as_uint(odd[e]), false, false);
    s.lo[e] = __uint_as_float(r[0]);
    s.hi[e] = __uint_as_float(r[1]);
  }
  return s;
}

// Of two tiles' sums of tokens 0..7 (even) and 8..15 (odd lanes of eight): lanes 8..15 of a row of sixteen give the first tile to the lanes eight below
// and take the second.  Then x0 holds tile (xc >> 3) of token xc & 7, x1 that of token 8 + (xc & 7).
__device__ __forceinline__ void trade_tiles(f32x4& x0, f32x4& x1, bool late) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float got = __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(late ? x0[e] : x1[e]), 0x128 /* row_ror:8 */, 0xf, 0xf, true));
    const float a = x0[e], b = x1[e];
    x0[e] = late ? got : a;
    x1[e] = late ? b : got;
  }
}

// A wave with more sums than there are vector registers beside them: the sums of a tile of tokens leave the accumulator registers when it is
// their turn (left alone the compiler brings all of them out first, and spills 24 to 240 registers a lane).
template <int TN, int TM>
__device__ __forceinline__ void in_turn(f32x4 (&acc)[TN][TM], int j) {
  if constexpr (TN * TM > 32) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < TN; ++i) asm volatile("" : "+a"(acc[i][j]));
  }
}

// Whether the outputs of all of a wave's tiles exist and a token's four neighbours are one store (`tiles` from `tile0`, `cols` outputs each)
__device__ __forceinline__ bool whole_tiles(const WideEpiArgs& a, int tile0, int tiles, int n_tiles, int cols) {
  return tile0 + tiles <= n_tiles && (tile0 + tiles) * cols <= a.N && ((a.ldo | a.N) & 3) == 0;
}

// EPI_RELU_PAIR: the tiles that exist, of n_tiles in all (their widths are whole tiles: there is no other epilogue for this one).  Other epilogues: all of
// the wave's tiles exist.
template <int EPI, int TN, int TM>
__device__ __forceinline__ void emit_tiles(const PromptArgs& p, f32x4 (&acc)[TN][TM], int tile0, int n_tiles, int row0, int lane) {
  const WideEpiArgs& a = p.epi;
  const int xc = lane & 15, xq = lane >> 4;
  if constexpr (EPI == SD_EPI_SILU_MUL) {
    bf16_t* out = reinterpret_cast<bf16_t*>(a.out) + (size_t)(row0 + xc) * a.ldo + (tile0 + (xq >> 1)) * 8 + (xq & 1) * 4;
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      const bool here = row0 + 16 * j + xc < p.M;
      in_turn(acc, j);
#pragma unroll
      for (int i = 0; i < TN; i += 2) {
        const TileSums s = split_halves(acc[i][j], acc[i + 1 < TN ? i + 1 : i][j]);
        const bf16x4 r = gated_of(s.lo, s.hi);
        if (here && (i + 1 < TN || xq < 2)) *reinterpret_cast<bf16x4*>(out + (size_t)16 * j * a.ldo + i * 8) = r;
      }
    }
  } else if constexpr (EPI == EPI_RELU_PAIR) {
    bf16_t* out = reinterpret_cast<bf16_t*>(a.out) + (size_t)(row0 + xc) * a.ldo + tile0 * 16 + xq * 4;
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      in_turn(acc, j);
      if (row0 + 16 * j + xc < p.M) {
#pragma unroll
        for (int i = 0; i < TN / 2; ++i) {
          if (tile0 + i >= n_tiles) break;
          bf16x4 r;
#pragma unroll
          for (int e = 0; e < 4; ++e) r[e] = (bf16_t)(fmaxf(acc[i][j][e], 0.f) * acc[i + TN / 2][j][e]);
          *reinterpret_cast<bf16x4*>(out + (size_t)16 * j * a.ldo + i * 16) = r;
        }
      }
    }
  } else if constexpr (EPI == SD_EPI_F32) {
    const int64_t ld = a.ldo;
    float* out = reinterpret_cast<float*>(a.out) + tile0 * 16 + xq * 4;
    const bool late = xc & 8;
    f32x4 bias[TN];
    if (a.bias) {
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        const bf16x4 b = *reinterpret_cast<const bf16x4*>(a.bias + (tile0 + i) * 16 + xq * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) bias[i][e] = (float)b[e];
      }
    }
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      in_turn(acc, j);
      const int m = row0 + 16 * j;
#pragma unroll
      for (int i = 0; i < TN; i += 2) {
        f32x4 y[2] = {acc[i][j], acc[i + 1 < TN ? i + 1 : i][j]};
        if (a.bias)
#pragma unroll
          for (int n = 0; n < 2; ++n) y[n] += bias[i + n < TN ? i + n : i];
        if (i + 1 < TN) {
          trade_tiles(y[0], y[1], late);
          float* to = out + (size_t)(m + (xc & 7)) * ld + (i + late) * 16;
          if (m + (xc & 7) < p.M) *reinterpret_cast<f32x4*>(to) = y[0];
          if (m + 8 + (xc & 7) < p.M) *reinterpret_cast<f32x4*>(to + 8 * ld) = y[1];
        } else if (m + xc < p.M) {
          *reinterpret_cast<f32x4*>(out + (size_t)(m + xc) * ld + i * 16) = y[0];
        }
      }
    }
  } else {
    const size_t at = (size_t)(row0 + xc) * a.ldo + tile0 * 16 + xq * 4;
    bf16_t* out = reinterpret_cast<bf16_t*>(a.out) + at;
    const bf16_t* residual = a.residual + at;
    // residuals of kBatch tiles of tokens at once, before the first store, which may change them for all the compiler knows
    constexpr int kBatch = EPI == SD_EPI_RESIDUAL && TN * TM > 32 ? 32 / TN : TM;
    bf16x4 bias[TN];
    if (a.bias) {
#pragma unroll
      for (int i = 0; i < TN; ++i) bias[i] = *reinterpret_cast<const bf16x4*>(a.bias + (tile0 + i) * 16 + xq * 4);
    }
#pragma unroll
    for (int j0 = 0; j0 < TM; j0 += kBatch) {
      bf16x4 res[kBatch][TN];
      if (EPI == SD_EPI_RESIDUAL) {
#pragma unroll
        for (int j = j0; j < TM && j < j0 + kBatch; ++j)
          if (row0 + 16 * j + xc < p.M) {
#pragma unroll
            for (int i = 0; i < TN; ++i) res[j - j0][i] = *reinterpret_cast<const bf16x4*>(residual + (size_t)16 * j * a.ldo + i * 16);
          }
      }
#pragma unroll
      for (int j = j0; j < TM && j < j0 + kBatch; ++j) {
        in_turn(acc, j);
        if (row0 + 16 * j + xc < p.M) {
#pragma unroll
          for (int i = 0; i < TN; ++i) {
            f32x4 y = acc[i][j];
            if (a.bias) {
#pragma unroll
              for (int e = 0; e < 4; ++e) y[e] += (float)bias[i][e];
            }
            *reinterpret_cast<bf16x4*>(out + (size_t)16 * j * a.ldo + i * 16) = four_of<EPI>(y, res[j - j0][i]);
          }
        }
        }
    }
  }
}

// The four tokens of a quad's lanes and four channels, turned: lane b of the quad has channel b's four tokens.
__device__ __forceinline__ bf16x4 turn_quad(const bf16x4& v, int lane) {
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  const u32x2 d = __builtin_bit_cast(u32x2, v);
  unsigned t[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {   // (channel 2 e + (lane & 1) of this lane's token and its neighbour's)
    const unsigned other = __builtin_amdgcn_mov_dpp(d[e], 0xB1, 0xf, 0xf, true);
    const bool odd = lane & 1;
    t[e] = __builtin_amdgcn_perm(odd ? d[e] : other, odd ? other : d[e], odd ? 0x07060302u : 0x05040100u);
  }
  const bool late = lane & 2;
  const unsigned other = __builtin_amdgcn_mov_dpp(late ? t[0] : t[1], 0x4E, 0xf, 0xf, true);
  const u32x2 r = {late ? other : t[0], late ? t[1] : other};
  return __builtin_bit_cast(bf16x4, r);
}

// One position for four neighbouring channels of a row (sections of them begin at multiples of four), four cosines in one load
__device__ __forceinline__ bool one_position_of_four(const WideRope& rp) {
  return (reinterpret_cast<uintptr_t>(rp.cs) & 15) == 0 && (!rp.mp.pos || ((rp.mp.s_t | rp.mp.s_th) & 3) == 0);
}

// A wave's tiles of a QKV product (those of n_tiles that exist): queries and keys rotated, keys and values into their pages.  A key's eight
// channels of a page are 16 bytes, next to the next token's; a page row of a value's channel holds its tokens side by side, so four tokens of
// a channel go in one store where they lie at neighbouring positions from a multiple of four on (others one by one).
// Two tiles of a head at a time: an even number of tiles a wave.  us of products whose rows have three positions or none, through LDS with a row's place
// looked up for every four outputs / this way: 4608 x 3584, three, 1024 rows 50.6 / 42.9, 2946 122 / 107; 2304 x 768, none, 2946 rows 25.0 / 19.7.
// kBatch tiles of tokens from J0 on: 8 x 8 tiles go four at a time (all eight's cosines and sines beside the accumulators: 19 registers a
// lane were spilled).
constexpr int heads_batch(int tn, int tm) { return tn * tm > 32 && tm % 4 == 0 ? 4 : tm; }
// PLAIN: all of the wave's tiles exist and one position turns four neighbouring channels, by cosines in one load (with the tests for the others
// inside, 18432 x 2048 at 4096 rows 325 us for 307).
template <int TN, int TM, bool PLAIN, int J0 = 0>
__device__ __forceinline__ void emit_heads(const PromptArgs& p, f32x4 (&acc)[TN][TM], int tile0, int row0, int lane) {
  const WideEpiArgs& a = p.epi;
  const WideRope& rp = a.rope;
  const int xc = lane & 15, xq = lane >> 4, D = rp.D, half = D / 2, tph = D / 16;
  static_assert(TN % 2 == 0, "two tiles of a head at a time");
  constexpr int kBatch = heads_batch(TN, TM);
  const bool fours = PLAIN || one_position_of_four(rp);
  auto turn_of = [&](int at) { return min(max(at, 0), rp.max_pos - 1); };
  int pos[kBatch], page[kBatch], turn[kBatch];   // position (-1: no such row), page, row of the cosines (without positions of their own)
  auto row_of = [&](int j) { return min(row0 + 16 * (J0 + j) + xc, p.M - 1); };
#pragma unroll
  for (int j = 0; j < kBatch; ++j) {
    const int m = row_of(j), b = qkv_sequence(rp, m);
    pos[j] = row0 + 16 * (J0 + j) + xc < p.M ? qkv_position(rp, m, b) : -1;
    turn[j] = !PLAIN && rp.mp.pos ? 0 : turn_of(sd_rope_position(rp.mp, pos[j], b, m, 0));
  }
  if ((tile0 + TN - 1) / tph >= rp.Hq) {
#pragma unroll
    for (int j = 0; j < kBatch; ++j) page[j] = pos[j] >= 0 ? qkv_page(rp, qkv_sequence(rp, row_of(j)), pos[j]) : 0;
  }
#pragma unroll
  for (int i = 0; i < TN; i += 2) {
    if (!PLAIN && tile0 + i >= p.n_tiles) break;
    if constexpr (TN * TM > 32) {   // (as in_turn)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = J0; j < J0 + kBatch; ++j) {
        asm volatile("" : "+a"(acc[i][j]));
        asm volatile("" : "+a"(acc[i + 1][j]));
      }
    }
    const int head = (tile0 + i) / tph, in_head = (tile0 + i - head * tph) * 8;
    if (head >= rp.Hq + rp.Hkv) {
      bf16_t* vp = rp.vc + (size_t)(head - rp.Hq - rp.Hkv) * D * 16;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int i0 = in_head + 8 * e + (xq & 1) * 4 + (xq >> 1) * half;   // channel of acc[..][0]
        f32x4 bias = {0.f, 0.f, 0.f, 0.f};
        if (a.bias)
#pragma unroll
          for (int c = 0; c < 4; ++c) bias[c] = (float)a.bias[head * D + i0 + c];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
          const f32x4& y = acc[i + e][J0 + j];
          bf16x4 v;
#pragma unroll
          for (int c = 0; c < 4; ++c) v[c] = (bf16_t)(a.bias ? y[c] + bias[c] : y[c]);
          const int p0 = __builtin_amdgcn_mov_dpp(pos[j], 0, 0xf, 0xf, true), g0 = __builtin_amdgcn_mov_dpp(page[j], 0, 0xf, 0xf, true);
          const unsigned long long ok = __ballot(pos[j] >= 0 && (p0 & 3) == 0 && pos[j] == p0 + (lane & 3) && page[j] == g0);
          const bf16x4 t = turn_quad(v, lane);
          bf16_t* to = vp + (size_t)page[j] * rp.Hkv * D * 16;
          if ((ok >> (lane & 60) & 15) == 15) {
            *reinterpret_cast<bf16x4*>(to + (i0 + (lane & 3)) * 16 + sd_v_slot(p0 & 15)) = t;
          } else if (pos[j] >= 0) {
#pragma unroll
            for (int c = 0; c < 4; ++c) to[(i0 + c) * 16 + sd_v_slot(pos[j] & 15)] = v[c];
          }
        }
      }
      continue;
    }
    const int i0 = in_head + (xq >> 1) * 8 + (xq & 1) * 4;   // channel of the even halves' first sum
    f32x4 b_lo = {0.f, 0.f, 0.f, 0.f}, b_hi = b_lo;
    if (a.bias)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        b_lo[c] = (float)a.bias[head * D + i0 + c];
        b_hi[c] = (float)a.bias[head * D + i0 + half + c];
      }
    auto put = [&](auto rotated) __attribute__((always_inline)) {
      constexpr bool kRotated = decltype(rotated)::value;
      f32x4 cs[kBatch], sn[kBatch];
      if constexpr (kRotated) {
        int at[kBatch];
        if (!PLAIN && rp.mp.pos) {
#pragma unroll
          for (int j = 0; j < kBatch; ++j) at[j] = turn_of(sd_rope_position(rp.mp, 0, 0, row_of(j), i0));
        } else {
#pragma unroll
          for (int j = 0; j < kBatch; ++j) at[j] = turn[j];
        }
        if (fours) {
#pragma unroll
          for (int j = 0; j < kBatch; ++j) {
            cs[j] = *reinterpret_cast<const f32x4*>(rp.cs + (size_t)at[j] * D + i0);
            sn[j] = *reinterpret_cast<const f32x4*>(rp.cs + (size_t)at[j] * D + i0 + half);
          }
        } else {
#pragma unroll
          for (int j = 0; j < kBatch; ++j)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              const int to = rp.mp.pos && c ? turn_of(sd_rope_position(rp.mp, 0, 0, row_of(j), i0 + c)) : at[j];
              cs[j][c] = rp.cs[(size_t)to * D + i0 + c];
              sn[j][c] = rp.cs[(size_t)to * D + i0 + half + c];
            }
        }
      }
#pragma unroll
      for (int j = 0; j < kBatch; ++j) {
        const TileSums s = split_halves(acc[i][J0 + j], acc[i + 1][J0 + j]);
        bf16x4 l, h;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float lo = round_bf16(a.bias ? s.lo[c] + b_lo[c] : s.lo[c]), hi = round_bf16(a.bias ? s.hi[c] + b_hi[c] : s.hi[c]);
          if constexpr (kRotated) {
            l[c] = (bf16_t)(lo * cs[j][c] - hi * sn[j][c]);
            h[c] = (bf16_t)(hi * cs[j][c] + lo * sn[j][c]);
          } else {
            l[c] = (bf16_t)lo;
            h[c] = (bf16_t)hi;
          }
        }
        if (pos[j] < 0) {
        } else if (head < rp.Hq) {
          bf16_t* q = reinterpret_cast<bf16_t*>(a.out) + (size_t)(row0 + 16 * (J0 + j) + xc) * a.ldo + head * D + i0;
          *reinterpret_cast<bf16x4*>(q) = l;
          *reinterpret_cast<bf16x4*>(q + half) = h;
        } else {
          bf16_t* k = rp.kc + ((size_t)page[j] * rp.Hkv + (head - rp.Hq)) * D * 16 + (pos[j] & 15) * 8 + (i0 & 7);
          *reinterpret_cast<bf16x4*>(k + (i0 >> 3) * 128) = l;
          *reinterpret_cast<bf16x4*>(k + ((i0 + half) >> 3) * 128) = h;
        }
      }
    };
    if constexpr (PLAIN) put(std::true_type{});
    else if (rp.cs) put(std::true_type{});
    else put(std::false_type{});
  }
  if constexpr (J0 + kBatch < TM) emit_heads<TN, TM, PLAIN, J0 + kBatch>(p, acc, tile0, row0, lane);
}

// Blocks a CU has room for: LDS, and the registers of two sets of accumulators.
constexpr int blocks_per_cu(int tn, int tm, int stages, bool split) {
  const int lds = 160 / (4 * (tn + tm) * stages), regs = !split || tn * tm > 16 ? 1 : tn * tm <= 4 ? 3 : 2;
  return lds < regs ? lds : regs;
}

// AHEAD: how many stages behind the one being loaded a line is asked for (0: none).
template <int TN, int TM, int STAGES, bool SPLIT, int EPI, int AHEAD>
__global__ __launch_bounds__(256, blocks_per_cu(TN, TM, STAGES, SPLIT)) void prompt_gemm_kernel(PromptArgs a) {
  constexpr bool kAccV = SPLIT && TN * TM <= 16;       // accumulators in vector registers: both sets fit beside the fragments
  constexpr int BN = 2 * TN, BM = 2 * TM * 16;         // weight tiles and token rows of the block
  constexpr int kABytes = BN * 2 * 1024, kBBytes = BM * 128;
  constexpr int kAPieces = BN * 2 / 4, kBPieces = BM / 8 / 4;  // 1 KiB direct loads per wave and stage
  __shared__ __attribute__((aligned(1024))) char s0[kABytes + kBBytes];
  __shared__ __attribute__((aligned(1024))) char s1[kABytes + kBBytes];
  __shared__ __attribute__((aligned(1024))) char s2[STAGES >= 3 ? kABytes + kBBytes : 1024];
  __shared__ __attribute__((aligned(1024))) char s3[STAGES == 4 ? kABytes + kBBytes : 1024];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int blocks = EPI == EPI_PARTIAL ? a.n_blocks * a.m_blocks : (int)gridDim.x;
  const int split = EPI == EPI_PARTIAL ? (int)blockIdx.x / blocks : 0;
  const int work = xcd_order(blockIdx.x - split * blocks, blocks);
  const int grp = work / (a.n_blocks * kRowGroup), in_grp = work - grp * a.n_blocks * kRowGroup;
  const int grp_rows = min(kRowGroup, a.m_blocks - grp * kRowGroup);
  const int nb = in_grp / grp_rows, mb = grp * kRowGroup + in_grp - nb * grp_rows;
  // EPI_RELU_PAIR: half of the block's tiles are gate tiles, half the up tiles that belong to them, in every wave
  constexpr bool PAIR = EPI == EPI_RELU_PAIR;
  static_assert(!PAIR || TN % 2 == 0, "gate and up tiles of a wave");
  const int tile0 = PAIR ? nb * TN : nb * BN, row0 = mb * BM;
  const int up_tiles = a.up_tiles;
  const int k0 = split * a.ks_per_split;               // first k-step (EPI_PARTIAL)
  const int n_it = EPI == EPI_PARTIAL ? min(a.ks_per_split, a.KS - k0) >> 1 : a.KS >> 1;

  // this wave's direct loads: weights, piece p = (tile p >> 1, k-step p & 1) of the block's tiles
  const char* wbase = reinterpret_cast<const char*>(a.W) + (size_t)tile0 * a.KS * 1024;
  const int live_tiles = PAIR ? a.up_tiles + min(TN, a.n_tiles / 2 - tile0) : min(BN, a.n_tiles - tile0);
  const auto wr = buffer_of(wbase, (unsigned)min((size_t)live_tiles * a.KS * 1024, (size_t)0xffffffffu));
  const int w_step = a.KS * 1024;
  // rows, piece p = rows 8p .. 8p + 7 of the block
  const char* xbase = reinterpret_cast<const char*>(a.x) + (size_t)row0 * a.ldx * 2;
  const int live_rows = min(BM, a.M - row0);
  const auto xr = buffer_of(xbase, (unsigned)((size_t)(live_rows - 1) * a.ldx * 2 + (size_t)a.KS * 64));
  const unsigned x_lane = (unsigned)(lane >> 3) * (unsigned)a.ldx * 2 + (((lane & 7) ^ (lane >> 3)) << 4);
  const unsigned x_step = 8u * (unsigned)a.ldx * 2;
  constexpr int kPieces = kAPieces + kBPieces;
  auto stage_piece = [&](char* s, int it, int i) __attribute__((always_inline)) {
    if (i < kAPieces) {
      const int p = wave + 4 * i;
      // (the tile is part of the lane offset: that is what the bounds check sees)
      const int at = lane * 16 + tile_at<PAIR, TN>(p >> 1, up_tiles) * w_step;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)(s + p * 1024), 16, at,
                                               (k0 + 2 * it + (p & 1)) * 1024, 0, 0);
    } else {
      const int p = wave + 4 * (i - kAPieces);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void*)(s + kABytes + p * 1024), 16, x_lane + p * x_step,
                                               k0 * 64 + it * 128, 0, 0);
    }
  };

  // Lines of a later stage, asked for by one load a wave into a place nobody reads, so that the direct loads find them
  // in the XCD's L2.  The row blocks of a weight block, next to each other on an XCD, share its lines; a row block's
  // lines are shared by the four weight blocks that an XCD runs at a time.  (128 x 128: weights alone; its rows' lines
  // cost more than they give, 128 -> 124 us.)
  __shared__ __attribute__((aligned(1024))) char unread[AHEAD ? 1024 : 16];
  unsigned ahead_off = 0xffffffffu;  // (out of bounds: no access)
  if (AHEAD) {
    const int l = (wave & 1) * 64 + lane;
    if (wave < 2) {
      constexpr int kLines = BN * 16;
      const int n = (kLines + grp_rows - 1) / grp_rows, line = (mb - grp * kRowGroup) * n + l;
      if (l < n && line < kLines) ahead_off = (unsigned)tile_at<PAIR, TN>(line >> 4, up_tiles) * (unsigned)w_step + (line & 15) * 128;
    } else if (!SPLIT) {
      const int line = (nb & 3) * (BM / 4) + l;
      if (l < BM / 4) ahead_off = (unsigned)line * (unsigned)a.ldx * 2;
    }
  }
  const auto ahead_of = wave < 2 ? wr : xr;
  auto prefetch = [&](int it) __attribute__((always_inline)) {
    it = min(it, n_it - 1);
    if (AHEAD)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ahead_of, (lds_void*)(unread + (AHEAD ? wave * 256 : 0)), 4, ahead_off,
                                               wave < 2 ? (k0 + 2 * it) * 1024 : k0 * 64 + it * 128, 0, 0);
  };

  const int wn = wave & 1, wm = wave >> 1;
  const int xc = lane & 15, xq = lane >> 4;
  const int a_off = wn * TN * 2048 + lane * 16;
  const int b_row = kABytes + (wm * TM * 16 + xc) * 128;
  const int b_sw[2] = {((xq ^ (xc & 7)) << 4), (((xq + 4) ^ (xc & 7)) << 4)};
  bf16x8 fa[2][TN], fb[2][TM];
  constexpr int kReads = TN + TM, kMfma = TN * TM;
  constexpr int kOver = kMfma * 3 / 4 > kReads ? kMfma * 3 / 4 : kReads;
  // A stage's direct loads: the first kEarly behind the barrier that frees its place, the others behind the next
  // stage's first products (two stages: no time for that).  Splits of K of more than 128 rows ask for all of them at once: their
  // blocks have few stages, and the rows' part of one is most of it.  us, spread / at once: 3584 x 18944 192 rows 47.3 / 44.9, 4096 x
  // 14336 256 rows 47.0 / 45.4, 8192 x 8192 224 rows 51.0 / 46.5, 2048 x 8192 256 rows 29.6 / 28.4 (3584 x 3584 23.2 / 23.7); but 4096 x 4096
  // 100 rows 18.0 / 18.4, 8192 x 8192 128 rows 37.9 / 38.9.
  constexpr int kEarly = STAGES >= 3 && !(EPI == EPI_PARTIAL && TM >= 6) ? kPieces / 2 : kPieces;
  static_assert(kReads <= kMfma && kEarly <= kMfma && kPieces - kEarly <= kMfma, "at most one LDS read and one direct load an MFMA");
  // what is in flight and newer than the next stage at a step's barrier
  constexpr int kAheadLeft = AHEAD == 0 ? 0 : STAGES >= 3 ? STAGES - 2 : 1;
  static_assert(AHEAD == 0 || AHEAD >= kAheadLeft, "the barriers of the first steps count as many prefetches as later ones");
  auto read_piece = [&](const char* s, int ks, int i) __attribute__((always_inline)) {
    if (i < TN)
      fa[ks][i] = *reinterpret_cast<const bf16x8*>(s + a_off + i * 2048 + ks * 1024);
    else
      fb[ks][i - TN] = *reinterpret_cast<const bf16x8*>(s + b_row + (i - TN) * 2048 + b_sw[ks]);
  };
  f32x4 acc[TN][TM], tot[SPLIT ? TN : 1][SPLIT ? TM : 1];
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      acc[i][j] = zero;
      if (SPLIT) tot[i][j] = zero;
    }
  // Left to itself the compiler moves accumulators between registers around its MFMAs (two moves per MFMA in the
  // largest shape: 876 TFLOP/s where 1050 are reached in place, 8192 x 2 x 1024 outputs of 4096), so the instruction
  // is written out with its accumulator tied in place.  The wait states that the compiler would insert between it
  // and other accesses of the accumulators are then placed by hand (settle).
  auto settle = [&]() __attribute__((always_inline)) {
    asm volatile("s_nop 15\n\ts_nop 15");
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        if constexpr (kAccV) asm volatile("" : "+v"(acc[i][j]));
        else asm volatile("" : "+a"(acc[i][j]));
      }
    asm volatile("s_nop 15");
  };
  auto mfma = [&](int ks, int i, int j) __attribute__((always_inline)) {
    if constexpr (kAccV)
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc[i][j]) : "v"(fa[ks][i]), "v"(fb[ks][j]));
    else
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(fa[ks][i]), "v"(fb[ks][j]));
  };
  // The MFMAs of one k-step with the next one's LDS reads (`from`) and direct loads FIRST .. LAST - 1 of stage `it`
  // between them
  auto phase = [&](auto k_step, const char* from, auto first, auto last, char* to, int it) __attribute__((always_inline)) {
    constexpr int ks = decltype(k_step)::value;
    constexpr int kFirst = decltype(first)::value, kLoads = decltype(last)::value - kFirst;
#pragma unroll
    for (int n = 0; n < kMfma; ++n) {
      mfma(ks, n / TM, n % TM);
      // (the reads in the first three quarters: the last one has its latency behind it at the phase's end)
      if (n < kOver && (n + 1) * kReads / kOver > n * kReads / kOver) read_piece(from, ks ^ 1, n * kReads / kOver);
      if (kLoads && (n + 1) * kLoads / kMfma > n * kLoads / kMfma) stage_piece(to, min(it, n_it - 1), kFirst + n * kLoads / kMfma);
    }
  };
  const int its_per_split = SPLIT ? a.ks_per_split >> 1 : 0;
  int next_split = its_per_split;
  // One stage of 64 columns: `cur` holds it (its first k-step's fragments are in registers already), `nxt` the
  // stage behind it; cur's place is then loaded with the stage STAGES further on (`prev`: the stage before, whose place
  // is being loaded).
  auto step = [&](char* cur, char* nxt, char* prev, int it) __attribute__((always_inline)) {
    constexpr std::integral_constant<int, 0> zero_c{};
    constexpr std::integral_constant<int, 1> one_c{};
    constexpr std::integral_constant<int, kEarly> early{};
    constexpr std::integral_constant<int, kPieces> all{};
    phase(zero_c, cur, early, all, prev, it - 1 + STAGES);
    // every wave has read `cur` and its own part of `nxt` has landed
    meet<(STAGES - 2) * kPieces + kAheadLeft>();
    phase(one_c, nxt, zero_c, early, cur, it + STAGES);
    prefetch(it + STAGES + AHEAD);
    if (SPLIT && it + 1 == next_split && it + 1 < n_it) {
      settle();
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) {
          tot[i][j] += acc[i][j];
          acc[i][j] = zero;
        }
      next_split += its_per_split;
      settle();
    }
  };
  auto fill = [&](char* s, int it) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < (it == STAGES - 1 ? kEarly : kPieces); ++i) stage_piece(s, min(it, n_it - 1), i);
  };
  fill(s0, 0);
  fill(s1, 1);
  if constexpr (STAGES >= 3) fill(s2, 2);
  if constexpr (STAGES == 4) fill(s3, 3);
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) prefetch(STAGES + i);
  meet<(STAGES - 2) * kPieces + kEarly + AHEAD>();
#pragma unroll
  for (int i = 0; i < kReads; ++i) read_piece(s0, 0, i);
  settle();
  int it = 0;
  if constexpr (STAGES == 4) {
    for (; it + 3 < n_it; it += 4) {
      step(s0, s1, s3, it);
      step(s1, s2, s0, it + 1);
      step(s2, s3, s1, it + 2);
      step(s3, s0, s2, it + 3);
    }
    if (it < n_it) step(s0, s1, s3, it);
    if (it + 1 < n_it) step(s1, s2, s0, it + 1);
    if (it + 2 < n_it) step(s2, s3, s1, it + 2);
  } else if constexpr (STAGES == 3) {
    for (; it + 2 < n_it; it += 3) {
      step(s0, s1, s2, it);
      step(s1, s2, s0, it + 1);
      step(s2, s0, s1, it + 2);
    }
    if (it < n_it) step(s0, s1, s2, it);
    if (it + 1 < n_it) step(s1, s2, s0, it + 1);
  } else {
    for (; it + 1 < n_it; it += 2) {
      step(s0, s1, s1, it);
      step(s1, s0, s0, it + 1);
    }
    if (it < n_it) step(s0, s1, s1, it);
  }
  meet<0>();  // no direct load outlives the workgroup's use of LDS
  settle();

  if (SPLIT) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) acc[i][j] = tot[i][j] + acc[i][j];
  }
  if constexpr (PAIR) {
    emit_tiles<EPI, TN, TM>(a, acc, tile0 + wn * (TN / 2), a.n_tiles / 2, row0 + wm * TM * 16, lane);
    return;
  } else if constexpr (EPI == EPI_QKV_ROPE) {
    const int first = tile0 + wn * TN;
    if (a.epi.rope.cs && !a.epi.rope.mp.pos && one_position_of_four(a.epi.rope) && first + TN <= a.n_tiles)
      emit_heads<TN, TM, true>(a, acc, first, row0 + wm * TM * 16, lane);
    else emit_heads<TN, TM, false>(a, acc, first, row0 + wm * TM * 16, lane);
    return;
  } else if constexpr (EPI != EPI_PARTIAL) {
    const int first = tile0 + wn * TN;
    if (whole_tiles(a.epi, first, TN, a.n_tiles, EPI == SD_EPI_SILU_MUL ? 8 : 16) && !(EPI == SD_EPI_SILU_MUL && a.epi.bias)) {
      emit_tiles<EPI, TN, TM>(a, acc, first, a.n_tiles, row0 + wm * TM * 16, lane);
      return;
    }
  }
  // Other outputs, and the partial sums of splits (3584 x 3584 at 107 / 192 / 256 rows 15.9 / 19.8 / 23.2 us with their epilogue's launch, from
  // registers 16.3 / 20.6 / 23.9), through LDS, 16 token rows at a time and each wave for itself, so that the lanes of a store hold
  // neighbouring outputs of a row (and the epilogue is there once per token tile, not once per pair of tiles).
  constexpr bool PAIRED = EPI == SD_EPI_SILU_MUL;
  constexpr int kLd = TN * 16 + 4;                        // floats; 16 rows start on different banks
  constexpr int kUnits = PAIRED ? TN * 2 : TN * 4;        // of a row; 64 lanes take 64 / kUnits rows at once
  float* img = reinterpret_cast<float*>(wave < 2 ? s0 : s1) + (wave & 1) * 16 * kLd;
  const int u = lane % kUnits, ui = PAIRED ? u >> 1 : u >> 2, r0 = PAIRED ? (u & 1) * 4 : (u & 3) * 4;
  const int tile = tile0 + wn * TN + ui;
#pragma unroll
  for (int j = 0; j < TM; ++j) {
#pragma unroll
    for (int i = 0; i < TN; ++i) *reinterpret_cast<f32x4*>(img + xc * kLd + i * 16 + 4 * xq) = acc[i][j];
    asm volatile("" ::: "memory");  // (other lanes read them: the stores of a lane without a unit stay here)
#pragma unroll 1
    for (int r = lane < 64 / kUnits * kUnits ? lane / kUnits : 16; r < 16; r += 64 / kUnits) {
      const int m = row0 + (wm * TM + j) * 16 + r;
      const float* src = img + r * kLd + ui * 16 + r0;
      const f32x4 lo = *reinterpret_cast<const f32x4*>(src);
      f32x4 hi = zero;
      if (PAIRED) hi = *reinterpret_cast<const f32x4*>(src + 8);
      if (tile < a.n_tiles && m < a.M) {
        if constexpr (EPI == EPI_PARTIAL)
          *reinterpret_cast<f32x4*>(a.part + ((size_t)split * a.M + m) * a.n_tiles * 16 + tile * 16 + r0) = lo;
        else emit_unit<EPI>(a.epi, m, tile, r0, lo, hi);
      }
    }
  }
}

template <int TN, int TM, int STAGES, bool SPLIT, int EPI, int AHEAD = 0>
int launch_prompt(PromptArgs a, hipStream_t st) {
  a.n_blocks = (a.n_tiles + 2 * TN - 1) / (2 * TN);
  a.m_blocks = (a.M + 32 * TM - 1) / (32 * TM);
  hipLaunchKernelGGL((prompt_gemm_kernel<TN, TM, STAGES, SPLIT, EPI, AHEAD>), dim3(a.n_blocks * a.m_blocks), dim3(256), 0, st, a);
  SD_CHECK_LAUNCH("sd_prompt_linear");
  return SD_OK;
}

// ---- passes of at most 256 rows: one block holds all of them, so every weight is read once; four waves, three stages.
// The MFMAs need the accumulators in place here too; 192 rows x 10 weight tiles a block are 120 of them a lane.
template <int TN, int EPI>
int launch_few(PromptArgs a, int S, hipStream_t st) {
  a.n_blocks = (a.n_tiles + 2 * TN - 1) / (2 * TN);
  a.m_blocks = 1;
  const dim3 grid(a.n_blocks * S);
  if (a.M <= 64) hipLaunchKernelGGL((prompt_gemm_kernel<TN, 2, 3, false, EPI, 0>), grid, dim3(256), 0, st, a);
  else if (a.M <= 128) hipLaunchKernelGGL((prompt_gemm_kernel<TN, 4, 3, false, EPI, 0>), grid, dim3(256), 0, st, a);
  else if (a.M <= 192) hipLaunchKernelGGL((prompt_gemm_kernel<TN, 6, 3, false, EPI, 0>), grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((prompt_gemm_kernel<TN, 8, 3, false, EPI, 0>), grid, dim3(256), 0, st, a);
  SD_CHECK_LAUNCH("sd_rows_linear");
  return SD_OK;
}

// Tiles a wave of a matrix whose K is whole: the fewest rounds of 256 blocks x tiles a block, larger blocks where that is
// the same.
int few_cost(int n_tiles, int tn) { return ((n_tiles + 2 * tn - 1) / (2 * tn) + 255) / 256 * tn; }
int few_tiles(int n_tiles) {
  const int c2 = few_cost(n_tiles, 2), c4 = few_cost(n_tiles, 4), c5 = few_cost(n_tiles, 5);
  return c5 <= c4 && c5 <= c2 ? 5 : c4 <= c2 ? 4 : 2;
}

template <int EPI>
int few_shape(const PromptArgs& a, hipStream_t st) {
  const int tn = few_tiles(a.n_tiles);
  if (tn == 5) return launch_few<5, EPI>(a, 1, st);
  return tn == 4 ? launch_few<4, EPI>(a, 1, st) : launch_few<2, EPI>(a, 1, st);
}

// The block of a prompt pass: the shape whose time by this model is the least.  The blocks go over the chip in rounds of 256 x
// per_cu; a round takes `fixed` us (launch, first loads, epilogue), `split` us a split of K (its sums join the others')
// and `stage` us a stage of 64 columns, which depends on how many blocks share a CU.  Fitted to 342 passes with epilogues through LDS, which took 2 to
// 8 us a block longer than those from registers; with these, over 672 passes (N 512..32000, K 768..18944, 272..4096 rows, weights from memory),
// the shapes it takes are .7 % (368 of split K), .6 % (128 QKV products), .4 % (96 gated, whole K) and 1.4 % (80 plain, whole K) slower than the
// best of all, where constants fitted to these times are .7, 1.5, .2 and .5 %.  128 x 128 throughout, two a CU, is 43, 29, 24 and 15 %
// slower than the shapes chosen.  us, chosen shape against 128 x 128: 1024 x 2048 at 1024 rows 13.3 (64 x 64) and 26.7; 4096 x 4096 at 512 rows 28.1
// (64 x 128) and 55.3; 6144 x 4096 with rotation at 1024 rows 63.6 (128 x 256) and 72.5; 3584 x 18944 at 2946 rows 345 (128 x 192) and 467; whole K,
// 14336 x 4096 gated: 1024 rows 181 (224 x 256) and 264, 300 rows 82 (256 x 192) and 117.
struct Shape {
  int tn, tm, per_cu;
  float fixed, split, stage[3];
};
constexpr Shape kSplitShapes[] = {
    {2, 2, 3, 3.8f, 0.f, {.283f, .419f, .590f}}, {4, 2, 2, 5.2f, 0.f, {.384f, .624f}}, {2, 4, 1, 5.5f, .09f, {.310f}},
    {4, 3, 1, 7.2f, .03f, {.397f}},              {4, 4, 1, 9.2f, .04f, {.480f}},       {4, 4, 2, 6.9f, 0.f, {.712f, .978f}},
    {4, 5, 1, 10.8f, .28f, {.522f}},             {4, 6, 1, 12.6f, .31f, {.577f}},      {4, 8, 1, 15.4f, .47f, {.715f}}};
constexpr Shape kWholeShapes[] = {
    {8, 8, 1, 16.2f, 0.f, {1.236f}},      {7, 8, 1, 8.7f, 0.f, {1.295f}},  {8, 6, 1, 12.3f, 0.f, {1.023f}},
    {4, 4, 2, 4.1f, 0.f, {.813f, .958f}}, {4, 4, 1, 5.8f, 0.f, {.477f}},   {4, 6, 1, 8.9f, 0.f, {.562f}}};

float shape_us(const Shape& s, int M, int n_tiles, int K, int S, int epi) {
  const long blocks = (long)((n_tiles + 2 * s.tn - 1) / (2 * s.tn)) * ((M + 32 * s.tm - 1) / (32 * s.tm));
  const long round = 256l * s.per_cu, full = blocks / round, rest = blocks - full * round;
  // The epilogue that rotates and writes pages is longer than a plain one, and nothing covers that of a large block alone on its CU.
  // Of 128 QKV products (1152 x 896 to 10240 x 8192, 272..4096 rows) the shapes with .25 a tile are .6 % slower than the best of all, with 0 .7 %, with
  // .5 (which the epilogue through LDS took) 1.0 %; any from .16 to .37 chooses the same.  us with .5 (128 x 128, two a CU) / with .25 (128 x 256):
  // 6144 x 4096 at 1024 rows 72.5 / 63.6, 2500 130 / 125, 4096 201 / 190; 10240 x 8192 at 1300 240 / 206.
  const float rope = epi == EPI_QKV_ROPE && S > 1 && s.tn * s.tm > 16 ? .25f * (s.tn * s.tm - 16) : 0.f;
  const float fixed = s.fixed + s.split * S + rope, stages = K / 64;
  float us = full * (fixed + s.stage[s.per_cu - 1] * stages);
  if (rest) {
    // blocks a CU of the last round, which starts as the one before it ends here and there
    const long per_cu = full && s.per_cu > 1 ? (rest <= 384 ? 1 : (rest - 128 + 255) / 256) : (rest + 255) / 256;
    us += fixed + s.stage[(per_cu < s.per_cu ? per_cu : s.per_cu) - 1] * stages;
  }
  return us;
}

// Shapes with an odd number of tiles a wave are not for the epilogues that take two at a time: gate and up (EPI_RELU_PAIR), and a head's
// (18432 x 2048 with rotation at 700 / 2000 rows: 224 x 256 blocks through LDS 79 / 216 us, what is chosen without them 66 / 194).
constexpr bool even_tiles(int epi) { return epi == EPI_RELU_PAIR || epi == EPI_QKV_ROPE; }
template <int N>
const Shape& best_shape(const Shape (&shapes)[N], int M, int n_tiles, int K, int S, int epi, float& us) {
  int best = 0;
  us = shape_us(shapes[0], M, n_tiles, K, S, epi);
  for (int i = 1; i < N; ++i) {
    if (even_tiles(epi) && shapes[i].tn % 2) continue;
    const float t = shape_us(shapes[i], M, n_tiles, K, S, epi);
    if (t < us) us = t, best = i;
  }
  return shapes[best];
}
const Shape& best_shape(int M, int n_tiles, int K, int S, int epi, float& us) {
  return S == 1 ? best_shape(kWholeShapes, M, n_tiles, K, S, epi, us) : best_shape(kSplitShapes, M, n_tiles, K, S, epi, us);
}

int shape_number(int M, int n_tiles, int K, int S, int epi) {
  float us;
  const Shape& s = best_shape(M, n_tiles, K, S, epi, us);
  return s.tn * 100 + s.tm * 10 + s.per_cu;
}

template <int EPI>
int prompt_shape(const PromptArgs& a, int S, hipStream_t st) {
  constexpr bool even = even_tiles(EPI);
  const int shape = shape_number(a.M, a.n_tiles, a.KS * 32, S, EPI);
  switch (shape) {
    case 881: return launch_prompt<8, 8, 2, false, EPI, 2>(a, st);
    case 781:
      if constexpr (!even) return launch_prompt<7, 8, 2, false, EPI, 2>(a, st);
      break;
    case 861: return launch_prompt<8, 6, 2, false, EPI, 2>(a, st);
    case 223: return launch_prompt<2, 2, 3, true, EPI>(a, st);
    case 422: return launch_prompt<4, 2, 3, true, EPI>(a, st);
    case 241: return launch_prompt<2, 4, 4, true, EPI>(a, st);
    case 431: return launch_prompt<4, 3, 4, true, EPI>(a, st);
    case 441: return launch_prompt<4, 4, 4, true, EPI, 3>(a, st);
    case 442: return launch_prompt<4, 4, 2, true, EPI>(a, st);
    case 451: return launch_prompt<4, 5, 4, true, EPI>(a, st);
    case 461: return launch_prompt<4, 6, 4, true, EPI>(a, st);
    case 481: return launch_prompt<4, 8, 3, true, EPI>(a, st);
  }
  sd_set_error("sd_prompt_linear: no kernel of shape %d", shape);
  return SD_ERR_UNSUPPORTED;
}

}  // namespace

// The block that a product of `n_tiles` of a matrix's `all_tiles` takes, tn * 100 + tm * 10 + blocks a CU, and 1000 where K
// is split (tests ask whether their sizes reach every block).
int sd_prompt_shape_(int M, int n_tiles, int all_tiles, int K, int epi) {
  int S, ksp, g;
  plan_split(all_tiles, K, S, ksp, g);
  return shape_number(M, n_tiles, K, S, epi) + (S > 1 ? 1000 : 0);
}

// What the QKV epilogue of this file takes: two tiles of a head at a time, four neighbours in a store.
bool sd_prompt_heads_fit_(const WideEpiArgs& e) {
  const uintptr_t at = reinterpret_cast<uintptr_t>(e.out) | reinterpret_cast<uintptr_t>(e.rope.kc) | reinterpret_cast<uintptr_t>(e.rope.vc);
  return e.rope.D % 32 == 0 && (e.ldo & 3) == 0 && (at & 7) == 0;
}

bool sd_prompt_linear_fits_(int M, int K, int64_t ldx) {
  // 256 rows are one pass of the kernels for fewer.  A block takes a long K's time however few blocks there are, and two or
  // three passes split it over the chip; us against those passes, weights from memory, 264 / 300 / 384 / 512 / 640 / 768
  // rows: 4096 x 14336 72 / 74 / 90 / 92 / 111 / 120 against 68 / 70 / 77 / 88 / 123 / 132; 3584 x 18944 89 / 92 / 112 / 113
  // / 133 / 143 against 78 / 81 / 88 / 100 / 136 / 147; 2048 x 8192 46 / 46 / 46 / 46 / 49 / 49 against 42 / 44 / 48 / 53 /
  // 74 / 80; 896 x 4864 25 to 26 against 31 / 34 / 39 / 41 / 59 / 60.  A K of up to 4096: 4096 x 4096 29 against 50 at 512
  // rows, 2048 x 2048 12.5 against 35.  (Gated matrices that make a short second round lose a little right behind 256
  // rows: 18944 x 3584 115 / 119 against 111 / 138 at 264 and 320.)
  return M > 256 && K % 64 == 0 && K >= 128 && (K <= 4096 || M > 512 || M > K / 24) && 512 * ldx < 0x7fffffff;
}

// At most 256 rows of a matrix whose K is split: its splits chained in a block instead of a workgroup each, with the epilogue
// inside.  us against the split products and the epilogue's launch, 64 / 128 / 256 rows: 2048 x 2048 12.4 / 12.4 / 12.5
// against 14.8 / 20.0 / 22.8, 1024 x 2048 12.4 / 12.5 / 12.6 against 12.5 / 15.8 / 22.2, 896 x 896 7.5 / 7.6 / 7.7 against
// 8.9 / 10.9 / 15.4; but 3584 x 3584 23.3 / 23.4 / 23.5 against 15.0 / 17.3 / 22.9.  Fewer rows, 17 / 24 / 33 / 48: 2048 x
// 2048 12.1 / 12.0 / 12.3 / 12.3 against 11.2 / 11.9 / 12.8 / 14.0, 7552 x 2048 13.9 / 14.0 / 14.2 / 14.3 against 12.3 / 12.7 /
// 13.3 / 14.1 (64: 14.6, 15.4); 1024 x 1024 7.6 / 7.6 / 7.8 / 7.8 against 7.4 / 8.0 / 8.2 / 8.8, 13312 x 1024 9.5 / 9.4 / 9.6 / 9.7
// against 11.3 / 11.5 / 12.4 / 13.6.
// A narrow matrix leaves that block alone on the chip while the splits' workgroups share its K, so it takes more rows: 64 x 2048
// 49 / 100 / 160 rows 11.7 / 11.8 / 11.9 against 9.3 / 10.5 / 11.4; 384 x 2048 49 / 64 12.0 / 12.0 against 10.9 / 11.7; 1024 x 2048 49 12.5 against
// 12.0; 64 x 1024 24 / 49 7.2 / 7.6 against 6.5 / 7.2, 384 x 1024 24 7.6 against 7.4.
bool sd_rows_chain_fits_(int M, int n_tiles, int K, int64_t ldx, int S) {
  return S > 1 && M >= (K <= 1024 ? 24 + 128 / n_tiles : 49 + 512 / n_tiles) && K <= 2048 && K % 64 == 0 && K >= 128 &&
         512 * ldx < 0x7fffffff;
}

// At most 256 rows: the products themselves (splits of K: the partial sums, for the caller's epilogue kernel).  Against
// the wide kernels, whose weights go through registers, with the epilogue's launch, weights from memory (us):
//   whole K, one round of blocks (gate and up of 8192 x 2048, 14336 x 4096, 18944 x 3584): 24 rows 20.7 -> 17.4, 44.3 ->
//   46.2, 56.1 -> 53.1, so not below 33; 128 rows 27.9 -> 20.2, 55.8 -> 55.5, 72.8 -> 60.2; 256 rows 42 -> 27, 76 -> 68,
//   127 -> 81 (the wide kernels leave CUs without a group, and spill at 256 rows);
//   more rounds (heads of 128256 x 2048, 152064 x 3584): 128 rows 110 -> 122, 228 -> 249; 256 rows 180 -> 154, 331 -> 317;
//   splits of 512 columns or more: 64 rows even, 96 rows 23.4 -> 20.1 (6144 x 4096) and never slower, 256 rows 62 -> 50
//   (3584 x 18944); of 256 columns: 96 rows 15.0 -> 15.3, 128 rows even, 256 rows 22.9 -> 20.2 (3072 x 2048); of 128
//   columns (2 stages) 5% slower up to 192 rows.
bool sd_rows_linear_fits_(int M, int n_tiles, int K, int64_t ldx, int S, int ks_per_split, int epi) {
  if (M > 256 || K % 64 != 0 || K < 128 || 512 * ldx >= 0x7fffffff) return false;
  if (S > 1) return M > 64 && (ks_per_split >= 16 || (M > 128 && ks_per_split >= 8));
  const int tn = few_tiles(n_tiles);
  return M > 32 && (epi == SD_EPI_SILU_MUL || epi == SD_EPI_F32) && (M > 192 || few_cost(n_tiles, tn) == tn);
}

int sd_rows_linear_(const void* W, const void* x, int64_t ldx, int M, int K, int n_tiles, int S, int ks_per_split, int epi,
                    const WideEpiArgs& epi_args, float* part, sd_stream_t stream) {
  SD_REQUIRE(!epi_args.w_scale && !epi_args.x_scale, SD_ERR_UNSUPPORTED, "sd_rows_linear: fp8 weights or activations");
  PromptArgs a{(const bf16_t*)W, (const bf16_t*)x, ldx, M, K / 32, n_tiles, ks_per_split, 0, 0, part, 0, epi_args};
  hipStream_t st = (hipStream_t)stream;
  if (S > 1) return launch_few<4, EPI_PARTIAL>(a, S, st);
  return epi == SD_EPI_F32 ? few_shape<SD_EPI_F32>(a, st) : few_shape<SD_EPI_SILU_MUL>(a, st);
}

// epi: an SD_EPI_* number or EPI_QKV_ROPE, with what that epilogue reads in `e` (no fp8 scales: the epilogues of this file know none).
int sd_prompt_linear_(const void* W, const void* x, int64_t ldx, int M, int K, int n_tiles, int epi,
                      const WideEpiArgs& epi_args, sd_stream_t stream) {
  SD_REQUIRE(!epi_args.w_scale && !epi_args.x_scale, SD_ERR_UNSUPPORTED, "sd_prompt_linear: fp8 weights or activations");
  SD_REQUIRE(epi != EPI_QKV_ROPE || sd_prompt_heads_fit_(epi_args), SD_ERR_UNSUPPORTED, "sd_prompt_linear: heads of %d, or unaligned outputs",
             epi_args.rope.D);
  int S, ksp, g;
  WideEpiArgs e = epi_args;
  e.M = M;
  e.NR = n_tiles * 16;
  e.S = 1;
  plan_split(n_tiles, K, S, ksp, g);
  PromptArgs a{(const bf16_t*)W, (const bf16_t*)x, ldx, M, K / 32, n_tiles, ksp, 0, 0, nullptr, 0, e};
  hipStream_t st = (hipStream_t)stream;
  switch (epi) {
    case SD_EPI_F32: return prompt_shape<SD_EPI_F32>(a, S, st);
    case SD_EPI_STORE: return prompt_shape<SD_EPI_STORE>(a, S, st);
    case SD_EPI_RESIDUAL: return prompt_shape<SD_EPI_RESIDUAL>(a, S, st);
    case SD_EPI_SILU_MUL: return prompt_shape<SD_EPI_SILU_MUL>(a, S, st);
    case SD_EPI_RELU: return prompt_shape<SD_EPI_RELU>(a, S, st);
    case SD_EPI_GELU_TANH: return prompt_shape<SD_EPI_GELU_TANH>(a, S, st);
    case EPI_QKV_ROPE: return prompt_shape<EPI_QKV_ROPE>(a, S, st);
  }
  sd_set_error("sd_prompt_linear: unknown epilogue %d", epi);
  return SD_ERR_INVALID;
}

// The stacked matrix of a gated layer (W [.. | gate [F] | up [F] | ..] of `n_tiles` tiles in all, gate's first tile
// `gate_tile`): act = bf16(relu(gate) * up) from one launch, the other columns f32 into y from one or two.  Against all columns
// in f32 and sd_relu_mul_rows (2048 rows of 2048 columns, 10240 or 14336 + 2 x 8192 outputs, us): 222 and 238 + 37 -> 108 + 90 and
// 108 + 109, the f32 stores of gate and up and their reads gone.  The splits of K are those of the whole matrix: so are the sums' bits.
//
// Two launches more are longer than that where they leave CUs without a block: the modelled times decide (sd_relu_mul_rows: 3 us
// and 4.5 TB/s), with a margin for what the model is off.  us of product and activation, all columns in f32 / this way: 10240 + 2 x
// 8192 outputs of 2048 columns 257 rows 54 / 51, 512 68 / 70, 1024 125 / 104, 2048 250 / 201; with 64 columns behind the pair 54 / 65, 66 / 87,
// 127 / 119, 247 / 214; 6144 + 2 x 4096 of 1024 columns 22 / 26, 29 / 32, 54 / 45, 100 / 81; 10240 + 2 x 1024 of 2048 30 / 33, 46 / 42, 77 / 71,
// 122 / 125.  Of 90 such measurements the rule takes no slower way than all columns in f32, and is 1.6 % behind the better one.
bool sd_prompt_relu_pair_fits_(int M, int n_tiles, int K, int64_t ldx, int gate_tile, int F) {
  if (!sd_prompt_linear_fits_(M, K, ldx)) return false;
  if ((int64_t)(F / 16 + 16) * K * 32 >= 0x7fffffff) return false;   // (an up tile's byte offset from its gate tile is an int)
  int S, ksp, g;
  plan_split(n_tiles, K, S, ksp, g);
  const int rest = n_tiles - gate_tile - F / 8;
  float whole, pair, us;
  best_shape(M, n_tiles, K, S, SD_EPI_F32, whole);
  best_shape(M, F / 8, K, S, EPI_RELU_PAIR, pair);
  for (const int tiles : {gate_tile, rest}) {
    if (tiles <= 0) continue;
    best_shape(M, tiles, K, S, SD_EPI_F32, us);
    pair += us;
  }
  return 1.08f * pair < whole + 3.f + (float)M * F * (10 / 4.5e6f);
}

int sd_prompt_relu_pair_(const void* W, const void* x, int64_t ldx, int M, int K, int n_tiles, int gate_tile, int F, float* y,
                         int64_t ldy, void* act, sd_stream_t stream) {
  int S, ksp, g;
  plan_split(n_tiles, K, S, ksp, g);
  hipStream_t st = (hipStream_t)stream;
  WideEpiArgs e{};
  e.M = M;
  e.S = 1;
  const auto at = [&](int tile) { return (const bf16_t*)W + (size_t)tile * (K / 32) * 512; };
  const int rest = gate_tile + F / 8;   // the tile behind the up range
  const int ranges[2][2] = {{0, gate_tile}, {rest, n_tiles - rest}};
  for (const auto& r : ranges) {
    if (r[1] <= 0) continue;
    e.N = e.NR = r[1] * 16;
    e.out = y + (size_t)r[0] * 16;
    e.ldo = ldy;
    const PromptArgs a{at(r[0]), (const bf16_t*)x, ldx, M, K / 32, r[1], ksp, 0, 0, nullptr, 0, e};
    const int rc = prompt_shape<SD_EPI_F32>(a, S, st);
    if (rc != SD_OK) return rc;
  }
  e.N = F;
  e.NR = 2 * F;
  e.out = act;
  e.ldo = F;
  const PromptArgs a{at(gate_tile), (const bf16_t*)x, ldx, M, K / 32, F / 8, ksp, 0, 0, nullptr, F / 16, e};
  return prompt_shape<EPI_RELU_PAIR>(a, S, st);
}

extern "C" int sd_linear_prompt(const void* W, const void* x, int64_t ldx, const void* bias, const void* residual,
                                void* out, int64_t ldo, int M, int N, int K, int epilogue, sd_stream_t stream) {
  SD_REQUIRE(W && x && out, SD_ERR_INVALID, "sd_linear_prompt: null pointer");
  SD_REQUIRE(epilogue >= SD_EPI_STORE && epilogue <= SD_EPI_GELU_TANH && (epilogue != SD_EPI_RESIDUAL || residual),
             SD_ERR_INVALID, "sd_linear_prompt: unknown epilogue %d, or a residual missing", epilogue);
  SD_REQUIRE(M >= 0 && N >= 1 && ldo >= N && ldx >= K && ldx % 8 == 0 && 512 * ldx < 0x7fffffff && sd_aligned16(W) &&
                 sd_aligned16(x), SD_ERR_INVALID, "sd_linear_prompt: rows must be 16-byte aligned (M=%d N=%d K=%d ldx=%lld)",
             M, N, K, (long long)ldx);
  SD_REQUIRE(K % 64 == 0 && K >= 128, SD_ERR_UNSUPPORTED, "sd_linear_prompt: K must be a multiple of 64, at least 128 (K=%d)", K);
  if (M == 0) return SD_OK;
  WideEpiArgs e{};
  e.N = N;
  e.bias = (const bf16_t*)bias;
  e.residual = (const bf16_t*)residual;
  e.out = out;
  e.ldo = ldo;
  return sd_prompt_linear_(W, x, ldx, M, K, tiles_of(N, epilogue), epilogue, e, stream);
}

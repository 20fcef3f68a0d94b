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
//     accumulator register there is;
//   4 x 4 (128 x 128), two stages: two blocks a CU, and room for a second set of sums; four stages where there is at most
//     one block a CU, whose loads nothing else covers;
//   2, 4 or 5 x 2, 4, 6 or 8 (all rows of a pass of 33..256), three stages: what is left is the weights' way from memory.
// The second set is for matrices whose K the narrower kernels split: a row's bits must not depend on how many
// rows share its pass, so the sums of a split are chained in one accumulator, and the splits' sums are added in
// index order from zero, as wide_epilogue_kernel adds them; in registers, without a second launch.
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
  WideEpiArgs epi;
};

typedef __attribute__((address_space(3))) void lds_void;
constexpr int EPI_PARTIAL = -1;  // the sums of one split of K, for wide_epilogue_kernel

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00027000);
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

// Barrier of the workgroup behind this wave's LDS reads and all but the newest LEFT of its direct loads
// (__syncthreads() would wait for every load in flight in some places and for none in others: it does not count
// direct loads as LDS writes).
template <int LEFT>
__device__ __forceinline__ void meet() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LEFT) : "memory");
}

template <int TN, int TM, int STAGES, bool SPLIT, int EPI>
__global__ __launch_bounds__(256, SPLIT ? 2 : 1) void prompt_gemm_kernel(PromptArgs a) {
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
  const int tile0 = nb * BN, row0 = mb * BM;
  const int k0 = split * a.ks_per_split;               // first k-step (EPI_PARTIAL)
  const int n_it = EPI == EPI_PARTIAL ? min(a.ks_per_split, a.KS - k0) >> 1 : a.KS >> 1;

  // this wave's direct loads: weights, piece p = (tile p >> 1, k-step p & 1) of the block's tiles
  const char* wbase = reinterpret_cast<const char*>(a.W) + (size_t)tile0 * a.KS * 1024;
  const int live_tiles = min(BN, a.n_tiles - tile0);
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
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)(s + p * 1024), 16, lane * 16 + (p >> 1) * w_step,
                                               (k0 + 2 * it + (p & 1)) * 1024, 0, 0);
    } else {
      const int p = wave + 4 * (i - kAPieces);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void*)(s + kABytes + p * 1024), 16, x_lane + p * x_step,
                                               k0 * 64 + it * 128, 0, 0);
    }
  };

  const int wn = wave & 1, wm = wave >> 1;
  const int xc = lane & 15, xq = lane >> 4;
  const int a_off = wn * TN * 2048 + lane * 16;
  const int b_row = kABytes + (wm * TM * 16 + xc) * 128;
  const int b_sw[2] = {((xq ^ (xc & 7)) << 4), (((xq + 4) ^ (xc & 7)) << 4)};
  bf16x8 fa[2][TN], fb[2][TM];
  constexpr int kReads = TN + TM, kMfma = TN * TM;
  constexpr int kOver = kMfma * 3 / 4 > kReads ? kMfma * 3 / 4 : kReads;
  static_assert(kReads <= kMfma && kPieces <= kMfma, "at most one LDS read and one direct load an MFMA");
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
        if constexpr (SPLIT) asm volatile("" : "+v"(acc[i][j]));
        else asm volatile("" : "+a"(acc[i][j]));
      }
    asm volatile("s_nop 15");
  };
  auto mfma = [&](int ks, int i, int j) __attribute__((always_inline)) {
    if constexpr (SPLIT)
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc[i][j]) : "v"(fa[ks][i]), "v"(fb[ks][j]));
    else
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(fa[ks][i]), "v"(fb[ks][j]));
  };
  // The MFMAs of one k-step with the next one's LDS reads (`from`) and the direct loads of a later stage between them
  auto phase = [&](auto k_step, const char* from, auto loads, char* to, int it) __attribute__((always_inline)) {
    constexpr int ks = decltype(k_step)::value;
    constexpr bool kLoads = decltype(loads)::value;
#pragma unroll
    for (int n = 0; n < kMfma; ++n) {
      mfma(ks, n / TM, n % TM);
      // (the reads in the first three quarters: the last one has its latency behind it at the phase's end)
      if (n < kOver && (n + 1) * kReads / kOver > n * kReads / kOver) read_piece(from, ks ^ 1, n * kReads / kOver);
      if (kLoads && (n + 1) * kPieces / kMfma > n * kPieces / kMfma) stage_piece(to, it, n * kPieces / kMfma);
    }
  };
  const int its_per_split = SPLIT ? a.ks_per_split >> 1 : 0;
  int next_split = its_per_split;
  // One stage of 64 columns: `cur` holds it (its first k-step's fragments are in registers already), `nxt` the
  // stage behind it; cur's place is then loaded with the stage STAGES further on.
  auto step = [&](char* cur, char* nxt, int it) __attribute__((always_inline)) {
    phase(std::integral_constant<int, 0>{}, cur, std::false_type{}, nullptr, 0);
    // every wave has read `cur` and its own part of `nxt` has landed
    meet<(STAGES - 2) * kPieces>();
    phase(std::integral_constant<int, 1>{}, nxt, std::true_type{}, cur, min(it + STAGES, n_it - 1));
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
    for (int i = 0; i < kPieces; ++i) stage_piece(s, min(it, n_it - 1), i);
  };
  fill(s0, 0);
  fill(s1, 1);
  if constexpr (STAGES >= 3) fill(s2, 2);
  if constexpr (STAGES == 4) fill(s3, 3);
  meet<(STAGES - 1) * kPieces>();
#pragma unroll
  for (int i = 0; i < kReads; ++i) read_piece(s0, 0, i);
  settle();
  int it = 0;
  if constexpr (STAGES == 4) {
    for (; it + 3 < n_it; it += 4) {
      step(s0, s1, it);
      step(s1, s2, it + 1);
      step(s2, s3, it + 2);
      step(s3, s0, it + 3);
    }
    if (it < n_it) step(s0, s1, it);
    if (it + 1 < n_it) step(s1, s2, it + 1);
    if (it + 2 < n_it) step(s2, s3, it + 2);
  } else if constexpr (STAGES == 3) {
    for (; it + 2 < n_it; it += 3) {
      step(s0, s1, it);
      step(s1, s2, it + 1);
      step(s2, s0, it + 2);
    }
    if (it < n_it) step(s0, s1, it);
    if (it + 1 < n_it) step(s1, s2, it + 1);
  } else {
    for (; it + 1 < n_it; it += 2) {
      step(s0, s1, it);
      step(s1, s0, it + 1);
    }
    if (it < n_it) step(s0, s1, it);
  }
  meet<0>();  // no direct load outlives the workgroup's use of LDS
  settle();

  if (SPLIT) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) acc[i][j] = tot[i][j] + acc[i][j];
  }
  // acc[i][j][reg] = (tile row 4 * xq + reg of tile i, token 16 j + xc).  Through LDS, 16 token rows at a time
  // and each wave for itself, so that the lanes of a store hold neighbouring outputs of a row (and the epilogue
  // is there once per token tile, not once per pair of tiles).
  constexpr bool PAIRED = EPI == SD_EPI_SILU_MUL || EPI == EPI_QKV_ROPE;
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

template <int TN, int TM, int STAGES, bool SPLIT, int EPI>
int launch_prompt(PromptArgs a, hipStream_t st) {
  a.n_blocks = (a.n_tiles + 2 * TN - 1) / (2 * TN);
  a.m_blocks = (a.M + 32 * TM - 1) / (32 * TM);
  hipLaunchKernelGGL((prompt_gemm_kernel<TN, TM, STAGES, SPLIT, EPI>), dim3(a.n_blocks * a.m_blocks), dim3(256), 0, st, a);
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
  if (a.M <= 64) hipLaunchKernelGGL((prompt_gemm_kernel<TN, 2, 3, false, EPI>), grid, dim3(256), 0, st, a);
  else if (a.M <= 128) hipLaunchKernelGGL((prompt_gemm_kernel<TN, 4, 3, false, EPI>), grid, dim3(256), 0, st, a);
  else if (a.M <= 192) hipLaunchKernelGGL((prompt_gemm_kernel<TN, 6, 3, false, EPI>), grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((prompt_gemm_kernel<TN, 8, 3, false, EPI>), grid, dim3(256), 0, st, a);
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

// The block of a prompt pass, us of 256 x 256 (whole K only), 128 x 128 with four stages, with two:
//   one block a CU at most (`small` <= 256): 6144 x 4096 at 512 rows 31.9 with four stages, 42.1 with two; 4096 x 14336 at
//   1024 rows 103 against 145; above, two blocks a CU cover each other's loads: 2048 rows 206 against 192;
//   whole K: 256 x 256 from 200 blocks on (14336 x 4096 gated: 272 rows 94, 101, 95; 1024 rows 195, 243, 231; 4096 rows 705,
//   1010, 866; 18944 x 3584 gated, 1024 rows 262, 337, 289; 32000 x 2048, 512 rows 59, 83, 66).  Between the line at 128
//   blocks and there both sides win: 18432 x 2048 at 512 rows (144 blocks) 52, 58, 54, at 272 rows 51, 37, 32; gated 8192 x
//   2048 at 512 rows (128 blocks, 50, 41, 36); and where the second round is short (18944 x 3584, 272 rows, 296 blocks): 161,
//   109, 107.
template <int EPI>
int prompt_shape(const PromptArgs& a, int S, hipStream_t st) {
  const long big = (long)((a.n_tiles + 15) / 16) * ((a.M + 255) / 256);
  const long small = (long)((a.n_tiles + 7) / 8) * ((a.M + 127) / 128);
  if (S == 1 && big >= 128) return launch_prompt<8, 8, 2, false, EPI>(a, st);
  if (small <= 256) return launch_prompt<4, 4, 4, true, EPI>(a, st);
  return launch_prompt<4, 4, 2, true, EPI>(a, st);
}

}  // namespace

bool sd_prompt_linear_fits_(int M, int n_tiles, int K, int64_t ldx) {
  // 256 rows are one pass of the kernels for fewer.  A block takes a long K's time however few blocks there are, and two or
  // three passes split it over the chip; us against those passes, weights from memory, 300 / 512 / 640 / 768 / 1024 rows:
  // 4096 x 14336 107 / 135 / 136 / 136 / 138 against 69 / 87 / 122 / 133 / 173; 3584 x 18944 131 / 164 / 164 / 165 / 169
  // against 78 / 98 / 135 / 146 / 193; 2048 x 8192 65 / 74 / 75 / 74 / 75 against 45 / 55 / 75 / 81 / 109.  A K of up to
  // 4096: 4096 x 4096 39 / 45 / 46 / 45 / 47 against 52 / 59 / 69 / 75 / 100, 2048 x 2048 24 / 24 / 26 / 27 / 28 against 37
  // / 46 / 61 / 68 / 90.  (Gated matrices whose blocks of 256 rows make a short second round lose too: 18944 x 3584 171 /
  // 181 against 134 / 165 up to 512 rows, 8192 x 2048 54 / 57 against 40 / 50, 14336 x 4096 193 / 196 against 164 / 178 at
  // 640 and 768.)
  const long blocks = (long)((n_tiles + 7) / 8) * ((M + 127) / 128);
  return M > 256 && K % 64 == 0 && K >= 128 && (K <= 4096 || (M > 768 && blocks > 64)) && 512 * ldx < 0x7fffffff;
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
  PromptArgs a{(const bf16_t*)W, (const bf16_t*)x, ldx, M, K / 32, n_tiles, ks_per_split, 0, 0, part, epi_args};
  hipStream_t st = (hipStream_t)stream;
  if (S > 1) return launch_few<4, EPI_PARTIAL>(a, S, st);
  return epi == SD_EPI_F32 ? few_shape<SD_EPI_F32>(a, st) : few_shape<SD_EPI_SILU_MUL>(a, st);
}

// epi: an SD_EPI_* number or EPI_QKV_ROPE, with what that epilogue reads in `e`.
int sd_prompt_linear_(const void* W, const void* x, int64_t ldx, int M, int K, int n_tiles, int epi,
                      const WideEpiArgs& epi_args, sd_stream_t stream) {
  int S, ksp, g;
  WideEpiArgs e = epi_args;
  e.M = M;
  e.NR = n_tiles * 16;
  e.S = 1;
  plan_split(n_tiles, K, S, ksp, g);
  PromptArgs a{(const bf16_t*)W, (const bf16_t*)x, ldx, M, K / 32, n_tiles, ksp, 0, 0, nullptr, e};
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

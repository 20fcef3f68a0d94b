// Row products of f32 models: y [M, N] = x [M, K] W^T (+ bias), or of relu(x) * x2, for more than 16 rows, on the f32 matrix
// instruction.
//
// v_mfma_f32_16x16x4_f32 is four fused multiply-adds in ascending k for every element (as v_mfma_f32_32x32x2_f32 is two; tests
// compare the bits), so a sum has the bits of the kernels for fewer rows whatever the block.  The op is bound by the matrix
// pipe (64 FLOP a clock and SIMD), so all that matters is that the pipe never waits and that every CU has its share: operands come by direct
// loads (16 bytes a lane, no registers), 32 columns a stage, three or four stages ahead of their use, one barrier a stage
// with the fragments read two pieces of 4 k before their products; blocks of 64 x 64 or 128 x 64, whichever costs less rounds
// over the chip.
//
// A stage of a row is 128 bytes, 8 pieces of 4 k; piece c of row r lies at slot c ^ (r & 7), which spreads the fragment
// reads over the banks; the source address carries the permutation.  Lane (r, q) of a product multiplies k = 4 c + q of row r
// of either operand: one value of piece c.  Rows past the matrix and k past K are out of the buffers' bounds and arrive as
// zeros.
//
// us, both operands through registers into two LDS buffers / this way with four waves a block / with eight: 777 rows of 13312 x 1024 251 / 182 /
// 180, 32000 x 1024 528 / 412 / 406 (125 TFLOP/s), 1024 x 4096 gated 122 / 89 / 81, 1024 x 1024 33 / 21.7 / 20.3; 300 rows of 13312 x
// 1024 166 / 86 / 83, 4096 x 4096 - / 133 / 128; 2048 rows of 4096 x 4096 615 / 489 / 485 (142 TFLOP/s), gated 1024 x 4096 - / 157 / 142.
#include "sd_common.h"

namespace {

struct F32Args {
  const float *x, *x2, *w, *bias;
  float* y;
  bf16_t* yb;
  int64_t ldx, ldy, bx, bw, by;
  int M, N, K, n_blocks, m_blocks;
};

constexpr int kRow = 128;                    // bytes of a row and stage

constexpr int stage_bytes(int nt, int mt, bool gated) { return (64 * nt + 64 * mt * (gated ? 2 : 1)) * kRow; }
// as many as leave room for two blocks a CU (128 x 64 gated: one)
constexpr int stages_of(int nt, int mt, bool gated) { return stage_bytes(nt, mt, gated) * 8 <= 160 * 1024 ? 4 : 3; }

// Eight waves, a quarter of the rows and half the columns each: two on a SIMD where a block is alone on its CU, so that one multiplies
// while the other reads its fragments or waits for the barrier (four waves before: see the figures above).
constexpr int kWaves = 8;
template <int NT, int MT, bool GATED>
__global__ __launch_bounds__(64 * kWaves, NT > 1 && GATED ? 1 : 2) void rows_f32_kernel(F32Args a) {
  constexpr int BN = 64 * NT, BM = 64 * MT, S = stages_of(NT, MT, GATED), kStage = stage_bytes(NT, MT, GATED);
  constexpr int kWLoads = BN / (8 * kWaves), kXLoads = BM / (8 * kWaves), kLoads = kWLoads + kXLoads * (GATED ? 2 : 1);   // of a wave and stage
  __shared__ __attribute__((aligned(1024))) char s0[kStage];
  __shared__ __attribute__((aligned(1024))) char s1[kStage];
  __shared__ __attribute__((aligned(1024))) char s2[kStage];
  __shared__ __attribute__((aligned(1024))) char s3[S == 4 ? kStage : 16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wn = wave & 1, wm = wave >> 1;
  const int r = lane & 15, kq = lane >> 4;
  const int work = xcd_order(blockIdx.x, a.n_blocks * a.m_blocks);
  const int grp = work / (a.n_blocks * kRowGroup), in_grp = work - grp * a.n_blocks * kRowGroup;
  const int grp_rows = min(kRowGroup, a.m_blocks - grp * kRowGroup);
  const int nb = in_grp / grp_rows, mb = grp * kRowGroup + in_grp - nb * grp_rows;
  const int n0 = nb * BN, m0 = mb * BM;
  const int live_n = min(BN, a.N - n0), live_m = min(BM, a.M - m0);
  const size_t xo = (size_t)blockIdx.z * a.bx + (size_t)m0 * a.ldx;
  const size_t x_bytes = ((size_t)(live_m - 1) * a.ldx + a.K) * 4;
  const auto wr = buffer_of(a.w + (size_t)blockIdx.z * a.bw + (size_t)n0 * a.K, (size_t)live_n * a.K * 4);
  const auto xr = buffer_of(a.x + xo, x_bytes);
  const auto gr = buffer_of(GATED ? a.x2 + xo : a.x, GATED ? x_bytes : 0);
  // this wave's direct loads: eight rows each
  const unsigned piece = ((lane & 7) ^ (lane >> 3)) << 4;
  unsigned w_at[kWLoads], x_at[kXLoads];
#pragma unroll
  for (int i = 0; i < kWLoads; ++i) {
    const int n = (wave * kWLoads + i) * 8 + (lane >> 3);
    w_at[i] = n < live_n ? (unsigned)n * (unsigned)a.K * 4 + piece : kOutside;
  }
#pragma unroll
  for (int i = 0; i < kXLoads; ++i) {
    const int m = (wave * kXLoads + i) * 8 + (lane >> 3);
    x_at[i] = m < live_m ? (unsigned)m * (unsigned)a.ldx * 4 + piece : kOutside;
  }
  const int n_it = (a.K + 31) / 32;
  auto put = [&](__amdgpu_buffer_rsrc_t b, char* to, unsigned at) __attribute__((always_inline)) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(b, (lds_void*)to, 16, at, 0, 0, 0);
  };
  // loads FIRST .. LAST - 1 of stage `it`
  auto load = [&](char* s, int it, int first, int last) __attribute__((always_inline)) {
    const unsigned k = it * kRow;
    const bool in = k + piece < (unsigned)a.K * 4;   // (stages past the last: none)
#pragma unroll
    for (int i = first; i < last; ++i) {
      const int j = i < kWLoads ? i : (i - kWLoads) % kXLoads;
      const unsigned row = i < kWLoads ? w_at[i] : x_at[j];
      const int at = i < kWLoads ? wave * kWLoads + i : (BN + (i < kWLoads + kXLoads ? 0 : BM)) / 8 + wave * kXLoads + j;
      put(i < kWLoads ? wr : i < kWLoads + kXLoads ? xr : gr, s + at * 1024, in && row != kOutside ? row + k : kOutside);
    }
  };
  constexpr int TN = 2 * NT, TM = 8 * MT / kWaves;   // tiles of 16 x 16 of a wave
  f32x4 acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int w_row = (wn * TN * 16 + r) * kRow + kq * 4, x_row = BN * kRow + (wm * TM * 16 + r) * kRow + kq * 4;
  float fa[4][TN], fb[4][TM], fg[4][GATED ? TM : 1];
  auto read = [&](const char* s, int p) __attribute__((always_inline)) {
    const int at = (p ^ (r & 7)) << 4;
#pragma unroll
    for (int i = 0; i < TN; ++i) fa[p & 3][i] = *reinterpret_cast<const float*>(s + w_row + i * 16 * kRow + at);
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      fb[p & 3][j] = *reinterpret_cast<const float*>(s + x_row + j * 16 * kRow + at);
      if (GATED) fg[p & 3][GATED ? j : 0] = *reinterpret_cast<const float*>(s + BM * kRow + x_row + j * 16 * kRow + at);
    }
  };
  auto gate = [&](int p) __attribute__((always_inline)) {
    if (GATED) {
#pragma unroll
      for (int j = 0; j < TM; ++j) fb[p & 3][j] = fmaxf(fb[p & 3][j], 0.f) * fg[p & 3][GATED ? j : 0];
    }
  };
  // `cur` holds the stage, its first piece is in registers; `nxt` the one behind it.  Left to itself the compiler puts a
  // piece's reads right before their use (4096 x 4096 at 2048 rows 571 us, 547 in this order): the scheduling barriers keep
  // them a piece ahead.
  // A stage's loads are spread over the eight pieces behind the barrier that frees its place: two of them in the step that
  // ends with `cur`, six in the next one, whose `prev` that place is.
  auto share = [](int p) { return kLoads * p / 8; };
  auto step = [&](char* cur, const char* nxt, char* prev, int it) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < 8; ++p) {
      if (p < 6) {
        read(cur, p + 2);
      } else {
        // every wave has read `cur`, and its own part of `nxt` has landed
        if (p == 6) meet<(S - 2) * kLoads>();
        read(nxt, p - 6);
      }
      gate(p + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[p & 3][i], fb[p & 3][j], acc[i][j], 0, 0, 0);
          if (i == 0 && j == 0) {
            if (p < 6) load(prev, it - 1 + S, share(p + 2), share(p + 3));
            else load(cur, it + S, share(p - 6), share(p - 5));
          }
        }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  load(s0, 0, 0, kLoads);
  load(s1, 1, 0, kLoads);
  load(s2, 2, 0, S == 4 ? kLoads : share(2));
  if constexpr (S == 4) load(s3, 3, 0, share(2));
  meet<(S - 2) * kLoads + kLoads * 2 / 8>();
  read(s0, 0);
  read(s0, 1);
  gate(0);
  int it = 0;
  if constexpr (S == 4) {
    for (; it + 3 < n_it; it += 4) {
      step(s0, s1, s3, it);
      step(s1, s2, s0, it + 1);
      step(s2, s3, s1, it + 2);
      step(s3, s0, s2, it + 3);
    }
    if (it < n_it) step(s0, s1, s3, it);
    if (it + 1 < n_it) step(s1, s2, s0, it + 1);
    if (it + 2 < n_it) step(s2, s3, s1, it + 2);
  } else {
    for (; it + 2 < n_it; it += 3) {
      step(s0, s1, s2, it);
      step(s1, s2, s0, it + 1);
      step(s2, s0, s1, it + 2);
    }
    if (it < n_it) step(s0, s1, s2, it);
    if (it + 1 < n_it) step(s1, s2, s0, it + 1);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no direct load outlives the workgroup's use of LDS
  // acc[i][j][e]: column n0 + (wn TN + i) 16 + 4 kq + e of row m0 + (wm TM + j) 16 + r
  float* Y = a.y + (size_t)blockIdx.z * a.by;
  bf16_t* Yb = a.yb ? a.yb + (size_t)blockIdx.z * a.by : nullptr;
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    const int m = m0 + (wm * TM + j) * 16 + r;
    if (m >= a.M) continue;
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      const int n = n0 + (wn * TN + i) * 16 + 4 * kq;
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = acc[i][j][e] + (a.bias && n + e < a.N ? a.bias[n + e] : 0.f);
      const size_t at = (size_t)m * a.ldy + n;
      if (n + 3 < a.N && (a.ldy & 3) == 0) {
        *reinterpret_cast<f32x4*>(Y + at) = o;
        if (Yb) *reinterpret_cast<bf16x4*>(Yb + at) = bf16x4{(bf16_t)o[0], (bf16_t)o[1], (bf16_t)o[2], (bf16_t)o[3]};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < a.N) {
            Y[at + e] = o[e];
            if (Yb) Yb[at + e] = (bf16_t)o[e];
          }
      }
    }
  }
}

template <int NT, int MT>
int launch(F32Args a, int batch, hipStream_t st) {
  a.n_blocks = (a.N + 64 * NT - 1) / (64 * NT);
  a.m_blocks = (a.M + 64 * MT - 1) / (64 * MT);
  const dim3 grid(a.n_blocks * a.m_blocks, 1, batch);
  if (a.x2) rows_f32_kernel<NT, MT, true><<<grid, 64 * kWaves, 0, st>>>(a);
  else rows_f32_kernel<NT, MT, false><<<grid, 64 * kWaves, 0, st>>>(a);
  SD_CHECK_LAUNCH("sd_matmul_rows");
  return SD_OK;
}

}  // namespace

// Whether blocks of 128 x 64 are quicker than 64 x 64 ones.  Blocks go over the CUs in rounds; us a stage of 32 columns and round, of a first
// round alone / of further ones (medians of 308 sizes, 64..32000 x 512..4096, 33..2048 rows, with eight waves a block): 64 x 64 .60 / .53, gated .71 / .62;
// 128 x 64 1.08 / 1.00, gated (one a CU) 1.18 / 1.17.  The rule's choice is .005 % slower than the better of the two on average, 0.7 % at most
// (6144 x 2048 at 130 rows).  us of 64 x 64 / 128 x 64: 13312 x 1024 at 2048 rows 422 / 407, 1024 216 / 223; 32000 x 1024 at 777 421 / 406, 33 38.8 / 41.9;
// 4096 x 1024 at 512 37.0 / 37.7; 4096 x 4096 at 300 127.8 / 127.7, gated 153 / 140; 1024 x 4096 gated at 1500 150 / 139, 777 81 / 136.
// 128 x 128, 192 x 128 and 256 x 128 (of four waves) are slower than the better of the two everywhere (13312 x 1024 at 2048 rows 481, 503, 528).
bool sd_rows_f32_wide_(int M, int N, int batch, bool gated) {
  const long n1 = ((long)((N + 63) / 64) * ((M + 63) / 64) * batch + 255) / 256;
  const long n2 = ((long)((N + 127) / 128) * ((M + 63) / 64) * batch + 255) / 256;
  const float us1 = n1 == 1 ? (gated ? .71f : .60f) : (gated ? .62f : .53f) * n1;
  const float us2 = n2 == 1 ? (gated ? 1.18f : 1.08f) : (gated ? 1.17f : 1.00f) * n2;
  return us2 < us1;
}

// 16-byte aligned rows (K, ldx and the batch strides multiples of four)
int sd_rows_f32_(const float* x, const float* x2, int64_t ldx, const float* w, const float* bias, float* y, int64_t ldy, int M,
                 int N, int K, int batch, int64_t bx, int64_t bw, int64_t by, bf16_t* yb, hipStream_t st) {
  const F32Args a{x, x2, w, bias, y, yb, ldx, ldy, bx, bw, by, M, N, K, 0, 0};
  return sd_rows_f32_wide_(M, N, batch, x2) ? launch<2, 1>(a, batch, st) : launch<1, 1>(a, batch, st);
}

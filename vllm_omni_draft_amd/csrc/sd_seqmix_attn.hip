// Softmax attention of layer-list models for the many rows of a prompt, over bf16 caches of plain rows (page, kv head,
// token): grouped heads, and latent rows whose first channels are the values.
//
// The queries and the weights of these models are f32 and stay so: each enters the bf16 matrix instruction as the sum
// of three bf16 parts (8 + 8 + 8 bits: all of an f32's), keys and values are the cache's bf16 values, so products are
// exact and sums f32, as on the vector pipe, at a third of the matrix rate.  The kernel before took one workgroup a row
// and read every key and value from L2 for it on the vector pipe (18 TFLOP/s of f32 work).
//
// A workgroup takes one kv head and 64 query rows (64 / (H/G) tokens x the heads of the group) of one portion, a wave
// 16 of them; 64 keys (four pages) a stage pass through LDS by direct loads, two stages, one barrier a stage.  A page of
// a head is contiguous, so a wave brings one page; 16-byte piece c of row r of a page lies at c ^ (r & 7) within its
// 128 bytes, which spreads the fragment reads over the banks.  S^T = K Q^T has a query's scores in one accumulator
// column, as they are the right operand of O^T = V^T P^T; V^T comes out of the row-major tile by the transposing LDS
// read (a group of 16 lanes reads 4 keys x 16 channels, a lane receives 4 keys of one channel).
// Bound by the matrix pipe and the exponentials between its parts (one wave a SIMD for latent rows, whose queries and
// sums fill the registers): 1024 rows of 16 latent heads (576 / 512 channels) 972 -> 135 us, 1024 rows of 16 heads over 4
// of 128 channels 344 -> 40 us, 2048 rows of 16 heads over 4 with a window of 1024 and pooled blocks 816 -> 87 us.
// A weight of 0 does not clear a value that is no number: in the stages that not all rows of a workgroup see whole, such
// values become 0 as they arrive (clear_odd: 1-5 %, 10 % of 65 pooled rows behind 4000 tokens), and the rows that see them
// get them added (add_odd).  Scores that are no numbers: see redo_query.
#include <math.h>
#include <type_traits>

#include "sd_common.h"

namespace {

struct RowsAttnArgs {
  const float* q;
  int64_t ldq;
  const bf16_t* kc;
  const bf16_t* vc;
  const int32_t* block_tables;
  const int32_t* entries;
  float* out;
  bf16_t* out_b;
  int64_t ldo;
  float scale;
  int max_blocks, n_entries, H, G, window, keep_first, above;   // above: portions of more rows than this
  // pooled keys and values of whole blocks of `pool` tokens behind the window (f32), `pslots` a page
  const float *pk, *pv, *head_bias;
  int pool, pslots;
};

typedef __attribute__((address_space(1))) const void global_void;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
template <int N>
using Number = std::integral_constant<int, N>;
constexpr int kPage = 16, kKeys = 64, kRowsPerBlock = 64, kPooled = 32;

// Two f32 values as three pairs of bf16 whose sums they are: 8 bits of the significand each, cut off (the differences
// are exact), the first value in the low halves.  INF: the values may be infinite, and are their first part then.
template <bool INF = false>
__device__ __forceinline__ void three_parts(float x, float y, unsigned& a, unsigned& b, unsigned& c) {
  auto upper = [](float v) { return __uint_as_float(__float_as_uint(v) & 0xffff0000u); };
  auto pack = [](float u, float v) { return __builtin_amdgcn_perm(__float_as_uint(v), __float_as_uint(u), 0x07060302u); };
  auto rest = [&](float v) { return INF && fabsf(v) == INFINITY ? 0.f : v - upper(v); };
  const float xr = rest(x), yr = rest(y);
  a = pack(x, y);
  b = pack(xr, yr);
  c = pack(xr - upper(xr), yr - upper(yr));
}

// e^x for x <= 0 (-inf: 0), to about one unit in the last place: the product with log2 e in two parts, no branch.
// (The limit lets a NaN through, as fmaxf would not: one instruction either way.)
__device__ __forceinline__ float exp_neg(float x) {
  x = __builtin_elementwise_maximum(x, -200.f);   // (e^-200 is 0 in f32)
  const float hi = x * 1.44269502f;
  const float lo = fmaf(x, 1.92596300e-8f, fmaf(x, 1.44269502f, -hi));
  const float y = __builtin_amdgcn_exp2f(hi);
  return fmaf(y, lo * 0.693147181f, y);
}

// 1 / (1 + e^-x) of a finite x, to about two units in the last place (below e^-87: 0 or next to it)
__device__ __forceinline__ float sigmoid_of(float x) {
  x = -fmaxf(x, -87.f);
  const float hi = x * 1.44269502f;
  const float lo = fmaf(x, 1.92596300e-8f, fmaf(x, 1.44269502f, -hi));
  const float y = __builtin_amdgcn_exp2f(hi);
  const float d = 1.f + fmaf(y, lo * 0.693147181f, y), r = __builtin_amdgcn_rcpf(d);
  return fmaf(fmaf(-d, r, 1.f), r, r);
}

// KS: key channels / 32 (even); VT: value channels / 16 (a multiple of 4); LATENT: values are the keys' first channels;
// POOLED: weights are sigmoids of the scores plus a bias, and the blocks behind the window take part as their means.
// The means are f32: stages of 32 of them take the f32 matrix instruction, whose fragments of 4 channels are the 8
// channels of a lane in turn; the scores' accumulators are its right operand as they are.
template <int KS, int VT, bool LATENT, bool POOLED>
__global__ __launch_bounds__(256, KS > 4 ? 1 : 2) void rows_attn_kernel(RowsAttnArgs g) {
  constexpr int DK = 32 * KS, DV = 16 * VT;
  constexpr int kKeyPage = kPage * DK * 2, kValPage = LATENT ? 0 : kPage * DV * 2;   // bytes of a page of one head
  constexpr int kStage = 4 * (kKeyPage + kValPage);
  __shared__ __attribute__((aligned(1024))) char s0[kStage];
  __shared__ __attribute__((aligned(1024))) char s1[kStage];
  __shared__ unsigned odd[2][4];   // of a stage and a wave's part of it: the rows that held values that are no numbers
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kvh = blockIdx.y, qh = g.H / g.G, per = kRowsPerBlock / qh;
  // the portion and the first token of this group of tokens; the last ones, which see most, first
  int e = 0, first = gridDim.x - 1 - blockIdx.x;
  for (; e < g.n_entries; ++e) {
    const int rows = g.entries[4 * e + 2], n = rows > g.above ? (rows + per - 1) / per : 0;
    if (first < n) break;
    first -= n;
  }
  if (e == g.n_entries) return;
  first *= per;
  const int slot = g.entries[4 * e], row0 = g.entries[4 * e + 1], pos0 = g.entries[4 * e + 3] + first;
  const int n_tok = min(per, g.entries[4 * e + 2] - first), m_rows = n_tok * qh;
  const int32_t* tbl = g.block_tables + (size_t)slot * g.max_blocks;
  const int last = pos0 + n_tok - 1;                         // the workgroup's last position
  int base0 = max(pos0 - g.window + 1, 0) & ~(kPage - 1);    // the window's first page
  // what is seen before it, in stages of their own: kept tokens, or pooled blocks
  auto blocks_of = [&](int pos) { return max(pos - g.window + 1, 0) / g.pool; };
  const int n_kept = POOLED ? blocks_of(last) : min(g.keep_first, base0);
  constexpr int kKept0 = POOLED ? kPooled : kKeys;
  const int kept_stages = (n_kept + kKept0 - 1) / kKept0, stages = kept_stages + (last - base0) / kKeys + 1;
  auto stage_base = [&](int s) { return s < kept_stages ? s * kKeys : base0 + (s - kept_stages) * kKeys; };

  const int m = min(16 * wave + col, m_rows - 1), t = m / qh, h = kvh * qh + m - t * qh;   // this lane's query
  const bool mine = 16 * wave + col < m_rows;
  const int p = pos0 + t;
  const bool works = 16 * wave < m_rows;
  const int wave_last = works ? pos0 + (min(16 * wave + 16, m_rows) - 1) / qh : -1;
  // The query times the scale.  Its parts are kept where the registers allow; wide rows (kKept false) keep the f32
  // values and take them apart at every use, which the vector pipe does beside the matrix pipe.
  constexpr bool kKept = KS <= 4;
  f32x4 qf[kKept ? 1 : KS][2];
  bf16x8 qp[kKept ? KS : 1][3];
  auto parts = [&](const f32x4 (&x)[2], bf16x8 (&y)[3], auto inf) __attribute__((always_inline)) {
    u32x4 a, b, c;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      unsigned pa, pb, pc;
      three_parts<decltype(inf)::value>(x[i >> 1][2 * (i & 1)], x[i >> 1][2 * (i & 1) + 1], pa, pb, pc);
      a[i] = pa;
      b[i] = pb;
      c[i] = pc;
    }
    y[0] = __builtin_bit_cast(bf16x8, a);
    y[1] = __builtin_bit_cast(bf16x8, b);
    y[2] = __builtin_bit_cast(bf16x8, c);
  };
  const float* qr = g.q + (size_t)(row0 + first + t) * g.ldq + (size_t)h * DK;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const f32x4 x[2] = {*reinterpret_cast<const f32x4*>(qr + 32 * s + 8 * quad) * g.scale,
                        *reinterpret_cast<const f32x4*>(qr + 32 * s + 8 * quad + 4) * g.scale};
    if constexpr (kKept) parts(x, qp[s], std::true_type{});
    else {
      qf[s][0] = x[0];
      qf[s][1] = x[1];
    }
  }
  // wave w brings page w of the stage (behind the stage's last key: that key's page), its number asked for a stage ahead
  auto stage_last = [&](int s) { return s < kept_stages ? n_kept - 1 : last; };
  auto page_of = [&](int st) {
    st = max(min(st, stages - 1), POOLED ? kept_stages : 0);
    return tbl[min(stage_base(st) + wave * kPage, stage_last(st)) / kPage];
  };
  int page = page_of(0);
  auto load = [&](char* s, int st) __attribute__((always_inline)) {
    if (POOLED && st < kept_stages) {   // wave w: means 8w on of the stage (behind the last one: that one)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 2 * i + (lane >> 5), idx = min(st * kPooled + wave * 8 + r, n_kept - 1);
        const int lp = (idx * g.pool + g.pool - 1) / kPage;   // the page whose slots hold block idx
        const size_t at = (((size_t)tbl[lp] * g.G + kvh) * g.pslots + idx - lp * kPage / g.pool) * 512 + (((lane & 31) ^ r) << 4);
        static_assert(!POOLED || (DK == 128 && DV == 128), "rows of 512 bytes");
        __builtin_amdgcn_global_load_lds((global_void*)((const char*)g.pk + at), (lds_void*)(s + wave * 4096 + i * 1024), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((global_void*)((const char*)g.pv + at), (lds_void*)(s + kPooled * 512 + wave * 4096 + i * 1024),
                                         16, 0, 0);
      }
      return;
    }
    const int blk = __builtin_amdgcn_readfirstlane(page);
    page = page_of(st + 1);
    const size_t row = ((size_t)blk * g.G + kvh) * kPage;
    const auto kr = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(g.kc + row * DK), 0, kKeyPage, 0x00027000);
#pragma unroll
    for (int i = 0; i < kKeyPage / 1024; ++i) {
      const int r = (i * 8 + (lane >> 3)) / (DK / 64);       // the row of the page that this lane's 128 bytes belong to
      __builtin_amdgcn_raw_ptr_buffer_load_lds(kr, (lds_void*)(s + wave * kKeyPage + i * 1024), 16,
                                               i * 1024 + (lane >> 3) * 128 + (((lane & 7) ^ (r & 7)) << 4), 0, 0, 0);
    }
    if constexpr (!LATENT) {
      const auto vr = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(g.vc + row * DV), 0, kValPage, 0x00027000);
#pragma unroll
      for (int i = 0; i < kValPage / 1024; ++i) {
        const int r = (i * 8 + (lane >> 3)) / (DV / 64);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(vr, (lds_void*)(s + 4 * kKeyPage + wave * kValPage + i * 1024), 16,
                                                 i * 1024 + (lane >> 3) * 128 + (((lane & 7) ^ (r & 7)) << 4), 0, 0, 0);
      }
    }
  };
  f32x4 o[VT];
#pragma unroll
  for (int v = 0; v < VT; ++v) o[v] = f32x4{0.f, 0.f, 0.f, 0.f};
  // (a query's sum is spread over its four lanes; the largest score, pooled: the largest absolute value, is NaN once one
  // was no number)
  float m_run = POOLED ? 0.f : -INFINITY, l_run = 0.f;
  const int k_off = col * DK * 2;
  const int k_sw[2] = {(quad ^ (col & 7)) << 4, ((quad + 4) ^ (col & 7)) << 4};
  constexpr int kVRow = (LATENT ? DK : DV) * 2;
  const int v_key = 4 * quad + (col >> 2);                   // of the 16 keys of a half; channels 4 (col & 3) on
  const int v_off = (LATENT ? 0 : 4 * kKeyPage) + v_key * kVRow + (col & 1) * 8;
  int v_sw[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) v_sw[i] = ((2 * i + ((col & 3) >> 1)) ^ (v_key & 7)) << 4;

  const float bias = POOLED && g.head_bias ? g.head_bias[h] : 0.f;
  const int my_blocks = POOLED ? blocks_of(p) : 0, wave_blocks = POOLED ? blocks_of(wave_last) : 0;
  auto attend_pooled = [&](const char* s, int st) __attribute__((always_inline)) {
    if (!works || st * kPooled >= wave_blocks) return;
    int cl = col, qd = quad;
    asm volatile("" : "+v"(cl), "+v"(qd));   // (or every address would be formed ahead of the loop and kept)
    f32x4 sc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      f32x4 a[2][2];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          a[u][i] = *reinterpret_cast<const f32x4*>(s + (16 * u + cl) * 512 + (((8 * ks + 2 * qd + i) ^ (cl & 7)) << 4));
      bf16x8 y[3] = {qp[kKept ? ks : 0][0], qp[kKept ? ks : 0][1], qp[kKept ? ks : 0][2]};
      asm volatile("" : "+v"(y[0]), "+v"(y[1]), "+v"(y[2]));   // (formed here, not ahead of the loop and kept)
#pragma unroll
      for (int j = 0; j < 8; ++j) {   // (the three parts make up the query's f32 value again)
        const float x = ((float)y[2][j] + (float)y[1][j]) + (float)y[0][j];
#pragma unroll
        for (int u = 0; u < 2; ++u) sc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][j >> 2][j & 3], x, sc[u], 0, 0, 0);
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 16 * u + 4 * qd + i;
        m_run = __builtin_elementwise_maximum(m_run, fabsf(sc[u][i]));
        const float wt = sigmoid_of(sc[u][i] + bias);
        sc[u][i] = st * kPooled + r < my_blocks ? wt : 0.f;
      }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 16 * u + 4 * qd + i;
        const char* at = s + (kPooled + r) * 512 + (cl & 3) * 4;
#pragma unroll
        for (int v = 0; v < VT; ++v)
          o[v] = __builtin_amdgcn_mfma_f32_16x16x4f32(*reinterpret_cast<const float*>(at + (((4 * v + (cl >> 2)) ^ (r & 7)) << 4)),
                                                      sc[u][i], o[v], 0, 0, 0);
      }
  };
  auto attend = [&](const char* s, int st) __attribute__((always_inline)) {
    const int base = stage_base(st);
    // (a stage of kept tokens holds no key of the window; in the window's stages kept tokens are seen too)
    const int key_end = st < kept_stages ? n_kept : 0x7fffffff;
    if (!works || base > wave_last) return;
    f32x4 sc[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) sc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    // (the four tiles of 16 keys side by side: four chains of sums)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      bf16x8 a[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) a[u] = *reinterpret_cast<const bf16x8*>(s + u * kKeyPage + k_off + (ks >> 1) * 128 + k_sw[ks & 1]);
      bf16x8 y[3];
      if constexpr (kKept) {
#pragma unroll
        for (int c = 0; c < 3; ++c) y[c] = qp[ks][c];
      } else {
        f32x4 x[2] = {qf[ks][0], qf[ks][1]};
        asm volatile("" : "+v"(x[0]), "+v"(x[1]));   // (or the parts would be formed ahead of the loop and kept)
        parts(x, y, std::false_type{});
      }
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int u = 0; u < 4; ++u) sc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u], y[c], sc[u], 0, 0, 0);
    }
    if constexpr (POOLED) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int d = p - (base + 16 * u + 4 * quad + i);
          m_run = __builtin_elementwise_maximum(m_run, fabsf(sc[u][i]));
          const float wt = sigmoid_of(sc[u][i] + bias);
          sc[u][i] = ((d >= 0) & (d < g.window)) ? wt : 0.f;
        }
    } else {
      float mx = m_run;
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int j = base + 16 * u + 4 * quad + i, d = p - j;
          // (bitwise: a chain of && would become branches)
          const bool seen = (d >= 0) & ((d < g.window) | (j < g.keep_first)) & (j < key_end);
          sc[u][i] = seen ? sc[u][i] : -INFINITY;
          mx = __builtin_elementwise_maximum(mx, sc[u][i]);
        }
      mx = __builtin_elementwise_maximum(mx, __shfl_xor(mx, 16, SD_WAVE));
      mx = __builtin_elementwise_maximum(mx, __shfl_xor(mx, 32, SD_WAVE));
      const float ref = mx == -INFINITY ? 0.f : mx;            // (no key seen yet)
      const float corr = exp_neg(m_run - ref);   // (nothing summed yet: 0)
      m_run = mx;
      float sum = 0.f;
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          sc[u][i] = exp_neg(sc[u][i] - ref);
          sum += sc[u][i];
        }
      l_run = fmaf(l_run, corr, sum);
      if (__any(corr != 1.f)) {
#pragma unroll
        for (int v = 0; v < VT; ++v) o[v] *= corr;
      }
    }
    bf16x8 pw[2][3];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const f32x4 x[2] = {sc[2 * u], sc[2 * u + 1]};
      parts(x, pw[u], std::false_type{});
    }
    // (two tiles of 16 channels side by side)
#pragma unroll
    for (int v = 0; v < VT; v += 2)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        bf16x8 a[2];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          const char* at = s + 32 * u * kVRow + v_off + (v >> 2) * 128 + v_sw[(v + w) & 3];
          const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at));
          const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 16 * kVRow));
          a[w] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int w = 0; w < 2; ++w) o[v + w] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[w], pw[u][c], o[v + w], 0, 0, 0);
      }
  };
  // Whether some row of the workgroup does not see all of stage st: the last of the kept stages' pooled blocks, and the
  // window's first and last stages
  const int kept_mixed = POOLED ? blocks_of(pos0) / kPooled : kept_stages;
  auto mixed = [&](int st) {
    if (st < kept_stages) return st >= kept_mixed;
    const int base = stage_base(st);
    return base + kKeys - 1 > pos0 || base <= last - g.window;
  };
  // This wave's rows of a stage's values (BYTES of them), once they are in LDS: what is no number becomes 0.  Returns the
  // rows.
  auto clear_odd = [&](char* rows, auto element, auto row_bytes, auto n_bytes) __attribute__((always_inline)) {
    constexpr bool kWide = sizeof(element) == 4;
    constexpr int kRow = decltype(row_bytes)::value, kBytes = decltype(n_bytes)::value;
    // (the top bit of each element whose exponent is all ones)
    auto bad = [](unsigned d) { return kWide ? ((d & 0x7f800000u) + 0x00800000u) & 0x80000000u : ((d & 0x7f807f80u) + 0x00800080u) & 0x80008000u; };
    unsigned any = 0;
#pragma unroll
    for (int at = 0; at < kBytes; at += 64 * 16) {
      const u32x4 d = *reinterpret_cast<const u32x4*>(rows + at + lane * 16);
#pragma unroll
      for (int i = 0; i < 4; ++i) any |= bad(d[i]);
    }
    unsigned found = 0;
    if (__any(any != 0)) {
#pragma unroll 1
      for (int at = lane * 16; at < kBytes; at += 64 * 16) {
        u32x4 d = *reinterpret_cast<const u32x4*>(rows + at);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const unsigned b = bad(d[i]);
          found |= b ? 1u << at / kRow : 0u;
          if (b & 0x80000000u) d[i] &= kWide ? 0u : 0x0000ffffu;
          if (b & 0x00008000u) d[i] &= 0xffff0000u;
        }
        *reinterpret_cast<u32x4*>(rows + at) = d;
      }
#pragma unroll
      for (int x = 1; x < 64; x <<= 1) found |= __shfl_xor(found, x, SD_WAVE);
    }
    return found;
  };
  // ... and reaches the queries that see its row: of latent rows, whose scores are no numbers then, as a whole.
  auto add_odd = [&](int st, bool means) __attribute__((always_inline)) {
#pragma unroll 1
    for (int w = 0; w < 4; ++w)
#pragma unroll 1
      for (unsigned rows = odd[st & 1][w]; rows; rows &= rows - 1) {
        const int j = means ? st * kPooled + 8 * w + __builtin_ctz(rows) : stage_base(st) + kPage * w + __builtin_ctz(rows);
        const int d = p - j;
        const bool seen = means ? j < my_blocks : (d >= 0) & ((d < g.window) | (j < g.keep_first));
        if constexpr (LATENT) {
          l_run = seen ? NAN : l_run;
        } else {
          const int jj = means ? min(j, n_kept - 1) : j, lp = means ? (jj * g.pool + g.pool - 1) / kPage : jj / kPage;
          const size_t head = (size_t)tbl[lp] * g.G + kvh;
          const float* pv = g.pv + (head * g.pslots + jj - lp * kPage / g.pool) * DV + 4 * quad;
          const bf16_t* vc = g.vc + (head * kPage + (jj & (kPage - 1))) * DV + 4 * quad;
#pragma unroll
          for (int v = 0; v < VT; ++v)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float x = means ? pv[16 * v + i] : (float)vc[16 * v + i];
              if (seen & !(fabsf(x) < INFINITY)) o[v][i] += x;
            }
        }
      }
  };
  // stage st is in `cur` once this wave's loads have landed and every wave is here; then nobody reads `nxt` any more
  auto step = [&](char* cur, char* nxt, int st) __attribute__((always_inline)) {
    // Rows behind the stage's last key hold what a page's earlier owner left, or nothing: they are cleared here, by the
    // wave that brought them.
    const bool means = POOLED && st < kept_stages, some = mixed(st);
    const int left = means ? kPage : stage_last(st) + 1 - stage_base(st) - wave * kPage;
    if (left < kPage || some) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      char* rows = cur + (LATENT ? wave * kKeyPage : 4 * kKeyPage + wave * kValPage);
      if (left < kPage) {
        for (int at = max(left, 0) * kVRow + lane * 16; at < kPage * kVRow; at += 64 * 16) *reinterpret_cast<u32x4*>(rows + at) = u32x4{0, 0, 0, 0};
        if (POOLED)   // (the keys too: their scores must be numbers)
          for (int at = max(left, 0) * DK * 2 + lane * 16; at < kKeyPage; at += 64 * 16)
            *reinterpret_cast<u32x4*>(cur + wave * kKeyPage + at) = u32x4{0, 0, 0, 0};
      }
      if (some) {
        unsigned found;
        if (means) found = clear_odd(cur + kPooled * 512 + wave * 4096, float(), Number<512>{}, Number<4096>{});
        else found = clear_odd(rows, bf16_t(), Number<kVRow>{}, Number<kPage * kVRow>{});
        if (lane == 0) odd[st & 1][wave] = found;
      }
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (st + 1 < stages) load(nxt, st + 1);
    if (means) attend_pooled(cur, st);
    else attend(cur, st);
    if (some && (odd[st & 1][0] | odd[st & 1][1] | odd[st & 1][2] | odd[st & 1][3])) add_odd(st, means);
  };
  // Query m of the workgroup by a whole wave: a lane a key for the scores, two channels for the sums.
  auto redo_query = [&](int m) __attribute__((always_inline)) {
    const int t = m / qh, h = kvh * qh + m - t * qh, p = pos0 + t;
    const float* q = g.q + (size_t)(row0 + first + t) * g.ldq + (size_t)h * DK;
    const int t_first = max(p - g.window + 1, 0);
    const int before = POOLED ? blocks_of(p) : min(g.keep_first, t_first), total = before + p - t_first + 1;
    const float add = POOLED && g.head_bias ? g.head_bias[h] : 0.f;
    // (row of the cache of key idx: pooled blocks or kept tokens first)
    auto row_of = [&](int idx) {
      if (POOLED && idx < before) {
        const int lp = (idx * g.pool + g.pool - 1) / kPage;
        return ((size_t)tbl[lp] * g.G + kvh) * g.pslots + idx - lp * kPage / g.pool;
      }
      const int j = idx < before ? idx : t_first + idx - before;
      return ((size_t)tbl[j / kPage] * g.G + kvh) * kPage + j % kPage;
    };
    float top = -INFINITY, l = 0.f, y[2] = {0.f, 0.f};
#pragma unroll 1
    for (int base = 0; base < total; base += SD_WAVE) {
      const int idx = min(base + lane, total - 1);
      const size_t row = row_of(idx);
      const bool block = POOLED && idx < before;
      float score = 0.f;
#pragma unroll 1
      for (int c = 0; c < DK; ++c) score = fmaf(q[c], block ? g.pk[row * DK + c] : (float)g.kc[row * DK + c], score);
      score *= g.scale;
      float w;
      if constexpr (POOLED) {
        w = 1.f / (1.f + expf(-(score + add)));
      } else {
        float mx = base + lane < total ? score : -INFINITY;
#pragma unroll
        for (int x = 1; x < SD_WAVE; x <<= 1) mx = fmaxf(mx, __shfl_xor(mx, x, SD_WAVE));
        mx = fmaxf(mx, top);
        const float corr = top == -INFINITY ? 0.f : expf(top - mx);
        top = mx;
        w = expf(score - mx);
        float sum = base + lane < total ? w : 0.f;
#pragma unroll
        for (int x = 1; x < SD_WAVE; x <<= 1) sum += __shfl_xor(sum, x, SD_WAVE);
        l = l * corr + sum;
        y[0] *= corr;
        y[1] *= corr;
      }
#pragma unroll 1
      for (int i = 0; i < min(SD_WAVE, total - base); ++i) {
        const float wi = __shfl(w, i, SD_WAVE);
        const size_t v = row_of(base + i) * DV + 2 * lane;
        const bool of_block = POOLED && base + i < before;
#pragma unroll
        for (int x = 0; x < 2; ++x) y[x] = fmaf(wi, of_block ? g.pv[v + x] : (float)g.vc[v + x], y[x]);
      }
    }
    static_assert(LATENT || (DK == 128 && DV == 128), "two channels a lane");
    const size_t at = (size_t)(row0 + first + t) * g.ldo + (size_t)h * DV + 2 * lane;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const float r = POOLED ? y[x] : y[x] * (1.f / l);
      if (g.out) g.out[at + x] = r;
      if (g.out_b) g.out_b[at + x] = (bf16_t)r;
    }
  };
  load(s0, 0);
#pragma unroll 1
  for (int st = 0; st < stages; st += 2) {
    step(s0, s1, st);
    if (st + 1 < stages) step(s1, s0, st + 1);
  }
  // A part of a query that is 0 makes a NaN of an infinite key, where the query's product with it is infinite and its weight
  // a number, and sigmoid_of wants finite scores: queries that met a score that is no number are done again, a key at a
  // time as on the vector pipe.  (Not of latent rows, where an infinite channel is an infinite value too.)
  bool done = !mine;
  if constexpr (!LATENT) {
    int odd_score = mine & (int)(POOLED ? !(m_run + fabsf(bias) < INFINITY) : m_run != m_run);
    odd_score |= __shfl_xor(odd_score, 16, SD_WAVE);
    odd_score |= __shfl_xor(odd_score, 32, SD_WAVE);
    done |= odd_score;
#pragma unroll 1
    for (unsigned left = (unsigned)__ballot(odd_score) & 0xffffu; left; left &= left - 1) redo_query(16 * wave + __builtin_ctz(left));
  }
  float inv = 1.f;
  if constexpr (!POOLED) {
    l_run += __shfl_xor(l_run, 16, SD_WAVE);
    l_run += __shfl_xor(l_run, 32, SD_WAVE);
    inv = 1.f / l_run;
  }
  if (done) return;
  const size_t at = (size_t)(row0 + first + t) * g.ldo + (size_t)h * DV + 4 * quad;
#pragma unroll
  for (int v = 0; v < VT; ++v) {
    const f32x4 y = o[v] * inv;
    if (g.out) *reinterpret_cast<f32x4*>(g.out + at + 16 * v) = y;
    if (g.out_b)
      *reinterpret_cast<bf16x4*>(g.out_b + at + 16 * v) = bf16x4{(bf16_t)y[0], (bf16_t)y[1], (bf16_t)y[2], (bf16_t)y[3]};
  }
}

}  // namespace

// Whether sd_rows_softmax_attention takes these sizes (v_cache nullptr: latent rows).
bool sd_rows_softmax_attention_fits_(int H, int G, int dk, int dv, int page, bool latent) {
  if (page != kPage || H % G || H / G > kRowsPerBlock) return false;
  return latent ? dk == 576 && dv == 512 : dk == 128 && dv == 128;
}

extern "C" int sd_rows_softmax_attention(const float* q, int64_t ldq, const void* k_cache, const void* v_cache,
                                         const int32_t* block_tables, int max_blocks, int page, int n_rows, int H, int G,
                                         int dk, int dv, int window, int keep_first, float scale, const int32_t* entries,
                                         int n_entries, float* out, void* out_b, int64_t ldo, sd_stream_t stream) {
  return sd_rows_softmax_attention_(q, ldq, k_cache, v_cache, block_tables, max_blocks, page, n_rows, H, G, dk, dv, window,
                                    keep_first, scale, entries, n_entries, false, out, out_b, ldo, stream);
}

int sd_rows_softmax_attention_(const float* q, int64_t ldq, const void* k_cache, const void* v_cache,
                               const int32_t* block_tables, int max_blocks, int page, int n_rows, int H, int G, int dk,
                               int dv, int window, int keep_first, float scale, const int32_t* entries, int n_entries,
                               bool long_only, float* out, void* out_b, int64_t ldo, sd_stream_t stream) {
  SD_REQUIRE(q && k_cache && block_tables && entries && (out || out_b) && max_blocks >= 1 && n_rows >= 1 && n_entries >= 1 &&
                 n_rows >= n_entries && H >= 1 && G >= 1 && window >= 1 && keep_first >= 0,
             SD_ERR_INVALID, "sd_rows_softmax_attention: bad argument");
  SD_REQUIRE(sd_rows_softmax_attention_fits_(H, G, dk, dv, page, !v_cache), SD_ERR_UNSUPPORTED,
             "sd_rows_softmax_attention: %d heads over %d of %d / %d channels, pages of %d", H, G, dk, dv, page);
  RowsAttnArgs g{q, ldq, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables, entries, out, (bf16_t*)out_b, ldo,
                 scale, max_blocks, n_entries, H, G, window, keep_first, long_only ? kLongPortion : 0, nullptr, nullptr, nullptr,
                 1, 0};
  SD_REQUIRE(ldq % 4 == 0 && ldo % 4 == 0 && ldq >= (int64_t)H * dk && ldo >= (int64_t)H * dv && sd_aligned16(q) &&
                 sd_aligned16(k_cache) && (!v_cache || sd_aligned16(v_cache)) && (!out || sd_aligned16(out)) &&
                 (!out_b || (reinterpret_cast<uintptr_t>(out_b) & 7) == 0),
             SD_ERR_INVALID, "sd_rows_softmax_attention: rows must be 16-byte aligned");
  const dim3 grid(n_rows / (kRowsPerBlock / (H / G)) + n_entries, G);
  if (v_cache) hipLaunchKernelGGL((rows_attn_kernel<4, 8, false, false>), grid, dim3(256), 0, (hipStream_t)stream, g);
  else hipLaunchKernelGGL((rows_attn_kernel<18, 32, true, false>), grid, dim3(256), 0, (hipStream_t)stream, g);
  SD_CHECK_LAUNCH("sd_rows_softmax_attention");
  return SD_OK;
}

// Window and pooled blocks with sigmoid weights (the means of the rows' own blocks are in the cache already).
int sd_rows_pool_attention_(const float* q, int64_t ldq, const void* k_cache, const void* v_cache, const float* pk, const float* pv,
                            const int32_t* block_tables, int max_blocks, int n_rows, int H, int G, int window, int pool, int pslots,
                            float scale, const float* head_bias, const int32_t* entries, int n_entries, bool long_only,
                            float* out, sd_stream_t stream) {
  RowsAttnArgs g{q, ldq, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables, entries, out, nullptr, (int64_t)H * 128,
                 scale, max_blocks, n_entries, H, G, window, 0, long_only ? kLongPortion : 0, pk, pv, head_bias, pool, pslots};
  SD_REQUIRE(ldq % 4 == 0 && sd_aligned16(q) && sd_aligned16(k_cache) && sd_aligned16(v_cache) && sd_aligned16(pk) &&
                 sd_aligned16(pv) && sd_aligned16(out),
             SD_ERR_INVALID, "sd_rows_pool_attention: rows must be 16-byte aligned");
  hipLaunchKernelGGL((rows_attn_kernel<4, 8, false, true>), dim3(n_rows / (kRowsPerBlock / (H / G)) + n_entries, G), dim3(256), 0,
                     (hipStream_t)stream, g);
  SD_CHECK_LAUNCH("sd_rows_pool_attention");
  return SD_OK;
}

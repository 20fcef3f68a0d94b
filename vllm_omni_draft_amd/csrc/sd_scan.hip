// Decayed outer-product recurrences token by token: S <- d_t S + (a_t k_t) v_t^T, o_t = S^T q_t (+ skip v_t), per (entry, head).
// d_t: a factor per head, per (row, head) or per (row, key channel).
//
// The order of every sum is fixed: strips of 16 key channels, a strip's products in ascending channel by fused multiply-adds,
// the strips' sums in order (the skip term on strip 0), so a row's bits do not depend on how a prompt is cut.  A token needs the one
// before it, so a head has only dk x dv independent chains, and what bounds the op is how few instructions a wave needs for a token:
//   - Two lanes share a strip of a value column, eight channels each.  The upper one is a token behind the lower one and starts from its
//     sum (v_permlane32_swap, one instruction): the same chain of sixteen products at half the instructions a lane and token.
//   - Sixteen lanes side by side hold sixteen columns of a strip, and its k and q arrive as one value a lane (eight of k, eight of
//     q): the products take them by row broadcast, an operand modifier, instead of reading them from LDS for every lane.  (A strip a
//     lane and 16-byte LDS reads of k, q and d for all: 1200 clocks a token, most of them the LDS pipe's, of 192 for the products.)
//   - 64 workgroups of 8 heads of 128 x 128 instead of 32, a wave a SIMD.
// us, before (256 threads of a strip a lane, 32 columns a workgroup) / now: 777 rows of 8 heads of 128 x 128, a decay per channel 404 / 92,
// per head 284 / 80, per row 312 / 95; 400 rows of 32 heads of 128 x 64 per row 165 / 53; 64 portions of 60 rows of 16 heads per channel
// 357 / 228, per head 286 / 199; one row of each of 4 requests, 32 heads of 128 x 64, 7.7 / 5.2; 16 heads of 64 x 64 per row,
// 16 portions of 24 rows 16.1 / 9.8, 300 rows 123 / 35; of 32 x 128 per channel 21.7 / 10.9, 166 / 39; of 16 x 16 per head 19.2 / 5.7, 182 / 29.  The products alone are 31 us of the 92.
#include <type_traits>

#include "sd_common.h"

namespace {

constexpr int kStrip = 16, kHalf = 8, kCols = 16;
constexpr int kPerHead = 0, kPerRow = 1, kPerChannel = 2;

struct ScanArgs {
  const float *q, *k, *v;
  int64_t ldqk, ldv;
  const float *decay, *k_scale;
  const void* skip;
  int w_f32;
  float* state;
  const int32_t* entries;
  float* out;
  int H, hpg, dk, dv, tiles, strips, max_rows;
};

// One token of a lane's eight channels: S[r] = fma(d, S[r], k[r] v), sum = fma(q[r], S[r], sum) for r = 0..7, with lane r of sixteen
// holding k[r] and, if D_LANES, d[r], lane r + 8 holding q[r].  Written out because the compiler folds a row broadcast into a
// product but not into a fused multiply-add (40 instructions instead of 24).  A row broadcast must not read what a vector
// instruction right before it wrote, which only the first ones could: s_nop.
#define SD_BCAST(r) " row_newbcast:" #r " row_mask:0xf bank_mask:0xf\n\t"
#define SD_MUL(r) "v_mul_f32_dpp %" #r ", %17, %19" SD_BCAST(r)
#define SD_DECAY_LANES(r, s) "v_fmac_f32_dpp %" #r ", %18, %" #s SD_BCAST(r)
#define SD_DECAY_ONE(r, s) "v_fmac_f32_e32 %" #r ", %18, %" #s "\n\t"
#define SD_ADD(r, lane) "v_fmac_f32_dpp %8, %17, %" #r SD_BCAST(lane)
#define SD_TOKEN(D)                                                                                                             \
  asm("s_nop 1\n\t" SD_MUL(0) SD_MUL(1) D(0, 9) SD_MUL(2) D(1, 10) SD_ADD(0, 8) SD_MUL(3) D(2, 11) SD_ADD(1, 9) SD_MUL(4) D(3, 12) \
          SD_ADD(2, 10) SD_MUL(5) D(4, 13) SD_ADD(3, 11) SD_MUL(6) D(5, 14) SD_ADD(4, 12) SD_MUL(7) D(6, 15) SD_ADD(5, 13) D(7, 16)  \
              SD_ADD(6, 14) SD_ADD(7, 15)                                                                                       \
      : "=&v"(T[0]), "=&v"(T[1]), "=&v"(T[2]), "=&v"(T[3]), "=&v"(T[4]), "=&v"(T[5]), "=&v"(T[6]), "=&v"(T[7]), "+&v"(sum)       \
      : "v"(S[0]), "v"(S[1]), "v"(S[2]), "v"(S[3]), "v"(S[4]), "v"(S[5]), "v"(S[6]), "v"(S[7]), "v"(kq), "v"(d), "v"(v))
template <bool D_LANES>
__device__ __forceinline__ void token_products(float (&S)[kHalf], float& sum, float kq, float d, float v) {
  float T[kHalf];
  if constexpr (D_LANES) SD_TOKEN(SD_DECAY_LANES);
  else SD_TOKEN(SD_DECAY_ONE);
#pragma unroll
  for (int r = 0; r < kHalf; ++r) S[r] = T[r];
}
// The lower half of the wave's `x` in the upper half, zero in the lower one
__device__ __forceinline__ float behind(float x) {
  return __int_as_float(__builtin_amdgcn_permlane32_swap(0, __float_as_int(x), false, false)[0]);
}

// Half of a workgroup's waves multiply; the others bring tokens and carry results, in chunks of CH tokens between barriers: global ->
// registers -> LDS, a ring of three chunks (the one in use and the last token of the one before it, which the upper lanes are at;
// the next one), while the one behind that is on its way, and add the strips' sums of the chunk before.  (Every wave doing
// all of that: 158 us instead of 92, per channel as above.)  A group of 16 lanes has its own ring, so a token's place is an
// immediate offset, and rings lie 16 (8) banks apart.
template <int CH, int COLS>
struct Lds {
  static constexpr int kq = (3 * CH + 1) * kStrip;   // floats of a group's ring: [token][8 of k, 8 of q]
  static constexpr int d = (3 * CH + 1) * kHalf;     // [token][8]
  static constexpr int part = (2 * CH + 1) * COLS;   // a strip's sums: [token][COLS]
  static constexpr int v = (3 * CH + 1) * COLS;      // [token][COLS]  (a token behind the ring's last one is read and not used)
  static constexpr int row = (3 * CH + 1) * 2;       // per row: [token][decay, keys' scale]
};

// COLS: columns of a workgroup; 32: two groups of sixteen columns of the one strip that sixteen key channels or fewer are.
template <int DECAY, int CH, int COLS>
__global__ __launch_bounds__(1024) void decay_scan_kernel(ScanArgs a) {
  using L = Lds<CH, COLS>;
  const int nthr = blockDim.x / 2, lane = threadIdx.x & 63;
  const int strips = COLS > kCols ? 1 : nthr / 32;   // (else an even number of strips: a wave has two)
  const bool carries = (int)threadIdx.x >= nthr;
  const int tid = carries ? threadIdx.x - nthr : threadIdx.x, wave = tid >> 6;
  const int work = xcd_order(blockIdx.x, gridDim.x);
  const int tile = work % a.tiles, h = work / a.tiles % a.H, e = work / a.tiles / a.H;
  const int slot = a.entries[4 * e], row0 = a.entries[4 * e + 1], len = a.entries[4 * e + 2], pos0 = a.entries[4 * e + 3];
  if (len > a.max_rows || len < 1) return;
  const int dk = a.dk, dv = a.dv;
  extern __shared__ float lds[];
  float* kq = lds;
  float* ds = kq + 2 * strips * L::kq;
  float* vs = ds + (DECAY == kPerChannel ? 2 * strips * L::d : DECAY == kPerRow ? L::row : 0);
  float* part = vs + L::v;
  const int n_chunks = len / CH + 1;     // of len + 1 steps; step i: token i of the lower lanes, token i - 1 of the upper ones
  int ring = 0;

  if (carries) {
    // What this thread brings of every chunk: one value of a token's k or q, half as many decays, and values of v
    const int kr = (tid >> 4) * kHalf + (tid & 7), dr = tid % (nthr / 2), d_late = tid >= nthr / 2;
    const float* kq_src = ((tid & 8) ? a.q : a.k) + (size_t)row0 * a.ldqk + (size_t)(h / a.hpg) * dk + min(kr, dk - 1);
    const float* d_src = a.decay + (DECAY == kPerChannel ? (size_t)row0 * a.H * dk + (size_t)h * dk + min(dr, dk - 1)
                                                         : (size_t)row0 * a.H + h);
    const int64_t d_step = DECAY == kPerChannel ? (int64_t)a.H * dk : a.H;
    const float* v_src = a.v + (size_t)row0 * a.ldv + (size_t)h * dv + min(tile * COLS + tid % COLS, dv - 1);
    float* kq_to = kq + (tid >> 4) * L::kq + (tid & 15);
    float* d_to = ds + (dr >> 3) * L::d + (dr & 7) + d_late * kHalf;
    constexpr int kV = CH * COLS / 64;  // (of a wave alone)
    const int v_loads = (CH * COLS + nthr - 1) / nthr;
    float pkq[CH], pd[CH / 2], pv[kV], pa = 1.f;
    // (every load is issued, on an address clamped into the portion: a guarded load would become a branch whose join waits
    // for the loads in flight)
    auto fetch = [&](int t0, auto tokens) __attribute__((always_inline)) {
      constexpr int N = decltype(tokens)::value;
      const bool whole = N == CH && t0 + N <= len;
      const float* p = kq_src + t0 * a.ldqk;
      if (whole) {
#pragma unroll
        for (int i = 0; i < N; ++i, p += a.ldqk) pkq[i] = *p;
      } else {
#pragma unroll
        for (int i = 0; i < N; ++i) pkq[i] = kq_src[min(t0 + i, len - 1) * a.ldqk];
      }
      if (DECAY == kPerChannel) {
        p = d_src + (t0 + d_late) * d_step;
        if (whole) {
#pragma unroll
          for (int i = 0; i < N / 2; ++i, p += 2 * d_step) pd[i] = *p;
        } else {
#pragma unroll
          for (int i = 0; i < N / 2; ++i) pd[i] = d_src[min(t0 + 2 * i + d_late, len - 1) * d_step];
        }
      }
      if (DECAY == kPerRow) {
        const int64_t at = min(t0 + tid % CH, len - 1) * d_step;
        pd[0] = d_src[at];
        if (a.k_scale) pa = a.k_scale[(size_t)row0 * a.H + h + at];
      }
#pragma unroll
      for (int i = 0; i < (kV * N + CH - 1) / CH; ++i) {
        if (i >= v_loads) break;
        pv[i] = v_src[min(t0 + (tid + i * nthr) / COLS, len - 1) * a.ldv];
      }
    };
    auto put = [&](int at) __attribute__((always_inline)) {   // (in tokens)
#pragma unroll
      for (int i = 0; i < CH; ++i)
        if (COLS == kCols || kr < kStrip) kq_to[(at + i) * kStrip] = kr < dk ? pkq[i] : 0.f;
      if (DECAY == kPerChannel) {
#pragma unroll
        for (int i = 0; i < CH / 2; ++i)
          if (COLS == kCols || dr < kStrip) d_to[(at + 2 * i) * kHalf] = dr < dk ? pd[i] : 0.f;
      }
      if (DECAY == kPerRow && tid < CH) {
        ds[(at + tid) * 2] = pd[0];
        ds[(at + tid) * 2 + 1] = pa;
      }
#pragma unroll
      for (int i = 0; i < kV; ++i) {
        if (i >= v_loads) break;
        const int idx = tid + i * nthr;
        if (idx < CH * COLS) vs[at * COLS + idx] = tile * COLS + idx % COLS < dv ? pv[i] : 0.f;
      }
    };
    // The strips' sums of tokens lo .. hi - 1
    auto emit = [&](int lo, int hi) __attribute__((always_inline)) {
      for (int idx = tid; idx < (hi - lo) * COLS; idx += nthr) {
        const int t = lo + idx / COLS, cc = idx % COLS;
        const float* p = part + (t & (2 * CH - 1)) * COLS + cc;
        float o = p[0];
        for (int i = 1; i < a.strips; i += 7) {
          float x[7];
#pragma unroll
          for (int j = 0; j < 7; ++j) x[j] = p[min(i + j, a.strips - 1) * L::part];
#pragma unroll
          for (int j = 0; j < 7; ++j) o = i + j < a.strips ? o + x[j] : o;
        }
        if (tile * COLS + cc < dv) a.out[(size_t)(row0 + t) * ((size_t)a.H * dv) + (size_t)h * dv + tile * COLS + cc] = o;
      }
    };
    // (nobody uses a token behind the last one: a portion of half a chunk asks for no more where a token has three values of a channel, and
    // a portion of one chunk does not ask for a second one.  16 heads of 128 x 256 per channel, 256 portions of one row 440 / 338, 300 of three 552 /
    // 429; per head 351 / 270 and 458 / 343.  The half for all decays, or the tokens one by one: up to 20 % slower.)
    using Chunk = std::integral_constant<int, CH>;
    if (DECAY == kPerChannel && CH == 8 && len <= CH / 2) fetch(0, std::integral_constant<int, CH / 2>());
    else fetch(0, Chunk());
    put(0);
    if (len > CH) fetch(CH, Chunk());
    for (int ch = 0; ch < n_chunks; ++ch) {
      __syncthreads();
      ring = ring == 2 * CH ? 0 : ring + CH;
      if (ch + 1 < n_chunks) put(ring);
      if (ch + 2 < n_chunks) fetch((ch + 2) * CH, Chunk());
      if (ch > 0) emit(max((ch - 1) * CH - 1, 0), ch * CH - 1);
    }
    __syncthreads();
    emit(max((n_chunks - 1) * CH - 1, 0), len);
    return;
  }

  const int upper = lane >> 5, s = COLS > kCols ? 0 : wave * 2 + ((lane >> 4) & 1), c = lane % COLS;   // (an upper lane: that of lane - 32)
  const int col = tile * COLS + c, r0 = s * kStrip + upper * kHalf;
  float* st = a.state + ((size_t)slot * a.H + h) * dk * dv;
  float S[kHalf];
#pragma unroll
  for (int r = 0; r < kHalf; ++r) S[r] = pos0 > 0 && r0 + r < dk && col < dv ? st[(size_t)(r0 + r) * dv + col] : 0.f;
  const float dh = DECAY == kPerHead ? a.decay[h] : 0.f;
  const float skip_h = DECAY == kPerRow && a.skip
                           ? a.w_f32 ? ((const float*)a.skip)[h] : (float)((const bf16_t*)a.skip)[h] : 0.f;
  const float* kq_mine = kq + (s * 2 + upper) * L::kq + (lane & 15);
  const float* d_mine = DECAY == kPerChannel ? ds + (s * 2 + upper) * L::d + (c & 7) : ds;
  const float* v_mine = vs + c;
  struct Token {
    float kq, d, a, v;
  };
  auto read = [&](int at, int i) __attribute__((always_inline)) {
    Token x;
    x.kq = kq_mine[at * kStrip + i * kStrip];
    x.d = DECAY == kPerChannel ? d_mine[at * kHalf + i * kHalf] : DECAY == kPerRow ? d_mine[at * 2 + i * 2] : dh;
    x.a = DECAY == kPerRow ? d_mine[at * 2 + i * 2 + 1] : 1.f;
    x.v = v_mine[at * COLS + i * COLS];
    return x;
  };
  float sum = 0.f;                       // of the token this lane has just seen
  auto products = [&](const Token& x) __attribute__((always_inline)) {
    token_products<DECAY == kPerChannel>(S, sum, x.kq, x.d, DECAY == kPerRow ? x.a * x.v : x.v);
  };
  // A token's sum of a strip, from its upper lanes (the lower lanes' values go where nobody reads)
  float* part_mine = upper ? part + s * L::part + c : part + strips * L::part + lane;
  auto keep = [&](float* to, const Token& x) __attribute__((always_inline)) {
    *to = DECAY == kPerRow && s == 0 ? fmaf(skip_h, x.v, sum) : sum;
  };
  for (int ch = 0; ch < n_chunks; ++ch) {
    __syncthreads();
    const int t0 = ch * CH, at = ring + 1 - upper;   // of the step behind t0
    Token x = read(upper ? (ring == 0 ? 3 * CH : ring) - 1 : ring, 0);
    float* kept = part_mine + (ch & 1) * CH * COLS - COLS;   // places of tokens t0 - 1 and t0
    float* before = ch & 1 ? kept : part_mine + (2 * CH - 1) * COLS;
    if (ch > 0 && t0 + CH <= len) {
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const Token y = read(at, i < CH - 1 ? i : 0);    // (the last one's is not used)
        __builtin_amdgcn_sched_barrier(0);               // (a token ahead of its use: left to itself the compiler reads it right there)
        sum = behind(sum);
        products(x);
        keep(i == 0 ? before : kept + i * COLS, x);
        x = y;
      }
    } else {
      for (int i = 0; i < CH && t0 + i <= len; ++i) {
        const Token y = read(at, i);     // (a token behind the last one is read and not used)
        sum = behind(sum);
        // the first token's step is the lower lanes' alone, the one behind the last token's the upper lanes'
        if (t0 + i == 0 ? !upper : t0 + i < len || upper) products(x);
        if (t0 + i > 0) keep(i == 0 ? before : kept + i * COLS, x);
        x = y;
      }
    }
    ring = ring == 2 * CH ? 0 : ring + CH;
  }
  __syncthreads();
  if (col < dv) {
#pragma unroll
    for (int r = 0; r < kHalf; ++r)
      if (r0 + r < dk) st[(size_t)(r0 + r) * dv + col] = S[r];
  }
}

template <int DECAY, int CH, int COLS>
void launch_scan(const ScanArgs& a, int grid, int nthr, hipStream_t st) {
  using L = Lds<CH, COLS>;
  const int strips = COLS > kCols ? 1 : nthr / 32, d = DECAY == kPerChannel ? 2 * strips * L::d : DECAY == kPerRow ? L::row : 0;
  // (64 floats and a ring's length behind the last strip's sums: the lower lanes' places)
  const size_t lds = sizeof(float) * (2 * strips * L::kq + d + L::v + (strips + 1) * L::part + 64);
  decay_scan_kernel<DECAY, CH, COLS><<<grid, 2 * nthr, lds, st>>>(a);
}

// Workgroups of 16 columns from which keys of one strip take 32: a wave's second strip would be nothing but padding, and the chip has more to do than
// it holds at once.  16 heads of 16 x 128 in workgroups of 64 columns and no carrying waves / of 16 / of 32: 256 portions of one row per channel 27.6 / 46 /
// 25.5, per row 28.8 / 36 / 20.5, per head 26.0 / 36 / 21.7; 64 of 24 tokens per channel 25.5 / 30.1 / 20.1; below it 16 / 32: one of 300 tokens per channel 34 /
// 42, 16 of 60 of 16 x 64 11.6 / 12.3.
constexpr int kManyGroups = 4096;
template <int DECAY>
int scan(ScanArgs a, int n_entries, const char* name, hipStream_t st) {
  SD_REQUIRE(a.dk >= 1 && a.dk <= 256, SD_ERR_UNSUPPORTED, "%s: key size %d outside 1..256", name, a.dk);
  a.strips = (a.dk + kStrip - 1) / kStrip;
  const int nthr = (a.strips + 1) / 2 * 64;
  const bool wide = a.strips == 1 && (int64_t)((a.dv + kCols - 1) / kCols) * a.H * n_entries >= kManyGroups;
  const int cols = wide ? 2 * kCols : kCols;
  a.tiles = (a.dv + cols - 1) / cols;
  const int64_t grid = (int64_t)a.tiles * a.H * n_entries;
  SD_REQUIRE(grid < INT_MAX, SD_ERR_UNSUPPORTED, "%s: more than 2^31 workgroups", name);
  // Chunks of eight tokens are at most 52 KB of LDS up to 128 channels, chunks of four beyond; three workgroups a CU up to 160 channels, two of
  // twelve waves or more from there on.  us in chunks of four / eight, 16 heads of 128 x 128 per channel: 300 tokens 47.9 / 34.4, 8 portions of 100 41.2 / 36.8, 32 of one
  // row 19.1 / 23.9; of 256 x 128: 73.8 / 50.5, 76.1 / 76.8, 36.5 / 59.4.
  if (wide) launch_scan<DECAY, 8, 2 * kCols>(a, (int)grid, nthr, st);
  else if (nthr <= 256) launch_scan<DECAY, 8, kCols>(a, (int)grid, nthr, st);
  else launch_scan<DECAY, 4, kCols>(a, (int)grid, nthr, st);
  SD_CHECK_LAUNCH(name);
  return SD_OK;
}

}  // namespace

int sd_decay_scan_(const float* q, const float* k, const float* v, int64_t ld, const float* decay, int per_channel,
                   float* state, const int32_t* entries, int n_entries, int max_rows, float* out, int H, int dk, int dv,
                   sd_stream_t stream) {
  SD_REQUIRE(q && k && v && decay && state && entries && out && n_entries >= 1 && H >= 1 && dv >= 1,
             SD_ERR_INVALID, "sd_decay_scan: bad argument");
  const ScanArgs a{q, k, v, ld, ld, decay, nullptr, nullptr, 0, state, entries, out, H, 1, dk, dv, 0, 0, max_rows};
  return per_channel ? scan<kPerChannel>(a, n_entries, "sd_decay_scan", (hipStream_t)stream)
                     : scan<kPerHead>(a, n_entries, "sd_decay_scan", (hipStream_t)stream);
}

int sd_decay_scan_rows_(const float* q, const float* k, int64_t ldqk, const float* v, int64_t ldv, const float* decay,
                        const float* k_scale, const void* skip, int w_f32, float* state, const int32_t* entries,
                        int n_entries, int max_rows, float* out, int H, int Gq, int dk, int dv, sd_stream_t stream) {
  SD_REQUIRE(q && k && v && decay && state && entries && out && n_entries >= 1 && H >= 1 && Gq >= 1 && H % Gq == 0 &&
                 dv >= 1,
             SD_ERR_INVALID, "sd_decay_scan_rows: bad argument");
  SD_REQUIRE(H <= 4096, SD_ERR_UNSUPPORTED, "sd_decay_scan_rows: more than 4096 heads");
  const ScanArgs a{q, k, v, ldqk, ldv, decay, k_scale, skip, w_f32, state, entries, out, H, H / Gq, dk, dv, 0, 0, max_rows};
  return scan<kPerRow>(a, n_entries, "sd_decay_scan_rows", (hipStream_t)stream);
}

extern "C" int sd_decay_scan(const float* q, const float* k, const float* v, int64_t ld, const float* decay,
                             int per_channel, float* state, const int32_t* entries, int n_entries,
                             float* out, int H, int dk, int dv, sd_stream_t stream) {
  return sd_decay_scan_(q, k, v, ld, decay, per_channel, state, entries, n_entries, INT_MAX, out, H, dk, dv, stream);
}

extern "C" int sd_decay_scan_rows(const float* q, const float* k, int64_t ldqk, const float* v, int64_t ldv,
                                  const float* decay, const float* k_scale, const void* skip, int w_f32, float* state,
                                  const int32_t* entries, int n_entries, float* out, int H, int Gq, int dk, int dv,
                                  sd_stream_t stream) {
  return sd_decay_scan_rows_(q, k, ldqk, v, ldv, decay, k_scale, skip, w_f32, state, entries, n_entries, INT_MAX, out, H,
                             Gq, dk, dv, stream);
}

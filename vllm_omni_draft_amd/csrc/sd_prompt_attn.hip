// Attention of prompt passes over the paged cache: the rows of a pass belong to runs of consecutive tokens
// (items), each of one sequence, whose keys and values are in the cache already.
//
// sd_paged_attention is made for a handful of rows: a workgroup streams a split of the keys for at most 64 rows and
// leaves partial sums to a second launch.  For a prompt that meant 64 rows per read of the keys, f32 partials of
// every split (rows x splits x heads x D, written and read) and a merge through LDS per workgroup: 43 of 157 ms of a
// 4096-token prompt of an 8B model.  Here a workgroup of four waves takes 128 query rows of one KV head (128 / (Hq/Hkv)
// tokens) through all their keys, K and V passing through LDS by direct loads (a page of 16 tokens of a head is one
// contiguous piece of K and one of V), two stages, one barrier a stage.  A wave owns 32 rows; the score tile has keys
// on the matrix instruction's row index, so a lane holds 16 scores of ONE row, the online softmax is lane-local plus
// one exchange, and the exponentials are the B operand of the second product as they are (see sd_v_slot).
//
// The arithmetic is that of sd_paged_attention with the same split_tokens, sum for sum: a split's tiles of 32 keys
// belong to four chains (tile j to chain j % 4), each with an online softmax of its own; the chains are weighted and
// added in order, then the splits, against the maximum over all splits.  A row thus has the bits that a decode pass
// gives it, and the bits do not depend on how a prompt is cut.  The weights of chains and splits need the maxima of
// everything first: a first sweep computes the scores for the maxima alone (a third of the matrix work), which costs
// less than keeping the splits' sums.  It needs keys only and no order, so its stages are 128 keys (64: see kKeys), half the barriers of the
// second sweep's, in which a stage is one chain of a split (tiles c and c + 4 of eight), so that only one chain's sums, a quarter of the
// channels at a time, are live beside the split's and the row's.
// What bounds it: products and vector work of a wave follow each other (two waves a SIMD: 55 % and 36 % of the time at 4096 tokens).  us, stages of
// one chain in both sweeps and exchanges through LDS / now, the call by itself in a graph, 32 heads over 8 in splits of 256: 4096 tokens of
// size 128 288 / 271, 1024 59.2 / 54.3, of size 64 36.0 / 33.5; 8 prompts of 64..1000, 28 over 4, 64.8 / 59.5 (in an 8B
// model's prompt, with cold keys, 4096 tokens take 338 / 319).  Size 128 in splits of 256 keeps 22 registers a lane in scratch at two blocks a CU.  Four stages in flight where a block is alone on its CU, both tiles' products before
// their weights, and raised wave priority around products were no faster.
#include <mutex>
#include <type_traits>

#include "sd_common.h"

namespace {

struct PromptAttnArgs {
  const bf16_t* q;
  int64_t ldq;
  const bf16_t* kc;
  const bf16_t* vc;
  const int32_t* block_tables;
  int max_blocks;
  const int32_t* items;  // [n][4]: first row, tokens, block-table row, position of the first token
  bf16_t* out;
  int64_t ldo;
  int Hq, Hkv;
  float scale_log2;
};

constexpr int kTable = 1024;       // page numbers kept in LDS at a time
constexpr int kRows = SD_PROMPT_BLOCK_ROWS;

// TPC: tiles of a chain (split_tokens / 128): 1 or 2
template <int D, int TPC>
__global__ __launch_bounds__(256, 2) void prompt_attn_kernel(PromptAttnArgs a) {
  constexpr int KS = D / 16, DT = D / 32;
  constexpr int kPage = D * 32;                 // bytes of a page of K (or V) of one head
  constexpr int kLoads = kPage / 1024;          // direct loads of a page
  constexpr int kPages = 2 * TPC;               // pages of a stage: a wave brings one (of K and of V)
  constexpr int kSplit = 128 * TPC, kSplitPages = kSplit / 16;
  // Keys of a stage of the first sweep: 128, but 64 where 128 of K alone are more than the second sweep's K and V and cost the room of a second
  // workgroup on the CU (size 128 in splits of 128: 4096 tokens 284 us, with 128 keys a stage 408; of size 64 1024 tokens 37.6, with 128 36.9).
  constexpr int kKeyPages = D == 64 ? 8 : 2 * kPages, kKeys = 16 * kKeyPages;
  static_assert(kKeyPages >= 2 * kPages && kKeyPages % 4 == 0 && (kKeys == kSplit || 2 * kKeys == kSplit), "a stage of either sweep; a split's stages");
  __shared__ __attribute__((aligned(1024))) char s0[kKeyPages * kPage];
  __shared__ __attribute__((aligned(1024))) char s1[kKeyPages * kPage];
  __shared__ int32_t table[kTable];
  extern __shared__ float split_max[];          // [splits][kRows]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5;
  const int kvh = blockIdx.x;
  const int4 item = reinterpret_cast<const int4*>(a.items)[blockIdx.y];
  const int row0 = item.x, n_tok = item.y, pos0 = item.w;
  const int32_t* bt = a.block_tables + (size_t)item.z * a.max_blocks;
  const int G = a.Hq / a.Hkv;
  const int m_rows = n_tok * G;
  const int kv_len = pos0 + n_tok;
  const int last_page = (kv_len - 1) >> 4;
  const int n_st = (kv_len + kSplit - 1) / kSplit * 4;   // stages of the second sweep
  const int n_max = (kv_len + 2 * kKeys - 1) / (2 * kKeys) * 2;   // and of the first, an even number: half a split or a whole one each

  // this lane's query row, its keys, and how far the wave's rows see
  const int m = wave * 32 + r;
  const bool valid = m < m_rows;
  const int t = valid ? m / G : 0, g = valid ? m - t * G : 0;
  const int see = valid ? pos0 + t + 1 : 0;
  const bool live_wave = wave * 32 < m_rows;
  const int wave_first = live_wave ? pos0 + (wave * 32) / G + 1 : 0;                        // fewest keys of a row
  const int wave_last = live_wave ? pos0 + min(wave * 32 + 31, m_rows - 1) / G + 1 : 0;     // most
  bf16x8 qf[KS];
  const bf16_t* qrow = a.q + (size_t)(row0 + t) * a.ldq + (size_t)(kvh * G + g) * D;
#pragma unroll
  for (int s = 0; s < KS; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(qrow + 16 * s + 8 * h);

  f32x16 o_split[DT], o_row[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o_split[dt][i] = o_row[dt][i] = 0.f;
  float l_split = 0.f, l_row = 0.f, top_split = -INFINITY, top_row = -INFINITY;

  int table0 = 0;  // first page in the table
  auto fill_table = [&](int first) {
    table0 = first;
    for (int e = tid; e < kTable; e += 256) table[e] = bt[min(min(first + e, last_page), a.max_blocks - 1)];
  };
  auto first_page = [&](int st) { return (st >> 2) * kSplitPages; };
  auto bring = [&](char* to, const bf16_t* pool, int page) __attribute__((always_inline)) {
    const int blk = __builtin_amdgcn_readfirstlane(table[max(min(page, last_page) - table0, 0)]);
    const size_t at = ((size_t)blk * a.Hkv + kvh) * (size_t)(D * 16);
    const auto from = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(pool + at), 0, kPage, 0x00027000);
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (lds_void*)(to + i * 1024), 16, lane * 16 + i * 1024, 0, 0, 0);
  };
  // first sweep: stage st holds K pages alone, a quarter of them a wave
  auto load_keys = [&](char* s, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kKeyPages / 4; ++i) {
      const int page = wave * (kKeyPages / 4) + i;
      bring(s + page * kPage, a.kc, st * kKeyPages + page);
    }
  };
  // second sweep: stage st is chain st & 3 of split st >> 2; wave w brings page w & 1 of tile chain + 4 (w >> 1): K, and V behind
  // the K pages
  auto load = [&](char* s, int st) __attribute__((always_inline)) {
    if (wave >= kPages) return;
    const int page = first_page(st) + 2 * ((st & 3) + 4 * (wave >> 1)) + (wave & 1);
    bring(s + wave * kPage, a.kc, page);
    bring(s + (kPages + wave) * kPage, a.vc, page);
  };
  // scores of tile u of a stage's K pages (key0: its first key), what a row does not see at -inf
  auto scores = [&](const char* s, int u, int key0, f32x16& sc) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 16; ++i) sc[i] = 0.f;
    // key r of the tile: token r & 15 of page r >> 4, channels in pieces of 8
    const char* kp = s + (2 * u + (r >> 4)) * kPage + (r & 15) * 16 + h * 256;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(kp + ks * 512), qf[ks], sc, 0, 0, 0);
    if (key0 + 32 > wave_first) {  // some row does not see all of the tile
      const int left = see - key0 - 4 * h;
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if ((i & 3) + 8 * (i >> 2) >= left) sc[i] = -INFINITY;
    }
  };
  auto max_of = [&](const f32x16& sc) __attribute__((always_inline)) {
    float top = sc[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) top = fmaxf(top, sc[i]);
    return top;
  };
  auto key_of = [&](int st, int u) { return (st >> 2) * kSplit + ((st & 3) + 4 * u) * 32; };
  auto find_max = [&](const char* s, int st) __attribute__((always_inline)) {
#pragma unroll 2   // (all four: 288 us for 278, registers in scratch)
    for (int u = 0; u < kKeys / 32; ++u)
      if (st * kKeys + u * 32 < wave_last) {
        f32x16 sc;
        scores(s, u, st * kKeys + u * 32, sc);
        top_split = fmaxf(top_split, max_of(sc));
      }
    if (kKeys == kSplit ? st * kKeys < kv_len : st & 1) {   // (the split's last stage)
      top_split = halves_max(top_split * a.scale_log2);  // (positive: rounding keeps the order, the maximum is that of the scaled scores)
      if (h == 0) split_max[st * kKeys / kSplit * kRows + m] = top_split;
      top_row = fmaxf(top_row, top_split);
      top_split = -INFINITY;
    }
  };
  auto attend = [&](const char* s, int st) __attribute__((always_inline)) {
    if ((st >> 2) * kSplit >= wave_last) return;  // nothing of the split for the wave's rows
    const float top_all = split_max[(st >> 2) * kRows + m];
    if (key_of(st, 0) < wave_last) {
      bf16x8 pf[TPC][2];
      float top = -INFINITY, l = 0.f, alpha = 1.f;
#pragma unroll
      for (int u = 0; u < TPC; ++u) {
        const int key0 = key_of(st, u);
        if (u > 0 && key0 >= wave_last) {  // (a tile nobody sees: factor 1, weights 0)
          const bf16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
          pf[u][0] = pf[u][1] = z;
          alpha = 1.f;
          continue;
        }
        f32x16 sc;
        scores(s, u, key0, sc);
        const float top_new = fmaxf(top, halves_max(max_of(sc) * a.scale_log2));
        const float use = top_new == -INFINITY ? 0.f : top_new;
        alpha = __builtin_amdgcn_exp2f(top - use);
        top = top_new;
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float p = __builtin_amdgcn_exp2f(sc[i] * a.scale_log2 - use);
          sum += p;
          pf[u][i >> 3][i & 7] = (bf16_t)p;
        }
        l = l * alpha + sum;
      }
      l = halves_sum(l);
      const float w = top_all == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(top - top_all);
      l_split += w * l;
      const bool rescale = TPC > 1 && __any(alpha != 1.f);  // (a factor of exactly 1 in every lane changes nothing)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        f32x16 o;
#pragma unroll
        for (int i = 0; i < 16; ++i) o[i] = 0.f;
#pragma unroll
        for (int u = 0; u < TPC; ++u) {
          if (u > 0 && rescale) {
#pragma unroll
            for (int i = 0; i < 16; ++i) o[i] *= alpha;
          }
#pragma unroll
          for (int p = 0; p < 2; ++p)
            o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                *reinterpret_cast<const bf16x8*>(s + (kPages + 2 * u + p) * kPage + (dt * 32 + r) * 32 + h * 16), pf[u][p],
                o, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) o_split[dt][i] += w * o[i];
      }
    }
    if ((st & 3) == 3) {
      const float f = __builtin_amdgcn_exp2f(top_all - top_row);
      l_row += f * l_split;
      l_split = 0.f;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          o_row[dt][i] += f * o_split[dt][i];
          o_split[dt][i] = 0.f;
        }
    }
  };
  // stage x (the first sweep's, then the second's) is in `cur` once this wave's loads have landed and every wave is here; then
  // nobody reads `nxt` any more
  auto step = [&](char* cur, char* nxt, int x, auto sweep) __attribute__((always_inline)) {
    constexpr bool kFirst = decltype(sweep)::value == 0;
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int y = x + 1;
    if (y < n_max + n_st) {  // (uniform)
      const bool keys = kFirst && y < n_max;
      const int first = keys ? y * kKeyPages : first_page(y - n_max), pages = keys ? kKeyPages : kSplitPages;
      if (first < table0 || first + pages > table0 + kTable) {
        fill_table(first);
        __syncthreads();
      }
      if (keys) load_keys(nxt, y);
      else load(nxt, y - n_max);
    }
    if constexpr (kFirst) find_max(cur, x);
    else attend(cur, x - n_max);
  };
  fill_table(0);
  __syncthreads();
  load_keys(s0, 0);
  // (an even number of stages in each sweep)
  for (int x = 0; x < n_max; x += 2) {
    step(s0, s1, x, std::integral_constant<int, 0>{});
    step(s1, s0, x + 1, std::integral_constant<int, 0>{});
  }
  for (int x = n_max; x < n_max + n_st; x += 2) {
    step(s0, s1, x, std::integral_constant<int, 1>{});
    step(s1, s0, x + 1, std::integral_constant<int, 1>{});
  }
  if (!valid) return;
  bf16_t* orow = a.out + (size_t)(row0 + t) * a.ldo + (size_t)(kvh * G + g) * D;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      bf16x4 v;
#pragma unroll
      for (int c = 0; c < 4; ++c) v[c] = (bf16_t)(l_row > 0.f ? o_row[dt][4 * j + c] / l_row : 0.f);
      *reinterpret_cast<bf16x4*>(orow + dt * 32 + 8 * j + 4 * h) = v;
    }
}

template <int D, int TPC>
int launch_prompt_attn(const PromptAttnArgs& a, int n_items, int max_ctx, hipStream_t st) {
  static std::once_flag once;
  static hipError_t err = hipSuccess;
  std::call_once(once, [] {
    err = hipFuncSetAttribute(reinterpret_cast<const void*>(prompt_attn_kernel<D, TPC>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, 88 * 1024);
  });
  SD_REQUIRE(err == hipSuccess, SD_ERR_HIP, "sd_prompt_attention: hipFuncSetAttribute failed: %s", hipGetErrorString(err));
  const size_t lds = (size_t)((max_ctx + 128 * TPC - 1) / (128 * TPC)) * kRows * sizeof(float);
  SD_REQUIRE(lds <= 88 * 1024, SD_ERR_UNSUPPORTED, "sd_prompt_attention: max_ctx %d with splits of %d keys", max_ctx, 128 * TPC);
  hipLaunchKernelGGL((prompt_attn_kernel<D, TPC>), dim3(a.Hkv, n_items), dim3(256), lds, st, a);
  SD_CHECK_LAUNCH("sd_prompt_attention");
  return SD_OK;
}

}  // namespace

extern "C" int sd_prompt_attention(const void* q, int64_t ldq, const void* k_cache, const void* v_cache,
                                   const int32_t* block_tables, int max_blocks_per_seq, const int32_t* items, int n_items,
                                   void* out, int64_t ldo, int Hq, int Hkv, int D, float scale, int max_ctx,
                                   int split_tokens, sd_stream_t stream) {
  SD_REQUIRE(q && k_cache && v_cache && block_tables && items && out, SD_ERR_INVALID, "sd_prompt_attention: null pointer");
  SD_REQUIRE(Hq >= 1 && Hkv >= 1 && Hq % Hkv == 0 && Hq / Hkv <= SD_PROMPT_BLOCK_ROWS && (D == 64 || D == 128),
             SD_ERR_UNSUPPORTED, "sd_prompt_attention: %d query heads over %d of size %d", Hq, Hkv, D);
  SD_REQUIRE(n_items >= 0 && n_items <= 65535 && max_blocks_per_seq >= 1 && scale > 0.f && ldq % 8 == 0 && ldo % 4 == 0 &&
                 ldq >= (int64_t)Hq * D && ldo >= (int64_t)Hq * D && sd_aligned16(q) && sd_aligned16(items) &&
                 sd_aligned16(k_cache) && sd_aligned16(v_cache) && (reinterpret_cast<uintptr_t>(out) & 7) == 0,
             SD_ERR_INVALID, "sd_prompt_attention: bad arguments (%d items, ldq %lld, ldo %lld)", n_items, (long long)ldq,
             (long long)ldo);
  // (other splits' chains are longer than the two tiles whose sums fit beside the others: sd_paged_attention takes them)
  SD_REQUIRE((split_tokens == 128 || split_tokens == 256) && max_ctx >= 1, SD_ERR_UNSUPPORTED,
             "sd_prompt_attention: splits of %d keys (128 or 256), max_ctx %d", split_tokens, max_ctx);
  if (n_items == 0) return SD_OK;
  PromptAttnArgs a{(const bf16_t*)q, ldq, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables, max_blocks_per_seq,
                   items, (bf16_t*)out, ldo, Hq, Hkv, scale * 1.44269504088896340736f};
  hipStream_t st = (hipStream_t)stream;
  if (D == 64) return split_tokens == 128 ? launch_prompt_attn<64, 1>(a, n_items, max_ctx, st)
                                          : launch_prompt_attn<64, 2>(a, n_items, max_ctx, st);
  return split_tokens == 128 ? launch_prompt_attn<128, 1>(a, n_items, max_ctx, st)
                             : launch_prompt_attn<128, 2>(a, n_items, max_ctx, st);
}

// Attention whose heads exchange their softmax weights, for portions of a prompt in bfloat16 (`attention_talk.hip` states
// the formula and serves decoded tokens, float32 and every other size), with no table of scores and the mixed weights alone in
// memory:
//
//   1. `talk_tile_stats_kernel`: a block of eight wavefronts a (32 rows, key/value head, heads of its group) walks the keys
//      once and leaves every (row, head)'s maximum and the inverse of its normaliser, the sink included;
//   2. `talk_tile_mix_kernel`: a block of eight wavefronts has 32 rows (16 of more than 16 heads), ALL heads and some steps of 32
//      keys.  A wavefront makes the finished float32 weights of its own heads (their scores on the matrix cores again) and puts
//      them into LDS, the block mixes them there (talk [H, H] times the weights [H, pairs of row and key] on the float32
//      matrix instruction, v_mfma_f32_16x16x4_f32) and writes them in bfloat16;
//   3. `talk_tile_values_kernel`: a block of four wavefronts a (rows, key/value head, heads of its group) adds weights times
//      values over all keys; a wavefront takes every fourth step, the four sums are added in their order.
// Keys and values are read from the pages as they lie there, [slot][dim] and [slot / 8][dim][slot % 8], straight into
// registers as the matrix instruction's operands.  Blocks of one key/value head are eight apart where there are eight, so
// that each XCD's L2 holds its own.
//
// A prompt of 1,500 tokens, 16 heads of 128 on 8, us: statistics 24, weights 35, values 18, where the score table in memory between a library's
// products took 213.  The weights' kernel is bound by its vector instructions and the float32 matrix instructions (2.9 of 3.7 us a step of
// 32 x 32; 16 of the mixing product's 128 cycles a pair tile would be bfloat16's, but weights stay float32 until they are mixed).  All in one
// kernel, the outputs kept in registers, took 59 to 87 with 10 for the sum of cut ranges: with them there is room for 16 rows only, and a
// compute unit then reads 128 KB of keys and values a step at about 50 GB/s.
#include "common.h"
#include <algorithm>
#include <type_traits>

CWM_DEFINE_ERROR_API

#define TILE_KEYS 32      // keys of a step
#define STATS_ROWS 32     // rows of a block of the first kernel
#define TILE_WAVES 8      // of the first two
#define VALUE_WAVES 4
#define TILE_PORTIONS 16  // portions of one launch
#define LOG2E 1.4426950408889634f

// A portion: tokens t0 .. t0 + n - 1 of the step, positions pos0 .. of sequence `seq`, of which this launch takes rows r0 .. r1 - 1
// (r0 a multiple of 32).  `table`: its mixed weights, [head][row - r0][column], `columns` of a row: column i of a row is the key i
// after the first that the row's tile of 32 rows reads, rounded down to a step.  `at`: its first block of each kernel.
struct TalkPortion {
  int seq, t0, n, pos0, r0, r1, columns, at[3];
  long table;
};
struct TalkPortions {
  int count;
  TalkPortion of[TILE_PORTIONS];
};

struct TalkTileArgs {
  const bf16_t* q;
  long q_stride;
  const bf16_t* cache;
  const int* block_table;
  int table_width, n_q_heads, n_kv_heads, page_size, page_shift, num_pages, window_left;  // page_shift: -1 where the page is no power of two
  float scale_log2e;
};

__device__ __forceinline__ const TalkPortion& portion_of(const TalkPortions& P, int kernel) {
  int i = 0;
  while (i + 1 < P.count && (int)blockIdx.x >= P.of[i + 1].at[kernel]) ++i;
  return P.of[i];
}
__device__ __forceinline__ int page_number(const TalkTileArgs& A, int key) { return A.page_shift >= 0 ? key >> A.page_shift : key / A.page_size; }
__device__ __forceinline__ int first_key(const TalkTileArgs& A, int p) { return A.window_left >= 0 ? max(0, p - A.window_left) : 0; }
// the first key of a row's table: of its tile of 32 rows
__device__ __forceinline__ int table_base(const TalkTileArgs& A, const TalkPortion& po, int row) { return first_key(A, po.pos0 + (row & ~31)) & ~(TILE_KEYS - 1); }

// the page of the 32 keys from `kt` on (pages hold a multiple of 32 keys); a page that is not there, in the table or behind its end: page 0
__device__ __forceinline__ int tile_page(const int* table, const TalkTileArgs& A, int kt, int& slot, bool* there = nullptr) {
  const int lp = page_number(A, kt);
  slot = kt - lp * A.page_size;
  const int page = lp < A.table_width ? table[lp] : -1;
  const bool known = (unsigned)page < (unsigned)A.num_pages;
  if (there) *there = known;
  return known ? page : 0;
}
// the same of one thread's own range
__device__ __forceinline__ bool row_lacks_page(const int* table, const TalkTileArgs& A, int first, int last) {
  for (int lp = page_number(A, first); lp <= page_number(A, last); ++lp)
    if (lp >= A.table_width || (unsigned)table[lp] >= (unsigned)A.num_pages) return true;
  return false;
}
// whether a key of [first, last] lies in a page that is not there, of a wavefront's range
__device__ __forceinline__ bool lacks_page(const int* table, const TalkTileArgs& A, int first, int last) {
  bool bad = false;
  for (int lp = page_number(A, first) + (int)(threadIdx.x & 63); lp <= page_number(A, last); lp += 64) {
    const int page = lp < A.table_width ? table[lp] : -1;
    bad = bad || (unsigned)page >= (unsigned)A.num_pages;
  }
  return __any(bad);
}

// ---- maxima and normalisers ------------------------------------------------------------------------------------------ //
// stats: [token][head][2], the maximum of the scores times log2 e and 1 / the sum of 2^(score - maximum).
// A wavefront takes every eighth tile of 32 keys for 32 rows and HEADS heads, which share the keys' operands.
template <int HD, int HEADS>
__global__ void __launch_bounds__(64 * TILE_WAVES, 2)
talk_tile_stats_kernel(TalkTileArgs A, TalkPortions P, float* __restrict__ stats, const float* __restrict__ sink) {
  constexpr int KS = HD / 32;
  const TalkPortion& po = portion_of(P, 0);
  const int per = A.n_q_heads / A.n_kv_heads, parts = (per + HEADS - 1) / HEADS, groups = A.n_kv_heads * parts;
  const int block = blockIdx.x - po.at[0], tiles = (po.r1 - po.r0 + STATS_ROWS - 1) / STATS_ROWS;
  const int row0 = po.r0 + (tiles - 1 - block / groups) * STATS_ROWS;  // the rows with most keys start first
  const int c = block % A.n_kv_heads, g0 = block % groups / A.n_kv_heads * HEADS;
  const int lane = threadIdx.x & 63, n = lane & 15, j = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int* table = A.block_table + (size_t)po.seq * A.table_width;
  const float none = -__builtin_inff();

  int p[2], first[2];
  Frag8 qf[2][HEADS][KS];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int r = min(row0 + 16 * u + n, po.n - 1);  // rows past the last are the last again
    p[u] = po.pos0 + r;
    first[u] = first_key(A, p[u]);
#pragma unroll
    for (int g = 0; g < HEADS; ++g) {
      const bf16_t* row = A.q + (size_t)(po.t0 + r) * A.q_stride + (size_t)(c * per + min(g0 + g, per - 1)) * HD + 8 * j;
#pragma unroll
      for (int s = 0; s < KS; ++s) qf[u][g][s].u = *(const uint4*)(row + 32 * s);
    }
  }
  const int p_first = po.pos0 + row0, p_last = po.pos0 + min(row0 + STATS_ROWS, po.n) - 1;
  const int lo = first_key(A, p_first);
  const int lo_all = first_key(A, p_last);  // from here to p_first every row reads every key
  const size_t plane = (size_t)A.n_kv_heads * A.page_size * HD;
  const bf16_t* keys = A.cache + (size_t)c * A.page_size * HD + (size_t)n * HD + 8 * j;

  auto load = [&](Frag8 (&kf)[2][KS], int kt) {
    int slot;
    const int page = tile_page(table, A, kt, slot);
    const bf16_t* from = keys + (size_t)page * 2 * plane + (size_t)slot * HD;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int s = 0; s < KS; ++s) kf[t][s].u = *(const uint4*)(from + (size_t)t * 16 * HD + 32 * s);
  };
  float m[2][HEADS], l[2][HEADS];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int g = 0; g < HEADS; ++g) m[u][g] = none, l[u][g] = 0.f;

  const int step = TILE_KEYS * TILE_WAVES;
  Frag8 kf[2][KS], next[2][KS];
  int kt = lo - lo % TILE_KEYS + TILE_KEYS * wave;
  if (kt <= p_last) load(kf, kt);
  for (; kt <= p_last; kt += step) {
    load(next, min(kt + step, p_last - p_last % TILE_KEYS));
    const bool edge = kt + TILE_KEYS - 1 > p_first || kt < lo_all;
#pragma unroll
    for (int g = 0; g < HEADS; ++g)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float s[8];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          float4v a = (float4v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int d = 0; d < KS; ++d) a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][d].v, qf[u][g][d].v, a, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) s[4 * t + e] = a[e];
        }
        if (edge) {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int key = kt + 16 * (e >> 2) + 4 * j + (e & 3);
            s[e] = key >= first[u] && key <= p[u] ? s[e] : none;
          }
        }
        float top = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
        if (__any(top > m[u][g])) {
          top = fmaxf(top, m[u][g]);
          if (top > m[u][g]) l[u][g] *= __builtin_amdgcn_exp2f((m[u][g] - top) * A.scale_log2e);
          m[u][g] = top;
        }
        const float minus = m[u][g] == none ? 0.f : -m[u][g] * A.scale_log2e;  // nothing yet: every term is 2^-inf, or NaN
#pragma unroll
        for (int e = 0; e < 8; ++e) l[u][g] += __builtin_amdgcn_exp2f(fmaf(s[e], A.scale_log2e, minus));
      }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int s = 0; s < KS; ++s) kf[t][s] = next[t][s];
  }
  // the four lanes of a row, then the wavefronts
  __shared__ float all_m[TILE_WAVES][HEADS][STATS_ROWS], all_l[TILE_WAVES][HEADS][STATS_ROWS];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int g = 0; g < HEADS; ++g) {
      float top = fmaxf(m[u][g], __shfl_xor(m[u][g], 16, 64));
      top = fmaxf(top, __shfl_xor(top, 32, 64));
      float sum = m[u][g] == none ? l[u][g] : l[u][g] * __builtin_amdgcn_exp2f((m[u][g] - top) * A.scale_log2e);
      sum += __shfl_xor(sum, 16, 64);
      sum += __shfl_xor(sum, 32, 64);
      if (j == 0) all_m[wave][g][16 * u + n] = top, all_l[wave][g][16 * u + n] = sum;
    }
  __syncthreads();
  for (int e = threadIdx.x; e < HEADS * STATS_ROWS; e += 64 * TILE_WAVES) {
    const int g = e / STATS_ROWS, r = e % STATS_ROWS;
    if (g0 + g >= per || row0 + r >= po.n) continue;
    const int h = c * per + g0 + g;
    float top = all_m[0][g][r], sum = 0.f;
#pragma unroll
    for (int w = 1; w < TILE_WAVES; ++w) top = fmaxf(top, all_m[w][g][r]);
    float top2 = top * A.scale_log2e;
    if (sink) top2 = fmaxf(top2, sink[h] * LOG2E);
#pragma unroll
    for (int w = 0; w < TILE_WAVES; ++w) {
      const float mw = all_m[w][g][r];
      sum += mw == none ? all_l[w][g][r] : all_l[w][g][r] * __builtin_amdgcn_exp2f(fmaf(mw, A.scale_log2e, -top2));
    }
    if (sink) sum += __builtin_amdgcn_exp2f(fmaf(sink[h], LOG2E, -top2));
    float* to = stats + ((size_t)(po.t0 + row0 + r) * A.n_q_heads + h) * 2;
    to[0] = top2, to[1] = 1.0f / sum;
  }
}

// ---- weights and their mixture ---------------------------------------------------------------------------------------- //
// SLOTS: heads the block has room for (8, 16 or 32); HPW: heads a wavefront has, all of one key/value head; RT: row tiles of 16.
// `steps`: of a block.
template <int HD, int SLOTS, int HPW, int RT>
__global__ void __launch_bounds__(64 * TILE_WAVES, 2)
talk_tile_mix_kernel(TalkTileArgs A, TalkPortions P, const float* __restrict__ stats, const float* __restrict__ talk, bf16_t* __restrict__ weights, int steps) {
  constexpr int KS = HD / 32, MT = (SLOTS + 15) / 16, GS = SLOTS / 4, ROWS = 16 * RT;
  constexpr int PROB = TILE_KEYS + 4;  // a row's elements in LDS: neighbouring rows start four banks further
  __shared__ __attribute__((aligned(16))) float prob[2][SLOTS][ROWS][PROB];
  __shared__ float mix[MT][GS][64];
  const TalkPortion& po = portion_of(P, 1);
  const int tiles = (po.r1 - po.r0 + ROWS - 1) / ROWS, block = blockIdx.x - po.at[1];
  const int row0 = po.r0 + (tiles - 1 - block % tiles) * ROWS;  // blocks of the same keys follow one another
  const int p_first = po.pos0 + row0, p_last = po.pos0 + min(row0 + ROWS, po.n) - 1;
  const int base = table_base(A, po, row0), lo_all = first_key(A, p_last);
  const int begin = (first_key(A, p_first) & ~(TILE_KEYS - 1)) + block / tiles * steps * TILE_KEYS, end = min(p_last + 1, begin + steps * TILE_KEYS);
  if (begin >= end) return;

  const int lane = threadIdx.x & 63, n = lane & 15, j = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int H = A.n_q_heads, per = H / A.n_kv_heads, side = TILE_WAVES / A.n_kv_heads;  // side: wavefronts of a key/value head
  const int c = wave / side, g0 = wave % side * HPW;
  const int mine = c < A.n_kv_heads ? min(HPW, per - g0) : 0;  // heads of this wavefront; it may have none and only mixes
  const int h0 = c * per + g0;
  const int* table = A.block_table + (size_t)po.seq * A.table_width;

  const size_t plane = (size_t)A.n_kv_heads * A.page_size * HD;
  const bf16_t* keys = A.cache + (size_t)min(c, A.n_kv_heads - 1) * A.page_size * HD + (size_t)n * HD + 8 * j;
  Frag8 kf[2][KS];
  auto load_keys = [&](int kt) {
    int slot;
    const int page = tile_page(table, A, kt, slot);
    const bf16_t* from = keys + (size_t)page * 2 * plane + (size_t)slot * HD;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int s = 0; s < KS; ++s) kf[t][s].u = *(const uint4*)(from + (size_t)t * 16 * HD + 32 * s);
  };
  load_keys(begin);

  int p[RT], first[RT];
  Frag8 qf[RT][HPW][KS];
  float top[RT][HPW], inverse[RT][HPW];
#pragma unroll
  for (int u = 0; u < RT; ++u) {
    const int r = min(row0 + 16 * u + n, po.n - 1);  // rows past the last are the last again
    p[u] = po.pos0 + r, first[u] = first_key(A, p[u]);
#pragma unroll
    for (int g = 0; g < HPW; ++g) {
      const int h = min(h0 + min(g, max(mine, 1) - 1), H - 1);
      const bf16_t* row = A.q + (size_t)(po.t0 + r) * A.q_stride + (size_t)h * HD + 8 * j;
#pragma unroll
      for (int s = 0; s < KS; ++s) qf[u][g][s].u = *(const uint4*)(row + 32 * s);
      const float* st = stats + ((size_t)(po.t0 + r) * H + h) * 2;
      top[u][g] = -st[0], inverse[u][g] = st[1];
    }
  }
  // the mixing matrix as left operands: row h = 16 mt + n, column 4 s + j; zeros beyond the heads
  if (wave == 0)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int s = 0; s < GS; ++s) {
        const int h = 16 * mt + n, g = 4 * s + j;
        mix[mt][s][lane] = h < H && g < H ? talk[(size_t)h * H + g] : 0.f;
      }
  // the weights of heads that are not there stay zero
#pragma unroll
  for (int b = 0; b < 2; ++b)
    for (int e = threadIdx.x; e < (SLOTS - H) * ROWS * PROB; e += 64 * TILE_WAVES) (&prob[b][H][0][0])[e] = 0.f;

  const size_t head_stride = (size_t)(po.r1 - po.r0) * po.columns;
  bf16_t* to = weights + po.table + (size_t)(row0 - po.r0) * po.columns - base;
  int b = 0;
  for (int kt = begin; kt < end; kt += TILE_KEYS, b ^= 1) {
    const bool edge = kt + TILE_KEYS - 1 > p_first || kt < lo_all;
    float4v s[RT][HPW][2];
#pragma unroll
    for (int u = 0; u < RT; ++u)
#pragma unroll
      for (int g = 0; g < HPW; ++g)
#pragma unroll
        for (int t = 0; t < 2; ++t) s[u][g][t] = (float4v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < KS; ++d)
#pragma unroll
      for (int u = 0; u < RT; ++u)
#pragma unroll
        for (int g = 0; g < HPW; ++g) {
          if (g >= mine) continue;
#pragma unroll
          for (int t = 0; t < 2; ++t) s[u][g][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][d].v, qf[u][g][d].v, s[u][g][t], 0, 0, 0);
        }
    load_keys(min(kt + TILE_KEYS, (end - 1) & ~(TILE_KEYS - 1)));  // under way while the weights are made and mixed
#pragma unroll
    for (int u = 0; u < RT; ++u)
#pragma unroll
      for (int g = 0; g < HPW; ++g) {
        if (g >= mine) continue;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          float w[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = __builtin_amdgcn_exp2f(fmaf(s[u][g][t][e], A.scale_log2e, top[u][g])) * inverse[u][g];
          if (edge) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int key = kt + 16 * t + 4 * j + e;
              w[e] = key >= first[u] && key <= p[u] ? w[e] : 0.f;
            }
          }
          *(float4*)&prob[b][h0 + g][16 * u + n][16 * t + 4 * j] = make_float4(w[0], w[1], w[2], w[3]);
        }
      }
    __syncthreads();  // and everyone has left the other buffer
    // 64 pairs of two rows a time: lane n of each quarter has four keys of one row
#pragma unroll
    for (int u = 0; u < RT; ++u) {
      const int row = 16 * u + 2 * wave + (n >> 3), key = 4 * (n & 7);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        float4v sum[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] = (float4v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < GS; ++i) {
          const float4v w = *(const float4v*)&prob[b][4 * i + j][row][key];
          const float t = mix[mt][i][lane];
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(t, w[e], sum[e], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int h = 16 * mt + 4 * j + i;
          if (h < H && row0 + row < po.r1)
            *(uint2*)(to + h * head_stride + (size_t)row * po.columns + kt + key) = make_uint2(pack2_bf16(sum[0][i], sum[1][i]), pack2_bf16(sum[2][i], sum[3][i]));
        }
      }
    }
  }
}

// ---- values ------------------------------------------------------------------------------------------------------------ //
// A row of a tile has weight zero for the tile's keys that it does not read, and zero times an infinity or a NaN is a NaN.  So a block with a
// result that is not finite, or a missing page, goes over its keys once more.  Keys that a row does not read lie in the steps at the tile's two
// ends alone (`TileEnds`): there values that are not finite, and all of a missing page, are zeros to the matrix instruction then, and a row's own
// products with the former are added to its sums.  An infinite or NaN value reaches its readers only, whatever rows lie beside them, and every
// other result has the bits that it has without; rows that read a missing page are NaN, the others are not.
struct TileEnds {
  int lo, lo_all, p_first, p_last;  // the first key that any row reads; from lo_all to p_first every row reads every key; the last key
  __device__ __forceinline__ bool of(int kt) const { return kt < lo_all || kt + TILE_KEYS - 1 > p_first; }
};
__device__ __forceinline__ bool not_finite(uint32_t half) { return (half & 0x7f80u) == 0x7f80u; }
__device__ __forceinline__ uint32_t finite_only(uint32_t two) {
  return (not_finite(two) ? 0u : two & 0x0000ffffu) | (not_finite(two >> 16) ? 0u : two & 0xffff0000u);
}
// a row's products of the tile's ends with values that are not finite, onto `sum`, four dims from d on
__device__ __forceinline__ float4v add_not_finite(const TalkTileArgs& A, const TileEnds& ends, const int* table, const bf16_t* weights, const bf16_t* values,
                                                  size_t page_stride, int head_dim, int d, int first, int p, float4v sum) {
  for (int kt = ends.lo & ~(TILE_KEYS - 1); kt <= p; kt += TILE_KEYS) {
    if (!ends.of(kt)) {
      kt = max(kt, (ends.p_first & ~(TILE_KEYS - 1)) - TILE_KEYS);
      continue;
    }
    int slot;
    bool there;
    const bf16_t* from = values + (size_t)tile_page(table, A, kt, slot, &there) * page_stride;
    if (!there) continue;
    for (int key = max(kt, first); key <= min(kt + TILE_KEYS - 1, p); ++key) {
      const int s = slot + key - kt;
      const bf16_t* v = from + ((size_t)(s / 8) * head_dim + d) * 8 + s % 8;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (not_finite(v[8 * i])) sum[i] = fmaf(bf16_to_f32(weights[key]), bf16_to_f32(v[8 * i]), sum[i]);
    }
  }
  return sum;
}

// HEADS: heads of a block, which share the values' operands.
template <int HD, int HEADS, int RT>
__global__ void __launch_bounds__(64 * VALUE_WAVES, 2)
talk_tile_values_kernel(TalkTileArgs A, TalkPortions P, const bf16_t* __restrict__ weights, bf16_t* __restrict__ out) {
  constexpr int DT = HD / 16, ROWS = 16 * RT;
  __shared__ __attribute__((aligned(16))) float sums[VALUE_WAVES][HEADS][16][HD + 4];
  const TalkPortion& po = portion_of(P, 2);
  const int per = A.n_q_heads / A.n_kv_heads, groups = A.n_kv_heads * ((per + HEADS - 1) / HEADS);
  const int block = blockIdx.x - po.at[2], tiles = (po.r1 - po.r0 + ROWS - 1) / ROWS;
  const int row0 = po.r0 + (tiles - 1 - block / groups) * ROWS;  // the rows with most keys start first
  const int c = block % A.n_kv_heads, g0 = block % groups / A.n_kv_heads * HEADS;
  const int lane = threadIdx.x & 63, n = lane & 15, j = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int* table = A.block_table + (size_t)po.seq * A.table_width;
  const int p_last = po.pos0 + min(row0 + ROWS, po.r1) - 1, lo = first_key(A, po.pos0 + row0), base = table_base(A, po, row0);
  const TileEnds ends = {lo, first_key(A, p_last), po.pos0 + row0, p_last};

  const bf16_t* from_w[RT][HEADS];
#pragma unroll
  for (int u = 0; u < RT; ++u)
#pragma unroll
    for (int g = 0; g < HEADS; ++g)
      from_w[u][g] = weights + po.table + ((size_t)(c * per + min(g0 + g, per - 1)) * (po.r1 - po.r0) + min(row0 + 16 * u + n, po.r1 - 1) - po.r0) * po.columns - base + 8 * j;
  const size_t plane = (size_t)A.n_kv_heads * A.page_size * HD;
  const bf16_t* values = A.cache + plane + (size_t)c * A.page_size * HD + (size_t)n * 8;

  Frag8 vf[DT], wf[RT][HEADS];
  bool there;
  auto load = [&](int kt) {
    int slot;
    const int page = tile_page(table, A, kt, slot, &there);
    const bf16_t* from = values + (size_t)page * 2 * plane + (size_t)(slot / 8 + j) * HD * 8;
#pragma unroll
    for (int u = 0; u < RT; ++u)
#pragma unroll
      for (int g = 0; g < HEADS; ++g) wf[u][g].u = *(const uint4*)(from_w[u][g] + kt);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) vf[dt].u = *(const uint4*)(from + dt * 16 * 8);
  };
  // whether all is finite and no page missing
  auto pass = [&](auto once_more) {
    constexpr bool again = decltype(once_more)::value;
    float4v acc[RT][HEADS][DT];
#pragma unroll
    for (int u = 0; u < RT; ++u)
#pragma unroll
      for (int g = 0; g < HEADS; ++g)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[u][g][dt] = (float4v){0.f, 0.f, 0.f, 0.f};
    for (int kt = (lo & ~(TILE_KEYS - 1)) + TILE_KEYS * wave; kt <= p_last; kt += TILE_KEYS * VALUE_WAVES) {
      load(kt);
      if (kt < lo || kt + TILE_KEYS - 1 > p_last) {  // values that no row reads may be anything
        uint32_t keep[4] = {0xffffffffu, 0xffffffffu, 0xffffffffu, 0xffffffffu};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int key = kt + 8 * j + e;
          if (key < lo || key > p_last) keep[e >> 1] &= (e & 1) ? 0x0000ffffu : 0xffff0000u;
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) vf[dt].u.x &= keep[0], vf[dt].u.y &= keep[1], vf[dt].u.z &= keep[2], vf[dt].u.w &= keep[3];
      }
      if (again && ends.of(kt)) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          vf[dt].u = there ? make_uint4(finite_only(vf[dt].u.x), finite_only(vf[dt].u.y), finite_only(vf[dt].u.z), finite_only(vf[dt].u.w)) : make_uint4(0u, 0u, 0u, 0u);
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int u = 0; u < RT; ++u)
#pragma unroll
          for (int g = 0; g < HEADS; ++g) acc[u][g][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dt].v, wf[u][g].v, acc[u][g][dt], 0, 0, 0);
    }
    // lane 16 j + n holds row n, dims 16 dt + 4 j + i
    const bool missing = lacks_page(table, A, lo, p_last);
    bool plain = !missing;
#pragma unroll
    for (int u = 0; u < RT; ++u) {
      if (u > 0) __syncthreads();
#pragma unroll
      for (int g = 0; g < HEADS; ++g)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) *(float4v*)&sums[wave][g][n][16 * dt + 4 * j] = acc[u][g][dt];
      __syncthreads();
      for (int e = threadIdx.x; e < HEADS * 16 * (HD / 4); e += 64 * VALUE_WAVES) {
        const int d = e % (HD / 4) * 4, g = e / (HD / 4) % HEADS, r = e / (HD / 4) / HEADS, row = row0 + 16 * u + r;
        if (g0 + g >= per || row >= po.r1) continue;
        float4v v = *(const float4v*)&sums[0][g][r][d];
#pragma unroll
        for (int w = 1; w < VALUE_WAVES; ++w) v += *(const float4v*)&sums[w][g][r][d];
        plain = plain && fabsf(v[0]) + fabsf(v[1]) + fabsf(v[2]) + fabsf(v[3]) < __builtin_inff();
        if constexpr (again) {
          const int p = po.pos0 + row, first = first_key(A, p);
          const float nan = __uint_as_float(0x7fc00000u);
          const bf16_t* w = weights + po.table + ((size_t)(c * per + g0 + g) * (po.r1 - po.r0) + row - po.r0) * po.columns - base;
          if (missing && row_lacks_page(table, A, first, p)) v = (float4v){nan, nan, nan, nan};
          else v = add_not_finite(A, ends, table, w, A.cache + plane + (size_t)c * A.page_size * HD, 2 * plane, HD, d, first, p, v);
        }
        *(uint2*)(out + (size_t)(po.t0 + row) * A.n_q_heads * HD + (size_t)(c * per + g0 + g) * HD + d) = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
      }
    }
    return plain;
  };
  if (__builtin_expect(__syncthreads_and(pass(std::false_type())), 1)) return;
  pass(std::true_type());
}

// ---- entry points ---------------------------------------------------------------------------------------------------- //
// heads a wavefront of the second kernel has, or 0: sizes it has no room for
extern "C" int cwm_talking_tile_heads(int n_q_heads, int n_kv_heads, int head_dim) {
  if (n_q_heads < 1 || n_q_heads > 32 || n_kv_heads < 1 || n_kv_heads > TILE_WAVES || n_q_heads % n_kv_heads != 0) return 0;
  if (head_dim != 64 && head_dim != 128) return 0;
  const int side = TILE_WAVES / n_kv_heads, each = (n_q_heads / n_kv_heads + side - 1) / side;
  return each <= 4 ? each : 0;
}
// steps of keys that a tile of the second kernel reads
static int tile_steps(const TalkPortion& po, int row0, int rows, int window_left) {
  const int first = po.pos0 + row0, last = po.pos0 + (row0 + rows < po.n ? row0 + rows : po.n) - 1;
  return last / TILE_KEYS - (window_left >= 0 && first > window_left ? first - window_left : 0) / TILE_KEYS + 1;
}
// heads of a block of the first and the third kernel
static int tile_heads_together(int per) { return per <= 4 ? per : per % 3 == 0 ? 3 : 4; }
// blocks of those kernels for a tile of rows; 0: sizes there are no kernels for
extern "C" int cwm_talking_tile_groups(int n_q_heads, int n_kv_heads, int head_dim) {
  if (cwm_talking_tile_heads(n_q_heads, n_kv_heads, head_dim) == 0) return 0;
  const int per = n_q_heads / n_kv_heads, together = tile_heads_together(per);
  return n_kv_heads * ((per + together - 1) / together);
}
extern "C" int cwm_talking_tile_portions() { return TILE_PORTIONS; }

// Steps of a block of the second kernel.  No sum goes from one step to the next, so they may be cut anywhere: where the rounds of blocks take
// least, a block costing 7 us and 3.7 a step.  A compute unit has room for one block (148 KB of LDS).  A round is counted in two ways, and the
// larger number holds: as 224 blocks, since not all of 256 units are had at once, and as the fullest of 32 lots of 8 units, which a launch's blocks are
// dealt to in turn: tiles whose number is a multiple of 32 leave the rows with most keys in few lots.  Up to 8 heads (74 KB) two blocks share a
// unit beyond 192 blocks, which makes a round of twice as many 1.6 times as long.  us by steps: 16 heads of 128, 1,500 tokens 91 (4), 78 (6), 85 (8),
// 100 (12) and 174 (32); 2,048, whose 221 blocks of 11 steps leave 9 in a lot, 145 (11), 117 (13); 8 heads, 1,500 tokens 65 (3), 77 (6), 69 (8).  Over 88
// portions of 8 to 32 heads of 64 and 128, 64 to 4,096 tokens, the choice is within 8% of the best of all steps, 1.1% in the mean; without the lots
// and the second block within 30% and 3.4%.
#define MIX_LOTS 32
static int mix_steps(const TalkPortions& P, int count, int mix_rows, int n_q_heads, int window_left) {
  const int room = n_q_heads <= 8 ? 2 : 1;
  int best = 2;
  float least = 0.f;
  for (int steps = 2; steps <= 32; ++steps) {
    long blocks = 0, at = 0;
    int lots[MIX_LOTS] = {}, fullest = 0;
    for (int i = 0; i < count; ++i) {
      const TalkPortion& po = P.of[i];
      const int tiles = (po.r1 - po.r0 + mix_rows - 1) / mix_rows;
      int most = 0;
      for (int tile = 0; tile < tiles; ++tile) {
        const int cuts = (tile_steps(po, po.r0 + tile * mix_rows, mix_rows, window_left) + steps - 1) / steps;
        blocks += cuts, most = cuts > most ? cuts : most;
        if (blocks > 4 * 224 * room) continue;  // (many rounds even out, and are not worth the counting)
        for (int cut = 0; cut < cuts; ++cut) fullest = std::max(fullest, ++lots[(at + (long)cut * tiles + tiles - 1 - tile) % MIX_LOTS]);
      }
      at += (long)tiles * most;
    }
    if (blocks > 4 * 224 * room) fullest = 0;
    const bool alone = room == 1 || (blocks <= 192 && fullest <= 8);
    const long rounds = std::max((blocks + 224 * room - 1) / (224 * room), (long)(fullest + 8 * room - 1) / (8 * room));
    const float us = (float)rounds * (7.f + 3.7f * steps) * (alone ? 1.f : 1.6f);
    if (steps == 2 || us < least) best = steps, least = us;
  }
  return best;
}
static int tile_mix_rows(int n_q_heads) { return n_q_heads <= 16 ? 32 : 16; }
// the steps of a launch that takes `n` tokens after `pos0` whole
extern "C" int cwm_talking_tile_steps(int n, int pos0, int n_q_heads, int window_left) {
  TalkPortions P = {};
  P.count = 1, P.of[0].n = P.of[0].r1 = n, P.of[0].pos0 = pos0;
  return mix_steps(P, 1, tile_mix_rows(n_q_heads), n_q_heads, window_left);
}

// `portions`: for every portion sequence, first token, tokens, position of the first, the rows that this launch takes (from a multiple
// of 32 on, and their end) and the columns of their table (a multiple of 32 that holds the keys of every tile of 32 rows): seven ints,
// `count` of them.  q: bfloat16 [T, H, hd], tokens q_stride apart, 16-byte aligned.  cache, block_table as `cwm_talking_attention`, pages
// of a multiple of 32 keys.  stats: float32 [T, H, 2] scratch; weights: bfloat16 scratch, heads * rows * columns of every portion, one after
// the other.  out: bfloat16 [T, H * hd].
extern "C" int cwm_talking_tiles(const void* q, long q_stride, const void* cache, const int* block_table, int table_width, const int* portions,
                                 int count, int n_q_heads, int n_kv_heads, int head_dim, int page_size, int num_pages, int window_left,
                                 float scale, const float* sink, const float* talk, float* stats, void* weights, void* out, hipStream_t stream) {
  const int each = cwm_talking_tile_heads(n_q_heads, n_kv_heads, head_dim);
  CWM_REQUIRE(each > 0, "talking_tiles: no kernel for %d heads of %d on %d", n_q_heads, head_dim, n_kv_heads);
  CWM_REQUIRE(count >= 1 && count <= TILE_PORTIONS && portions, "talking_tiles: %d portions in a launch", count);
  CWM_REQUIRE(page_size > 0 && page_size % TILE_KEYS == 0 && num_pages > 0 && table_width > 0, "talking_tiles: bad cache sizes");
  CWM_REQUIRE(q && cache && block_table && talk && stats && weights && out, "talking_tiles: arguments missing");
  CWM_REQUIRE(scale > 0.f, "talking_tiles: the maxima are those of unscaled scores, which takes a positive scale");
  CWM_REQUIRE(q_stride % 8 == 0 && ((uintptr_t)q % 16) == 0 && ((uintptr_t)cache % 16) == 0 && ((uintptr_t)out % 8) == 0 && ((uintptr_t)weights % 16) == 0,
              "talking_tiles: rows must be 16-byte aligned");
  const int per = n_q_heads / n_kv_heads, together = tile_heads_together(per);
  const int mix_rows = tile_mix_rows(n_q_heads), value_rows = together <= 2 ? 32 : 16, groups = cwm_talking_tile_groups(n_q_heads, n_kv_heads, head_dim);
  TalkPortions P;
  P.count = count;
  long blocks[3] = {0, 0, 0}, at = 0;
  int most_steps[TILE_PORTIONS];
  for (int i = 0; i < count; ++i) {
    const int* d = portions + 7 * i;
    TalkPortion& po = P.of[i];
    po.seq = d[0], po.t0 = d[1], po.n = d[2], po.pos0 = d[3], po.r0 = d[4], po.r1 = d[5], po.columns = d[6], po.table = at;
    CWM_REQUIRE(po.seq >= 0 && po.t0 >= 0 && po.pos0 >= 0 && po.r0 >= 0 && po.r0 % 32 == 0 && po.r1 > po.r0 && po.r1 <= po.n && po.columns % TILE_KEYS == 0, "talking_tiles: bad portion");
    most_steps[i] = 0;
    for (int row0 = po.r0; row0 < po.r1; row0 += mix_rows) {
      const int tile = po.pos0 + row0 / 32 * 32, last = po.pos0 + (row0 + mix_rows < po.n ? row0 + mix_rows : po.n) - 1;
      const int base = window_left >= 0 && tile > window_left ? tile - window_left : 0, steps = tile_steps(po, row0, mix_rows, window_left);
      CWM_REQUIRE(last / TILE_KEYS - base / TILE_KEYS < po.columns / TILE_KEYS, "talking_tiles: %d columns do not hold a row's keys", po.columns);
      most_steps[i] = steps > most_steps[i] ? steps : most_steps[i];
    }
    at += (long)n_q_heads * (po.r1 - po.r0) * po.columns;
  }
  const int steps = mix_steps(P, count, mix_rows, n_q_heads, window_left);
  for (int i = 0; i < count; ++i) {
    TalkPortion& po = P.of[i];
    const int rows = po.r1 - po.r0;
    for (int k = 0; k < 3; ++k) po.at[k] = (int)blocks[k];
    blocks[0] += (long)((rows + STATS_ROWS - 1) / STATS_ROWS) * groups;
    blocks[1] += (long)((rows + mix_rows - 1) / mix_rows) * ((most_steps[i] + steps - 1) / steps);
    blocks[2] += (long)((rows + value_rows - 1) / value_rows) * groups;
    for (int k = 0; k < 3; ++k) CWM_REQUIRE(blocks[k] < (1L << 30), "talking_tiles: too many blocks");
  }
  int page_shift = -1;
  if ((page_size & (page_size - 1)) == 0)
    for (page_shift = 0; (1 << page_shift) < page_size;) ++page_shift;
  const TalkTileArgs A = {(const bf16_t*)q, q_stride, (const bf16_t*)cache, block_table, table_width, n_q_heads, n_kv_heads, page_size, page_shift, num_pages, window_left,
                          scale * LOG2E};
#define CWM_STATS(HD, HEADS)                                                                                                                hipLaunchKernelGGL((talk_tile_stats_kernel<HD, HEADS>), dim3((unsigned)blocks[0]), dim3(64 * TILE_WAVES), 0, stream, A, P, stats, sink)
#define CWM_MIX(HD, SLOTS, HPW, RT)                                                                                                         hipLaunchKernelGGL((talk_tile_mix_kernel<HD, SLOTS, HPW, RT>), dim3((unsigned)blocks[1]), dim3(64 * TILE_WAVES), 0, stream, A, P, stats, talk, (bf16_t*)weights, steps)
#define CWM_VALUES(HD, HEADS, RT)                                                                                                           hipLaunchKernelGGL((talk_tile_values_kernel<HD, HEADS, RT>), dim3((unsigned)blocks[2]), dim3(64 * VALUE_WAVES), 0, stream, A, P, (const bf16_t*)weights, (bf16_t*)out)
#define CWM_ALL(HD)                                                                      \
  do {                                                                                   \
    if (together == 1) CWM_STATS(HD, 1);                                                 \
    else if (together == 2) CWM_STATS(HD, 2);                                            \
    else if (together == 3) CWM_STATS(HD, 3);                                            \
    else CWM_STATS(HD, 4);                                                               \
    if (n_q_heads <= 8) CWM_MIX(HD, 8, 1, 2); /* never more than one head a wavefront */ \
    else if (n_q_heads <= 16 && each <= 2) CWM_MIX(HD, 16, 2, 2);                        \
    else if (n_q_heads <= 16) CWM_MIX(HD, 16, 3, 2);                                     \
    else if (each <= 3) CWM_MIX(HD, 32, 3, 1);                                           \
    else CWM_MIX(HD, 32, 4, 1);                                                          \
    if (together == 1) CWM_VALUES(HD, 1, 2);                                             \
    else if (together == 2) CWM_VALUES(HD, 2, 2);                                        \
    else if (together == 3) CWM_VALUES(HD, 3, 1);                                        \
    else CWM_VALUES(HD, 4, 1);                                                           \
  } while (0)
  if (head_dim == 128) CWM_ALL(128);
  else CWM_ALL(64);
#undef CWM_ALL
#undef CWM_VALUES
#undef CWM_MIX
#undef CWM_STATS
  return cwm_launch_status("talking_tiles");
}

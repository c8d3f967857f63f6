// C[M, N] = A[M, K] * W[N, K]^T in bfloat16 with float32 sums for the many rows of a prompt, where the library's own tiles
// would leave a good part of the chip idle: its largest (256 x 256, 256 x 192) reach 1.3 to 1.5 PFLOP/s when they fill the 256
// compute units to the last round, and half of that when they do not.  The loop is gemm_wide.h's; here are its tiles, the
// choice between them, and the epilogue silu(gate) * up.
//
// Measured, library / this, us: 1,040 x 4,096 x 4,096 46 / 39, 1,040 x 4,096 x 14,336 147 / 130, 2,296 x 2,048 x 2,048 27.5 / 21.7,
// 1,500 x 2,048 x 2,048 21.4 / 17.0, 2,048 x 10,304 x 2,048 95 / 87, 600 x 4,096 x 4,096 37 / 29; but 4,096 x 8,192 x 6,144, two full rounds of
// 256 x 256, 284 / 338, and 3,000 x 512 x 14,336, where the library cuts K, 73 / 85.
//
// Every sum adds its 64-wide steps of K in their order whatever the tile, so a row's bits depend on its own values alone.
//
// Replaces torch.nn.functional.linear at cwm/fastgen/forward.py:593-606,763,776-782,820 for prompts.  Needs K % 64 == 0,
// N % 16 == 0 and 16-byte aligned rows.
#include "gemm_wide.h"

#include <math.h>

CWM_DEFINE_ERROR_API

#define WIDE_BAND 8  // row tiles whose column tiles follow one another

struct WideOrder {
  int m_tiles, n_tiles;
  // tile t: bands of WIDE_BAND row tiles, in a band column by column, so that the 32 blocks of an XCD, which take
  // consecutive tiles, share 8 row panels of A and 4 of W in its L2
  __device__ __forceinline__ void place(int t, int& tm, int& tn) const {
    const int band = t / (WIDE_BAND * n_tiles), in_band = t - band * WIDE_BAND * n_tiles;
    const int rows = min(WIDE_BAND, m_tiles - band * WIDE_BAND);
    tn = in_band / rows;
    tm = band * WIDE_BAND + in_band - tn * rows;
  }
};

template <int WM, int WN>
struct PlainSource {
  const bf16_t *A, *W;
  long lda, ldw;
  int M, N, lane, wave;
  WideOrder order;
  const bf16_t *a, *w;
  uint32_t off[WideShape<WM, WN>::ND];
  static constexpr bool W_TILES = false;
  __device__ __forceinline__ const bf16_t* base(int p) const { return p < WideShape<WM, WN>::BM / 8 ? a : w; }
  __device__ __forceinline__ void enter(int tile) {
    constexpr int BM = WideShape<WM, WN>::BM, BN = WideShape<WM, WN>::BN;
    int tm, tn;
    order.place(tile, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    a = A + (size_t)m0 * lda;
    w = W + (size_t)n0 * ldw;
#pragma unroll
    for (int i = 0; i < WideShape<WM, WN>::ND; ++i) {
      const int p = min(wave + 8 * i, WideShape<WM, WN>::PIECES - 1);
      const int row = 8 * p + (lane >> 3);
      // rows past the matrix read its last one: their sums are not stored
      if (p < BM / 8)
        off[i] = (uint32_t)(((size_t)min(row, M - 1 - m0) * lda + 8 * ((lane & 7) ^ ((row >> 1) & 7))) * 2);
      else
        off[i] = (uint32_t)(((size_t)min(row - BM, N - 1 - n0) * ldw + 8 * ((lane & 7) ^ wide_w_key<WN>(row - BM))) * 2);
    }
  }
};

// GLU: the columns are eight gates, then the eight ups of the same outputs, in turn; C[M, N / 2] = silu(gate) * up, both
// rounded to bfloat16 first, as the product and the kernel after it would have done.  With four tiles of columns a lane
// holds both eights; with two it holds one, and trades with its neighbour: the lanes of even j finish the even rows.
template <int WM, int WN, typename TC, bool GLU>
struct PlainSink {
  TC* C;
  long ldc;
  int M, N, lane, wave;
  WideOrder order;
  static constexpr int STORES = GLU ? WM * WN / 4 : WM * (sizeof(TC) == 4 ? WN : WN / 2);

  static __device__ __forceinline__ float gated(float g, float u) {
    g = bf16_to_f32(f32_to_bf16(g)), u = bf16_to_f32(f32_to_bf16(u));
    return g / (1.0f + expf(-g)) * u;
  }
  static __device__ __forceinline__ uint4 gated8(const float4v& g0, const float4v& g1, const float4v& u0, const float4v& u1) {
    return make_uint4(pack2_bf16(gated(g0[0], u0[0]), gated(g0[1], u0[1])), pack2_bf16(gated(g0[2], u0[2]), gated(g0[3], u0[3])),
                      pack2_bf16(gated(g1[0], u1[0]), gated(g1[1], u1[1])), pack2_bf16(gated(g1[2], u1[2]), gated(g1[3], u1[3])));
  }

  __device__ __forceinline__ bool store(int tile, float4v (&acc)[WM][WN]) const {
    constexpr int BM = WideShape<WM, WN>::BM, BN = WideShape<WM, WN>::BN;
    int tm, tn;
    order.place(tile, tm, tn);
    const int r = lane & 15, j = lane >> 4, wm = wave >> 2, wn = wave & 3;
    const int m0 = tm * BM + wm * WM * 16 + r;            // this lane's first row
    const int n0 = tn * BN + wn * WN * 16 + 4 * WN * j;  // and its 4 WN columns
    const bool full = (tm + 1) * BM <= M && (tn + 1) * BN <= N;
    if constexpr (GLU && WN == 4) {
      if (n0 < N) {
#pragma unroll
        for (int a = 0; a < WM; ++a) {
          const int m = m0 + 16 * a;
          if (m < M) *(uint4*)((bf16_t*)C + (size_t)m * ldc + n0 / 2) = gated8(acc[a][0], acc[a][1], acc[a][2], acc[a][3]);
        }
      }
    } else if constexpr (GLU) {
      static_assert(!GLU || WN == 4 || (WN == 2 && WM % 2 == 0), "rows are traded in pairs");
      const bool odd = j & 1;
#pragma unroll
      for (int a = 0; a < WM; a += 2) {
        float4v got[2], have[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const float4v give = odd ? acc[a][b] : acc[a + 1][b];
          have[b] = odd ? acc[a + 1][b] : acc[a][b];
#pragma unroll
          for (int e = 0; e < 4; ++e) got[b][e] = __shfl_xor(give[e], 16, 64);
        }
        const int m = m0 + 16 * (a + (odd ? 1 : 0));
        const uint4 v = odd ? gated8(got[0], got[1], have[0], have[1]) : gated8(have[0], have[1], got[0], got[1]);
        if (m < M && n0 < N) *(uint4*)((bf16_t*)C + (size_t)m * ldc + (n0 / 16) * 8) = v;
      }
    } else {
#pragma unroll
      for (int a = 0; a < WM; ++a) {
        const int m = m0 + 16 * a;
        if (m >= M) continue;
        TC* row = C + (size_t)m * ldc + n0;
#pragma unroll
        for (int b = 0; b < WN; b += 2) {  // eight columns, which lie before or past the end together
          if (n0 + 4 * b >= N) continue;
          if constexpr (sizeof(TC) == 4) {
            *(float4v*)(row + 4 * b) = acc[a][b];
            *(float4v*)(row + 4 * b + 4) = acc[a][b + 1];
          } else {
            *(uint4*)(row + 4 * b) = make_uint4(pack2_bf16(acc[a][b][0], acc[a][b][1]), pack2_bf16(acc[a][b][2], acc[a][b][3]),
                                                pack2_bf16(acc[a][b + 1][0], acc[a][b + 1][1]), pack2_bf16(acc[a][b + 1][2], acc[a][b + 1][3]));
          }
        }
      }
    }
    return full;
  }
};

template <int WM, int WN, typename TC, bool GLU>
__global__ void __launch_bounds__(512, 2)
gemm_wide_kernel(const bf16_t* __restrict__ A, long lda, const bf16_t* __restrict__ W, long ldw, TC* __restrict__ C, long ldc,
                 int M, int N, int steps, int m_tiles, int n_tiles) {
  typedef WideShape<WM, WN> Shape;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[Shape::S * Shape::STAGE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the XCDs (block number modulo 8) take consecutive runs of tiles, their blocks in turn
  const int total = m_tiles * n_tiles, groups = min(8, (int)gridDim.x);
  const int xcd = blockIdx.x % groups, idx = blockIdx.x / groups;
  const int blocks = ((int)gridDim.x + groups - 1 - xcd) / groups;  // of this XCD, at least one
  const int per = total / groups, rest = total % groups;
  const int first = xcd * per + min(xcd, rest), count = per + (xcd < rest ? 1 : 0);
  const int mine = (count - idx + blocks - 1) / blocks;
  const WideOrder order = {m_tiles, n_tiles};
  PlainSource<WM, WN> src = {A, W, lda, ldw, M, N, lane, wave, order};
  PlainSink<WM, WN, TC, GLU> sink = {C, ldc, M, N, lane, wave, order};
  wide_loop<WM, WN, PlainSink<WM, WN, TC, GLU>::STORES>(lds, src, sink, first + idx, blocks, mine, steps);
}

// What a product costs with one tile, us: to start, each round of a block's tiles, each step of a round, and of each step
// `fill` in proportion to the tiles there are, since the chip's power and its L2 are shared.
struct TileCost {
  int rows, columns;
  float start, round, step, fill;
};
static float tile_us(const TileCost& t, int M, int N, int K, int units, float more_a_round) {
  const float tiles = (float)((M + t.rows - 1) / t.rows) * (float)((N + t.columns - 1) / t.columns);
  const float rounds = ceilf(tiles / (float)units), steps = (float)K / WIDE_BK;
  return t.start + rounds * (t.round + more_a_round + steps * t.step) + tiles / (float)units * steps * t.fill;
}
// This kernel's tiles.  Fitted to 1,100 products of 130 to 4,096 rows, 512 to 28,672 columns and a K of 512 to 14,336, within 8% (a K below
// 512 takes up to a fifth longer); the tile it picks is on average 1% slower than the best one.  Tiles of 192 columns are not among them: at 42 of those
// sizes one was ahead of all of these by more than 3%, by 17% at the most (3,538 x 3,072 x 6,144 112 / 131, 1,040 x 28,672 x 6,144 317 / 351).
static const TileCost wide_tiles[] = {
    {256, 128, 2.18f, 2.96f, 0.54f, 0.30f}, {192, 128, 2.64f, 2.31f, 0.43f, 0.24f}, {128, 128, 3.18f, 1.29f, 0.35f, 0.18f},
    {64, 128, 2.94f, 0.61f, 0.26f, 0.10f},  {128, 256, 2.37f, 2.70f, 0.58f, 0.28f}, {160, 256, 2.39f, 3.40f, 0.69f, 0.31f},
    // heights of an odd number of tiles a wavefront, which the gated epilogue cannot trade between lanes
    {224, 128, 2.34f, 2.55f, 0.53f, 0.25f}, {160, 128, 3.01f, 1.52f, 0.43f, 0.20f}, {96, 128, 3.20f, 0.92f, 0.32f, 0.14f}};
#define WIDE_TILES 9
#define WIDE_GLU_TILES 6
static int wide_tile(int M, int N, int K, int units, bool glu, float* us) {
  int best = 0;
  for (int i = 0; i < (glu ? WIDE_GLU_TILES : WIDE_TILES); ++i) {
    // the gated epilogue costs a tile of 256 x 128 0.6 us more than storing the sums
    const float t = tile_us(wide_tiles[i], M, N, K, units, glu ? 0.64f / (256 * 128) * wide_tiles[i].rows * wide_tiles[i].columns : 0.f);
    if (i == 0 || t < *us) best = i, *us = t;
  }
  return best;
}
// The library's product, as if it picked the best of these tiles: fitted to its times for the same sizes, within 14%.  It wins
// where its large tiles fill whole rounds (4,096 x 8,192 x 6,144).
static const TileCost library_tiles[] = {
    {256, 256, 6.9f, 6.4f, 0.97f, 0.43f}, {256, 192, 3.2f, 5.3f, 1.25f, 0.f},  {192, 256, 0.f, 10.3f, 0.72f, 0.42f},  {256, 128, 0.f, 12.7f, 0.38f, 0.58f},
    {128, 256, 9.4f, 0.f, 0.31f, 0.58f},  {128, 128, 12.f, 1.3f, 0.f, 0.49f}, {160, 128, 0.f, 13.5f, 0.64f, 0.f}};

// the share of the chip that a tile of the library fills over all its rounds
static float library_fill(const TileCost& t, int M, int N, int units) {
  const float tiles = (float)((M + t.rows - 1) / t.rows) * (float)((N + t.columns - 1) / t.columns);
  return (float)M * (float)N / (ceilf(tiles / (float)units) * (float)units * (float)(t.rows * t.columns));
}

// Whether this kernel takes a product from the library, with `glu` also the kernel that gates its result (3 us and three passes that mostly
// stay in the memory-side cache): where the library's largest tiles (the first three) leave a quarter of the chip idle, or by the costs above, by
// 4% at least.  Of 2,127 products that drawn steps of all designs bring it, timed on the GPU with weights from memory, it is 1.09 times as fast in
// the mean, and 338 times slower by more than 5%, 20 times by more than 10 us: small results, where the library cuts a K of 1,536 and more and this
// kernel does not (library / this, us: 450 x 512 x 3,072 9.5 / 18.0, 384 x 2,048 x 2,048 12.4 / 14.9).  They stay all the same, down to a few
// hundredths of the chip: a call of the library takes the host 20 us more in a step, and steps of such products wait for the host (60 drawn steps with the
// library for most of those 338 took 3.2% longer, up to 10%; 380 tokens with three of them 1,614 us and 1,485).  Results of fewer columns than a
// tile (a router's 16: 2,048 x 16 x 2,048 11.5 / 12.2) stay with the library.
extern "C" int cwm_gemm_bf16_wide_pays(int M, int N, int K, int units, int glu) {
  if (M <= 0 || N < 128 || K <= 0 || K % WIDE_BK || N % 16 || units <= 0) return 0;
  const float share = (float)M * (float)N / (65536.f * (float)units);
  if (K > (share < 0.04f ? 3072 : share < 0.08f ? 4096 : K)) return 0;
  float us = 0.f, library = 0.f, fill = 0.f;
  wide_tile(M, N, K, units, glu != 0, &us);
  for (int i = 0; i < (int)(sizeof(library_tiles) / sizeof(library_tiles[0])); ++i) {
    const float t = tile_us(library_tiles[i], M, N, K, units, 0.f);
    if (i == 0 || t < library) library = t;
    if (i < 3) fill = fmaxf(fill, library_fill(library_tiles[i], M, N, units));
  }
  // a width that its tiles do not end with costs the library a tenth: 777 to 4,096 rows, a K of 1,536 to 3,072, library / this in the mean 1.03 at
  // 4,096, 6,144, 8,192, 10,240 and 12,288 columns, 1.15 at 4,128, 6,208, 8,224, 10,304 and 12,352 (2,048 x 10,304 x 2,048 97 / 87)
  if (N % 128) library *= 1.1f;
  if (glu) library += 3.f + 3e-7f * (float)M * (float)N;
  return fill < 0.75f || us < 0.96f * library;
}

// C [M][ldc] of c_dtype; glu: W holds gate and up rows in alternating groups of 8 and C [M, N / 2] receives silu(gate) * up in
// bfloat16.  `tile`: -1, or the number of a tile of the list above (tests).
extern "C" int cwm_gemm_bf16_wide(const void* A, long lda, const void* W, long ldw, void* C, int c_dtype, long ldc, int M, int N, int K,
                                  int units, int glu, int tile, hipStream_t stream) {
  CWM_REQUIRE(M >= 0 && N > 0 && K > 0 && units > 0, "gemm_bf16_wide: bad sizes M=%d N=%d K=%d units=%d", M, N, K, units);
  CWM_REQUIRE(K % WIDE_BK == 0, "gemm_bf16_wide: K=%d must be a multiple of %d", K, WIDE_BK);
  CWM_REQUIRE(N % 16 == 0, "gemm_bf16_wide: N=%d must be a multiple of 16", N);
  CWM_REQUIRE(lda % 8 == 0 && ldw % 8 == 0 && ldc % 8 == 0, "gemm_bf16_wide: row strides must be multiples of 8 elements");
  CWM_REQUIRE(((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0 && ((uintptr_t)C % 16) == 0, "gemm_bf16_wide: operands must be 16-byte aligned");
  CWM_REQUIRE(lda >= K && ldw >= K && ldc >= (glu ? N / 2 : N), "gemm_bf16_wide: row strides shorter than rows");
  CWM_REQUIRE(lda < (1L << 22) && ldw < (1L << 22), "gemm_bf16_wide: row strides too long for 32-bit offsets");
  CWM_REQUIRE(c_dtype == CWM_F32 || c_dtype == CWM_BF16, "gemm_bf16_wide: unknown output dtype %d", c_dtype);
  CWM_REQUIRE(!glu || c_dtype == CWM_BF16, "gemm_bf16_wide: the gated epilogue gives a bfloat16 result");
  if (M == 0) return 0;
  float us = 0.f;
  if (tile < 0) tile = wide_tile(M, N, K, units, glu != 0, &us);
  CWM_REQUIRE(tile < (glu ? WIDE_GLU_TILES : WIDE_TILES), "gemm_bf16_wide: no tile %d", tile);
  const int wm = wide_tiles[tile].rows / 32, wn = wide_tiles[tile].columns / 64;
  const long m_tiles = (M + 32 * wm - 1) / (32 * wm), n_tiles = (N + 64 * wn - 1) / (64 * wn);
  CWM_REQUIRE(m_tiles * n_tiles * (K / WIDE_BK) < (1L << 31), "gemm_bf16_wide: too many steps of tiles");
  dim3 grid((unsigned)(m_tiles * n_tiles < units ? m_tiles * n_tiles : units));
#define CWM_WIDE_RUN(WM, WN, TC, GLU)                                                                                                \
  hipLaunchKernelGGL((gemm_wide_kernel<WM, WN, TC, GLU>), grid, dim3(512), 0, stream, (const bf16_t*)A, lda, (const bf16_t*)W, ldw,   \
                     (TC*)C, ldc, M, N, K / WIDE_BK, (int)m_tiles, (int)n_tiles)
#define CWM_WIDE_TILE(WM, WN, GATED)                        \
  if (wm == WM && wn == WN) {                               \
    if (glu) {                                              \
      if constexpr (GATED) CWM_WIDE_RUN(WM, WN, bf16_t, true); \
    } else if (c_dtype == CWM_F32)                          \
      CWM_WIDE_RUN(WM, WN, float, false);                   \
    else                                                    \
      CWM_WIDE_RUN(WM, WN, bf16_t, false);                  \
  }
  CWM_WIDE_TILE(8, 2, true)
  CWM_WIDE_TILE(6, 2, true)
  CWM_WIDE_TILE(4, 2, true)
  CWM_WIDE_TILE(2, 2, true)
  CWM_WIDE_TILE(4, 4, true)
  CWM_WIDE_TILE(5, 4, true)
  CWM_WIDE_TILE(7, 2, false)
  CWM_WIDE_TILE(5, 2, false)
  CWM_WIDE_TILE(3, 2, false)
#undef CWM_WIDE_TILE
#undef CWM_WIDE_RUN
  return cwm_launch_status("gemm_bf16_wide");
}

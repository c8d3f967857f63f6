// The loop of a matrix product whose operands both pass through LDS: C[m, n] = sum over k of A[m, k] * W[n, k],
// bfloat16 operands, float32 sums.  Shared by the plain product of many rows (gemm_bf16_wide.hip) and the routed
// experts' (routed.hip), which differ in where a tile's rows lie and in what becomes of its sums.
//
// Persistent blocks of eight wavefronts, two along the rows and four along the columns; a wavefront holds WM x WN tiles
// of 16 x 16 sums.  K goes in steps of 64.  A step's rows of A and W (BM + BN rows of 128 bytes, a cache line each) reach
// LDS by direct loads, up to S steps ahead into S buffers; the stream of loads runs on across tiles, so a block fills its
// pipeline once.  While a wavefront multiplies half a step, it reads the other half's operands from LDS into a second set
// of registers and issues the loads of a step to come, a few of each after every row of matrix instructions: issued in one
// go they queue up before the memory pipe while the matrix cores wait.  One barrier a step.
//
// What bounds it: on all 256 compute units the chip's power (a loop of nothing but these instructions on varied operands,
// ceilings.hip, reaches 1.45 PFLOP/s; the library's best product 1.58); below that a step's loads (64 KB in flight a compute
// unit against 1.3 to 1.6 us of latency), which is why smaller tiles with three to five buffers are used and no tile of
// 256 x 256 with two.  A load of 64-byte instead of 128-byte rows is slower by a third, two groups of wavefronts that take turns between
// reading and multiplying by 5 to 15%.
//
//   v_mfma_f32_16x16x32_bf16:  C^T[n, m] += W[n, k] * A[m, k]
//     A operand = W (lane 16 j + r: row r, k = 32 s + 8 j .. + 7), B operand = A^T (same); lane 16 j + r gets C[r][4 j .. + 3]
// Row r of tile b of a wavefront's WN is the column 4 WN (r / 4) + 4 b + r % 4 of its 16 WN, so that a lane's sums are
// 4 WN consecutive columns of a row of C.
//
// In LDS the 16-byte piece p of a row lies at p ^ key(row); the keys spread the 16 rows of one operand read over all
// banks: rows of A follow one another, (row / 2) % 8; rows of W come in fours 4 WN apart.
//
// A SOURCE with W_TILES has W in operand tiles, [16 rows][32 k][64 lanes][8 values]: 1 KB is an operand, in memory as in LDS, row r of
// tile b is the column 16 b + r, and a lane's sums are 4 consecutive columns of each tile.
#pragma once

#include "common.h"

#define WIDE_BK 64
#define WIDE_LDS (160 * 1024)

template <int WM, int WN>
struct WideShape {
  static constexpr int BM = 2 * WM * 16, BN = 4 * WN * 16;
  static constexpr int PIECES = (BM + BN) / 8;        // loads a step, of eight rows each
  static constexpr int ND = (PIECES + 7) / 8;         // of a wavefront (the last ones may be double)
  static constexpr int STAGE = PIECES * 1024;
  static constexpr int S = WIDE_LDS / STAGE < 5 ? WIDE_LDS / STAGE : 5;
  static_assert(S >= 3, "a tile needs three buffers");
};

template <int WN>
__device__ __forceinline__ int wide_w_key(int row) {  // of a row of W within the tile (a wavefront's rows are 16 WN in turn)
  return ((row >> 1) & 1) | (((row / (4 * WN)) & 3) << 1);
}

// SOURCE: enter(tile) sets what base(p) answers, where piece p of a step lies (a uniform pointer; pieces p < BM / 8 are A's rows
// 8 p .., the others eight rows of W, or an operand of half a step), and `off[ND]`, this lane's byte offsets of its loads from there.  SINK: store(tile, acc) writes
// the sums, with exactly STORES store instructions if it answers true.
template <int WM, int WN, int STORES, typename SOURCE, typename SINK>
__device__ __forceinline__ void wide_loop(unsigned char* lds, SOURCE& src, SINK& sink, int tile, int tile_stride, int n_tiles, int steps) {
  typedef WideShape<WM, WN> Shape;
  constexpr int BM = Shape::BM, ND = Shape::ND, STAGE = Shape::STAGE, S = Shape::S, PIECES = Shape::PIECES;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, j = lane >> 4;
  const int wm = wave >> 2, wn = wave & 3;
  if (n_tiles <= 0) return;

  // ---- the stream of loads: the step it is at, and how many are left
  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
  int i_tile = tile, i_step = 0, i_left = n_tiles * steps;
  src.enter(i_tile);
  auto issue_one = [&](int i, uint32_t stage) __attribute__((always_inline)) {
    const int p = min(wave + 8 * i, PIECES - 1);
    dma16(src.base(p) + (size_t)i_step * (SOURCE::W_TILES && p >= BM / 8 ? 1024 : WIDE_BK), src.off[i], lds0 + stage + p * 1024);
  };
  auto advance = [&]() __attribute__((always_inline)) {  // past the last step: that step again, into a buffer nobody reads
    if (i_left > 1) {
      --i_left;
      if (++i_step == steps) {
        i_step = 0;
        i_tile += tile_stride;
        src.enter(i_tile);
      }
    }
  };

  const int a_key = (r >> 1) & 7;
  const int w_row = 4 * WN * (r >> 2) + (r & 3);  // of tile b: + 4 b, the key's row bits of which follow from b alone
  const unsigned char* const a_base = lds + (wm * WM * 16 + r) * 128;
  const unsigned char* const w_base = lds + BM * 128 + (SOURCE::W_TILES ? wn * WN * 2048 + lane * 16 : (wn * WN * 16 + w_row) * 128);
  int w_piece[WN];  // of the first half; the second half's is ^ 64 bytes, or 1 KB further
#pragma unroll
  for (int b = 0; b < WN; ++b) w_piece[b] = SOURCE::W_TILES ? b * 2048 : b * 512 + ((j ^ wide_w_key<WN>(wn * WN * 16 + w_row + 4 * b)) * 16);
  const int a_piece = (j ^ a_key) * 16;

  float4v acc[WM][WN];
  Frag8 a0[WM], b0[WN], a1[WM], b1[WN];
#define WIDE_READ_A(FA, ST, HALF, i) FA[i].u = *(const uint4*)(a_base + (ST) + (i) * 2048 + (a_piece ^ ((HALF) * 64)))
#define WIDE_READ_W(FB, ST, HALF, i) FB[i].u = *(const uint4*)(w_base + (ST) + (w_piece[i] ^ ((HALF) * (SOURCE::W_TILES ? 1024 : 64))))
#define WIDE_ROW(FA, FB, i) \
  _Pragma("unroll") for (int b = 0; b < WN; ++b) acc[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(FB[b].v, FA[i].v, acc[i][b], 0, 0, 0);
  constexpr int READS = (WN + WM + WM - 2) / (WM - 1);  // after a row of matrix instructions, so that none follow the last
#define WIDE_READS(FA, FB, ST, HALF, i)                                           \
  _Pragma("unroll") for (int q = (i) * READS; q < (i) * READS + READS; ++q) {     \
    if (q < WN) { WIDE_READ_W(FB, ST, HALF, q); }                                 \
    else if (q < WN + WM) { WIDE_READ_A(FA, ST, HALF, q - WN); }                  \
  }

#pragma unroll 1  // entering a tile is much code
  for (int s = 0; s < S; ++s) {
#pragma unroll
    for (int i = 0; i < ND; ++i) issue_one(i, s * STAGE);
    advance();
  }
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"((S - 1) * ND) : "memory");
  int cur = 0;
#pragma unroll
  for (int b = 0; b < WN; ++b) WIDE_READ_W(b0, 0, 0, b);
#pragma unroll
  for (int a = 0; a < WM; ++a) WIDE_READ_A(a0, 0, 0, a);

  bool stored = false;  // the last tile's stores may be under way, STORES of them, after the loads that are waited for next
  for (int left = n_tiles; left > 0; --left, tile += tile_stride) {
#pragma unroll
    for (int a = 0; a < WM; ++a)
#pragma unroll
      for (int b = 0; b < WN; ++b) acc[a][b] = (float4v){0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < steps; ++k) {
      const int nxt = cur + STAGE == S * STAGE ? 0 : cur + STAGE;
#pragma unroll
      for (int a = 0; a < WM; ++a) {
        WIDE_ROW(a0, b0, a)
        __builtin_amdgcn_sched_barrier(0);
        WIDE_READS(a1, b1, cur, 1, a)
        __builtin_amdgcn_sched_barrier(0);
      }
      // this wavefront's loads of the next step have landed and it has read all of this step; after the barrier so has everyone
      if (k == 0 && stored)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((S - 2) * ND + STORES < 63 ? (S - 2) * ND + STORES : 63) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((S - 2) * ND) : "memory");
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int a = 0; a < WM; ++a) {
        WIDE_ROW(a1, b1, a)
        __builtin_amdgcn_sched_barrier(0);
        WIDE_READS(a0, b0, nxt, 0, a)
#pragma unroll
        for (int i = a * ND / WM; i < (a + 1) * ND / WM; ++i) issue_one(i, cur);
        __builtin_amdgcn_sched_barrier(0);
      }
      advance();
      cur = nxt;
    }
    stored = sink.store(tile, acc);
  }
  asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // the loads past the last step, and the last stores
#undef WIDE_READ_A
#undef WIDE_READ_W
#undef WIDE_ROW
#undef WIDE_READS
}

// C[M, N] = A[M, K] * W[N, K]^T (+ bias[N]) in float32 on the matrix cores
// (v_mfma_f32_32x32x2_f32: float32 operands, exact products, float32 sums; float32 operands with
// K a multiple of 32 and up to 65,536 in exact bfloat16 parts instead, with an entry of their own, see below): the matrix
// product of the 32-bit path.  Operands may be stored as float32 or bfloat16 (converted
// exactly on load).  Every output
// element is the sum over k = 0, 1, ... in one fixed grouping (eight values at a time, as the
// pairs (j, j + 4), j = 0..3; 32 at a time in parts), whatever tile of the result it lies in, so
// a row's result does not depend on the other rows of the call.  Any M, N, K.
//
// A block takes a BM x BN tile of C (128 x 128 with 4 wavefronts; 32 x 32 with one for at most 32
// rows); tiles of A and W of BK values of k go through LDS, the next ones waiting in registers.
// Lane l of a 32 x 32 matrix instruction supplies A[l % 32][l / 32] and W[l % 32][l / 32]; a
// lane reads four consecutive k of its row at once (16 bytes) and feeds them to four
// instructions, so the two halves of the lanes pair k with k + 4: any pairing gives the
// same sum of products as long as both operands use it.
//
// Replaces torch.nn.functional.linear at cwm/fastgen/forward.py:593-606,763,
// 776-782,820 (weights [out, in] row-major, y = x W^T + b).
#include "common.h"

CWM_DEFINE_ERROR_API

typedef float float16v __attribute__((ext_vector_type(16)));

// a step takes BK values of k; a row of a tile in LDS is padded to BK + 4 floats (16-byte pieces stay aligned)

// four consecutive elements of a row from element `k` on, zeros from K on; `vec`: the row is
// 16-byte (float32) or 8-byte (bfloat16) aligned at multiples of 4 elements
template <typename T>
__device__ __forceinline__ void load4(const T* row, int k, int K, bool vec, float (&v)[4]) {
  if (vec && k + 4 <= K) {
    if constexpr (sizeof(T) == 4) {
      const float4 f = *(const float4*)(row + k);
      v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
    } else {
      const uint2 u = *(const uint2*)(row + k);
      v[0] = bf16_to_f32((bf16_t)(u.x & 0xffffu)); v[1] = bf16_to_f32((bf16_t)(u.x >> 16));
      v[2] = bf16_to_f32((bf16_t)(u.y & 0xffffu)); v[3] = bf16_to_f32((bf16_t)(u.y >> 16));
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (k + i < K) ? Elem<T>::load(row + k + i) : 0.f;
  }
}

// WAVES_M x WAVES_N wavefronts, each with TM x TN matrix-instruction tiles of 32 x 32; BK: a multiple of 8
// One block's tile of the result, from row m0 and column n0 on; As, Ws: BM and BN rows of BK + 4 floats of LDS.  MARKED: only the
// elements of the tile's rows and columns with a mark are stored.
template <typename TA, typename TW, typename TC, int WAVES_M, int WAVES_N, int TM, int TN, int BK, bool MARKED = false>
__device__ __forceinline__ void gemm_f32_tile(const TA* __restrict__ A, long lda, const TW* __restrict__ W, long ldw, TC* __restrict__ C, long ldc,
                                              const void* __restrict__ bias, int bias_dtype, int M, int N, int K, int vec_a, int vec_w, const int m0,
                                              const int n0, float* As, float* Ws, const unsigned char* marked_rows = nullptr,
                                              const unsigned char* marked_columns = nullptr) {
  constexpr int BM = 32 * TM * WAVES_M, BN = 32 * TN * WAVES_N, THREADS = 64 * WAVES_M * WAVES_N;
  constexpr int BKP = BK + 4, Q = BK / 4;  // Q: 16-byte pieces in a row of a step
  constexpr int A_LOADS = (BM * Q + THREADS - 1) / THREADS, W_LOADS = (BN * Q + THREADS - 1) / THREADS;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  const int r32 = lane & 31;  // the lane's row of a 32 x 32 operand
  const int kh = lane >> 5;   // and its half of the k values

  float16v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  float ra[A_LOADS][4], rw[W_LOADS][4];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
      const int f = tid + i * THREADS;  // piece f: row f / Q, values 4 * (f % Q) .. + 3 of the step
      const int m = m0 + f / Q;
      if (f / Q < BM && m < M)
        load4(A + (size_t)m * lda, k0 + 4 * (f % Q), K, vec_a != 0, ra[i]);
      else
        ra[i][0] = ra[i][1] = ra[i][2] = ra[i][3] = 0.f;
    }
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) {
      const int f = tid + i * THREADS;
      const int n = n0 + f / Q;
      if (f / Q < BN && n < N)
        load4(W + (size_t)n * ldw, k0 + 4 * (f % Q), K, vec_w != 0, rw[i]);
      else
        rw[i][0] = rw[i][1] = rw[i][2] = rw[i][3] = 0.f;
    }
  };
  auto stash = [&]() {
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
      const int f = tid + i * THREADS;
      if (f / Q < BM) *(float4*)(&As[(f / Q) * BKP + 4 * (f % Q)]) = make_float4(ra[i][0], ra[i][1], ra[i][2], ra[i][3]);
    }
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) {
      const int f = tid + i * THREADS;
      if (f / Q < BN) *(float4*)(&Ws[(f / Q) * BKP + 4 * (f % Q)]) = make_float4(rw[i][0], rw[i][1], rw[i][2], rw[i][3]);
    }
  };

  fetch(0);
  for (int k0 = 0; k0 < K; k0 += BK) {
    stash();
    __syncthreads();
    if (k0 + BK < K) fetch(k0 + BK);  // in flight while this step is multiplied
#pragma unroll
    for (int o = 0; o < BK / 8; ++o) {  // the step's k values 8 o .. 8 o + 7
      float4 fa[TM], fw[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[i] = *(const float4*)(&As[((wm * TM + i) * 32 + r32) * BKP + 8 * o + 4 * kh]);
#pragma unroll
      for (int j = 0; j < TN; ++j) fw[j] = *(const float4*)(&Ws[((wn * TN + j) * 32 + r32) * BKP + 8 * o + 4 * kh]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            const float a = e == 0 ? fa[i].x : e == 1 ? fa[i].y : e == 2 ? fa[i].z : fa[i].w;
            const float w = e == 0 ? fw[j].x : e == 1 ? fw[j].y : e == 2 ? fw[j].z : fw[j].w;
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, w, acc[i][j], 0, 0, 0);
          }
    }
    __syncthreads();
  }

  // lane l of a result tile holds column l % 32 and the rows 8 (e / 4) + 4 (l / 32) + e % 4, e = 0..15
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + (wn * TN + j) * 32 + r32;
    if (n >= N) continue;
    float b = 0.f;
    if (bias) b = bias_dtype == CWM_BF16 ? bf16_to_f32(((const bf16_t*)bias)[n]) : ((const float*)bias)[n];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + (wm * TM + i) * 32 + 8 * (e >> 2) + 4 * kh + (e & 3);
        if (MARKED && !(marked_rows[m - m0] | marked_columns[n - n0])) continue;
        if (m < M) Elem<TC>::store(C + (size_t)m * ldc + n, acc[i][j][e] + b);
      }
  }
}

template <typename TA, typename TW, typename TC, int WAVES_M, int WAVES_N, int TM, int TN, int BK>
__global__ void __launch_bounds__(64 * WAVES_M * WAVES_N)
gemm_f32_kernel(const TA* __restrict__ A, long lda, const TW* __restrict__ W, long ldw, TC* __restrict__ C,
                long ldc, const void* __restrict__ bias, int bias_dtype, int M, int N, int K, int vec_a, int vec_w) {
  constexpr int BM = 32 * TM * WAVES_M, BN = 32 * TN * WAVES_N;
  __shared__ __attribute__((aligned(16))) float As[BM * (BK + 4)];
  __shared__ __attribute__((aligned(16))) float Ws[BN * (BK + 4)];
  gemm_f32_tile<TA, TW, TC, WAVES_M, WAVES_N, TM, TN, BK>(A, lda, W, ldw, C, ldc, bias, bias_dtype, M, N, K, vec_a, vec_w, blockIdx.y * BM, blockIdx.x * BN,
                                                          As, Ws);
}

// ---- float32 operands in three parts of eight bits ------------------------------------------------------------------ //
// a = a1 + a2 + a3 exactly, each part a bfloat16: a1 = a rounded, a2 = a - a1 rounded (the difference is exact and has at
// most 16 bits), a3 what is left (at most 8 bits).  a * w is then the sum of nine products of parts, exact in float32, of which
// the six largest are added up on the bfloat16 matrix instruction (v_mfma_f32_16x16x32_bf16, float32 sums), 16 times the
// rate of the float32 one: the three left out are below 2^-24 of the product together, and a sum takes 6 K / 32 roundings
// instead of K / 2.  Against float64 (normal operands, K = 512, 4,096 and 14,336) a result is 3.3e-7, 9.7e-7 and 1.8e-6 off,
// 4.0e-7, 1.15e-6 and 2.1e-6 with float32 operands; with positive operands 2.6e-7, 6.1e-7 and 1.1e-6 against 3.5e-7, 9.9e-7
// and 1.8e-6.  743 rows, float32 operands and parts: 28,672 x 4,096 1,847 and 828 us, 2,048 x 2,048 191 and 61 us.
// Memory holds float32: W's parts are made in registers.  Both operands are multiplied by 2^23 first, and
// the sums by 2^-46 at the end, which rounds nothing: the last bit of the smallest float32 is then a normal bfloat16, so that the parts
// of small values are exact too (without it the third part is lost below 2^-110 and the second below 2^-118).  Rows of A and W with a
// value of 2^32 or more, or an infinity, are left to float32 operands, element by element of the result: with smaller ones the sums of
// up to 65,536 scaled products stay below 2^126.  So an element's order of k and of the parts depends on its own row and column alone.
// The bfloat16 instruction rounds its sums down, not to the nearest: left alone, every result is low by the same amount (2.5e-8, 1.0e-7
// and 4.1e-7 of the results' size at K = 512, 2,048 and 8,192), which adds up over a model's layers (16 layers of width 2,048: logits
// 2.9e-6 off float64 where float32 operands are 2.4e-6).  So the 8 steps in the middle of every 16 go into the sum with its sign turned,
// where rounding down is up: logits 2.0e-6 off, at the same times.
#define SPLIT_STEP 32
#define SPLIT_MOST_K 65536
#define SPLIT_SCALE 8388608.0f               // 2^23
#define SPLIT_UNSCALE 1.4210854715202004e-14f  // 2^-46
#define SPLIT_TURN 4                         // steps after which the sum's sign turns, and 8 later again, of every 16
#define SPLIT_LIMIT 3.602879701896397e16f    // 2^55: 2^32 once scaled

//
// What bounded a kernel whose blocks made both operands' parts on their way into LDS was the making: vector instructions, which add to the
// matrix cores' time, two thirds as many cycles in a block of 128 x 128, and again in every block that read the row (28,672 x 4,096 986 us,
// 128,256 x 4,096 4,290, 6,144 x 4,096 283, 4,096 x 14,336 693, 2,048 x 2,048 72).  So A's parts are made once, by a kernel that writes them as operands of the
// matrix instruction, [tile of 16 rows][step of 32 k][part][64 lanes][8 values], signs turned with their steps; and a block takes up to 256
// rows, so that few blocks take a row of W apart, and the one wavefront that multiplies it does: the wavefronts lie side by side along the
// columns, 16 each, with all WM tiles of 16 rows.  Operands of A and raw rows of W reach LDS by direct loads, W two steps further ahead; a
// wavefront takes the next step's W apart while it multiplies; one barrier a step.  Now 828, 3,440 (1.36 PFLOP/s of bfloat16 products; a
// loop of nothing but these instructions reaches 1.45, ceilings.hip), 198, 495 and 60 us, and the same bits.
#define PARTS_STEPS 8  // of K whose parts a block of the first kernel makes

struct PartRows {  // a row's marks: bit r of [row tile][group of PARTS_STEPS steps]
  const uint32_t* flags;
  int groups;
};

// Eight values of a row at step `s`, turned with it, as their three parts in the matrix instruction's order; the largest of them, once scaled.
__device__ __forceinline__ float take_eight_apart(const float4v& x, const float4v& y, int s, bool live, uint4 (&part)[3]) {
  float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]}, largest = 0.f;
  const float scale = ((s + SPLIT_TURN) / (2 * SPLIT_TURN)) & 1 ? -SPLIT_SCALE : SPLIT_SCALE;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    v[e] = live ? v[e] * scale : 0.f;
    largest = fmaxf(largest, fabsf(v[e]));
  }
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      w[e] = pack2_bf16(v[2 * e], v[2 * e + 1]);
      v[2 * e] -= __uint_as_float(w[e] << 16), v[2 * e + 1] -= __uint_as_float(w[e] & 0xffff0000u);
    }
    part[p] = make_uint4(w[0], w[1], w[2], w[3]);
  }
  return largest;
}
// Bit r: the wavefront's lanes 16 j + r saw a value beyond the parts.
__device__ __forceinline__ uint32_t rows_beyond(float largest) {
  const unsigned long long over = __ballot(!(largest < SPLIT_LIMIT));
  return (uint32_t)((over | over >> 16 | over >> 32 | over >> 48) & 0xffffu);
}

// A block makes the parts of PARTS_STEPS steps of a row tile, each of its four wavefronts of two.  (A wavefront that took eight steps one after the
// other waited for its loads eight times: 4,096 x 256 10.7 us.)
__global__ void __launch_bounds__(256) f32_parts_kernel(const float* __restrict__ A, long lda, int M, int steps, uint4* __restrict__ parts, uint32_t* __restrict__ flags,
                                                        int groups) {
  constexpr int EACH = PARTS_STEPS / 4;
  __shared__ uint32_t beyond[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, j = lane >> 4;
  const int tile = blockIdx.x, first = blockIdx.y * PARTS_STEPS + wave * EACH;
  const int m = tile * 16 + r;
  const float* src = A + (size_t)min(m, M - 1) * lda + 8 * j;
  float4v x[EACH], y[EACH];
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    const float* from = src + 32 * min(first + i, steps - 1);
    x[i] = *(const float4v*)from, y[i] = *(const float4v*)(from + 4);
  }
  float largest = 0.f;
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    const int s = first + i;
    if (s >= steps) break;
    uint4 part[3];
    largest = fmaxf(largest, take_eight_apart(x[i], y[i], s, m < M, part));
#pragma unroll
    for (int p = 0; p < 3; ++p) parts[(((size_t)tile * steps + s) * 3 + p) * 64 + lane] = part[p];
  }
  const uint32_t over = rows_beyond(largest);
  if (lane == 0) beyond[wave] = over;
  __syncthreads();
  if (threadIdx.x == 0) flags[(size_t)tile * groups + blockIdx.y] = beyond[0] | beyond[1] | beyond[2] | beyond[3];
}

// ALONE: not 0: a K of up to so many steps, all of which fit the LDS, in one launch: a block makes the parts of its rows of A itself.  Bound by a
// launch and one trip to memory.  A kernel that took both operands apart, two launches, this, us: 4 rows of 1,024 x 32 4.6, 5.7, 3.7; of 2,048 x
// 64 5.3, 6.2, 4.0; of 512 x 256 9.1, 8.6, 7.0; 300 rows of 2,048 x 64 10.9, 8.2, 5.6.  And no scratch memory, and less of the host's time a call.
#define ALONE_STEPS 8
template <typename TC, int WM, int WAVES, int ALONE>
__global__ void __launch_bounds__(64 * WAVES, 2)
gemm_f32_parts_kernel(const unsigned char* __restrict__ parts, PartRows marks, const float* __restrict__ A, long lda, const float* __restrict__ W, long ldw,
                      TC* __restrict__ C, long ldc, const void* __restrict__ bias, int bias_dtype, int M, int N, int K, int row_blocks, int total) {
  constexpr int BM = 16 * WM, BN = 16 * WAVES;
  constexpr int A_STAGE = WM * 3 * 1024, W_STAGE = BN * 128;
  // steps of A under way or in use, and of W
  constexpr int SA = ALONE ? ALONE : 4 * A_STAGE + 6 * W_STAGE <= 160 * 1024 ? 4 : 3 * A_STAGE + 5 * W_STAGE <= 160 * 1024 ? 3 : 2;
  constexpr int SW = ALONE ? SA : SA + 2;
  constexpr int NA = (WM * 3 + WAVES - 1) / WAVES, NW = W_STAGE / 1024 / WAVES;  // a wavefront's loads a step
  static_assert(SA * A_STAGE + SW * W_STAGE <= 160 * 1024, "the steps fit the LDS");
  static_assert(WM % 2 == 0, "row tiles go in pairs");
  static_assert(!ALONE || WAVES % WM == 0, "a wavefront makes the parts of one row tile");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[SA * A_STAGE + SW * W_STAGE];
  const int run = (total + 7) >> 3, at = (int)(blockIdx.x & 7) * run + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= run || at >= total) return;
  const int m0 = at % row_blocks * BM, n0 = at / row_blocks * BN;
  const int lane = threadIdx.x & 63, r = lane & 15, j = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int steps = K / SPLIT_STEP, last = steps - 1, row_tiles = (M + 15) / 16;
  const uint32_t lds_a = (uint32_t)(uintptr_t)(&lds[0]), lds_w = lds_a + SA * A_STAGE;

  // this wavefront's loads: 1 KB pieces of A's operands (tiles past the last are the last again), eight rows of W each
  const unsigned char* a_src[NA];
  uint32_t a_dst[NA], w_off[NW];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int p = min(wave + WAVES * i, WM * 3 - 1), tile = min(m0 / 16 + p / 3, row_tiles - 1);
    a_src[i] = parts + ((size_t)tile * steps * 3 + p % 3) * 1024;
    a_dst[i] = p * 1024;
  }
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int row = 8 * (NW * wave + i) + (lane >> 3);
    w_off[i] = (uint32_t)((size_t)min(row, N - 1 - n0) * ldw * 4) + 16 * ((lane & 7) ^ ((row >> 1) & 7));
  }
  const float* w_src = W + (size_t)n0 * ldw;
  auto load_a = [&](int i, int step, int buf) { dma16((const bf16_t*)(a_src[i] + (size_t)step * 3072), lane * 16, lds_a + buf * A_STAGE + a_dst[i]); };
  auto load_w = [&](int i, int step, int buf) { dma16((const bf16_t*)(w_src + (size_t)step * 32), w_off[i], lds_w + buf * W_STAGE + (NW * wave + i) * 1024); };

  float largest = 0.f;
  // the wavefront's 16 rows of W of a step, taken apart
  const int w_row = (wave * 16 + r) * 128, w_key = (r >> 1) & 7;
  auto raw = [&](int buf, float4v& x, float4v& y) {
    const unsigned char* row = lds + SA * A_STAGE + buf * W_STAGE + w_row;
    x = *(const float4v*)(row + ((2 * j) ^ w_key) * 16);
    y = *(const float4v*)(row + ((2 * j + 1) ^ w_key) * 16);
  };
  auto take_apart = [&](float4v x, float4v y, Frag8 (&fw)[3]) {
    x *= SPLIT_SCALE, y *= SPLIT_SCALE;
    largest = fmaxf(fmaxf(fmaxf(fmaxf(largest, fabsf(x[0])), fabsf(x[1])), fabsf(x[2])), fabsf(x[3]));
    largest = fmaxf(fmaxf(fmaxf(fmaxf(largest, fabsf(y[0])), fabsf(y[1])), fabsf(y[2])), fabsf(y[3]));
#pragma unroll
    for (int part = 0; part < 3; ++part) {
      const uint32_t w0 = pack2_bf16(x[0], x[1]), w1 = pack2_bf16(x[2], x[3]), w2 = pack2_bf16(y[0], y[1]), w3 = pack2_bf16(y[2], y[3]);
      fw[part].u = make_uint4(w0, w1, w2, w3);
      if (part < 2) {
        x[0] -= __uint_as_float(w0 << 16), x[1] -= __uint_as_float(w0 & 0xffff0000u), x[2] -= __uint_as_float(w1 << 16), x[3] -= __uint_as_float(w1 & 0xffff0000u);
        y[0] -= __uint_as_float(w2 << 16), y[1] -= __uint_as_float(w2 & 0xffff0000u), y[2] -= __uint_as_float(w3 << 16), y[3] -= __uint_as_float(w3 & 0xffff0000u);
      }
    }
  };

  float4v acc[WM];
#pragma unroll
  for (int a = 0; a < WM; ++a) acc[a] = (float4v){0.f, 0.f, 0.f, 0.f};
  __shared__ uint32_t beyond[ALONE ? WAVES : 1];  // of the row tile whose parts a wavefront made
  if constexpr (ALONE) {
    for (int s = 0; s < steps; ++s)
#pragma unroll
      for (int i = 0; i < NW; ++i) load_w(i, s, s);
    const int tile = wave % WM, m = m0 + tile * 16 + r;
    const float* src = A + (size_t)min(m, M - 1) * lda + 8 * j;
    float most = 0.f;
    for (int s = wave / WM; s < steps; s += WAVES / WM) {
      uint4 part[3];
      most = fmaxf(most, take_eight_apart(*(const float4v*)(src + 32 * s), *(const float4v*)(src + 32 * s + 4), s, m < M, part));
#pragma unroll
      for (int p = 0; p < 3; ++p) *(uint4*)(lds + s * A_STAGE + (tile * 3 + p) * 1024 + lane * 16) = part[p];
    }
    const uint32_t over = rows_beyond(most);
    if (lane == 0) beyond[wave] = over;
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
  } else {
    // the loads in the order in which the waits below count them: step s of A with step s + 2 of W
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < NW; ++i) load_w(i, min(s, last), s);
#pragma unroll
    for (int s = 0; s < SA - 1; ++s) {
#pragma unroll
      for (int i = 0; i < NA; ++i) load_a(i, min(s, last), s);
#pragma unroll
      for (int i = 0; i < NW; ++i) load_w(i, min(s + 2, last), s + 2);
    }
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(NW + (SA - 2) * (NA + NW)) : "memory");
  }
  Frag8 fw[3], fn[3];
  {
    float4v x, y;
    raw(0, x, y);
    take_apart(x, y, fw);
  }
  float sign = 1.f;
  int a_buf = 0, w_buf = 0;  // of the step that is multiplied
  for (int k = 0; k < steps; ++k) {
    // this wavefront's loads of this step of A and the next of W have landed and it has left the step before; after the barrier
    // so has everyone
    if constexpr (!ALONE) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(NW + (SA - 2) * (NA + NW)) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    const int a_free = a_buf == 0 ? SA - 1 : a_buf - 1, w_free = w_buf == 0 ? SW - 1 : w_buf - 1;
    const int w_next = ALONE ? min(k + 1, last) : w_buf + 1 == SW ? 0 : w_buf + 1;
    if (k % (2 * SPLIT_TURN) == SPLIT_TURN) {
      sign = -sign;
#pragma unroll
      for (int a = 0; a < WM; ++a) acc[a] = -acc[a];
    }
    const unsigned char* st = lds + a_buf * A_STAGE + lane * 16;
    float4v x, y;
    raw(w_next, x, y);
    Frag8 fa[2][2][3];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int part = 0; part < 3; ++part) fa[0][u][part].u = *(const uint4*)(st + (u * 3 + part) * 1024);
#pragma unroll
    for (int p = 0; p < WM / 2; ++p) {
      if (p + 1 < WM / 2) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int part = 0; part < 3; ++part) fa[(p + 1) & 1][u][part].u = *(const uint4*)(st + ((2 * (p + 1) + u) * 3 + part) * 1024);
      }
      __builtin_amdgcn_sched_barrier(0);
      constexpr int PART_A[6] = {2, 0, 1, 1, 0, 0}, PART_W[6] = {0, 2, 1, 0, 1, 0};  // the smaller products first
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int u = 0; u < 2; ++u)
          acc[2 * p + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[PART_W[q]].v, fa[p & 1][u][PART_A[q]].v, acc[2 * p + u], 0, 0, 0);
      if (p == 0) take_apart(x, y, fn);
      // the loads of a step to come, a few after each pair
#pragma unroll
      for (int i = 0; i < NA + NW; ++i) {
        if (ALONE || i * (WM / 2) / (NA + NW) != p) continue;
        if (i < NA)
          load_a(i, min(k + SA - 1, last), a_free);
        else
          load_w(i - NA, min(k + SW - 1, last), w_free);
      }
    }
#pragma unroll
    for (int part = 0; part < 3; ++part) fw[part] = fn[part];
    a_buf = a_buf + 1 == SA ? 0 : a_buf + 1;
    w_buf = w_next;
  }
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");  // the loads past the last step; everyone has left the buffers

  // rows and columns with a value beyond the parts
  constexpr int WHOLE = 64 * 20 + BN * 20;  // floats of the tile of whole operands
  unsigned char* marked_rows = lds + WHOLE * 4;
  unsigned char* marked_columns = marked_rows + (BM + 63) / 64 * 64;
  uint32_t* any_of = (uint32_t*)(marked_columns + BN);
  largest = fmaxf(largest, __shfl_xor(largest, 16, CWM_WAVE));
  largest = fmaxf(largest, __shfl_xor(largest, 32, CWM_WAVE));
  const bool column = !(largest < SPLIT_LIMIT);
  if (j == 0) marked_columns[wave * 16 + r] = column;
  uint32_t rows = 0;  // of the row tiles wave, wave + WAVES, ...
#pragma unroll
  for (int t = 0; t < (WM + WAVES - 1) / WAVES; ++t) {
    const int tile = wave + WAVES * t;
    uint32_t f = 0;
    if constexpr (ALONE) {
#pragma unroll
      for (int w = 0; w < WAVES; ++w) f |= w % WM == tile ? beyond[w] : 0u;
    } else if (tile < WM && m0 / 16 + tile < row_tiles)
      for (int g = lane; g < marks.groups; g += 64) f |= marks.flags[(size_t)(m0 / 16 + tile) * marks.groups + g];
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) f |= __shfl_xor(f, off, CWM_WAVE);
    if (tile < WM && lane < 16) marked_rows[tile * 16 + lane] = (f >> lane) & 1;
    rows |= f;
  }
  if (lane == 0) any_of[wave] = rows;
  if (__any(column) && lane == 0) any_of[wave] = 1;
  __syncthreads();
  uint32_t any = 0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) any |= any_of[w];

  // lane 16 j + r of a tile holds row r, columns 4 j + i
  const int n = n0 + wave * 16 + 4 * j;
  float add[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    add[i] = 0.f;
    if (bias && n + i < N) add[i] = bias_dtype == CWM_BF16 ? bf16_to_f32(((const bf16_t*)bias)[n + i]) : ((const float*)bias)[n + i];
  }
  const bool whole = sizeof(TC) == 4 && any == 0 && ldc % 4 == 0 && ((uintptr_t)C & 15) == 0 && n + 3 < N;
#pragma unroll
  for (int a = 0; a < WM; ++a) {
    const int m = m0 + a * 16 + r;
    if (m >= M) continue;
    const float4v v = acc[a] * (sign * SPLIT_UNSCALE);
    if (whole) {
      *(float4*)((float*)C + (size_t)m * ldc + n) = make_float4(v[0] + add[0], v[1] + add[1], v[2] + add[2], v[3] + add[3]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n + i < N && !(any && (marked_rows[m - m0] | marked_columns[n + i - n0]))) Elem<TC>::store(C + (size_t)m * ldc + n + i, v[i] + add[i]);
    }
  }
  if (any) {
    for (int sub = 0; sub < BM && m0 + sub < M; sub += 64) {
      gemm_f32_tile<float, float, TC, 2, WAVES / 2, 1, 1, 16, true>(A, lda, W, ldw, C, ldc, bias, bias_dtype, min(M, m0 + BM), N, K, 1, 1, m0 + sub, n0, (float*)lds,
                                                            (float*)lds + 64 * 20, marked_rows + sub, marked_columns);
      __syncthreads();
    }
  }
}

template <typename TA, typename TW, typename TC>
static void launch(const void* A, long lda, const void* W, long ldw, void* C, long ldc, const void* bias,
                   int bias_dtype, int M, int N, int K, hipStream_t stream) {
  // 16-byte loads of four values where every row allows them
  const int vec_a = lda % 4 == 0 && ((uintptr_t)A % 16) == 0;
  const int vec_w = ldw % 4 == 0 && ((uintptr_t)W % 16) == 0;
  if (M > 32) {
    dim3 grid((N + 127) / 128, (M + 127) / 128);
    hipLaunchKernelGGL((gemm_f32_kernel<TA, TW, TC, 2, 2, 2, 2, 16>), grid, dim3(256), 0, stream, (const TA*)A, lda, (const TW*)W,
                       ldw, (TC*)C, ldc, bias, bias_dtype, M, N, K, vec_a, vec_w);
  } else {
    // few rows: one row tile, one wavefront a block and long steps, so that many blocks stream the
    // weight with much of it in flight
    dim3 grid((N + 31) / 32, 1);
    hipLaunchKernelGGL((gemm_f32_kernel<TA, TW, TC, 1, 1, 1, 1, 64>), grid, dim3(64), 0, stream, (const TA*)A, lda, (const TW*)W,
                       ldw, (TC*)C, ldc, bias, bias_dtype, M, N, K, vec_a, vec_w);
  }
}

extern "C" int cwm_gemm_f32(const void* A, int a_dtype, long lda, const void* W, int w_dtype, long ldw, void* C,
                            int c_dtype, long ldc, const void* bias, int bias_dtype, int M, int N, int K,
                            hipStream_t stream) {
  CWM_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  CWM_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gemm_f32: row strides shorter than rows");
  if (M == 0) return 0;
  CWM_REQUIRE((M + 127) / 128 <= 65535, "gemm_f32: M=%d has too many row tiles", M);
  const int key = (a_dtype << 2) | (w_dtype << 1) | c_dtype;
  switch (key) {
    case 0: launch<float, float, float>(A, lda, W, ldw, C, ldc, bias, bias_dtype, M, N, K, stream); break;
    case 1: launch<float, float, bf16_t>(A, lda, W, ldw, C, ldc, bias, bias_dtype, M, N, K, stream); break;
    case 2: launch<float, bf16_t, float>(A, lda, W, ldw, C, ldc, bias, bias_dtype, M, N, K, stream); break;
    case 3: launch<float, bf16_t, bf16_t>(A, lda, W, ldw, C, ldc, bias, bias_dtype, M, N, K, stream); break;
    case 4: launch<bf16_t, float, float>(A, lda, W, ldw, C, ldc, bias, bias_dtype, M, N, K, stream); break;
    case 5: launch<bf16_t, float, bf16_t>(A, lda, W, ldw, C, ldc, bias, bias_dtype, M, N, K, stream); break;
    case 6: launch<bf16_t, bf16_t, float>(A, lda, W, ldw, C, ldc, bias, bias_dtype, M, N, K, stream); break;
    case 7: launch<bf16_t, bf16_t, bf16_t>(A, lda, W, ldw, C, ldc, bias, bias_dtype, M, N, K, stream); break;
    default: return cwm_fail("gemm_f32: unknown dtypes a=%d w=%d c=%d", a_dtype, w_dtype, c_dtype);
  }
  return cwm_launch_status("gemm_f32");
}

// The blocks of the product in parts, (row tiles, wavefronts), and what a step of one costs, us, with most of the chip busy: 743 rows,
// 128 steps.  Blocks of 64 columns and four wavefronts share a compute unit by two, and a step of both takes 0.64; taller ones of four
// wavefronts or short ones of eight were nowhere ahead.  30 and 60 rows of 4,096 x 4,096: 32 rows and 64 columns 55 and 57 us, 64 x 128 101 and 102.
struct PartsBlock {
  int row_tiles, waves;
  float step;
};
static const PartsBlock parts_blocks[] = {{16, 8, 2.05f}, {12, 8, 1.62f}, {10, 8, 1.44f}, {8, 8, 1.19f}, {6, 8, 1.03f}, {4, 8, 0.80f}, {2, 4, 0.44f}};
#define PARTS_BLOCKS 7
#define PARTS_ALONE -2  // the number that asks for the product in one launch (32 rows and 64 columns a block)
#define PARTS_ALONE_SHORT -3
static int parts_block(int M, int N) {
  int best = 0;
  float least = 0.f;
  for (int i = 0; i < PARTS_BLOCKS; ++i) {
    const PartsBlock& b = parts_blocks[i];
    const long blocks = (long)((M + 16 * b.row_tiles - 1) / (16 * b.row_tiles)) * ((N + 16 * b.waves - 1) / (16 * b.waves));
    const float us = b.waves == 4 && blocks > 256 ? (float)((blocks + 511) / 512) * 0.64f : (float)((blocks + 255) / 256) * b.step;
    if (i == 0 || us < least) best = i, least = us;
  }
  return best;
}
// float32 A and W, K a multiple of 32.  `scratch`: for every started 16 rows 3,072 bytes a step of 32 k and 4 every 256 k, 16-byte
// aligned; none with PARTS_ALONE.  `block`: -1, PARTS_ALONE, or the number of one of the list above (tests).
extern "C" int cwm_gemm_f32_parts(const void* A, long lda, const void* W, long ldw, void* C, int c_dtype, long ldc, const void* bias, int bias_dtype, int M, int N,
                                  int K, void* scratch, int block, hipStream_t stream) {
  CWM_REQUIRE(M > 0 && N > 0 && K > 0 && K % SPLIT_STEP == 0 && K <= SPLIT_MOST_K, "gemm_f32_parts: bad sizes M=%d N=%d K=%d", M, N, K);
  CWM_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gemm_f32_parts: row strides shorter than rows");
  CWM_REQUIRE(lda % 4 == 0 && ldw % 4 == 0 && ldw < (1L << 23) && ((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0 && ((uintptr_t)scratch % 16) == 0,
              "gemm_f32_parts: rows must be 16-byte aligned");
  CWM_REQUIRE(c_dtype == CWM_F32 || c_dtype == CWM_BF16, "gemm_f32_parts: unknown output dtype %d", c_dtype);
  const int row_tiles = (M + 15) / 16, steps = K / SPLIT_STEP, groups = (steps + PARTS_STEPS - 1) / PARTS_STEPS;
  unsigned char* parts = (unsigned char*)scratch;
  uint32_t* flags = (uint32_t*)(parts + (size_t)row_tiles * steps * 3072);
  CWM_REQUIRE(block == PARTS_ALONE ? steps <= ALONE_STEPS : scratch != nullptr && block >= -1, "gemm_f32_parts: K=%d takes two launches and scratch memory", K);
  if (block != PARTS_ALONE)
    hipLaunchKernelGGL(f32_parts_kernel, dim3((unsigned)row_tiles, (unsigned)groups), dim3(256), 0, stream, (const float*)A, lda, M, steps, (uint4*)parts, flags, groups);
  const PartRows marks = {flags, groups};
  if (block == -1) block = parts_block(M, N);
  if (block == PARTS_ALONE && steps <= ALONE_STEPS / 2) block = PARTS_ALONE_SHORT;  // two blocks a compute unit
#define CWM_PARTS(AT, WM, WAVES, ALONE)                                                                                                           \
  case AT: {                                                                                                                                      \
    const int row_blocks = (M + 16 * WM - 1) / (16 * WM), total = row_blocks * ((N + 16 * WAVES - 1) / (16 * WAVES));                             \
    if (c_dtype == CWM_F32)                                                                                                                       \
      hipLaunchKernelGGL((gemm_f32_parts_kernel<float, WM, WAVES, ALONE>), dim3((total + 7) / 8 * 8), dim3(64 * WAVES), 0, stream, parts, marks,  \
                         (const float*)A, lda, (const float*)W, ldw, (float*)C, ldc, bias, bias_dtype, M, N, K, row_blocks, total);               \
    else                                                                                                                                          \
      hipLaunchKernelGGL((gemm_f32_parts_kernel<bf16_t, WM, WAVES, ALONE>), dim3((total + 7) / 8 * 8), dim3(64 * WAVES), 0, stream, parts, marks, \
                         (const float*)A, lda, (const float*)W, ldw, (bf16_t*)C, ldc, bias, bias_dtype, M, N, K, row_blocks, total);              \
  } break;
  switch (block) {
    CWM_PARTS(0, 16, 8, 0)
    CWM_PARTS(1, 12, 8, 0)
    CWM_PARTS(2, 10, 8, 0)
    CWM_PARTS(3, 8, 8, 0)
    CWM_PARTS(4, 6, 8, 0)
    CWM_PARTS(5, 4, 8, 0)
    CWM_PARTS(6, 2, 4, 0)
    CWM_PARTS(PARTS_ALONE, 2, 4, ALONE_STEPS)
    CWM_PARTS(PARTS_ALONE_SHORT, 2, 4, ALONE_STEPS / 2)
    default: return cwm_fail("gemm_f32_parts: no block %d", block);
  }
#undef CWM_PARTS
  return cwm_launch_status("gemm_f32_parts");
}

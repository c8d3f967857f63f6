// C[M, N] = A[M, K] * W[N, K]^T (+ bias[N]) in float32 on the matrix cores
// (v_mfma_f32_32x32x2_f32: float32 operands, exact products, float32 sums; float32 operands with
// K a multiple of 32 and up to 65,536 in exact bfloat16 parts instead, see below): the matrix
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
// and 1.8e-6.  Bound by the matrix cores and the vector instructions that make the parts (times that add).  743 rows, float32
// operands and parts: 28,672 x 4,096 1,847 and 1,034 us (169 TFLOP/s of float32 products), 2,048 x 2,048 191 and 74 us; 64 rows
// 6,144 x 4,096 361 and 136 us; 32 rows 168 and 91 us.
// The parts are made on the way into LDS, so memory holds float32 as before.  Both operands are multiplied by 2^23 first, and
// the sums by 2^-46 at the end, which rounds nothing: the last bit of the smallest float32 is then a normal bfloat16, so that the parts
// of small values are exact too (without it the third part is lost below 2^-110 and the second below 2^-118).  Rows of A and W with a
// value of 2^32 or more, or an infinity, are left to float32 operands, element by element of the result: with smaller ones the sums of
// up to 65,536 scaled products stay below 2^126.  So an element's order of k and of the parts depends on its own row and column alone.
// The bfloat16 instruction rounds its sums down, not to the nearest: left alone, every result is low by the same amount (2.5e-8, 1.0e-7
// and 4.1e-7 of the results' size at K = 512, 2,048 and 8,192), which adds up over a model's layers (16 layers of width 2,048: logits
// 2.9e-6 off float64 where float32 operands are 2.4e-6).  So the 8 steps in the middle of every 16 go into the sum with its sign turned,
// where rounding down is up: logits 2.0e-6 off, at the same times.
#define SPLIT_STEP 32
#define SPLIT_LD (SPLIT_STEP + 8)      // a row of a part in LDS: 80 bytes, so that 16 rows' pieces lie in different banks
#define SPLIT_MOST_K 65536
#define SPLIT_SCALE 8388608.0f               // 2^23
#define SPLIT_UNSCALE 1.4210854715202004e-14f  // 2^-46
#define SPLIT_TURN 4                         // steps after which the sum's sign turns, and 8 later again, of every 16
#define SPLIT_LIMIT 3.602879701896397e16f    // 2^55: 2^32 once scaled

typedef __bf16 bf16_pair __attribute__((ext_vector_type(2)));
// c plus the product of two pairs of bfloat16 values (v_dot2_f32_bf16); with (-1, 0) or (0, -1) for `by`: c less one of the pair
__device__ __forceinline__ float plus_pairs(uint32_t pair, uint32_t by, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16_pair, pair), __builtin_bit_cast(bf16_pair, by), c, false);
}

// WAVES_M x WAVES_N wavefronts, each with TM x TN tiles of 16 x 16.  PAIRS: a value less its part in one instruction instead of two.
// It has the shorter chain and the lower rate, so it pays where blocks wait for themselves: with 64 x 128 blocks and 300 rows of 4,096 x
// 14,336 (160 blocks) 487 us and 504, 743 rows of 2,048 x 2,048 (192) 76 and 87, but 743 rows of 6,144 x 4,096 (576) 306 and 295.
template <typename TC, int WAVES_M, int WAVES_N, int TM, int TN, bool PAIRS>
__global__ void __launch_bounds__(64 * WAVES_M * WAVES_N, TM * TN <= 8 ? 3 : 2)
gemm_f32_split_kernel(const float* __restrict__ A, long lda, const float* __restrict__ W, long ldw, TC* __restrict__ C, long ldc,
                      const void* __restrict__ bias, int bias_dtype, int M, int N, int K, int row_blocks, int total) {
  constexpr int BM = 16 * TM * WAVES_M, BN = 16 * TN * WAVES_N, THREADS = 64 * WAVES_M * WAVES_N;
  constexpr int A_LOADS = BM * (SPLIT_STEP / 4) / THREADS, W_LOADS = BN * (SPLIT_STEP / 4) / THREADS;
  constexpr int PARTS_BYTES = 3 * (BM + BN) * SPLIT_LD * 2, WHOLE_BYTES = (BM + BN) * (16 + 4) * 4;
  __shared__ __attribute__((aligned(16))) unsigned char lds[PARTS_BYTES > WHOLE_BYTES ? PARTS_BYTES : WHOLE_BYTES];
  __shared__ unsigned char marked_rows[BM], marked_columns[BN];
  bf16_t* a_parts = (bf16_t*)lds;                  // [3][BM][SPLIT_LD]
  bf16_t* w_parts = a_parts + 3 * BM * SPLIT_LD;   // [3][BN][SPLIT_LD]
  // an XCD gets a run of neighbours, the row blocks of a panel of W one after the other: its L2 reads the panel once
  const int run = (total + 7) >> 3, at = (int)(blockIdx.x & 7) * run + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= run || at >= total) return;
  const int m0 = at % row_blocks * BM, n0 = at / row_blocks * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, j = lane >> 4;
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  // piece f of a step: row f / 8, values 4 (f % 8) .. + 3; rows past the last are read from the last, their results not written
  const float* src_a[A_LOADS];
  const float* src_w[W_LOADS];
#pragma unroll
  for (int i = 0; i < A_LOADS; ++i) src_a[i] = A + (size_t)min(m0 + (tid + i * THREADS) / 8, M - 1) * lda + 4 * (tid & 7);
#pragma unroll
  for (int i = 0; i < W_LOADS; ++i) src_w[i] = W + (size_t)min(n0 + (tid + i * THREADS) / 8, N - 1) * ldw + 4 * (tid & 7);
  // two steps of operands on their way: what is fetched while step k is multiplied goes into LDS before step k + 2
  float4v ra[2][A_LOADS], rw[2][W_LOADS];
  auto fetch = [&](int set, int k) {
    const int k0 = min(k, K - SPLIT_STEP);
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) ra[set][i] = *(const float4v*)(src_a[i] + k0);
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) rw[set][i] = *(const float4v*)(src_w[i] + k0);
  };
  // (-1, 0) and (0, -1), in registers: as an inline constant the instruction reads -1.0 as something else
  uint32_t less_first = 0x0000bf80u, less_second = 0xbf800000u;
  asm("" : "+v"(less_first), "+v"(less_second));
  float largest_a[A_LOADS] = {}, largest_w[W_LOADS] = {};  // of a thread's pieces, which are the same rows' in every step
  float sign = 1.f;  // of the sums, and so of A's parts
  auto stage = [&](float4v v, float scale, bf16_t* parts, int plane, int f, float& largest) {
    v *= scale;
    if constexpr (TM * TN > 8)  // two instructions, or three in a shorter chain
      largest = fmaxf(fmaxf(fmaxf(fmaxf(largest, fabsf(v[0])), fabsf(v[1])), fabsf(v[2])), fabsf(v[3]));
    else
      largest = fmaxf(largest, fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
    bf16_t* to = parts + (f / 8) * SPLIT_LD + 4 * (f % 8);
#pragma unroll
    for (int part = 0; part < 3; ++part) {
      const uint32_t lo = pack2_bf16(v[0], v[1]), hi = pack2_bf16(v[2], v[3]);
      *(uint2*)(to + part * plane) = make_uint2(lo, hi);
      // what is left, exactly
      if constexpr (PAIRS) {
        v[0] = plus_pairs(lo, less_first, v[0]), v[1] = plus_pairs(lo, less_second, v[1]);
        v[2] = plus_pairs(hi, less_first, v[2]), v[3] = plus_pairs(hi, less_second, v[3]);
      } else {
        v[0] -= __uint_as_float(lo << 16), v[1] -= __uint_as_float(lo & 0xffff0000u);
        v[2] -= __uint_as_float(hi << 16), v[3] -= __uint_as_float(hi & 0xffff0000u);
      }
    }
  };
  float4v acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b) acc[a][b] = (float4v){0.f, 0.f, 0.f, 0.f};
  auto step = [&](int set, int next) {
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) stage(ra[set][i], sign * SPLIT_SCALE, a_parts, BM * SPLIT_LD, tid + i * THREADS, largest_a[i]);
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) stage(rw[set][i], SPLIT_SCALE, w_parts, BN * SPLIT_LD, tid + i * THREADS, largest_w[i]);
    __syncthreads();
    fetch(set, next);
    Frag8 fa[3][TM];
#pragma unroll
    for (int part = 0; part < 3; ++part)
#pragma unroll
      for (int a = 0; a < TM; ++a) fa[part][a].u = *(const uint4*)(a_parts + (part * BM + (wm * TM + a) * 16 + r) * SPLIT_LD + 8 * j);
#pragma unroll
    for (int b = 0; b < TN; ++b) {
      Frag8 fw[3];
#pragma unroll
      for (int part = 0; part < 3; ++part) fw[part].u = *(const uint4*)(w_parts + (part * BN + (wn * TN + b) * 16 + r) * SPLIT_LD + 8 * j);
      constexpr int PART_A[6] = {2, 0, 1, 1, 0, 0}, PART_W[6] = {0, 2, 1, 0, 1, 0};  // the smaller products first
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int a = 0; a < TM; ++a) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[PART_W[q]].v, fa[PART_A[q]][a].v, acc[a][b], 0, 0, 0);
    }
    __syncthreads();
  };
  fetch(0, 0);
  fetch(1, SPLIT_STEP);
  int k0 = 0;
  for (; k0 + 2 * SPLIT_STEP <= K; k0 += 2 * SPLIT_STEP) {
    if (k0 / SPLIT_STEP % (2 * SPLIT_TURN) == SPLIT_TURN) {
      sign = -sign;
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[a][b] = -acc[a][b];
    }
    step(0, k0 + 2 * SPLIT_STEP);
    step(1, k0 + 3 * SPLIT_STEP);
  }
  if (k0 < K) step(0, K);
  float largest = 0.f;
#pragma unroll
  for (int i = 0; i < A_LOADS; ++i) largest = fmaxf(largest, largest_a[i]);
#pragma unroll
  for (int i = 0; i < W_LOADS; ++i) largest = fmaxf(largest, largest_w[i]);
  const bool any = __syncthreads_or(!(largest < SPLIT_LIMIT));
  if (any) {
    // eight neighbouring threads have a row's pieces
    auto mark = [&](float largest, unsigned char* marks, int f) {
#pragma unroll
      for (int off = 1; off < 8; off <<= 1) largest = fmaxf(largest, __shfl_xor(largest, off, CWM_WAVE));
      if ((f & 7) == 0) marks[f / 8] = !(largest < SPLIT_LIMIT);
    };
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) mark(largest_a[i], marked_rows, tid + i * THREADS);
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) mark(largest_w[i], marked_columns, tid + i * THREADS);
    __syncthreads();
  }
  // lane 16 j + r of a tile holds row r, columns 4 j + i
#pragma unroll
  for (int b = 0; b < TN; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = n0 + (wn * TN + b) * 16 + 4 * j + i;
      if (n >= N) continue;
      float add = 0.f;
      if (bias) add = bias_dtype == CWM_BF16 ? bf16_to_f32(((const bf16_t*)bias)[n]) : ((const float*)bias)[n];
#pragma unroll
      for (int a = 0; a < TM; ++a) {
        const int m = m0 + (wm * TM + a) * 16 + r;
        if (any && (marked_rows[m - m0] | marked_columns[n - n0])) continue;
        if (m < M) Elem<TC>::store(C + (size_t)m * ldc + n, acc[a][b][i] * (sign * SPLIT_UNSCALE) + add);
      }
    }
  if (any) {
    constexpr int WHOLE_M = BM / 32, WHOLE_N = BN / 32;
    gemm_f32_tile<float, float, TC, WAVES_M, WAVES_N, WHOLE_M / WAVES_M, WHOLE_N / WAVES_N, 16, true>(
        A, lda, W, ldw, C, ldc, bias, bias_dtype, M, N, K, 1, 1, m0, n0, (float*)lds, (float*)lds + BM * 20, marked_rows, marked_columns);
  }
}

template <typename TC>
static void launch_split(const float* A, long lda, const float* W, long ldw, TC* C, long ldc, const void* bias, int bias_dtype, int M, int N, int K,
                         hipStream_t stream) {
#define CWM_SPLIT(WAVES_M, WAVES_N, TM, TN, PAIRS)                                                                                          \
  do {                                                                                                                                     \
    const int row_blocks = (M + 16 * TM * WAVES_M - 1) / (16 * TM * WAVES_M), total = row_blocks * ((N + 16 * TN * WAVES_N - 1) / (16 * TN * WAVES_N)); \
    hipLaunchKernelGGL((gemm_f32_split_kernel<TC, WAVES_M, WAVES_N, TM, TN, PAIRS>), dim3((total + 7) / 8 * 8), dim3(64 * WAVES_M * WAVES_N), 0, stream, A,   \
                       lda, W, ldw, C, ldc, bias, bias_dtype, M, N, K, row_blocks, total);                                                \
  } while (0)
  const long wide = (long)((M + 127) / 128) * ((N + 127) / 128);
  if (M <= 32)
    CWM_SPLIT(1, 2, 2, 2, true);
  else if (M <= 64 || wide < 512)  // too few blocks of 128 x 128 for two a compute unit
    if ((long)((M + 63) / 64) * ((N + 127) / 128) <= 256) CWM_SPLIT(2, 2, 2, 4, true); else CWM_SPLIT(2, 2, 2, 4, false);
  else
    CWM_SPLIT(2, 2, 4, 4, false);
#undef CWM_SPLIT
}

template <typename TA, typename TW, typename TC>
static void launch(const void* A, long lda, const void* W, long ldw, void* C, long ldc, const void* bias,
                   int bias_dtype, int M, int N, int K, hipStream_t stream) {
  // 16-byte loads of four values where every row allows them
  const int vec_a = lda % 4 == 0 && ((uintptr_t)A % 16) == 0;
  const int vec_w = ldw % 4 == 0 && ((uintptr_t)W % 16) == 0;
  if constexpr (sizeof(TA) == 4 && sizeof(TW) == 4) {
    if (vec_a && vec_w && K % SPLIT_STEP == 0 && K <= SPLIT_MOST_K) {  // whatever M is: a row's result does not depend on the others
      launch_split<TC>((const float*)A, lda, (const float*)W, ldw, (TC*)C, ldc, bias, bias_dtype, M, N, K, stream);
      return;
    }
  }
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

// A layer's own input from the token: every token has a second embedding row of which each layer reads its part e
// (side_dim values), gated by the residual and added to it after a norm,
//   g = gelu_tanh(W_gate x) * e;   y = W_proj g;   x <- x + y / sqrt(mean(y^2) + eps) * n
// with x the float32 residual [T, D], W_gate [side_dim, D], W_proj [D, side_dim] (handed over transposed, a row a side
// value, so that neighbouring threads read neighbouring elements), n [D].  side_dim is small (tens), so
// the two products are a few dot products a token: one block a token keeps the row of x in LDS, its wavefronts take
// the gate's outputs in turn (a dot product over D each, added up by shuffles in a fixed order), then every thread
// makes elements of y from the side_dim gated values, the block adds up their squares, and the scaled row goes into
// the residual (several tokens a block where the step has many, so that the matrices are read once for all of them).
// `round_inputs`: x and g are rounded to bfloat16 before they enter their products, as a model does
// that keeps its activations in bfloat16; the sums, the activation and the norm are float32 either way.
#include "common.h"
#include <type_traits>

CWM_DEFINE_ERROR_API

#define SIDE_THREADS 1024
#define SIDE_MAX_DIM 256    // side_dim
#define SIDE_MAX_WIDTH 15360
#define SIDE_LDS_LIMIT 61440
#define SIDE_GATE_ROWS 4   // rows of the gate that a wavefront reads side by side
#define SIDE_MAX_ADDENDS 4

// What is still to be added to the residual before the input is made (the layer's sublayers' results): each addend a
// [T, D] tensor (rows may lie apart) or float32 partial sums [P, T, D], times a constant; added in their order, in
// float32, the partial sums of an addend first among themselves, as the layer norm kernel adds them.
struct SideAddend {
  const void* ptr;
  long ld;              // elements between rows
  long partial_stride;  // elements between partial sums
  int n_partials;
  int dtype;
  float scale;
};

struct SideAddends {
  SideAddend a[SIDE_MAX_ADDENDS];
  int n;
};

// Which tokens a launch serves, where a step holds portions of both kinds: those of portions of at least SIDE_TILE_FROM tokens
// go to the matrix cores, the others to the kernel without them, so that a token's bits do not depend on the rest of the step.
#define SIDE_TILE_FROM 256
struct SidePortions {
  const int* seq_of_token;  // null: every token of the step is served
  const int* cu_q;
  __device__ __forceinline__ bool serves(int t, int n_tokens, bool tiles) const {
    if (t >= n_tokens) return false;
    if (!seq_of_token) return true;
    const int b = seq_of_token[t];
    return (cu_q[b + 1] - cu_q[b] >= SIDE_TILE_FROM) == tiles;
  }
};

extern "C" int cwm_token_side_tile_from() { return SIDE_TILE_FROM; }

extern "C" int cwm_token_side_max_addends() { return SIDE_MAX_ADDENDS; }

extern "C" int cwm_token_side_max_dim() { return SIDE_MAX_DIM; }
extern "C" int cwm_token_side_max_width() { return SIDE_MAX_WIDTH; }

__device__ __forceinline__ float side_round(float v, bool round) { return round ? bf16_to_f32(f32_to_bf16(v)) : v; }

template <typename T> struct SideVec;
template <> struct SideVec<bf16_t> {
  static constexpr int N = 8;  // elements of a 16-byte load
  static __device__ __forceinline__ void load(const bf16_t* p, float (&v)[8]) {
    const uint4 x = *(const uint4*)p;
    v[0] = __uint_as_float(x.x << 16), v[1] = __uint_as_float(x.x & 0xffff0000u);
    v[2] = __uint_as_float(x.y << 16), v[3] = __uint_as_float(x.y & 0xffff0000u);
    v[4] = __uint_as_float(x.z << 16), v[5] = __uint_as_float(x.z & 0xffff0000u);
    v[6] = __uint_as_float(x.w << 16), v[7] = __uint_as_float(x.w & 0xffff0000u);
  }
};
template <> struct SideVec<float> {
  static constexpr int N = 4;
  static __device__ __forceinline__ void load(const float* p, float (&v)[4]) {
    const float4 x = *(const float4*)p;
    v[0] = x.x, v[1] = x.y, v[2] = x.z, v[3] = x.w;
  }
};

// TOK tokens a block: the two matrices are read once for all of them.  The gate's rows are dealt to the block's
// wavefronts, which read them 16 bytes a lane; every sum runs in one order whatever TOK is.
template <typename TW, int TOK>
__device__ __forceinline__ void
token_side_rows(const int block, float* __restrict__ h, const int* __restrict__ tokens, const TW* __restrict__ table, long table_ld,
                  int column0, const TW* __restrict__ w_gate, const TW* __restrict__ w_proj_t, const float* __restrict__ weight,
                  int n_tokens, int dim, int side_dim, int vocab, float eps, bool round_inputs, SideAddends addends, SidePortions portions) {
  extern __shared__ __attribute__((aligned(16))) float rows[];  // [TOK][dim], then the gated values [TOK][side_dim]
  __shared__ float scratch[16];
  float* gated = rows + (size_t)TOK * dim;
  const int t0 = block * TOK;
  bool mine[TOK], any = false;
#pragma unroll
  for (int tok = 0; tok < TOK; ++tok) any |= mine[tok] = portions.serves(t0 + tok, n_tokens, false);
  if (!any) return;
  for (int e = threadIdx.x; e < TOK * dim; e += SIDE_THREADS) {
    const int tok = e / dim, el = e - tok * dim;
    const size_t t = (size_t)t0 + tok;
    float x = 0.f;
    bool serve = false;
#pragma unroll
    for (int i = 0; i < TOK; ++i) serve = tok == i ? mine[i] : serve;
    if (serve) {
      x = h[t * dim + el];
      for (int a = 0; a < addends.n; ++a) {
        const SideAddend& ad = addends.a[a];
        float y = 0.f;
        for (int p = 0; p < ad.n_partials; ++p) {
          const size_t at = (size_t)p * ad.partial_stride + t * ad.ld + el;
          y += ad.dtype == CWM_F32 ? ((const float*)ad.ptr)[at] : bf16_to_f32(((const bf16_t*)ad.ptr)[at]);
        }
        x = fmaf(ad.scale, y, x);
      }
      if (addends.n > 0) h[t * dim + el] = x;  // read again at the end, after the block's barriers
    }
    rows[e] = side_round(x, round_inputs);
  }
  __syncthreads();
  const int lane = threadIdx.x & (CWM_WAVE - 1), wave = threadIdx.x / CWM_WAVE;
  constexpr int N = SideVec<TW>::N;
  const bool vec = dim % N == 0 && ((uintptr_t)w_gate % 16) == 0;
  // a wavefront takes SIDE_GATE_ROWS rows of the gate at a time, so that as many loads are in flight
  for (int k0 = wave * SIDE_GATE_ROWS; k0 < side_dim; k0 += (SIDE_THREADS / CWM_WAVE) * SIDE_GATE_ROWS) {
    float a[SIDE_GATE_ROWS][TOK];
#pragma unroll
    for (int kk = 0; kk < SIDE_GATE_ROWS; ++kk)
#pragma unroll
      for (int tok = 0; tok < TOK; ++tok) a[kk][tok] = 0.f;
    if (vec) {
      for (int e0 = lane * N; e0 < dim; e0 += CWM_WAVE * N) {
        float w[SIDE_GATE_ROWS][N];
#pragma unroll
        for (int kk = 0; kk < SIDE_GATE_ROWS; ++kk) SideVec<TW>::load(w_gate + (size_t)min(k0 + kk, side_dim - 1) * dim + e0, w[kk]);
#pragma unroll
        for (int tok = 0; tok < TOK; ++tok)
#pragma unroll
          for (int i = 0; i < N; ++i) {
            const float x = rows[tok * dim + e0 + i];
#pragma unroll
            for (int kk = 0; kk < SIDE_GATE_ROWS; ++kk) a[kk][tok] = fmaf(w[kk][i], x, a[kk][tok]);
          }
      }
    } else {
      for (int e = lane; e < dim; e += CWM_WAVE) {
#pragma unroll
        for (int kk = 0; kk < SIDE_GATE_ROWS; ++kk) {
          const float w = Elem<TW>::load(w_gate + (size_t)min(k0 + kk, side_dim - 1) * dim + e);
#pragma unroll
          for (int tok = 0; tok < TOK; ++tok) a[kk][tok] = fmaf(w, rows[tok * dim + e], a[kk][tok]);
        }
      }
    }
#pragma unroll
    for (int kk = 0; kk < SIDE_GATE_ROWS; ++kk) {
      const int k = k0 + kk;
#pragma unroll
      for (int tok = 0; tok < TOK; ++tok) {
        const float sum = wave_sum(a[kk][tok]);
        if (lane == 0 && k < side_dim && mine[tok]) {
          const float z = side_round(sum, round_inputs);
          const float gelu = 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
          const int token = tokens[t0 + tok];
          const bool known = token >= 0 && token < vocab;
          const float e_k = known ? Elem<TW>::load(table + (size_t)token * table_ld + column0 + k) : __uint_as_float(0x7fc00000u);
          gated[tok * side_dim + k] = side_round(gelu * e_k, round_inputs);
        }
      }
    }
  }
  __syncthreads();
  // y stays in registers: a thread's elements are e = threadIdx.x + i * SIDE_THREADS
  constexpr int MAXE = SIDE_MAX_WIDTH / SIDE_THREADS;
  float y[TOK][MAXE];
  float sq[TOK];
#pragma unroll
  for (int tok = 0; tok < TOK; ++tok) sq[tok] = 0.f;
#pragma unroll
  for (int i = 0; i < MAXE; ++i) {
    const int e = threadIdx.x + i * SIDE_THREADS;
#pragma unroll
    for (int tok = 0; tok < TOK; ++tok) y[tok][i] = 0.f;
    if (e < dim) {
#pragma unroll 8
      for (int k = 0; k < side_dim; ++k) {
        const float w = Elem<TW>::load(w_proj_t + (size_t)k * dim + e);
#pragma unroll
        for (int tok = 0; tok < TOK; ++tok) y[tok][i] = fmaf(w, gated[tok * side_dim + k], y[tok][i]);
      }
#pragma unroll
      for (int tok = 0; tok < TOK; ++tok) sq[tok] += y[tok][i] * y[tok][i];
    }
  }
#pragma unroll
  for (int tok = 0; tok < TOK; ++tok) {
    const float rstd = 1.0f / sqrtf(block_sum(sq[tok], scratch) / (float)dim + eps);
    if (mine[tok]) {
      float* hrow = h + (size_t)(t0 + tok) * dim;
#pragma unroll
      for (int i = 0; i < MAXE; ++i) {
        const int e = threadIdx.x + i * SIDE_THREADS;
        if (e < dim) hrow[e] += y[tok][i] * rstd * weight[e];
      }
    }
  }
}

template <typename TW, int TOK>
__global__ void __launch_bounds__(SIDE_THREADS)
token_side_kernel(float* __restrict__ h, const int* __restrict__ tokens, const TW* __restrict__ table, long table_ld,
                  int column0, const TW* __restrict__ w_gate, const TW* __restrict__ w_proj_t, const float* __restrict__ weight,
                  int n_tokens, int dim, int side_dim, int vocab, float eps, bool round_inputs, SideAddends addends, SidePortions portions) {
  token_side_rows<TW, TOK>(blockIdx.x, h, tokens, table, table_ld, column0, w_gate, w_proj_t, weight, n_tokens, dim, side_dim, vocab, eps, round_inputs,
                           addends, portions);
}

// The same for bfloat16 weights whose inputs are rounded, on the matrix cores: TOK tokens a block of sixteen wavefronts.  The
// gate's product (16 tokens x side_dim, K = dim) is split over the wavefronts by columns and K, whose parts meet in LDS; the
// projection's (16 x dim, K = side_dim) by columns.  w_proj is [dim, side_dim] here.  The kernel above is bound by its
// multiply-adds and by LDS (every product's x and gated value is a read of its own): of width 2,048 with 64 side values and two
// addends, 1,500 tokens take it 88 us; here 21.  A block's stages follow one another (rows, gate's product, projection, each bound
// by its loads), so what can be asked for before a stage is: the tokens' values and the gate's first weights before the rows, the projection's
// before the gate's sums, the norm's before the squares; a row's pieces four at a time; the rows stay in LDS in float32 and are
// written once.  (38 us with a piece at a time, rows written and read again, and operands fetched a row a lane.)  Sixteen tokens a block, whose
// rows are bfloat16 in LDS and lie in the residual meanwhile: a token's sums have one order whatever TOK is.  Builds for short rows have no more
// loads than such a row has pieces and steps: a build for 2,048 took 256 tokens of width 512 12.1 us, of width 64 10.7, these 8.3 and 6.0.
// dim: a multiple of 64 and at most 256 MAXT; side_dim: a multiple of 32, at most SIDE_TILE_MAX; rows of h, the addends and the
// norm's weight start at multiples of 16 bytes (bfloat16 addends: of 8).
#define SIDE_TILE_MAX 128
#define SIDE_TURN_BYTES 1024  // an operand of 16 rows of 64 bytes
// bytes of LDS for `tok` tokens a block, whose rows stay there in float32 (`kept`) or, of bfloat16, for the gate's product alone
static inline size_t side_tile_lds(int tok, int dim, bool kept) {
  const int waves = SIDE_THREADS / CWM_WAVE, parts = 16 * tok * (int)sizeof(float);
  return (size_t)tok * (kept ? (dim + 4) * sizeof(float) : (dim + 8) * sizeof(bf16_t)) + (size_t)waves * (parts > SIDE_TURN_BYTES ? parts : SIDE_TURN_BYTES) +
         (size_t)tok * (SIDE_TILE_MAX + 8) * 2 + (size_t)waves * tok * sizeof(float);
}

// Tokens a block.  A block has a compute unit to itself beyond rows of 1,024 elements, so sixteen where eight would need a second round of blocks
// (64 side values, us with eight and sixteen: 2,500 tokens of width 1,024 28 and 19, of 2,048 42 and 31, of 4,096 82 and 57; 8,192 of 2,048 94 and
// 83), but not where three short rounds are less than two long ones (32 side values, 5,000 tokens of width 2,048 49 and 56); of the widest rows four
// where eight would leave more than half the chip idle (256 tokens of width 4,096 24.4 and 26.9; 1,000 tokens 35.3 and 36).
extern "C" int cwm_token_side_tile_tokens(int n_tokens, int dim, int side_dim) {
  if (side_dim <= 32 && dim > 1024 && n_tokens > 16 * 256 && n_tokens <= 24 * 256) return 8;
  if (n_tokens > 8 * 256) return 16;
  return dim > 3456 && n_tokens <= 4 * 256 ? 4 : 8;
}
extern "C" long cwm_token_side_tile_lds(int tok, int dim) { return (long)side_tile_lds(tok, dim, tok < 16); }

template <int TOK, int MAXT>
__device__ __forceinline__ void
token_side_tile(const int block, float* __restrict__ h, const int* __restrict__ tokens, const bf16_t* __restrict__ table, long table_ld, int column0,
                       const bf16_t* __restrict__ w_gate, const bf16_t* __restrict__ w_proj, const float* __restrict__ weight, int n_tokens,
                       int dim, int side_dim, int vocab, float eps, SideAddends addends, SidePortions portions) {
  extern __shared__ __attribute__((aligned(16))) unsigned char tile_lds[];
  constexpr int WAVES = SIDE_THREADS / CWM_WAVE, A_TOKEN = WAVES / TOK;  // wavefronts that load a token's row
  constexpr int AHEAD = MAXT <= 2 ? 2 * MAXT : MAXT == 4 && TOK == 16 ? 4 : 8;  // steps of the gate's product whose weights are in flight
  constexpr int RUN = MAXT <= 2 ? (MAXT * TOK + 15) / 16 : MAXT == 4 && TOK == 16 ? 2 : 4;  // pieces of a row that a thread has in flight
  constexpr int GATED = TOK * SIDE_TILE_MAX / SIDE_THREADS > 1 ? TOK * SIDE_TILE_MAX / SIDE_THREADS : 1;  // gated values a thread makes at most
  constexpr bool KEPT = TOK < 16;  // sixteen rows of float32 are more than the LDS holds
  typedef std::conditional_t<KEPT, float, bf16_t> Row;
  const int x_ld = dim + (KEPT ? 4 : 8);
  Row* xs = (Row*)tile_lds;                                      // [TOK][x_ld]
  // a wavefront's part of the gate's product, [16 side values][TOK], where its operands are turned before and after
  constexpr int PART = 16 * TOK * 4 > SIDE_TURN_BYTES ? 16 * TOK : SIDE_TURN_BYTES / 4;
  float* parts = (float*)(xs + (size_t)TOK * x_ld);
  bf16_t* gated = (bf16_t*)(parts + WAVES * PART);               // [TOK][SIDE_TILE_MAX + 8]
  float* squares = (float*)(gated + TOK * (SIDE_TILE_MAX + 8));  // [WAVES][TOK]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, j = lane >> 4;
  // A weight operand of 16 rows and 32 values is fetched four lanes a row (64 consecutive bytes) and turned to a lane's row through a place of
  // the wavefront's own in LDS: fetched as the instruction takes it, neighbouring lanes lie in 16 rows, which costs a lookup a lane.  A row's
  // four pieces change places with the row, so that no bank is met twice.
  unsigned char* turn = (unsigned char*)(parts + wave * PART);
  const int turn_row = lane >> 2, turn_piece = lane & 3;
  auto turned = [&](uint4 w) {
    Frag8 f;
    __builtin_amdgcn_wave_barrier();
    *(uint4*)(turn + turn_row * 64 + (turn_piece ^ (turn_row >> 2)) * 16) = w;
    __builtin_amdgcn_wave_barrier();
    f.u = *(const uint4*)(turn + r * 64 + (j ^ (r >> 2)) * 16);
    __builtin_amdgcn_wave_barrier();
    return f;
  };
  const int t0 = block * TOK;
  bool any = false;
#pragma unroll
  for (int tok = 0; tok < TOK; ++tok) any |= portions.serves(t0 + tok, n_tokens, true);
  if (!any) return;
  // what does not hang on the rows is asked for before them: the tokens' own values and the gate's first steps
  float own[GATED];
  {
    int token[GATED];
#pragma unroll
    for (int u = 0; u < GATED; ++u) token[u] = tokens[min(t0 + (int)(threadIdx.x + u * SIDE_THREADS) % TOK, n_tokens - 1)];
#pragma unroll
    for (int u = 0; u < GATED; ++u) {
      const int k = (threadIdx.x + u * SIDE_THREADS) / TOK;
      const bool known = token[u] >= 0 && token[u] < vocab;
      const bf16_t e_k = table[(size_t)(known ? token[u] : 0) * table_ld + column0 + min(k, side_dim - 1)];
      own[u] = known ? bf16_to_f32(e_k) : __uint_as_float(0x7fc00000u);
    }
  }
  // the gate's product: wavefront w has the side values 16 (w % columns) .. + 15 and part w / columns of K.  The wavefronts' parts lie
  // apart and each starts at a place of its own (of the column, not of the block, so that a sum has one order): rows lie a power of two
  // apart, and in step they would all ask the same few channels of the caches
  const int columns = side_dim / 16, k_parts = WAVES / columns, steps = dim / 32;
  const int gate_column = wave % columns, gate_part = wave / columns, part_steps = (steps + k_parts - 1) / k_parts;
  const int gate_from = min(gate_part * part_steps, steps - 1);
  const int gate_count = gate_part < k_parts ? max(min(part_steps, steps - gate_part * part_steps), 0) : 0;  // wavefronts left over have no part
  const int gate_start = gate_count > 0 ? 4 * gate_column % gate_count : 0;
  auto gate_step = [&](int u) {  // the u-th of the wavefront's steps
    const int v = u + gate_start;
    return gate_from + (v >= gate_count ? v - gate_count : v);
  };
  const bf16_t* gate_row = w_gate + (size_t)(16 * gate_column + turn_row) * dim + 8 * turn_piece;
  uint4 gate_w[AHEAD];
  auto fetch_gate = [&](int first) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      if (first + u < gate_count) gate_w[u] = *(const uint4*)(gate_row + 32 * gate_step(first + u));
  };
  fetch_gate(0);
  // 1. the rows: pending addends onto the residual, into LDS
  {
    const int tok = wave / A_TOKEN, t = t0 + tok;
    const bool serve = portions.serves(t, n_tokens, true);
    Row* x_row = xs + (size_t)tok * x_ld;
    const int e0 = 4 * ((wave % A_TOKEN) * CWM_WAVE + lane);
    for (int at = e0; at < dim; at += RUN * 4 * CWM_WAVE * A_TOKEN) {
      float4v x[RUN];
      int e[RUN];
#pragma unroll
      for (int u = 0; u < RUN; ++u) {
        e[u] = min(at + u * 4 * CWM_WAVE * A_TOKEN, dim - 4);  // a piece past the end: the row's last once more
        x[u] = (float4v){0.f, 0.f, 0.f, 0.f};
      }
      if (serve) {
#pragma unroll
        for (int u = 0; u < RUN; ++u) x[u] = *(const float4v*)(h + (size_t)t * dim + e[u]);
        for (int a = 0; a < addends.n; ++a) {
          const SideAddend& ad = addends.a[a];
          float4v y[RUN];
#pragma unroll
          for (int u = 0; u < RUN; ++u) y[u] = (float4v){0.f, 0.f, 0.f, 0.f};
          if (ad.dtype == CWM_F32) {
            for (int p = 0; p < ad.n_partials; ++p) {
              const float* from = (const float*)ad.ptr + (size_t)p * ad.partial_stride + (size_t)t * ad.ld;
#pragma unroll
              for (int u = 0; u < RUN; ++u) y[u] += *(const float4v*)(from + e[u]);
            }
          } else {
            const bf16_t* from = (const bf16_t*)ad.ptr + (size_t)t * ad.ld;
            uint2 w[RUN];
#pragma unroll
            for (int u = 0; u < RUN; ++u) w[u] = *(const uint2*)(from + e[u]);
#pragma unroll
            for (int u = 0; u < RUN; ++u)
              y[u] += (float4v){__uint_as_float(w[u].x << 16), __uint_as_float(w[u].x & 0xffff0000u), __uint_as_float(w[u].y << 16), __uint_as_float(w[u].y & 0xffff0000u)};
          }
#pragma unroll
          for (int u = 0; u < RUN; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) x[u][i] = fmaf(ad.scale, y[u][i], x[u][i]);
        }
      }
#pragma unroll
      for (int u = 0; u < RUN; ++u) {
        if constexpr (KEPT) {
          *(float4v*)(x_row + e[u]) = x[u];
        } else {
          if (at + u * 4 * CWM_WAVE * A_TOKEN >= dim) continue;  // (the row's last piece may have been written by its own thread before it was read here)
          if (serve && addends.n > 0) *(float4v*)(h + (size_t)t * dim + e[u]) = x[u];  // read again at the end, after the block's barriers
          *(uint2*)(x_row + e[u]) = make_uint2(pack2_bf16(x[u][0], x[u][1]), pack2_bf16(x[u][2], x[u][3]));
        }
      }
    }
  }
  __syncthreads();
  // 2. the gate's product
  {
    float4v acc = {0.f, 0.f, 0.f, 0.f};
    const Row* x_row = xs + (size_t)min(r, TOK - 1) * x_ld + 8 * j;
    for (int first = 0; first < gate_count; first += AHEAD) {
      uint4 now[AHEAD];
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) now[u] = gate_w[u];
      fetch_gate(first + AHEAD);
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        const int s = gate_step(first + u);
        if (first + u < gate_count) {
          Frag8 fx;
          if constexpr (KEPT) {
            const float4v a = *(const float4v*)(x_row + 32 * s), b = *(const float4v*)(x_row + 32 * s + 4);
            fx.u = make_uint4(pack2_bf16(a[0], a[1]), pack2_bf16(a[2], a[3]), pack2_bf16(b[0], b[1]), pack2_bf16(b[2], b[3]));
          } else {
            fx.u = *(const uint4*)(x_row + 32 * s);
          }
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(turned(now[u]).v, fx.v, acc, 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (r < TOK) parts[wave * PART + (4 * j + i) * TOK + r] = acc[i];
  }
  // the projection: wavefront w has the tiles w, w + 16, ... of 16 elements; its first weights are on their way past the barriers
  // (eight tiles at a time: with sixteen tiles' weights and results both in registers they spill)
  constexpr int GROUP = MAXT < 8 ? MAXT : 8;
  static_assert(MAXT % GROUP == 0, "whole groups of tiles");
  uint4 proj_w[GROUP];
  auto fetch_proj = [&](int q0, int k) {
#pragma unroll
    for (int q = 0; q < GROUP; ++q)
      proj_w[q] = *(const uint4*)(w_proj + (size_t)(min(16 * ((q0 + q) * WAVES + wave), dim - 16) + turn_row) * side_dim + k + 8 * turn_piece);
  };
  fetch_proj(0, 0);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < GATED; ++u) {
    const int id = threadIdx.x + u * SIDE_THREADS;
    if (id < TOK * side_dim) {
      const int tok = id % TOK, k = id / TOK;
      float sum = 0.f;
      for (int part = 0; part < k_parts; ++part) sum += parts[(part * columns + k / 16) * PART + k % 16 * TOK + tok];
      const float z = side_round(sum, true);
      const float gelu = 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
      gated[tok * (SIDE_TILE_MAX + 8) + k] = f32_to_bf16(gelu * own[u]);
    }
  }
  __syncthreads();
  // 3. the projection; its squares; the scaled row into the residual
  float4v y[MAXT];
#pragma unroll
  for (int q = 0; q < MAXT; ++q) y[q] = (float4v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q0 = 0; q0 < MAXT; q0 += GROUP)
    for (int k = 0; k < side_dim; k += 32) {
      Frag8 fg;
      fg.u = *(const uint4*)(gated + min(r, TOK - 1) * (SIDE_TILE_MAX + 8) + k + 8 * j);
#pragma unroll
      for (int q = 0; q < GROUP; ++q)
        if (16 * ((q0 + q) * WAVES + wave) < dim) y[q0 + q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(turned(proj_w[q]).v, fg.v, y[q0 + q], 0, 0, 0);
      const bool more = k + 32 < side_dim;
      fetch_proj(more ? q0 : min(q0 + GROUP, MAXT - GROUP), more ? k + 32 : 0);
    }
  float sq = 0.f;
#pragma unroll
  for (int q = 0; q < MAXT; ++q)
#pragma unroll
    for (int i = 0; i < 4; ++i) sq = fmaf(y[q][i], y[q][i], sq);
  sq += __shfl_xor(sq, 16, CWM_WAVE);
  sq += __shfl_xor(sq, 32, CWM_WAVE);
  if (j == 0 && r < TOK) squares[wave * TOK + r] = sq;
  float4v norm[GROUP];  // of the first group; the others' behind the barrier
#pragma unroll
  for (int q = 0; q < GROUP; ++q) norm[q] = *(const float4v*)(weight + min(16 * (q * WAVES + wave), dim - 16) + 4 * j);
  __syncthreads();
  if (r < TOK && (KEPT || portions.serves(t0 + r, n_tokens, true))) {
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) total += squares[w * TOK + r];
    const float rstd = 1.0f / sqrtf(total / (float)dim + eps);
    float* x_row;  // the row before the input: in LDS, or where the first stage has left it
    if constexpr (KEPT) x_row = xs + (size_t)r * x_ld;
    else x_row = h + (size_t)(t0 + r) * dim;
#pragma unroll
    for (int q = 0; q < MAXT; ++q) {
      const int e = 16 * (q * WAVES + wave) + 4 * j;
      if (e < dim) {
        const float4v n = q < GROUP ? norm[q % GROUP] : *(const float4v*)(weight + e);
        float4v x = *(const float4v*)(x_row + e);
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] += y[q][i] * rstd * n[i];
        *(float4v*)(x_row + e) = x;
      }
    }
  }
  if constexpr (!KEPT) return;
  __syncthreads();
  // whole rows, a wavefront 1 KB at a time
  const int tok = wave / A_TOKEN, t = t0 + tok;
  if (!portions.serves(t, n_tokens, true)) return;
  for (int e = 4 * ((wave % A_TOKEN) * CWM_WAVE + lane); e < dim; e += 4 * CWM_WAVE * A_TOKEN)
    *(float4v*)(h + (size_t)t * dim + e) = *(const float4v*)((const float*)xs + (size_t)tok * x_ld + e);
}

template <int TOK, int MAXT>
__global__ void __launch_bounds__(SIDE_THREADS)
token_side_tile_kernel(float* __restrict__ h, const int* __restrict__ tokens, const bf16_t* __restrict__ table, long table_ld, int column0,
                       const bf16_t* __restrict__ w_gate, const bf16_t* __restrict__ w_proj, const float* __restrict__ weight, int n_tokens,
                       int dim, int side_dim, int vocab, float eps, SideAddends addends, SidePortions portions) {
  token_side_tile<TOK, MAXT>(blockIdx.x, h, tokens, table, table_ld, column0, w_gate, w_proj, weight, n_tokens, dim, side_dim, vocab, eps, addends, portions);
}

// Both in one launch, for a step whose short portions hold few tokens: the first `tile_blocks` blocks take the long portions' tokens,
// then a block a token the short ones', beside them and not behind them.  1,006 and 48 tokens of width 3,072: 29.9 us,
// 28.1 of them the tiles alone; two launches 51.7.
#define SIDE_FEW 128
template <int TOK, int MAXT>
__global__ void __launch_bounds__(SIDE_THREADS)
token_side_both_kernel(float* __restrict__ h, const int* __restrict__ tokens, const bf16_t* __restrict__ table, long table_ld, int column0,
                       const bf16_t* __restrict__ w_gate, const bf16_t* __restrict__ w_proj, const bf16_t* __restrict__ w_proj_t,
                       const float* __restrict__ weight, int n_tokens, int dim, int side_dim, int vocab, float eps, SideAddends addends,
                       SidePortions portions, int tile_blocks) {
  if ((int)blockIdx.x < tile_blocks)
    token_side_tile<TOK, MAXT>(blockIdx.x, h, tokens, table, table_ld, column0, w_gate, w_proj, weight, n_tokens, dim, side_dim, vocab, eps, addends, portions);
  else
    token_side_rows<bf16_t, 1>(blockIdx.x - tile_blocks, h, tokens, table, table_ld, column0, w_gate, w_proj_t, weight, n_tokens, dim, side_dim, vocab, eps,
                               true, addends, portions);
}

// h: float32 [T, dim], changed in place.  Addend a (n_addends of them, or none): ptrs[a] of dtypes[a], rows lds[a]
// elements apart, n_partials[a] slabs partial_strides[a] elements apart, times scales[a]; they are added to h first.
// tokens: int32 [T].  table: [vocab, >= column0 + side_dim] of `w_dtype`, rows
// table_ld apart; w_gate [side_dim, dim] and w_proj_t [side_dim, dim] (the projection transposed) of `w_dtype`, contiguous;
// w_proj: the projection as [dim, side_dim], or null (then the matrix cores are not used);
// weight: float32 [dim].  seq_of_token, cu_q: the step's portions where some have SIDE_TILE_FROM tokens and more and some fewer,
// null where all tokens are one kind (then n_tokens stands for the portion); n_few: the tokens of the shorter ones.
extern "C" int cwm_token_side(float* h, const int* tokens, const void* table, long table_ld, int column0, const void* w_gate,
                              const void* w_proj_t, const void* w_proj, int w_dtype, const float* weight, int n_tokens, int dim, int side_dim, int vocab,
                              float eps, int round_inputs, int n_addends, const void* const* ptrs, const int* dtypes,
                              const long* lds_, const int* n_partials, const long* partial_strides, const float* scales,
                              const int* seq_of_token, const int* cu_q, int n_few, hipStream_t stream) {
  CWM_REQUIRE(n_tokens >= 0 && vocab >= 1 && column0 >= 0, "token_side: bad sizes");
  CWM_REQUIRE(dim >= 1 && dim <= SIDE_MAX_WIDTH, "token_side: rows of %d elements are outside 1..%d", dim, SIDE_MAX_WIDTH);
  CWM_REQUIRE(side_dim >= 1 && side_dim <= SIDE_MAX_DIM, "token_side: %d side values are outside 1..%d", side_dim, SIDE_MAX_DIM);
  CWM_REQUIRE(h && tokens && table && w_gate && w_proj_t && weight, "token_side: arguments missing");
  CWM_REQUIRE(eps > 0.f, "token_side: eps must be positive");
  CWM_REQUIRE(!seq_of_token == !cu_q, "token_side: the portions need both their lists");
  CWM_REQUIRE(n_addends >= 0 && n_addends <= SIDE_MAX_ADDENDS, "token_side: %d addends, at most %d are taken", n_addends, SIDE_MAX_ADDENDS);
  if (n_tokens == 0) return 0;
  SideAddends ad;
  ad.n = n_addends;
  for (int a = 0; a < n_addends; ++a) {
    CWM_REQUIRE(ptrs[a] && n_partials[a] >= 1, "token_side: addend %d is empty", a);
    CWM_REQUIRE(n_partials[a] == 1 || dtypes[a] == CWM_F32, "token_side: partial sums must be float32");
    ad.a[a] = SideAddend{ptrs[a], lds_[a], partial_strides[a], n_partials[a], dtypes[a], scales[a]};
  }
  // portions from SIDE_TILE_FROM tokens on (32 blocks of eight): with few the other kernel's blocks of one or two tokens spread over more of the chip (8 to
  // 64 tokens of width 2,048: 14.2 to 14.6 us against 15.8 to 16.1 in tiles; 128 to 255 tokens 21.9 to 22.5 against 16.3 to 16.6, so the line could lie
  // at 128; 300 tokens 40 against 16.7)
  bool tiled = n_tokens >= SIDE_TILE_FROM && w_proj && w_dtype == CWM_BF16 && round_inputs && dim % 64 == 0 && dim <= 4096 && side_dim % 32 == 0 && side_dim <= SIDE_TILE_MAX &&
               (((uintptr_t)h | (uintptr_t)w_gate | (uintptr_t)w_proj | (uintptr_t)weight) % 16) == 0;
  for (int a = 0; a < n_addends; ++a)
    tiled = tiled && lds_[a] % 4 == 0 && partial_strides[a] % 4 == 0 && ((uintptr_t)ptrs[a] % (dtypes[a] == CWM_F32 ? 16 : 8)) == 0;
  const SidePortions portions = {tiled ? seq_of_token : nullptr, cu_q};
  if (tiled) {
    const int tok = cwm_token_side_tile_tokens(n_tokens, dim, side_dim);
    const size_t lds_tile = side_tile_lds(tok, dim, tok < 16);
    const bool both = seq_of_token && n_few < SIDE_FEW;
    const size_t lds_row = sizeof(float) * ((size_t)dim + side_dim), lds = both && lds_row > lds_tile ? lds_row : lds_tile;
    const int tile_blocks = (n_tokens + tok - 1) / tok;
#define CWM_SIDE_TILE(TOK, MAXT)                                                                                                          \
  do {                                                                                                                                     \
    const void* kernel = both ? (const void*)token_side_both_kernel<TOK, MAXT> : (const void*)token_side_tile_kernel<TOK, MAXT>;           \
    if (lds > 65536) (void)hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                              \
    if (both)                                                                                                                              \
      hipLaunchKernelGGL((token_side_both_kernel<TOK, MAXT>), dim3(tile_blocks + n_tokens), dim3(SIDE_THREADS), lds, stream, h, tokens,     \
                         (const bf16_t*)table, table_ld, column0, (const bf16_t*)w_gate, (const bf16_t*)w_proj, (const bf16_t*)w_proj_t,    \
                         weight, n_tokens, dim, side_dim, vocab, eps, ad, portions, tile_blocks);                                          \
    else                                                                                                                                   \
      hipLaunchKernelGGL((token_side_tile_kernel<TOK, MAXT>), dim3(tile_blocks), dim3(SIDE_THREADS), lds, stream, h, tokens,                \
                         (const bf16_t*)table, table_ld, column0, (const bf16_t*)w_gate, (const bf16_t*)w_proj, weight, n_tokens, dim,      \
                         side_dim, vocab, eps, ad, portions);                                                                              \
  } while (0)
    if (tok == 4) CWM_SIDE_TILE(4, 16);
    else if (tok == 8 && dim <= 256) CWM_SIDE_TILE(8, 1);
    else if (tok == 8 && dim <= 512) CWM_SIDE_TILE(8, 2);
    else if (tok == 8 && dim <= 1024) CWM_SIDE_TILE(8, 4);
    else if (tok == 8 && dim <= 2048) CWM_SIDE_TILE(8, 8);
    else if (tok == 8) CWM_SIDE_TILE(8, 16);
    else if (dim <= 256) CWM_SIDE_TILE(16, 1);
    else if (dim <= 512) CWM_SIDE_TILE(16, 2);
    else if (dim <= 1024) CWM_SIDE_TILE(16, 4);
    else if (dim <= 2048) CWM_SIDE_TILE(16, 8);
    else CWM_SIDE_TILE(16, 16);
#undef CWM_SIDE_TILE
    if (!seq_of_token || both) return cwm_launch_status("token_side");
  }
  // tokens a block: as many (4, 2, 1) as fit the LDS and still leave the chip a block a few tokens
  const int served = tiled ? n_few : n_tokens;
  int tok = 4;
  while (tok > 1 && (sizeof(float) * (size_t)tok * (dim + side_dim) > SIDE_LDS_LIMIT || served < 64 * tok)) tok /= 2;
  CWM_REQUIRE(sizeof(float) * ((size_t)dim + side_dim) <= SIDE_LDS_LIMIT, "token_side: a row of %d and %d side values do not fit the LDS", dim, side_dim);
  const size_t lds = sizeof(float) * (size_t)tok * (dim + side_dim);
  const int blocks = (n_tokens + tok - 1) / tok;
#define CWM_SIDE_TOK(TW, TOK)                                                                                            \
  hipLaunchKernelGGL((token_side_kernel<TW, TOK>), dim3(blocks), dim3(SIDE_THREADS), lds, stream, h, tokens, (const TW*)table, \
                     table_ld, column0, (const TW*)w_gate, (const TW*)w_proj_t, weight, n_tokens, dim, side_dim, vocab, eps, round_inputs != 0, ad, portions)
#define CWM_SIDE(TW)                            \
  do {                                          \
    if (tok == 4) CWM_SIDE_TOK(TW, 4);          \
    else if (tok == 2) CWM_SIDE_TOK(TW, 2);     \
    else CWM_SIDE_TOK(TW, 1);                   \
  } while (0)
  if (w_dtype == CWM_F32) CWM_SIDE(float);
  else if (w_dtype == CWM_BF16) CWM_SIDE(bf16_t);
  else return cwm_fail("token_side: unknown element type %d", w_dtype);
#undef CWM_SIDE
#undef CWM_SIDE_TOK
  return cwm_launch_status("token_side");
}

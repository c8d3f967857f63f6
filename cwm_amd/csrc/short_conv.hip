// A short causal convolution over time on every channel, added to its own input: what a sublayer reads in place of h,
//   out_t = h_t + sum_(lag = 0 .. taps - 1) w[taps - 1 - lag] h_(t - lag)      element by element; the last tap is h_t's own
// where nothing (zero) precedes a sequence's first token.  Up to two such convolutions of the same input (two sublayers that read one
// norm's rows, each through weights of its own) are made in one pass.  The last taps - 1 inputs of a sequence are its
// state (float32 [taps - 1, D], oldest first; zero when the request is admitted), so a portion's first tokens find
// what the step before left.  `short_conv_kernel` (a thread a (token, channel)) only reads the state;
// `short_conv_state_kernel` (a thread a (sequence, channel)) replaces it afterwards, in the same stream, so no block
// waits for another.  In a step whose portions are all one token long (a decode step) the token's own thread is the
// only reader of its channel's state, and moves the rows up and appends its input itself: one launch.  Prompts in bfloat16 take
// `short_conv_runs_kernel`, one launch as well.  float32 arithmetic; the sum runs over the taps from the oldest to the newest.
#include "common.h"

CWM_DEFINE_ERROR_API

#define SCONV_THREADS 256
#define SCONV_MAX_TAPS 16

extern "C" int cwm_short_conv_max_taps() { return SCONV_MAX_TAPS; }

template <typename T>
__global__ void __launch_bounds__(SCONV_THREADS)
short_conv_kernel(const T* __restrict__ x, long x_ld, const float* __restrict__ w1, const float* __restrict__ w2,
                  T* __restrict__ out1, T* __restrict__ out2, float* __restrict__ state, long state_ld,
                  const int* __restrict__ slots, const int* __restrict__ cu_q, const int* __restrict__ seq_of_token,
                  int n_slots, int dim, int taps, bool update_inline) {
  const int t = blockIdx.x;
  const int d = blockIdx.y * SCONV_THREADS + threadIdx.x;
  if (d >= dim) return;
  const int b = seq_of_token[t];
  const int start = cu_q[b];
  const int slot = slots[b];
  float* srow = (state && slot >= 0 && slot < n_slots) ? state + (size_t)slot * state_ld : nullptr;
  const bool moves_state = update_inline && srow && cu_q[b + 1] - start == 1;  // then t == start, and tap j reads row j
  const float own = Elem<T>::load(x + (size_t)t * x_ld + d);
  float a1 = 0.f, a2 = 0.f;
  for (int j = 0; j < taps; ++j) {
    const int s = t - (taps - 1) + j;
    float v;
    if (s >= start)
      v = j == taps - 1 ? own : Elem<T>::load(x + (size_t)s * x_ld + d);
    else
      v = srow ? srow[(size_t)(taps - 1 + (s - start)) * dim + d] : 0.f;
    a1 = fmaf(w1[(size_t)j * dim + d], v, a1);
    if (w2) a2 = fmaf(w2[(size_t)j * dim + d], v, a2);
    if (moves_state && j >= 1) srow[(size_t)(j - 1) * dim + d] = v;  // row j - 1 was read in the round before
  }
  Elem<T>::store(out1 + (size_t)t * dim + d, own + a1);
  if (w2) Elem<T>::store(out2 + (size_t)t * dim + d, own + a2);
}

template <typename T>
__global__ void __launch_bounds__(SCONV_THREADS)
short_conv_state_kernel(const T* __restrict__ x, long x_ld, float* __restrict__ state, long state_ld,
                        const int* __restrict__ slots, const int* __restrict__ cu_q, int n_slots, int dim, int taps) {
  const int b = blockIdx.x;
  const int d = blockIdx.y * SCONV_THREADS + threadIdx.x;
  if (d >= dim) return;
  const int slot = slots[b];
  if (slot < 0 || slot >= n_slots) return;
  float* srow = state + (size_t)slot * state_ld;
  const int start = cu_q[b], n = cu_q[b + 1] - start;
  // row r of the new state is the input n - (taps - 1) + r of the portion, or, before the portion, row r + n of the
  // old state: rows are written in rising order, each after the higher row it may come from has been read
  for (int r = 0; r < taps - 1; ++r) {
    const int rel = n - (taps - 1) + r;
    const float v = rel >= 0 ? Elem<T>::load(x + (size_t)(start + rel) * x_ld + d) : srow[(size_t)(r + n) * dim + d];
    srow[(size_t)r * dim + d] = v;
  }
}

// Prompts in bfloat16, eight channels a thread: a unit of threads has SCONV_RUN consecutive tokens, whose rows and the TAPS - 1 before
// them it reads once, all in flight, and makes those that read no state; a further unit a sequence makes that sequence's first TAPS - 1
// tokens, which do, and then leaves the new state.  The sums run as above, so the bits are the same.  What bounded the kernel above was its loads, two
// bytes of every tap's row a thread: 1,500 tokens of 2,048, four taps, two convolutions 19.5 us and 4.0 for the state, 4,000 52.6; here 7.6 and 13.6 (18 and
// 31 MB: what is left is a launch and the way to memory).
#define SCONV_RUN 4
template <int TAPS, bool TWO>
__global__ void __launch_bounds__(SCONV_THREADS)
short_conv_runs_kernel(const bf16_t* __restrict__ x, long x_ld, const float* __restrict__ w1, const float* __restrict__ w2, bf16_t* __restrict__ out1,
                       bf16_t* __restrict__ out2, float* __restrict__ state, long state_ld, const int* __restrict__ slots, const int* __restrict__ cu_q,
                       const int* __restrict__ seq_of_token, int n_slots, int n_tokens, int n_seqs, int dim, bool write_state) {
  constexpr int HIST = TAPS - 1;
  const int per = dim / 8, at = blockIdx.x * SCONV_THREADS + threadIdx.x, runs = (n_tokens + SCONV_RUN - 1) / SCONV_RUN;
  int unit = at / per;
  const int c = 8 * (at - unit * per);
  if (unit >= runs + n_seqs) return;
  float wa[TAPS][8], wb[TWO ? TAPS : 1][8];
  auto eight = [](const float* p, float (&v)[8]) {
    const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
  };
#pragma unroll
  for (int j = 0; j < TAPS; ++j) {
    eight(w1 + (size_t)j * dim + c, wa[j]);
    if constexpr (TWO) eight(w2 + (size_t)j * dim + c, wb[j]);
  }
  auto leave = [&](int t, const float (&in)[TAPS][8]) {  // in: the oldest input first
    float a[8], b[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] = b[e] = 0.f;
#pragma unroll
    for (int j = 0; j < TAPS; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        a[e] = fmaf(wa[j][e], in[j][e], a[e]);
        if constexpr (TWO) b[e] = fmaf(wb[j][e], in[j][e], b[e]);
      }
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] = in[HIST][e] + a[e], b[e] = in[HIST][e] + b[e];
    *(uint4*)(out1 + (size_t)t * dim + c) = make_uint4(pack2_bf16(a[0], a[1]), pack2_bf16(a[2], a[3]), pack2_bf16(a[4], a[5]), pack2_bf16(a[6], a[7]));
    if constexpr (TWO)
      *(uint4*)(out2 + (size_t)t * dim + c) = make_uint4(pack2_bf16(b[0], b[1]), pack2_bf16(b[2], b[3]), pack2_bf16(b[4], b[5]), pack2_bf16(b[6], b[7]));
  };
  auto widen = [](const Frag8& f, float (&v)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = bf16_to_f32(f.h[e]);
  };
  if (unit < runs) {
    const int t0 = unit * SCONV_RUN;
    Frag8 rows[SCONV_RUN + HIST];
    int place[SCONV_RUN];
#pragma unroll
    for (int i = 0; i < SCONV_RUN + HIST; ++i) rows[i].u = *(const uint4*)(x + (size_t)max(0, min(t0 + i - HIST, n_tokens - 1)) * x_ld + c);
#pragma unroll
    for (int i = 0; i < SCONV_RUN; ++i) {
      const int t = min(t0 + i, n_tokens - 1);
      place[i] = t - cu_q[seq_of_token[t]];
    }
#pragma unroll
    for (int i = 0; i < SCONV_RUN; ++i) {
      if (t0 + i >= n_tokens || place[i] < HIST) continue;
      float in[TAPS][8];
#pragma unroll
      for (int j = 0; j < TAPS; ++j) widen(rows[i + j], in[j]);
      leave(t0 + i, in);
    }
    return;
  }
  unit -= runs;
  const int start = cu_q[unit], n = cu_q[unit + 1] - start, slot = slots[unit];
  if (n == 0) return;
  float* st = slot >= 0 && slot < n_slots ? state + (size_t)slot * state_ld + c : nullptr;
  // the state, then the portion's first HIST inputs (the last again where it has fewer)
  float in[2 * HIST][8];
#pragma unroll
  for (int r = 0; r < HIST; ++r) {
    Frag8 f;
    f.u = *(const uint4*)(x + (size_t)(start + min(r, n - 1)) * x_ld + c);
    widen(f, in[HIST + r]);
#pragma unroll
    for (int e = 0; e < 8; ++e) in[r][e] = 0.f;
    if (st) eight(st + (size_t)r * dim, in[r]);
  }
#pragma unroll
  for (int i = 0; i < HIST; ++i) {
    if (i >= n) continue;
    float taps[TAPS][8];
#pragma unroll
    for (int j = 0; j < TAPS; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) taps[j][e] = in[i + j][e];
    leave(start + i, taps);
  }
  if (!st || !write_state) return;
  // row r of the new state is the input n - HIST + r of the portion, or row r + n of what was
#pragma unroll
  for (int r = 0; r < HIST; ++r) {
    float v[8];
    if (n >= HIST) {
      Frag8 f;
      f.u = *(const uint4*)(x + (size_t)(start + n - HIST + r) * x_ld + c);
      widen(f, v);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = 0.f;
#pragma unroll
      for (int k = 1; k < HIST; ++k)
        if (n == k)
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = in[r + k][e];
    }
    *(float4*)(st + (size_t)r * dim) = make_float4(v[0], v[1], v[2], v[3]);
    *(float4*)(st + (size_t)r * dim + 4) = make_float4(v[4], v[5], v[6], v[7]);
  }
}

static long short_conv_runs_threads(int n_tokens, int n_seqs, int dim) { return (((long)n_tokens + SCONV_RUN - 1) / SCONV_RUN + n_seqs) * (dim / 8); }
// Whether a step's sizes go through the kernel of runs, whose threads are numbered in 31 bits; larger ones keep the kernels above
extern "C" int cwm_short_conv_in_runs(int n_tokens, int n_seqs, int taps, int dim) {
  return n_tokens > n_seqs && taps >= 2 && taps <= 4 && dim % 8 == 0 && short_conv_runs_threads(n_tokens, n_seqs, dim) < (1L << 31) - SCONV_THREADS;
}

// x: [T, dim] of `dtype`, rows x_ld elements apart.  w1 (and w2, or null): float32 [taps, dim], a row a tap, the last
// row the current token's.  out1 (and out2): contiguous [T, dim] of `dtype`.  state: float32 [n_slots, state_ld] with
// (taps - 1) * dim <= state_ld (null where taps == 1); slots: int32 [n_seqs]; cu_q: int32 [n_seqs + 1]; seq_of_token:
// int32 [T].  write_state 0: the state is read and left as it was; 1: replaced by a second launch; 2: every portion of
// the step is one token long, and the first launch moves the state itself.
extern "C" int cwm_short_conv(const void* x, long x_ld, int dtype, const float* w1, const float* w2, void* out1, void* out2,
                              float* state, long state_ld, const int* slots, const int* cu_q, const int* seq_of_token,
                              int n_slots, int n_tokens, int n_seqs, int dim, int taps, int write_state, hipStream_t stream) {
  CWM_REQUIRE(n_tokens >= 0 && n_seqs >= 0 && dim >= 1, "short_conv: bad sizes");
  CWM_REQUIRE(taps >= 1 && taps <= SCONV_MAX_TAPS, "short_conv: %d taps are outside 1..%d", taps, SCONV_MAX_TAPS);
  CWM_REQUIRE(x && w1 && out1 && (!w2 || out2) && slots && cu_q && seq_of_token, "short_conv: arguments missing");
  CWM_REQUIRE(taps == 1 || (state && state_ld >= (long)(taps - 1) * dim), "short_conv: the state does not hold %d rows of %d", taps - 1, dim);
  if (n_tokens == 0) return 0;
  const int gy = (dim + SCONV_THREADS - 1) / SCONV_THREADS;
  auto aligned = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  if (dtype == CWM_BF16 && write_state != 2 && cwm_short_conv_in_runs(n_tokens, n_seqs, taps, dim) && x_ld % 8 == 0 && state_ld % 4 == 0 && aligned(x) &&
      aligned(w1) && aligned(w2) && aligned(out1) && aligned(out2) && aligned(state)) {
    const dim3 grid((unsigned)((short_conv_runs_threads(n_tokens, n_seqs, dim) + SCONV_THREADS - 1) / SCONV_THREADS));
#define CWM_SCONV_RUNS(TAPS, TWO)                                                                                                             \
  hipLaunchKernelGGL((short_conv_runs_kernel<TAPS, TWO>), grid, dim3(SCONV_THREADS), 0, stream, (const bf16_t*)x, x_ld, w1, w2, (bf16_t*)out1, \
                     (bf16_t*)out2, state, state_ld, slots, cu_q, seq_of_token, n_slots, n_tokens, n_seqs, dim, write_state == 1)
    if (taps == 2 && w2) CWM_SCONV_RUNS(2, true);
    else if (taps == 2) CWM_SCONV_RUNS(2, false);
    else if (taps == 3 && w2) CWM_SCONV_RUNS(3, true);
    else if (taps == 3) CWM_SCONV_RUNS(3, false);
    else if (w2) CWM_SCONV_RUNS(4, true);
    else CWM_SCONV_RUNS(4, false);
#undef CWM_SCONV_RUNS
    return cwm_launch_status("short_conv");
  }
#define CWM_SCONV(T)                                                                                                       \
  do {                                                                                                                     \
    hipLaunchKernelGGL((short_conv_kernel<T>), dim3(n_tokens, gy), dim3(SCONV_THREADS), 0, stream, (const T*)x, x_ld, w1,   \
                       w2, (T*)out1, (T*)out2, state, state_ld, slots, cu_q, seq_of_token, n_slots, dim, taps,               \
                       write_state == 2);                                                                                   \
    if (write_state == 1 && taps > 1)                                                                                      \
      hipLaunchKernelGGL((short_conv_state_kernel<T>), dim3(n_seqs, gy), dim3(SCONV_THREADS), 0, stream, (const T*)x, x_ld, \
                         state, state_ld, slots, cu_q, n_slots, dim, taps);                                                 \
  } while (0)
  if (dtype == CWM_F32) CWM_SCONV(float);
  else if (dtype == CWM_BF16) CWM_SCONV(bf16_t);
  else return cwm_fail("short_conv: unknown element type %d", dtype);
#undef CWM_SCONV
  return cwm_launch_status("short_conv");
}

// The two sequential pieces of a selective state-space mixer, each going on from a per-request state.
//
//   causal convolution + SiLU, per channel c of a token t at place j of its sequence:
//       out[t][c] = silu(bias[c] + sum_k w[c][k] * in[j - (taps - 1 - k)][c]),   inputs before the sequence's start are 0;
//     a portion's first taps - 1 tokens read the inputs that the step before left in the state (oldest first),
//     and the portion leaves its own last taps - 1 inputs there.
//   the recurrence, per head h (group g = h / (heads / groups)), state S [N][P] in float32:
//       dt = softplus(dt_raw + dt_bias[h]);  a = exp(-exp(A_log[h]) * dt)
//       S <- a S + dt B_t x_t^T;   y_t = S^T C_t + D[h] x_t
//     with x_t [P], B_t and C_t [N] from the convolution's output row [x: heads * P | B: groups * N | C: groups * N].
//     A head's state lies in memory in the order its threads hold it (see the kernel), padded to 16 * split rows.
//
// Both are exact under any cut of a sequence into portions: a portion starts from the state as the previous one
// left it and performs the same operations in the same order as the whole sequence would.
#include "three_parts.h"
#include <type_traits>

CWM_DEFINE_ERROR_API

#define CONV_MAX_TAPS 8
#define SCAN_ROWS 16  // rows of the state that one thread holds

extern "C" int cwm_conv_max_taps() { return CONV_MAX_TAPS; }
extern "C" int cwm_scan_max_state() { return SCAN_ROWS * 16; }
// lanes that share a column of a head's state of N rows: 1, 2, 4, 8 or 16; the head's state takes SCAN_ROWS * split * P floats
extern "C" int cwm_scan_split(int N) {
  int split = 1;
  while (split * SCAN_ROWS < N) split <<= 1;
  return split;
}

__device__ __forceinline__ float silu_f32(float z) { return z / (1.f + expf(-z)); }

// The block of a sequence's first token in this step computes the first taps - 1 tokens of the portion (all that
// read the state) and then writes the new state, so reads and writes of one sequence's state stay in one thread
// per channel.  Blocks of the other tokens read inputs of this step only.
template <typename T>
__global__ void __launch_bounds__(256) conv_silu_kernel(const T* __restrict__ in, long in_ld, const float* __restrict__ w,
                                                        const float* __restrict__ bias, float* state, long state_ld, long state_off,
                                                        const int* __restrict__ slots, const int* __restrict__ cu_q,
                                                        const int* __restrict__ seq_of_token, T* __restrict__ out, int channels,
                                                        int taps, int n_slots) {
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  const int t = blockIdx.x, b = seq_of_token[t];
  const int first = cu_q[b];
  const int j = t - first;
  const int q = cu_q[b + 1] - first;
  const int hist = taps - 1;
  float wk[CONV_MAX_TAPS];
#pragma unroll
  for (int k = 0; k < CONV_MAX_TAPS; ++k) wk[k] = k < taps ? w[(size_t)c * taps + k] : 0.f;
  const float bc = bias[c];
  if (j >= hist) {
    float acc = bc;
#pragma unroll
    for (int k = 0; k < CONV_MAX_TAPS; ++k)
      if (k < taps) acc = fmaf(wk[k], Elem<T>::load(in + (size_t)(t - (hist - k)) * in_ld + c), acc);
    Elem<T>::store(out + (size_t)t * channels + c, silu_f32(acc));
    return;
  }
  if (j != 0) return;
  const int slot = slots[b];
  float* st = (slot >= 0 && slot < n_slots) ? state + (size_t)slot * state_ld + state_off : nullptr;
  float old[CONV_MAX_TAPS];  // old[m]: the input m places after the oldest one kept, m < hist
#pragma unroll
  for (int m = 0; m < CONV_MAX_TAPS; ++m) old[m] = (st && m < hist) ? st[(size_t)m * channels + c] : 0.f;
  // input at place i of the sequence as this step sees it: i < 0 lies in the state
  auto input = [&](int i) -> float {
    if (i >= 0) return Elem<T>::load(in + (size_t)(first + i) * in_ld + c);
    float v = 0.f;
#pragma unroll
    for (int m = 0; m < CONV_MAX_TAPS; ++m)
      if (m == hist + i) v = old[m];
    return v;
  };
  const int n_head = q < hist ? q : hist;
  for (int jj = 0; jj < n_head; ++jj) {
    float acc = bc;
#pragma unroll
    for (int k = 0; k < CONV_MAX_TAPS; ++k)
      if (k < taps) acc = fmaf(wk[k], input(jj - (hist - k)), acc);
    Elem<T>::store(out + (size_t)(first + jj) * channels + c, silu_f32(acc));
  }
  if (st) {
    float fresh[CONV_MAX_TAPS];
#pragma unroll
    for (int m = 0; m < CONV_MAX_TAPS; ++m) fresh[m] = m < hist ? input(q - hist + m) : 0.f;
#pragma unroll
    for (int m = 0; m < CONV_MAX_TAPS; ++m)
      if (m < hist) st[(size_t)m * channels + c] = fresh[m];
  }
}

// Portions of a prompt in bfloat16, eight channels a thread: a unit of threads has CONV_RUN consecutive tokens, whose rows and the TAPS - 1
// before them it reads once, all in flight, and makes those that read no state (place >= TAPS - 1 in their portion); a further unit a sequence
// makes the first TAPS - 1 tokens, which do, and then leaves the new state.  The sums run in the order of the kernel above.  A thread a (token, eight channels)
// for the former, which read every row TAPS times, and a launch of the kernel above for the latter took 21.7 and 5.3 us (2,048 tokens, 6,144
// channels, four taps); this takes 20.9, most of it the activation's exponential and division, 300 tokens 6.4 instead of 9.5.
// w_by_tap: the weights tap by tap ([taps][channels]): a thread's eight are 32 bytes, the threads' side by side.
#define CONV_RUN 4
template <int TAPS>
__global__ void __launch_bounds__(256) conv_silu_runs_kernel(const bf16_t* __restrict__ in, long in_ld, const float* __restrict__ w_by_tap,
                                                             const float* __restrict__ bias, float* __restrict__ state, long state_ld, long state_off,
                                                             const int* __restrict__ slots, const int* __restrict__ cu_q,
                                                             const int* __restrict__ seq_of_token, bf16_t* __restrict__ out, int n_tokens, int n_seqs,
                                                             int channels, int n_slots) {
  constexpr int HIST = TAPS - 1;
  const int per = channels / 8, at = blockIdx.x * 256 + threadIdx.x, runs = (n_tokens + CONV_RUN - 1) / CONV_RUN;
  int unit = at / per;
  const int c = 8 * (at - unit * per);
  if (unit >= runs + (HIST > 0 ? n_seqs : 0)) return;
  auto eight = [](const float* p, float (&v)[8]) {
    const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
  };
  float wk[TAPS][8], bc[8];
  eight(bias + c, bc);
#pragma unroll
  for (int k = 0; k < TAPS; ++k) eight(w_by_tap + (size_t)k * channels + c, wk[k]);
  auto leave = [&](int t, const float (&x)[TAPS][8]) {  // x: the oldest input first
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = bc[e];
#pragma unroll
    for (int k = 0; k < TAPS; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = fmaf(wk[k][e], x[k][e], acc[e]);
    uint4 o;
    o.x = pack2_bf16(silu_f32(acc[0]), silu_f32(acc[1]));
    o.y = pack2_bf16(silu_f32(acc[2]), silu_f32(acc[3]));
    o.z = pack2_bf16(silu_f32(acc[4]), silu_f32(acc[5]));
    o.w = pack2_bf16(silu_f32(acc[6]), silu_f32(acc[7]));
    *(uint4*)(out + (size_t)t * channels + c) = o;
  };
  auto widen = [](const Frag8& f, float (&v)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = bf16_to_f32(f.h[e]);
  };
  if (unit < runs) {
    const int t0 = unit * CONV_RUN;
    Frag8 rows[CONV_RUN + HIST];
    int place[CONV_RUN];
#pragma unroll
    for (int i = 0; i < CONV_RUN + HIST; ++i) rows[i].u = *(const uint4*)(in + (size_t)max(0, min(t0 + i - HIST, n_tokens - 1)) * in_ld + c);
#pragma unroll
    for (int i = 0; i < CONV_RUN; ++i) {
      const int t = min(t0 + i, n_tokens - 1);
      place[i] = t - cu_q[seq_of_token[t]];
    }
#pragma unroll
    for (int i = 0; i < CONV_RUN; ++i) {
      if (t0 + i >= n_tokens || place[i] < HIST) continue;
      float x[TAPS][8];
#pragma unroll
      for (int k = 0; k < TAPS; ++k) widen(rows[i + k], x[k]);
      leave(t0 + i, x);
    }
    return;
  }
  unit -= runs;
  const int start = cu_q[unit], n = cu_q[unit + 1] - start, slot = slots[unit];
  if (n == 0) return;
  float* st = slot >= 0 && slot < n_slots ? state + (size_t)slot * state_ld + state_off + c : nullptr;
  // the state, then the portion's first HIST inputs (the last again where it has fewer)
  float x[HIST > 0 ? 2 * HIST : 1][8];
#pragma unroll
  for (int m = 0; m < HIST; ++m) {
    Frag8 f;
    f.u = *(const uint4*)(in + (size_t)(start + min(m, n - 1)) * in_ld + c);
    widen(f, x[HIST + m]);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[m][e] = 0.f;
    if (st) eight(st + (size_t)m * channels, x[m]);
  }
#pragma unroll
  for (int i = 0; i < HIST; ++i) {
    if (i >= n) continue;
    float taps[TAPS][8];
#pragma unroll
    for (int k = 0; k < TAPS; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e) taps[k][e] = x[i + k][e];
    leave(start + i, taps);
  }
  if (!st) return;
#pragma unroll
  for (int m = 0; m < HIST; ++m) {
    float v[8];
    if (n >= HIST) {
      Frag8 f;
      f.u = *(const uint4*)(in + (size_t)(start + n - HIST + m) * in_ld + c);
      widen(f, v);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = 0.f;
#pragma unroll
      for (int k = 1; k < HIST; ++k)
        if (n == k)
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = x[m + k][e];
    }
    *(float4*)(st + (size_t)m * channels) = make_float4(v[0], v[1], v[2], v[3]);
    *(float4*)(st + (size_t)m * channels + 4) = make_float4(v[4], v[5], v[6], v[7]);
  }
}

static long conv_runs_threads(int n_tokens, int n_seqs, int channels) { return (((long)n_tokens + CONV_RUN - 1) / CONV_RUN + n_seqs) * (channels / 8); }
// Whether a step's sizes go through the kernel of runs, whose threads are numbered in 31 bits; larger ones keep the kernel of a thread a channel
extern "C" int cwm_conv_silu_in_runs(int n_tokens, int n_seqs, int channels) {
  return n_seqs > 0 && n_tokens > n_seqs && channels % 8 == 0 && conv_runs_threads(n_tokens, n_seqs, channels) < (1L << 31) - 256;
}

// w_by_tap: the same weights as [taps][channels], or null (then every token goes through the kernel of a thread a channel)
extern "C" int cwm_conv_silu(const void* in, long in_ld, int dtype, const float* w, const float* w_by_tap, const float* bias, float* state, long state_ld,
                             long state_off, const int* slots, const int* cu_q, const int* seq_of_token, void* out, int n_tokens,
                             int n_seqs, int channels, int taps, int n_slots, hipStream_t stream) {
  CWM_REQUIRE(in && w && bias && state && slots && cu_q && seq_of_token && out, "conv_silu: arguments missing");
  CWM_REQUIRE(taps >= 1 && taps <= CONV_MAX_TAPS, "conv_silu: %d taps, the kernel takes 1..%d", taps, CONV_MAX_TAPS);
  CWM_REQUIRE(channels > 0 && in_ld >= channels && n_tokens >= 0, "conv_silu: bad sizes");
  CWM_REQUIRE(state_off >= 0 && state_off + (long)(taps - 1) * channels <= state_ld, "conv_silu: the state row is too short");
  if (n_tokens == 0) return 0;
  dim3 grid(n_tokens, (channels + 255) / 256);
  if (dtype == CWM_BF16 && w_by_tap && cwm_conv_silu_in_runs(n_tokens, n_seqs, channels) && in_ld % 8 == 0 && state_ld % 4 == 0 &&
      state_off % 4 == 0 && ((uintptr_t)in % 16) == 0 && ((uintptr_t)out % 16) == 0 && ((uintptr_t)w_by_tap % 16) == 0 && ((uintptr_t)bias % 16) == 0 &&
      ((uintptr_t)state % 16) == 0) {
    const long threads = conv_runs_threads(n_tokens, n_seqs, channels);
#define CWM_CONV_RUNS(TAPS)                                                                                                              \
  hipLaunchKernelGGL(conv_silu_runs_kernel<TAPS>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, (const bf16_t*)in, in_ld, \
                     w_by_tap, bias, state, state_ld, state_off, slots, cu_q, seq_of_token, (bf16_t*)out, n_tokens, n_seqs, channels, n_slots)
    static_assert(CONV_MAX_TAPS == 8, "a build for every number of taps");
    switch (taps) {
      case 1: CWM_CONV_RUNS(1); break;
      case 2: CWM_CONV_RUNS(2); break;
      case 3: CWM_CONV_RUNS(3); break;
      case 4: CWM_CONV_RUNS(4); break;
      case 5: CWM_CONV_RUNS(5); break;
      case 6: CWM_CONV_RUNS(6); break;
      case 7: CWM_CONV_RUNS(7); break;
      default: CWM_CONV_RUNS(8);
    }
#undef CWM_CONV_RUNS
  } else if (dtype == CWM_BF16)
    hipLaunchKernelGGL(conv_silu_kernel<bf16_t>, grid, dim3(256), 0, stream, (const bf16_t*)in, in_ld, w, bias, state, state_ld, state_off,
                       slots, cu_q, seq_of_token, (bf16_t*)out, channels, taps, n_slots);
  else if (dtype == CWM_F32)
    hipLaunchKernelGGL(conv_silu_kernel<float>, grid, dim3(256), 0, stream, (const float*)in, in_ld, w, bias, state, state_ld, state_off,
                       slots, cu_q, seq_of_token, (float*)out, channels, taps, n_slots);
  else
    return cwm_fail("conv_silu: unknown dtype %d", dtype);
  return cwm_launch_status("conv_silu");
}

// One block per (tile of P, head, sequence).  Thread (p, s) holds 16 rows of column p of the head's state: with
// `split` lanes a column (a power of two, adjacent in a wavefront), lane s has rows 4 (s + q split) + j, q, j < 4,
// so that its B and C values are four 16-byte pieces of LDS.  The block walks the sequence's tokens of this step in
// order, a chunk of up to 16 at a time: while it computes on one chunk from LDS (B, C and the tile's x as float32, the step
// sizes and decays computed once a token), the next chunk's values are already on their way into registers.  The
// split lanes add their parts of y_t[p] by shuffles in a fixed order.  The state is read once before and written
// once after the walk; what a token's result is made of, and in which order, does not depend on how the
// sequence is cut into steps.
#define SCAN_PF 36  // most values of a chunk that one thread fetches

// THREADS a block, TC tokens a chunk.  VEC: the rows of xbc start at multiples of 16 bytes and N and P are multiples
// of the values in 16 bytes, so a chunk is fetched in pieces of 16 bytes; otherwise value by value.
#define SCAN_PFV 6  // most 16-byte pieces of a chunk that one thread fetches

//
// Long portions are cut into segments that run side by side (PHASE 1 and 2; PHASE 0 is the walk of whole portions):
// `segments` holds, for every block z, {sequence, first token, end token, number j of the segment in its sequence,
// the sequence's first entry in the scratch lists, segments of the sequence}.  PHASE 1: segment j < last walks its
// tokens from a zero state and leaves that state and the product of its decays in entry 1 + j; the last segment's
// block copies the sequence's state into entry 0.  PHASE 2: segment j starts from entry 0 carried through the
// entries 1 .. j (S <- decay_i S + state_i), walks its tokens and writes y; the last one leaves the sequence's state.
// No block reads a state that another block of the same launch writes.  PHASE 3: the portions of one segment alone, walked as in
// PHASE 0.
template <typename T, int THREADS, int TC, bool VEC, int PHASE>
__global__ void __launch_bounds__(THREADS) selective_scan_kernel(const T* __restrict__ xbc, long xbc_ld, const T* __restrict__ dt_raw,
                                                                 long dt_ld, const float* __restrict__ dt_bias,
                                                                 const float* __restrict__ a_log, const float* __restrict__ d_skip,
                                                                 float* state, long state_ld, const int* __restrict__ slots,
                                                                 const int* __restrict__ cu_q, float* __restrict__ y, int heads, int P,
                                                                 int N, int groups, int split, int n_slots,
                                                                 const int* __restrict__ segments, float* seg_state, float* seg_decay) {
  extern __shared__ float lds[];
  const int h = blockIdx.y;
  int b = blockIdx.z, t0, t1, seg = 0, seg_base = 0, n_segs = 1;
  if (PHASE == 0) {
    t0 = cu_q[b], t1 = cu_q[b + 1];
  } else {
    const int* entry = segments + 6 * blockIdx.z;
    b = entry[0], t0 = entry[1], t1 = entry[2], seg = entry[3], seg_base = entry[4], n_segs = entry[5];
  }
  if (PHASE == 3 && n_segs > 1) return;
  const int cols = THREADS / split;
  const int s = threadIdx.x % split;
  const int col = threadIdx.x / split;
  const int p0 = blockIdx.x * cols;
  const int p = p0 + col;
  const bool live = p < P;
  const int g = h / (heads / groups);
  const int inner = heads * P;
  const int NB = SCAN_ROWS * split;  // rows of B (and of C) in LDS, zeros from N on
  const int row = 2 * NB + cols;     // a token's values in LDS: B, C, the tile's x
  float* dtv = lds + TC * row;       // the chunk's step sizes
  float* av = dtv + TC;              // and decays
  const int slot = slots[b];
  // A head's state in memory, as its threads hold it: [q][p][s][j] for row 4 (s + q split) + j of column p, so that a
  // thread's four rows are 16 bytes and the split lanes of a column lie side by side (rows from N on stay zero).
  float* st = (slot >= 0 && slot < n_slots) ? state + (size_t)slot * state_ld + (size_t)h * SCAN_ROWS * split * P : nullptr;
  float S[SCAN_ROWS];
  const size_t head_elems = (size_t)SCAN_ROWS * split * P;
  auto load_state = [&](const float* from) {  // null: zeros
#pragma unroll
    for (int q = 0; q < SCAN_ROWS / 4; ++q) {
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (from && live) v = *(const float4*)(from + (((size_t)q * P + p) * split + s) * 4);
      S[4 * q + 0] = v.x, S[4 * q + 1] = v.y, S[4 * q + 2] = v.z, S[4 * q + 3] = v.w;
    }
  };
  auto store_state = [&](float* to) {
    if (to && live) {
#pragma unroll
      for (int q = 0; q < SCAN_ROWS / 4; ++q)
        *(float4*)(to + (((size_t)q * P + p) * split + s) * 4) = make_float4(S[4 * q + 0], S[4 * q + 1], S[4 * q + 2], S[4 * q + 3]);
    }
  };
  auto entry_state = [&](int k) { return seg_state + ((size_t)(seg_base + k) * heads + h) * head_elems; };
  if (PHASE == 0 || PHASE == 3) {
    load_state(st);
  } else if (PHASE == 1) {
    if (seg == n_segs - 1) {  // the whole block: the sequence's state as it is, for the segments of the next launch
      load_state(st);
      store_state(entry_state(0));
      return;
    }
    load_state(nullptr);
  } else {
    load_state(entry_state(0));
    for (int i = 0; i < seg; ++i) {
      const float d = seg_decay[(size_t)(seg_base + 1 + i) * heads + h];
      const float* local = entry_state(1 + i);
#pragma unroll
      for (int q = 0; q < SCAN_ROWS / 4; ++q) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (live) v = *(const float4*)(local + (((size_t)q * P + p) * split + s) * 4);
        S[4 * q + 0] = d * S[4 * q + 0] + v.x, S[4 * q + 1] = d * S[4 * q + 1] + v.y;
        S[4 * q + 2] = d * S[4 * q + 2] + v.z, S[4 * q + 3] = d * S[4 * q + 3] + v.w;
      }
    }
  }
  const float bias = dt_bias[h];
  const float rate = -expf(a_log[h]);
  const float skip = d_skip[h];
  float decays = 1.f;  // PHASE 1: the product of the segment's decays

  constexpr int U = 16 / sizeof(T);  // values in 16 bytes
  float pf[VEC ? 1 : SCAN_PF];
  uint4 pfv[VEC ? SCAN_PFV : 1];
  int pfv_at[VEC ? SCAN_PFV : 1];  // where in LDS each piece goes (-1: nowhere)
  float pf_dt = 0.f, pf_a = 0.f;
  auto fetch = [&](int start) {  // the chunk that starts at token `start`, into registers
    const int n_tok = min(TC, t1 - start);  // what lies behind the sequence's end is not read (nor used)
    if constexpr (VEC) {
      const int pieces = row / U;  // of one token
      int tc = threadIdx.x / pieces, e = threadIdx.x - tc * pieces;
      const int step_tc = THREADS / pieces, step_e = THREADS - step_tc * pieces;
#pragma unroll
      for (int k = 0; k < SCAN_PFV; ++k) {
        uint4 v = make_uint4(0, 0, 0, 0);
        pfv_at[k] = tc < TC ? tc * row + e * U : -1;
        if (tc < n_tok) {
          const T* src = xbc + (size_t)(start + tc) * xbc_ld;
          const int at = e * U;
          if (at < NB) {
            if (at < N) v = *(const uint4*)(src + inner + (size_t)g * N + at);
          } else if (at < 2 * NB) {
            if (at - NB < N) v = *(const uint4*)(src + inner + (size_t)(groups + g) * N + (at - NB));
          } else if (p0 + at - 2 * NB < P) {
            v = *(const uint4*)(src + (size_t)h * P + p0 + (at - 2 * NB));
          }
        }
        pfv[k] = v;
        tc += step_tc;
        e += step_e;
        if (e >= pieces) e -= pieces, ++tc;
      }
    } else {
      const int total = n_tok * row;
      int tc = 0, e = threadIdx.x;  // this thread's k-th value, number threadIdx.x + k * THREADS of the chunk, is value e of token tc
      while (e >= row) e -= row, ++tc;
#pragma unroll
      for (int k = 0; k < SCAN_PF; ++k) {
        float v = 0.f;
        if (tc * row + e < total) {
          const T* src = xbc + (size_t)(start + tc) * xbc_ld;
          if (e < NB) {
            if (e < N) v = Elem<T>::load(src + inner + (size_t)g * N + e);
          } else if (e < 2 * NB) {
            if (e - NB < N) v = Elem<T>::load(src + inner + (size_t)(groups + g) * N + (e - NB));
          } else if (p0 + e - 2 * NB < P) {
            v = Elem<T>::load(src + (size_t)h * P + p0 + (e - 2 * NB));
          }
        }
        pf[k] = v;
        e += THREADS;
        while (e >= row) e -= row, ++tc;
      }
    }
    if (threadIdx.x < TC) {
      const int t = start + threadIdx.x;
      if (t < t1) {
        const float z = Elem<T>::load(dt_raw + (size_t)t * dt_ld + h) + bias;
        pf_dt = z > 20.f ? z : log1pf(expf(z));
        pf_a = expf(rate * pf_dt);
      }
    }
  };
  auto stage = [&]() {  // registers -> LDS
    if constexpr (VEC) {
#pragma unroll
      for (int k = 0; k < SCAN_PFV; ++k) {
        if (pfv_at[k] < 0) continue;
        float* dst = lds + pfv_at[k];
        if constexpr (sizeof(T) == 4) {
          *(uint4*)dst = pfv[k];
        } else {
          const uint32_t w[4] = {pfv[k].x, pfv[k].y, pfv[k].z, pfv[k].w};
          *(float4*)dst = make_float4(__uint_as_float(w[0] << 16), __uint_as_float(w[0] & 0xffff0000u), __uint_as_float(w[1] << 16),
                                      __uint_as_float(w[1] & 0xffff0000u));
          *(float4*)(dst + 4) = make_float4(__uint_as_float(w[2] << 16), __uint_as_float(w[2] & 0xffff0000u), __uint_as_float(w[3] << 16),
                                            __uint_as_float(w[3] & 0xffff0000u));
        }
      }
    } else {
#pragma unroll
      for (int k = 0; k < SCAN_PF; ++k) {
        const int idx = threadIdx.x + k * THREADS;
        if (idx < TC * row) lds[idx] = pf[k];
      }
    }
    if (threadIdx.x < TC) {
      dtv[threadIdx.x] = pf_dt;
      av[threadIdx.x] = pf_a;
    }
  };
  // One chunk from LDS.  The walk itself holds no wait on another lane: every token leaves its lane's part of y in
  // a register, and the parts of the whole chunk are added across the split lanes afterwards, side by side.  A full
  // chunk runs without a condition in it, so that a token's reads from LDS can start while the one before computes.
  auto walk = [&](auto full_tag, int start, int n_here) {
    constexpr bool FULL = decltype(full_tag)::value;
    float part[TC], xs[TC];
#pragma unroll
    for (int tc = 0; tc < TC; ++tc) {
      part[tc] = 0.f;
      xs[tc] = 0.f;
      if (FULL || tc < n_here) {
        const float* tok = lds + tc * row;
        const float a = av[tc];
        if (PHASE == 1) decays *= a;
        const float x = tok[2 * NB + col];
        const float dx = dtv[tc] * x;
        float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < SCAN_ROWS / 4; ++q) {
          const float4 Bq = *(const float4*)(tok + 4 * (s + q * split));
          const float4 Cq = *(const float4*)(tok + NB + 4 * (s + q * split));
          S[4 * q + 0] = fmaf(a, S[4 * q + 0], Bq.x * dx);
          S[4 * q + 1] = fmaf(a, S[4 * q + 1], Bq.y * dx);
          S[4 * q + 2] = fmaf(a, S[4 * q + 2], Bq.z * dx);
          S[4 * q + 3] = fmaf(a, S[4 * q + 3], Bq.w * dx);
          acc[0] = fmaf(S[4 * q + 0], Cq.x, acc[0]);
          acc[1] = fmaf(S[4 * q + 1], Cq.y, acc[1]);
          acc[2] = fmaf(S[4 * q + 2], Cq.z, acc[2]);
          acc[3] = fmaf(S[4 * q + 3], Cq.w, acc[3]);
        }
        part[tc] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
        xs[tc] = x;
      }
    }
    if (PHASE == 1) return;  // only the state is wanted
    for (int off = 1; off < split; off <<= 1) {
#pragma unroll
      for (int tc = 0; tc < TC; ++tc)
        if (FULL || tc < n_here) part[tc] += __shfl_xor(part[tc], off, CWM_WAVE);
    }
    if (live && s == 0) {
#pragma unroll
      for (int tc = 0; tc < TC; ++tc)
        if (FULL || tc < n_here) y[(size_t)(start + tc) * inner + (size_t)h * P + p] = part[tc] + skip * xs[tc];
    }
  };

  fetch(t0);
  stage();
  __syncthreads();
  for (int start = t0; start < t1; start += TC) {
    const bool more = start + TC < t1;
    if (more) fetch(start + TC);
    const int n_here = min(TC, t1 - start);
    if (n_here == TC)
      walk(std::true_type{}, start, TC);
    else
      walk(std::false_type{}, start, n_here);
    __syncthreads();
    if (more) {
      stage();
      __syncthreads();
    }
  }
  if (PHASE == 0 || PHASE == 3) {
    store_state(st);
  } else if (PHASE == 1) {
    store_state(entry_state(1 + seg));
    if (threadIdx.x == 0) seg_decay[(size_t)(seg_base + 1 + seg) * heads + h] = decays;
  } else if (seg == n_segs - 1) {
    store_state(st);
  }
}

// A step in which every sequence brings one token (decoding): no chunk, no LDS.  Thread (p, s) as above; its 16 values
// of B and of C, x, dt and its 16 state values are all asked for at once, so the step waits for memory once.
template <typename T>
__global__ void __launch_bounds__(256) selective_scan_single_kernel(const T* __restrict__ xbc, long xbc_ld, const T* __restrict__ dt_raw,
                                                                    long dt_ld, const float* __restrict__ dt_bias,
                                                                    const float* __restrict__ a_log, const float* __restrict__ d_skip,
                                                                    float* state, long state_ld, const int* __restrict__ slots,
                                                                    float* __restrict__ y, int heads, int P, int N, int groups, int split,
                                                                    int n_slots) {
  const int h = blockIdx.y;
  const int t = blockIdx.z;  // the sequence, and its one token
  const int cols = 256 / split;
  const int s = threadIdx.x % split;
  const int p = blockIdx.x * cols + threadIdx.x / split;
  const bool live = p < P;
  const int pc = live ? p : P - 1;
  const int g = h / (heads / groups);
  const int inner = heads * P;
  const int slot = slots[t];
  float* st = (slot >= 0 && slot < n_slots) ? state + (size_t)slot * state_ld + (size_t)h * SCAN_ROWS * split * P : nullptr;
  const T* row = xbc + (size_t)t * xbc_ld;
  const T* Bt = row + inner + (size_t)g * N;
  const T* Ct = Bt + (size_t)groups * N;
  float S[SCAN_ROWS], Bv[SCAN_ROWS], Cv[SCAN_ROWS];
#pragma unroll
  for (int q = 0; q < SCAN_ROWS / 4; ++q) {
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (st && live) v = *(const float4*)(st + (((size_t)q * P + p) * split + s) * 4);
    S[4 * q + 0] = v.x, S[4 * q + 1] = v.y, S[4 * q + 2] = v.z, S[4 * q + 3] = v.w;
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int n = 4 * (s + q * split) + jj;
      Bv[4 * q + jj] = n < N ? Elem<T>::load(Bt + n) : 0.f;
      Cv[4 * q + jj] = n < N ? Elem<T>::load(Ct + n) : 0.f;
    }
  }
  const float x = Elem<T>::load(row + (size_t)h * P + pc);
  const float z = Elem<T>::load(dt_raw + (size_t)t * dt_ld + h) + dt_bias[h];
  const float dt = z > 20.f ? z : log1pf(expf(z));
  const float a = expf(-expf(a_log[h]) * dt);
  const float dx = dt * x;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < SCAN_ROWS; ++i) {  // the same operations in the same order as the walk of a chunk
    S[i] = fmaf(a, S[i], Bv[i] * dx);
    acc[i & 3] = fmaf(S[i], Cv[i], acc[i & 3]);
  }
  float part = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  for (int off = 1; off < split; off <<= 1) part += __shfl_xor(part, off, CWM_WAVE);
  if (live && s == 0) y[(size_t)t * inner + (size_t)h * P + p] = part + d_skip[h] * x;
  if (st && live) {
#pragma unroll
    for (int q = 0; q < SCAN_ROWS / 4; ++q)
      *(float4*)(st + (((size_t)q * P + p) * split + s) * 4) = make_float4(S[4 * q + 0], S[4 * q + 1], S[4 * q + 2], S[4 * q + 3]);
  }
}

// Segments of bfloat16 rows on the matrix cores, 64 tokens at a time.  With L_t the sum of the block's log decays up to its
// token t, S the state before the block, and everything per head:
//       y_t = e^(L_t) S^T C_t + sum_(s <= t) (C_t . B_s) dt_s e^(L_t - L_s) x_s + D x_t
//       S  <- e^(L_end) S + sum_s B_s (e^(L_end - L_s) dt_s x_s)^T
// C_t . B_s are products of bfloat16 values (exact, float32 sums).  The other products have one float32 operand each (S, the
// weighted x, the scores), which goes in as three bfloat16 parts that hold all its bits, so that every single product is exact
// and no value is rounded that the walk keeps: three v_mfma_f32_16x16x32_bf16 of 16 cycles for eight v_mfma_f32_16x16x4_f32 of
// 32 (2,048 tokens 154 us with those; off float64, on the same 1,025 tokens of 8 heads of 64 x 128, 3.9e-7 instead of 2.4e-7).  The L are summed in float64: a difference of two
// of them is as exact as the decays between them.  A wavefront has 16 columns of the head: its part of the state stays in
// registers as the matrix instruction leaves it (lane 16 j + r: column r, rows 16 q + 4 j + i), and two such tiles are also the
// operand that C needs, with its values of k in the order 4 j + i, 16 + 4 j + i; likewise two tiles of x.  The other operand is
// read from LDS in that order.
// MODE 1 leaves the state that every segment but a sequence's last makes from zero, and the segment's decay; then
// `scan_carry_kernel` turns those into the states at the segments' starts; MODE 2 walks every segment from there and writes y.
// Portions of one segment, decoded tokens among them, are left to the walk: their bits and their cost are what they are without a
// long portion beside them (in blocks a decoded token pays for 64).
// A step of 64 tokens takes a block 9 us, 1.5 of them matrix instructions: scores 2 us (ten tiles of keys for four wavefronts, three at most),
// S^T C and the state's update 1.4 each, y's stores 1.4, staging 1.2.  Step sizes and sums of logs are made a step ahead by the first
// wavefront, which has one tile of scores, instead of while the others wait (58 to 55 us with the dealt tiles).  Two blocks a compute unit
// (three in MODE 1; asked for, since the registers beyond the first 256 would leave one); bound by the vector units and by splitting values on them (looking for infinities among B and C costs 2 of 115 us); the walk was bound by its reads of B and C from LDS.
#define BLOCK_TOKENS 64

// What is made of this value is made after this place: the compiler would move what both ways of a branch have in common
// before it, and hold all of it in registers.
__device__ __forceinline__ int keep_apart(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// Four bfloat16 values of an operand as float32.
__device__ __forceinline__ void four_floats(const bf16_t* at, float (&c)[4]) {
  const uint2 w = *(const uint2*)at;
  c[0] = __uint_as_float(w.x << 16), c[1] = __uint_as_float(w.x & 0xffff0000u);
  c[2] = __uint_as_float(w.y << 16), c[3] = __uint_as_float(w.y & 0xffff0000u);
}

// Sixteen bytes of an operand whose eight values of k are 4 j .. + 3 and 16 + 4 j .. + 3 of 32: the order in which two tiles of a
// matrix instruction's result hold them.
__device__ __forceinline__ Frag8 two_fours(const bf16_t* at) {
  const uint2 low = *(const uint2*)at, high = *(const uint2*)(at + 16);
  Frag8 f;
  f.u = make_uint4(low.x, low.y, high.x, high.y);
  return f;
}

template <int NT, int MODE>  // NT: tiles of 16 rows of the state (even)
__global__ void __launch_bounds__(256, MODE == 1 ? 3 : 2) scan_block_kernel(const bf16_t* __restrict__ xbc, long xbc_ld, const bf16_t* __restrict__ dt_raw, long dt_ld,
                                                         const float* __restrict__ dt_bias, const float* __restrict__ a_log,
                                                         const float* __restrict__ d_skip, float* __restrict__ state, long state_ld,
                                                         const int* __restrict__ slots, float* __restrict__ y, int heads, int P, int N, int groups,
                                                         int split, int n_slots, const int* __restrict__ segments, float* __restrict__ seg_state,
                                                         float* __restrict__ seg_decay) {
  constexpr int ROWS = 16 * NT, PIECES = ROWS / 8, LOADS = BLOCK_TOKENS * PIECES / 256;
  constexpr int ROW_LD = ROWS + 8, COL_LD = BLOCK_TOKENS + 4, SCORE_LD = BLOCK_TOKENS + 4;
  static_assert(NT % 2 == 0, "the state's rows go into products of 32");
  typedef uint32_t Words4 __attribute__((ext_vector_type(4)));
  __shared__ __attribute__((aligned(16))) bf16_t b_rows[MODE == 2 ? BLOCK_TOKENS : 1][ROW_LD];
  __shared__ __attribute__((aligned(16))) bf16_t c_rows[MODE == 2 ? BLOCK_TOKENS : 1][ROW_LD];
  __shared__ __attribute__((aligned(16))) bf16_t b_cols[ROWS][COL_LD];
  __shared__ __attribute__((aligned(16))) bf16_t scores[MODE == 2 ? 3 : 1][MODE == 2 ? BLOCK_TOKENS : 1][SCORE_LD];  // in three parts
  // of this block of tokens and of the next, in turn
  __shared__ double sum_log_of[2][BLOCK_TOKENS];
  __shared__ __attribute__((aligned(16))) float step_size_of[2][BLOCK_TOKENS], from_start_of[2][BLOCK_TOKENS], to_end_of[2][BLOCK_TOKENS];
  __shared__ int spoilt;  // whether a B or C of the segment so far was not finite: from there on its products are the float32 instruction's
  const int* entry = segments + 6 * blockIdx.z;
  const int t0 = entry[1], t1 = entry[2], seg = entry[3], seg_base = entry[4], n_segs = entry[5];
  if (n_segs == 1) return;                     // a short portion is walked
  if (MODE == 1 && seg == n_segs - 1) return;  // nothing follows it
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, j = lane >> 4;
  const int h = blockIdx.y, g = h / (heads / groups), inner = heads * P;
  const int p = blockIdx.x * 64 + wave * 16 + r;
  const bool live = p < P;  // P: a multiple of 16, so a wavefront's columns all exist or none does
  const size_t head_elems = (size_t)SCAN_ROWS * split * P;
  const float bias = dt_bias[h], rate = -expf(a_log[h]), skip = d_skip[h];

  // rows 16 q + 4 j .. + 3 of column p as they lie in a head's state (rows past SCAN_ROWS * split do not exist)
  auto state_at = [&](int q, int quarter) -> long {
    const int four = 4 * q + quarter;
    return live && four < 4 * split ? (((long)(four / split) * P + p) * split + four % split) * 4 : -1;
  };
  float4v S[NT];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const long at = state_at(q, j);
    S[q] = MODE == 2 && at >= 0 ? *(const float4v*)(seg_state + ((size_t)(seg_base + seg) * heads + h) * head_elems + at) : (float4v){0.f, 0.f, 0.f, 0.f};
  }

  Words4 rb[LOADS], rc[MODE == 2 ? LOADS : 1];
  uint32_t rx[16];
  uint32_t r_dt = 0;
  const bf16_t* b_src = xbc + (size_t)t0 * xbc_ld + inner + (size_t)g * N;  // (a segment's offsets take 32 bits)
  const bf16_t* c_src = b_src + (size_t)groups * N;
  const bf16_t* x_src = xbc + (size_t)t0 * xbc_ld + (size_t)h * P;
  const uint32_t x_col = live ? p : 0;
  const uint32_t y_lane = 4 * j * inner + p;
  // a thread fetches pieces of 16 bytes, the lanes of a wavefront those of its tokens at one place of the row (with a row's in neighbouring
  // lanes the stores into b_cols meet in a bank four at a time: MODE 1 28 us instead of 24)
  auto fetch = [&](int c0) {
#pragma unroll
    for (int k = 0; k < LOADS; ++k) {
      const int t = c0 + lane, n = 8 * (4 * k + wave);
      // what lies past the end or beyond the state's rows (N: a multiple of 8) is read from a place that exists and left out when it is staged
      const uint32_t at = (uint32_t)(min(t, t1 - 1) - t0) * (uint32_t)xbc_ld + min(n, N - 8);
      rb[k] = *(const Words4*)(b_src + at);
      if constexpr (MODE == 2) rc[k] = *(const Words4*)(c_src + at);
    }
#pragma unroll
    // tokens 16 (k / 4) + 4 j + k % 4 of the lane's column; what lies past the end is the last token's and is left out when the
    // values are used: a value put together or a branch taken here waits for its load (16 waits one after the other: 2,048 tokens of
    // 64 heads 71 us instead of 58 in MODE 2, 38 instead of 24 in MODE 1)
    for (int k = 0; k < 16; ++k) rx[k] = x_src[(uint32_t)(min(c0 + 16 * (k >> 2) + 4 * j + (k & 3), t1 - 1) - t0) * (uint32_t)xbc_ld + x_col];
  };
  auto fetch_dt = [&](int c0) {
    if (wave == 0) r_dt = dt_raw[(size_t)min(c0 + lane, t1 - 1) * dt_ld + h];
  };
  double segment_log = 0.0;  // MODE 1, the first wavefront: of the segment's decay

  // step sizes and sums of log decays of a block of tokens, by the first wavefront, which has the fewest scores to make
  auto weigh = [&](int c0, int place, uint32_t raw) {
    const bool inside = c0 + lane < t1;
    const float zt = bf16_to_f32((bf16_t)raw) + bias, dt = inside ? (zt > 20.f ? zt : log1pf(expf(zt))) : 0.f;
    // e^-128 is 0 in float32, as the decays of more are; bounded, they leave differences of sums finite and exact
    const float log_decay = inside ? rate * dt : 0.f;
    double through = (double)(log_decay < -128.f ? -128.f : log_decay);
#pragma unroll
    for (int off = 1; off < CWM_WAVE; off <<= 1) {
      const double o = __shfl_up(through, off, CWM_WAVE);
      if (lane >= off) through += o;
    }
    const double all = __shfl(through, CWM_WAVE - 1, CWM_WAVE);
    sum_log_of[place][lane] = through;
    step_size_of[place][lane] = dt;
    from_start_of[place][lane] = expf((float)through);
    to_end_of[place][lane] = expf((float)(all - through)) * dt;
    if constexpr (MODE == 1) segment_log += all;
  };

  if (tid == 0) spoilt = 0;
  fetch_dt(t0);
  fetch(t0);
  if (wave == 0) weigh(t0, 0, r_dt);
  fetch_dt(t0 + BLOCK_TOKENS);
  for (int c0 = t0; c0 < t1; c0 += BLOCK_TOKENS) {
    const int place = ((c0 - t0) / BLOCK_TOKENS) & 1;
    const double* sum_log = sum_log_of[place];
    const float *step_size = step_size_of[place], *from_start = from_start_of[place], *to_end = to_end_of[place];
    __syncthreads();  // the block of tokens before is done with
    Halves most = {0, 0};
#pragma unroll
    for (int k = 0; k < LOADS; ++k) {
      const int token = lane, n = 8 * (4 * k + wave);
      const uint32_t inside = c0 + token < t1 && n < N ? 0xffffffffu : 0u;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        rb[k][e] &= inside;
        if constexpr (MODE == 2) rc[k][e] &= inside;
        most = larger_magnitudes(most, rb[k][e]);
        if constexpr (MODE == 2) most = larger_magnitudes(most, rc[k][e]);
      }
      if constexpr (MODE == 2) {
        *(Words4*)&b_rows[token][n] = rb[k];
        *(Words4*)&c_rows[token][n] = rc[k];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) b_cols[n + e][token] = (bf16_t)(rb[k][e >> 1] >> (16 * (e & 1)));
    }
    if (max(most.x, most.y) >= 0x7f80) spoilt = 1;
    uint32_t rx_now[8];  // (the next block's come into rx meanwhile)
    Halves largest = {0, 0};
#pragma unroll
    for (int k = 0; k < 16; k += 2) {
      const int t = c0 + 16 * (k >> 2) + 4 * j + (k & 3);
      const uint32_t low = live && t < t1 ? rx[k] : 0, high = live && t + 1 < t1 ? rx[k + 1] : 0;
      rx_now[k >> 1] = low | high << 16;
      largest = larger_magnitudes(largest, rx_now[k >> 1]);
    }
    auto x_of = [&](int k) { return __uint_as_float(k & 1 ? rx_now[k >> 1] & 0xffff0000u : rx_now[k >> 1] << 16); };
    const uint32_t dt_next = keep_apart(r_dt);  // (taken here, where the loads are waited for)
    const bool all_finite = __ballot(max(largest.x, largest.y) >= 0x7f80) == 0;  // of the wavefront's columns
    __syncthreads();
    const bool all_plain = __builtin_amdgcn_readfirstlane(spoilt) == 0;
    fetch_dt(c0 + 2 * BLOCK_TOKENS);
    if (c0 + BLOCK_TOKENS < t1) fetch(c0 + BLOCK_TOKENS);  // in flight while this block of tokens is worked on
    if constexpr (MODE == 2) {
      // scores of the wavefront's 16 queries and the keys up to them; of the last wavefront's four tiles of keys the second wavefront,
      // which has two of its own, makes the first
      for (int tile = wave == 3 ? 1 : 0; tile < (wave == 1 ? 3 : wave + 1); ++tile) {
        const bool lent = wave == 1 && tile == 2;
        const int b = lent ? 0 : tile, t = 16 * (lent ? 3 : wave) + r;
        const double mine = sum_log[t];
        float4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < NT / 2; ++q) {
          Frag8 fb, fc;
          fb.u = *(const uint4*)&b_rows[16 * b + r][32 * q + 8 * j];
          fc.u = *(const uint4*)&c_rows[t][32 * q + 8 * j];
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb.v, fc.v, acc, 0, 0, 0);
        }
        const float4v dts = *(const float4v*)&step_size[16 * b + 4 * j];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = 16 * b + 4 * j + i;
          acc[i] = key <= t ? acc[i] * dts[i] * expf((float)(mine - sum_log[key])) : 0.f;
        }
        uint32_t w[3][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          w[0][i] = __float_as_uint(acc[i]);
          float rest = acc[i] - __uint_as_float(w[0][i] & 0xffff0000u);
          rest = (w[0][i] & 0x7f800000u) == 0x7f800000u ? 0.f : rest;
          w[1][i] = __float_as_uint(rest);
          w[2][i] = __float_as_uint(rest - __uint_as_float(w[1][i] & 0xffff0000u));
        }
#pragma unroll
        for (int k = 0; k < 3; ++k)
          *(uint2*)&scores[k][t][16 * b + 4 * j] =
              make_uint2(__builtin_amdgcn_perm(w[k][1], w[k][0], 0x07060302u), __builtin_amdgcn_perm(w[k][3], w[k][2], 0x07060302u));
      }
      if (wave == 0) weigh(c0 + BLOCK_TOKENS, place ^ 1, dt_next);
      if (wave % 2 == 0)  // keys go in pairs of tiles
#pragma unroll
        for (int k = 0; k < 3; ++k) *(uint2*)&scores[k][16 * wave + r][16 * (wave + 1) + 4 * j] = make_uint2(0u, 0u);
      __syncthreads();
      if (live) {
        float4v out[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) out[a] = (float4v){0.f, 0.f, 0.f, 0.f};
        if (__builtin_expect(all_plain, 1)) {
#pragma unroll
          for (int q = 0; q < NT; q += 2) {
            const float v[8] = {S[q][0], S[q][1], S[q][2], S[q][3], S[q + 1][0], S[q + 1][1], S[q + 1][2], S[q + 1][3]};
            Frag8 part[3];
            three_parts(v, part);
#pragma unroll
            for (int a = 0; a < 4; ++a) {
              const Frag8 c = two_fours(&c_rows[16 * a + r][16 * q + 4 * j]);
#pragma unroll
              for (int k = 2; k >= 0; --k) out[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c.v, part[k].v, out[a], 0, 0, 0);
            }
          }
        } else {
          const int row = keep_apart(r);
#pragma unroll
          for (int q = 0; q < NT; ++q)
#pragma unroll
            for (int a = 0; a < 4; ++a) {
              float c[4];
              four_floats(&c_rows[16 * a + row][16 * q + 4 * j], c);
#pragma unroll
              for (int i = 0; i < 4; ++i) out[a] = __builtin_amdgcn_mfma_f32_16x16x4f32(c[i], S[q][i], out[a], 0, 0, 0);
              __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const float4v f = *(const float4v*)&from_start[16 * a + 4 * j];
#pragma unroll
          for (int i = 0; i < 4; ++i) out[a][i] *= f[i];
        }
        auto score = [&](int row, int key) {
          return (bf16_to_f32(scores[0][row][key]) + bf16_to_f32(scores[1][row][key])) + bf16_to_f32(scores[2][row][key]);
        };
        if (all_finite) {
#pragma unroll
          for (int b = 0; b < 4; b += 2) {
            Frag8 xs;  // x is bfloat16
            xs.u = make_uint4(rx_now[2 * b], rx_now[2 * b + 1], rx_now[2 * b + 2], rx_now[2 * b + 3]);
#pragma unroll
            for (int a = b; a < 4; ++a)
#pragma unroll
              for (int k = 2; k >= 0; --k)
                out[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(two_fours(&scores[k][16 * a + r][16 * b + 4 * j]).v, xs.v, out[a], 0, 0, 0);
          }
        } else {
#pragma unroll
          for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int a = b + 1; a < 4; ++a)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                out[a] = __builtin_amdgcn_mfma_f32_16x16x4f32(score(16 * a + r, 16 * b + 4 * j + i), x_of(4 * b + i), out[a], 0, 0, 0);
        }
        if (!all_finite) {
          // a later key's score of 0 does not leave an infinity or a NaN out: the tiles on the diagonal key by key
#pragma unroll
          for (int k = 0; k < 16; ++k) {
            const int b = k >> 2;
            for (int from = 0; from < 4; ++from) {
              const int key = 4 * from + (k & 3);
              const float value = __shfl(x_of(k), 16 * from + r, CWM_WAVE);
#pragma unroll
              for (int i = 0; i < 4; ++i)
                if (4 * j + i >= key) out[b][i] = fmaf(score(16 * b + 4 * j + i, 16 * b + key), value, out[b][i]);
            }
          }
        }
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int at = c0 + 16 * a + i;  // of the lane's quarter 0
            if (at + 4 * j < t1) y[(size_t)at * inner + (size_t)h * P + y_lane] = out[a][i] + skip * x_of(4 * a + i);
          }
      }
    }
    if (MODE == 1 && wave == 0 && c0 + BLOCK_TOKENS < t1) weigh(c0 + BLOCK_TOKENS, place ^ 1, dt_next);
    // the state after the block of tokens
    const float whole = from_start[BLOCK_TOKENS - 1];
    if (__builtin_expect(all_plain, 1)) {
#pragma unroll
      for (int q = 0; q < NT; ++q) {
#pragma unroll
        for (int i = 0; i < 4; ++i) S[q][i] *= whole;
      }
#pragma unroll
      for (int b = 0; b < 4; b += 2) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = x_of(4 * b + k) * to_end[16 * (b + (k >> 2)) + 4 * j + (k & 3)];
        Frag8 part[3];
        three_parts(v, part);
#pragma unroll
        for (int q = 0; q < NT; ++q) {
          const Frag8 c = two_fours(&b_cols[16 * q + r][16 * b + 4 * j]);
#pragma unroll
          for (int k = 2; k >= 0; --k) S[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c.v, part[k].v, S[q], 0, 0, 0);
        }
      }
    } else {
      const int row = keep_apart(r), group = keep_apart(4 * j);
#pragma unroll
      for (int q = 0; q < NT; ++q) {
#pragma unroll
        for (int i = 0; i < 4; ++i) S[q][i] *= whole;
      }
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        float xs[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) xs[i] = x_of(4 * b + i) * to_end[16 * b + group + i];
#pragma unroll
        for (int q = 0; q < NT; ++q) {
          float c[4];
          four_floats(&b_cols[16 * q + row][16 * b + group], c);
#pragma unroll
          for (int i = 0; i < 4; ++i) S[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(c[i], xs[i], S[q], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);  // few values at a time: this seldom walked way must not cost the other one registers
        }
      }
    }
  }
  float* home = nullptr;
  if (MODE == 1) {
    home = seg_state + ((size_t)(seg_base + seg) * heads + h) * head_elems;
    if (blockIdx.x == 0 && tid == 0) seg_decay[(size_t)(seg_base + seg) * heads + h] = expf((float)segment_log);
  } else if (seg == n_segs - 1) {
    const int slot = slots[entry[0]];
    if (slot >= 0 && slot < n_slots) home = state + (size_t)slot * state_ld + (size_t)h * head_elems;
  }
  if (!home) return;
  const int quarter = keep_apart(j);  // (the places are worked out again, not kept through the walk)
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const long at = state_at(q, quarter);
    if (at >= 0) *(float4v*)(home + at) = S[q];
  }
}

// What the segments make from zero -> the states at their starts, in place: a thread an element of a sequence's state walks
// the sequence's segments in order.
__global__ void __launch_bounds__(256) scan_carry_kernel(const int* __restrict__ segments, const float* __restrict__ state, long state_ld,
                                                         const int* __restrict__ slots, int n_slots, int heads, long head_elems,
                                                         float* __restrict__ seg_state, const float* __restrict__ seg_decay) {
  const int* entry = segments + 6 * blockIdx.y;
  if (entry[3] != 0 || entry[5] == 1) return;  // the sequence's first segment stands for all of them; a short portion is walked
  const long i = (long)blockIdx.x * 256 + threadIdx.x, elems = heads * head_elems;
  if (i >= elems) return;
  const int h = (int)(i / head_elems), slot = slots[entry[0]], first = entry[4], count = entry[5];
  float cur = slot >= 0 && slot < n_slots ? state[(size_t)slot * state_ld + i] : 0.f;
  for (int s = 0; s < count; s += 8) {
    float add[8], keep[8];
#pragma unroll
    for (int a = 0; a < 8; ++a) {  // the last segment has neither: what lies past the others is not used
      const size_t at = first + min(s + a, count - 2);
      add[a] = seg_state[at * elems + i], keep[a] = seg_decay[at * heads + h];
    }
#pragma unroll
    for (int a = 0; a < 8; ++a) {
      if (s + a < count) seg_state[(size_t)(first + s + a) * elems + i] = cur;
      cur = fmaf(keep[a], cur, add[a]);
    }
  }
}

// ONLY: the one phase to launch, or -1: the walk, or with a list of segments both phases.
template <typename T, bool VEC, int ONLY = -1>
static void launch_scan(dim3 grid, int split, hipStream_t stream, const void* xbc, long xbc_ld, const void* dt_raw, long dt_ld,
                        const float* dt_bias, const float* a_log, const float* d_skip, float* state, long state_ld, const int* slots,
                        const int* cu_q, float* y, int heads, int P, int N, int groups, int n_slots, const int* segments, float* seg_state,
                        float* seg_decay) {
  constexpr int THREADS = 256, TC = 16;
  const int row = 2 * SCAN_ROWS * split + THREADS / split;
  const size_t lds_bytes = (size_t)(TC * row + 2 * TC) * sizeof(float);
#define CWM_SCAN_PHASE(PHASE)                                                                                                              \
  hipLaunchKernelGGL((selective_scan_kernel<T, THREADS, TC, VEC, PHASE>), grid, dim3(THREADS), lds_bytes, stream, (const T*)xbc, xbc_ld,     \
                     (const T*)dt_raw, dt_ld, dt_bias, a_log, d_skip, state, state_ld, slots, cu_q, y, heads, P, N, groups, split, n_slots, \
                     segments, seg_state, seg_decay)
  if constexpr (ONLY >= 0) {
    CWM_SCAN_PHASE(ONLY);
  } else if (!segments) {
    CWM_SCAN_PHASE(0);
  } else {
    CWM_SCAN_PHASE(1);
    CWM_SCAN_PHASE(2);
  }
#undef CWM_SCAN_PHASE
}

extern "C" int cwm_selective_scan(const void* xbc, long xbc_ld, const void* dt_raw, long dt_ld, int dtype, const float* dt_bias,
                                  const float* a_log, const float* d_skip, float* state, long state_ld, const int* slots,
                                  const int* cu_q, float* y, int n_tokens, int n_seqs, int heads, int P, int N, int groups, int n_slots,
                                  const int* segments, int n_segments, int n_short, float* seg_state, float* seg_decay, hipStream_t stream) {
  CWM_REQUIRE(xbc && dt_raw && dt_bias && a_log && d_skip && state && slots && cu_q && y, "selective_scan: arguments missing");
  CWM_REQUIRE(heads > 0 && P > 0 && N > 0 && groups > 0 && heads % groups == 0, "selective_scan: bad sizes");
  CWM_REQUIRE(N <= SCAN_ROWS * 16, "selective_scan: a state of %d rows, the kernel takes up to %d", N, SCAN_ROWS * 16);
  CWM_REQUIRE(xbc_ld >= (long)heads * P + 2L * groups * N && dt_ld >= heads, "selective_scan: rows too short");
  CWM_REQUIRE(heads <= 65535 && n_seqs <= 65535, "selective_scan: too many heads or sequences for one launch");
  const int split = cwm_scan_split(N);
  CWM_REQUIRE((long)heads * SCAN_ROWS * split * P <= state_ld && state_ld % 4 == 0 && ((uintptr_t)state % 16) == 0,
              "selective_scan: the state row is too short or not a multiple of 16 bytes");
  if (n_tokens == 0 || n_seqs == 0) return 0;
  const int cols = 256 / split;
  const int row = 2 * SCAN_ROWS * split + cols;
  CWM_REQUIRE(16 * row <= SCAN_PF * 256, "selective_scan: a chunk of tokens does not fit the threads' registers");
  // with a list of segments (6 numbers each; its scratch lists have an entry for every segment) the blocks' z counts those;
  // n_short of the portions are one segment each
  CWM_REQUIRE(!segments || (n_segments > 0 && n_segments <= 65535 && seg_state && seg_decay && ((uintptr_t)seg_state % 16) == 0),
              "selective_scan: a list of segments needs its scratch lists and at most 65535 entries");
  dim3 grid((P + cols - 1) / cols, heads, segments ? n_segments : n_seqs);
  if (!segments && n_tokens == n_seqs) {  // one token a sequence
    dim3 single((P + cols - 1) / cols, heads, n_seqs);
    if (dtype == CWM_BF16)
      hipLaunchKernelGGL(selective_scan_single_kernel<bf16_t>, single, dim3(256), 0, stream, (const bf16_t*)xbc, xbc_ld, (const bf16_t*)dt_raw, dt_ld,
                         dt_bias, a_log, d_skip, state, state_ld, slots, y, heads, P, N, groups, split, n_slots);
    else if (dtype == CWM_F32)
      hipLaunchKernelGGL(selective_scan_single_kernel<float>, single, dim3(256), 0, stream, (const float*)xbc, xbc_ld, (const float*)dt_raw, dt_ld,
                         dt_bias, a_log, d_skip, state, state_ld, slots, y, heads, P, N, groups, split, n_slots);
    else
      return cwm_fail("selective_scan: unknown dtype %d", dtype);
    return cwm_launch_status("selective_scan");
  }
  const int unit = dtype == CWM_BF16 ? 8 : 4;
  const bool vec = N % unit == 0 && P % unit == 0 && xbc_ld % unit == 0 && ((uintptr_t)xbc % 16) == 0 && 16 * row / unit <= SCAN_PFV * 256;
  if (segments && dtype == CWM_BF16 && vec && N <= 128 && P % 16 == 0 && ((uintptr_t)seg_state % 16) == 0) {
    // on the matrix cores: 2,048 tokens of 64 heads, 64 columns and 128 rows in 115 us (91 since no load of the next
    // tokens is waited for where it is issued) instead of 565 (launches included), 300 tokens in 77 instead of 170, 4,096 in 213 instead of 1,126; off float64, on the same 1,025 tokens
    // of 8 heads, 2.4e-7, the walk of segments token by token 2.4e-6
    const dim3 blocks((P + 63) / 64, heads, n_segments);
    const long head_elems = (long)SCAN_ROWS * split * P;
#define CWM_SCAN_BLOCK(NT, MODE)                                                                                                           \
  hipLaunchKernelGGL((scan_block_kernel<NT, MODE>), blocks, dim3(256), 0, stream, (const bf16_t*)xbc, xbc_ld, (const bf16_t*)dt_raw, dt_ld,  \
                     dt_bias, a_log, d_skip, state, state_ld, slots, y, heads, P, N, groups, split, n_slots, segments, seg_state, seg_decay)
    if (N <= 64) CWM_SCAN_BLOCK(4, 1); else CWM_SCAN_BLOCK(8, 1);
    hipLaunchKernelGGL(scan_carry_kernel, dim3((unsigned)((heads * head_elems + 255) / 256), n_segments), dim3(256), 0, stream, segments, state, state_ld,
                       slots, n_slots, heads, head_elems, seg_state, seg_decay);
    if (N <= 64) CWM_SCAN_BLOCK(4, 2); else CWM_SCAN_BLOCK(8, 2);
#undef CWM_SCAN_BLOCK
    if (n_short > 0)
      launch_scan<bf16_t, true, 3>(grid, split, stream, xbc, xbc_ld, dt_raw, dt_ld, dt_bias, a_log, d_skip, state, state_ld, slots, cu_q, y, heads, P, N,
                                   groups, n_slots, segments, seg_state, seg_decay);
    return cwm_launch_status("selective_scan");
  }
#define CWM_SCAN(T, VEC) \
  launch_scan<T, VEC>(grid, split, stream, xbc, xbc_ld, dt_raw, dt_ld, dt_bias, a_log, d_skip, state, state_ld, slots, cu_q, y, heads, P, N, groups, n_slots, \
                      segments, seg_state, seg_decay)
  if (dtype == CWM_BF16) {
    if (vec) CWM_SCAN(bf16_t, true); else CWM_SCAN(bf16_t, false);
  } else if (dtype == CWM_F32) {
    if (vec) CWM_SCAN(float, true); else CWM_SCAN(float, false);
  } else {
    return cwm_fail("selective_scan: unknown dtype %d", dtype);
  }
#undef CWM_SCAN
  return cwm_launch_status("selective_scan");
}

// Row-wise kernels of layers that normalise a sublayer's output before the residual sum:
//
//   group norm    dst[r] (+)= w * x_g / sqrt(mean(x_g^2) + eps) for each of `groups` equal consecutive parts x_g of
//                 the row x = sum_p src[p][row] (* silu(gate[row]) if a gate is given), float32 arithmetic.
//                 One entry point serves the norm of chosen rows into a fresh tensor, the norm of rows where they
//                 lie (dst == src; the rows may be columns of a wider tensor) and the norm that adds into the
//                 float32 residual stream (accumulate); the rows as they then stand can be left in a second tensor of
//                 another type as well (the next sublayer's input).
//   token shift   s_t = h_t + (h_(t-1) - h_t) * mu on the float32 stream, the previous token of a portion's first
//                 token coming from the sequence's state, which receives the portion's last h.
//   sigmoid gate  out = a * sigmoid(g).
//
// Sums run in a fixed order that depends on the row's own length only.
#include "common.h"

CWM_DEFINE_ERROR_API

__device__ __forceinline__ float load_as_f32(const void* p, int dtype, size_t i) {
  return dtype == CWM_F32 ? ((const float*)p)[i] : bf16_to_f32(((const bf16_t*)p)[i]);
}

__device__ __forceinline__ void store_from_f32(void* p, int dtype, size_t i, float v) {
  if (dtype == CWM_F32)
    ((float*)p)[i] = v;
  else
    ((bf16_t*)p)[i] = f32_to_bf16(v);
}

__device__ __forceinline__ float silu_f32(float z) { return z / (1.f + expf(-z)); }

typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
typedef float float8v __attribute__((ext_vector_type(8)));

// Eight consecutive elements as they lie: 32 bytes of float32, or 16 of bfloat16 (`hi` then repeats them, so that both loads
// are issued without a branch between them).
struct Eight {
  uint4v lo, hi;
};

template <bool WIDE>
__device__ __forceinline__ Eight load_eight(const void* p, int dtype, size_t i, int n) {
  Eight x;
  if (WIDE) {
    const char* at = (const char*)p + i * (dtype == CWM_F32 ? 4 : 2);
    x.lo = *(const uint4v*)at;
    x.hi = *(const uint4v*)(at + (dtype == CWM_F32 ? 16 : 0));
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (dtype == CWM_F32) {
        x.lo[c] = c < n ? ((const uint32_t*)p)[i + c] : 0u;
        x.hi[c] = c + 4 < n ? ((const uint32_t*)p)[i + c + 4] : 0u;
      } else {
        const uint32_t even = 2 * c < n ? ((const bf16_t*)p)[i + 2 * c] : 0u, odd = 2 * c + 1 < n ? ((const bf16_t*)p)[i + 2 * c + 1] : 0u;
        x.lo[c] = x.hi[c] = even | odd << 16;
      }
    }
  }
  return x;
}

// Element c (a compile-time number) of eight.
__device__ __forceinline__ float eight_at(const Eight& x, int dtype, int c) {
  const uint32_t f = c < 4 ? x.lo[c & 3] : x.hi[c & 3], h = x.lo[c >> 1];
  return __uint_as_float(dtype == CWM_F32 ? f : c & 1 ? h & 0xffff0000u : h << 16);
}

template <bool WIDE>
__device__ __forceinline__ void store_eight(void* p, int dtype, size_t i, int n, const float8v& y) {
  if (!WIDE) {
#pragma unroll
    for (int c = 0; c < 8; ++c)
      if (c < n) store_from_f32(p, dtype, i + c, y[c]);
  } else if (dtype == CWM_F32) {
    *(float4v*)((float*)p + i) = (float4v){y[0], y[1], y[2], y[3]};
    *(float4v*)((float*)p + i + 4) = (float4v){y[4], y[5], y[6], y[7]};
  } else {
    uint4v w;
#pragma unroll
    for (int c = 0; c < 4; ++c) w[c] = pack2_bf16(y[2 * c], y[2 * c + 1]);
    *(uint4v*)((bf16_t*)p + i) = w;
  }
}

// `team` threads (a power of two) serve a part, eight consecutive elements each, which stay in registers between the sum and
// the result; the weights and what is added to are under way while the sum is formed.  Only a part beyond 8,192 elements goes
// round twice.  Memory bounds it: 2,048 rows of 2,048, two float32 partial sums added into the residual, with the copy, take
// 13.6 us (5.5 TB/s) where one element a load and 256 threads a part took 20.9; in 8 parts 13.2 against 28.9, in 32 parts 13.2
// against 68.9; one row of 2,048 3.0 against 8.1.  WIDE: every row starts at a multiple of 16 bytes and parts are multiples
// of eight elements; the sums' order is the same either way.
template <bool WIDE, bool GATED, bool ADDED>
__global__ void __launch_bounds__(1024) group_norm_kernel(const void* src, int src_dtype, long src_ld, int n_partials,
                                                          long partial_stride, const void* gate, int gate_dtype,
                                                          long gate_ld, const void* __restrict__ weight, int w_dtype, void* dst,
                                                          int dst_dtype, long dst_ld, const int* __restrict__ rows, long n_parts, int groups, int part,
                                                          int team, float eps, void* __restrict__ copy, int copy_dtype, long copy_ld) {
  __shared__ float scratch[16];
  const int per = blockDim.x / team, mine = 8 * (threadIdx.x & (team - 1));
  for (long base = (long)blockIdx.x * per; base < n_parts; base += (long)gridDim.x * per) {
    const long asked = base + threadIdx.x / team, id = asked < n_parts ? asked : n_parts - 1;
    const long r = id / groups;
    const int g = (int)(id - r * groups);
    const size_t row = rows ? (size_t)rows[r] : (size_t)r;
    const size_t s0 = row * src_ld + (size_t)g * part;
    const size_t g0 = row * gate_ld + (size_t)g * part;
    const size_t d0 = (size_t)r * dst_ld + (size_t)g * part;
    const size_t w0 = (size_t)g * part;
    auto inputs = [&](int i, Eight& x, Eight& z) {
      x = load_eight<WIDE>(src, src_dtype, s0 + i, part - i);
      if (GATED) z = load_eight<WIDE>(gate, gate_dtype, g0 + i, part - i);
    };
    auto values = [&](int i, const Eight& x, const Eight& z) {
      float8v v;
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = eight_at(x, src_dtype, c);
      for (int p = 1; p < n_partials; ++p) {
        const Eight more = load_eight<WIDE>(src, src_dtype, (size_t)p * partial_stride + s0 + i, part - i);
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] += eight_at(more, src_dtype, c);
      }
      if (GATED)
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] *= silu_f32(eight_at(z, gate_dtype, c));
      return v;
    };
    auto squares = [&](const float8v& v, int n) {
      float ss = 0.f;
#pragma unroll
      for (int c = 0; c < 8; ++c) ss += c < n ? v[c] * v[c] : 0.f;
      return ss;
    };
    // a thread without elements reads the part's last ones again and leaves them out
    const int i0 = mine < part ? mine : WIDE ? part - 8 : part - 1;
    Eight x, z, w, old;
    inputs(i0, x, z);
    w = load_eight<WIDE>(weight, w_dtype, w0 + i0, part - i0);
    if (ADDED) old = load_eight<WIDE>(dst, dst_dtype, d0 + i0, part - i0);
    const float8v first = values(i0, x, z);
    float ss = squares(first, part - mine);
    for (int i = mine + 8 * team; i < part; i += 8 * team) {
      inputs(i, x, z);
      ss += squares(values(i, x, z), part - i);
    }
    float total;
    if (team <= CWM_WAVE) {
      total = ss;
      for (int m = 1; m < team; m <<= 1) total += __shfl_xor(total, m, CWM_WAVE);
    } else {
      total = block_sum(ss, scratch);
    }
    if (asked >= n_parts) continue;
    const float inv = 1.f / sqrtf(total / (float)part + eps);
    auto leave = [&](int i, const float8v& v, const Eight& w, const Eight& old) {
      float8v y;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        y[c] = v[c] * inv * eight_at(w, w_dtype, c);
        if (ADDED) y[c] += eight_at(old, dst_dtype, c);
      }
      store_eight<WIDE>(dst, dst_dtype, d0 + i, part - i, y);
      if (copy) store_eight<WIDE>(copy, copy_dtype, (size_t)r * copy_ld + w0 + i, part - i, y);  // what dst now holds, in another type
    };
    if (mine < part) leave(mine, first, w, old);
    for (int i = mine + 8 * team; i < part; i += 8 * team) {
      inputs(i, x, z);
      w = load_eight<WIDE>(weight, w_dtype, w0 + i, part - i);
      if (ADDED) old = load_eight<WIDE>(dst, dst_dtype, d0 + i, part - i);
      leave(i, values(i, x, z), w, old);
    }
  }
}

// src: [n_partials][.][src_ld] (rows `rows[r]` or r), dst: [n_rows][dst_ld]; dim = groups * part elements of a row.
extern "C" int cwm_group_norm(const void* src, int src_dtype, long src_ld, int n_partials, long partial_stride, const void* gate,
                              int gate_dtype, long gate_ld, const void* weight, int w_dtype, void* dst, int dst_dtype, long dst_ld,
                              const int* rows, int n_rows, int dim, int groups, float eps, int accumulate, void* copy, int copy_dtype,
                              long copy_ld, hipStream_t stream) {
  CWM_REQUIRE(src && weight && dst, "group_norm: arguments missing");
  CWM_REQUIRE(n_rows >= 0 && dim > 0 && groups > 0 && dim % groups == 0, "group_norm: %d elements do not divide into %d groups", dim, groups);
  CWM_REQUIRE(n_partials >= 1 && src_ld >= dim && dst_ld >= dim && (!gate || gate_ld >= dim), "group_norm: rows shorter than %d", dim);
  CWM_REQUIRE(groups <= 65535, "group_norm: too many groups");
  // a thread re-reads what it has not kept after it has written its own elements only: in place is safe
  if (n_rows == 0) return 0;
  const int part = dim / groups;
  int team = 1;
  while (team < 1024 && 8 * team < part) team *= 2;
  const int threads = team <= CWM_WAVE ? 256 : team, per = threads / team;
  const long n_parts = (long)n_rows * groups, blocks = (n_parts + per - 1) / per;
  auto wide_rows = [](const void* p, int dtype, long ld) { return ((uintptr_t)p % 16) == 0 && ld % (dtype == CWM_F32 ? 4 : 8) == 0; };
  const bool wide = part % 8 == 0 && wide_rows(src, src_dtype, src_ld) && wide_rows(src, src_dtype, partial_stride) && wide_rows(weight, w_dtype, 0) &&
                    wide_rows(dst, dst_dtype, dst_ld) && (!gate || wide_rows(gate, gate_dtype, gate_ld)) && (!copy || wide_rows(copy, copy_dtype, copy_ld));
#define CWM_GROUP_NORM(WIDE, GATED, ADDED)                                                                                                      \
  hipLaunchKernelGGL((group_norm_kernel<WIDE, GATED, ADDED>), dim3((unsigned)(blocks < 1 << 20 ? blocks : 1 << 20)), dim3(threads), 0, stream, \
                     src, src_dtype, src_ld, n_partials, partial_stride, gate, gate_dtype, gate_ld, weight, w_dtype, dst, dst_dtype, dst_ld, rows, \
                     n_parts, groups, part, team, eps, copy, copy_dtype, copy_ld)
#define CWM_GROUP_NORM_WIDE(GATED, ADDED)                                                      \
  do {                                                                                         \
    if (wide) CWM_GROUP_NORM(true, GATED, ADDED); else CWM_GROUP_NORM(false, GATED, ADDED);     \
  } while (0)
  if (gate) {
    if (accumulate) CWM_GROUP_NORM_WIDE(true, true); else CWM_GROUP_NORM_WIDE(true, false);
  } else {
    if (accumulate) CWM_GROUP_NORM_WIDE(false, true); else CWM_GROUP_NORM_WIDE(false, false);
  }
#undef CWM_GROUP_NORM_WIDE
#undef CWM_GROUP_NORM
  return cwm_launch_status("group_norm");
}

__global__ void __launch_bounds__(256) token_shift_kernel(const float* __restrict__ h, const float* __restrict__ mu, float* state,
                                                          const int* __restrict__ slots, const int* __restrict__ cu_q,
                                                          const int* __restrict__ seq_of_token, const int* __restrict__ positions,
                                                          void* __restrict__ out, int out_dtype, int dim, int n_slots, int write_state) {
  const int t = blockIdx.x;
  const int b = seq_of_token[t];
  const int first = cu_q[b];
  const bool head = t == first;
  const int slot = slots[b];
  const bool slot_ok = slot >= 0 && slot < n_slots;
  const bool fresh = positions[t] == 0;
  const size_t last = (size_t)(cu_q[b + 1] - 1) * dim;
  for (int i = threadIdx.x; i < dim; i += blockDim.x) {
    const float x = h[(size_t)t * dim + i];
    float prev;
    if (head) {
      prev = (fresh || !slot_ok) ? 0.f : state[(size_t)slot * dim + i];
      // the block of a portion's first token is the only one that touches the sequence's state: it reads what
      // the step before left and then leaves the portion's last row, element by element in one thread
      if (write_state && slot_ok) state[(size_t)slot * dim + i] = h[last + i];
    } else {
      prev = h[(size_t)(t - 1) * dim + i];
    }
    store_from_f32(out, out_dtype, (size_t)t * dim + i, x + (prev - x) * mu[i]);
  }
}

// The same, four values a thread at a time (dim: a multiple of 4, rows at multiples of 16 bytes, 8 for bfloat16 results): 2,048 tokens of width
// 2,048 7.6 instead of 10.7 us.
template <typename TO>
__global__ void __launch_bounds__(256) token_shift_four_kernel(const float* __restrict__ h, const float* __restrict__ mu, float* state,
                                                               const int* __restrict__ slots, const int* __restrict__ cu_q,
                                                               const int* __restrict__ seq_of_token, const int* __restrict__ positions,
                                                               TO* __restrict__ out, int dim, int n_slots, int write_state) {
  const int t = blockIdx.x;
  const int b = seq_of_token[t];
  const int first = cu_q[b];
  const bool head = t == first;
  const int slot = slots[b];
  const bool slot_ok = slot >= 0 && slot < n_slots;
  const bool fresh = positions[t] == 0;
  const size_t last = (size_t)(cu_q[b + 1] - 1) * dim;
  for (int i = 4 * threadIdx.x; i < dim; i += 4 * blockDim.x) {
    const float4 x = *(const float4*)(h + (size_t)t * dim + i), m = *(const float4*)(mu + i);
    float4 prev = make_float4(0.f, 0.f, 0.f, 0.f);
    if (head) {
      if (!fresh && slot_ok) prev = *(const float4*)(state + (size_t)slot * dim + i);
      if (write_state && slot_ok) *(float4*)(state + (size_t)slot * dim + i) = *(const float4*)(h + last + i);
    } else {
      prev = *(const float4*)(h + (size_t)(t - 1) * dim + i);
    }
    const float y0 = x.x + (prev.x - x.x) * m.x, y1 = x.y + (prev.y - x.y) * m.y, y2 = x.z + (prev.z - x.z) * m.z, y3 = x.w + (prev.w - x.w) * m.w;
    if constexpr (sizeof(TO) == 2)
      *(uint2*)(out + (size_t)t * dim + i) = make_uint2(pack2_bf16(y0, y1), pack2_bf16(y2, y3));
    else
      *(float4*)(out + (size_t)t * dim + i) = make_float4(y0, y1, y2, y3);
  }
}

extern "C" int cwm_token_shift(const float* h, const float* mu, float* state, const int* slots, const int* cu_q,
                               const int* seq_of_token, const int* positions, void* out, int out_dtype, int n_tokens, int dim,
                               int n_slots, int write_state, hipStream_t stream) {
  CWM_REQUIRE(h && mu && state && slots && cu_q && seq_of_token && positions && out, "token_shift: arguments missing");
  CWM_REQUIRE(n_tokens >= 0 && dim > 0 && n_slots > 0, "token_shift: bad sizes");
  if (n_tokens == 0) return 0;
  if (dim % 4 == 0 && (((uintptr_t)h | (uintptr_t)mu | (uintptr_t)state | (uintptr_t)out) % 16) == 0 && (out_dtype == CWM_BF16 || out_dtype == CWM_F32)) {
    if (out_dtype == CWM_BF16)
      hipLaunchKernelGGL(token_shift_four_kernel<bf16_t>, dim3(n_tokens), dim3(256), 0, stream, h, mu, state, slots, cu_q, seq_of_token, positions,
                         (bf16_t*)out, dim, n_slots, write_state);
    else
      hipLaunchKernelGGL(token_shift_four_kernel<float>, dim3(n_tokens), dim3(256), 0, stream, h, mu, state, slots, cu_q, seq_of_token, positions,
                         (float*)out, dim, n_slots, write_state);
    return cwm_launch_status("token_shift");
  }
  hipLaunchKernelGGL(token_shift_kernel, dim3(n_tokens), dim3(256), 0, stream, h, mu, state, slots, cu_q, seq_of_token, positions, out,
                     out_dtype, dim, n_slots, write_state);
  return cwm_launch_status("token_shift");
}

__global__ void __launch_bounds__(256) sigmoid_mul_kernel(const void* __restrict__ a, long a_ld, const void* __restrict__ g, long g_ld,
                                                          void* __restrict__ out, long out_ld, int dtype, int width) {
  const size_t t = blockIdx.x;
  for (int i = blockIdx.y * blockDim.x + threadIdx.x; i < width; i += gridDim.y * blockDim.x) {
    const float z = load_as_f32(g, dtype, t * g_ld + i);
    store_from_f32(out, dtype, t * out_ld + i, load_as_f32(a, dtype, t * a_ld + i) / (1.f + expf(-z)));
  }
}

// The same for bfloat16, eight values a thread (width and rows: multiples of 8 values, 16 bytes): 2,296 rows of 2,048 8.0 instead of 15.4 us.
__global__ void __launch_bounds__(256) sigmoid_mul_eight_kernel(const bf16_t* __restrict__ a, long a_ld, const bf16_t* __restrict__ g, long g_ld,
                                                                bf16_t* __restrict__ out, long out_ld, int width) {
  const size_t t = blockIdx.x;
  const int i = 8 * (blockIdx.y * blockDim.x + threadIdx.x);
  if (i >= width) return;
  const uint4 x = *(const uint4*)(a + t * a_ld + i), z = *(const uint4*)(g + t * g_ld + i);
  const uint32_t xs[4] = {x.x, x.y, x.z, x.w}, zs[4] = {z.x, z.y, z.z, z.w};
  uint32_t o[4];
#pragma unroll
  for (int c = 0; c < 4; ++c)
    o[c] = pack2_bf16(__uint_as_float(xs[c] << 16) / (1.f + expf(-__uint_as_float(zs[c] << 16))),
                      __uint_as_float(xs[c] & 0xffff0000u) / (1.f + expf(-__uint_as_float(zs[c] & 0xffff0000u))));
  *(uint4*)(out + t * out_ld + i) = make_uint4(o[0], o[1], o[2], o[3]);
}

extern "C" int cwm_sigmoid_mul(const void* a, long a_ld, const void* g, long g_ld, void* out, long out_ld, int dtype, int n_rows,
                               int width, hipStream_t stream) {
  CWM_REQUIRE(a && g && out && n_rows >= 0 && width > 0, "sigmoid_mul: bad arguments");
  if (n_rows == 0) return 0;
  if (dtype == CWM_BF16 && (width | a_ld | g_ld | out_ld) % 8 == 0 && (((uintptr_t)a | (uintptr_t)g | (uintptr_t)out) % 16) == 0 && width <= 8 * 256 * 65535) {
    hipLaunchKernelGGL(sigmoid_mul_eight_kernel, dim3(n_rows, (width / 8 + 255) / 256), dim3(256), 0, stream, (const bf16_t*)a, a_ld, (const bf16_t*)g, g_ld,
                       (bf16_t*)out, out_ld, width);
    return cwm_launch_status("sigmoid_mul");
  }
  int gy = (width + 1023) / 1024;
  hipLaunchKernelGGL(sigmoid_mul_kernel, dim3(n_rows, gy), dim3(256), 0, stream, a, a_ld, g, g_ld, out, out_ld, dtype, width);
  return cwm_launch_status("sigmoid_mul");
}

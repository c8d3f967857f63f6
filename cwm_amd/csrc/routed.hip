// Routed experts and other products in which every row has a weight matrix of its own choosing.
//
//   route_top        per token: the `top` largest of its router logits (the lower index wins a tie) and the softmax
//                    over those alone, float32; or, mode 1, the softmax over all experts, a choice by score plus a
//                    correction per expert, and weights that are the chosen scores times a scale.  Experts may form
//                    equal groups of neighbours, of which only those with the best members stay open to the choice.
//   group_by_expert  the step's (token, choice) pairs grouped by expert, each group padded to whole tiles of 16
//                    rows: row_token[row] (-1 in the padding), pair_row[pair], tile_expert[tile] (-1 beyond the
//                    last tile), and in a place of its own the number of tiles up to the last.  One block; no count leaves the
//                    device.  The order of a group's rows is whatever the block's atomic counters give: a row's
//                    result does not depend on its place.
//   grouped product  out[row] = W[e(row)] a[row] on the matrix cores, e from tile_expert (16 rows a tile share it)
//                    or, for a batch of independent products (one weight per head, say), from the block's z.
//                    bfloat16 operands on v_mfma_f32_16x16x32_bf16, float32 operands on v_mfma_f32_16x16x4_f32
//                    (exact products); float32 sums, in the order of k, or in four parts of it where the weights are
//                    streamed (the rows an expert has on average choose: a row's bits hang on the step by that rounding).
//                    With two weights the epilogue forms silu(W0 a) * (W1 a), or another form of `GateAct`.
//   combine          out[t] = sum_k weight[t][k] * rows[pair_row[t][k]] in the order of k, float32.
//
// Matrix-core layout as in the other products of this package: operand A = the weight tile (lane 16 j + r: row
// n0 + r, 8 values of k from 32 s + 8 j), operand B = the rows (lane 16 j + r: row r, the same k), result lane
// 16 j + r holds out[r][n0 + 4 j + i], i = 0..3.
#include "gemm_wide.h"

#include <type_traits>

CWM_DEFINE_ERROR_API

#define ROUTE_MAX_TOP 16
#define ROUTE_MAX_EXPERTS 256
#define TILE_ROWS 16

extern "C" int cwm_route_max_top() { return ROUTE_MAX_TOP; }
extern "C" int cwm_route_max_experts() { return ROUTE_MAX_EXPERTS; }
extern "C" int cwm_route_tile_rows() { return TILE_ROWS; }

// mode 0: the `top` largest logits, weights = softmax over those alone.
// mode 1: scores s = softmax over all experts; the `top` largest of s + correction (correction: null for none) are
//         chosen; weights = scale * s of the chosen, divided by their sum first if `renormalize`.
// One wavefront a token: lane l holds the experts l, l + 64, ...; a choice is a vote of the lanes (the larger value, the
// lower index among equals), so a token's router costs `top` rounds of shuffles whatever the number of experts.
#define ROUTE_PER_LANE (ROUTE_MAX_EXPERTS / CWM_WAVE)
// One token's router, by one wavefront: score[i] holds the logit of expert lane + 64 i (-inf beyond the last expert) on
// entry; the chosen experts and their weights are written by lane 0, to chosen_out / weights_out (`top` entries each)
// and, if given, to chosen_lds.
__device__ __forceinline__ void route_wave(float (&score)[ROUTE_MAX_EXPERTS / CWM_WAVE], int lane, int n_experts, int top, int mode,
                                           const float* __restrict__ correction, float scale, int renormalize,
                                           int n_groups, int keep_groups, int* __restrict__ chosen_out, float* __restrict__ weights_out,
                                              int* chosen_lds) {
  const float neg_inf = -__builtin_inff();
  float choice[ROUTE_PER_LANE];  // what an expert is chosen by; score: what a weight is made of
#pragma unroll
  for (int i = 0; i < ROUTE_PER_LANE; ++i) choice[i] = score[i];
  if (mode == 1) {
    float largest = score[0];
#pragma unroll
    for (int i = 1; i < ROUTE_PER_LANE; ++i) largest = fmaxf(largest, score[i]);
    largest = wave_max(largest);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < ROUTE_PER_LANE; ++i) {
      score[i] = lane + CWM_WAVE * i < n_experts ? expf(score[i] - largest) : 0.f;
      sum += score[i];
    }
    const float inv = 1.f / wave_sum(sum);
#pragma unroll
    for (int i = 0; i < ROUTE_PER_LANE; ++i) {
      const int e = lane + CWM_WAVE * i;
      score[i] *= inv;
      choice[i] = e < n_experts ? (correction ? score[i] + correction[e] : score[i]) : neg_inf;
    }
  }
  if (keep_groups < n_groups) {
    // the groups with the best members stay open: `keep_groups` votes, each for the best expert of the groups that are not
    // open yet (the lower index among equals), which opens its group; every other expert then leaves the choice
    const int size = n_experts / n_groups;
    bool open[ROUTE_PER_LANE];
#pragma unroll
    for (int i = 0; i < ROUTE_PER_LANE; ++i) open[i] = false;
    for (int k = 0; k < keep_groups; ++k) {
      float bv = neg_inf;
      int be = 0x7fffffff;
#pragma unroll
      for (int i = 0; i < ROUTE_PER_LANE; ++i) {
        const int e = lane + CWM_WAVE * i;
        if (e < n_experts && !open[i] && (be == 0x7fffffff || choice[i] > bv)) {
          bv = choice[i];
          be = e;
        }
      }
#pragma unroll
      for (int off = CWM_WAVE / 2; off > 0; off >>= 1) {
        const float ov = __shfl_xor(bv, off, CWM_WAVE);
        const int oe = __shfl_xor(be, off, CWM_WAVE);
        if (oe != 0x7fffffff && (be == 0x7fffffff || ov > bv || (ov == bv && oe < be))) {
          bv = ov;
          be = oe;
        }
      }
#pragma unroll
      for (int i = 0; i < ROUTE_PER_LANE; ++i) open[i] = open[i] || (lane + CWM_WAVE * i) / size == be / size;
    }
#pragma unroll
    for (int i = 0; i < ROUTE_PER_LANE; ++i)
      if (!open[i]) choice[i] = neg_inf;  // open experts are at least `top`, so the votes below end before these
  }
  int idx[ROUTE_MAX_TOP];
  float val[ROUTE_MAX_TOP];
#pragma unroll
  for (int k = 0; k < ROUTE_MAX_TOP; ++k) {
    idx[k] = -1;
    val[k] = 0.f;
  }
#pragma unroll
  for (int k = 0; k < ROUTE_MAX_TOP; ++k) {
    if (k < top) {
      // this lane's best expert that is not taken yet, then the wavefront's
      float bv = neg_inf, bs = 0.f;
      int be = 0x7fffffff;
#pragma unroll
      for (int i = 0; i < ROUTE_PER_LANE; ++i) {
        const int e = lane + CWM_WAVE * i;
        if (e < n_experts && (be == 0x7fffffff || choice[i] > bv)) {  // taken experts have left the vote (below)
          bool taken = false;
#pragma unroll
          for (int m = 0; m < ROUTE_MAX_TOP; ++m) taken |= (m < k && idx[m] == e);
          if (!taken) {
            bv = choice[i];
            bs = score[i];
            be = e;
          }
        }
      }
#pragma unroll
      for (int off = CWM_WAVE / 2; off > 0; off >>= 1) {
        const float ov = __shfl_xor(bv, off, CWM_WAVE), os = __shfl_xor(bs, off, CWM_WAVE);
        const int oe = __shfl_xor(be, off, CWM_WAVE);
        const bool theirs = oe != 0x7fffffff && (be == 0x7fffffff || ov > bv || (ov == bv && oe < be));
        if (theirs) {
          bv = ov;
          bs = os;
          be = oe;
        }
      }
      idx[k] = be;
      val[k] = bs;
    }
  }
  if (lane != 0) return;
  float sum = 0.f;
  if (mode == 0) {
    const float largest = val[0];  // the first chosen is the largest
#pragma unroll
    for (int k = 0; k < ROUTE_MAX_TOP; ++k)
      if (k < top) {
        val[k] = expf(val[k] - largest);
        sum += val[k];
      }
  } else {
#pragma unroll
    for (int k = 0; k < ROUTE_MAX_TOP; ++k)
      if (k < top) sum += val[k];
    if (!renormalize) sum = 1.f;
  }
#pragma unroll
  for (int k = 0; k < ROUTE_MAX_TOP; ++k)
    if (k < top) {
      chosen_out[k] = idx[k];
      if (chosen_lds) chosen_lds[k] = idx[k];
      weights_out[k] = mode == 0 ? val[k] / sum : scale * (val[k] / sum);
    }
}

// How many experts come before this lane's, by the larger value and the lower index among equals (a NaN before everything); the
// lanes beyond the experts keep their own number, so that all 64 are different.
__device__ __forceinline__ int route_place(float choice, int lane, int n_experts) {
  const uint32_t bits = __float_as_uint(choice + 0.f);  // -0 as 0
  const uint32_t key = choice != choice ? 0xffffffffu : bits >> 31 ? ~bits : bits | 0x80000000u;
  int place = 0;
#pragma unroll 8
  for (int e = 0; e < n_experts; ++e) {
    const uint32_t other = __builtin_amdgcn_readlane(key, e);
    place += other > key || (other == key && e < lane);
  }
  return lane < n_experts ? place : lane;
}

// The same choice for at most 64 experts, one a lane, without votes: every expert counts those before it and sends its score to
// the lane of its place.  A vote is a chain of 18 shuffles, and the kernel is nothing but that
// latency: 4 of 16 experts for eight tokens take 2.5 us, 7.0 with votes; 8 of 64 take 4.5, 10.2 with votes.
__device__ __forceinline__ void route_few(float score, int lane, int n_experts, int top, int mode, const float* __restrict__ correction,
                                          float scale, int renormalize, int n_groups, int keep_groups, int* __restrict__ chosen_out,
                                          float* __restrict__ weights_out) {
  float choice = score;
  if (mode == 1) {
    const float bias = correction && lane < n_experts ? correction[lane] : 0.f;
    const float largest = wave_max(score);
    score = lane < n_experts ? expf(score - largest) : 0.f;
    score *= 1.f / wave_sum(score);
    choice = correction ? score + bias : score;
  }
  int place = route_place(choice, lane, n_experts);
  if (keep_groups < n_groups) {
    // the groups whose best members come first stay open: a lane's group is as far forward as its first member
    const int size = n_experts / n_groups, group = lane / size;
    int front = CWM_WAVE;
    for (int e = 0; e < n_experts; ++e) {
      const int other = __builtin_amdgcn_readlane(place, e);
      if (e / size == group) front = min(front, other);
    }
    int before = 0;
    for (int g = 0; g < n_groups; ++g) before += __builtin_amdgcn_readlane(front, g * size) < front;
    if (before >= keep_groups) choice = -__builtin_inff();  // open experts are at least `top`
    place = route_place(choice, lane, n_experts);
  }
  const int expert = __builtin_amdgcn_ds_permute(4 * place, lane);
  float val = __int_as_float(__builtin_amdgcn_ds_permute(4 * place, __float_as_int(score)));
  auto of_lane = [&](int k) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(val), k)); };
  float sum = 1.f;
  if (mode == 0) val = expf(val - of_lane(0));  // the first chosen is the largest
  if (mode == 0 || renormalize) {
    sum = 0.f;
    for (int k = 0; k < top; ++k) sum += of_lane(k);
  }
  if (lane < top) {
    chosen_out[lane] = expert;
    weights_out[lane] = mode == 0 ? val / sum : scale * (val / sum);
  }
}

// FEW: at most as many experts as lanes.
template <bool FEW>
__global__ void __launch_bounds__(256) route_top_kernel(const float* __restrict__ logits, int* __restrict__ chosen,
                                                        float* __restrict__ weights, int n_tokens, int n_experts, int top, int mode,
                                                        const float* __restrict__ correction, float scale, int renormalize,
                                                        int n_groups, int keep_groups) {
  const int lane = threadIdx.x & (CWM_WAVE - 1);
  const int t = blockIdx.x * (blockDim.x / CWM_WAVE) + threadIdx.x / CWM_WAVE;
  if (t >= n_tokens) return;
  const float* z = logits + (size_t)t * n_experts;
  if constexpr (FEW) {
    route_few(lane < n_experts ? z[lane] : -__builtin_inff(), lane, n_experts, top, mode, correction, scale, renormalize, n_groups, keep_groups,
              chosen + (size_t)t * top, weights + (size_t)t * top);
    return;
  }
  float score[ROUTE_PER_LANE];
#pragma unroll
  for (int i = 0; i < ROUTE_PER_LANE; ++i) {
    const int e = lane + CWM_WAVE * i;
    score[i] = e < n_experts ? z[e] : -__builtin_inff();
  }
  route_wave(score, lane, n_experts, top, mode, correction, scale, renormalize, n_groups, keep_groups, chosen + (size_t)t * top, weights + (size_t)t * top, nullptr);
}

extern "C" int cwm_route_top(const float* logits, int* chosen, float* weights, int n_tokens, int n_experts, int top, int mode,
                             const float* correction, float scale, int renormalize, int n_groups, int keep_groups, hipStream_t stream) {
  CWM_REQUIRE(logits && chosen && weights, "route_top: arguments missing");
  CWM_REQUIRE(top >= 1 && top <= ROUTE_MAX_TOP && top <= n_experts, "route_top: %d of %d experts, the kernel takes up to %d", top, n_experts,
              ROUTE_MAX_TOP);
  CWM_REQUIRE(n_experts <= ROUTE_MAX_EXPERTS, "route_top: %d experts, the kernel takes up to %d", n_experts, ROUTE_MAX_EXPERTS);
  CWM_REQUIRE(mode == 0 || mode == 1, "route_top: unknown mode %d", mode);
  CWM_REQUIRE(n_groups >= 1 && n_experts % n_groups == 0 && keep_groups >= 1 && keep_groups <= n_groups &&
                  top <= keep_groups * (n_experts / n_groups),
              "route_top: %d of %d groups of %d experts do not hold %d choices", keep_groups, n_groups, n_experts, top);
  if (n_tokens <= 0) return 0;
  auto kernel = n_experts <= CWM_WAVE ? route_top_kernel<true> : route_top_kernel<false>;
  hipLaunchKernelGGL(kernel, dim3((n_tokens + 3) / 4), dim3(256), 0, stream, logits, chosen, weights, n_tokens, n_experts, top,
                     mode, correction, scale, renormalize, n_groups, keep_groups);
  return cwm_launch_status("route_top");
}

// The grouping, by one block; `chosen` may lie in global memory or in LDS.
__device__ __forceinline__ void group_pairs(const int* chosen, int n_pairs, int n_experts, int* __restrict__ row_token,
                                            int* __restrict__ pair_row, int* __restrict__ tile_expert, int* __restrict__ used, int n_tiles,
                                            int top, int tile_align, int* count, int* start) {
  for (int e = threadIdx.x; e < n_experts; e += blockDim.x) count[e] = 0;
  for (int i = threadIdx.x; i < n_tiles * TILE_ROWS; i += blockDim.x) row_token[i] = -1;
  __syncthreads();
  constexpr int HELD = 8;  // a thread's first choices stay in registers
  int held[HELD];
#pragma unroll
  for (int q = 0; q < HELD; ++q) {
    const int i = threadIdx.x + q * blockDim.x;
    held[q] = i < n_pairs ? chosen[i] : -1;
  }
  auto each_pair = [&](auto&& f) {
#pragma unroll
    for (int q = 0; q < HELD; ++q) {
      const int i = threadIdx.x + q * blockDim.x;
      if (i < n_pairs) f(i, held[q]);
    }
    for (int i = threadIdx.x + HELD * blockDim.x; i < n_pairs; i += blockDim.x) f(i, chosen[i]);
  };
  each_pair([&](int, int e) {
    if (e >= 0 && e < n_experts) atomicAdd(&count[e], 1);
  });
  __syncthreads();
  if (threadIdx.x < CWM_WAVE) {
    // four neighbouring experts a lane: an expert's tiles start at a multiple of tile_align behind the ones before
    const int lane = threadIdx.x;
    int tiles[4], sum = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int e = 4 * lane + q;
      tiles[q] = e < n_experts ? ((count[e] + TILE_ROWS - 1) / TILE_ROWS + tile_align - 1) / tile_align * tile_align : 0;
      sum += tiles[q];
    }
    int through = sum;
#pragma unroll
    for (int off = 1; off < CWM_WAVE; off <<= 1) {
      const int o = __shfl_up(through, off, CWM_WAVE);
      if (lane >= off) through += o;
    }
    int tile = through - sum;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (4 * lane + q < n_experts) start[4 * lane + q] = tile * TILE_ROWS;
      tile += tiles[q];
    }
    if (lane == CWM_WAVE - 1) *used = min(through, n_tiles);
  }
  __syncthreads();
  // tile by tile: the last expert that starts at it or before (those without rows start where the next one does)
  for (int i = threadIdx.x; i < n_tiles; i += blockDim.x) {
    int low = 0, high = n_experts - 1;
    while (low < high) {
      const int mid = (low + high + 1) >> 1;
      if (start[mid] <= i * TILE_ROWS) low = mid; else high = mid - 1;
    }
    tile_expert[i] = i * TILE_ROWS < start[low] + count[low] ? low : -1;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < n_experts; e += blockDim.x) count[e] = 0;
  __syncthreads();
  each_pair([&](int i, int e) {
    int row = -1;
    if (e >= 0 && e < n_experts) {
      row = start[e] + atomicAdd(&count[e], 1);
      if (row < n_tiles * TILE_ROWS)
        row_token[row] = i / top;
      else
        row = -1;
    }
    pair_row[i] = row;
  });
}

__global__ void __launch_bounds__(1024) group_by_expert_kernel(const int* __restrict__ chosen, int n_pairs, int n_experts,
                                                               int* __restrict__ row_token, int* __restrict__ pair_row,
                                                               int* __restrict__ tile_expert, int* __restrict__ used, int n_tiles, int top, int tile_align) {
  __shared__ int count[ROUTE_MAX_EXPERTS];
  __shared__ int start[ROUTE_MAX_EXPERTS];
  group_pairs(chosen, n_pairs, n_experts, row_token, pair_row, tile_expert, used, n_tiles, top, tile_align, count, start);
}

// Few tokens (a decode step): the router's product, the choice and the grouping in one launch of one block, each of which is a few
// microseconds of latency as a launch of its own (eight tokens, 16 experts, K = 2,048: 4.8 + 4.4 + 4.3 us).  The
// product is that of gemm_bf16_stream.hip on one tile of columns after the other, its sums in the same order: the 16 wavefronts
// share K, and add their parts through LDS.  Bound by its rounds of loads, four steps of 32 a wavefront at a time and one tile of 16
// experts after the other: `route_group_pays` says up to where that is less than three launches.  w: the router's streaming copy
// [tiles of 16 experts][K / 32][64][8].
#define ROUTE_GROUP_TOKENS 16
#define ROUTE_GROUP_STEPS 16  // of 32 along K, at most, a wavefront

// Without GROUP a block for every 16 tokens makes logits and choices alone: any number of tokens.  Logits as a product and then the choice /
// this, us, 16 experts: K = 2,048 17 tokens 8.6 / 6.0, 128 12.1 / 6.3, 2,048 8.3 / 6.4, 4,096 9.1 / 7.0; K = 1,024 7.1 to 12.2 / 6.0 to 6.5, 4,096 9.0 to 13.2 / 8.1 to 9.3.
template <bool GROUP>
__global__ void __launch_bounds__(1024) route_group_kernel(const bf16_t* __restrict__ x, long x_ld, const bf16_t* __restrict__ w,
                                                           const float* __restrict__ bias, int K, int n_tokens, int n_experts, int top, int mode,
                                                           const float* __restrict__ correction, float scale, int renormalize, int n_groups,
                                                           int keep_groups, int* __restrict__ chosen, float* __restrict__ weights,
                                                           int* __restrict__ row_token, int* __restrict__ pair_row, int* __restrict__ tile_expert,
                                                           int* __restrict__ used, int n_tiles, int tile_align) {
  __shared__ __attribute__((aligned(16))) float parts[16][256];
  __shared__ float logits[ROUTE_GROUP_TOKENS][CWM_WAVE];
  __shared__ int picks[ROUTE_GROUP_TOKENS * ROUTE_MAX_TOP];
  __shared__ int count[ROUTE_MAX_EXPERTS], start[ROUTE_MAX_EXPERTS];
  const int lane = threadIdx.x & (CWM_WAVE - 1), wave = threadIdx.x / CWM_WAVE;
  const int r = lane & 15, j = lane >> 4;
  const int steps = K / 32, each = (steps + 15) / 16, first = wave * each, last = min(steps, first + each);
  if constexpr (!GROUP) {
    const int done = blockIdx.x * ROUTE_GROUP_TOKENS;
    x += (size_t)done * x_ld;
    chosen += (size_t)done * top;
    weights += (size_t)done * top;
    n_tokens = min(ROUTE_GROUP_TOKENS, n_tokens - done);
  }
  const bf16_t* row = x + (size_t)min(r, n_tokens - 1) * x_ld + 8 * j;
  for (int n0 = 0; n0 < n_experts; n0 += 16) {
    const bf16_t* tile = w + ((size_t)(n0 / 16) * steps * 64 + lane) * 8;
    float4v acc = (float4v){0.f, 0.f, 0.f, 0.f};
    for (int s = first; s < last; s += 4) {
      Frag8 fx[4], fw[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int at = min(s + u, last - 1);
        fx[u].u = *(const uint4*)(row + 32 * at);
        fw[u].u = *(const uint4*)(tile + (size_t)at * 512);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (s + u < last) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[u].v, fx[u].v, acc, 0, 0, 0);
    }
    __syncthreads();
    *(float4v*)&parts[wave][r * 16 + 4 * j] = acc;  // [token][expert]
    __syncthreads();
    if (threadIdx.x < 256) {
      float sum = 0.f;
#pragma unroll
      for (int v = 0; v < 16; ++v) sum += parts[v][threadIdx.x];
      const int e = n0 + (threadIdx.x & 15);
      if (bias && e < n_experts) sum += bias[e];
      logits[threadIdx.x >> 4][e] = sum;
    }
  }
  __syncthreads();
  if (wave < n_tokens)
    route_few(lane < n_experts ? logits[wave][lane] : -__builtin_inff(), lane, n_experts, top, mode, correction, scale, renormalize, n_groups,
              keep_groups, GROUP ? picks + wave * top : chosen + (size_t)wave * top, weights + (size_t)wave * top);
  if constexpr (!GROUP) return;
  __syncthreads();
  for (int i = threadIdx.x; i < n_tokens * top; i += blockDim.x) chosen[i] = picks[i];
  group_pairs(picks, n_tokens * top, n_experts, row_token, pair_row, tile_expert, used, n_tiles, top, tile_align, count, start);
}

extern "C" int cwm_route_group_tokens() { return ROUTE_GROUP_TOKENS; }
extern "C" int cwm_route_group_experts() { return CWM_WAVE; }
extern "C" int cwm_route_group_max_k() { return 16 * 32 * ROUTE_GROUP_STEPS; }

// x: bfloat16 [n_tokens][x_ld]; w: the router's streaming copy; bias: float32 [n_experts] or null; the choice as in
// `cwm_route_top` for at most 64 experts, the lists as in `cwm_group_by_expert`.
extern "C" int cwm_route_group(const void* x, long x_ld, const void* w, const float* bias, int K, int n_tokens, int n_experts, int top, int mode,
                               const float* correction, float scale, int renormalize, int n_groups, int keep_groups, int* chosen,
                               float* weights, int* row_token, int* pair_row, int* tile_expert, int* used, int n_tiles, int tile_align,
                               hipStream_t stream) {
  CWM_REQUIRE(x && w && chosen && weights && row_token && pair_row && tile_expert && used, "route_group: arguments missing");
  CWM_REQUIRE(n_tokens >= 0 && n_tokens <= ROUTE_GROUP_TOKENS, "route_group: %d tokens, the kernel takes up to %d", n_tokens, ROUTE_GROUP_TOKENS);
  CWM_REQUIRE(n_experts >= 1 && n_experts <= CWM_WAVE && top >= 1 && top <= ROUTE_MAX_TOP && top <= n_experts, "route_group: %d of %d experts, the kernel takes up to %d of %d",
              top, n_experts, ROUTE_MAX_TOP, CWM_WAVE);
  CWM_REQUIRE(K >= 32 && K % 32 == 0 && K <= 16 * 32 * ROUTE_GROUP_STEPS && x_ld >= K && x_ld % 8 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0,
              "route_group: rows of %d elements must be a multiple of 32, up to %d, at multiples of 16 bytes", K, 16 * 32 * ROUTE_GROUP_STEPS);
  CWM_REQUIRE(mode == 0 || mode == 1, "route_group: unknown mode %d", mode);
  CWM_REQUIRE(n_groups >= 1 && n_experts % n_groups == 0 && keep_groups >= 1 && keep_groups <= n_groups && top <= keep_groups * (n_experts / n_groups),
              "route_group: %d of %d groups of %d experts do not hold %d choices", keep_groups, n_groups, n_experts, top);
  CWM_REQUIRE(tile_align >= 1 && (long)n_tiles >= ((long)n_tokens * top + TILE_ROWS - 1) / TILE_ROWS + (long)n_experts * tile_align,
              "route_group: %d tiles do not hold %d pairs of %d experts", n_tiles, n_tokens * top, n_experts);
  if (n_tokens == 0) return 0;
  hipLaunchKernelGGL(route_group_kernel<true>, dim3(1), dim3(1024), 0, stream, (const bf16_t*)x, x_ld, (const bf16_t*)w, bias, K, n_tokens, n_experts, top,
                     mode, correction, scale, renormalize, n_groups, keep_groups, chosen, weights, row_token, pair_row, tile_expert, used, n_tiles,
                     tile_align);
  return cwm_launch_status("route_group");
}

// The same without the lists, for any number of tokens.
extern "C" int cwm_route_rows(const void* x, long x_ld, const void* w, const float* bias, int K, int n_tokens, int n_experts, int top, int mode,
                              const float* correction, float scale, int renormalize, int n_groups, int keep_groups, int* chosen, float* weights,
                              hipStream_t stream) {
  CWM_REQUIRE(x && w && chosen && weights && n_tokens >= 0, "route_rows: arguments missing");
  CWM_REQUIRE(n_experts >= 1 && n_experts <= CWM_WAVE && top >= 1 && top <= ROUTE_MAX_TOP && top <= n_experts, "route_rows: %d of %d experts, the kernel takes up to %d of %d",
              top, n_experts, ROUTE_MAX_TOP, CWM_WAVE);
  CWM_REQUIRE(K >= 32 && K % 32 == 0 && K <= 16 * 32 * ROUTE_GROUP_STEPS && x_ld >= K && x_ld % 8 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0,
              "route_rows: rows of %d elements must be a multiple of 32, up to %d, at multiples of 16 bytes", K, 16 * 32 * ROUTE_GROUP_STEPS);
  CWM_REQUIRE(mode == 0 || mode == 1, "route_rows: unknown mode %d", mode);
  CWM_REQUIRE(n_groups >= 1 && n_experts % n_groups == 0 && keep_groups >= 1 && keep_groups <= n_groups && top <= keep_groups * (n_experts / n_groups),
              "route_rows: %d of %d groups of %d experts do not hold %d choices", keep_groups, n_groups, n_experts, top);
  if (n_tokens == 0) return 0;
  hipLaunchKernelGGL(route_group_kernel<false>, dim3((n_tokens + ROUTE_GROUP_TOKENS - 1) / ROUTE_GROUP_TOKENS), dim3(1024), 0, stream, (const bf16_t*)x, x_ld,
                     (const bf16_t*)w, bias, K, n_tokens, n_experts, top, mode, correction, scale, renormalize, n_groups, keep_groups, chosen, weights,
                     nullptr, nullptr, nullptr, nullptr, 0, 1);
  return cwm_launch_status("route_rows");
}

// used: one number, the tiles up to the last one that has rows, rounded up to tile_align.  tile_align: an expert's first tile lies at a multiple of so many tiles (the tiles that one block of the product takes).
extern "C" int cwm_group_by_expert(const int* chosen, int n_tokens, int top, int n_experts, int* row_token, int* pair_row,
                                   int* tile_expert, int* used, int n_tiles, int tile_align, hipStream_t stream) {
  CWM_REQUIRE(chosen && row_token && pair_row && tile_expert && used, "group_by_expert: arguments missing");
  CWM_REQUIRE(n_experts >= 1 && n_experts <= ROUTE_MAX_EXPERTS && top >= 1, "group_by_expert: %d experts, the kernel takes up to %d", n_experts,
              ROUTE_MAX_EXPERTS);
  const long n_pairs = (long)n_tokens * top;
  CWM_REQUIRE(tile_align >= 1 && (long)n_tiles >= (n_pairs + TILE_ROWS - 1) / TILE_ROWS + (long)n_experts * tile_align,
              "group_by_expert: %d tiles do not hold %ld pairs of %d experts", n_tiles, n_pairs, n_experts);
  if (n_tokens <= 0) return 0;
  hipLaunchKernelGGL(group_by_expert_kernel, dim3(1), dim3(1024), 0, stream, chosen, (int)n_pairs, n_experts, row_token, pair_row, tile_expert,
                     used, n_tiles, top, tile_align);
  return cwm_launch_status("group_by_expert");
}

// ---- the grouped product ------------------------------------------------------------------------------------- //
// What the epilogue of a product with two weights makes of g = W0 a and u = W1 a:
//   kind 0: silu(g) * u
//   kind 1: g' * sigmoid(alpha g') * (u' + 1) with g' = min(g, limit), u' = clamp(u, -limit, limit)
//   kind 2: gelu(g) * u, the tanh form of gelu
struct GateAct {
  int kind;
  float alpha, limit;
};
__device__ __forceinline__ float gated_value(float g, float u, const GateAct act) {
  if (act.kind == 1) {
    g = fminf(g, act.limit);
    u = fminf(fmaxf(u, -act.limit), act.limit);
    return g / (1.f + expf(-act.alpha * g)) * (u + 1.f);
  }
  if (act.kind == 2) return 0.5f * g * (1.f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g))) * u;
  return g / (1.f + expf(-g)) * u;
}

template <typename T> struct Frag;
template <> struct Frag<bf16_t> {
  static constexpr int K_STEP = 32;  // values of k one matrix instruction takes
  static constexpr int PER_LANE = 8;
  Frag8 f;
  __device__ __forceinline__ void zero() { f.u = make_uint4(0, 0, 0, 0); }
  __device__ __forceinline__ void load16(const bf16_t* p) { f.u = *(const uint4*)p; }
  __device__ __forceinline__ void load16_once(const bf16_t* p) { f.w = __builtin_nontemporal_load((const decltype(f.w)*)p); }
  __device__ __forceinline__ void load_some(const bf16_t* p, int n) {
    zero();
    for (int i = 0; i < PER_LANE; ++i)
      if (i < n) f.h[i] = p[i];
  }
  static __device__ __forceinline__ float4v mma(const Frag& w, const Frag& a, float4v acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.f.v, a.f.v, acc, 0, 0, 0);
  }
};
template <> struct Frag<float> {
  static constexpr int K_STEP = 16;  // four instructions of 4: lane group j supplies k = 4 j + e to instruction e
  static constexpr int PER_LANE = 4;
  float4 f;
  __device__ __forceinline__ void zero() { f = make_float4(0.f, 0.f, 0.f, 0.f); }
  __device__ __forceinline__ void load16(const float* p) { f = *(const float4*)p; }
  __device__ __forceinline__ void load_some(const float* p, int n) {
    f.x = n > 0 ? p[0] : 0.f;
    f.y = n > 1 ? p[1] : 0.f;
    f.z = n > 2 ? p[2] : 0.f;
    f.w = n > 3 ? p[3] : 0.f;
  }
  static __device__ __forceinline__ float4v mma(const Frag& w, const Frag& a, float4v acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w.f.x, a.f.x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w.f.y, a.f.y, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w.f.z, a.f.z, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w.f.w, a.f.w, acc, 0, 0, 0);
    return acc;
  }
};

// A block of four wavefronts, WR of them down the rows and 4 / WR along the columns, takes WR * RT row tiles of one
// expert (they follow one another in the list, and an expert's tiles start at a multiple of that many) and
// (4 / WR) * CT * 16 columns; a wavefront multiplies RT row tiles by CT column tiles, so each piece of a weight tile
// it loads serves RT tiles of rows and each piece of rows CT tiles of columns.  Shapes in use: 1 x 1 tiles a
// wavefront, four wavefronts along the columns (few rows an expert: many blocks stream the weights); 4 x 1 likewise;
// 4 x 4 (4 x 2 with two weights) with the wavefronts 2 x 2 (many rows an expert).
// VEC: rows of a and W start at multiples of 16 bytes and K is a multiple of a lane's piece.
template <typename T, int RT, int CT, int WR, bool GATED, bool VEC>
__global__ void __launch_bounds__(256) grouped_product_kernel(const T* __restrict__ a, long a_ld, long a_batch, const int* __restrict__ row_token,
                                                              const T* __restrict__ w0, const T* __restrict__ w1, long w_stride,
                                                              const int* __restrict__ tile_expert, int n_tiles, void* __restrict__ out,
                                                              int out_dtype, long out_ld, long out_batch, int n_rows, int N, int K, GateAct act) {
  constexpr int WC = 4 / WR;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wave_r = wave / WC, wave_c = wave % WC;
  const int r = lane & 15, j = lane >> 4;
  const int block_tile0 = blockIdx.x * (WR * RT);
  const int tile0 = block_tile0 + wave_r * RT;
  int expert;
  if (tile_expert) {
    expert = block_tile0 < n_tiles ? tile_expert[block_tile0] : -1;
    if (expert < 0) return;
  } else {
    expert = blockIdx.z;
  }
  const int n0 = (blockIdx.y * WC + wave_c) * CT * 16;
  if (n0 >= N) return;
  const T* wrow0[CT];
  const T* wrow1[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int col = n0 + ct * 16 + r;
    const size_t at = (size_t)expert * w_stride + (size_t)(col < N ? col : N - 1) * K;
    wrow0[ct] = w0 + at;
    wrow1[ct] = GATED ? w1 + at : nullptr;
  }
  const T* arow[RT];
  bool tile_live[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int tile = tile0 + rt;
    // a tile of another expert, or beyond the rows, is left out
    tile_live[rt] = tile_expert ? (tile < n_tiles && tile_expert[tile] == expert) : tile * TILE_ROWS < n_rows;
    const int row = tile * TILE_ROWS + r;
    long src = -1;
    if (tile_live[rt]) src = row_token ? row_token[row] : (row < n_rows ? row : -1);
    arow[rt] = src >= 0 ? a + (size_t)blockIdx.z * a_batch + (size_t)src * a_ld : nullptr;
  }
  float4v acc0[RT][CT], acc1[RT][CT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc0[rt][ct] = acc1[rt][ct] = (float4v){0.f, 0.f, 0.f, 0.f};
  constexpr int STEP = Frag<T>::K_STEP, PIECE = Frag<T>::PER_LANE;
  // two sets of operands: while one is multiplied, the loads of the next step are in flight
  auto load_set = [&](Frag<T> (&fw0)[CT], Frag<T> (&fw1)[CT], Frag<T> (&fa)[RT], int k0) {
    const int k = k0 + j * PIECE;
    const int left = K - k;  // values of this lane's piece inside K
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      if (VEC) {
        if (left > 0) {
          fw0[ct].load16(wrow0[ct] + k);
          if (GATED) fw1[ct].load16(wrow1[ct] + k);
        } else {
          fw0[ct].zero();
          if (GATED) fw1[ct].zero();
        }
      } else {
        fw0[ct].load_some(wrow0[ct] + k, left);
        if (GATED) fw1[ct].load_some(wrow1[ct] + k, left);
      }
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      if (!arow[rt] || left <= 0)
        fa[rt].zero();
      else if (VEC)
        fa[rt].load16(arow[rt] + k);
      else
        fa[rt].load_some(arow[rt] + k, left);
    }
  };
  auto multiply = [&](const Frag<T> (&fw0)[CT], const Frag<T> (&fw1)[CT], const Frag<T> (&fa)[RT]) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        acc0[rt][ct] = Frag<T>::mma(fw0[ct], fa[rt], acc0[rt][ct]);
        if (GATED) acc1[rt][ct] = Frag<T>::mma(fw1[ct], fa[rt], acc1[rt][ct]);
      }
  };
  Frag<T> w0a[CT], w1a[CT], ra[RT], w0b[CT], w1b[CT], rb[RT];
  load_set(w0a, w1a, ra, 0);
  for (int k0 = 0; k0 < K; k0 += 2 * STEP) {
    load_set(w0b, w1b, rb, k0 + STEP);  // beyond K: zeros
    multiply(w0a, w1a, ra);
    load_set(w0a, w1a, ra, k0 + 2 * STEP);
    multiply(w0b, w1b, rb);
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    if (!tile_live[rt]) continue;
    const int row = (tile0 + rt) * TILE_ROWS + r;
    if (!tile_expert && row >= n_rows) continue;
    const size_t base = (size_t)blockIdx.z * out_batch + (size_t)row * out_ld;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = n0 + ct * 16 + 4 * j + i;
        if (c >= N) continue;
        float v = acc0[rt][ct][i];
        if (GATED) v = gated_value(v, acc1[rt][ct][i], act);
        if (out_dtype == CWM_F32)
          ((float*)out)[base + c] = v;
        else
          ((bf16_t*)out)[base + c] = f32_to_bf16(v);
      }
  }
}

// Few rows an expert (a decode step): the product is bound by streaming the chosen experts' weights once.  A block
// takes one row tile and 16 columns; its four wavefronts split K (wavefront w the steps w, w + 4, ...: together they
// read whole lines of a weight row), each with STREAM_DEPTH steps of operands in flight while the ones before are
// multiplied, and add their sums through LDS in the order of w.  Rows of a and W start at multiples of 16 bytes.  TILED: weights in
// operand tiles, whose lines are read once and past the caches (eight tokens, 14 of 16 experts of 2,048 x 1,024: gate and up 24 us,
// row-major 27).
#define STREAM_DEPTH 4

template <typename T, bool GATED, bool TILED>
__global__ void __launch_bounds__(256) grouped_stream_kernel(const T* __restrict__ a, long a_ld, long a_batch, const int* __restrict__ row_token,
                                                             const T* __restrict__ w0, const T* __restrict__ w1, long w_stride,
                                                             const int* __restrict__ tile_expert, int n_tiles, void* __restrict__ out,
                                                             int out_dtype, long out_ld, long out_batch, int n_rows, int N, int K, GateAct act,
                                                             int tile_align) {
  __shared__ float sums[4][GATED ? 2 : 1][64][4];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int r = lane & 15, j = lane >> 4;
  int tile = blockIdx.x;
  int expert;
  if (tile_expert) {
    // the first tiles of the list's multiples, then the second ones, ...: few experts have a second tile, and blocks without
    // work in regular places would leave whole XCDs without (they are dealt to the XCDs in turn; 22 and 35 us)
    const int multiples = n_tiles / tile_align;
    if (tile < multiples * tile_align) tile = tile % multiples * tile_align + tile / multiples;
    expert = tile < n_tiles ? tile_expert[tile] : -1;
    if (expert < 0) return;
  } else {
    expert = blockIdx.z;
  }
  const int n0 = blockIdx.y * 16;
  const int col = n0 + r;
  const size_t at = (size_t)expert * w_stride + (TILED ? ((size_t)blockIdx.y * (K / 32) * 64 + lane) * 8 : (size_t)(col < N ? col : N - 1) * K);
  const T* wrow0 = w0 + at;
  const T* wrow1 = GATED ? w1 + at : nullptr;
  const int row = tile * TILE_ROWS + r;
  long src = row_token ? row_token[row] : (row < n_rows ? row : -1);
  const T* arow = src >= 0 ? a + (size_t)blockIdx.z * a_batch + (size_t)src * a_ld : nullptr;
  constexpr int STEP = Frag<T>::K_STEP, PIECE = Frag<T>::PER_LANE;
  const int steps = (K + STEP - 1) / STEP;
  float4v acc0 = (float4v){0.f, 0.f, 0.f, 0.f}, acc1 = acc0;
  auto load_group = [&](Frag<T> (&fw0)[STREAM_DEPTH], Frag<T> (&fw1)[STREAM_DEPTH], Frag<T> (&fa)[STREAM_DEPTH], int first) {
#pragma unroll
    for (int d = 0; d < STREAM_DEPTH; ++d) {
      const int step = wave + 4 * (first + d);
      const int k = step * STEP + j * PIECE;
      if (step < steps && k < K) {
        if constexpr (TILED) {
          fw0[d].load16_once(wrow0 + (size_t)step * 512);
          if (GATED) fw1[d].load16_once(wrow1 + (size_t)step * 512);
        } else {
          fw0[d].load16(wrow0 + k);
          if (GATED) fw1[d].load16(wrow1 + k);
        }
        if (arow) fa[d].load16(arow + k); else fa[d].zero();
      } else {
        fw0[d].zero();
        if (GATED) fw1[d].zero();
        fa[d].zero();
      }
    }
  };
  auto multiply_group = [&](const Frag<T> (&fw0)[STREAM_DEPTH], const Frag<T> (&fw1)[STREAM_DEPTH], const Frag<T> (&fa)[STREAM_DEPTH]) {
#pragma unroll
    for (int d = 0; d < STREAM_DEPTH; ++d) {
      acc0 = Frag<T>::mma(fw0[d], fa[d], acc0);
      if (GATED) acc1 = Frag<T>::mma(fw1[d], fa[d], acc1);
    }
  };
  Frag<T> w0a[STREAM_DEPTH], w1a[STREAM_DEPTH], ra[STREAM_DEPTH], w0b[STREAM_DEPTH], w1b[STREAM_DEPTH], rb[STREAM_DEPTH];
  const int groups = (steps + 4 * STREAM_DEPTH - 1) / (4 * STREAM_DEPTH);  // of STREAM_DEPTH steps a wavefront
  load_group(w0a, w1a, ra, 0);
  for (int g = 0; g < groups; g += 2) {
    load_group(w0b, w1b, rb, (g + 1) * STREAM_DEPTH);  // beyond K: zeros
    multiply_group(w0a, w1a, ra);
    load_group(w0a, w1a, ra, (g + 2) * STREAM_DEPTH);
    multiply_group(w0b, w1b, rb);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    sums[wave][0][lane][i] = acc0[i];
    if (GATED) sums[wave][GATED ? 1 : 0][lane][i] = acc1[i];
  }
  __syncthreads();
  if (wave != 0) return;
  if (!tile_expert && row >= n_rows) return;
  const size_t base = (size_t)blockIdx.z * out_batch + (size_t)row * out_ld;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = n0 + 4 * j + i;
    if (c >= N) continue;
    float v = ((sums[0][0][lane][i] + sums[1][0][lane][i]) + sums[2][0][lane][i]) + sums[3][0][lane][i];
    if (GATED) {
      const float u = ((sums[0][GATED ? 1 : 0][lane][i] + sums[1][GATED ? 1 : 0][lane][i]) + sums[2][GATED ? 1 : 0][lane][i]) + sums[3][GATED ? 1 : 0][lane][i];
      v = gated_value(v, u, act);
    }
    if (out_dtype == CWM_F32)
      ((float*)out)[base + c] = v;
    else
      ((bf16_t*)out)[base + c] = f32_to_bf16(v);
  }
}

// Many rows an expert, bfloat16, K a multiple of 64: a block of four wavefronts takes RT row tiles of one expert and 64 CT
// rows of weights, 64 values of k a step.  Every wavefront multiplies all of the block's rows by CT weight tiles of its own
// (with two weights half of them of each), so a piece of a weight tile is needed by one wavefront alone: it goes straight
// to registers, half a step ahead of its use, and only the rows go through LDS (two buffers; 16-byte pieces, a row's pieces
// XOR-swizzled by the row so that the lanes of a matrix operand read different banks).  That leaves LDS, which bounds a
// block whose wavefronts share both operands, 40% busy beside the matrix cores.
// With a list the blocks are numbered so that an XCD gets a run of neighbours in the order (group of WIDE_GROUP row blocks,
// columns, row block): the row blocks of an expert then share its weights in one L2, where dealing them to the XCDs in turn
// has every XCD read every expert's weights.  `used` says how many tiles of the list are in use, so the runs are equally long.
// TILED: the weights lie in operand tiles (an expert's [N / 16][K / 32][64 lanes][8 values]), 1 KB of consecutive memory a load.
// Read from row-major weights, a load is 16 rows' pieces of 64 bytes, four neighbouring lanes in four rows, which costs the
// vector memory path a lookup a lane: with half or all of a block's products left out the kernel took as long.  An expert's
// last block multiplies as many row tiles as it has (2, 4 or 8).
// 16 experts of 2,048 x 1,024, four a token, gate and up / down, operand tiles and row-major: 2,048 tokens evenly loaded 74 / 46 us
// (924 / 743 TFLOP/s) and 105 / 58; with a router's uneven loads 100 / 58 and 135 / 76 (a CU that gets three blocks where others
// get two decides), 1,500 tokens 72 / 42 and 97 / 53, 4,096 tokens 159 / 99 and 204 / 121, 300 tokens 38 / 20 and 42 / 21.
#define WIDE_GROUP 4

// A wavefront's and a block's place in a wide product, and what its loop needs of the kernel's arguments.
struct WideBlock {
  const bf16_t* a;
  long a_ld;
  const int* row_token;  // with a list: the token of each of its rows, or null
  const bf16_t *w0, *w1;  // the block's expert's
  const int* tile_expert;
  int n_tiles, expert, tile0, n0, n_rows, N, K;
};

// A barrier that waits for the wavefront's LDS accesses only, not for the global loads on their way.
__device__ __forceinline__ void wide_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory"); }

template <int RT, int CT, bool GATED, bool TILED, int BLOCK_ROWS>
__device__ __forceinline__ void wide_rows(const WideBlock& wb, uint4 (*lds_rows)[BLOCK_ROWS * 8], void* __restrict__ out, int out_dtype,
                                          size_t out_base, long out_ld, int vec_out, GateAct act) {
  constexpr int ROWS = RT * TILE_ROWS, FETCH = ROWS * 8 / 256;  // 16-byte pieces of the rows that a thread fetches a step
  constexpr int WT = GATED ? CT / 2 : CT;                       // column tiles of the result a wavefront makes
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, j = lane >> 4;
  const int tile0 = wb.tile0, n0 = wb.n0, N = wb.N, K = wb.K;
  // rows that do not exist, and those of tiles that are another expert's, are read from a row that does; nothing uses the results
  uint32_t src_a[FETCH];  // in pieces: rows are whole pieces long
#pragma unroll
  for (int i = 0; i < FETCH; ++i) {
    const int list_row = tile0 * TILE_ROWS + (threadIdx.x >> 3) + 32 * i;
    int src;
    if (wb.tile_expert)
      src = list_row >= wb.n_tiles * TILE_ROWS ? 0 : wb.row_token ? max(wb.row_token[list_row], 0) : min(list_row, wb.n_rows - 1);
    else
      src = min(list_row, wb.n_rows - 1);
    src_a[i] = (uint32_t)src * (uint32_t)(wb.a_ld / 8) + (threadIdx.x & 7);
  }
  uint32_t src_w[CT];  // N * K < 2^31
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int n = n0 + (ct % WT) * 16;
    src_w[ct] = TILED ? (uint32_t)min(n, N - 16) * (uint32_t)K + lane * 8 : (uint32_t)min(n + r, N - 1) * (uint32_t)K + j * 8;
  }
  typedef uint32_t Words4 __attribute__((ext_vector_type(4)));
  Words4 ra[FETCH];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < FETCH; ++i) ra[i] = *((const Words4*)wb.a + src_a[i] + (uint32_t)k0 / 8);
  };
  const int staged = (threadIdx.x & ~7) + ((threadIdx.x & 7) ^ ((threadIdx.x >> 3) & 7));
  auto stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < FETCH; ++i) *(Words4*)&lds_rows[buf][staged + 256 * i] = ra[i];
  };
  Frag8 fw[2][CT];
  auto load_weights = [&](int half, int k0) {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) fw[half][ct].u = *(const uint4*)((ct < WT ? wb.w0 : wb.w1) + (src_w[ct] + (TILED ? (uint32_t)(k0 * 16 + 512 * half) : (uint32_t)(k0 + 32 * half))));
  };
  float4v acc[RT][CT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = (float4v){0.f, 0.f, 0.f, 0.f};
  const int steps = K / 64;
  auto place = [&](int step) { return min(step, steps - 1) * 64; };
  fetch(0);
  load_weights(0, 0);
  load_weights(1, 0);
  stage(0);
  fetch(place(1));
  wide_barrier();
  // No branch in the loop (the last steps load again what they have): with one around a load the compiler waits for the
  // load where the paths meet.  The scheduling barriers keep the loads where they are, ahead of the other half's products.
  for (int step = 0; step < steps; ++step) {
    const uint4* rows = lds_rows[step & 1];
    const int next = place(step + 1);
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int piece = half * 4 + j;
      Frag8 fa[RT];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) fa[rt].u = rows[(rt * 16 + r) * 8 + (piece ^ (r & 7))];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[half][ct].v, fa[rt].v, acc[rt][ct], 0, 0, 0);
      load_weights(half, next);
      __builtin_amdgcn_sched_barrier(0);
    }
    stage((step + 1) & 1);
    __builtin_amdgcn_sched_barrier(0);
    fetch(place(step + 2));
    wide_barrier();
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int tile = tile0 + rt, row = tile * TILE_ROWS + r;
    if (wb.tile_expert ? !(tile < wb.n_tiles && wb.tile_expert[tile] == wb.expert) : row >= wb.n_rows) continue;
    const size_t base = out_base + (size_t)row * out_ld;
#pragma unroll
    for (int ct = 0; ct < WT; ++ct) {
      const int c = n0 + ct * 16 + 4 * j;  // four adjacent columns
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = GATED ? gated_value(acc[rt][ct][i], acc[rt][ct + (GATED ? WT : 0)][i], act) : acc[rt][ct][i];
      if (vec_out && c + 3 < N) {
        if (out_dtype == CWM_F32)
          *(float4*)((float*)out + base + c) = make_float4(v[0], v[1], v[2], v[3]);
        else
          *(uint2*)((bf16_t*)out + base + c) = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
        continue;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (c + i >= N) continue;
        if (out_dtype == CWM_F32)
          ((float*)out)[base + c + i] = v[i];
        else
          ((bf16_t*)out)[base + c + i] = f32_to_bf16(v[i]);
      }
    }
  }
}

template <int RT, int CT, bool GATED, bool TILED>
__global__ void __launch_bounds__(256, 2) grouped_wide_kernel(const bf16_t* __restrict__ a, long a_ld, long a_batch, const int* __restrict__ row_token,
                                                              const bf16_t* __restrict__ w0, const bf16_t* __restrict__ w1, long w_stride,
                                                              const int* __restrict__ tile_expert, const int* __restrict__ used, int n_tiles,
                                                              int row_blocks, int col_blocks,
                                                              void* __restrict__ out, int out_dtype, long out_ld, long out_batch, int vec_out,
                                                              int n_rows, int N, int K, GateAct act) {
  constexpr int WT = GATED ? CT / 2 : CT;
  __shared__ uint4 lds_rows[2][RT * TILE_ROWS * 8];
  const int wave = threadIdx.x >> 6;
  int bx, by, expert, live_tiles;
  if (tile_expert) {
    const int live = ((used ? min(*used, n_tiles) : n_tiles) + RT - 1) / RT, total = live * col_blocks;
    const int run = (total + 7) >> 3, at = (int)(blockIdx.x & 7) * run + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= run || at >= total) return;
    const int first = at / (WIDE_GROUP * col_blocks) * WIDE_GROUP, rest = at - first * col_blocks;
    const int together = min(WIDE_GROUP, live - first);
    bx = first + rest % together;
    by = rest / together;
    expert = tile_expert[bx * RT];
    if (expert < 0) return;
    live_tiles = 1;
#pragma unroll
    for (int t = 1; t < RT; ++t) live_tiles += bx * RT + t < n_tiles && tile_expert[min(bx * RT + t, n_tiles - 1)] == expert;
  } else {
    bx = blockIdx.x % row_blocks;
    by = blockIdx.x / row_blocks;
    expert = blockIdx.z;
    live_tiles = (n_rows + TILE_ROWS - 1) / TILE_ROWS - bx * RT;
  }
  const WideBlock wb = {a + (size_t)blockIdx.z * a_batch, a_ld, row_token, w0 + (size_t)expert * w_stride, GATED ? w1 + (size_t)expert * w_stride : nullptr,
                        tile_expert, n_tiles, expert, bx * RT, by * (64 * WT) + wave * (16 * WT), n_rows, N, K};
  const size_t out_base = (size_t)blockIdx.z * out_batch;
  // an expert's last block takes as many row tiles as it has, rounded up to 2, 4 or 8: the others' products would be for padding
  auto go = [&](auto tiles) {
    if constexpr (decltype(tiles)::value <= RT)
      wide_rows<decltype(tiles)::value, CT, GATED, TILED, RT * TILE_ROWS>(wb, lds_rows, out, out_dtype, out_base, out_ld, vec_out, act);
  };
  if (RT >= 8 && live_tiles > 4)
    go(std::integral_constant<int, 8>());
  else if (RT >= 4 && live_tiles > 2)
    go(std::integral_constant<int, 4>());
  else
    go(std::integral_constant<int, 2>());
}

// ---- many rows an expert, weights in operand tiles: the loop of gemm_wide.h ---------------------------------------------- //
// What bounded the kernel above was its last round of blocks (two a compute unit; 576 on 512 places take 100 us where 512 take 74) and
// the weights' way through registers, a step ahead.  Here 256 blocks stay, one a compute unit, and rows and weights are on their way two steps
// ahead by direct loads, the rows gathered by the loads' own addresses.  A tile is a list's block of 128 rows of one expert and 256 columns
// of its weights (gated: 128 gates and the same ups).  What whole rounds of such tiles leave over, where it would fill less than half of a
// round, goes in quarters, 64 rows by 128 columns, over all blocks.  The sums' order is that of the kernel above, and so are the bits.
// 16 experts of 2,048 x 1,024, four a token, uneven loads, the kernel above / this, gate and up, then down, us: 2,048 tokens 111 / 92 and 59 / 51,
// 700 50 / 43 and 25 / 25, 4,096 161 / 153 and 101 / 95; 32 of 3,072 x 1,536, 1,000 tokens 174 / 156 and 105 / 90; 8 of 512 x 320, 300 tokens
// 14.0 / 8.6 and 8.3 / 6.5; but 1,500 tokens, whose second round is two thirds full, 72 / 75 and 40 / 41:
// the caller's rule (`_loop_pays`) leaves such, and others that were not ahead, to it.
#define GROUPED_BLOCKS 256
typedef const __attribute__((address_space(4))) int* list_ints;  // read by scalar loads, which do not wait for the loads under way

struct GroupedWide {
  const bf16_t* a;
  long a_ld;
  list_ints row_token;  // or null: the list's own rows
  const bf16_t *w0, *w1;
  long w_stride;
  list_ints tile_expert;
  int n_tiles, N, K;
  int row_blocks, col_blocks;  // of whole tiles: 8 row tiles, 256 columns of weights
  void* out;
  long out_ld;
  GateAct act;
  // tile t in the order (group of WIDE_GROUP row blocks, column block, row block of the group); quarters of a tile follow one another
  __host__ __device__ __forceinline__ void place(int t, bool quarters, int& tile0, int& col) const {
    const int whole = quarters ? t >> 2 : t;
    const int first = whole / (WIDE_GROUP * col_blocks) * WIDE_GROUP, rest = whole - first * col_blocks;
    const int together = min(WIDE_GROUP, row_blocks - first);
    tile0 = (first + rest % together) * 8 + (quarters ? (t & 1) * 4 : 0);
    col = rest / together * 2 + (quarters ? (t >> 1) & 1 : 0);
    if (!quarters) col >>= 1;
  }
  // the row that a tile's loads start from, and how far past it its row `row` is read: rows past the list are its last one again.  A list whose
  // tiles in use are not counted may end inside a block, and the lower quarters of that block begin past it
  __host__ __device__ __forceinline__ int first_row(int tile0) const { return min(tile0, n_tiles - 1) * TILE_ROWS; }
  __host__ __device__ __forceinline__ int from_first(int tile0, int row) const { return min(row, n_tiles * TILE_ROWS - 1 - first_row(tile0)); }
};

// for tests: what `from_first` gives for tile `t` of a list of `n_tiles`, and the row it counts from
extern "C" int cwm_grouped_loop_rows(int n_tiles, int col_blocks, int t, int quarters, int row, int* first) {
  GroupedWide g = {};
  g.n_tiles = n_tiles, g.row_blocks = (n_tiles + 7) / 8, g.col_blocks = col_blocks;
  int tile0, col;
  g.place(t, quarters != 0, tile0, col);
  *first = g.first_row(tile0);
  return g.from_first(tile0, row);
}

// the same for all lanes, which the compiler cannot see behind a list's entry
__device__ __forceinline__ const bf16_t* same_for_all(const bf16_t* p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t high = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32)), low = __builtin_amdgcn_readfirstlane((uint32_t)v);  // unsigned: the builtin's int would extend its sign
  return (const bf16_t*)((uint64_t)high << 32 | low);
}

template <int WM, int WN, bool GATED, bool QUARTERS>
struct GroupedSource {
  const GroupedWide g;
  int lane, wave;
  const bf16_t *a, *u0;
  long up;  // from the gates' weights to the ups'
  uint32_t off[WideShape<WM, WN>::ND];
  static constexpr bool W_TILES = true;
  static constexpr int BM = WideShape<WM, WN>::BM;
  __device__ __forceinline__ const bf16_t* base(int p) const {
    const int q = p - BM / 8;
    return q < 0 ? a : u0 + (GATED && (q >> 1) % WN >= WN / 2 ? up : 0);
  }
  __device__ __forceinline__ void enter(int tile) {
    int tile0, col;
    g.place(tile, QUARTERS, tile0, col);
    const int expert = __builtin_amdgcn_readfirstlane(max(0, g.tile_expert[tile0 / 8 * 8]));
    a = g.row_token ? g.a : g.a + (size_t)g.first_row(tile0) * g.a_ld;
    u0 = g.w0 + (size_t)expert * g.w_stride;
    a = same_for_all(a), u0 = same_for_all(u0);
    const int last_row = g.n_tiles * TILE_ROWS - 1;
#pragma unroll
    for (int i = 0; i < WideShape<WM, WN>::ND; ++i) {
      const int p = min(wave + 8 * i, WideShape<WM, WN>::PIECES - 1);
      if (p < BM / 8) {
        const int row = 8 * p + (lane >> 3);
        int from = g.from_first(tile0, row);
        if (g.row_token) {  // eight rows, eight scalars; padding reads token 0
          const int at = min(tile0 * TILE_ROWS + 8 * p, last_row - 7);
          int token[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            token[e] = g.row_token[at + e];
            asm volatile("" : "+s"(token[e]));  // or the compiler makes it a load of each lane's own, behind all that are under way
          }
          from = token[0];
#pragma unroll
          for (int e = 1; e < 8; ++e) from = (lane >> 3) == e ? token[e] : from;
          from = max(0, from);
        }
        off[i] = (uint32_t)(from * (int)(g.a_ld / 8) + ((lane & 7) ^ ((row >> 1) & 7))) * 16u;
      } else {
        const int q = p - BM / 8, wn = q / (2 * WN), b = (q >> 1) % WN, half = q & 1;
        constexpr int WT = GATED ? WN / 2 : WN;  // column tiles of a wavefront
        const int n_tile = min((col * 4 + wn) * WT + b % WT, g.N / 16 - 1);  // columns past the last: theirs are not stored
        off[i] = (uint32_t)(n_tile * (g.K / 32) + half) * 1024u + 16u * lane;
      }
    }
  }
};

template <int WM, int WN, typename TC, bool GATED, bool QUARTERS>
struct GroupedSink {
  const GroupedWide g;
  int lane, wave;
  static constexpr int WT = GATED ? WN / 2 : WN, STORES = WM * WT;
  __device__ __forceinline__ bool store(int tile, float4v (&acc)[WM][WN]) const {
    int tile0, col;
    g.place(tile, QUARTERS, tile0, col);
    const int expert = g.tile_expert[tile0 / 8 * 8];
    const int r = lane & 15, j = lane >> 4, wm = wave >> 2, wn = wave & 3;
    const int n0 = (col * 4 + wn) * WT * 16 + 4 * j;
    bool whole = (col + 1) * 4 * WT * 16 <= g.N;
#pragma unroll
    for (int a = 0; a < WM; ++a) {
      const int t = tile0 + wm * WM + a;
      const bool live = t < g.n_tiles && expert >= 0 && g.tile_expert[t] == expert;
      whole = whole && live;
      if (!live) continue;
      TC* row = (TC*)g.out + (size_t)(t * TILE_ROWS + r) * g.out_ld + n0;
#pragma unroll
      for (int b = 0; b < WT; ++b) {
        if (n0 + 16 * b >= g.N) continue;  // N is a multiple of 16: four columns lie before or past the end together
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = GATED ? gated_value(acc[a][b][i], acc[a][b + (GATED ? WT : 0)][i], g.act) : acc[a][b][i];
        if constexpr (sizeof(TC) == 4)
          *(float4*)(row + 16 * b) = make_float4(v[0], v[1], v[2], v[3]);
        else
          *(uint2*)(row + 16 * b) = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
      }
    }
    return whole;
  }
};

template <typename TC, bool GATED>
__global__ void __launch_bounds__(512, 2) grouped_loop_kernel(const GroupedWide args, const int* __restrict__ used) {
  constexpr int WM = 4, WN = 4, QM = 2, QN = 2;
  typedef WideShape<WM, WN> Whole;
  typedef WideShape<QM, QN> Quarter;
  constexpr int BYTES = Whole::S * Whole::STAGE > Quarter::S * Quarter::STAGE ? Whole::S * Whole::STAGE : Quarter::S * Quarter::STAGE;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[BYTES];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  GroupedWide g = args;
  g.row_blocks = __builtin_amdgcn_readfirstlane(((used ? min(*used, g.n_tiles) : g.n_tiles) + 7) / 8);
  const int total = g.row_blocks * g.col_blocks, blocks = (int)gridDim.x;
  // whole rounds of whole tiles, and one more where what is left fills more than half of it
  int whole = total / blocks * blocks;
  if (2 * (total - whole) > blocks) whole = total;
  // the XCDs (block number modulo 8) take consecutive runs, their blocks in turn
  const int groups = min(8, blocks), xcd = blockIdx.x % groups, idx = blockIdx.x / groups, peers = (blocks + groups - 1 - xcd) / groups;
  auto share = [&](int n, int& first, int& mine) {
    const int per = n / groups, rest = n % groups;
    first = xcd * per + min(xcd, rest) + idx;
    mine = (per + (xcd < rest ? 1 : 0) - idx + peers - 1) / peers;
  };
  const int steps = g.K / WIDE_BK;
  int first, mine;
  share(whole, first, mine);
  if (mine > 0) {
    GroupedSource<WM, WN, GATED, false> src = {g, lane, wave, nullptr, nullptr, GATED ? g.w1 - g.w0 : 0};
    GroupedSink<WM, WN, TC, GATED, false> sink = {g, lane, wave};
    wide_loop<WM, WN, GroupedSink<WM, WN, TC, GATED, false>::STORES>(lds, src, sink, first, peers, mine, steps);
    asm volatile("s_barrier" ::: "memory");  // everyone has left the buffers
  }
  share(4 * (total - whole), first, mine);
  if (mine > 0) {
    GroupedSource<QM, QN, GATED, true> src = {g, lane, wave, nullptr, nullptr, GATED ? g.w1 - g.w0 : 0};
    GroupedSink<QM, QN, TC, GATED, true> sink = {g, lane, wave};
    wide_loop<QM, QN, GroupedSink<QM, QN, TC, GATED, true>::STORES>(lds, src, sink, 4 * whole + first, peers, mine, steps);
  }
}

template <typename T, int RT, int CT, int WR, bool GATED>
static void launch_grouped(bool vec, int tiles, int n_batch, hipStream_t stream, const T* a, long a_ld, long a_batch, const int* row_token,
                           const T* w0, const T* w1, long w_stride, const int* tile_expert, int n_tiles, void* out, int out_dtype,
                           long out_ld, long out_batch, int n_rows, int N, int K, GateAct act) {
  constexpr int block_tiles = WR * RT, block_cols = (4 / WR) * CT * 16;
  dim3 grid((tiles + block_tiles - 1) / block_tiles, (N + block_cols - 1) / block_cols, n_batch);
  if (vec)
    hipLaunchKernelGGL((grouped_product_kernel<T, RT, CT, WR, GATED, true>), grid, dim3(256), 0, stream, a, a_ld, a_batch, row_token, w0, w1,
                       w_stride, tile_expert, n_tiles, out, out_dtype, out_ld, out_batch, n_rows, N, K, act);
  else
    hipLaunchKernelGGL((grouped_product_kernel<T, RT, CT, WR, GATED, false>), grid, dim3(256), 0, stream, a, a_ld, a_batch, row_token, w0, w1,
                       w_stride, tile_expert, n_tiles, out, out_dtype, out_ld, out_batch, n_rows, N, K, act);
}

// a: rows of K values, `a_ld` apart (row `row_token[row]` for list row `row` if it is given, else row `row`; batch z starts
// `a_batch` further).  w0 (and w1 for the gated form): [experts or batches][N][K], `w_stride` apart.  With
// `tile_expert` the rows are the list's n_tiles * 16 and out is [rows][out_ld]; without, every batch z < n_batch
// multiplies the same n_rows rows by its own weight into out + z * out_batch.  tiles_a_block: 1, 2, 4 or 8 row tiles
// a block; with a list, an expert's tiles start at a multiple of `tile_align`, itself a multiple of tiles_a_block.  used: how many
// of the list's tiles may have rows (`cwm_group_by_expert` leaves the number), or null: any of them.  act_kind, act_alpha, act_limit: the gated
// form's activation (`GateAct`).  tiled: the weights are in operand tiles (bfloat16, [experts][N / 16][K / 32][64][8]).  loop: products of
// eight row tiles a block with such weights go to persistent blocks, where the rows' offsets fit 32 bits.
extern "C" int cwm_grouped_product(const void* a, long a_ld, long a_batch, int dtype, const int* row_token, const void* w0, const void* w1,
                                   long w_stride, const int* tile_expert, const int* used, int n_tiles, int n_batch, void* out, int out_dtype, long out_ld,
                                   long out_batch, int n_rows, int N, int K, int tiles_a_block, int tile_align, int act_kind,
                                   float act_alpha, float act_limit, int tiled, int loop, hipStream_t stream) {
  CWM_REQUIRE(a && w0 && out, "grouped_product: arguments missing");
  CWM_REQUIRE(!tiled || (dtype == CWM_BF16 && N % 16 == 0 && K % 64 == 0 && (long)N * K < (1l << 31)),
              "grouped_product: weights in operand tiles are bfloat16, N a multiple of 16 and K of 64");
  CWM_REQUIRE(act_kind >= 0 && act_kind <= 2, "grouped_product: unknown gated activation %d", act_kind);
  const GateAct act = {act_kind, act_alpha, act_limit};
  CWM_REQUIRE(N > 0 && K > 0 && a_ld >= K && out_ld >= 0, "grouped_product: bad sizes");
  CWM_REQUIRE(tile_expert ? (n_tiles >= 0 && n_batch == 1 && (row_token || n_rows >= n_tiles * TILE_ROWS)) : (n_batch >= 1 && n_batch <= 65535), "grouped_product: give a tile list or a number of batches");
  const int tiles = tile_expert ? n_tiles : (n_rows + TILE_ROWS - 1) / TILE_ROWS;
  if (tiles <= 0) return 0;
  const int esize = dtype == CWM_BF16 ? 2 : 4;
  const int piece = dtype == CWM_BF16 ? 8 : 4;
  const bool vec = K % piece == 0 && (a_ld * esize) % 16 == 0 && (a_batch * esize) % 16 == 0 && (w_stride * esize) % 16 == 0 &&
                   ((uintptr_t)a % 16) == 0 && ((uintptr_t)w0 % 16) == 0 && (!w1 || ((uintptr_t)w1 % 16) == 0);
  CWM_REQUIRE(tiles_a_block == 1 || tiles_a_block == 2 || tiles_a_block == 4 || tiles_a_block == 8, "grouped_product: a block takes 1, 2, 4 or 8 row tiles");
  CWM_REQUIRE(!tile_expert || (tile_align >= 1 && tile_align % tiles_a_block == 0), "grouped_product: the list's tiles start at multiples of %d, a block takes %d",
              tile_align, tiles_a_block);
  CWM_REQUIRE((N + 15) / 16 <= 65535, "grouped_product: too many columns");
  const int nb = tile_expert ? 1 : n_batch;
#define CWM_GROUPED(T, RT, CT, WR, GATED)                                                                                                 \
  launch_grouped<T, RT, CT, WR, GATED>(vec, tiles, nb, stream, (const T*)a, a_ld, a_batch, row_token, (const T*)w0, (const T*)w1, w_stride, \
                                       tile_expert, n_tiles, out, out_dtype, out_ld, out_batch, n_rows, N, K, act)
#define CWM_GROUPED_SHAPES(T)                                                   \
  do {                                                                          \
    if (w1) {                                                                   \
      if (tiles_a_block == 8) CWM_GROUPED(T, 4, 2, 2, true);                    \
      else if (tiles_a_block == 4) CWM_GROUPED(T, 4, 1, 1, true);               \
      else CWM_GROUPED(T, 1, 1, 1, true);                                       \
    } else {                                                                    \
      if (tiles_a_block == 8) CWM_GROUPED(T, 4, 4, 2, false);                   \
      else if (tiles_a_block == 4) CWM_GROUPED(T, 4, 1, 1, false);              \
      else CWM_GROUPED(T, 1, 1, 1, false);                                      \
    }                                                                           \
  } while (0)
  if (tiles_a_block > 1 && vec && dtype == CWM_BF16 && K % 64 == 0 && (long)N * K < (1l << 31) && (long)n_rows * (a_ld / 8) < (1l << 32)) {
    // the shape whose rows go through LDS
    const int osize = out_dtype == CWM_F32 ? 4 : 2;
    const int vec_out = (out_ld * osize) % (4 * osize) == 0 && (out_batch * osize) % (4 * osize) == 0 && ((uintptr_t)out % (4 * osize)) == 0;
    if (loop && tiled && tiles_a_block == 8 && tile_expert && tile_align == 8 && vec_out && (unsigned long long)n_rows * a_ld * 2 < (1ull << 32) &&
        out_dtype == (w1 ? CWM_BF16 : CWM_F32)) {
      GroupedWide g = {(const bf16_t*)a, a_ld, (list_ints)row_token, (const bf16_t*)w0, (const bf16_t*)w1, w_stride, (list_ints)tile_expert, n_tiles, N, K,
                       0, (N + (w1 ? 127 : 255)) / (w1 ? 128 : 256), out, out_ld, act};
      if (w1)
        hipLaunchKernelGGL((grouped_loop_kernel<bf16_t, true>), dim3(GROUPED_BLOCKS), dim3(512), 0, stream, g, used);
      else
        hipLaunchKernelGGL((grouped_loop_kernel<float, false>), dim3(GROUPED_BLOCKS), dim3(512), 0, stream, g, used);
      return cwm_launch_status("grouped_product");
    }
    const int row_blocks = (tiles + tiles_a_block - 1) / tiles_a_block;
#define CWM_WIDE_AS(RT, CT, GATED, TILED)                                                                                                            \
  do {                                                                                                                                     \
    const int cols = (GATED ? 32 : 64) * CT, col_blocks = (N + cols - 1) / cols;                                                           \
    dim3 grid((row_blocks * col_blocks + 7) / 8 * 8, 1, nb);                                                                               \
    if (!tile_expert) grid.x = row_blocks * col_blocks;                                                                                    \
    hipLaunchKernelGGL((grouped_wide_kernel<RT, CT, GATED, TILED>), grid, dim3(256), 0, stream, (const bf16_t*)a, a_ld, a_batch, row_token,        \
                       (const bf16_t*)w0, (const bf16_t*)w1, w_stride, tile_expert, used, n_tiles, row_blocks, col_blocks, out, out_dtype,       \
                       out_ld, out_batch, vec_out, n_rows, N, K, act);                                                                     \
  } while (0)
    // Four weight tiles a wavefront where that still makes about two blocks a compute unit, else two, which makes twice as
    // many blocks (measured with 16 experts of 2,048 x 1,024, gate and up: 200 rows an expert 96 and 81 us, 1,024 rows 214 and
    // 220 us; 32 of 3,072 x 1,536: 256 rows 320 and 363 us).  Blocks of two row tiles stream the weights: always two.
    const int blocks4 = row_blocks * ((N + (w1 ? 127 : 255)) / (w1 ? 128 : 256));
    const bool many = tiles_a_block == 8 ? blocks4 >= 500 : tiles_a_block == 4 && blocks4 >= 560;
#define CWM_WIDE(RT, CT, GATED)            \
  do {                                     \
    if (tiled)                             \
      CWM_WIDE_AS(RT, CT, GATED, true);    \
    else                                   \
      CWM_WIDE_AS(RT, CT, GATED, false);   \
  } while (0)
#define CWM_WIDE_COLS(RT, GATED)   \
  do {                             \
    if (many)                      \
      CWM_WIDE(RT, 4, GATED);      \
    else                           \
      CWM_WIDE(RT, 2, GATED);      \
  } while (0)
    if (w1) {
      if (tiles_a_block == 8) CWM_WIDE_COLS(8, true);
      else if (tiles_a_block == 4) CWM_WIDE_COLS(4, true);
      else CWM_WIDE(2, 2, true);
    } else {
      if (tiles_a_block == 8) CWM_WIDE_COLS(8, false);
      else if (tiles_a_block == 4) CWM_WIDE_COLS(4, false);
      else CWM_WIDE(2, 2, false);
    }
#undef CWM_WIDE_COLS
#undef CWM_WIDE
#undef CWM_WIDE_AS
    return cwm_launch_status("grouped_product");
  }
  if (tiles_a_block <= 2 && vec && (dtype == CWM_BF16 || dtype == CWM_F32)) {
    // the weight-streaming shape
    dim3 grid(tiles, (N + 15) / 16, nb);
#define CWM_STREAMED(T, GATED, TILED)                                                                                                             \
  hipLaunchKernelGGL((grouped_stream_kernel<T, GATED, TILED>), grid, dim3(256), 0, stream, (const T*)a, a_ld, a_batch, row_token, (const T*)w0,     \
                     (const T*)w1, w_stride, tile_expert, n_tiles, out, out_dtype, out_ld, out_batch, n_rows, N, K, act, tile_align)
    if (dtype == CWM_BF16) {
      if (tiled) {
        if (w1) CWM_STREAMED(bf16_t, true, true); else CWM_STREAMED(bf16_t, false, true);
      } else {
        if (w1) CWM_STREAMED(bf16_t, true, false); else CWM_STREAMED(bf16_t, false, false);
      }
    } else {
      if (w1) CWM_STREAMED(float, true, false); else CWM_STREAMED(float, false, false);
    }
#undef CWM_STREAMED
    return cwm_launch_status("grouped_product");
  }
  CWM_REQUIRE(!tiled, "grouped_product: weights in operand tiles need rows at multiples of 16 bytes");
  if (dtype == CWM_BF16)
    CWM_GROUPED_SHAPES(bf16_t);
  else if (dtype == CWM_F32)
    CWM_GROUPED_SHAPES(float);
  else
    return cwm_fail("grouped_product: unknown dtype %d", dtype);
#undef CWM_GROUPED_SHAPES
#undef CWM_GROUPED
  return cwm_launch_status("grouped_product");
}

__global__ void __launch_bounds__(256) combine_routed_kernel(const float* __restrict__ rows, long rows_ld, const int* __restrict__ pair_row,
                                                             const float* __restrict__ weights, float* __restrict__ out, int top, int dim) {
  const size_t t = blockIdx.x;
  for (int i = blockIdx.y * blockDim.x + threadIdx.x; i < dim; i += gridDim.y * blockDim.x) {
    float acc = 0.f;
    for (int k = 0; k < top; ++k) {
      const int row = pair_row[t * top + k];
      if (row >= 0) acc += weights[t * top + k] * rows[(size_t)row * rows_ld + i];
    }
    out[t * dim + i] = acc;
  }
}

// The same sums, four adjacent elements a lane, four rows under way at a time (a choice without a row reads row 0 and
// is left out): 2,296 tokens of 4 choices of 2,048 take 14.9 us where one element a load took 21.7, 300 tokens 2.4 of
// 4.7 and one 1.9 of 3.9.  dim: a multiple of 4; rows at multiples of 16 bytes.
__global__ void __launch_bounds__(256) combine_four_kernel(const float* __restrict__ rows, long rows_ld, const int* __restrict__ pair_row,
                                                           const float* __restrict__ weights, float* __restrict__ out, int top, int dim) {
  const size_t t = blockIdx.x;
  for (int i = 4 * (blockIdx.y * blockDim.x + threadIdx.x); i < dim; i += 4 * gridDim.y * blockDim.x) {
    float4v acc = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < top; k0 += 4) {
      float4v x[4];
      int row[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        row[u] = k0 + u < top ? pair_row[t * top + k0 + u] : -1;
        x[u] = *(const float4v*)(rows + (size_t)(row[u] < 0 ? 0 : row[u]) * rows_ld + i);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (row[u] >= 0) acc += weights[t * top + k0 + u] * x[u];
    }
    *(float4v*)(out + t * dim + i) = acc;
  }
}

extern "C" int cwm_combine_routed(const float* rows, long rows_ld, const int* pair_row, const float* weights, float* out, int n_tokens,
                                  int top, int dim, hipStream_t stream) {
  CWM_REQUIRE(rows && pair_row && weights && out && top >= 1 && dim > 0, "combine_routed: bad arguments");
  if (n_tokens <= 0) return 0;
  if (dim % 4 == 0 && rows_ld % 4 == 0 && (((uintptr_t)rows | (uintptr_t)out) % 16) == 0) {
    hipLaunchKernelGGL(combine_four_kernel, dim3(n_tokens, (dim + 1023) / 1024), dim3(256), 0, stream, rows, rows_ld, pair_row, weights, out, top, dim);
    return cwm_launch_status("combine_routed");
  }
  hipLaunchKernelGGL(combine_routed_kernel, dim3(n_tokens, (dim + 1023) / 1024), dim3(256), 0, stream, rows, rows_ld, pair_row, weights, out, top, dim);
  return cwm_launch_status("combine_routed");
}

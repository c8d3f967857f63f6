// Next-token choice from float32 logits, one block per row: greedy argmax, or a
// draw from softmax(logits / T) restricted to the nucleus of mass top_p.
//
// Reference semantics: argmax when sampling is off (cwm/fastgen/generate.py:1012);
// probs = softmax(logits / T) in float32 (:1003); nucleus = the entries whose
// preceding mass in descending order does not exceed top_p, renormalised
// (cwm/fastgen/utils/sampling.py:38-45).  The draw itself uses a uniform number
// u in [0, 1) that the caller supplies per row: the first kept entry, in vocabulary
// order, at which the running kept mass exceeds u * (kept mass).  That is a draw
// from the same distribution as torch.multinomial, made reproducible per request.
//
// Also returned per row: logprob = log softmax(logits)[token] (the reference's
// -cross_entropy, generate.py:1010) and sample_logprob = log of the probability
// under the temperature / nucleus distribution (0 for greedy rows).
//
// The nucleus is found without sorting: with e_i = exp((x_i - max) / T) and
// f(t) = sum of e_i > t, the kept set is {e_i >= t*} for the smallest float t*
// with f(t*) <= top_p * sum(e); t* is found by cutting the interval of bit patterns.
// Entries exactly equal to the threshold are all kept.  Without a nucleus (top_p = 1)
// nothing is stored: the draw recomputes e_i where it walks.  A row of 128k logits done so
// takes about 22 us greedy, 44 us at a temperature and 170 us with a nucleus; rows of more than
// 8,192 entries are cut into segments instead (below): 6, 11 and, by the logits' spread, 21 to 62 us replayed
// from a graph (launched one by one 15, 16 and 21 to 62); 743 such rows 97, 129 and 205 to 396 us.
#include "common.h"
#include "no_alloc.h"

#include <mutex>
#include <type_traits>

CWM_DEFINE_ERROR_API

#define SAMPLE_THREADS 1024

struct MaxIdx {
  float v;
  int i;
};

__device__ __forceinline__ MaxIdx better(MaxIdx a, MaxIdx b) {
  if (b.v > a.v || (b.v == a.v && b.i < a.i)) return b;
  return a;
}

// f(i, x[i]) for every i < n, thread t taking i = t, t + THREADS, ... in increasing order; VEC (n a multiple of 4
// and x 16-byte aligned): four adjacent entries at a time, so a pass over a row of 128k logits is 32 loads a thread
template <bool VEC, typename F>
__device__ __forceinline__ void each_strided(const float* x, int n, int tid, F&& f) {
  if (VEC) {
    const float4* x4 = (const float4*)x;
#pragma unroll 2
    for (int i = tid; i < (n >> 2); i += SAMPLE_THREADS) {
      const float4 v = x4[i];
      f(4 * i, v.x);
      f(4 * i + 1, v.y);
      f(4 * i + 2, v.z);
      f(4 * i + 3, v.w);
    }
  } else {
#pragma unroll 4
    for (int i = tid; i < n; i += SAMPLE_THREADS) f(i, x[i]);
  }
}

#ifndef SEARCH_WAYS
#define SEARCH_WAYS 2  // thresholds tried in one pass over the row (measured at 128k entries: 2 169 us, 3 187, 4 196, 8 242)
#endif

struct WholeRowShared {
  float scratch[16];
  float mv[SAMPLE_THREADS / CWM_WAVE];
  int mi[SAMPLE_THREADS / CWM_WAVE];
  float seg_sum[2 * SAMPLE_THREADS / CWM_WAVE];  // masses of the 16 regions, then of the chosen region's 16 parts
  float above_part[SAMPLE_THREADS / CWM_WAVE][SEARCH_WAYS];
};

// One block does a whole row by itself.
template <bool VEC>
__device__ __forceinline__ void sample_whole_row(WholeRowShared& sh, const int row, const float* __restrict__ logits, long row_stride, int vocab,
                                 const float* __restrict__ temperature, const float* __restrict__ top_p, const float* __restrict__ uniform,
                                 float* __restrict__ workspace, int* __restrict__ token_out, float* __restrict__ logprob_out,
                                 float* __restrict__ sample_logprob_out) {
  float* scratch = sh.scratch;
  float* mv = sh.mv;
  int* mi = sh.mi;
  float* seg_sum = sh.seg_sum;
  auto& above_part = sh.above_part;
  const int tid = threadIdx.x;
  const float* x = logits + (size_t)row * row_stride;
  float* e = workspace + (size_t)row * vocab;

  // 1. maximum and its first index
  MaxIdx best = {-__builtin_inff(), 0x7fffffff};
  each_strided<VEC>(x, vocab, tid, [&](int i, float v) {
    if (v > best.v) {  // a thread visits its indices in increasing order
      best.v = v;
      best.i = i;
    }
  });
#pragma unroll
  for (int off = CWM_WAVE / 2; off > 0; off >>= 1) {
    MaxIdx o;
    o.v = __shfl_xor(best.v, off, CWM_WAVE);
    o.i = __shfl_xor(best.i, off, CWM_WAVE);
    best = better(best, o);
  }
  if ((tid & (CWM_WAVE - 1)) == 0) {
    mv[tid / CWM_WAVE] = best.v;
    mi[tid / CWM_WAVE] = best.i;
  }
  __syncthreads();
  best.v = mv[0];
  best.i = mi[0];
  for (int w = 1; w < SAMPLE_THREADS / CWM_WAVE; ++w) {
    MaxIdx o = {mv[w], mi[w]};
    best = better(best, o);
  }
  if (best.i >= vocab) best.i = 0;  // every logit NaN or -inf: still return a valid id
  const float xmax = best.v;

  // 2. log-sum-exp at temperature 1
  float s1 = 0.f;
  each_strided<VEC>(x, vocab, tid, [&](int, float v) { s1 += expf(v - xmax); });
  s1 = block_sum(s1, scratch);
  const float lse = xmax + logf(s1);

  const float temp = temperature[row];
  if (!(temp > 0.f)) {  // greedy
    if (tid == 0) {
      token_out[row] = best.i;
      logprob_out[row] = xmax - lse;
      sample_logprob_out[row] = 0.f;
    }
    return;
  }

  // 3. the nucleus threshold (top_p < 1 only): unnormalised probabilities at temperature T go to the
  //    workspace, and the search reads them from there.  f(t) = sum of e_i > t, summed in a fixed order, does
  //    not grow with t, so the smallest t with f(t) <= top_p * sum(e) is found by cutting the interval of bit
  //    patterns: SEARCH_WAYS thresholds a pass, each with a sum of its own.
  const float inv_t = 1.0f / temp;
  const float tp = top_p[row];
  const bool nucleus = tp < 1.0f;
  float thresh = 0.f;
  if (nucleus) {
    float z = 0.f;
    if (VEC) {
      float4* e4 = (float4*)e;
      const float4* x4 = (const float4*)x;
#pragma unroll 2
      for (int i = tid; i < (vocab >> 2); i += SAMPLE_THREADS) {
        const float4 v = x4[i];
        float4 ev;
        ev.x = expf((v.x - xmax) * inv_t);
        ev.y = expf((v.y - xmax) * inv_t);
        ev.z = expf((v.z - xmax) * inv_t);
        ev.w = expf((v.w - xmax) * inv_t);
        e4[i] = ev;
        z += ev.x;
        z += ev.y;
        z += ev.z;
        z += ev.w;
      }
    } else {
#pragma unroll 4
      for (int i = tid; i < vocab; i += SAMPLE_THREADS) {
        const float ev = expf((x[i] - xmax) * inv_t);
        e[i] = ev;
        z += ev;
      }
    }
    z = block_sum(z, scratch);  // (its first barrier also orders the writes of e before the reads below)
    const float target = tp * z;
    uint32_t lo = 0u, hi = __float_as_uint(1.0f);  // f(1) = 0: the answer lies in [lo, hi]
    while (lo < hi) {
      // thresholds lo <= m_0 < m_1 < ... < hi, evenly spread (the same one several times once the interval is short)
      uint32_t m[SEARCH_WAYS];
      float above[SEARCH_WAYS];
      const uint32_t span = hi - lo;
#pragma unroll
      for (int j = 0; j < SEARCH_WAYS; ++j) {
        m[j] = lo + (uint32_t)(((unsigned long long)span * (j + 1)) / (SEARCH_WAYS + 1));
        if (m[j] >= hi) m[j] = hi - 1;
        above[j] = 0.f;
      }
      each_strided<VEC>(e, vocab, tid, [&](int, float ev) {
#pragma unroll
        for (int j = 0; j < SEARCH_WAYS; ++j) above[j] += ev > __uint_as_float(m[j]) ? ev : 0.f;
      });
#pragma unroll
      for (int j = 0; j < SEARCH_WAYS; ++j) above[j] = wave_sum(above[j]);
      __syncthreads();
      if ((tid & (CWM_WAVE - 1)) == 0) {
#pragma unroll
        for (int j = 0; j < SEARCH_WAYS; ++j) above_part[tid / CWM_WAVE][j] = above[j];
      }
      __syncthreads();
      // the first threshold whose sum is small enough becomes the upper end, the one before it (plus one) the lower
      int first = SEARCH_WAYS;
#pragma unroll
      for (int j = SEARCH_WAYS - 1; j >= 0; --j) {
        float total = 0.f;
        for (int w = 0; w < SAMPLE_THREADS / CWM_WAVE; ++w) total += above_part[w][j];
        if (total <= target) first = j;
      }
      if (first > 0) lo = m[first - 1] + 1;
      if (first < SEARCH_WAYS) hi = m[first];
    }
    thresh = __uint_as_float(hi);
  }
  // the kept mass of entry i (0 for an entry outside the nucleus); without a nucleus it is computed anew
  // wherever it is needed, which is cheaper than a trip through memory
  auto kept = [&](int i) -> float {
    const float ev = nucleus ? e[i] : expf((x[i] - xmax) * inv_t);
    return ev >= thresh ? ev : 0.f;
  };

  // 4. inverse CDF over the kept entries in vocabulary order, in three levels: the vocabulary is cut into 16
  //    regions of whole groups of 64 entries, one per wavefront, whose masses say in which region the drawn
  //    point lies; that region into 16 parts likewise; the part is then walked group by group by one wavefront.
  //    Every load is of 64 adjacent entries.  The sums of the three levels are rounded differently, so a level
  //    may find the point beyond its last mass: it then takes its last entry with mass.
  const int lane = tid & (CWM_WAVE - 1);
  const int wave = tid / CWM_WAVE;
  constexpr int WAVES = SAMPLE_THREADS / CWM_WAVE;
  const int n_groups = (vocab + CWM_WAVE - 1) / CWM_WAVE;
  // mass of the entries [begin, end) that this wavefront's lanes read side by side
  auto wave_mass = [&](int begin, int end) -> float {
    float m = 0.f;
    if (VEC) {  // begin is a multiple of 64 and end of 4
      const float4* src = (const float4*)((nucleus ? e : x) + begin);
#pragma unroll 2
      for (int i = lane; i < ((end - begin) >> 2); i += CWM_WAVE) {
        const float4 v = src[i];
        const float e0 = nucleus ? v.x : expf((v.x - xmax) * inv_t), e1 = nucleus ? v.y : expf((v.y - xmax) * inv_t);
        const float e2 = nucleus ? v.z : expf((v.z - xmax) * inv_t), e3 = nucleus ? v.w : expf((v.w - xmax) * inv_t);
        m += e0 >= thresh ? e0 : 0.f;
        m += e1 >= thresh ? e1 : 0.f;
        m += e2 >= thresh ? e2 : 0.f;
        m += e3 >= thresh ? e3 : 0.f;
      }
    } else {
#pragma unroll 4
      for (int i = begin + lane; i < end; i += CWM_WAVE) m += kept(i);
    }
    return wave_sum(m);
  };
  // the first of the WAVES masses in `part` at which the running sum from `before` passes `target` (the last
  // one with mass if none does); the running sum before it is returned through `before`
  auto pick_part = [&](const float* part, float target, float& before) -> int {
    float run = before;
    int pick = -1, last = 0;
    float pick_before = before, last_before = before;
    for (int w = 0; w < WAVES; ++w) {
      const float m = part[w];
      if (m > 0.f) {
        last = w;
        last_before = run;
        if (pick < 0 && run + m > target) {
          pick = w;
          pick_before = run;
        }
      }
      run += m;
    }
    before = pick < 0 ? last_before : pick_before;
    return pick < 0 ? last : pick;
  };

  const int region_groups = (n_groups + WAVES - 1) / WAVES;
  {
    const int begin = min(vocab, wave * region_groups * CWM_WAVE);
    const float m = wave_mass(begin, min(vocab, begin + region_groups * CWM_WAVE));
    if (lane == 0) seg_sum[wave] = m;
  }
  __syncthreads();
  float total = 0.f;
  for (int w = 0; w < WAVES; ++w) total += seg_sum[w];
  const float target = uniform[row] * total;
  float before = 0.f;
  const int region = pick_part(seg_sum, target, before);  // the same in every thread

  const int part_groups = (region_groups + WAVES - 1) / WAVES;
  const int region_begin = min(vocab, region * region_groups * CWM_WAVE);
  const int region_end = min(vocab, region_begin + region_groups * CWM_WAVE);
  {
    const int begin = min(region_end, region_begin + wave * part_groups * CWM_WAVE);
    const float m = wave_mass(begin, min(region_end, begin + part_groups * CWM_WAVE));
    if (lane == 0) seg_sum[WAVES + wave] = m;
  }
  __syncthreads();
  const int part = pick_part(seg_sum + WAVES, target, before);

  if (wave == 0) {
    const int begin = min(region_end, region_begin + part * part_groups * CWM_WAVE);
    const int end = min(region_end, begin + part_groups * CWM_WAVE);
    float run = before;
    int tok = -1;  // the entry at which the running sum passes the target
    int last_tok = -1;  // the last entry with mass so far, in case rounding puts the target beyond the part's mass
    for (int g = begin; g < end && tok < 0; g += CWM_WAVE) {
      const int i = g + lane;
      const float v = i < end ? kept(i) : 0.f;
      float scan = v;  // inclusive sum over the lanes up to this one
#pragma unroll
      for (int off = 1; off < CWM_WAVE; off <<= 1) {
        const float o = __shfl_up(scan, off, CWM_WAVE);
        if (lane >= off) scan += o;
      }
      const unsigned long long has_mass = __ballot(v > 0.f);
      const unsigned long long passes = __ballot(v > 0.f && run + scan > target);
      if (passes) tok = g + __ffsll((long long)passes) - 1;
      if (has_mass) last_tok = g + 63 - __clzll((long long)has_mass);
      run += __shfl(scan, CWM_WAVE - 1, CWM_WAVE);
    }
    if (tok < 0) tok = last_tok;
    if (lane == 0) {
      if (tok < 0) tok = best.i;  // no entry with mass at all (every logit NaN)
      token_out[row] = tok;
      logprob_out[row] = x[tok] - lse;
      sample_logprob_out[row] = logf(kept(tok) / total);
    }
  }
}

template <bool VEC>
__global__ void __launch_bounds__(SAMPLE_THREADS)
sample_kernel(const float* __restrict__ logits, long row_stride, int vocab, const float* __restrict__ temperature,
              const float* __restrict__ top_p, const float* __restrict__ uniform, float* __restrict__ workspace,
              int* __restrict__ token_out, float* __restrict__ logprob_out, float* __restrict__ sample_logprob_out) {
  __shared__ WholeRowShared sh;
  sample_whole_row<VEC>(sh, blockIdx.x, logits, row_stride, vocab, temperature, top_p, uniform, workspace, token_out, logprob_out,
                        sample_logprob_out);
}

// ---- rows cut into segments ----------------------------------------------------------- //
// One compute unit reads a row of 128k logits at a hundredth of the memory's rate and needs 8 us for as many exponentials,
// so a row is cut into segments of at most 2,048 entries, a block each, read once; a second kernel of one block a row puts
// the segments' records together.  The nucleus is found through a histogram of mass instead of passes over the row: a bin
// is floor(x * 8 / (T ln 2)), an eighth of an octave of e^(x/T), the same bin in every segment whatever its maximum, and the
// bin in which the mass from the top passes top_p * z is the only one whose entries have to be looked at.  Masses that
// several threads add to one place are integers, so their order does not matter and a row's result is the same every time: units
// of 2^-52 of a segment's largest entry (the 2,048 entries of a segment fit 64 bits), of 2^-44 of the row's where all of its entries may
// meet.  Entries of up to 29 octaves below the segment's largest are exact in them; what the smaller ones are rounded by is below
// 2^-25 of the kept mass together (at most 2^19 entries, half a unit each), less than the rounding of a float32 sum.
#define SEG_THREADS 256
#define SEG_PER_THREAD 8
#define SEG_ENTRIES (SEG_THREADS * SEG_PER_THREAD)
#define SEG_MOST 256     // segments of a row
#define SEG_BINS 256     // the last one holds everything 32 octaves and more below the segment's maximum
#define SEGMENTS_FROM 8192  // longer rows are cut: the second launch costs 4 us, and a nucleus in a row of 8,192 takes 37 us as a whole, 20 to 28 in segments
#define SEG_LIST 4096    // entries of the decisive bin that are kept in LDS
#define SEG_SORT 1024    // and those of its decisive part that are put in order
#define SEG_RANK 256     // so few of them by counting: 2 entries 0.6 instead of 2.2 us by exchanges, 224 3.9 instead of 4.3 (the comparisons grow with the square)
#define SEG_FIXED 4503599627370496.0f  // 2^52
#define ROW_FIXED 17592186044416.0f    // 2^44

struct SegRecord {
  float max;
  int argmax;
  float sum;   // of exp(x - max)
  float mass;  // of exp((x - max) / T)
};

// Where the records and histograms of a row lie in its part of the workspace (vocab floats).
__host__ __device__ __forceinline__ int seg_length(int vocab) {
  const int n = (vocab + SEG_ENTRIES - 1) / SEG_ENTRIES;
  return (((vocab + n - 1) / n) + 63) / 64 * 64;
}
__device__ __forceinline__ SegRecord* seg_records(float* row_workspace) {
  return (SegRecord*)(((uintptr_t)row_workspace + 15) & ~(uintptr_t)15);
}
__device__ __forceinline__ float* seg_histogram(float* row_workspace, int n_segs, int seg) {
  return (float*)(seg_records(row_workspace) + n_segs) + (size_t)seg * SEG_BINS;
}

// the bin of x counted downwards from the one of `top` (both times 8 / (T ln 2))
__device__ __forceinline__ int bins_below(float top_floor, float scaled) { return (int)fminf(top_floor - floorf(scaled), (float)(SEG_BINS - 1)); }

// The part of its bin in which `scaled` (x * 8 / (T ln 2), rounded) lies, counted downwards.  The fraction comes from the same rounded
// number as the bin: contracted with the multiplication before it, it may be negative and the part lie outside the bin.
__device__ __forceinline__ int part_of_bin(float scaled) {
#pragma clang fp contract(off)
  const float fraction = scaled - floorf(scaled);
  return SEG_BINS - 1 - max(0, min(SEG_BINS - 1, (int)(fraction * SEG_BINS)));
}

template <bool VEC>
__global__ void __launch_bounds__(SEG_THREADS)
sample_segment_kernel(const float* __restrict__ logits, long row_stride, int vocab, int seg_len, const float* __restrict__ temperature,
                      const float* __restrict__ top_p, float* __restrict__ workspace) {
  __shared__ float wv[SEG_THREADS / CWM_WAVE];
  __shared__ int wi[SEG_THREADS / CWM_WAVE];
  __shared__ float ws[SEG_THREADS / CWM_WAVE], wz[SEG_THREADS / CWM_WAVE], wt[SEG_THREADS / CWM_WAVE];
  __shared__ unsigned long long bins[SEG_BINS];
  const int seg = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, lane = tid & (CWM_WAVE - 1), wave = tid / CWM_WAVE;
  const int begin = seg * seg_len, end = min(vocab, begin + seg_len);
  const float* x = logits + (size_t)row * row_stride;
  bins[tid] = 0;
  float v[SEG_PER_THREAD];
  int at[SEG_PER_THREAD / 4];  // first entry of every four
#pragma unroll
  for (int q = 0; q < SEG_PER_THREAD / 4; ++q) {
    at[q] = begin + 4 * (q * SEG_THREADS + tid);
    if (VEC) {  // begin, end: multiples of 4
      const float4 f = at[q] < end ? *(const float4*)(x + at[q]) : make_float4(-__builtin_inff(), -__builtin_inff(), -__builtin_inff(), -__builtin_inff());
      v[4 * q] = f.x, v[4 * q + 1] = f.y, v[4 * q + 2] = f.z, v[4 * q + 3] = f.w;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[4 * q + j] = at[q] + j < end ? x[at[q] + j] : -__builtin_inff();
    }
  }
  MaxIdx best = {-__builtin_inff(), 0x7fffffff};
#pragma unroll
  for (int j = 0; j < SEG_PER_THREAD; ++j)
    if (v[j] > best.v) best.v = v[j], best.i = at[j / 4] + j % 4;
#pragma unroll
  for (int off = CWM_WAVE / 2; off > 0; off >>= 1) best = better(best, MaxIdx{__shfl_xor(best.v, off, CWM_WAVE), __shfl_xor(best.i, off, CWM_WAVE)});
  if (lane == 0) wv[wave] = best.v, wi[wave] = best.i;
  __syncthreads();
  best = MaxIdx{wv[0], wi[0]};
#pragma unroll
  for (int w = 1; w < SEG_THREADS / CWM_WAVE; ++w) best = better(best, MaxIdx{wv[w], wi[w]});

  const float temp = temperature[row];
  const bool draw = temp > 0.f, nucleus = draw && top_p[row] < 1.0f;
  const float inv_t = draw ? 1.0f / temp : 0.f, inv_w = inv_t * 11.541560327f;  // 8 / ln 2
  const float top_floor = floorf(best.v * inv_w);
  float s = 0.f, z = 0.f, tail = 0.f;
#pragma unroll
  for (int j = 0; j < SEG_PER_THREAD; ++j) {
    const float d = v[j] == -__builtin_inff() ? v[j] : v[j] - best.v;  // (a segment may hold nothing else; a NaN stays one)
    s += expf(d);
    if (draw) {
      const float e = expf(d * inv_t);
      z += e;
      if (nucleus) {
        const int k = bins_below(top_floor, v[j] * inv_w);
        if (k < SEG_BINS - 1 && e > 0.f) atomicAdd(&bins[k], __float2ull_rn(e * SEG_FIXED));
        else tail += e;
      }
    }
  }
  s = wave_sum(s), z = wave_sum(z), tail = wave_sum(tail);
  if (lane == 0) ws[wave] = s, wz[wave] = z, wt[wave] = tail;
  __syncthreads();
  float* row_workspace = workspace + (size_t)row * vocab;
  if (nucleus) {
    float* out = seg_histogram(row_workspace, gridDim.x, seg);
    out[tid] = tid < SEG_BINS - 1 ? (float)bins[tid] * (1.0f / SEG_FIXED) : wt[0] + wt[1] + wt[2] + wt[3];
  }
  if (tid == 0) seg_records(row_workspace)[seg] = SegRecord{best.v, best.i, ws[0] + ws[1] + ws[2] + ws[3], wz[0] + wz[1] + wz[2] + wz[3]};
}

// Inclusive sums over the block's threads in a fixed order, of values that are not negative; `scratch` holds 32 floats.
// With `total` the sum over the block as join_sum forms it.
__device__ __forceinline__ float block_scan(float v, float* scratch, float* total = nullptr) {
  const int lane = threadIdx.x & (CWM_WAVE - 1), wave = threadIdx.x / CWM_WAVE;
  const float wave_total = total ? wave_sum(v) : 0.f;
#pragma unroll
  for (int off = 1; off < CWM_WAVE; off <<= 1) {
    const float o = __shfl_up(v, off, CWM_WAVE);
    if (lane >= off) v += o;
  }
  __syncthreads();
  if (lane == CWM_WAVE - 1) {
    scratch[wave] = v;
    if (total) scratch[SAMPLE_THREADS / CWM_WAVE + wave] = wave_total;
  }
  __syncthreads();
  if (total) {
    *total = 0.f;
#pragma unroll
    for (int w = 0; w < SAMPLE_THREADS / CWM_WAVE; ++w) *total += scratch[SAMPLE_THREADS / CWM_WAVE + w];
  }
  float before = 0.f;
#pragma unroll
  for (int w = 0; w < SAMPLE_THREADS / CWM_WAVE - 1; ++w) before += w < wave ? scratch[w] : 0.f;  // read together
  return before + v;
}

// block_sum of SAMPLE_THREADS threads: its bits, with the wavefronts' sums read together.
__device__ __forceinline__ float join_sum(float v, float* scratch) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & (CWM_WAVE - 1)) == 0) scratch[threadIdx.x / CWM_WAVE] = v;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < SAMPLE_THREADS / CWM_WAVE; ++w) total += scratch[w];
  return total;
}

struct JoinShared {
  float scratch[32];
  int first, last, count, smallest;
  int argmax[SEG_MOST];
  float max[SEG_MOST], scale[SEG_MOST], mass[SEG_MOST];
  int below[SEG_MOST];  // bins from the row's top bin down to the segment's
  unsigned long long kept[SEG_MOST];
  union {
    float part[4][SEG_BINS];
    float sorted[SEG_SORT];
  };
  unsigned long long sub[SEG_BINS];
  float list_x[SEG_LIST];
  int list_i[SEG_LIST];
  float before;
};

// The index of the first thread, in order, whose inclusive sum `cum` passes `target` while it has mass; the last one with
// mass if none does.  `before` receives the sum before it.  All threads call it and get the same answer.
__device__ __forceinline__ int first_past(JoinShared& sh, float mass, float cum, float target, float& before) {
  if (threadIdx.x == 0) sh.first = 0x7fffffff, sh.last = -1;
  __syncthreads();
  const int lane = threadIdx.x & (CWM_WAVE - 1), wave_first = threadIdx.x - lane;
  const unsigned long long with = __ballot(mass > 0.f), past = __ballot(mass > 0.f && cum > target);
  if (lane == 0) {
    if (past) atomicMin(&sh.first, wave_first + __ffsll(past) - 1);
    if (with) atomicMax(&sh.last, wave_first + CWM_WAVE - 1 - __clzll((long long)with));
  }
  __syncthreads();
  const int pick = sh.first != 0x7fffffff ? sh.first : sh.last;
  if ((int)threadIdx.x == pick) sh.before = cum - mass;
  __syncthreads();
  before = pick >= 0 ? sh.before : 0.f;
  return pick;
}

// False where the row has to be done by `sample_whole_row`; the block's threads agree.
template <bool VEC>
__device__ __forceinline__ bool join_segments(JoinShared& sh, const int row, const float* __restrict__ logits, long row_stride, int vocab, int seg_len, int n_segs, const float* __restrict__ temperature,
                   const float* __restrict__ top_p, const float* __restrict__ uniform, float* __restrict__ workspace,
                   int* __restrict__ token_out, float* __restrict__ logprob_out, float* __restrict__ sample_logprob_out) {
  const int tid = threadIdx.x, lane = tid & (CWM_WAVE - 1), wave = tid / CWM_WAVE;
  const float* x = logits + (size_t)row * row_stride;
  float* row_workspace = workspace + (size_t)row * vocab;
  const float temp = temperature[row], row_top_p = top_p[row], u = uniform[row];

  // 1. the row's maximum, its first index and the log of the sum at temperature 1
  SegRecord rec = {-__builtin_inff(), 0x7fffffff, 0.f, 0.f};
  if (tid < n_segs) rec = seg_records(row_workspace)[tid];
  MaxIdx best = {rec.max, rec.argmax};
#pragma unroll
  for (int off = CWM_WAVE / 2; off > 0; off >>= 1) best = better(best, MaxIdx{__shfl_xor(best.v, off, CWM_WAVE), __shfl_xor(best.i, off, CWM_WAVE)});
  if (lane == 0 && wave < SEG_MOST / CWM_WAVE) sh.max[wave] = best.v, sh.argmax[wave] = best.i;
  __syncthreads();
  best = MaxIdx{sh.max[0], sh.argmax[0]};
#pragma unroll
  for (int w = 1; w < SEG_MOST / CWM_WAVE; ++w) best = better(best, MaxIdx{sh.max[w], sh.argmax[w]});
  const float xmax = best.v;
  const float sum = join_sum(tid < n_segs ? (rec.max == -__builtin_inff() ? rec.sum : rec.sum * expf(rec.max - xmax)) : 0.f, sh.scratch);
  const float lse = xmax + logf(sum);
  // NaN among the logits, infinities, temperatures at which a bin's number would not be exact: one block, pass by pass
  const float inv_t = 1.0f / temp, inv_w = inv_t * 11.541560327f;
  if (!(sum > 0.f) || !(fabsf(xmax) < __builtin_inff()) || (temp > 0.f && !(fabsf(xmax) * inv_w < 1e6f && inv_w < 1e6f))) {
    return false;
  }
  if (!(temp > 0.f)) {  // greedy
    if (tid == 0) {
      token_out[row] = best.i;
      logprob_out[row] = xmax - lse;
      sample_logprob_out[row] = 0.f;
    }
    return true;
  }

  // 2. every segment's mass over the row's maximum
  const float top_floor = floorf(xmax * inv_w);
  __syncthreads();  // (sh.max, sh.argmax have been read)
  float seg_mass = 0.f;
  if (tid < SEG_MOST) {
    const float scale = tid < n_segs && rec.max > -__builtin_inff() ? expf((rec.max - xmax) * inv_t) : 0.f;
    seg_mass = scale > 0.f ? rec.mass * scale : 0.f;
    sh.scale[tid] = scale;
    sh.below[tid] = scale > 0.f ? bins_below(top_floor, rec.max * inv_w) : SEG_BINS;
    sh.kept[tid] = 0;
  }
  const float z = join_sum(seg_mass, sh.scratch);
  const bool nucleus = row_top_p < 1.0f;
  int bin = SEG_BINS, sub = SEG_BINS;  // kept whole: the bins before `bin`, and of that one the parts before `sub`
  float least = 0.f;                   // kept of part `sub` (of the whole bin if it is not divided): the entries from here on
  auto e_of = [&](float v) { return expf((v - xmax) * inv_t); };
  auto bin_of = [&](float scaled) { return bins_below(top_floor, scaled); };
  auto kept = [&](float v) {
    if (!nucleus) return v > -__builtin_inff() ? e_of(v) : 0.f;
    const float scaled = v * inv_w;
    const int k = v > -__builtin_inff() ? bin_of(scaled) : SEG_BINS;
    if (k != bin) return k < bin ? e_of(v) : 0.f;
    if (sub < SEG_BINS) {
      const int j = part_of_bin(scaled);
      if (j != sub) return j < sub ? e_of(v) : 0.f;
    }
    const float e = e_of(v);
    return e >= least ? e : 0.f;
  };

  if (nucleus) {
    // 3. the bin in which the mass from the top passes top_p * z
    const float target = row_top_p * z;
    const int g = tid & (SEG_BINS - 1);
    float m = 0.f;
    constexpr int APART = SAMPLE_THREADS / SEG_BINS, TOGETHER = 4;  // histograms whose loads are in flight at once
    for (int s0 = tid / SEG_BINS; s0 < n_segs; s0 += APART * TOGETHER) {
      float h[TOGETHER];
#pragma unroll
      for (int q = 0; q < TOGETHER; ++q) {
        const int s = min(s0 + q * APART, n_segs - 1), k = g - sh.below[s];
        h[q] = 0.f;
        if (s0 + q * APART < n_segs && k >= 0 && k < SEG_BINS - 1) h[q] = seg_histogram(row_workspace, n_segs, s)[k];
      }
#pragma unroll
      for (int q = 0; q < TOGETHER; ++q) m = fmaf(h[q], sh.scale[min(s0 + q * APART, n_segs - 1)], m);
    }
    sh.part[tid / SEG_BINS][g] = m;
    __syncthreads();
    m = tid < SEG_BINS - 1 ? sh.part[0][tid] + sh.part[1][tid] + sh.part[2][tid] + sh.part[3][tid] : 0.f;
    const float cum = block_scan(m, sh.scratch);
    if (tid == 0) sh.first = SEG_BINS, sh.count = 0, sh.smallest = 0x7f800000;
    __syncthreads();
    const unsigned long long past = __ballot(m > 0.f && cum > target);
    if (lane == 0 && past) atomicMin(&sh.first, tid + __ffsll(past) - 1);
    __syncthreads();
    bin = sh.first;
    if (bin >= SEG_BINS - 1) {  // the passing point lies below 32 octaves
      return false;
    }
    if (tid == bin) sh.before = cum - m;
    if (tid < SEG_BINS) sh.sub[tid] = 0;
    __syncthreads();
    float above = sh.before;

    // of every segment the bins before it, a wavefront a segment: used at the end, read with the loads that follow
    constexpr int WAVES = SAMPLE_THREADS / CWM_WAVE, SEGS = 4;  // segments of a wavefront at once
    const int first_seg = __builtin_amdgcn_readfirstlane(wave);
    for (int s0 = first_seg; s0 < n_segs; s0 += WAVES * SEGS) {
      float h[SEGS][SEG_BINS / CWM_WAVE] = {};
#pragma unroll
      for (int g = 0; g < SEGS; ++g) {
        const int s = s0 + g * WAVES;
        if (s < n_segs) {
          const int below = sh.below[s];
          const float* hist = seg_histogram(row_workspace, n_segs, s);
#pragma unroll
          for (int q = 0; q < SEG_BINS / CWM_WAVE; ++q) {
            const int k = q * CWM_WAVE + lane;
            if (k < SEG_BINS - 1 && k + below < bin) h[g][q] = hist[k];
          }
        }
      }
#pragma unroll
      for (int g = 0; g < SEGS; ++g) {
        const int s = s0 + g * WAVES;
        if (s < n_segs) {
          float whole = 0.f;
#pragma unroll
          for (int q = 0; q < SEG_BINS / CWM_WAVE; ++q) whole += h[g][q];
          whole = wave_sum(whole);
          if (lane == 0) sh.mass[s] = whole;
        }
      }
    }

    // 4. that bin's entries, a segment a wavefront, where the segment has mass in it: take(segment, its first entry,
    //    the lane's entries that lie in the bin)
    const float edge = top_floor - bin;  // x lies in the bin if edge <= x * inv_w < edge + 1
    static_assert(SEG_MOST <= SAMPLE_THREADS, "a lane looks at one of its wavefront's segments");
    const int looked = wave + lane * (SAMPLE_THREADS / CWM_WAVE);
    const int looked_bin = looked < n_segs ? bin - sh.below[looked] : -1;
    const unsigned long long with_mass =
        __ballot(looked_bin >= 0 && seg_histogram(row_workspace, n_segs, looked)[min(looked_bin, SEG_BINS - 1)] > 0.f);
    auto scan_bin = [&](auto&& take) {
      for (unsigned long long left = with_mass; left; left &= left - 1) {
        const int s = wave + (__ffsll(left) - 1) * (SAMPLE_THREADS / CWM_WAVE);
        const int begin = s * seg_len, end = min(vocab, begin + seg_len);
        constexpr int LOADS = SEG_ENTRIES / (4 * CWM_WAVE);
        uint32_t marked = 0;
#pragma unroll 1
        for (int h = 0; h < LOADS; h += LOADS / 2) {
          float4 f[LOADS / 2];  // in flight at once
#pragma unroll
          for (int q = 0; q < LOADS / 2; ++q) {
            const int i = begin + 4 * ((h + q) * CWM_WAVE + lane);
            f[q] = make_float4(-__builtin_inff(), -__builtin_inff(), -__builtin_inff(), -__builtin_inff());
            if (VEC) {
              if (i < end) f[q] = *(const float4*)(x + i);
            } else {
              if (i < end) f[q].x = x[i];
              if (i + 1 < end) f[q].y = x[i + 1];
              if (i + 2 < end) f[q].z = x[i + 2];
              if (i + 3 < end) f[q].w = x[i + 3];
            }
          }
          auto in_bin = [&](float v) { return v * inv_w >= edge && v * inv_w < edge + 1.0f; };
#pragma unroll
          for (int q = 0; q < LOADS / 2; ++q) {
            const uint32_t four = (in_bin(f[q].x) ? 1u : 0u) | (in_bin(f[q].y) ? 2u : 0u) | (in_bin(f[q].z) ? 4u : 0u) | (in_bin(f[q].w) ? 8u : 0u);
            marked |= four << (4 * (h + q));
          }
        }
        take(s, begin, marked);
      }
      __syncthreads();
    };
    auto entry_at = [&](int begin, int j) { return begin + 4 * ((j / 4) * CWM_WAVE + lane) + j % 4; };
    // the marked entries go to the list; a wavefront takes its places there with one addition
    auto list = [&](int begin, uint32_t marked) {
      const int mine = __popc(marked);
      int through = mine;
#pragma unroll
      for (int off = 1; off < CWM_WAVE; off <<= 1) {
        const int o = __shfl_up(through, off, CWM_WAVE);
        if (lane >= off) through += o;
      }
      int place = 0;
      if (lane == CWM_WAVE - 1 && through > 0) place = atomicAdd(&sh.count, through);
      place = __shfl(place, CWM_WAVE - 1, CWM_WAVE) + through - mine;
      for (; marked; marked &= marked - 1, ++place) {
        const int i = entry_at(begin, __ffs(marked) - 1);
        if (place < SEG_LIST) sh.list_x[place] = x[i], sh.list_i[place] = i;
      }
    };
    scan_bin([&](int, int begin, uint32_t marked) { list(begin, marked); });
    int n = sh.count;
    const bool all_listed = n <= SEG_LIST;
    if (n > SEG_SORT) {
      // 5. too many to put in order: the bin's 256 parts by their masses, and the entries of the part in which the point lies
      auto add = [&](float v) { atomicAdd(&sh.sub[part_of_bin(v * inv_w)], __float2ull_rn(e_of(v) * ROW_FIXED)); };
      if (all_listed) {
        for (int j = tid; j < n; j += SAMPLE_THREADS) add(sh.list_x[j]);
        __syncthreads();
      } else {
        scan_bin([&](int, int begin, uint32_t marked) {
          for (; marked; marked &= marked - 1) add(x[entry_at(begin, __ffs(marked) - 1)]);
        });
      }
      const float part = tid < SEG_BINS ? (float)sh.sub[tid] * (1.0f / ROW_FIXED) : 0.f;
      const float run = block_scan(part, sh.scratch);
      float before;
      sub = first_past(sh, part, run, target - above, before);
      if (sub < 0) {  // no part with mass
        return false;
      }
      above += before;
      if (tid == 0) sh.count = 0;
      __syncthreads();
      if (all_listed) {
        // the list's entries before the part are kept; the part's go to the list's front, once everything has been read
        float v[SEG_LIST / SAMPLE_THREADS];
        int at[SEG_LIST / SAMPLE_THREADS];
#pragma unroll
        for (int q = 0; q < SEG_LIST / SAMPLE_THREADS; ++q) {
          const int j = q * SAMPLE_THREADS + tid;
          v[q] = j < n ? sh.list_x[j] : 0.f;
          at[q] = j < n ? sh.list_i[j] : -1;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < SEG_LIST / SAMPLE_THREADS; ++q) {
          if (at[q] < 0) continue;
          const int p = part_of_bin(v[q] * inv_w);
          if (p < sub) atomicAdd(&sh.kept[at[q] / seg_len], __float2ull_rn(e_of(v[q]) * ROW_FIXED));
          if (p == sub) {
            const int place = atomicAdd(&sh.count, 1);
            sh.list_x[place] = v[q], sh.list_i[place] = at[q];
          }
        }
        __syncthreads();
      } else {
        scan_bin([&](int s, int begin, uint32_t marked) {
          float whole = 0.f;
          uint32_t in_part = 0;
          for (; marked; marked &= marked - 1) {
            const int j = __ffs(marked) - 1;
            const float v = x[entry_at(begin, j)];
            const int p = part_of_bin(v * inv_w);
            if (p < sub) whole += e_of(v);
            if (p == sub) in_part |= 1u << j;
          }
          whole = wave_sum(whole);
          if (lane == 0) sh.kept[s] = __float2ull_rn(whole * ROW_FIXED);
          list(begin, in_part);
        });
      }
      n = sh.count;
      if (n > SEG_SORT) {  // over a thousand entries within a 2,048th of an octave
        return false;
      }
    }
    // 6. an entry is kept if the mass of the larger ones does not pass the target: the listed ones in descending order
    const float own = tid < n ? e_of(sh.list_x[tid]) : 0.f;
    const int owner = tid < n ? sh.list_i[tid] / seg_len : 0;
    float key = own;
    if (n <= SEG_RANK) {
      // an entry's place is the number of larger ones and of equal ones before it, counted by RANKERS threads
      constexpr int RANKERS = SAMPLE_THREADS / SEG_RANK;
      if (tid < SEG_RANK) sh.part[0][tid] = own;
      __syncthreads();
      const int entry = tid / RANKERS, at = tid % RANKERS;
      const float mine = sh.part[0][entry];
      int place = 0;
      for (int j = at; j < n; j += RANKERS) place += sh.part[0][j] > mine || (sh.part[0][j] == mine && j < entry);
#pragma unroll
      for (int off = 1; off < RANKERS; off <<= 1) place += __shfl_xor(place, off, CWM_WAVE);
      if (at == 0 && entry < n) sh.part[1][place] = mine;
      __syncthreads();
      key = tid < n ? sh.part[1][tid] : 0.f;
    }
    int size = n <= SEG_RANK ? 1 : CWM_WAVE;
    while (size > 1 && size < n) size <<= 1;
    for (int k = 2; k <= size; k <<= 1)
      for (int j = k >> 1; j > 0; j >>= 1) {
        float other;
        if (j < CWM_WAVE) {
          other = __shfl_xor(key, j, CWM_WAVE);
        } else {
          __syncthreads();
          sh.sorted[tid] = key;
          __syncthreads();
          other = sh.sorted[tid ^ j];
        }
        key = ((tid & k) == 0) == ((tid & j) == 0) ? fmaxf(key, other) : fminf(key, other);
      }
    const float through = block_scan(key, sh.scratch);
    const unsigned long long fits = __ballot(tid < n && above + (through - key) <= target);
    if (fits && lane == CWM_WAVE - 1 - __clzll((long long)fits)) atomicMin(&sh.smallest, __float_as_int(key));  // the wavefront's smallest: keys descend
    __syncthreads();
    least = __int_as_float(sh.smallest);
    if (tid < n && own >= least) atomicAdd(&sh.kept[owner], __float2ull_rn(own * ROW_FIXED));
    __syncthreads();
    // the kept mass of every segment: its bins before `bin` and what the list gave
    seg_mass = tid < n_segs ? sh.mass[tid] * sh.scale[tid] + (float)sh.kept[tid] * (1.0f / ROW_FIXED) : 0.f;
  }

  // 7. inverse CDF: the segment in which the running mass passes u * (kept mass), then the entry.  The two levels' sums are
  //    rounded differently, so a level may find the point beyond its last mass: it then takes its last entry with mass.
  float total;
  const float run = block_scan(seg_mass, sh.scratch, &total);
  const float target = u * total;
  float before;
  const int seg = first_past(sh, seg_mass, run, target, before);
  if (seg < 0) {
    return false;
  }
  const int begin = seg * seg_len, end = min(vocab, begin + seg_len);
  const int i = begin + 2 * tid;  // two adjacent entries a thread
  const float e0 = i < end ? kept(x[i]) : 0.f, e1 = i + 1 < end ? kept(x[i + 1]) : 0.f;
  const float cum = block_scan(e0 + e1, sh.scratch);
  float entry_before;
  const int pick = first_past(sh, e0 + e1, cum, target - before, entry_before);
  if (pick < 0) {
    if (tid == 0) token_out[row] = best.i, logprob_out[row] = xmax - lse, sample_logprob_out[row] = logf(1.0f / total);
    return true;
  }
  if (tid == pick) {
    const bool second = !(e0 > 0.f) || (e1 > 0.f && entry_before + e0 <= target - before);
    token_out[row] = second ? i + 1 : i;
    logprob_out[row] = x[second ? i + 1 : i] - lse;
    sample_logprob_out[row] = logf((second ? e1 : e0) / total);
  }
  return true;
}

// One block a row, so it is bound by its own chain: records, histograms, the bin's entries, the kept segments' masses and the
// segment with the draw are read one after the other, with barriers and sums over the block between them.  So that a link costs
// one trip to memory, loads of one kind are issued together: four histograms (only where they count: the rows of all 63 without
// condition were 7 instead of 3 us), the segments that hold the bin by one look, the masses before the bin with the first of
// these; the wavefronts' sums are read as a block, and a wavefront sends one atomic, not one a lane.  A row of 128,256 with a
// nucleus of few entries 16.2 instead of 22.7 us, of 32,768 14.6 instead of 19.8; at top_p = 1 the choice as a whole 11 instead of 19.
template <bool VEC>
__global__ void __launch_bounds__(SAMPLE_THREADS, 8)
sample_join_kernel(const float* __restrict__ logits, long row_stride, int vocab, int seg_len, int n_segs, const float* __restrict__ temperature,
                   const float* __restrict__ top_p, const float* __restrict__ uniform, float* __restrict__ workspace,
                   int* __restrict__ token_out, float* __restrict__ logprob_out, float* __restrict__ sample_logprob_out) {
  __shared__ union {
    JoinShared join;
    WholeRowShared whole;
  } shared;
  if (join_segments<VEC>(shared.join, blockIdx.x, logits, row_stride, vocab, seg_len, n_segs, temperature, top_p, uniform, workspace, token_out,
                         logprob_out, sample_logprob_out))
    return;
  __syncthreads();
  sample_whole_row<VEC>(shared.whole, blockIdx.x, logits, row_stride, vocab, temperature, top_p, uniform, workspace, token_out, logprob_out,
                        sample_logprob_out);
}

static void launch_sample(const float* logits, long row_stride, int n_rows, int vocab, const float* temperature, const float* top_p,
                          const float* uniform, float* workspace, int* token_out, float* logprob_out, float* sample_logprob_out,
                          hipStream_t stream) {
  // four entries a load where every row of the logits and of the workspace starts at a multiple of 16 bytes
  const bool vec = vocab % 4 == 0 && row_stride % 4 == 0 && (uintptr_t)logits % 16 == 0 && (uintptr_t)workspace % 16 == 0;
  // in segments where the row is long enough and their number fits the second kernel's lists; the records and histograms
  // (1,040 bytes for every 1,024 entries or more) fit the row's part of the workspace
  const int seg_len = seg_length(vocab), n_segs = (vocab + seg_len - 1) / seg_len;
  if (vocab > SEGMENTS_FROM && n_segs <= SEG_MOST && n_rows <= 65535) {
    auto launch = [&](auto v) {
      hipLaunchKernelGGL(sample_segment_kernel<decltype(v)::value>, dim3(n_segs, n_rows), dim3(SEG_THREADS), 0, stream, logits, row_stride, vocab,
                         seg_len, temperature, top_p, workspace);
      hipLaunchKernelGGL(sample_join_kernel<decltype(v)::value>, dim3(n_rows), dim3(SAMPLE_THREADS), 0, stream, logits, row_stride, vocab, seg_len,
                         n_segs, temperature, top_p, uniform, workspace, token_out, logprob_out, sample_logprob_out);
    };
    if (vec) launch(std::true_type());
    else launch(std::false_type());
    return;
  }
  if (vec)
    hipLaunchKernelGGL(sample_kernel<true>, dim3(n_rows), dim3(SAMPLE_THREADS), 0, stream, logits, row_stride, vocab, temperature,
                       top_p, uniform, workspace, token_out, logprob_out, sample_logprob_out);
  else
    hipLaunchKernelGGL(sample_kernel<false>, dim3(n_rows), dim3(SAMPLE_THREADS), 0, stream, logits, row_stride, vocab, temperature,
                       top_p, uniform, workspace, token_out, logprob_out, sample_logprob_out);
}

extern "C" int cwm_sample(const float* logits, long row_stride, int n_rows, int vocab, const float* temperature,
                          const float* top_p, const float* uniform, float* workspace, int* token_out,
                          float* logprob_out, float* sample_logprob_out, hipStream_t stream) {
  CWM_REQUIRE(n_rows >= 0 && vocab > 0, "sample: bad sizes rows=%d vocab=%d", n_rows, vocab);
  CWM_REQUIRE(row_stride >= vocab, "sample: row stride shorter than the vocabulary");
  CWM_REQUIRE(workspace != nullptr, "sample: workspace missing");
  if (n_rows == 0) return 0;
  launch_sample(logits, row_stride, n_rows, vocab, temperature, top_p, uniform, workspace, token_out, logprob_out, sample_logprob_out, stream);
  return cwm_launch_status("sample");
}

// ---- the same without a workspace argument: nothing is allocated ------------------ //
// The unnormalised probabilities go to a device array of this file; see no_alloc.h.
// In host code `sample_scratch` is only a stand-in for the symbol: its device address
// differs from GPU to GPU and is looked up once per device, with that device current.
static __device__ __align__(256) float sample_scratch[CWM_SAMPLE_STATIC_MAX_FLOATS];

#define CWM_MAX_DEVICES 64
static float* sample_scratch_ptr[CWM_MAX_DEVICES] = {nullptr};
static std::mutex sample_scratch_mutex;

extern "C" long cwm_sample_static_capacity() { return CWM_SAMPLE_STATIC_MAX_FLOATS; }

// The array's address on the current device, looked up at the first call there.  Sets `*out`; returns non-zero on failure.
static int sample_scratch_on_current_device(float** out) {
  int device = -1;
  hipError_t err = hipGetDevice(&device);
  if (err != hipSuccess) return cwm_fail("sample_static: hipGetDevice failed: %s", hipGetErrorString(err));
  CWM_REQUIRE(device >= 0 && device < CWM_MAX_DEVICES, "sample_static: device %d is outside 0..%d", device, CWM_MAX_DEVICES - 1);
  std::lock_guard<std::mutex> guard(sample_scratch_mutex);
  if (sample_scratch_ptr[device] == nullptr) {
    void* found = nullptr;
    err = hipGetSymbolAddress(&found, HIP_SYMBOL(sample_scratch));
    if (err != hipSuccess || found == nullptr)
      return cwm_fail("sample_static: the scratch array has no address on device %d: %s", device, hipGetErrorString(err));
    sample_scratch_ptr[device] = (float*)found;
  }
  *out = sample_scratch_ptr[device];
  return 0;
}

extern "C" int cwm_sample_static_init() {
  float* scratch = nullptr;
  return sample_scratch_on_current_device(&scratch);
}

extern "C" int cwm_sample_static(const float* logits, long row_stride, int n_rows, int vocab,
                                 const float* temperature, const float* top_p, const float* uniform,
                                 int* token_out, float* logprob_out, float* sample_logprob_out,
                                 hipStream_t stream) {
  CWM_REQUIRE(n_rows >= 0 && vocab > 0, "sample_static: bad sizes rows=%d vocab=%d", n_rows, vocab);
  CWM_REQUIRE(row_stride >= vocab, "sample_static: row stride shorter than the vocabulary");
  CWM_REQUIRE((long long)n_rows * vocab <= (long long)CWM_SAMPLE_STATIC_MAX_FLOATS,
              "sample_static: %d rows of %d logits need %lld floats of scratch, the fixed array holds %d", n_rows, vocab,
              (long long)n_rows * vocab, CWM_SAMPLE_STATIC_MAX_FLOATS);
  if (n_rows == 0) return 0;
  float* scratch = nullptr;
  if (int status = sample_scratch_on_current_device(&scratch)) return status;
  launch_sample(logits, row_stride, n_rows, vocab, temperature, top_p, uniform, scratch, token_out, logprob_out, sample_logprob_out, stream);
  return cwm_launch_status("sample_static");
}

// log softmax(logits[rows[i]])[targets[i]] for given tokens: the log-probabilities of a
// prompt's own tokens (cwm/fastgen/forward.py:908-924).  One block per entry.
__global__ void __launch_bounds__(SAMPLE_THREADS)
token_logprob_kernel(const float* __restrict__ logits, long row_stride, int vocab, const int* __restrict__ rows,
                     const int* __restrict__ targets, float* __restrict__ out) {
  __shared__ float scratch[16];
  const int i = blockIdx.x;
  const float* x = logits + (size_t)rows[i] * row_stride;
  float mx = -__builtin_inff();
#pragma unroll 4
  for (int v = threadIdx.x; v < vocab; v += SAMPLE_THREADS) mx = fmaxf(mx, x[v]);
  mx = block_max(mx, scratch);
  float sum = 0.f;
#pragma unroll 4
  for (int v = threadIdx.x; v < vocab; v += SAMPLE_THREADS) sum += expf(x[v] - mx);
  sum = block_sum(sum, scratch);
  if (threadIdx.x == 0) {
    const int t = targets[i];
    out[i] = (t >= 0 && t < vocab) ? x[t] - (mx + logf(sum)) : __uint_as_float(0x7fc00000u);
  }
}

extern "C" int cwm_token_logprob(const float* logits, long row_stride, int n_rows_total, int vocab, const int* rows,
                                 const int* targets, int n, float* out, hipStream_t stream) {
  CWM_REQUIRE(n >= 0 && vocab > 0 && n_rows_total >= 0, "token_logprob: bad sizes");
  CWM_REQUIRE(row_stride >= vocab, "token_logprob: row stride shorter than the vocabulary");
  if (n == 0) return 0;
  hipLaunchKernelGGL(token_logprob_kernel, dim3(n), dim3(SAMPLE_THREADS), 0, stream, logits, row_stride, vocab, rows,
                     targets, out);
  return cwm_launch_status("token_logprob");
}

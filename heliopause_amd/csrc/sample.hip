// sample.hip -- next-token sampling from top-k candidates, on the device.
//
// Restates tokenSamplingDistribution / sampleNextToken with their softmax,
// applyTopP and createDeterministicRng (packages/engine/src/generation.ts
// 78-165) over the [columns][k] candidates the top-k kernels leave in HBM, so
// a decode loop can pick the next token without a host round trip.  JS
// numbers are IEEE doubles: every step here is a double operation in the
// reference's order (no contraction), Math.exp is hp_exp (the JS engine's
// algorithm), and the sums the reference takes left to right (softmax total,
// top-p and draw cumulatives) are taken left to right.  Columns draw in order
// from one generator state, as the reference draws them one after another;
// greedy columns draw nothing.
//
// One workgroup, a wave per column (round robin past 16): the generator's
// state advances by a constant per draw, so column c's draw is known without
// the ones before it.  What bounds a column is the chain of its left-to-right
// sums; each takes its terms from the lanes' registers (readlane), four at a
// time, so that their reads do not wait for the sum.  A column of 64
// candidates after its top-k launch (default top-p) 9.6 us with one lane
// reading the terms back from LDS, 10.3 with a readlane and its loop per term,
// 8.1 as it is; in a loop of its own 5.0, 5.7, 5.3.  Five columns of 40
// candidates, which one wave took one after another, 33 -> 8.2 us.
#include "hp_common.h"
#include "hp_exp.h"

namespace hp {

namespace {

constexpr int kLanes = 64;
constexpr int kWaves = 16;

// createDeterministicRng (generation.ts:78-87): the JS operations are 32-bit
// wrapping ones (Math.imul, ToInt32 of a sum of two int32, >>> 0).  `state` is
// the generator's after its step (+ kRngStep).
constexpr uint32_t kRngStep = 0x6D2B79F5u;
__device__ __forceinline__ double rng_value(uint32_t state) {
  uint32_t v = state;
  v = (v ^ (v >> 15)) * (v | 1u);
  v ^= v + (v ^ (v >> 7)) * (v | 61u);
  return (double)(v ^ (v >> 14)) / 4294967296.0;
}

constexpr int kTerms = 4;  // terms of a left-to-right sum read at once
static_assert(kLanes % kTerms == 0, "whole groups of terms");

// Lane i's value (i the same in every lane).
__device__ __forceinline__ double lane_value(double v, int i) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, i);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), i);
  return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}

// softmax (generation.ts:157-165) of the n values held by lanes 0..n-1;
// returns this lane's probability (0 for lanes >= n).  The sum's terms past n
// are 0 and change nothing.
__device__ double softmax_lane(double x, int n) {
  const int lane = threadIdx.x & (kLanes - 1);
  const bool valid = lane < n;
  // Math.max over the values from -Infinity: NaN if any value is NaN.  The
  // sign of a zero maximum cannot change exp(x - max).
  const bool nan = valid && __builtin_isnan(x);
  double m = valid && !nan ? x : -__builtin_inf();
#pragma unroll
  for (int off = kLanes / 2; off > 0; off >>= 1) {
    const double o = __shfl_xor(m, off);
    m = o > m ? o : m;
  }
  if (__any(nan)) m = __builtin_nan("");
  const double e = valid ? hp_exp(x - m) : 0.0;
  double s = 0.0;
  for (int i = 0; i < n; i += kTerms) {
    double t[kTerms];
#pragma unroll
    for (int j = 0; j < kTerms; j++) t[j] = lane_value(e, i + j);
#pragma unroll
    for (int j = 0; j < kTerms; j++) s = s + t[j];
  }
  double p;
  if (s <= 0.0 || !__builtin_isfinite(s))
    p = lane == 0 ? 1.0 : 0.0;
  else
    p = e / s;
  return valid ? p : 0.0;
}

// Lanes 0 .. i, the first i < n at which the left-to-right sum of q passes:
// sum > limit, or (at_least) sum >= limit.  n when none does.  q are
// probabilities, 0 from lane n on, so the sum never falls: a group of terms
// holds the first i when its last sum passes.
__device__ int first_over(double q, int n, double limit, bool at_least) {
  auto passes = [&](double sum) { return at_least ? sum >= limit : limit < sum; };
  double cum = 0.0;
  for (int i = 0; i < n; i += kTerms) {
    double t[kTerms];
#pragma unroll
    for (int j = 0; j < kTerms; j++) t[j] = lane_value(q, i + j);
#pragma unroll
    for (int j = 0; j < kTerms; j++) t[j] = cum = cum + t[j];
    if (passes(cum)) {
      int at = i;
#pragma unroll
      for (int j = 0; j < kTerms - 1; j++) at += passes(t[j]) ? 0 : 1;
      return at;
    }
  }
  return n;
}

__global__ __launch_bounds__(kLanes * kWaves) void sample_kernel(const uint32_t *__restrict__ ids,
                                                        const float *__restrict__ vals, int cols, int k, int count,
                                                        SampleParams p, uint32_t *__restrict__ rng,
                                                        int32_t *__restrict__ tokens, double *__restrict__ probs,
                                                        int32_t *__restrict__ kept) {
  const int lane = threadIdx.x & (kLanes - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes), waves = blockDim.x / kLanes;
  const bool greedy = p.do_sample == 0 || p.temperature == 0.0;
  const uint32_t state = rng[0];
  __syncthreads();  // every wave has the state before it moves on
  if (threadIdx.x == 0 && !greedy) rng[0] = state + (uint32_t)cols * kRngStep;
  for (int c = wave; c < cols; c += waves) {
    const uint32_t id = lane < count ? ids[(size_t)c * k + lane] : 0u;
    const double v = lane < count ? (double)vals[(size_t)c * k + lane] : 0.0;
    if (greedy) {  // the best candidate with probability 1; no draw
      if (lane == 0) {
        tokens[c] = (int32_t)id;
        probs[(size_t)c * k] = 1.0;
        kept[c] = 1;
      }
      continue;
    }
    const int n1 = count < p.top_k ? count : p.top_k;  // topK slice of the sorted candidates
    int n2 = n1;
    if (!(p.top_p >= 1.0) && n1 > 1) {  // applyTopP (generation.ts:135-155)
      const int at = first_over(softmax_lane(v, n1), n1, p.top_p, true);
      n2 = at < n1 ? at + 1 : n1;
    }
    const double q = softmax_lane(v / p.temperature, n2);
    if (lane < n2) probs[(size_t)c * k + lane] = q;
    // sampleNextToken (generation.ts:89-108)
    const int at = first_over(q, n2, rng_value(state + (uint32_t)(c + 1) * kRngStep), false);
    const int32_t tok = __builtin_amdgcn_readlane((int)id, at < n2 ? at : n2 - 1);
    if (lane == 0) {
      tokens[c] = tok;
      kept[c] = n2;
    }
  }
}

}  // namespace

hipError_t launch_sample(const uint32_t *ids, const float *vals, int cols, int k, int count, const SampleParams &p,
                         uint32_t *rng, int32_t *tokens, double *probs, int32_t *kept, hipStream_t s) {
  if (cols < 1 || k < 1 || k > kLanes || count < 1 || count > k || p.top_k < 1) return hipErrorInvalidValue;
  const int waves = cols < kWaves ? cols : kWaves;
  hipLaunchKernelGGL(sample_kernel, dim3(1), dim3(kLanes * waves), 0, s, ids, vals, cols, k, count, p, rng, tokens, probs,
                     kept);
  return hipGetLastError();
}

}  // namespace hp

// Sampling from logits rows: temperature, top-k, top-p (HF's logits warpers,
// transformers generation/logits_process.py TemperatureLogitsWarper,
// TopKLogitsWarper, TopPLogitsWarper), then one draw from the softmax of the
// kept scores by the Gumbel-max method.  Declarations shared by the C ABI
// (qmk_api.hip) and the kernels (qmk_sample.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qmk_state.h"

namespace qmk {

// SplitMix64 finaliser with its golden-ratio increment (G. Steele, D. Lea,
// C. Flood, "Fast splittable pseudorandom number generators", OOPSLA 2014).
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// Per-draw base of the random numbers: (seed, counter).
__device__ __forceinline__ uint64_t draw_base(uint64_t seed, uint64_t counter) { return mix64(seed ^ mix64(counter)); }

// U in (0, 1) for token v: the top 24 bits of the hash, centred in their interval.
__device__ __forceinline__ float draw_uniform(uint64_t base, int v) {
  const uint64_t h = mix64(base + (uint64_t)(uint32_t)v);
  return ((float)(uint32_t)(h >> 40) + 0.5f) * (1.0f / 16777216.0f);
}

// Order-preserving uint32 key of a float.
__device__ __forceinline__ uint32_t key32(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Key of token v's Gumbel-perturbed score s: key32(s + G), G = -log(-log(U)).
__device__ __forceinline__ uint32_t gumbel_key_score(float s, uint64_t base, int v) {
  return key32(s + -logf(-logf(draw_uniform(base, v))));
}
__device__ __forceinline__ uint32_t gumbel_key(float logit, float temperature, uint64_t base, int v) {
  return gumbel_key_score(__fdiv_rn(logit, temperature), base, v);
}

struct SampleParams {
  float temperature;  // <= 0: greedy (first index of the maximum)
  int top_k;          // keep scores >= the top_k-th largest; <= 0 or >= vocab: off
  float top_p;        // keep the highest scores whose mass above them is < top_p; outside (0, 1): off
  uint64_t seed;
};

// Device work of one logits row between the launches of a sampling call: its selection state, and the
// histogram of one 8-bit radix digit (counts or fixed-point masses).  Zero between calls: the call's last
// launch clears it.
constexpr int kSampleBins = 2048, kSampleCand = 4096;
struct SampleWork {
  unsigned long long hist[256];
  unsigned long long z, target, need, best;  // need: top-k rank still sought / top-p mass above the prefix
  unsigned int maxkey, prefix, mask, kmin, pmin, ticket;
  // two-launch form: scores above the threshold's bin (both filters) and in it, ~(smallest key) and largest
  // key in the bin, largest key above it, whether the bin is one of the finer ones (and is to be cut so)
  unsigned int nabove, nbin, binmin, binmax, abovemax, finer;
  unsigned long long tied;  // best draw in the bin, if its keys are all the same
};
// What the two-launch form of a filtered draw needs besides, per row of its launches: a histogram (zero
// between calls) and, after it, the tokens in the threshold's bin; those above the bin; up to kSampleCand of each.
struct SampleLists {
  union {
    unsigned long long hist[kSampleBins];
    unsigned int bin[kSampleCand];
  };
  unsigned int above[kSampleCand];
};
// Rows per launch sequence of qmk_sample_rows (0.5 MB of work); of the two-launch form, whose lists would
// make that 8 MB, 128 (4 MB).  A draw of 256 rows without a filter takes 33-84 us in one sequence and 107-167
// in four.
constexpr int kSampleRowsMax = 256, kSampleListRows = 128;

// The work of up to `rows` rows, in one allocation: `rows` SampleWork, then the lists.
__host__ __device__ inline SampleLists* sample_lists(SampleWork* work, int rows) {
  return reinterpret_cast<SampleLists*>(work + rows);
}

// hipMalloc + zero fill of the work of `rows` rows.
int alloc_sample_work(SampleWork** out, int rows);

// Persistent-mode sampler of the generate loop: when the decode step just run
// produced `logits`, replace its greedy token in the state and the log by a
// sampled one (counter = the step's position) and set `done` for the stop token.
// `work`: one row's zeroed work, owned by the caller's stream.
int launch_sample_state(const float* logits, int vocab, const SampleParams& sp, DecodeState* st, int* log,
                        SampleWork* work, hipStream_t stream);

}  // namespace qmk

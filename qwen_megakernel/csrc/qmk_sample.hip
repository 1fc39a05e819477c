// Sampling kernels.  Each logits row is spread over G workgroups of 256
// threads (G from 8 to 128, so that a single row fills many CUs); the passes
// are separate launches and no workgroup ever waits for another.
//
//   s_v = logit_v / T                       (HF TemperatureLogitsWarper, fp32 divide)
//   top-k: keep s_v >= the k-th largest s   (HF TopKLogitsWarper: ties at the k-th value kept)
//   top-p: keep v iff the probability mass of the kept scores strictly above s_v is < p
//          (HF TopPLogitsWarper removes sorted tokens whose ascending cumulative
//          probability is <= 1 - p; at least the top token stays)
//   draw:  argmax over kept v of s_v + G_v, G_v = -log(-log(U_v)) (Gumbel-max: a draw
//          from softmax of the kept s), U_v from a counter-based hash of (seed, counter, v)
//
// Thresholds are exact: top-k over integer counts, top-p over probability masses held as 2^-40
// fixed-point integers (exp(s_v - max) rounded once).  Integer sums and integer maxima do not depend
// on the order of the atomics, so results are deterministic.  The random numbers use SplitMix64
// (G. Steele, D. Lea, C. Flood, "Fast splittable pseudorandom number generators", OOPSLA 2014).
//
// With a filter, a call is two launches over the row (three for top-p alone, whose masses need the
// row's maximum first; in the generate loop that is the decode step's own greedy logit over T), and one
// between them that rarely does anything:
// - k_first histograms the slices over 2048 bins in LDS, adds the non-zero bins to the row's with
//   integer atomics, and the last workgroup of the row (a ticket counter) finds the bin that holds the
//   threshold.  top-k: counts over the top 11 bits of the order-preserving 32-bit key of s;  top-p
//   alone: masses over (max - s) in steps of 1/64;
// - k_finer does the same within that bin, 2048 finer ones, where it holds more than kFinerAbove scores: a
//   key bin is up to a quarter of the score wide, so logits far from 0 for their spread fill it, and so
//   do flat ones at a high temperature;
// - k_finish draws among the scores above the bin, which are kept for certain (with both filters it
//   lists them, fewer than top_k), and lists the bin's own; the row's last workgroup finds the exact
//   thresholds among these by radix descent in LDS, draws among those that stay and writes the token.
//   A bin of equal scores, however many (a mask's -inf, bf16 logits), needs no list: they stay or go as one.
// A bin of more than kSampleCand scores even so, not equal but closer than 2^-13 of their value (top-p
// alone: 2^-17), is found again in the logits by the last workgroup, one pass over the row per digit.
// top-k above kFinishTopK keeps the general form: radix descent over the whole row, 8 bits per launch
// (k_hist, 4 launches per threshold, then k_draw).
// A launch that works costs 7-9 us whatever it does, which is what bounds a call; k_finer without work 2.3.
// Four rows of 151,936 scores, T 0.8, us, general form -> two launches without k_finer -> now: N(0,2) with a
// few raised, top-k 50 + top-p 0.9 83 -> 24.6 -> 28.2, top-k 4096 + top-p 0.95 91 -> 836 -> 59; N(10,2), top-k
// 200 + top-p 0.9 84 -> 727 -> 36; all but ten masked, top-k 50 + top-p 0.9 91 -> 1005 -> 43; N(0,0.01), top-p
// 0.9 60 -> 673 -> 44.  The general form is faster for 152,000 distinct scores within 0.01 (one row, top-k
// 4096: 36 against 44).

#include <hip/hip_runtime.h>

#include "../../include/qwen_megakernel.h"
#include "qmk_device.h"
#include "qmk_sample.h"

#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>

namespace qmk {
namespace sample {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr double kFix = 1099511627776.0;  // 2^40
constexpr int kPasses = 4;
constexpr int kBins = 256;  // 8-bit digits

struct Args {
  const float* logits;
  int V;
  SampleParams sp;
  const long long* counters;  // rows mode: per-row counters, out: per-row tokens
  int* out;
  DecodeState* st;            // state mode (one row): counter = st->pos - 1; the token replaces st->tok
  int* log;
  SampleWork* work;           // one per row, zero between calls
  SampleLists* lists;         // one per row (two-launch form)
};

__device__ __forceinline__ float from_key32(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

__device__ __forceinline__ unsigned long long mass_of(float s, float mx) {
  return (unsigned long long)((double)expf(s - mx) * kFix + 0.5);
}

struct Block {
  int row;
  const float* x;
  int v0, v1;           // this workgroup's slice of the row
  uint64_t counter;
  SampleWork* w;
  SampleLists* ls;
  uint32_t greedy_tok;  // state mode: the decode step's greedy token (its logit is the row maximum)
};

// Common prologue: the row and slice of this workgroup; false when the call
// has nothing to do (state mode after a step that only padded the log).
__device__ bool setup(const Args& a, Block& b) {
  __shared__ int run, tok;
  __shared__ long long ctr;
  b.row = blockIdx.y;
  if (threadIdx.x == 0) {
    if (a.st) {
      run = a.st->ran != 0 && a.st->err == 0;
      ctr = (long long)a.st->pos - 1;  // position of the step just run
      tok = a.st->tok;
      if (tok < 0 || tok >= a.V) run = 0;
    } else {
      run = 1;
      ctr = a.counters ? a.counters[b.row] : 0;
    }
  }
  __syncthreads();
  const int chunk = (a.V + gridDim.x - 1) / gridDim.x;
  b.x = a.logits + (size_t)b.row * a.V;
  b.v0 = min(a.V, (int)blockIdx.x * chunk);
  b.v1 = min(a.V, b.v0 + chunk);
  b.counter = (uint64_t)ctr;
  b.w = a.work + b.row;
  b.ls = a.lists + b.row;
  b.greedy_tok = a.st ? (uint32_t)tok : 0u;
  return run != 0;
}

template <class F>
__device__ unsigned long long block_reduce_u64(unsigned long long v, F&& op) {
  __shared__ unsigned long long red[kWaves];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int o = 32; o >= 1; o >>= 1) v = op(v, (unsigned long long)__shfl_xor(v, o));
  if (lane == 0) red[wave] = v;
  __syncthreads();
  v = red[0];
  for (int i = 1; i < kWaves; i++) v = op(v, red[i]);
  return v;
}

// True in every thread of the last workgroup of this pass to finish; the
// other workgroups' atomics are then visible to it.  Each thread waits until
// its device-scope atomics are acknowledged before the ticket is taken, and
// the last workgroup reads the results with agent-scope atomic loads; no
// fence, which on this part would write back the L2.
__device__ bool last_block(SampleWork* w) {
  __shared__ int last;
  wait_vmcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) last = atomicAdd(&w->ticket, 1u) == gridDim.x - 1;
  __syncthreads();
  return last != 0;
}

__device__ __forceinline__ unsigned long long load_u64(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned int load_u32(const unsigned int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Maximum key of s over the row (for the masses).
__global__ void __launch_bounds__(kThreads) k_max(Args a) {
  Block b;
  if (!setup(a, b)) return;
  const float T = a.sp.temperature;
  unsigned long long m = 0;
  for (int v = b.v0 + threadIdx.x; v < b.v1; v += kThreads) {
    const unsigned long long k = key32(__fdiv_rn(b.x[v], T));
    m = k > m ? k : m;
  }
  m = block_reduce_u64(m, [](unsigned long long p, unsigned long long q) { return p > q ? p : q; });
  if (threadIdx.x == 0) atomicMax(&b.w->maxkey, (unsigned int)m);
}

// The maximum score: the decode step's greedy logit over T (state mode), else
// the k_max result.
__device__ __forceinline__ float row_max(const Args& a, const Block& b) {
  return a.st ? __fdiv_rn(b.x[b.greedy_tok], a.sp.temperature) : from_key32(load_u32(&b.w->maxkey));
}

// One radix pass of the top-k (MASS = false: counts) or top-p (MASS = true:
// fixed-point masses of the scores >= kmin) threshold.  The first top-p pass
// also sums the mass Z of the scores >= kmin and sets the target max(1, p Z).
template <bool MASS>
__global__ void __launch_bounds__(kThreads) k_hist(Args a, int pass) {
  __shared__ unsigned long long wh[kWaves][kBins];
  __shared__ unsigned long long hs[kBins];
  __shared__ unsigned int ndig;
  Block b;
  if (!setup(a, b)) return;
  const int shift = 24 - 8 * pass;
  constexpr int nb = kBins;
  const float T = a.sp.temperature;
  SampleWork* w = b.w;
  const uint32_t prefix = load_u32(&w->prefix), mask = load_u32(&w->mask);
  const uint32_t kmin = MASS ? load_u32(&w->kmin) : 0u;
  const float mx = MASS ? row_max(a, b) : 0.f;
  const bool zsum = MASS && pass == 0;
  const int wave = threadIdx.x >> 6;
  for (int i = threadIdx.x; i < kWaves * kBins; i += kThreads) (&wh[0][0])[i] = 0;
  __syncthreads();
  unsigned long long z = 0;
  for (int v = b.v0 + threadIdx.x; v < b.v1; v += kThreads) {
    const float s = __fdiv_rn(b.x[v], T);
    const uint32_t k = key32(s);
    if (k < kmin) continue;
    const unsigned long long m = MASS ? mass_of(s, mx) : 1ull;
    if (zsum) z += m;
    if ((k & mask) == prefix) atomicAdd(&wh[wave][(k >> shift) & (uint32_t)(nb - 1)], m);
  }
  __syncthreads();
  for (int t = threadIdx.x; t < nb; t += kThreads) {
    unsigned long long h = 0;
    for (int q = 0; q < kWaves; q++) h += wh[q][t];
    if (h) atomicAdd(&w->hist[t], h);
  }
  if (zsum) {
    z = block_reduce_u64(z, [](unsigned long long p, unsigned long long q) { return p + q; });
    if (threadIdx.x == 0 && z) atomicAdd(&w->z, z);
  }
  if (!last_block(w)) return;

  // The last workgroup: suffix sums S[d] = sum of bins >= d, then the digit d,
  // the largest in [1, nb) with (mass above +) S[d] >= what is sought, else 0
  // (S is non-increasing, so d is the count of such d).
  for (int t = threadIdx.x; t < nb; t += kThreads) hs[t] = load_u64(&w->hist[t]);
  if (threadIdx.x == 0) ndig = 0;
  __syncthreads();
  for (int off = 1; off < nb; off <<= 1) {
    unsigned long long add[kBins / kThreads];
#pragma unroll
    for (int i = 0; i < kBins / kThreads; i++) {
      const int t = threadIdx.x + i * kThreads;
      add[i] = t < nb && t + off < nb ? hs[t + off] : 0ull;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kBins / kThreads; i++) {
      const int t = threadIdx.x + i * kThreads;
      if (t < nb) hs[t] += add[i];
    }
    __syncthreads();
  }
  unsigned long long target = 0;
  if (MASS) {
    if (zsum) {
      target = (unsigned long long)((double)a.sp.top_p * (double)load_u64(&w->z));
      if (target < 1) target = 1;
    } else {
      target = load_u64(&w->target);
    }
  }
  // top-k: `need` is the rank still sought (k at pass 0); top-p: the mass above the prefix
  const unsigned long long need = pass == 0 ? (MASS ? 0ull : (unsigned long long)a.sp.top_k) : load_u64(&w->need);
  for (int t = threadIdx.x; t < nb; t += kThreads) {
    const bool ok = t >= 1 && (MASS ? need + hs[t] >= target : hs[t] >= need);
    const unsigned long long bal = __ballot(ok);
    if ((threadIdx.x & 63) == 0 && bal) atomicAdd(&ndig, (unsigned int)__popcll(bal));
    w->hist[t] = 0;  // ready for the next pass
  }
  __syncthreads();
  const uint32_t d = ndig;
  if (threadIdx.x == 0) {
    const unsigned long long above = (int)d < nb - 1 ? hs[d + 1] : 0ull;
    const uint32_t np = prefix | (d << shift);
    if (zsum) w->target = target;
    if (pass < kPasses - 1) {
      w->prefix = np;
      w->mask = mask | ((uint32_t)(nb - 1) << shift);
      w->need = MASS ? need + above : need - above;
    } else {
      if (MASS) w->pmin = np;
      else w->kmin = np;
      w->prefix = 0;
      w->mask = 0;
      w->need = 0;
    }
    w->ticket = 0;
  }
}

// The row's token, and its work cleared for the next call (one thread of the row's last workgroup).
__device__ __forceinline__ void put_token(const Args& a, const Block& b, int tok) {
  SampleWork* w = b.w;
  if (a.st) {
    DecodeState* st = a.st;
    st->tok = tok;
    if (a.log) a.log[st->step - 1] = tok;
    st->done = (st->eos >= 0 && tok == st->eos) ? 1u : 0u;
  } else {
    a.out[b.row] = tok;
  }
  w->z = w->target = w->need = w->best = w->tied = 0;
  w->maxkey = w->prefix = w->mask = w->kmin = w->pmin = 0;
  w->nabove = w->nbin = w->binmin = w->binmax = w->abovemax = w->finer = 0;
  w->ticket = 0;
}

constexpr int kFirstShift = 21;       // top-k: bins are the key's top 11 bits
constexpr float kStepsPerUnit = 64.f;  // top-p alone: bins are steps of max - s
constexpr int kFinerBits = 11;          // finer bins: the next 11, steps of 1/2048 of those
constexpr int kFinishTopK = kSampleCand;  // largest top-k whose scores above the threshold's bin fit the list
constexpr unsigned long long kFinerAbove = 512;  // scores in the bin from which k_finer pays
constexpr int kUnroll = 8;            // logits in flight per thread
static_assert(kSampleBins == 8 * kThreads, "eight bins per thread");

// f(v, logit) for this thread's elements v = v0 + threadIdx.x, + kThreads, .. of [v0, v1), kUnroll
// loads at a time
template <class F>
__device__ __forceinline__ void for_slice(const float* x, int v0, int v1, F&& f) {
  for (int v = v0 + (int)threadIdx.x; v < v1; v += kThreads * kUnroll) {
    float l[kUnroll];
#pragma unroll
    for (int i = 0; i < kUnroll; i++) l[i] = v + i * kThreads < v1 ? x[v + i * kThreads] : 0.f;
#pragma unroll
    for (int i = 0; i < kUnroll; i++)
      if (v + i * kThreads < v1) f(v + i * kThreads, l[i]);
  }
}

// Sum over the threads after this one, of one value each (kThreads of them), and over all in `total`.
__device__ __forceinline__ unsigned long long block_sum_after(unsigned long long v, unsigned long long& total) {
  __shared__ unsigned long long ws[kWaves];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  unsigned long long incl = v;  // this lane's and the later ones'
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long x = __shfl_down(incl, o);
    if (lane + o < 64) incl += x;
  }
  __syncthreads();
  if (lane == 0) ws[wave] = incl;
  __syncthreads();
  unsigned long long after = incl - v;
  total = 0;
  for (int q = 0; q < kWaves; q++) {
    total += ws[q];
    if (q > wave) after += ws[q];
  }
  return after;
}

// Bin of a score, larger for larger scores.  Key bins: the key's top bits.  LINEAR: the steps of max - s,
// counted down from the top bin, 0 from 32 below the maximum on (whose mass rounds to 0), and for a NaN
// difference.  Scaling by powers of two is exact, so a finer bin lies in one first one.
// Level 0: the first 2048 bins, 1: the 2048 in each of those (22 bits).
template <bool LINEAR>
__device__ __forceinline__ uint32_t level_bin(float s, uint32_t key, float mx, int level) {
  uint32_t b = key >> (kFirstShift - kFinerBits);
  if (LINEAR) {
    const float d = (mx - s) * (kStepsPerUnit * kSampleBins);
    b = d < (float)(kSampleBins - 1) * kSampleBins ? kSampleBins * kSampleBins - 1 - (uint32_t)(int)fmaxf(d, 0.f) : 0u;
  }
  return level ? b : b >> kFinerBits;
}

// The last workgroup's end of a histogram pass.  Suffix sums: a thread holds bins 8t..8t+7.  The bin is the
// largest d >= 1 whose sum above + S[d] reaches what is sought, else 0 (S does not increase with d, so d is
// the count of such d); sought(total) says what.  Clears the histogram, and calls f(d, S[d + 1], h[d], sought)
// in one thread.
template <class P, class F>
__device__ __forceinline__ void select_bin(unsigned long long* hist, unsigned long long above, P&& sought_of, F&& f) {
  __shared__ unsigned int ndig;
  const int t = threadIdx.x;
  if (t == 0) ndig = 0;
  unsigned long long h[8], own = 0, total;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    h[i] = load_u64(&hist[8 * t + i]);
    own += h[i];
  }
  const unsigned long long after = block_sum_after(own, total), sought = sought_of(total);
  unsigned long long run = after, over[8];
  unsigned int n = 0;
#pragma unroll
  for (int i = 7; i >= 0; i--) {
    over[i] = run;  // S[8t + i + 1]
    run += h[i];
    n += (8 * t + i >= 1 && above + run >= sought) ? 1u : 0u;
    hist[8 * t + i] = 0;  // ready for the next pass
  }
  if (n) atomicAdd(&ndig, n);
  __syncthreads();
  const int d = (int)ndig;
  if (d >> 3 == t) {
    unsigned long long ov = 0, hd = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      ov = (d & 7) == i ? over[i] : ov;
      hd = (d & 7) == i ? h[i] : hd;
    }
    f(d, ov, hd, sought);
  }
}

// MASS: the masses of the whole row over linear bins (top-p alone); else counts over key bins (top-k).
// Leaves the threshold's bin in w->prefix, the rank still sought in it (top-k) or the mass above it
// (top-p) in w->need, the mass sought in w->target, and in w->finer whether k_finer is to cut the bin.
template <bool MASS>
__global__ void __launch_bounds__(kThreads) k_first(Args a) {
  typedef typename std::conditional<MASS, unsigned long long, unsigned int>::type bin_t;
  __shared__ bin_t wh[kSampleBins];
  Block b;
  if (!setup(a, b)) return;
  SampleWork* w = b.w;
  const float T = a.sp.temperature, mx = MASS ? row_max(a, b) : 0.f;
#pragma unroll
  for (int i = 0; i < 8; i++) wh[threadIdx.x + kThreads * i] = 0;
  __syncthreads();
  for_slice(b.x, b.v0, b.v1, [&](int, float l) {
    const float s = __fdiv_rn(l, T);
    const bin_t m = MASS ? (bin_t)mass_of(s, mx) : (bin_t)1;
    if (!MASS || m) atomicAdd(&wh[level_bin<MASS>(s, key32(s), mx, 0)], m);
  });
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const unsigned long long h = wh[threadIdx.x + kThreads * i];
    if (h) atomicAdd(&b.ls->hist[threadIdx.x + kThreads * i], h);
  }
  if (!last_block(w)) return;
  select_bin(
      b.ls->hist, 0,
      [&](unsigned long long total) {
        if (!MASS) return (unsigned long long)a.sp.top_k;
        const unsigned long long p = (unsigned long long)((double)a.sp.top_p * (double)total);
        return p < 1 ? 1ull : p;
      },
      [&](int d, unsigned long long over, unsigned long long h, unsigned long long sought) {
        w->prefix = (unsigned int)d;
        w->need = MASS ? over : sought - over;
        w->target = sought;
        // scores in the bin: its count; for a mass at most that over the smallest one's
        const unsigned long long least = MASS ? mass_of(-(float)(kSampleBins - d) / kStepsPerUnit, 0.f) : 1ull;
        w->finer = (MASS && (d == 0 || least == 0)) || h > kFinerAbove * least;
        w->ticket = 0;
      });
}

// The threshold's bin among the 2048 finer ones within k_first's, as k_first (if that asked for it).
template <bool MASS>
__global__ void __launch_bounds__(kThreads) k_finer(Args a) {
  typedef typename std::conditional<MASS, unsigned long long, unsigned int>::type bin_t;
  __shared__ bin_t wh[kSampleBins];
  if (load_u32(&a.work[blockIdx.y].finer) == 0) return;
  Block b;
  if (!setup(a, b)) return;
  SampleWork* w = b.w;
  const float T = a.sp.temperature, mx = MASS ? row_max(a, b) : 0.f;
  const uint32_t fd = load_u32(&w->prefix);
#pragma unroll
  for (int i = 0; i < 8; i++) wh[threadIdx.x + kThreads * i] = 0;
  __syncthreads();
  for_slice(b.x, b.v0, b.v1, [&](int, float l) {
    const float s = __fdiv_rn(l, T);
    const uint32_t bin = level_bin<MASS>(s, key32(s), mx, 1);
    if (bin >> kFinerBits == fd) atomicAdd(&wh[bin & (kSampleBins - 1)], MASS ? (bin_t)mass_of(s, mx) : (bin_t)1);
  });
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const unsigned long long h = wh[threadIdx.x + kThreads * i];
    if (h) atomicAdd(&b.ls->hist[threadIdx.x + kThreads * i], h);
  }
  if (!last_block(w)) return;
  const unsigned long long need = load_u64(&w->need), target = load_u64(&w->target);
  __syncthreads();  // read by every thread before one of them writes them
  select_bin(
      b.ls->hist, MASS ? need : 0, [&](unsigned long long) { return MASS ? target : need; },
      [&](int d, unsigned long long over, unsigned long long, unsigned long long) {
        w->prefix = fd << kFinerBits | (unsigned int)d;
        w->need = MASS ? need + over : need - over;
        w->ticket = 0;
      });
}

// Whole draw of a filtered call (after k_first and k_finer): TOPK, TOPP the filters that are on.
template <bool TOPK, bool TOPP>
__global__ void __launch_bounds__(kThreads) k_finish(Args a) {
  constexpr bool LINEAR = !TOPK, BOTH = TOPK && TOPP;
  // tokens above the bin and in it: this workgroup's, then, in the row's last one, the row's, with their keys
  __shared__ uint32_t tk[2][kSampleCand], ck[2 * kSampleCand];
  __shared__ unsigned long long hs[128];
  __shared__ unsigned int nlocal[2], base[2], digit;
  __shared__ unsigned long long s_above;
  Block b;
  if (!setup(a, b)) return;
  SampleWork* w = b.w;
  const float T = a.sp.temperature;
  const uint32_t fd = load_u32(&w->prefix);
  const int level = load_u32(&w->finer) ? 1 : 0;
  float mx = LINEAR ? row_max(a, b) : 0.f;
  const uint64_t dbase = draw_base(a.sp.seed, b.counter);
  if (threadIdx.x < 2) nlocal[threadIdx.x] = 0;
  __syncthreads();
  // best: draws of the scores that stay for certain; tied: of the bin's, which stay or go as one if their
  // keys are the same
  unsigned long long best = 0, tied = 0;
  uint32_t kmn = 0xffffffffu, kmx = 0, amx = 0;
  auto draw = [&](int v, float s) {
    return ((unsigned long long)gumbel_key_score(s, dbase, v) << 32) | (0xffffffffu - (uint32_t)v);
  };
  for_slice(b.x, b.v0, b.v1, [&](int v, float l) {
    const float s = __fdiv_rn(l, T);
    const uint32_t k = key32(s), bin = level_bin<LINEAR>(s, k, mx, level);
    if (bin < fd) return;
    const int in = bin == fd;
    if (!BOTH || in) {
      const unsigned long long g = draw(v, s);
      if (in) tied = g > tied ? g : tied;
      else best = g > best ? g : best;
    }
    if (in) {
      kmn = k < kmn ? k : kmn;
      kmx = k > kmx ? k : kmx;
    } else {
      amx = k > amx ? k : amx;
      if (!BOTH) return;
    }
    const unsigned int i = atomicAdd(&nlocal[in], 1u);
    if (i < (unsigned)kSampleCand) tk[in][i] = (uint32_t)v;
  });
  __syncthreads();
  if (threadIdx.x < 2 && nlocal[threadIdx.x])
    base[threadIdx.x] = atomicAdd(threadIdx.x ? &w->nbin : &w->nabove, nlocal[threadIdx.x]);
  auto mx64 = [](unsigned long long p, unsigned long long q) { return p > q ? p : q; };
  best = block_reduce_u64(best, mx64);
  __syncthreads();
  tied = block_reduce_u64(tied, mx64);
  __syncthreads();
  const unsigned long long ends = block_reduce_u64(((unsigned long long)(~kmn) << 32), mx64);
  __syncthreads();
  kmx = (uint32_t)block_reduce_u64((unsigned long long)kmx, mx64);
  if (BOTH) {
    __syncthreads();
    amx = (uint32_t)block_reduce_u64((unsigned long long)amx, mx64);
  }
  for (int q = 0; q < 2; q++) {
    uint32_t* const list = q ? b.ls->bin : b.ls->above;
    const unsigned int n = min(nlocal[q], (unsigned)kSampleCand);
    for (unsigned int i = threadIdx.x; i < n; i += kThreads)
      if (base[q] + i < (unsigned)kSampleCand)
        __hip_atomic_store(&list[base[q] + i], tk[q][i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (threadIdx.x == 0) {
    if (best) atomicMax(&w->best, best);
    if (BOTH && nlocal[0]) atomicMax(&w->abovemax, amx);
    if (nlocal[1]) {
      atomicMax(&w->tied, tied);
      atomicMax(&w->binmin, (unsigned int)(ends >> 32));
      atomicMax(&w->binmax, kmx);
    }
  }
  if (!last_block(w)) return;

  // ---- the row's last workgroup
  const unsigned int na = BOTH ? load_u32(&w->nabove) : 0u, nb = load_u32(&w->nbin);  // na < top_k <= kSampleCand
  const uint32_t bmin = ~load_u32(&w->binmin), bmax = load_u32(&w->binmax);
  const bool same = bmin == bmax, listed = nb <= (unsigned)kSampleCand;  // one score, however often; all in the list
  best = load_u64(&w->best);
  tied = load_u64(&w->tied);
  if (same && !BOTH) {  // the threshold is that score: it stays
    best = tied > best ? tied : best;
  } else {
    // the listed scores: those above the bin, then its own
    uint32_t* const rtk = &tk[0][0];
    const unsigned int nl = na + (listed && !same ? nb : 0u);
    for (unsigned int i = threadIdx.x; i < nl; i += kThreads) {
      const uint32_t v = load_u32(i < na ? &b.ls->above[i] : &b.ls->bin[i - na]);
      rtk[i] = v;
      ck[i] = key32(__fdiv_rn(b.x[v], T));
    }
    __syncthreads();
    // f(key, how many, token or -1) for the scores of the bin, or also for those above it (the list from 0)
    auto each = [&](bool all, auto&& f) {
      for (unsigned int i = threadIdx.x + (all ? 0u : na); i < nl; i += kThreads) f(ck[i], 1u, (int)rtk[i]);
      if (same) {
        if (threadIdx.x == 0) f(bmin, nb, -1);
      } else if (!listed) {
        for_slice(b.x, 0, a.V, [&](int v, float l) {
          const float s = __fdiv_rn(l, T);
          const uint32_t k = key32(s);
          if (level_bin<LINEAR>(s, k, mx, level) == fd) f(k, 1u, v);
        });
      }
    };
    // the largest key with (a sum above +) the sum over the bin's scores, or all, of keys >= it reaching
    // `sought`, among the keys from kmin to kmax: 7 bits at a time of those in which the two differ
    auto descend = [&](bool mass, bool all, uint32_t kmin, uint32_t kmax, unsigned long long above,
                       unsigned long long sought) {
      int hi = kmin == kmax ? 0 : 32 - __clz((int)(kmin ^ kmax));
      uint32_t mask = hi == 32 ? 0u : ~0u << hi, prefix = kmax & mask;
      while (hi > 0) {
        const int wd = hi < 7 ? hi : 7, sh = hi - wd;
        const uint32_t dm = (1u << wd) - 1u;
        for (int i = threadIdx.x; i < 128; i += kThreads) hs[i] = 0;
        __syncthreads();
        auto count = [&](uint32_t k, unsigned int n, int) {
          if ((k & mask) == prefix && k >= kmin)
            atomicAdd(&hs[(k >> sh) & dm], mass ? mass_of(from_key32(k), mx) * n : (unsigned long long)n);
        };
        each(all, count);
        __syncthreads();
        if (threadIdx.x < 64) {  // bins 2l, 2l + 1 per lane; suffix sums, then the digit
          const int lane = threadIdx.x;
          const unsigned long long h0 = hs[2 * lane], h1 = hs[2 * lane + 1];
          unsigned long long incl = h0 + h1;
          for (int o = 1; o < 64; o <<= 1) {
            const unsigned long long x = __shfl_down(incl, o);
            if (lane + o < 64) incl += x;
          }
          const unsigned long long s0 = above + incl, s1 = above + incl - h0;
          const unsigned int d = (unsigned)__popcll(__ballot(lane > 0 && s0 >= sought)) +
                                 (unsigned)__popcll(__ballot(s1 >= sought));
          if ((int)(d >> 1) == lane) {
            digit = d;
            s_above = (d & 1) ? s1 - h1 : s0 - h0;
          }
        }
        __syncthreads();
        prefix |= digit << sh;
        mask |= dm << sh;
        above = s_above;
        hi = sh;
        __syncthreads();
      }
      return prefix;
    };
    uint32_t keep = 0;
    if (TOPK) {
      // the rank still sought in the bin: it counts from the bin's top
      keep = descend(false, false, bmin, bmax, 0, load_u64(&w->need));
      if (BOTH) {
        const uint32_t kmax = na ? load_u32(&w->abovemax) : bmax;
        mx = from_key32(kmax);
        unsigned long long z = 0;
        each(true, [&](uint32_t k, unsigned int n, int) {
          if (k >= keep) z += mass_of(from_key32(k), mx) * n;
        });
        z = block_reduce_u64(z, [](unsigned long long p, unsigned long long q) { return p + q; });
        unsigned long long target = (unsigned long long)((double)a.sp.top_p * (double)z);
        if (target < 1) target = 1;
        const uint32_t pmin = descend(true, true, keep, kmax, 0, target);
        keep = pmin > keep ? pmin : keep;
      }
    } else {
      keep = descend(true, false, bmin, bmax, load_u64(&w->need), load_u64(&w->target));
    }
    unsigned long long g = 0;
    each(true, [&](uint32_t k, unsigned int, int v) {
      if (k < keep) return;
      const unsigned long long q = v < 0 ? tied : draw(v, from_key32(k));
      g = q > g ? q : g;
    });
    __syncthreads();
    g = block_reduce_u64(g, mx64);
    best = g > best ? g : best;
  }
  // the bin's list lies where the next call's histogram does
  for (unsigned int i = threadIdx.x; i < min(nb, (unsigned)kSampleCand); i += kThreads) b.ls->bin[i] = 0;
  __syncthreads();  // every wave has read the work that put_token clears
  if (threadIdx.x == 0) put_token(a, b, (int)(0xffffffffu - (uint32_t)best));
}

// The draw (GREEDY: the first index of the maximum logit); the last workgroup
// writes the token and clears the row's work for the next call.
template <bool GREEDY>
__global__ void __launch_bounds__(kThreads) k_draw(Args a) {
  Block b;
  if (!setup(a, b)) return;
  SampleWork* w = b.w;
  const float T = a.sp.temperature;
  const uint32_t kmin = load_u32(&w->kmin), pmin = load_u32(&w->pmin);
  const uint32_t keep = kmin > pmin ? kmin : pmin;
  const uint64_t base = GREEDY ? 0 : draw_base(a.sp.seed, b.counter);
  unsigned long long best = 0;
  for (int v = b.v0 + threadIdx.x; v < b.v1; v += kThreads) {
    uint32_t k;
    if (GREEDY) {
      k = key32(b.x[v]);
    } else {
      if (key32(__fdiv_rn(b.x[v], T)) < keep) continue;
      k = gumbel_key(b.x[v], T, base, v);
    }
    const unsigned long long key = ((unsigned long long)k << 32) | (0xffffffffu - (uint32_t)v);
    best = key > best ? key : best;
  }
  best = block_reduce_u64(best, [](unsigned long long p, unsigned long long q) { return p > q ? p : q; });
  if (threadIdx.x == 0) atomicMax(&w->best, best);
  if (!last_block(w)) return;
  if (threadIdx.x == 0) put_token(a, b, (int)(0xffffffffu - (uint32_t)load_u64(&w->best)));
}

// Workgroups per row: about 128 workgroups in all, at least 8 per row.
int groups_for(int rows) {
  int g = 128;
  while (g > 8 && g * rows > 128) g >>= 1;
  return g;
}

// Draws that take the two-launch form
bool two_launches(const SampleParams& sp, int V) {
  const bool topk = sp.top_k > 0 && sp.top_k < V, topp = sp.top_p > 0.f && sp.top_p < 1.f;
  return sp.temperature > 0.f && (topk || topp) && !(topk && sp.top_k > kFinishTopK);
}

int launch(const Args& a, int rows, hipStream_t stream) {
  const dim3 grid(groups_for(rows), rows), block(kThreads);
  const SampleParams& sp = a.sp;
  if (!(sp.temperature > 0.f)) {
    hipLaunchKernelGGL(k_draw<true>, grid, block, 0, stream, a);
  } else {
    const bool topk = sp.top_k > 0 && sp.top_k < a.V;
    const bool topp = sp.top_p > 0.f && sp.top_p < 1.f;
    if (topp && !a.st && (!topk || sp.top_k > kFinishTopK)) hipLaunchKernelGGL(k_max, grid, block, 0, stream, a);
    if (two_launches(sp, a.V)) {
      if (topk) {
        hipLaunchKernelGGL(k_first<false>, grid, block, 0, stream, a);
        hipLaunchKernelGGL(k_finer<false>, grid, block, 0, stream, a);
      } else {
        hipLaunchKernelGGL(k_first<true>, grid, block, 0, stream, a);
        hipLaunchKernelGGL(k_finer<true>, grid, block, 0, stream, a);
      }
      if (topk && topp) hipLaunchKernelGGL((k_finish<true, true>), grid, block, 0, stream, a);
      else if (topk) hipLaunchKernelGGL((k_finish<true, false>), grid, block, 0, stream, a);
      else hipLaunchKernelGGL((k_finish<false, true>), grid, block, 0, stream, a);
      return hipGetLastError() == hipSuccess ? QMK_OK : QMK_ERR_HIP;
    }
    if (topk)
      for (int p = 0; p < sample::kPasses; p++) hipLaunchKernelGGL(k_hist<false>, grid, block, 0, stream, a, p);
    if (topp)
      for (int p = 0; p < sample::kPasses; p++) hipLaunchKernelGGL(k_hist<true>, grid, block, 0, stream, a, p);
    hipLaunchKernelGGL(k_draw<false>, grid, block, 0, stream, a);
  }
  return hipGetLastError() == hipSuccess ? QMK_OK : QMK_ERR_HIP;
}

// Work of qmk_sample_rows per (device, stream), kSampleRowsMax rows, kept until
// the process ends: calls on one stream are ordered, so they may share it;
// calls on different streams may overlap, so they do not.
std::mutex g_mu;
std::map<std::pair<int, hipStream_t>, SampleWork*> g_work;

int stream_work(hipStream_t stream, SampleWork** out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return QMK_ERR_HIP;
  std::lock_guard<std::mutex> lk(g_mu);
  auto it = g_work.find({dev, stream});
  if (it == g_work.end()) {
    SampleWork* w = nullptr;
    if (alloc_sample_work(&w, kSampleRowsMax) != QMK_OK) return QMK_ERR_HIP;
    it = g_work.emplace(std::make_pair(dev, stream), w).first;
  }
  *out = it->second;
  return QMK_OK;
}

}  // namespace sample

int alloc_sample_work(SampleWork** out, int rows) {
  static_assert(sizeof(SampleWork) % alignof(SampleLists) == 0, "the lists follow the rows' work");
  const size_t bytes = (size_t)rows * sizeof(SampleWork) + (size_t)std::min(rows, kSampleListRows) * sizeof(SampleLists);
  if (hipMalloc(out, bytes) != hipSuccess) return QMK_ERR_HIP;
  // the fill runs on the null stream: wait for it, since the caller's stream need not
  if (hipMemset(*out, 0, bytes) != hipSuccess || hipStreamSynchronize(nullptr) != hipSuccess) {
    (void)hipFree(*out);
    *out = nullptr;
    return QMK_ERR_HIP;
  }
  return QMK_OK;
}

int launch_sample_state(const float* logits, int vocab, const SampleParams& sp, DecodeState* st, int* log,
                        SampleWork* work, hipStream_t stream) {
  sample::Args a{logits, vocab, sp, nullptr, nullptr, st, log, work, sample_lists(work, 1)};
  return sample::launch(a, 1, stream);
}

}  // namespace qmk

using namespace qmk;

extern "C" int qmk_sample_rows(const float* logits, int rows, int vocab, float temperature, int top_k, float top_p,
                               unsigned long long seed, const long long* counters, int* out_tokens,
                               hipStream_t stream) {
  if (!logits || !counters || !out_tokens || rows < 1 || rows > 65535 || vocab < 1) return QMK_ERR_ARG;
  if (!(top_p == top_p) || !(temperature == temperature)) return QMK_ERR_ARG;  // NaN
  const SampleParams sp{temperature, top_k, top_p, (uint64_t)seed};
  SampleWork* work = nullptr;
  int s = sample::stream_work(stream, &work);
  if (s != QMK_OK) return s;
  const int most = sample::two_launches(sp, vocab) ? kSampleListRows : kSampleRowsMax;
  for (int r0 = 0; r0 < rows && s == QMK_OK; r0 += most) {
    const int n = std::min(rows - r0, most);
    sample::Args a{logits + (size_t)r0 * vocab, vocab, sp, counters + r0, out_tokens + r0, nullptr, nullptr, work,
                   sample_lists(work, kSampleRowsMax)};
    s = sample::launch(a, n, stream);
  }
  return s;
}

// Token sampling on the device: top-k or top-p over one row of fp32 logits,
// so that sampled generation hands the next token to the next decode step
// without the logits leaving device memory.  The candidate set and its
// probabilities are those of the host samplers (largest logits first, ties
// toward the lower token id; softmax over the kept logits); the draw uses a
// counter-based generator, one uniform number per (seed, counter).
//
// One workgroup of 1024 threads.  A row is 128 KB at 32000 tokens, which one
// compute unit reads in ~1 us; what a draw spends beyond that are dependent
// steps, so there are few of them:
//   1. every logit becomes a 32-bit key of the same order; a thread keeps its
//      logits in registers (vocabularies of up to 32768) and the largest;
//   2. one wave raises a bound, bit by bit, as long as `keep` of the 1024 thread
//      maxima stay above it: at least `keep` logits do then;
//   3. the logits above the bound (little more than `keep` of them) are gathered
//      and ranked by counting, ties toward the lower id;
//   4. one wave walks the candidates in order: the softmax, for top-p the prefix
//      whose mass reaches p, and the draw.  The sums run in candidate order, as in
//      the host samplers.
// Top-p looks at the 64 most likely tokens first, which hold the mass wherever a
// model is sure of anything.  More than 256 candidates, or more than 1024 logits
// above the bound (many equal ones), take the general way: radix selection of the
// k-th largest 64-bit key (eight passes of one byte with a histogram in LDS) and a
// bitonic sort.  Measured over 32000 logits, us per launch, before (radix selection for
// all) and now: k = 1 90 / 10, k = 40 95 / 14, k = 256 113 / 30, top-p 0.9 of a row with
// one likely token 105 / 17, of a flat row (general way) 297 / 225, k = 1000 211 / 150.
#include "../../include/vkl_hip.h"
#include "vkl_common.h"

namespace
{
constexpr int kSampThreads = 1024;
constexpr int kMaxCand = 1024;

__device__ __forceinline__ uint64_t
logit_key (float v, uint32_t id)
{
  const uint32_t b = __float_as_uint (v);
  const uint32_t u = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
  return ((uint64_t)u << 32) | (uint64_t)(0xffffffffu - id);
}

__device__ __forceinline__ float
key_logit (uint64_t key)
{
  const uint32_t u = (uint32_t)(key >> 32);
  const uint32_t b = (u & 0x80000000u) ? (u & 0x7fffffffu) : ~u;
  return __uint_as_float (b);
}

// splitmix64 of (seed, counter) -> uniform in [0, 1) with 24 bits
__device__ __forceinline__ float
uniform01 (uint64_t seed, uint32_t counter)
{
  uint64_t z = seed + 0x9E3779B97F4A7C15ull * ((uint64_t)counter + 1);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (float)(z >> 40) * (1.0f / 16777216.0f);
}

struct SampleArgs
{
  const float *logits;
  int V, k;     // k: candidates kept by rank (top-p: the cap, kMaxCand)
  float p;      // < 0: top-k; else top-p
  uint64_t seed;
  uint32_t counter;
  const uint32_t *counter_dev; // if set, added to counter (e.g. a position kept on the device)
  uint32_t *tok;
  uint32_t *cand_ids; // optional: candidates of this draw, most likely first
  float *cand_probs;
  uint32_t *cand_n;
  // a step of a replayed decode loop (all three set): k, p and the seed come
  // from `dev` = {k, bits of p, seed low, seed high} in device memory, so that
  // one captured launch serves every request; loop = {index into ids,
  // position}; the token of position + 1 goes to ids[index + 1], drawn with
  // that position as the counter, and both loop words advance
  const uint32_t *dev;
  uint32_t *loop;
  uint32_t *ids;
};

constexpr int kRegs = 32;      // logits of a thread in registers
constexpr int kFewCand = 256;  // candidates ranked by counting
constexpr int kFirstTopP = 64; // candidates top-p looks at first

__device__ __forceinline__ uint32_t
ordered (float v)
{
  const uint32_t b = __float_as_uint (v);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

struct SampleShared
{
  uint64_t cand[kMaxCand]; // keys of the candidates, in the end sorted
  uint64_t found[kMaxCand];
  uint32_t hist[256];
  uint32_t maxima[kSampThreads];
  float red[kSampThreads];
  uint64_t prefix;
  uint32_t need, count, bound;
  float total;
  int short_of_mass;
};

// the row: f (logit, id) for every logit of this thread, ids tid + 1024 j
template <bool REGS> struct Row
{
  float v[REGS ? kRegs : 1];
  const float *logits;
  int V;

  __device__ __forceinline__ void
  load (const float *l, int n)
  {
    logits = l, V = n;
    if (REGS)
#pragma unroll
      for (int j = 0; j < kRegs; ++j)
        v[REGS ? j : 0] = vkl::ldg (l + min ((int)threadIdx.x + j * kSampThreads, n - 1));
  }
  template <class F>
  __device__ __forceinline__ void
  each (F f) const
  {
    if (REGS)
      {
        // (copies of its own: the 32 masks and keys of one walk are not kept for the next)
        int n = V;
        asm volatile ("" : "+s"(n));
#pragma unroll
        for (int j = 0; j < kRegs; ++j)
          {
            float x = v[REGS ? j : 0];
            asm volatile ("" : "+v"(x));
            if ((int)threadIdx.x + j * kSampThreads < n)
              f (x, (uint32_t)(threadIdx.x + j * kSampThreads));
          }
      }
    else
      for (int i = threadIdx.x; i < V; i += kSampThreads)
        f (vkl::ldg (logits + i), (uint32_t)i);
  }
};

// The `keep` (<= kFewCand) largest keys in order into sh.cand; false if too many
// logits lie above the bound (nothing is written then)
template <bool REGS>
__device__ bool
select_few (const Row<REGS> &row, int keep, SampleShared &sh)
{
  const int tid = threadIdx.x, lane = tid & 63;
  uint32_t big = 0; // below every real key, or equal to the lowest NaN's
  row.each ([&] (float x, uint32_t) { big = max (big, ordered (x)); });
  sh.maxima[tid] = big;
  if (tid == 0)
    sh.count = 0;
  __syncthreads ();
  if (tid < 64)
    {
      uint32_t m[kSampThreads / 64];
#pragma unroll
      for (int j = 0; j < kSampThreads / 64; ++j)
        m[j] = sh.maxima[64 * j + lane];
      // enough above the bound always; a few more than needed cost less than the
      // bits that would take them out
      const int enough = max (2 * keep, 96);
      uint32_t bound = 0;
      for (int bit = 31, above = kSampThreads; bit >= 0 && above > enough; --bit)
        {
          const uint32_t next = bound | (1u << bit);
          int n = 0;
#pragma unroll
          for (int j = 0; j < kSampThreads / 64; ++j)
            n += __popcll (__builtin_amdgcn_ballot_w64 (m[j] >= next));
          if (n >= keep)
            bound = next, above = n;
        }
      if (lane == 0)
        sh.bound = bound;
    }
  __syncthreads ();
  const uint32_t bound = sh.bound;
  row.each ([&] (float x, uint32_t id) {
    if (ordered (x) >= bound)
      {
        const uint32_t slot = atomicAdd (&sh.count, 1u);
        if (slot < (uint32_t)kMaxCand)
          sh.found[slot] = logit_key (x, id);
      }
  });
  __syncthreads ();
  const int n = (int)sh.count;
  if (n > kMaxCand)
    return false;
  // all keys differ: a key's rank is the number of larger ones
  if (tid < n)
    {
      const uint64_t mine = sh.found[tid];
      int rank = 0;
      for (int i = 0; i < n; ++i)
        rank += sh.found[i] > mine;
      if (rank < keep)
        sh.cand[rank] = mine;
    }
  __syncthreads ();
  return true;
}

// the same for any keep up to kMaxCand and any logits
__device__ void
select_radix (const Row<false> &row, int keep, SampleShared &sh)
{
  const int tid = threadIdx.x;
  __syncthreads ();
  // ---- the keep-th largest key ----------------------------------------------
  if (tid == 0)
    sh.prefix = 0, sh.need = (uint32_t)keep, sh.count = 0;
  for (int pass = 7; pass >= 0; --pass)
    {
      if (tid < 256)
        sh.hist[tid] = 0;
      __syncthreads ();
      const uint64_t prefix = sh.prefix;
      const int shift = 8 * pass;
      row.each ([&] (float x, uint32_t id) {
        const uint64_t key = logit_key (x, id);
        // keys that agree with the prefix in all bytes above this one
        if (pass == 7 || (key >> (shift + 8)) == (prefix >> (shift + 8)))
          atomicAdd (&sh.hist[(uint32_t)(key >> shift) & 255u], 1u);
      });
      __syncthreads ();
      if (tid == 0)
        {
          uint32_t need = sh.need, cum = 0;
          int bin = 255;
          for (; bin > 0; --bin)
            {
              if (cum + sh.hist[bin] >= need)
                break;
              cum += sh.hist[bin];
            }
          sh.need = need - cum;
          sh.prefix = prefix | ((uint64_t)bin << shift);
        }
      __syncthreads ();
    }
  const uint64_t kth = sh.prefix;

  // ---- gather and sort the candidates ------------------------------------------
  int P = 1;
  while (P < keep)
    P <<= 1;
  for (int i = tid; i < P; i += kSampThreads)
    sh.cand[i] = 0;
  __syncthreads ();
  row.each ([&] (float x, uint32_t id) {
    const uint64_t key = logit_key (x, id);
    if (key >= kth)
      {
        const uint32_t slot = atomicAdd (&sh.count, 1u);
        if (slot < (uint32_t)kMaxCand)
          sh.cand[slot] = key;
      }
  });
  __syncthreads ();
  // bitonic sort, descending, over P slots (unused slots hold key 0, below
  // every real key)
  for (int size = 2; size <= P; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1)
      {
        for (int i = tid; i < P; i += kSampThreads)
          {
            const int j = i ^ stride;
            if (j > i)
              {
                const uint64_t x = sh.cand[i], y = sh.cand[j];
                const bool desc = (i & size) == 0;
                if (desc ? x < y : x > y)
                  sh.cand[i] = y, sh.cand[j] = x;
              }
          }
        __syncthreads ();
      }
}

// value i of a wave, where every lane has one
__device__ __forceinline__ float
lane_value (float x, int i)
{
  return __int_as_float (__builtin_amdgcn_readlane (__float_as_int (x), i));
}

// exp (logit - top) of candidate i
__device__ __forceinline__ float
weight (const SampleShared &sh, int i, float top)
{
  return expf (key_logit (sh.cand[i]) - top);
}

template <bool REGS>
__global__ __launch_bounds__ (kSampThreads) void
sample_kernel (const SampleArgs args)
{
  SampleArgs a = args;
  if (a.dev)
    {
      a.p = __uint_as_float (vkl::ldg (a.dev + 1));
      const int k = (int)vkl::ldg (a.dev);
      a.k = a.p >= 0.f ? kMaxCand : (k > kMaxCand ? kMaxCand : max (k, 1));
      a.seed = (uint64_t)vkl::ldg (a.dev + 2) | ((uint64_t)vkl::ldg (a.dev + 3) << 32);
    }
  __shared__ SampleShared sh;
  const int tid = threadIdx.x, lane = tid & 63;
  const int most = min (min (a.k, kMaxCand), a.V);
  Row<REGS> row;
  row.load (a.logits, a.V);

  int keep = a.p >= 0.f ? min (kFirstTopP, most) : most;
  int n = 0;
  float top = 0.f;
  for (;;)
    {
      if (keep > kFewCand || !select_few (row, keep, sh))
        select_radix (Row<false>{ {}, a.logits, a.V }, keep, sh);
      top = key_logit (sh.cand[0]);
      n = keep;
      if (a.p < 0.f)
        break;
      // mass of the whole vocabulary relative to the top logit
      float part = 0.f;
      row.each ([&] (float x, uint32_t) { part += expf (x - top); });
      sh.red[tid] = part;
      __syncthreads ();
      for (int s = kSampThreads / 2; s >= 64; s >>= 1)
        {
          if (tid < s)
            sh.red[tid] += sh.red[tid + s];
          __syncthreads ();
        }
      if (tid < 64)
        {
          // the last six steps of that sum, lane i with lane i + s
          float sum = sh.red[lane];
          for (int s = 32; s > 0; s >>= 1)
            sum += __shfl_down (sum, s, 64);
          const float total = lane_value (sum, 0);
          // tokens are added while the mass so far is below p
          float mass = 0.f;
          n = 0;
          for (int c = 0; c < keep && mass < a.p; c += 64)
            {
              const float share = c + lane < keep ? weight (sh, c + lane, top) / total : 0.f;
              for (int i = 0; i < min (64, keep - c) && mass < a.p; ++i, ++n)
                mass += lane_value (share, i);
            }
          if (lane == 0)
            sh.short_of_mass = mass < a.p;
          n = max (n, 1);
        }
      __syncthreads ();
      if (keep == most || !sh.short_of_mass)
        break;
      keep = most;
    }
  if (tid >= 64)
    return;

  // ---- probabilities and the draw, in candidate order, by one wave -------------
  float sum = 0.f;
  for (int c = 0; c < n; c += 64)
    {
      const float e = c + lane < n ? weight (sh, c + lane, top) : 0.f;
      for (int i = 0; i < min (64, n - c); ++i)
        sum += lane_value (e, i);
    }
  uint32_t ctr = a.counter + (a.counter_dev ? vkl::ldg (a.counter_dev) : 0u);
  uint32_t index = 0, position = 0;
  if (a.loop)
    {
      index = vkl::ldg (a.loop), position = vkl::ldg (a.loop + 1);
      ctr = a.counter + position + 1u;
    }
  const float target = uniform01 (a.seed, ctr);
  float cum = 0.f;
  int pick = -1;
  for (int c = 0; c < n && (pick < 0 || a.cand_probs || a.cand_ids); c += 64)
    {
      const float pr = c + lane < n ? weight (sh, c + lane, top) / sum : 0.f;
      if (c + lane < n && a.cand_probs)
        a.cand_probs[c + lane] = pr;
      if (c + lane < n && a.cand_ids)
        a.cand_ids[c + lane] = 0xffffffffu - (uint32_t)sh.cand[c + lane];
      for (int i = 0; i < min (64, n - c) && pick < 0; ++i)
        {
          cum += lane_value (pr, i);
          if (cum > target)
            pick = c + i;
        }
    }
  if (pick < 0) // rounding left the total a hair below the target
    pick = n - 1;
  if (lane != 0)
    return;
  if (a.cand_n)
    *a.cand_n = (uint32_t)n;
  const uint32_t drawn = 0xffffffffu - (uint32_t)sh.cand[pick];
  if (a.loop)
    {
      a.ids[index + 1] = drawn;
      a.loop[0] = index + 1u, a.loop[1] = position + 1u;
    }
  else
    *a.tok = drawn;
}

void
launch (const SampleArgs &a, hipStream_t s)
{
  if (a.V <= kRegs * kSampThreads)
    sample_kernel<true><<<dim3 (1), dim3 (kSampThreads), 0, s>>> (a);
  else
    sample_kernel<false><<<dim3 (1), dim3 (kSampThreads), 0, s>>> (a);
}
} // namespace

namespace vkl
{
// the draw of a replayed decode step (see SampleArgs::dev)
int
sample_loop_launch (const float *logits, int V, const uint32_t *dev_params, uint32_t *loop,
                    uint32_t *ids, hipStream_t s)
{
  SampleArgs a = {};
  a.logits = logits, a.V = V;
  a.k = 1, a.p = -1.f;
  a.dev = dev_params, a.loop = loop, a.ids = ids;
  launch (a, s);
  return 0;
}
}

extern "C" int
vkl_sample_f32 (const float *logits, int V, int k, float p, uint64_t seed,
                uint32_t counter, const uint32_t *counter_dev, uint32_t *tok,
                uint32_t *cand_ids, float *cand_probs, uint32_t *cand_n,
                void *stream)
{
  VKL_CHECK_ARG (logits && tok && V > 0);
  VKL_CHECK_ARG (p >= 0.f || k >= 1);
  VKL_CHECK_ARG (p < 0.f || p <= 1.0f);
  SampleArgs a = {};
  a.logits = logits, a.V = V;
  a.k = p >= 0.f ? kMaxCand : (k > kMaxCand ? kMaxCand : k);
  a.p = p, a.seed = seed, a.counter = counter, a.counter_dev = counter_dev;
  a.tok = tok, a.cand_ids = cand_ids, a.cand_probs = cand_probs, a.cand_n = cand_n;
  launch (a, (hipStream_t)stream);
  return vkl_launch_status ();
}

// The layers of the decode step as ONE launch, for narrow rows.
//
// What bounds such a layer is not its weights (3 MB at 512 values Q8_0) but the five
// hand-overs of a row from all workgroups to all.  vkl_decode_layer.hip hands over with
// results stored and acknowledged, an arrival at a counter, a flag, and then the row: four
// trips through memory, 3.8 us per phase at 512 values with its product.  Here a value travels
// with its tag in one word {tag, fp16} and a reader polls the row itself: two trips, one for
// the store and one for the load that finds it.  Nothing is ordered against anything else, no
// store is waited for and no cache has to be clean: polls and stores go past the L2.
// Us per layer at 512 values: 21.5 with a launch per layer, 14.4 in this form with a head on
// some of the row workgroups and weights requested a phase ahead, 12.6 as below, 11.6 with a
// workgroup's results as 32-byte stores (words of single waves: memory takes the partial
// lines one by one), 11.1 with k, q and v gathered too and one SiLU for a wave's three pairs,
// 9.9 with two rows of up to 512 bytes side by side in a wave.
//
// Rows: dim / 8 workgroups of eight waves, a wave owns row g of each of the square matrices
// (k, q, v, o, down) and two or three up/gate pairs, g its number among dim waves; all its
// weights of a layer are in its registers.  A row goes to eight copies, one for the
// workgroups of each XCD (any copy would do, they differ in who else reads them): a hand-over
// takes 1.1 us where 32 workgroups poll the same lines and 2.4 where 256 do.  Heads:
// n_heads workgroups more, which do nothing but the attention and hold the cached rows when k,
// q and v arrive.
//
// The memory path of a compute unit returns loads in order, so a poll returns behind all
// weights requested before it: as much as the registers hold is requested at the one point of
// the layer where the wait is longer than the way from memory, while the heads are computed.
//
// Two launches have to fit the GPU at once, as two launches per layer of narrow rows do (two
// models on two streams would each wait for workgroups that the other one keeps out): a
// workgroup takes one of two places of its compute unit, 128 registers (Q8_0 rows of more than
// 1024 values spill nine) and at most 80 KB of LDS.  Rows of more than 512 bytes therefore request the down projection's, of more than 1024
// the next layer's K/Q/V too, only when the up/gate product has left its registers.  With 256
// registers and all of it requested at the one point above it was no faster, us per token: 512
// wide Q8_0 97 / now 88, 1024 68 / 66, 1536 83 / 82, 768 wide fp16 87 / 82.
//
// The tags of a step follow on those of the step before (a counter in the sync area,
// advanced at the end of a launch), and every word of a row is written once per layer, of the
// last layer's row and of the arg-maxima once per launch (a model's launches are all of one
// form): what a row holds before is always an older tag, of 2^16.  A row is not overwritten while somebody still
// waits for it: the next layer's needs a row that all workgroups have contributed to since.
// Waits are bounded and a wait that gave up is reported as in the layer launch; its
// workgroup publishes nothing from then on.  vkl_decode_status clears counter and rows with
// the error word.
#include "vkl_decode_shared.h"
#include <algorithm>

namespace vkl
{
namespace dec
{
namespace
{
constexpr int kLsTags = 2048; // word of the layer-sync area: layers done so far, modulo 2^16 a tag
static_assert ((kLsTags + 32) * 4 <= kLayerSyncBytes, "layer-sync area too small");
constexpr int kSyncErr = 1;   // word of Scratch::sync: a wait gave up
constexpr int kTagSpinLimit = 1 << 14;
constexpr int kPairs = kTaggedPairs;
enum Stage { ST_KQV = 0, ST_ATT, ST_WO, ST_UP, ST_DOWN, ST_HEAD };

typedef __amdgpu_buffer_rsrc_t rsrc_t;

__device__ __forceinline__ rsrc_t
tagged_row (uint32_t *base, int words)
{
  return __builtin_amdgcn_make_buffer_rsrc (base, 0, words * 4, 0x00020000);
}

constexpr int kPastL2 = 17; // sc0 sc1

// Eight words from word `at` on, once all carry `tag` (in the upper half): their values.
// False: `limit` polls have not seen that.
__device__ __forceinline__ bool
poll8 (rsrc_t row, int at, uint32_t tag, int limit, uint4 &v)
{
  for (int spin = 0; spin < limit; ++spin)
    {
      asm volatile ("" ::: "memory"); // (each poll reads anew)
      const vkl_u32x4 a = __builtin_bit_cast (vkl_u32x4, __builtin_amdgcn_raw_buffer_load_b128 (row, at * 4, 0, kPastL2));
      const vkl_u32x4 b
          = __builtin_bit_cast (vkl_u32x4, __builtin_amdgcn_raw_buffer_load_b128 (row, at * 4 + 16, 0, kPastL2));
      const uint32_t off = (a.x ^ tag) | (a.y ^ tag) | (a.z ^ tag) | (a.w ^ tag) | (b.x ^ tag) | (b.y ^ tag)
                           | (b.z ^ tag) | (b.w ^ tag);
      if ((off >> 16) == 0)
        {
          v = make_uint4 ((a.x & 0xffff) | a.y << 16, (a.z & 0xffff) | a.w << 16, (b.x & 0xffff) | b.y << 16,
                          (b.z & 0xffff) | b.w << 16);
          return true;
        }
    }
  return false;
}

// The number of a lane or thread as something to compute anew from in every layer: addresses
// and offsets that follow from it are cheap, and kept around the loop over the layers they
// would fill the registers.
__device__ __forceinline__ int
anew (int v)
{
  asm volatile ("" : "+v"(v));
  return v;
}

struct Wait
{
  uint32_t *err;  // the error word of the step
  uint32_t *dead; // LDS: set once a wait of this workgroup gave up
  int limit;
};

__device__ __forceinline__ void
give_up (const Wait &w, uint32_t stage)
{
  *w.dead = 1u;
  uint32_t expected = 0u; // (the word keeps the first cause)
  __hip_atomic_compare_exchange_strong (w.err, &expected, 0x100u | stage, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int
polls (const Wait &w)
{
  return *w.dead ? 1 : w.limit;
}

// a row that is multiplied as it is -> xl
template <int CH>
__device__ __forceinline__ void
row_in (uint32_t *base, int n, uint32_t tag, const Wait &w, uint32_t stage, uint16_t *xl)
{
  const rsrc_t row = tagged_row (base, n);
  const int limit = polls (w);
#pragma unroll
  for (int j = 0; j < CH; ++j)
    {
      const int c = (int)threadIdx.x + j * kDecThreads;
      uint4 v = make_uint4 (0, 0, 0, 0);
      if (c * 8 < n)
        {
          if (!poll8 (row, c * 8, tag, limit, v))
            give_up (w, stage);
          ((uint4 *)xl)[c] = v;
        }
    }
  __syncthreads ();
}

// a row that is normalised first (at most 4096 values, eight per thread; fetch (c) brings
// values 8 c .. 8 c + 7): the row itself -> xr,
// y = fp16 (x * g * (1 / sqrt (mean (x^2) + eps))) -> xl.  The sums are those of stage_row,
// thread for thread.
template <typename Fetch>
__device__ __forceinline__ void
row_in_norm (Fetch fetch, int n, const uint4 (&g)[2], float eps, uint16_t *xr, uint16_t *xl, float *red)
{
  const int c = (int)threadIdx.x;
  const bool in = c * 8 < n;
  uint4 v = make_uint4 (0, 0, 0, 0);
  float s = 0.f;
  if (in)
    {
      v = fetch (c);
      ((uint4 *)xr)[c] = v;
    }
  const uint32_t x[4] = { v.x, v.y, v.z, v.w };
#pragma unroll
  for (int i = 0; i < 4; ++i)
    {
      const float a = h2f ((uint16_t)(x[i] & 0xffff)), b = h2f ((uint16_t)(x[i] >> 16));
      s += a * a;
      s += b * b;
    }
  s = wave_sum (s);
  if ((threadIdx.x & 63) == 0)
    red[threadIdx.x >> 6] = s;
  __syncthreads ();
  float total = 0.f;
#pragma unroll
  for (int i = 0; i < kDecWaves; ++i)
    total += red[i];
  const float alpha = 1.0f / sqrtf (total / (float)n + eps);
  if (in)
    {
      const uint32_t gw[8] = { g[0].x, g[0].y, g[0].z, g[0].w, g[1].x, g[1].y, g[1].z, g[1].w };
      uint32_t r[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        {
          const float a = h2f ((uint16_t)(x[i] & 0xffff)), b = h2f ((uint16_t)(x[i] >> 16));
          r[i] = (uint32_t)f2h (a * __uint_as_float (gw[2 * i]) * alpha)
                 | ((uint32_t)f2h (b * __uint_as_float (gw[2 * i + 1]) * alpha) << 16);
        }
      ((uint4 *)xl)[c] = make_uint4 (r[0], r[1], r[2], r[3]);
    }
  __syncthreads ();
}

// values 8 c .. of a row of tagged words (0 where the wait gave up)
__device__ __forceinline__ uint4
tagged8 (uint32_t *base, int n, int c, uint32_t tag, const Wait &w, uint32_t stage)
{
  uint4 v = make_uint4 (0, 0, 0, 0);
  if (!poll8 (tagged_row (base, n), c * 8, tag, polls (w), v))
    give_up (w, stage);
  return v;
}

__device__ __forceinline__ void
load_norm_weights (const float *g, int n, uint4 (&v)[2])
{
  const int c = (int)threadIdx.x * 8 < n ? (int)threadIdx.x * 8 : 0;
  v[0] = ldg4 (g + c), v[1] = ldg4 (g + c + 4);
}

// The part of a product that a lane adds in one step: 16 bytes of a row.  The sums over a row
// are those of Gemv (vkl_decode_gemv.h), term for term, so the results are too.
template <int WT>
__device__ __forceinline__ float
add16 (float acc, const uint4 w, uint16_t d, const uint16_t *xl, int at)
{
  if (WT != 8)
    return dot8_f16 (w, *(const uint4 *)(xl + (at >> 1)), acc);
  const uint4 *xp = (const uint4 *)(xl + at);
  const uint4 x0 = xp[0], x1 = xp[1];
  const h16x2 xv[8] = { __builtin_bit_cast (h16x2, x0.x), __builtin_bit_cast (h16x2, x0.y),
                        __builtin_bit_cast (h16x2, x0.z), __builtin_bit_cast (h16x2, x0.w),
                        __builtin_bit_cast (h16x2, x1.x), __builtin_bit_cast (h16x2, x1.y),
                        __builtin_bit_cast (h16x2, x1.z), __builtin_bit_cast (h16x2, x1.w) };
  return acc + dot16_q8 (w, xv, 0.f) * h2f (d);
}

// a [N, K] matrix
template <int WT> struct Matrix
{
  const uint8_t *q;
  const uint16_t *d;
  int bytes, nb; // of a row

  __device__ __forceinline__
  Matrix (const void *base, int N, int K)
      : q ((const uint8_t *)base), d ((const uint16_t *)((const uint8_t *)base + (size_t)N * K)),
        bytes (WT == 8 ? K : 2 * K), nb (K >> 5)
  {
  }
};

// One row in a wave's registers: S steps of 1024 bytes, 16 per lane.  No branches: a lane
// past the end of the row requests its start and adds nothing.
template <int WT, bool NT, int S> struct Row
{
  uint4 w[S];
  uint16_t d[S];

  __device__ __forceinline__ void
  request (const Matrix<WT> m, int row, int lane)
  {
    const uint8_t *q = m.q + (size_t)row * m.bytes;
    const uint16_t *sc = m.d + (size_t)row * m.nb;
#pragma unroll
    for (int s = 0; s < S; ++s)
      {
        const int kk = s * 1024 + lane * 16;
        const uint32_t kc = kk < m.bytes ? (uint32_t)kk : 0u;
        w[s] = NT ? ldg4_stream (q + kc) : ldg4 (q + kc);
        if (WT == 8)
          d[s] = ldg (sc + (kc >> 5));
      }
  }

  // the sum over the row, in every lane
  __device__ __forceinline__ float
  dot (const uint16_t *xl, int K, int lane) const
  {
    const int bytes = WT == 8 ? K : 2 * K;
    float acc = 0.f;
#pragma unroll
    for (int s = 0; s < S; ++s)
      {
        const int kk = s * 1024 + lane * 16;
        const bool in = kk < bytes;
        const float sum = add16<WT> (acc, w[s], d[s], xl, in ? kk : 0);
        acc = in ? sum : acc;
      }
    return wave_sum (acc);
  }
};

// Two rows.  SD = 0: rows of up to 512 bytes, the halves of a wave take one each (half the
// loads, conversions and sums; the half that a row of its own would leave idle adds zeros).
template <int WT, bool NT, int SD> struct Duo
{
  Row<WT, NT, SD> a, b;

  __device__ __forceinline__ void
  request (const Matrix<WT> ma, int ra, const Matrix<WT> mb, int rb, int lane)
  {
    a.request (ma, ra, lane), b.request (mb, rb, lane);
  }
  __device__ __forceinline__ void
  dot (const uint16_t *xl, int K, int lane, float &ya, float &yb) const
  {
    ya = a.dot (xl, K, lane), yb = b.dot (xl, K, lane);
  }
};

template <int WT, bool NT> struct Duo<WT, NT, 0>
{
  uint4 w;
  uint16_t d;

  __device__ __forceinline__ void
  request (const Matrix<WT> ma, int ra, const Matrix<WT> mb, int rb, int lane)
  {
    const int kk = (lane & 31) * 16;
    const uint32_t kc = kk < ma.bytes ? (uint32_t)kk : 0u;
    const uint8_t *qa = ma.q + (size_t)ra * ma.bytes, *qb = mb.q + (size_t)rb * mb.bytes;
    const uint8_t *q = (lane < 32 ? qa : qb) + kc;
    w = NT ? ldg4_stream (q) : ldg4 (q);
    if (WT == 8)
      {
        const uint16_t *da = ma.d + (size_t)ra * ma.nb, *db = mb.d + (size_t)rb * mb.nb;
        d = ldg ((lane < 32 ? da : db) + (kc >> 5));
      }
  }
  __device__ __forceinline__ void
  dot (const uint16_t *xl, int K, int lane, float &ya, float &yb) const
  {
    const int kk = (lane & 31) * 16;
    const bool in = kk < (WT == 8 ? K : 2 * K);
    const float sum = add16<WT> (0.f, w, d, xl, in ? kk : 0);
    const float v = row_sum<16> (in ? sum : 0.f);
    ya = lane_value (v, 0) + lane_value (v, 16), yb = lane_value (v, 32) + lane_value (v, 48);
  }
};

// k, q and v of a head, and its output, as tagged words
struct HeadRows
{
  uint32_t *kqv, *att; // att: the first copy
  int stride, copy, threads;
  uint32_t tag;
  Wait w;
  bool silent;

  __device__ __forceinline__ int
  thread () const
  {
    return anew ((int)threadIdx.x);
  }
  __device__ __forceinline__ uint32_t
  pair (const Params &, bool is_k, bool is_v, int first, int pi) const
  {
    if ((int)threadIdx.x >= threads)
      return 0;
    const int at = (is_k ? 0 : (is_v ? 2 : 1)) * stride + first + 2 * pi;
    const rsrc_t r = tagged_row (kqv, 3 * stride);
    const int limit = polls (w);
    for (int spin = 0; spin < limit; ++spin)
      {
        asm volatile ("" ::: "memory");
        typedef uint32_t u32x2 __attribute__ ((ext_vector_type (2)));
        const u32x2 v = __builtin_bit_cast (
            u32x2, __builtin_amdgcn_raw_buffer_load_b64 (r, at * 4, 0, kPastL2));
        if ((((v.x ^ tag) | (v.y ^ tag)) >> 16) == 0)
          return (v.x & 0xffff) | v.y << 16;
      }
    give_up (w, ST_KQV);
    return 0;
  }
  __device__ __forceinline__ void
  put (const Params &, int at, int lane, float o, float) const
  {
    // four lanes per column: two copies each
    if (silent || *w.dead)
      return;
    uint32_t *dst = att + at + (lane & 3) * copy;
    st_coherent_u32 (dst, tag | f2h (o));
    st_coherent_u32 (dst + 4 * copy, tag | f2h (o));
  }
  __device__ __forceinline__ bool
  live () const
  {
    return *w.dead == 0u;
  }
};

// The workgroup's `n` values, at most eight per wave, from LDS to all copies of a row: eight
// lanes for eight neighbouring words of a copy.
// One store of 32 bytes per copy instead of one of four per value and copy.
__device__ __forceinline__ void
publish (uint32_t *row, int copy, int at, const uint32_t *out, int n, int wave, int lane, const uint32_t *dead)
{
  __syncthreads ();
  const int i = wave * 8 + (lane & 7);
  if (i < n && *dead == 0u)
    st_coherent_u32 (row + (lane >> 3) * copy + at + i, out[i]);
}

struct LdsMap
{
  int xa, xb, xc, xr, xd, words, attn, bytes; // byte offsets; words: reduction words and `dead`
};

__host__ __device__ inline LdsMap
lds_map (int dim, int ffn, int maxlen, int hd)
{
  LdsMap m;
  const int row = (dim * 2 + 15) & ~15;
  m.words = 0;
  // rows, or what a head needs: a workgroup has one or the other (the token is picked in a head's
  // place, behind the last row)
  m.attn = 128 + (5 + kPairs) * kDecWaves * 4;
  m.xa = m.attn, m.xb = m.xa + row, m.xc = m.xb + row, m.xr = m.xc + row, m.xd = m.xr + row;
  const int rpb = kDecThreads / (hd / 8);
  const int rows = m.xd + ((ffn * 2 + 15) & ~15), head = m.attn + 1024 + ((maxlen + 3) & ~3) * 4 + rpb * hd * 4 + 256;
  m.bytes = rows > head ? rows : head;
  return m;
}

// What a wave multiplies in a layer; the entry's part is on its way a layer ahead.
// SD: steps of 1024 bytes in a row of dim values, 0 where it takes half of one
template <int WT, int SD, bool NT> struct Entry
{
  Duo<WT, NT, SD> kq;
  Row<WT, NT, SD ? SD : 1> v;
  uint4 g[2]; // norm weights
};

template <int WT, int SD, bool NT> struct Rest
{
  Row<WT, NT, SD ? SD : 1> o;
  Duo<WT, NT, SD> ug[kPairs];
  Row<WT, NT, SD ? 3 * SD : 2> down;
  uint4 g[2];
};

// Where the step's token comes from and goes to, by scalar loads: nothing of it is written
// before every workgroup has read it.
typedef const __attribute__ ((address_space (4))) uint32_t *ScalarWord;

__device__ __forceinline__ uint32_t
this_token (const Params &p)
{
  const uint32_t t = p.loop ? ((ScalarWord)p.ids)[((ScalarWord)p.loop)[0]] : *(ScalarWord)p.tok;
  return t < (uint32_t)p.m.vocab ? t : 0u;
}

// values 8 c .. of the token's embedding row (the arithmetic of embed_row)
template <int WT>
__device__ __forceinline__ uint4
embedding8 (const Params &p, uint32_t tok, int c)
{
  const int dim = p.m.dim;
  if (WT != 8)
    return ldg4 ((const uint16_t *)p.m.tok_embd + (size_t)tok * dim + c * 8);
  const Matrix<8> t (p.m.tok_embd, p.m.vocab, dim);
  const unsigned long long q = ldg ((const unsigned long long *)(t.q + (size_t)tok * dim + c * 8));
  const float sc = h2f (ldg (t.d + (size_t)tok * (dim >> 5) + (c >> 2)));
  uint32_t o[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    o[j] = (uint32_t)f2h ((float)(int8_t)(q >> (16 * j)) * sc)
           | ((uint32_t)f2h ((float)(int8_t)(q >> (16 * j + 8)) * sc) << 16);
  return make_uint4 (o[0], o[1], o[2], o[3]);
}

// The vocabulary: the workgroups that have neither rows nor a head request their part of the
// output matrix when the launch begins and hold it in registers until the last layer's row
// arrives; each leaves its arg-max for workgroup 0.  From the last row to the next token 8.5 us
// (512 wide, 17 MB) where the lm_head launch, its arg-max and two launch boundaries took 33
// of 120 us per token.
constexpr int kVocabLoads = 16; // loads of 16 bytes per lane that a wave holds of it (24 do not fit 128 registers)

template <int WT, int SD, bool NT>
__device__ __forceinline__ void
vocabulary (const Params &p, int part, int parts, uint32_t tag, int layers, const Wait &w, uint32_t *x,
            uint32_t *best, uint16_t *xr, uint16_t *xa, float *red)
{
  constexpr int kDuos = kVocabLoads / (SD ? 2 * SD : 1);
  const vkl_decode_model &m = p.m;
  const int dim = m.dim, V = m.vocab;
  const int lane = (int)threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane ((int)(threadIdx.x >> 6));
  const Matrix<WT> out (m.output, V, dim);
  const int waves = parts * kDecWaves, mine = part * kDecWaves + wave;
  // (vocab is even: a wave's rows come in twos)
  const int lo = 2 * (int)((long)(V / 2) * mine / waves), hi = 2 * (int)((long)(V / 2) * (mine + 1) / waves);
  Duo<WT, NT, SD> r[kDuos];
  uint4 g[2];
  load_norm_weights (m.output_norm, dim, g);
  auto request = [&] (int row) {
#pragma unroll
    for (int i = 0; i < kDuos; ++i)
      {
        const int at = min (row + 2 * i, V - 2);
        r[i].request (out, at, out, at + 1, lane);
      }
  };
  request (lo);
  // Until the row of the layer before the last is there: seldom and one word, so that these
  // many workgroups stay out of the way of those that poll the row for its values.
  if (layers > 1)
    for (long spin = 0; spin < (long)w.limit * layers; ++spin)
      {
        if ((tag - (ld_coherent_u32 (x) & 0xffff0000u)) >> 16 <= 1u)
          break;
        __builtin_amdgcn_s_sleep (32);
      }
  row_in_norm ([&] (int c) { return tagged8 (x, dim, c, tag, w, ST_DOWN); }, dim, g, m.final_eps, xr, xa, red);
  float top = -INFINITY;
  uint32_t top_at = 0xffffffffu;
  for (int row = lo; row < hi; row += 2 * kDuos)
    {
      if (row != lo)
        request (row);
      // lane j takes row j of them
      float mine_v = 0.f;
#pragma unroll
      for (int i = 0; i < kDuos; ++i)
        {
          float a, b;
          r[i].dot (xa, dim, lane, a, b);
          mine_v = lane == 2 * i ? a : (lane == 2 * i + 1 ? b : mine_v);
        }
      const uint16_t h = f2h (mine_v);
      const float v = h2f (h);
      const int n = min (hi - row, 2 * kDuos);
      const bool in = lane < n;
      if (in && *w.dead == 0u)
        {
          stg (p.s.logits16 + row + lane, h);
          stg (p.logits32 + row + lane, v);
        }
      // the first of the largest (a NaN is never the largest)
      const float mx = wave_max (in ? v : -INFINITY);
      const unsigned long long at = __ballot (in && v == mx);
      if (at && better (mx, (uint32_t)(row + __builtin_ctzll (at)), top, top_at))
        top = mx, top_at = (uint32_t)(row + __builtin_ctzll (at));
    }
  uint32_t *idx = (uint32_t *)red + kDecWaves; // (red itself is not read any more: barriers since)
  if (lane == 0)
    red[wave] = top, idx[wave] = top_at;
  __syncthreads ();
  if (threadIdx.x == 0 && *w.dead == 0u)
    {
      for (int i = 1; i < kDecWaves; ++i)
        if (better (red[i], idx[i], red[0], idx[0]))
          red[0] = red[i], idx[0] = idx[i];
      const unsigned long long word = (unsigned long long)idx[0] << 32 | tag | f2h (red[0]);
      __hip_atomic_store ((unsigned long long *)best + part, word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// workgroup 0, last: the token from the `parts` arg-maxima
__device__ __forceinline__ void
pick_token (const Params &p, int parts, uint32_t tag, const Wait &w, uint32_t *best, uint8_t *lds)
{
  float v = -INFINITY;
  uint32_t at = 0xffffffffu;
  if ((int)threadIdx.x < parts)
    {
      const rsrc_t row = tagged_row (best, 2 * parts);
      const int limit = polls (w);
      bool ok = false;
      for (int spin = 0; spin < limit && !ok; ++spin)
        {
          asm volatile ("" ::: "memory");
          typedef uint32_t u32x2 __attribute__ ((ext_vector_type (2)));
          const u32x2 b = __builtin_bit_cast (
              u32x2, __builtin_amdgcn_raw_buffer_load_b64 (row, (int)threadIdx.x * 8, 0, kPastL2));
          ok = ((b.x ^ tag) >> 16) == 0;
          v = h2f ((uint16_t)(b.x & 0xffff)), at = b.y;
        }
      if (!ok)
        give_up (w, ST_HEAD);
    }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
    {
      const float ov = __shfl_xor (v, o, 64);
      const uint32_t oi = __shfl_xor (at, o, 64);
      if (better (ov, oi, v, at))
        v = ov, at = oi;
    }
  float *bv = (float *)lds;
  uint32_t *bi = (uint32_t *)(lds + 64);
  if ((threadIdx.x & 63) == 0)
    bv[threadIdx.x >> 6] = v, bi[threadIdx.x >> 6] = at;
  __syncthreads ();
  if (threadIdx.x == 0 && *w.dead == 0u)
    {
      for (int i = 1; i < kDecWaves; ++i)
        if (better (bv[i], bi[i], v, at))
          v = bv[i], at = bi[i];
      const uint32_t id = at == 0xffffffffu ? 0u : at;
      if (p.loop && !p.sample)
        {
          // to the next replay of the step
          const uint32_t i = ldg (p.loop), ps = ldg (p.loop + 1);
          stg (p.ids + i + 1, id);
          stg ((uint32_t *)p.loop, i + 1);
          stg ((uint32_t *)p.loop + 1, ps + 1);
        }
      else if (p.next_tok)
        stg (p.next_tok, id);
    }
}

// whole: a step from its token to the logits and the next token (the grid has workgroups for
// the vocabulary); otherwise the layers alone, from Scratch::x to Scratch::x
template <int WT, int SD, bool NT>
__global__ __launch_bounds__ (kDecThreads) __attribute__ ((amdgpu_waves_per_eu (4, 4))) void
decode_layers_kernel (const Params p, bool whole)
{
  extern __shared__ __align__ (16) uint8_t lds[];
  const vkl_decode_model &m = p.m;
  const int dim = m.dim, ffn = m.ffn;
  const LdsMap map = lds_map (dim, ffn, m.maxlen, m.head_dim);
  float *red = (float *)(lds + map.words);
  uint32_t *dead = (uint32_t *)(red + 2 * kDecWaves);
  uint32_t *out = dead + 16; // results of the four products
  const TaggedRows tr = tagged_rows (dim, ffn);
  uint32_t *rows = p.s.tagged;
  uint32_t *err = p.s.sync + kSyncErr;
  uint32_t *counter = p.s.lsync + kLsTags;
  const int copy = (int)(__builtin_amdgcn_s_getreg (20 | (0 << 6) | (3 << 11)) & 7u); // the XCD's number
  const uint32_t done = ld_coherent_u32 (counter);
  // (once a wait has given up the step is lost anyway)
  const Wait w = { err, dead, ld_coherent_u32 (err) != 0u ? 1 : (m.wait_polls > 0 ? m.wait_polls : kTagSpinLimit) };
  if (threadIdx.x == 0)
    *dead = 0u;
  __syncthreads ();
  // the table of layers is not written while a step runs: scalar loads
  typedef const __attribute__ ((address_space (4))) vkl_layer_weights *Table;
  const Table table = (Table)m.layers;
  const int count = m.n_layers;
  uint16_t *xa = (uint16_t *)(lds + map.xa), *xb = (uint16_t *)(lds + map.xb), *xc = (uint16_t *)(lds + map.xc);
  uint16_t *xr = (uint16_t *)(lds + map.xr), *xd = (uint16_t *)(lds + map.xd);
  const int G = dim / kDecWaves;
  const int parts = (int)gridDim.x - G - m.n_heads; // workgroups of the vocabulary
  const uint32_t last_tag = (done + (uint32_t)count) << 16;
  uint32_t *best = rows + tr.best;

  if ((int)blockIdx.x >= G + m.n_heads)
    {
      vocabulary<WT, SD, NT> (p, (int)blockIdx.x - G - m.n_heads, parts, last_tag, count, w,
                              rows + tr.x + copy * tr.copy_d, best, xr, xa, red);
      return;
    }

  // ---- the workgroups behind those of the rows: a head of the attention each -------------
  if ((int)blockIdx.x >= G)
    {
      for (int l = 0; l < count; ++l)
        {
          vkl_layer_weights lw;
          lw.kcache = table[l].kcache, lw.vcache = table[l].vcache;
          const HeadRows hr = { rows + tr.kqv, rows + tr.att, tr.copy_d, tr.copy_d, m.head_dim / 2 * 3,
                                (done + (uint32_t)l + 1u) << 16, w, m.wait_test != 0 };
          const int head = (int)blockIdx.x - G;
          if (m.head_dim == 128)
            attention_head<128, true, true> (p, lw, head, lds + map.attn, nullptr, NoWait (), hr);
          else
            attention_head<64, true, true> (p, lw, head, lds + map.attn, nullptr, NoWait (), hr);
          __syncthreads ();
        }
      return;
    }

  // (what is requested behind the up/gate product, see above)
  constexpr bool kLateDown = SD > 0, kLateEntry = SD > 1;
  const int wave = __builtin_amdgcn_readfirstlane ((int)(threadIdx.x >> 6));
  const int g = (int)blockIdx.x * kDecWaves + wave; // number of the wave: dim of them
  const int first_row = (int)blockIdx.x * kDecWaves;
  const int first_pair = (int)((unsigned)ffn * (unsigned)first_row / (unsigned)dim);
  const int end_pair = (int)((unsigned)ffn * (unsigned)(first_row + kDecWaves) / (unsigned)dim);
  const int lo = (int)((unsigned)ffn * (unsigned)g / (unsigned)dim);
  const int pairs = (int)((unsigned)ffn * (unsigned)(g + 1) / (unsigned)dim) - lo;
  int lane = (int)threadIdx.x & 63;

  auto request_entry = [&] (const void *wk, const void *wq, const void *wv, const float *norm) {
    Entry<WT, SD, NT> n;
    n.kq.request (Matrix<WT> (wk, dim, dim), g, Matrix<WT> (wq, dim, dim), g, lane);
    n.v.request (Matrix<WT> (wv, dim, dim), g, lane);
    load_norm_weights (norm, dim, n.g);
    return n;
  };
  const uint32_t tok = whole ? this_token (p) : 0u;
  Entry<WT, SD, NT> in = request_entry (table[0].wk, table[0].wq, table[0].wv, table[0].attn_norm);

  for (int l = 0;; ++l)
    {
      lane = anew (lane);
      // (the pointers come with scalar loads, here so that nobody waits for them; behind
      // the last layer those of the last layer again)
      const void *wo = table[l].wo, *w_gate = table[l].w_gate, *w_up = table[l].w_up, *w_down = table[l].w_down;
      const float *ffn_norm = table[l].ffn_norm;
      const int ln = min (l + 1, count - 1);
      const void *wk = table[ln].wk, *wq = table[ln].wq, *wv = table[ln].wv;
      const float *attn_norm = table[ln].attn_norm;
      const uint32_t tag = (done + (uint32_t)l + 1u) << 16;

      // ---- RMSNorm + K/Q/V ------------------------------------------------------
      row_in_norm (
          [&] (int c) {
            if (l > 0)
              return tagged8 (rows + tr.x + copy * tr.copy_d, dim, c, tag - 0x10000u, w, ST_DOWN);
            return whole ? embedding8<WT> (p, tok, c) : ldg4 (p.s.x + c * 8);
          },
          dim, in.g, m.eps, xr, xa, red);
      {
        float a, b;
        in.kq.dot (xa, dim, lane, a, b);
        const float c = in.v.dot (xa, dim, lane);
        uint32_t *ok = out + kDecWaves * (2 + kPairs);
        if (lane < 3)
          ok[lane * kDecWaves + wave] = tag | f2h (lane == 0 ? a : (lane == 1 ? b : c));
        // (one reader per head: no copies; the eight lanes of a row of k, q or v)
        __syncthreads ();
        if (wave == 0 && lane < 3 * kDecWaves && *dead == 0u)
          st_coherent_u32 (rows + tr.kqv + (lane >> 3) * tr.copy_d + first_row + (lane & 7), ok[lane]);
      }

      // ---- while the heads are computed: the weights up to the next layer's K/Q/V -------------
      // (a poll returns behind the weights requested before it, and any of the later
      // hand-overs is shorter than their way from memory; kLateDown and kLateEntry: what the
      // registers do not hold beside up/gate)
      Rest<WT, SD, NT> r;
      r.o.request (Matrix<WT> (wo, dim, dim), g, lane);
#pragma unroll
      for (int j = 0; j < kPairs; ++j)
        {
          // (a wave with fewer pairs repeats its last)
          const int u = min (lo + j, max (lo + pairs - 1, 0));
          r.ug[j].request (Matrix<WT> (w_up, ffn, dim), u, Matrix<WT> (w_gate, ffn, dim), u, lane);
        }
      load_norm_weights (ffn_norm, dim, r.g);
      if (!kLateDown)
        r.down.request (Matrix<WT> (w_down, dim, ffn), g, lane);
      if (!kLateEntry)
        in = request_entry (wk, wq, wv, attn_norm);

      // ---- Wo + residual ------------------------------------------------------------
      row_in<1> (rows + tr.att + copy * tr.copy_d, dim, tag, w, ST_ATT, xb);
      {
        const uint32_t y = f2h (h2f (f2h (r.o.dot (xb, dim, lane))) + h2f (xr[g]));
        if (lane == 0)
          out[wave] = tag | y;
        publish (rows + tr.xm, tr.copy_d, first_row, out, kDecWaves, wave, lane, dead);
      }

      // ---- RMSNorm + up/gate with SiLU -------------------------------------------------
      row_in_norm ([&] (int c) { return tagged8 (rows + tr.xm + copy * tr.copy_d, dim, c, tag, w, ST_WO); }, dim,
                   r.g, m.eps, xr, xc, red + kDecWaves);
      {
        uint32_t *ot = out + kDecWaves;
        // (lane j ends pair j)
        float u = 0.f, a = 0.f;
#pragma unroll
        for (int j = 0; j < kPairs; ++j)
          {
            float uj, aj;
            r.ug[j].dot (xc, dim, lane, uj, aj);
            u = lane == j ? uj : u, a = lane == j ? aj : a;
          }
        if (lane < pairs)
          ot[lo + lane - first_pair] = tag | f2h (silu (a) * u);
        publish (rows + tr.t, tr.copy_f, first_pair, ot, end_pair - first_pair, wave, lane, dead);
        if (kLateDown)
          r.down.request (Matrix<WT> (w_down, dim, ffn), g, lane);
        if (kLateEntry)
          in = request_entry (wk, wq, wv, attn_norm);
      }

      // ---- down + residual --------------------------------------------------------------
      row_in<2> (rows + tr.t + copy * tr.copy_f, ffn, tag, w, ST_UP, xd);
      const uint32_t y = f2h (h2f (f2h (r.down.dot (xd, ffn, lane))) + h2f (xr[g]));
      uint32_t *ox = out + kDecWaves * (1 + kPairs);
      if (l + 1 == count && !whole)
        {
          if (lane == 0 && *dead == 0u)
            stg (p.s.x + g, (uint16_t)y);
          break;
        }
      if (lane == 0)
        ox[wave] = tag | y;
      publish (rows + tr.x, tr.copy_d, first_row, ox, kDecWaves, wave, lane, dead);
      if (l + 1 == count)
        break;
    }
  if (blockIdx.x != 0)
    return;
  if (whole)
    {
      __syncthreads ();
      pick_token (p, parts, last_tag, w, best, lds + map.attn);
    }
  // (every workgroup has read the counter before it published its first word, and this one
  // has seen words of all, unless it gave up: what a workgroup that starts later leaves then is
  // cleared with the error word)
  if (threadIdx.x == 0)
    st_coherent_u32 (counter, done + (uint32_t)count);
}

template <int WT, int SD, bool NT>
int
launch_layers_t (const Params &p, int groups, hipStream_t s)
{
  const size_t lds = (size_t)lds_map (p.m.dim, p.m.ffn, p.m.maxlen, p.m.head_dim).bytes;
  static LdsLimit limit;
  if (int e = limit.raise ((const void *)decode_layers_kernel<WT, SD, NT>, lds))
    return e;
  const int own = p.m.dim / kDecWaves + p.m.n_heads;
  decode_layers_kernel<WT, SD, NT>
      <<<dim3 ((unsigned)std::max (own, groups)), dim3 (kDecThreads), lds, s>>> (p, groups > own);
  return 0;
}

template <int WT, int SD>
int
launch_layers_nt (const Params &p, int groups, hipStream_t s)
{
  return p.stream_once ? launch_layers_t<WT, SD, true> (p, groups, s)
                       : launch_layers_t<WT, SD, false> (p, groups, s);
}

int
row_bytes (const vkl_decode_model &m)
{
  return m.wtype == 8 ? m.dim : 2 * m.dim;
}

int
launch_any (const Params &p, int groups, hipStream_t s)
{
  const int bytes = row_bytes (p.m);
  if (p.m.wtype == 8)
    return bytes <= 512    ? launch_layers_nt<8, 0> (p, groups, s)
           : bytes <= 1024 ? launch_layers_nt<8, 1> (p, groups, s)
                           : launch_layers_nt<8, 2> (p, groups, s);
  return bytes <= 512    ? launch_layers_nt<1, 0> (p, groups, s)
         : bytes <= 1024 ? launch_layers_nt<1, 1> (p, groups, s)
                         : launch_layers_nt<1, 2> (p, groups, s);
}
} // namespace

// Where dim waves have at most three up/gate pairs each, a layer's weights fit the registers
// and all workgroups have a compute unit of their own, of which they take half.  Us per token
// of a greedy loop, 32000 ids, a launch per layer / this form with an lm_head launch / the whole
// step in one launch: 256 wide Q8_0, 6 layers 131 / 74 / 65; 512 wide, 8 layers 173 / 100 / 88,
// fp16 167 / 94 / 88; 768 wide, 6 layers 141 / 86 / 80, fp16 134 / 82 / -; 4 layers: 1024 wide
// 102 / 67 / -, fp16 102 / 68 / -; 1536 wide 116 / 82 / -; 1792 wide 122 / 88 / -.  2048 wide (all
// 256 compute units for the rows, the heads beside them, weights a phase ahead) it was slower:
// 144 / 158, fp16 160 / 212; there a layer is bound by its weights, and polls behind them come
// late.
bool
layers_launch_supported (const vkl_decode_model &m, int n_cu)
{
  return m.flags != nullptr && m.layers != nullptr && tagged_shape (m) && m.dim / kDecWaves + m.n_heads <= n_cu
         && 2 * lds_map (m.dim, m.ffn, m.maxlen, m.head_dim).bytes <= 160 * 1024;
}

int
launch_layers (const Params &p, hipStream_t s)
{
  return launch_any (p, 0, s);
}

// The workgroups left over hold the output matrix in their registers, or at most twice that.
bool
whole_step_supported (const vkl_decode_model &m, int n_cu)
{
  if (!layers_launch_supported (m, n_cu))
    return false;
  const long parts = n_cu - m.dim / kDecWaves - m.n_heads;
  if (parts < 1 || parts > kDecThreads || parts > kMaxParts)
    return false;
  const int steps = (row_bytes (m) + 1023) / 1024;
  const long held = row_bytes (m) <= 512 ? 2 * kVocabLoads : kVocabLoads / steps; // rows of a wave
  return m.vocab <= 2 * held * parts * kDecWaves;
}

int
launch_step_whole (const Params &p, int n_cu, hipStream_t s)
{
  return launch_any (p, n_cu, s);
}
} // namespace dec
} // namespace vkl

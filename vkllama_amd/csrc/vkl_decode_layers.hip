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
// lines one by one), 11.1 with k, q and v gathered too and one SiLU for a wave's three pairs.
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
// weights requested before it: everything up to the next layer's K/Q/V is requested at the one
// point of the layer where the wait is longer than the way from memory, while the heads are
// computed.
//
// The tags of a step follow on those of the step before (a counter in the sync area,
// advanced at the end of a launch), and every word of a row is written once per layer: what
// a row holds before is always an older tag.  A row is not overwritten while somebody still
// waits for it: the next layer's needs a row that all workgroups have contributed to since.
// Waits are bounded and a wait that gave up is reported as in the layer launch; its
// workgroup publishes nothing from then on.
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
constexpr int kPairs = 3;     // up/gate pairs of a wave, at most
enum Stage { ST_KQV = 0, ST_ATT, ST_WO, ST_UP, ST_DOWN };

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

// a row that is normalised first (at most 4096 values, eight per thread): the row itself ->
// xr, y = fp16 (x * g * (1 / sqrt (mean (x^2) + eps))) -> xl.  The sums are those of
// stage_row, thread for thread.
template <bool TAGGED>
__device__ __forceinline__ void
row_in_norm (uint32_t *base, const uint16_t *plain, int n, uint32_t tag, const Wait &w, uint32_t stage,
             const uint4 (&g)[2], float eps, uint16_t *xr, uint16_t *xl, float *red)
{
  const int c = (int)threadIdx.x;
  const bool in = c * 8 < n;
  uint4 v = make_uint4 (0, 0, 0, 0);
  float s = 0.f;
  if (in)
    {
      if (!TAGGED)
        v = ldg4 (plain + c * 8);
      else if (!poll8 (tagged_row (base, n), c * 8, tag, polls (w), v))
        give_up (w, stage);
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

__device__ __forceinline__ void
load_norm_weights (const float *g, int n, uint4 (&v)[2])
{
  const int c = (int)threadIdx.x * 8 < n ? (int)threadIdx.x * 8 : 0;
  v[0] = ldg4 (g + c), v[1] = ldg4 (g + c + 4);
}

// One row of a matrix in a wave's registers: S steps of 1024 bytes, 16 per lane.  The sums
// are those of Gemv (vkl_decode_gemv.h), so the results are too.  No branches: a lane past the
// end of the row requests its start and adds nothing.
template <int WT, bool NT, int S> struct Row
{
  uint4 w[S];
  uint16_t d[S];

  // the row of a [N, K] matrix
  __device__ __forceinline__ void
  request (const void *matrix, int N, int K, int row, int lane)
  {
    const int bytes = WT == 8 ? K : 2 * K, nb = K >> 5;
    const uint8_t *q = (const uint8_t *)matrix + (size_t)row * bytes;
    const uint16_t *sc = (const uint16_t *)((const uint8_t *)matrix + (size_t)N * K) + (size_t)row * nb;
#pragma unroll
    for (int s = 0; s < S; ++s)
      {
        const int kk = s * 1024 + lane * 16;
        const uint32_t kc = kk < bytes ? (uint32_t)kk : 0u;
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
        const int kc = in ? kk : 0;
        float sum;
        if (WT != 8)
          sum = dot8_f16 (w[s], *(const uint4 *)(xl + (kc >> 1)), acc);
        else
          {
            const uint4 *xp = (const uint4 *)(xl + kc);
            const uint4 x0 = xp[0], x1 = xp[1];
            const h16x2 xv[8]
                = { __builtin_bit_cast (h16x2, x0.x), __builtin_bit_cast (h16x2, x0.y),
                    __builtin_bit_cast (h16x2, x0.z), __builtin_bit_cast (h16x2, x0.w),
                    __builtin_bit_cast (h16x2, x1.x), __builtin_bit_cast (h16x2, x1.y),
                    __builtin_bit_cast (h16x2, x1.z), __builtin_bit_cast (h16x2, x1.w) };
            sum = acc + dot16_q8 (w[s], xv, 0.f) * h2f (d[s]);
          }
        acc = in ? sum : acc;
      }
    return wave_sum (acc);
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
  m.xa = 0, m.xb = row, m.xc = 2 * row, m.xr = 3 * row, m.xd = 4 * row;
  m.words = m.xd + ((ffn * 2 + 15) & ~15);
  m.attn = m.words + 128 + (5 + kPairs) * kDecWaves * 4;
  const int rpb = kDecThreads / (hd / 8);
  m.bytes = m.attn + 1024 + ((maxlen + 3) & ~3) * 4 + rpb * hd * 4 + 256;
  return m;
}

// What a wave multiplies in a layer; the entry's part is on its way a layer ahead.
template <int WT, int SD, bool NT> struct Entry
{
  Row<WT, NT, SD> k, q, v;
  uint4 g[2]; // norm weights
};

template <int WT, int SD, bool NT> struct Rest
{
  Row<WT, NT, SD> o, up[kPairs], gate[kPairs];
  Row<WT, NT, 3 * SD> down; // (SD: steps of 1024 bytes in a row of dim values)
  uint4 g[2];
};

template <int WT, int SD, bool NT>
__global__ __launch_bounds__ (kDecThreads) __attribute__ ((amdgpu_waves_per_eu (2, 2))) void
decode_layers_kernel (const Params p, int first, int count)
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
  const uint32_t done = ld_coherent_u32 (counter);
  // (once a wait has given up the step is lost anyway)
  const Wait w = { err, dead, ld_coherent_u32 (err) != 0u ? 1 : (m.wait_polls > 0 ? m.wait_polls : kTagSpinLimit) };
  if (threadIdx.x == 0)
    *dead = 0u;
  __syncthreads ();
  // the table of layers is not written while a step runs: scalar loads
  typedef const __attribute__ ((address_space (4))) vkl_layer_weights *Table;
  const Table table = (Table)m.layers + first;

  // ---- the workgroups behind those of the rows: a head of the attention each -------------
  const int G = dim / kDecWaves;
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

  uint16_t *xa = (uint16_t *)(lds + map.xa), *xb = (uint16_t *)(lds + map.xb), *xc = (uint16_t *)(lds + map.xc);
  uint16_t *xr = (uint16_t *)(lds + map.xr), *xd = (uint16_t *)(lds + map.xd);
  const int wave = __builtin_amdgcn_readfirstlane ((int)(threadIdx.x >> 6));
  const int g = (int)blockIdx.x * kDecWaves + wave; // number of the wave: dim of them
  const int first_row = (int)blockIdx.x * kDecWaves;
  const int first_pair = (int)((unsigned)ffn * (unsigned)first_row / (unsigned)dim);
  const int end_pair = (int)((unsigned)ffn * (unsigned)(first_row + kDecWaves) / (unsigned)dim);
  const int lo = (int)((unsigned)ffn * (unsigned)g / (unsigned)dim);
  const int pairs = (int)((unsigned)ffn * (unsigned)(g + 1) / (unsigned)dim) - lo;
  const int copy = (int)(__builtin_amdgcn_s_getreg (20 | (0 << 6) | (3 << 11)) & 7u); // the XCD's number
  int lane = (int)threadIdx.x & 63;

  auto request_entry = [&] (const void *wk, const void *wq, const void *wv, const float *norm) {
    Entry<WT, SD, NT> n;
    n.k.request (wk, dim, dim, g, lane);
    n.q.request (wq, dim, dim, g, lane);
    n.v.request (wv, dim, dim, g, lane);
    load_norm_weights (norm, dim, n.g);
    return n;
  };
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
      if (l == 0)
        row_in_norm<false> (nullptr, p.s.x, dim, 0, w, ST_DOWN, in.g, m.eps, xr, xa, red);
      else
        row_in_norm<true> (rows + tr.x + copy * tr.copy_d, nullptr, dim, tag - 0x10000u, w, ST_DOWN, in.g, m.eps, xr,
                           xa, red);
      {
        const float a = in.k.dot (xa, dim, lane), b = in.q.dot (xa, dim, lane), c = in.v.dot (xa, dim, lane);
        uint32_t *ok = out + kDecWaves * (2 + kPairs);
        if (lane < 3)
          ok[lane * kDecWaves + wave] = tag | f2h (lane == 0 ? a : (lane == 1 ? b : c));
        // (one reader per head: no copies; the eight lanes of a row of k, q or v)
        __syncthreads ();
        if (wave == 0 && lane < 3 * kDecWaves && *dead == 0u)
          st_coherent_u32 (rows + tr.kqv + (lane >> 3) * tr.copy_d + first_row + (lane & 7), ok[lane]);
      }

      // ---- while the heads are computed: all weights up to the next layer's K/Q/V -------------
      // (a poll returns behind the weights requested before it, and any of the later
      // hand-overs is shorter than their way from memory)
      Rest<WT, SD, NT> r;
      r.o.request (wo, dim, dim, g, lane);
#pragma unroll
      for (int j = 0; j < kPairs; ++j)
        {
          // (a wave with fewer pairs repeats its last)
          const int u = min (lo + j, max (lo + pairs - 1, 0));
          r.up[j].request (w_up, ffn, dim, u, lane);
          r.gate[j].request (w_gate, ffn, dim, u, lane);
        }
      load_norm_weights (ffn_norm, dim, r.g);
      r.down.request (w_down, dim, ffn, g, lane);
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
      row_in_norm<true> (rows + tr.xm + copy * tr.copy_d, nullptr, dim, tag, w, ST_WO, r.g, m.eps, xr, xc,
                         red + kDecWaves);
      {
        uint32_t *ot = out + kDecWaves;
        // (lane j ends pair j)
        float u = 0.f, a = 0.f;
#pragma unroll
        for (int j = 0; j < kPairs; ++j)
          {
            const float uj = r.up[j].dot (xc, dim, lane), aj = r.gate[j].dot (xc, dim, lane);
            u = lane == j ? uj : u, a = lane == j ? aj : a;
          }
        if (lane < pairs)
          ot[lo + lane - first_pair] = tag | f2h (silu (a) * u);
        publish (rows + tr.t, tr.copy_f, first_pair, ot, end_pair - first_pair, wave, lane, dead);
      }

      // ---- down + residual --------------------------------------------------------------
      row_in<2> (rows + tr.t + copy * tr.copy_f, ffn, tag, w, ST_UP, xd);
      const uint32_t y = f2h (h2f (f2h (r.down.dot (xd, ffn, lane))) + h2f (xr[g]));
      if (l + 1 == count)
        {
          if (lane == 0 && *dead == 0u)
            stg (p.s.x + g, (uint16_t)y);
          break;
        }
      uint32_t *ox = out + kDecWaves * (1 + kPairs);
      if (lane == 0)
        ox[wave] = tag | y;
      publish (rows + tr.x, tr.copy_d, first_row, ox, kDecWaves, wave, lane, dead);
    }
  // (every workgroup has read the counter before it published its first word, and this one
  // has seen words of all)
  if (blockIdx.x == 0 && threadIdx.x == 0)
    st_coherent_u32 (counter, done + (uint32_t)count);
}

template <int WT, int SD, bool NT>
int
launch_layers_t (const Params &p, int first, int count, hipStream_t s)
{
  const size_t lds = (size_t)lds_map (p.m.dim, p.m.ffn, p.m.maxlen, p.m.head_dim).bytes;
  static LdsLimit limit;
  if (int e = limit.raise ((const void *)decode_layers_kernel<WT, SD, NT>, lds))
    return e;
  decode_layers_kernel<WT, SD, NT>
      <<<dim3 ((unsigned)(p.m.dim / kDecWaves + p.m.n_heads)), dim3 (kDecThreads), lds, s>>> (p, first, count);
  return 0;
}

template <int WT, int SD>
int
launch_layers_nt (const Params &p, int first, int count, hipStream_t s)
{
  return p.stream_once ? launch_layers_t<WT, SD, true> (p, first, count, s)
                       : launch_layers_t<WT, SD, false> (p, first, count, s);
}
} // namespace

// Where dim waves have at most three up/gate pairs each, a layer's weights fit the registers
// and all workgroups have a compute unit of their own.  Us per token, a launch per layer / this
// form (greedy, 64 or 48 tokens, the lm_head launch included): 256 wide Q8_0, 6 layers 137 /
// 93; 512 wide, 8 layers 182 / 120, fp16 171 / 107; 4 layers: 1024 wide 112 / 83, fp16 110 /
// 82; 1536 wide 123 / 98.  2048 wide (all 256 compute units for the rows, the heads beside
// them, weights a phase ahead) it was slower: 144 / 158, fp16 160 / 212; there a layer is
// bound by its weights, and polls behind them come late.
bool
layers_launch_supported (const vkl_decode_model &m, int n_cu)
{
  return m.flags != nullptr && m.layers != nullptr && m.dim <= (m.wtype == 8 ? kTaggedMaxDim : kTaggedMaxDim / 2)
         && (m.dim % 64) == 0 && m.dim / kDecWaves + m.n_heads <= n_cu && m.ffn <= kPairs * m.dim
         && (m.ffn % 32) == 0 && m.ffn >= m.dim / kDecWaves
         && lds_map (m.dim, m.ffn, m.maxlen, m.head_dim).bytes <= 160 * 1024;
}

int
launch_layers (const Params &p, int first, int count, hipStream_t s)
{
  const int steps = ((p.m.wtype == 8 ? p.m.dim : 2 * p.m.dim) + 1023) / 1024;
  if (p.m.wtype == 8)
    return steps == 1 ? launch_layers_nt<8, 1> (p, first, count, s) : launch_layers_nt<8, 2> (p, first, count, s);
  return steps == 1 ? launch_layers_nt<1, 1> (p, first, count, s) : launch_layers_nt<1, 2> (p, first, count, s);
}
} // namespace dec
} // namespace vkl

// Attention of many query rows over the K/V rows of a prompt, one kernel per
// call: scores, masked softmax and the product with V without the [H, S, L]
// score and probability tensors ever reaching memory.
//
// One pass over the keys with a running maximum (online softmax): per tile of
// 64 keys the scores are formed (fp16: rounded like the stand-alone product: score =
// fp16(scale * q.k)), the maximum m is raised if needed - the products accumulated
// so far and the sum of exponentials are then multiplied by exp(m_old - m_new) -, the
// weights, rounded once as the operand of the second product, go into it as they
// are, and the division by their sum comes last, in fp32, before the one rounding
// of the output.  The separate operators round the NORMALISED probability to fp16
// instead; the two differ by two roundings of a weight (fp16: 2^-11 of it each), i.e. by at
// most 2 * 2^-11 * sum_l p[l] |v[l]|: 9.8e-3 of max (|o|, a tenth of that sum), inside the 1e-2
// the outputs are held to.  In bf16 weights and outputs are rounded to 2^-8 of themselves.
//
// Workgroup = 4 waves = 128 query rows of one head, 32 per wave; the keys come
// through LDS in tiles of 64.  Both products run on v_mfma_f32_32x32x16 in the
// transposed form, so that a lane's accumulator registers belong to ONE query:
//   S^T[key, q] = sum_d K[key, d] Q[q, d]      A = K tile (LDS), B = Q (regs)
//   O^T[d, q]   = sum_key V^T[d, key] P^T[key, q]   A = V^T tile (LDS), B = P^T
// Lane l of a wave owns query l % 32.  Of a 32-key block its 16 accumulator
// registers hold the keys 8*(r/4) + 4*(l/32) + r%4, so maximum and sum over
// keys are sums over a lane's own registers (the two lane halves are merged
// after every tile), and the weights it forms are, as they lie, the B
// operand of the second product: registers 8t .. 8t+7 are the eight k values
// of lane half l/32 in k-step t.
//
// Heads of 64 and 128 values (attn_tiles_kernel): K and V tiles go straight into LDS
// as they lie in memory (global_load_lds), the next tile while this one is multiplied,
// one barrier per tile; the V^T operand is read transposed (ds_read_b64_tr_b16: four
// keys of a column per lane, two reads make the eight k values above).  Other head sizes
// (attn_prefill_kernel): tiles travel through registers and V is written to LDS
// transposed, its keys permuted to the operand's order (slot 16t + 8h + j holds key
// 16t + 8*(j/4) + 4h + j%4 of the block).
//
// What bounds it: matrix cores 1024 cycles per wave and tile, vector ALU 13 instructions
// per two scores (two FMAs, two exponentials at a quarter of the rate, a maximum, one
// conversion, one dot product with ones for the sum) = 830, with rounded scores two more
// (mixed-precision FMAs round and widen on the way), LDS reads 32 KB; two workgroups on a
// compute unit overlap them.  The maximum is only raised by more than a
// factor of 2^6 in the weights at a time, which keeps nearly all tiles free of rescaling.
// Measured, us per call before (registers and two barriers per tile for all head sizes) and
// now: fp16, 32 heads of 128, 2048 rows 85 / 60, 40 heads, 3967 rows 308 / 224; bf16 in chunks
// with a sink, 2048 rows 100 / 51; 16 heads, 1500 rows behind 600 keys 67 / 46.
// Few query tiles (a turn of some dozen tokens behind a long context) would leave most
// compute units idle: then the keys of a query tile are divided among workgroups, whose
// unnormalised outputs a second launch adds up.
//
// The element type is a template parameter: fp16 (Llama-2) or bf16.  Query heads may share
// key/value heads, the score factor may grow with the query's position, and a head's output
// may be scaled by the sigmoid of a per-token gate.
//
// A second, small kernel in this file prepares the inputs of the first from
// the projection outputs: RoPE of Q (in place) and K, and the K/V cache write.
#include "../../include/vkl_hip.h"
#include "../../include/vkl_stack.h"
#include "vkl_common.h"
#include "vkl_gemm.h"
#include <algorithm>

namespace
{
typedef _Float16 half8 __attribute__ ((ext_vector_type (8)));
typedef __bf16 bf8 __attribute__ ((ext_vector_type (8)));
typedef float float16v __attribute__ ((ext_vector_type (16)));
typedef uint32_t u32x2 __attribute__ ((ext_vector_type (2)));

constexpr int kBQ = 128;      // query rows per workgroup
constexpr int kBKey = 64;     // keys per tile
constexpr int kThreads = 256;
constexpr float kNeg = -1.0e30f; // "no key seen yet": finite, so that kNeg - kNeg = 0

struct AttnArgs
{
  const uint16_t *q, *k, *v;
  uint16_t *out;
  int H, S, L, ntq;
  size_t qcs, qhs, kcs, khs, vcs, vhs, ors, ohs;
  float scale;
  int rep;            // query heads per key/value head
  float temp_coef;    // != 0: scale times 1 + coef ln (floor ((pos + 1) / every) + 1)
  int temp_every;
  const float *gate;  // optional [S, gs]: head h's output times sigmoid (gate[s, h])
  size_t gs;
  int chunk, sink;    // CHUNKED kernels: see vkl_attn_prefill_chunked_bf16
  int parts;          // workgroups that share the keys of a query tile (at most, with a span)
  int span;           // != 0: tiles of keys to a part, at most
  float *ws;          // parts > 1: their results, see part_row
};

// the two element types of the operands
struct F16Elem
{
  typedef half8 v8;
  static constexpr bool round_scores = true; // to fp16, as the stand-alone product stores them
  static __device__ __forceinline__ float16v
  mfma (v8 a, v8 b, float16v c)
  {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16 (a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint16_t
  bits (float f)
  {
    return vkl::f2h (f);
  }
  typedef _Float16 t;
  typedef _Float16 t2 __attribute__ ((ext_vector_type (2)));
  // sum + a[0] + a[1]
  static __device__ __forceinline__ float
  add2 (t2 a, float sum)
  {
    return __builtin_amdgcn_fdot2 (a, t2{ (_Float16)1.f, (_Float16)1.f }, sum, false);
  }
};

struct Bf16Elem
{
  typedef bf8 v8;
  static constexpr bool round_scores = false;
  static __device__ __forceinline__ float16v
  mfma (v8 a, v8 b, float16v c)
  {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16 (a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint16_t
  bits (float f)
  {
    return vkl::f2bf (f);
  }
  typedef __bf16 t;
  typedef __bf16 t2 __attribute__ ((ext_vector_type (2)));
  static __device__ __forceinline__ float
  add2 (t2 a, float sum)
  {
    return __builtin_amdgcn_fdot2_f32_bf16 (a, t2{ (__bf16)1.f, (__bf16)1.f }, sum, false);
  }
};

__device__ __align__ (16) const uint32_t g_zero16[4] = { 0, 0, 0, 0 };

__device__ __forceinline__ float
fast_exp (float x)
{
  return __builtin_amdgcn_exp2f (x * 1.44269504088896340736f);
}


// Which query tile of which head a workgroup has.
// Heavy query tiles (the last ones: most keys) first.  With a head count
// that is a multiple of 8 the workgroups of one head share id % 8, which
// keeps the head's K and V in the L2 of one XCD.
__device__ __forceinline__ void
tile_of (const AttnArgs &a, int b, int &head, int &qt)
{
  if ((a.H & 7) == 0)
    {
      // j: position in the XCD's queue.  Its 32 compute units take the first
      // 32 workgroups, then the next 32 beside them, and so on: every other
      // such layer runs in the opposite order, so that a heavy tile and a
      // light one share a compute unit.  (The order of the queue is reversed
      // within the layer, the last of which may be shorter: whatever the
      // number of tiles, every tile of every head has one place.)
      int j = b >> 3;
      const int queue = (a.H >> 3) * a.ntq, j0 = j & ~31;
      if ((j >> 5) & 1)
        j = j0 + min (queue, j0 + 32) - 1 - j;
      head = (b & 7) + 8 * (j / a.ntq);
      qt = a.ntq - 1 - (j % a.ntq);
    }
  else
    {
      head = b / a.ntq;
      qt = a.ntq - 1 - (b % a.ntq);
    }
}

template <int HD> struct Tile
{
  static constexpr int CPR = HD / 8;                       // 16-byte chunks per row
  static constexpr int KALL = kBKey * CPR, VALL = (kBKey / 2) * CPR;
  static constexpr int KCH = (KALL + kThreads - 1) / kThreads; // K chunks per thread
  static constexpr int VIT = (VALL + kThreads - 1) / kThreads; // (key pair, chunk) items per thread
  // item numbers past the last exist where the tile is not a multiple of the workgroup
  static constexpr bool KRAG = KALL % kThreads != 0, VRAG = VALL % kThreads != 0;
  uint4 k[KCH];
  uint4 v[VIT][2];
};

// K rows [t*64, t*64+64) of the head, as they lie; rows beyond L read zeros
template <int HD>
__device__ __forceinline__ void
load_k (const AttnArgs &a, const uint16_t *kb, int t, Tile<HD> &r)
{
  constexpr int CPR = Tile<HD>::CPR;
  const void *zeros = g_zero16;
#pragma unroll
  for (int i = 0; i < Tile<HD>::KCH; ++i)
    {
      const int c = threadIdx.x + i * kThreads;
      const int row = t * kBKey + c / CPR;
      r.k[i] = vkl::ldg4 (row < a.L && (!Tile<HD>::KRAG || c < Tile<HD>::KALL) ? (const void *)(kb + (size_t)row * a.khs + (c % CPR) * 8)
                                    : zeros);
    }
}

// key of slot s (0..63) of a tile
__device__ __forceinline__ int
slot_key (int s)
{
  const int blk = s >> 5, t = (s >> 4) & 1, h = (s >> 3) & 1, j = s & 7;
  return 32 * blk + 16 * t + 8 * (j >> 2) + 4 * h + (j & 3);
}

template <int HD>
__device__ __forceinline__ void
load_v (const AttnArgs &a, const uint16_t *vb, int t, Tile<HD> &r)
{
  const void *zeros = g_zero16;
#pragma unroll
  for (int i = 0; i < Tile<HD>::VIT; ++i)
    {
      const int it = threadIdx.x + i * kThreads;
      const int pair = it & 31, dc = it >> 5;
      // slots 2*pair and 2*pair+1 hold two adjacent keys
      const int row = t * kBKey + slot_key (2 * pair);
      const bool in = !Tile<HD>::VRAG || it < Tile<HD>::VALL;
      r.v[i][0] = vkl::ldg4 (row < a.L && in ? (const void *)(vb + (size_t)row * a.vhs + dc * 8) : zeros);
      r.v[i][1] = vkl::ldg4 (row + 1 < a.L && in ? (const void *)(vb + (size_t)(row + 1) * a.vhs + dc * 8)
                                           : zeros);
    }
}

template <int HD>
__device__ __forceinline__ void
store_k (const Tile<HD> &r, uint16_t *Ks)
{
  constexpr int CPR = Tile<HD>::CPR, LDK = HD + 8;
#pragma unroll
  for (int i = 0; i < Tile<HD>::KCH; ++i)
    {
      const int c = threadIdx.x + i * kThreads;
      if (Tile<HD>::KRAG && c >= Tile<HD>::KALL)
        continue;
      *(uint4 *)(Ks + (c / CPR) * LDK + (c % CPR) * 8) = r.k[i];
    }
}

// V^T: row = d, column = slot; a thread writes the two keys of its pair as one
// 32-bit word per d
template <int HD>
__device__ __forceinline__ void
store_v (const Tile<HD> &r, uint16_t *Vt)
{
  constexpr int LDV = kBKey + 8;
#pragma unroll
  for (int i = 0; i < Tile<HD>::VIT; ++i)
    {
      const int it = threadIdx.x + i * kThreads;
      const int pair = it & 31, dc = it >> 5;
      if (Tile<HD>::VRAG && it >= Tile<HD>::VALL)
        continue;
      const uint32_t va[4] = { r.v[i][0].x, r.v[i][0].y, r.v[i][0].z, r.v[i][0].w };
      const uint32_t vb[4] = { r.v[i][1].x, r.v[i][1].y, r.v[i][1].z, r.v[i][1].w };
      uint32_t *dst = (uint32_t *)(Vt + (size_t)(dc * 8) * LDV + 2 * pair);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        {
          dst[(2 * e) * (LDV / 2)] = (va[e] & 0xffffu) | (vb[e] << 16);
          dst[(2 * e + 1) * (LDV / 2)] = (va[e] >> 16) | (vb[e] & 0xffff0000u);
        }
    }
}

// S^T of one 32-key block: rows = keys 32*blk .. +31 of the tile in LDS
template <int HD, class E>
__device__ __forceinline__ float16v
score_block (const uint16_t *Ks, int blk, const typename E::v8 (&qf)[HD / 16], int lane)
{
  constexpr int LDK = HD + 8;
  float16v acc;
#pragma unroll
  for (int r = 0; r < 16; ++r)
    acc[r] = 0.f;
  const uint16_t *kp = Ks + (32 * blk + (lane & 31)) * LDK + (lane >> 5) * 8;
#pragma unroll
  for (int kt = 0; kt < HD / 16; ++kt)
    acc = E::mfma (*(const typename E::v8 *)(kp + kt * 16), qf[kt], acc);
  return acc;
}

// (heads wider than 128 values: one workgroup per compute unit, twice the registers)
// CHUNKED: a query sees keys from the start of its own chunk of positions on, and
// the softmax may have a sink (a score of 0 without a value)
template <int HD, class E, bool CHUNKED = false>
__global__ __launch_bounds__ (kThreads, HD <= 128 ? 2 : 1) void
attn_prefill_kernel (const AttnArgs a)
{
  typedef typename E::v8 v8;
  constexpr int KT = HD / 16, DB = HD / 32;
  constexpr int LDK = HD + 8, LDV = kBKey + 8;
  __shared__ __align__ (16) uint16_t Ks[kBKey * LDK];
  __shared__ __align__ (16) uint16_t Vt[HD * LDV];

  int head, qt;
  tile_of (a, (int)blockIdx.x, head, qt);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lq = lane & 31, hh = lane >> 5;
  const int q0 = qt * kBQ;
  const int qrow = q0 + wave * 32 + lq; // this lane's query
  const int shift = a.L - a.S;          // key l is visible iff l <= qrow + shift
  const int kmax = min (a.L, q0 + kBQ + shift);
  const int ntile = (kmax + kBKey - 1) / kBKey;
  const int wave_last = q0 + wave * 32 + 31 + shift; // last key any query of the wave sees
  // first key of the chunk of this lane's query, of the wave's first and last
  auto chunk_start = [&] (int row) { return CHUNKED && a.chunk ? (row + shift) / a.chunk * a.chunk : 0; };
  const int klow = chunk_start (qrow), wave_low = chunk_start (q0 + wave * 32);
  const int wave_high = chunk_start (q0 + wave * 32 + 31);
  const int t0 = CHUNKED ? chunk_start (q0) / kBKey : 0;
  const int kvh = head / a.rep;
  const uint16_t *kb = a.k + (size_t)kvh * a.kcs;
  const uint16_t *vb = a.v + (size_t)kvh * a.vcs;
  // this query's score factor
  float scale = a.scale;
  if (a.temp_coef != 0.f)
    scale *= 1.0f + a.temp_coef * logf ((float)((qrow + shift + 1) / a.temp_every + 1));

  v8 qf[KT];
  {
    const uint16_t *qp = a.q + (size_t)head * a.qcs + (size_t)min (qrow, a.S - 1) * a.qhs + hh * 8;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
      qf[kt] = __builtin_bit_cast (v8, vkl::ldg4 (qp + kt * 16));
  }

  Tile<HD> tl;
  // One pass over the keys with a running maximum: the accumulated products
  // and the sum of exponentials are rescaled whenever the maximum grows, and
  // the division by the sum comes last.
  // (the sink is a key that every query has seen before the first tile; the sums of
  // the two lane halves are added at the end, one of them has it)
  // (a tile may hold no key of a query's chunk: its first maximum lies far above the
  // score of a hidden key, whose weight is then zero)
  float m = !CHUNKED ? kNeg : a.sink ? 0.f : 0.1f * kNeg, sum = CHUNKED && a.sink && hh == 0 ? 1.f : 0.f;
  float16v oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      oacc[db][r] = 0.f;
  load_k<HD> (a, kb, t0, tl);
  load_v<HD> (a, vb, t0, tl);
  for (int t = t0; t < ntile; ++t)
    {
      __syncthreads ();
      store_k<HD> (tl, Ks);
      store_v<HD> (tl, Vt);
      __syncthreads ();
      if (t + 1 < ntile)
        {
          load_k<HD> (a, kb, t + 1, tl);
          load_v<HD> (a, vb, t + 1, tl);
        }
      if (t * kBKey > wave_last || (CHUNKED && t * kBKey + kBKey <= wave_low))
        continue;
      // scores of the tile's 64 keys; a key the query must not see counts as "never
      // seen"
      float sv[2][16];
      float bm = kNeg;
      const bool inner = t * kBKey + kBKey - 1 <= q0 + wave * 32 + shift // every key visible to every query of the wave
                         && (!CHUNKED || t * kBKey >= wave_high);
#pragma unroll
      for (int blk = 0; blk < 2; ++blk)
        {
          const float16v acc = score_block<HD, E> (Ks, blk, qf, lane);
          const int key0 = t * kBKey + 32 * blk + 4 * hh;
#pragma unroll
          for (int r = 0; r < 16; ++r)
            {
              const int key = key0 + 8 * (r >> 2) + (r & 3);
              const float sc = acc[r] * scale;
              sv[blk][r] = inner || (key <= qrow + shift && (!CHUNKED || key >= klow)) ? sc : kNeg;
              bm = fmaxf (bm, sv[blk][r]);
            }
        }
      // the two halves of the lanes hold different keys of the same query and
      // feed one product: they need the same maximum
      bm = fmaxf (bm, __shfl_xor (bm, 32, 64));
      const float mn = fmaxf (m, bm);
      if (__builtin_amdgcn_ballot_w64 (mn != m) != 0)
        {
          const float alpha = fast_exp (m - mn); // 0 before the first key, 1 where the maximum stays
          sum *= alpha;
#pragma unroll
          for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r)
              oacc[db][r] *= alpha;
          m = mn;
        }
      v8 pf[2][2];
#pragma unroll
      for (int blk = 0; blk < 2; ++blk)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          {
            // exp (kNeg - m) = 0.  The sum takes the weight as the product
            // below consumes it, rounded: the weights then add up to one exactly.
            const typename E::t e = (typename E::t)fast_exp (sv[blk][r] - m);
            sum += (float)e;
            pf[blk][r >> 3][r & 7] = e;
          }
#pragma unroll
      for (int db = 0; db < DB; ++db)
        {
          const uint16_t *vp = Vt + (size_t)(32 * db + lq) * LDV + 8 * hh;
#pragma unroll
          for (int blk = 0; blk < 2; ++blk)
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2)
              oacc[db] = E::mfma (*(const v8 *)(vp + 32 * blk + 16 * t2), pf[blk][t2], oacc[db]);
        }
    }
  // the other half of the lanes has summed the other keys of the same query
  sum += __shfl_xor (sum, 32, 64);
  float inv = 1.0f / sum;
  if (a.gate)
    inv = inv / (1.0f + expf (-vkl::ldg (a.gate + (size_t)min (qrow, a.S - 1) * a.gs + head)));
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      oacc[db][r] *= inv;

  if (qrow >= a.S)
    return;
  uint16_t *op = a.out + (size_t)qrow * a.ors + (size_t)head * a.ohs;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      {
        const int d = 32 * db + 8 * g + 4 * hh;
        u32x2 w;
        w.x = (uint32_t)E::bits (oacc[db][4 * g]) | ((uint32_t)E::bits (oacc[db][4 * g + 1]) << 16);
        w.y = (uint32_t)E::bits (oacc[db][4 * g + 2])
              | ((uint32_t)E::bits (oacc[db][4 * g + 3]) << 16);
        *(VKL_GLOBAL u32x2 *)(op + d) = w;
      }
}
// ---------------------------------------------------------------------------
// heads of 64 and 128 values
// ---------------------------------------------------------------------------
#define VKL_LDS __attribute__ ((address_space (3)))

// Weights grow by at most this power of two before the maximum is raised
constexpr float kRaise = 6.0f;

__device__ __forceinline__ float
max3 (float a, float b, float c)
{
  // (fmaxf would quiet its operands first)
  float r;
  asm ("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

template <class T>
__device__ __forceinline__ T
pk_max (T a, T b)
{
  T r;
  asm ("v_pk_max_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// the larger of a lane's value and of that of the lane 32 away
__device__ __forceinline__ float
max_halves (float x)
{
  const auto r = __builtin_amdgcn_permlane32_swap (__float_as_uint (x), __float_as_uint (x), false, false);
  return fmaxf (__uint_as_float (r[0]), __uint_as_float (r[1]));
}

// Results of a part of the keys: per part, head and query row the maximum (in powers of
// two), the sum of weights and HD unnormalised outputs
template <int HD>
__device__ __forceinline__ float *
part_row (const AttnArgs &a, int part, int head, int row)
{
  return a.ws + ((size_t)(part * a.H + head) * a.S + row) * (HD + 4);
}

// Tiles in LDS hold their rows as they lie, except that the 16-byte chunks of a row are
// exchanged: chunk c of key k is at slot c ^ swizzle (k).  Both kinds of reads, sixteen
// keys at one chunk (K) and four keys of 32 columns (V, transposed), then meet every bank
// once.
template <int HD>
__device__ __forceinline__ int
swizzle (int key)
{
  return HD == 128 ? ((key & 3) << 2) | ((key >> 2) & 3) : (((key >> 1) & 1) << 2) | ((key >> 2) & 3);
}

// Issue order of N products, each with PER reads, the reads of AHEAD products in front
template <int KIND, int PER, int N, int AHEAD> struct Alternate
{
  template <int I>
  static __device__ __forceinline__ void
  from ()
  {
    __builtin_amdgcn_sched_group_barrier (0x008, 1, 0);
    if constexpr (I + AHEAD < N)
      __builtin_amdgcn_sched_group_barrier (KIND, PER, 0);
    if constexpr (I + 1 < N)
      from<I + 1> ();
  }
  static __device__ __forceinline__ void
  run ()
  {
    __builtin_amdgcn_sched_group_barrier (KIND, PER * AHEAD, 0);
    from<0> ();
  }
};

// tiles of keys that the query tile from row q0 on sees
__host__ __device__ __forceinline__ int
key_tiles (const AttnArgs &a, int q0)
{
  const int shift = a.L - a.S, end = q0 + kBQ + shift;
  return ((end < a.L ? end : a.L) + kBKey - 1) / kBKey - (a.chunk ? (q0 + shift) / a.chunk * a.chunk : 0) / kBKey;
}

// parts of a query tile that sees n tiles of keys
__host__ __device__ __forceinline__ int
parts_of (const AttnArgs &a, int n)
{
  return a.span ? (n + a.span - 1) / a.span : a.parts;
}

// PAIR: two groups of four waves take every other tile of keys each, with a maximum and sums of their own, and meet in LDS
// at the end: a workgroup that has its compute unit alone then has a second wave per SIMD, which multiplies while the first
// one forms its weights.
template <int HD, class E, bool CHUNKED, bool PARTS, bool PAIR>
__global__ __launch_bounds__ (PAIR ? 2 * kThreads : kThreads, 2) void
attn_tiles_kernel (const AttnArgs a)
{
  typedef typename E::v8 v8;
  typedef typename E::t2 t2;
  constexpr int KT = HD / 16, DB = HD / 32, CPR = HD / 8, ROWB = HD * 2;
  constexpr int TILE = kBKey * ROWB;     // bytes of a K or V tile
  constexpr int RPI = 1024 / ROWB;       // keys per 1 KiB load
  constexpr int LPW = TILE / 1024 / 4;   // loads per wave and tile
  // four objects: a read of one is then not made to wait for the loads on their way into
  // another
  constexpr int GROUPS = PAIR ? 2 : 1;
  __shared__ __align__ (16) uint8_t lk0[GROUPS * TILE], lv0[GROUPS * TILE], lk1[GROUPS * TILE], lv1[GROUPS * TILE];

  int head, qt, part = 0;
  {
    int b = (int)blockIdx.x;
    if (PARTS)
      part = b / (a.ntq * a.H), b -= part * (a.ntq * a.H);
    tile_of (a, b, head, qt);
  }
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane ((threadIdx.x >> 6) & 3);
  const int group = PAIR ? __builtin_amdgcn_readfirstlane (threadIdx.x >> 8) : 0;
  const int lq = lane & 31, hh = lane >> 5;
  const int q0 = qt * kBQ;
  const int qrow = q0 + wave * 32 + lq; // this lane's query
  const int shift = a.L - a.S;          // key l is visible iff l <= qrow + shift
  const int kmax = min (a.L, q0 + kBQ + shift);
  const int wave_last = q0 + wave * 32 + 31 + shift; // last key any query of the wave sees
  // first key of the chunk of this lane's query, of the wave's first and last
  auto chunk_start = [&] (int row) { return CHUNKED && a.chunk ? (row + shift) / a.chunk * a.chunk : 0; };
  const int klow = chunk_start (qrow), wave_low = chunk_start (q0 + wave * 32);
  const int wave_high = chunk_start (q0 + wave * 32 + 31);
  int t0 = CHUNKED ? chunk_start (q0) / kBKey : 0, t1 = (kmax + kBKey - 1) / kBKey;
  if (PARTS)
    {
      const int n = t1 - t0, first = t0, parts = parts_of (a, n);
      if (part >= parts)
        return;
      t0 = first + n * part / parts, t1 = first + n * (part + 1) / parts;
    }
  const int kvh = head / a.rep;
  const uint16_t *kb = a.k + (size_t)kvh * a.kcs;
  const uint16_t *vb = a.v + (size_t)kvh * a.vcs;
  // from what the maximum is taken over to powers of two: rounded scores, or the products,
  // with this query's score factor
  float c = (E::round_scores ? 1.f : a.scale) * 1.44269504088896340736f;
  if (!E::round_scores && a.temp_coef != 0.f)
    c *= 1.0f + a.temp_coef * logf ((float)((qrow + shift + 1) / a.temp_every + 1));

  v8 qf[KT];
  {
    // the maximum is taken over the products: a negative factor goes into the query (of
    // the factor 0 all scores are 0)
    const uint32_t flip = c < 0.f ? 0x80008000u : 0u, keep = c == 0.f ? 0u : ~0u;
    c = c == 0.f ? 1.f : fabsf (c);
    const uint16_t *qp = a.q + (size_t)head * a.qcs + (size_t)min (qrow, a.S - 1) * a.qhs + hh * 8;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
      {
        uint4 w = vkl::ldg4 (qp + kt * 16);
        w.x = (w.x ^ flip) & keep, w.y = (w.y ^ flip) & keep, w.z = (w.z ^ flip) & keep, w.w = (w.w ^ flip) & keep;
        qf[kt] = __builtin_bit_cast (v8, w);
      }
  }

  // loads: instruction i of a wave covers RPI keys from (wave + 4 i) RPI on; lane l fetches
  // the chunk that belongs into slot l % CPR of its key (keys beyond the last repeat it:
  // no query sees them)
  const int lr = lane / CPR;
  auto issue = [&] (int t, uint8_t *lk, uint8_t *lv) {
#pragma unroll
    for (int i = 0; i < LPW; ++i)
      {
        const int r = (wave + 4 * i) * RPI + lr;
        const size_t key = (size_t)min (t * kBKey + r, a.L - 1);
        const int col = ((lane % CPR) ^ swizzle<HD> (r)) * 8;
        __builtin_amdgcn_global_load_lds ((const VKL_GLOBAL void *)(kb + key * a.khs + col),
                                          (VKL_LDS void *)(lk + group * TILE + (wave + 4 * i) * 1024), 16, 0, 0);
        __builtin_amdgcn_global_load_lds ((const VKL_GLOBAL void *)(vb + key * a.vhs + col),
                                          (VKL_LDS void *)(lv + group * TILE + (wave + 4 * i) * 1024), 16, 0, 0);
      }
  };
  // reads of K: key l % 32 of a block, values 16 kt + 8 (l / 32) .. + 7
  uint32_t koff[KT];
#pragma unroll
  for (int kt = 0; kt < KT; ++kt)
    koff[kt] = group * TILE + lq * ROWB + (((2 * kt + hh) ^ swizzle<HD> (lq)) << 4);
  // reads of V: of sixteen lanes four each give the columns 16 ((l / 16) % 2) .. + 15 of four
  // neighbouring keys from 8 g + 4 (l / 32) on, of which each receives one column
  uint32_t voff[DB][2];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int g = 0; g < 2; ++g)
      {
        const int key = 8 * g + 4 * hh + ((lane & 15) >> 2);
        const int chunk = 4 * db + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
        voff[db][g] = group * TILE + key * ROWB + ((chunk ^ swizzle<HD> (key)) << 4) + (lane & 1) * 8;
      }

  // (the sink is a key that every query has seen before the first tile; the sums of the
  // two lane halves are added at the end, one of them has it)
  // (a tile may hold no key that a query sees: its first maximum lies far above the score
  // of a hidden key, whose weight is then zero)
  const bool sink = CHUNKED && a.sink && part == 0 && group == 0;
  float m = sink ? 0.f : 0.1f * kNeg, sum = sink && hh == 0 ? 1.f : 0.f;
  float16v oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      oacc[db][r] = 0.f;
  // one tile, in (ks, vs); the next one goes to (kn, vn)
  auto step = [&] (int t, const uint8_t *ks, const uint8_t *vs, uint8_t *kn, uint8_t *vn) {
    // this tile has landed (the wave's part; the barrier covers the others'), and every
    // wave is done with the tile before, whose place the next one takes
    __builtin_amdgcn_s_waitcnt (0x0f70);
    __builtin_amdgcn_s_barrier ();
    __builtin_amdgcn_sched_barrier (0);
    if (t + GROUPS < t1)
      issue (t + GROUPS, kn, vn);
    if ((PAIR && t >= t1) || t * kBKey > wave_last || (CHUNKED && t * kBKey + kBKey <= wave_low))
      return;
    const bool inner = t * kBKey + kBKey - 1 <= q0 + wave * 32 + shift // every key visible to every query of the wave
                       && (!CHUNKED || t * kBKey >= wave_high);
    float16v s[2];
#pragma unroll
    for (int blk = 0; blk < 2; ++blk)
      {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          s[blk][r] = 0.f;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
          s[blk] = E::mfma (*(const v8 *)(ks + koff[kt] + blk * 32 * ROWB), qf[kt], s[blk]);
      }
    Alternate<0x100, 1, 2 * KT, 6>::run (); // reads stay six ahead of the products
    __builtin_amdgcn_sched_barrier (0);
    auto hidden = [&] (int blk, int r) {
      const int key = t * kBKey + 4 * hh + 32 * blk + 8 * (r >> 2) + (r & 3);
      return key > qrow + shift || (CHUNKED && key < klow);
    };
    float bm;
    t2 sh[2][8]; // the scores as fp16 pairs
    if constexpr (E::round_scores)
      {
#pragma unroll
        for (int blk = 0; blk < 2; ++blk)
#pragma unroll
          for (int r = 0; r < 16; r += 2)
            sh[blk][r / 2] = t2{ (typename E::t)__builtin_fmaf (s[blk][r], a.scale, 0.f),
                                 (typename E::t)__builtin_fmaf (s[blk][r + 1], a.scale, 0.f) };
        if (!inner)
          {
            const typename E::t never = -__builtin_inff ();
#pragma unroll
            for (int blk = 0; blk < 2; ++blk)
#pragma unroll
              for (int r = 0; r < 16; ++r)
                if (hidden (blk, r))
                  sh[blk][r / 2][r & 1] = never;
          }
        t2 top = sh[0][0];
#pragma unroll
        for (int i = 1; i < 16; ++i)
          top = pk_max (top, sh[i >> 3][i & 7]);
        bm = fmaxf ((float)top[0], (float)top[1]);
      }
    else
      {
        if (!inner)
          {
#pragma unroll
            for (int blk = 0; blk < 2; ++blk)
#pragma unroll
              for (int r = 0; r < 16; ++r)
                if (hidden (blk, r))
                  s[blk][r] = kNeg;
          }
        bm = kNeg;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          bm = max3 (s[0][r], s[1][r], bm);
      }
    // the two halves of the lanes hold different keys of the same query and feed one
    // product: they need the same maximum
    bm = max_halves (bm);
    const bool raise = (bm - m) * c > kRaise;
    if (__builtin_amdgcn_ballot_w64 (raise) != 0)
      {
        const float mn = raise ? bm : m;
        const float alpha = __builtin_amdgcn_exp2f ((m - mn) * c); // 0 before the first key, 1 where the maximum stays
        sum *= alpha;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            oacc[db][r] *= alpha;
        m = mn;
      }
    const float mc = m * c;
    v8 pf[2][2];
#pragma unroll
    for (int blk = 0; blk < 2; ++blk)
#pragma unroll
      for (int r = 0; r < 16; r += 2)
        {
          typedef float f32x2 __attribute__ ((ext_vector_type (2)));
          const float s0 = E::round_scores ? (float)sh[blk][r / 2][0] : s[blk][r];
          const float s1 = E::round_scores ? (float)sh[blk][r / 2][1] : s[blk][r + 1];
          const f32x2 e = { __builtin_amdgcn_exp2f (__builtin_fmaf (s0, c, -mc)),
                            __builtin_amdgcn_exp2f (__builtin_fmaf (s1, c, -mc)) };
          // the sum takes the weights as the product below consumes them, rounded: they
          // then add up to one exactly
          const t2 w = __builtin_convertvector (e, t2);
          sum = E::add2 (w, sum);
          pf[blk][r >> 3][r & 7] = w[0], pf[blk][r >> 3][(r & 7) + 1] = w[1];
        }
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int blk = 0; blk < 2; ++blk)
#pragma unroll
        for (int t2i = 0; t2i < 2; ++t2i)
          {
            typedef short i16x4 __attribute__ ((ext_vector_type (4)));
            typedef short i16x8 __attribute__ ((ext_vector_type (8)));
            const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16 (
                (VKL_LDS i16x4 *)(vs + voff[db][0] + (32 * blk + 16 * t2i) * ROWB));
            const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16 (
                (VKL_LDS i16x4 *)(vs + voff[db][1] + (32 * blk + 16 * t2i) * ROWB));
            const i16x8 v = __builtin_shufflevector (lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            oacc[db] = E::mfma (__builtin_bit_cast (v8, v), pf[blk][t2i], oacc[db]);
          }
    Alternate<0x100, 2, 4 * DB, 4>::run ();
    __builtin_amdgcn_sched_barrier (0);
  };
  if (t0 + group < t1)
    issue (t0 + group, lk0, lv0);
  // (both groups take as many steps, and barriers: the last of the second may be empty)
  for (int t = t0; t < t1; t += 2 * GROUPS)
    {
      step (t + group, lk0, lv0, lk1, lv1);
      if (t + GROUPS < t1)
        step (t + GROUPS + group, lk1, lv1, lk0, lv0);
    }
  // the other half of the lanes has summed the other keys of the same query
  sum += __shfl_xor (sum, 32, 64);
  if constexpr (PAIR)
    {
      typedef float f32x4 __attribute__ ((ext_vector_type (4)));
      typedef float f32x2 __attribute__ ((ext_vector_type (2)));
      static_assert (DB * 4 * 1024 + 512 <= GROUPS * TILE, "");
      __syncthreads (); // every wave has read its last tile
      uint8_t *at = wave == 0 ? lk0 : wave == 1 ? lv0 : wave == 2 ? lk1 : lv1;
      f32x4 *ov = (f32x4 *)at + lane;
      f32x2 *st = (f32x2 *)(at + DB * 4 * 1024) + lane;
      if (group)
        {
#pragma unroll
          for (int i = 0; i < DB * 4; ++i)
            ov[i * 64] = f32x4{ oacc[i / 4][4 * (i % 4)], oacc[i / 4][4 * (i % 4) + 1], oacc[i / 4][4 * (i % 4) + 2],
                                oacc[i / 4][4 * (i % 4) + 3] };
          *st = f32x2{ m, sum };
        }
      __syncthreads ();
      if (group)
        return;
      const f32x2 other = *st;
      const float mn = fmaxf (m, other.x);
      const float w0 = __builtin_amdgcn_exp2f ((m - mn) * c), w1 = __builtin_amdgcn_exp2f ((other.x - mn) * c);
      m = mn, sum = w0 * sum + w1 * other.y;
#pragma unroll
      for (int i = 0; i < DB * 4; ++i)
        {
          const f32x4 x = ov[i * 64];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            oacc[i / 4][4 * (i % 4) + e] = w0 * oacc[i / 4][4 * (i % 4) + e] + w1 * x[e];
        }
    }
  if (PARTS)
    {
      if (qrow >= a.S)
        return;
      typedef float f32x4 __attribute__ ((ext_vector_type (4)));
      float *pr = part_row<HD> (a, part, head, qrow);
      if (hh == 0)
        *(VKL_GLOBAL f32x4 *)(pr + HD) = f32x4{ m * c, sum, 0.f, 0.f };
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *(VKL_GLOBAL f32x4 *)(pr + 32 * db + 8 * g + 4 * hh)
              = f32x4{ oacc[db][4 * g], oacc[db][4 * g + 1], oacc[db][4 * g + 2], oacc[db][4 * g + 3] };
      return;
    }
  float inv = 1.0f / sum;
  if (a.gate)
    inv = inv / (1.0f + expf (-vkl::ldg (a.gate + (size_t)min (qrow, a.S - 1) * a.gs + head)));
  if (qrow >= a.S)
    return;
  uint16_t *op = a.out + (size_t)qrow * a.ors + (size_t)head * a.ohs;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      {
        const int d = 32 * db + 8 * g + 4 * hh;
        u32x2 w;
        w.x = (uint32_t)E::bits (oacc[db][4 * g] * inv) | ((uint32_t)E::bits (oacc[db][4 * g + 1] * inv) << 16);
        w.y = (uint32_t)E::bits (oacc[db][4 * g + 2] * inv) | ((uint32_t)E::bits (oacc[db][4 * g + 3] * inv) << 16);
        *(VKL_GLOBAL u32x2 *)(op + d) = w;
      }
}

// Adds the parts of the keys up: HD / 8 lanes per query row and head, eight values each.  Bound by latency: the maxima and
// sums and the values of four parts are requested at once (a wave per row with a trip to memory for each part took
// 2 to 3 us longer: 16 heads, 1500 rows behind 600 keys, both launches 43.8 / 41.0; 32 heads, one row behind 2047 14.9 / 12.4, 77
// behind 1500 18.7 / 17.7).
template <int HD, class E>
__global__ __launch_bounds__ (256) void
attn_parts_kernel (const AttnArgs a)
{
  typedef float f32x4 __attribute__ ((ext_vector_type (4)));
  constexpr int LPR = HD / 8, SPL = 16 / LPR; // lanes of a row; parts whose maxima a lane looks at
  const int i = (int)((blockIdx.x * 256 + threadIdx.x) / LPR), sub = (int)threadIdx.x % LPR;
  const int head = i % a.H, row = min (i / a.H, a.S - 1);
  const int parts = parts_of (a, key_tiles (a, row / kBQ * kBQ));
  f32x4 x[4][2];
  auto request = [&] (int p0) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      {
        const float *pr = part_row<HD> (a, min (p0 + j, parts - 1), head, row) + sub * 8;
        x[j][0] = *(const VKL_GLOBAL f32x4 *)pr, x[j][1] = *(const VKL_GLOBAL f32x4 *)(pr + 4);
      }
  };
  float pm[SPL], ps[SPL];
#pragma unroll
  for (int k = 0; k < SPL; ++k)
    {
      const float *pr = part_row<HD> (a, min (sub + k * LPR, parts - 1), head, row);
      pm[k] = vkl::ldg (pr + HD), ps[k] = vkl::ldg (pr + HD + 1);
    }
  request (0);
  float gate = 0.f;
  if (a.gate)
    gate = vkl::ldg (a.gate + (size_t)row * a.gs + head);
  float top = -3.0e38f;
#pragma unroll
  for (int k = 0; k < SPL; ++k)
    {
      pm[k] = sub + k * LPR < parts ? pm[k] : -3.0e38f;
      top = fmaxf (top, pm[k]);
    }
#pragma unroll
  for (int d = LPR / 2; d > 0; d >>= 1)
    top = fmaxf (top, __shfl_xor (top, d, 64));
  float w[SPL], total = 0.f;
#pragma unroll
  for (int k = 0; k < SPL; ++k)
    {
      const bool in = sub + k * LPR < parts;
      w[k] = in ? __builtin_amdgcn_exp2f (pm[k] - top) : 0.f;
      total += in ? w[k] * ps[k] : 0.f;
    }
#pragma unroll
  for (int d = LPR / 2; d > 0; d >>= 1)
    total += __shfl_xor (total, d, 64);
  float o[8];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    o[e] = 0.f;
  const int base = ((int)threadIdx.x & 63) - sub;
  for (int p0 = 0; p0 < a.parts; p0 += 4) // (a.parts: the most of any row)
    {
      if (p0 > 0)
        request (p0);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        {
          const int p = p0 + j;
          const float wp = __shfl (SPL == 2 && p >= LPR ? w[SPL - 1] : w[0], base + p % LPR, 64);
#pragma unroll
          for (int e = 0; e < 8; ++e)
            o[e] = p < parts ? __builtin_fmaf (wp, x[j][e >> 2][e & 3], o[e]) : o[e];
        }
    }
  if (i / a.H >= a.S)
    return;
  float inv = 1.0f / total;
  if (a.gate)
    inv = inv / (1.0f + expf (-gate));
  uint16_t *op = a.out + (size_t)row * a.ors + (size_t)head * a.ohs + sub * 8;
#pragma unroll
  for (int h = 0; h < 2; ++h)
    {
      u32x2 v;
      v.x = (uint32_t)E::bits (o[4 * h] * inv) | ((uint32_t)E::bits (o[4 * h + 1] * inv) << 16);
      v.y = (uint32_t)E::bits (o[4 * h + 2] * inv) | ((uint32_t)E::bits (o[4 * h + 3] * inv) << 16);
      *(VKL_GLOBAL u32x2 *)(op + 4 * h) = v;
    }
}

// Into how many parts the keys go, where two workgroups fit a compute unit and fewer than
// half of those would exist: the number with the lowest estimated time, from a model fitted
// to measurements at 8 to 40 heads, 1 to 900 query rows and 32 to 4000 keys (microseconds:
// a tile of the longest row takes 1.15; parts cost a second launch and 0.45 per MB that they
// write and it reads).  Measured, one part / as chosen: 32 heads of 128, 77 rows behind 1500
// keys 34 / 18, 10 rows behind 4000 83 / 22, 200 behind 1800 40 / 27; 384 rows of their own
// stay in one part (12; in two 20).  What counts are the keys that a query tile sees, from the
// start of its first row's chunk on; where a chunk ends inside the query tile, every tile of
// keys is masked and takes 2 (128 rows behind 8000 keys, 16 heads, chunks of 512: 13 us, 22 in the
// sixteen parts of 8128 keys; 32 heads, 128 rows behind 1000: 17, in one part 21).
// What one part takes is that of workgroups of four waves.  Two groups of waves (tile_pairs), which such a launch of ten tiles and
// more has, take some 2 + 1.02 per tile; the model does not know them, since tests/test_attention_spans.py holds the parts to
// those that it gives.  us, as chosen / in one part: 16 heads of 128, 1500 rows behind 300 keys 36.1 / 34.4, 600 38.3 / 36.6, 1200
// 45.3 / 46.1, 2400 62.3 / 63.1, 1024 behind 1024 36.6 / 34.6; 8 heads, 1500 behind 600 31.3 / 34.7; 32 heads, 200 behind 600 19.0 /
// 18.3; 16 heads of 64, 1500 behind 600 (two parts) 32.3 / 25.2.
int
key_parts (const AttnArgs &a, int hd)
{
  const int groups = a.ntq * a.H, shift = a.L - a.S;
  if (2 * groups > 512)
    return 1;
  int most = 0; // tiles of keys of a query tile
  double longest = 0;
  for (int q0 = 0; q0 < a.S; q0 += kBQ)
    {
      const int first = q0 + shift, last = std::min (a.S, q0 + kBQ) - 1 + shift;
      const int tiles = last / kBKey - (a.chunk ? first / a.chunk * a.chunk : 0) / kBKey + 1;
      most = std::max (most, tiles);
      longest = std::max (longest, tiles * (a.chunk && first / a.chunk != last / a.chunk ? 2.0 : 1.15));
    }
  const double mb = (double)a.H * a.S * (hd + 4) * sizeof (float) * 1e-6;
  int best = 1;
  double least = longest;
  for (int p = 2; p <= 16 && p * groups <= 512 && p <= most; ++p)
    {
      const double cost = 5 + longest / p + 0.45 * mb * p;
      if (cost < least)
        best = p, least = cost;
    }
  return best;
}

// How many tiles of keys a part gets where query tiles get different numbers of parts (0: all
// get the same).  Where two parts each leave a quarter of the 512 places empty or more (up to 200
// groups), the longest rows get three: the smallest span that needs no more than 500 places
// (of 512, as of 528, some cases took the time of three workgroups on a compute unit) and
// three parts.  A compute unit takes 1.1 us per tile however many workgroups it holds, and two
// long halves on one are what a launch waits for.  16 heads of 128, 1500 rows behind 300 / 600 /
// 1200 / 2400 keys, us: in two 42 / 46 / 55 / 72, as here 37 / 40 / 48 / 66.
// Over 700 shapes of 163 (fewer groups do not get two parts) to 255 groups, time as here / in two:
// heads that are dealt to XCDs (multiples of 8), 171 to 200 groups: 8 heads 0.86-0.96, 16 0.85-0.94,
// 24 0.93-0.97, 32 0.93-0.97, 40 0.93-0.99, but 48 1.05-1.09, 64 0.97-1.01, 88 and 96 1.09-1.19.
// Other numbers of heads: workgroups go to XCDs in turn, and what third parts add does not reach
// all alike.  With up to 440 places (55 of an XCD's 64) it was 0.74-0.93 for up to 5 heads, 0.78-1.02
// for more in up to 183 groups; 6 and 17 heads in 186 and 187 up to 1.11, 12 heads in 444 places
// 1.05, in 480 places and 198 groups up to 1.19 (18 heads, 1408 rows behind 1200), 192 groups (a
// tile's parts on one XCD) 1.07-1.26.  With more than 200 groups it was 0.81 to 1.15 (240 groups of 8
// heads 0.82-0.99, of 16 0.90-1.15): even parts.
int
key_span (const AttnArgs &a)
{
  const int groups = a.ntq * a.H;
  const bool dealt = a.H % 8 == 0;
  if (a.parts != 2 || groups > (dealt || a.H <= 5 ? 200 : 183) || (dealt ? a.H > 40 : groups % 8 == 0))
    return 0;
  int most = 0;
  for (int q0 = 0; q0 < a.S; q0 += kBQ)
    most = std::max (most, key_tiles (a, q0));
  for (int span = (most + 2) / 3; 2 * span < most; ++span)
    {
      int places = 0;
      for (int q0 = 0; q0 < a.S; q0 += kBQ)
        places += (key_tiles (a, q0) + span - 1) / span * a.H;
      if (places <= (dealt ? 500 : 440))
        return span;
    }
  return 0;
}

// parts of the keys (at most, with a span) and the span
void
plan_parts (AttnArgs &a, int hd)
{
  a.parts = key_parts (a, hd);
  const size_t part = (size_t)a.H * a.S * (hd + 4) * sizeof (float);
  if ((a.span = hd == 128 && 3 * part <= vkl::StreamScratch::bytes () ? key_span (a) : 0))
    a.parts = 3;
}

// Whether the workgroups of a launch in one part, each of which has a compute unit alone, are of two groups of waves: from ten
// tiles of keys on, where half of the tiles saves more than the meeting at the end costs (2 us).  us, four waves / eight: 16 heads of 128, 450 rows
// 13.0 / 13.1, 640 16.7 / 16.2, 1000 23.1 / 20.5, 1500 32.7 / 27.5, 2048 43.5 / 35.7; 32 heads, 768 rows 19.7 / 18.6, 1024 24.4 / 22.1; 16
// heads of 64, 700 rows 12.7 / 11.1; 128 rows 7.1 / 9.2.
constexpr int kPairTiles = 10;

bool
tile_pairs (const AttnArgs &a)
{
  int most = 0;
  for (int q0 = 0; q0 < a.S; q0 += kBQ)
    most = std::max (most, key_tiles (a, q0));
  return a.ntq * a.H <= 256 && most >= kPairTiles;
}

template <int HD, class E, bool CHUNKED>
int
launch_tiles (AttnArgs a, hipStream_t s)
{
  plan_parts (a, HD);
  const size_t part = (size_t)a.H * a.S * (HD + 4) * sizeof (float);
  vkl::StreamScratch own;
  if (a.parts > 1)
    {
      // scratch of the stream, not allocated while the stream is captured
      hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
      if (hipStreamIsCapturing (s, &capture) != hipSuccess)
        (void)hipGetLastError (); // (the default stream while another one is captured)
      else if (capture == hipStreamCaptureStatusNone
               && a.parts * part <= vkl::StreamScratch::bytes ())
        a.ws = own.take (s);
    }
  const int groups = a.ntq * a.H;
  if (!a.ws)
    {
      a.parts = 1, a.span = 0;
      if (tile_pairs (a))
        attn_tiles_kernel<HD, E, CHUNKED, false, true><<<dim3 ((unsigned)groups), dim3 (2 * kThreads), 0, s>>> (a);
      else
        attn_tiles_kernel<HD, E, CHUNKED, false, false><<<dim3 ((unsigned)groups), dim3 (kThreads), 0, s>>> (a);
      return vkl_launch_status ();
    }
  attn_tiles_kernel<HD, E, CHUNKED, true, false><<<dim3 ((unsigned)(groups * a.parts)), dim3 (kThreads), 0, s>>> (a);
  attn_parts_kernel<HD, E><<<dim3 ((unsigned)(((size_t)a.S * a.H * (HD / 8) + 255) / 256)), dim3 (256), 0, s>>> (a);
  return vkl_launch_status ();
}

// ---------------------------------------------------------------------------
// RoPE of Q and K and the K/V cache write, straight from the [S, H*hd]
// outputs of the projections: one thread per 8 consecutive elements of a
// (row, head).  Q is rotated in place (the attention kernel reads it with a
// row stride of H*hd), the rotated K and V go to cache rows (k_pos0 + s) %
// maxlen of their head.  Arithmetic of one pair as in the RoPE operator:
// (a, b) -> (fp16(a c - b s), fp16(a s + b c)) with fp32 tables.
// ---------------------------------------------------------------------------
struct RopeKvArgs
{
  uint16_t *q;
  const uint16_t *k, *v;
  uint16_t *kcache, *vcache;
  const float *fc, *fs;
  int S, H, hd, maxlen;
  int q_row0, q_rows;       // rows of q that are rotated, and their positions
  uint32_t q_pos0, k_pos0;  // q row q_row0 + i is at q_pos0 + i; k row s at k_pos0 + s
  size_t rs;                // row stride of q, k, v (elements)
};

__device__ __forceinline__ uint4
rotate8 (const uint4 x, const float *fc, const float *fs)
{
  const uint4 c4 = vkl::ldg4 (fc), s4 = vkl::ldg4 (fs);
  const float c[4] = { __uint_as_float (c4.x), __uint_as_float (c4.y), __uint_as_float (c4.z),
                       __uint_as_float (c4.w) };
  const float sn[4] = { __uint_as_float (s4.x), __uint_as_float (s4.y), __uint_as_float (s4.z),
                        __uint_as_float (s4.w) };
  const uint32_t w[4] = { x.x, x.y, x.z, x.w };
  uint32_t o[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    {
      const float a = vkl::h2f ((uint16_t)(w[j] & 0xffff)), b = vkl::h2f ((uint16_t)(w[j] >> 16));
      const float r0 = a * c[j] - b * sn[j];
      const float r1 = a * sn[j] + b * c[j];
      o[j] = (uint32_t)vkl::f2h (r0) | ((uint32_t)vkl::f2h (r1) << 16);
    }
  return make_uint4 (o[0], o[1], o[2], o[3]);
}

__global__ __launch_bounds__ (256) void
rope_kvwrite_kernel (const RopeKvArgs a, size_t total)
{
  const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= total)
    return;
  const int cpr = a.hd / 8;
  const int c = (int)(t % cpr);
  const int h = (int)((t / cpr) % a.H);
  const int s = (int)(t / ((size_t)cpr * a.H));
  const size_t src = (size_t)s * a.rs + (size_t)h * a.hd + c * 8;
  const int half = a.hd / 2;
  const uint32_t kpos = a.k_pos0 + (uint32_t)s;
  const size_t dst = ((size_t)h * a.maxlen + kpos % (uint32_t)a.maxlen) * a.hd + c * 8;
  const uint4 kr = rotate8 (vkl::ldg4 (a.k + src), a.fc + (size_t)kpos * half + c * 4,
                            a.fs + (size_t)kpos * half + c * 4);
  *(uint4 *)(a.kcache + dst) = kr;
  *(uint4 *)(a.vcache + dst) = vkl::ldg4 (a.v + src);
  if (s >= a.q_row0 && s < a.q_row0 + a.q_rows)
    {
      const uint32_t qpos = a.q_pos0 + (uint32_t)(s - a.q_row0);
      *(uint4 *)(a.q + src) = rotate8 (vkl::ldg4 (a.q + src), a.fc + (size_t)qpos * half + c * 4,
                                       a.fs + (size_t)qpos * half + c * 4);
    }
}
} // namespace

extern "C" int
vkl_rope_kvwrite_f16 (void *q, const void *k, const void *v, int S, int H,
                      int hd, size_t row_stride, int q_row0, int q_rows,
                      uint32_t q_pos0, uint32_t k_pos0, const float *freqc,
                      const float *freqs, int table_rows, void *kcache,
                      void *vcache, int maxlen, void *stream)
{
  VKL_CHECK_ARG (q && k && v && freqc && freqs && kcache && vcache);
  VKL_CHECK_ARG (S > 0 && H > 0 && hd > 0 && (hd % 8) == 0 && maxlen > 0 && S <= maxlen);
  VKL_CHECK_ARG (q_row0 >= 0 && q_rows >= 0 && q_row0 + q_rows <= S);
  // every position must have a row in the cos / sin tables
  VKL_CHECK_ARG ((size_t)k_pos0 + S <= (size_t)table_rows
                 && (size_t)q_pos0 + q_rows <= (size_t)table_rows);
  VKL_CHECK_ARG ((row_stride % 8) == 0 && row_stride >= (size_t)H * hd);
  VKL_CHECK_ARG (((uintptr_t)q % 16) == 0 && ((uintptr_t)k % 16) == 0 && ((uintptr_t)v % 16) == 0
                 && ((uintptr_t)kcache % 16) == 0 && ((uintptr_t)vcache % 16) == 0
                 && ((uintptr_t)freqc % 16) == 0 && ((uintptr_t)freqs % 16) == 0);
  RopeKvArgs a;
  a.q = (uint16_t *)q, a.k = (const uint16_t *)k, a.v = (const uint16_t *)v;
  a.kcache = (uint16_t *)kcache, a.vcache = (uint16_t *)vcache;
  a.fc = freqc, a.fs = freqs;
  a.S = S, a.H = H, a.hd = hd, a.maxlen = maxlen;
  a.q_row0 = q_row0, a.q_rows = q_rows, a.q_pos0 = q_pos0, a.k_pos0 = k_pos0;
  a.rs = row_stride;
  const size_t total = (size_t)S * H * (hd / 8);
  rope_kvwrite_kernel<<<dim3 ((unsigned)((total + 255) / 256)), dim3 (256), 0, (hipStream_t)stream>>> (
      a, total);
  return vkl_launch_status ();
}

extern "C" int
vkl_attn_prefill_causal_f16 (const void *q, const void *k, const void *v,
                             int H, int S, int L, int hd, size_t qcs,
                             size_t qhs, size_t kcs, size_t khs, size_t vcs,
                             size_t vhs, float scale, void *out, size_t ors,
                             size_t ohs, void *stream)
{
  VKL_CHECK_ARG (q && k && v && out);
  VKL_CHECK_ARG (H > 0 && S > 0 && L >= S);
  VKL_CHECK_ARG (hd == 64 || hd == 128);
  // 16-byte vector loads, 8-byte stores
  VKL_CHECK_ARG (((uintptr_t)q % 16) == 0 && ((uintptr_t)k % 16) == 0 && ((uintptr_t)v % 16) == 0
                 && ((uintptr_t)out % 8) == 0);
  VKL_CHECK_ARG ((qcs % 8) == 0 && (qhs % 8) == 0 && (kcs % 8) == 0 && (khs % 8) == 0
                 && (vcs % 8) == 0 && (vhs % 8) == 0 && (ors % 4) == 0 && (ohs % 4) == 0);
  AttnArgs a = {};
  a.rep = 1;
  a.q = (const uint16_t *)q, a.k = (const uint16_t *)k, a.v = (const uint16_t *)v;
  a.out = (uint16_t *)out;
  a.H = H, a.S = S, a.L = L, a.ntq = (S + kBQ - 1) / kBQ;
  a.qcs = qcs, a.qhs = qhs, a.kcs = kcs, a.khs = khs, a.vcs = vcs, a.vhs = vhs;
  a.ors = ors, a.ohs = ohs, a.scale = scale;
  return hd == 128 ? launch_tiles<128, F16Elem, false> (a, (hipStream_t)stream)
                   : launch_tiles<64, F16Elem, false> (a, (hipStream_t)stream);
}

namespace
{
template <bool CHUNKED>
int
launch_prefill_bf16 (const AttnArgs &a, int hd, hipStream_t s)
{
  const dim3 grid ((unsigned)(a.ntq * a.H)), block (kThreads);
  switch (hd)
    {
    case 32: attn_prefill_kernel<32, Bf16Elem, CHUNKED><<<grid, block, 0, s>>> (a); break;
    case 64: return launch_tiles<64, Bf16Elem, CHUNKED> (a, s);
    case 96: attn_prefill_kernel<96, Bf16Elem, CHUNKED><<<grid, block, 0, s>>> (a); break;
    case 128: return launch_tiles<128, Bf16Elem, CHUNKED> (a, s);
    case 160: attn_prefill_kernel<160, Bf16Elem, CHUNKED><<<grid, block, 0, s>>> (a); break;
    case 192: attn_prefill_kernel<192, Bf16Elem, CHUNKED><<<grid, block, 0, s>>> (a); break;
    case 224: attn_prefill_kernel<224, Bf16Elem, CHUNKED><<<grid, block, 0, s>>> (a); break;
    default: attn_prefill_kernel<256, Bf16Elem, CHUNKED><<<grid, block, 0, s>>> (a); break;
    }
  return vkl_launch_status ();
}

int
prefill_args_bf16 (AttnArgs &a, const void *q, const void *k, const void *v, int H, int G, int S, int L, int hd,
                   size_t qhs, size_t khs, size_t vhs, float scale, void *out, size_t ors)
{
  VKL_CHECK_ARG (q && k && v && out);
  VKL_CHECK_ARG (H > 0 && G > 0 && (H % G) == 0 && S > 0 && L >= S);
  VKL_CHECK_ARG (hd > 0 && (hd % 32) == 0 && hd <= 256);
  VKL_CHECK_ARG (((uintptr_t)q % 16) == 0 && ((uintptr_t)k % 16) == 0 && ((uintptr_t)v % 16) == 0
                 && ((uintptr_t)out % 8) == 0);
  VKL_CHECK_ARG ((qhs % 8) == 0 && (khs % 8) == 0 && (vhs % 8) == 0 && (ors % 4) == 0);
  VKL_CHECK_ARG (qhs >= (size_t)H * hd && khs >= (size_t)G * hd && vhs >= (size_t)G * hd && ors >= (size_t)H * hd);
  a.q = (const uint16_t *)q, a.k = (const uint16_t *)k, a.v = (const uint16_t *)v;
  a.out = (uint16_t *)out;
  a.H = H, a.S = S, a.L = L, a.ntq = (S + kBQ - 1) / kBQ;
  a.qcs = a.kcs = a.vcs = a.ohs = (size_t)hd;
  a.qhs = qhs, a.khs = khs, a.vhs = vhs, a.ors = ors;
  a.scale = scale, a.rep = H / G;
  return 0;
}
} // namespace

extern "C" int
vkl_attn_prefill_parts (int H, int S, int L, int hd, int chunk)
{
  if (H <= 0 || S <= 0 || L < S || chunk < 0 || (hd != 64 && hd != 128))
    return 1;
  AttnArgs a = {};
  a.H = H, a.S = S, a.L = L, a.ntq = (S + kBQ - 1) / kBQ, a.chunk = chunk;
  plan_parts (a, hd);
  return a.parts;
}

extern "C" int
vkl_attn_prefill_tile_parts (int H, int S, int L, int hd, int chunk, int row)
{
  if (H <= 0 || S <= 0 || L < S || chunk < 0 || (hd != 64 && hd != 128) || row < 0 || row >= S)
    return 1;
  AttnArgs a = {};
  a.H = H, a.S = S, a.L = L, a.ntq = (S + kBQ - 1) / kBQ, a.chunk = chunk;
  plan_parts (a, hd);
  return parts_of (a, key_tiles (a, row / kBQ * kBQ));
}

extern "C" int
vkl_attn_prefill_causal_bf16 (const void *q, const void *k, const void *v, int H, int G, int S, int L, int hd,
                              size_t qhs, size_t khs, size_t vhs, float scale, float temp_coef,
                              int temp_every, const float *gate, size_t gs, void *out, size_t ors,
                              void *stream)
{
  AttnArgs a = {};
  if (int e = prefill_args_bf16 (a, q, k, v, H, G, S, L, hd, qhs, khs, vhs, scale, out, ors))
    return e;
  VKL_CHECK_ARG ((temp_coef == 0.f || temp_every > 0) && (!gate || gs >= (size_t)H));
  a.temp_coef = temp_coef, a.temp_every = temp_every, a.gate = gate, a.gs = gs;
  return launch_prefill_bf16<false> (a, hd, (hipStream_t)stream);
}

extern "C" int
vkl_attn_prefill_chunked_bf16 (const void *q, const void *k, const void *v, int H, int G, int S, int L, int hd,
                               size_t qhs, size_t khs, size_t vhs, float scale, int chunk, int sink, void *out,
                               size_t ors, void *stream)
{
  AttnArgs a = {};
  if (int e = prefill_args_bf16 (a, q, k, v, H, G, S, L, hd, qhs, khs, vhs, scale, out, ors))
    return e;
  VKL_CHECK_ARG (chunk >= 0);
  a.chunk = chunk, a.sink = sink;
  return launch_prefill_bf16<true> (a, hd, (hipStream_t)stream);
}

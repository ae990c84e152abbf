// y[M,N] = x[M,K] W[N,K]^T for many token rows (prompt passes of 128 tokens
// and more), fp16 activations and dense fp16 or planar Q8_0 weights, fp32
// accumulation on the matrix cores; bf16 and 32-bit activations with bf16 weights.
//
// A k-step is 64 wide, so a tile row is one 128-byte cache line.  The tiles of x and W do
// not pass through registers on their way in: global_load_lds_dwordx4 writes them
// straight into LDS, two to six k-steps deep, one 1 KiB instruction
// per 8 tile rows.  Such an instruction writes its 64 x 16 bytes to consecutive
// LDS addresses, so rows cannot be padded against bank conflicts; instead every
// lane fetches the 16-byte chunk (slot ^ f(row)) of its row, which stores the
// row XOR-swizzled, and the fragment reads apply the same f.
//
// The k loop is scheduled by hand (sched_group_barrier): products alternate with the
// fragment reads of the next part of a k-step and with a share of the loads for a later
// k-step.  The barrier that hands over the next k-step sits inside a step, whose
// remaining products then overlap with the first fragment reads of the next one.
//
// Tiles of up to 256 x 256 (gemm_mix_kernel) multiply fp16 and bf16; those of 32 x 32
// products (wide_bf16_tile) are left for 64 rows of bf16, for short tiles of more and for 32-bit operands.
#include "../../include/vkl_stack.h"
#include "vkl_stack_dev.h"
#include "vkl_common.h"
#include "vkl_gemm.h"
#include <algorithm>
#include <type_traits>
#include "vkl_gemm_finish.h"

namespace vkl
{
namespace
{
typedef _Float16 half8 __attribute__ ((ext_vector_type (8)));
typedef __bf16 bf8 __attribute__ ((ext_vector_type (8)));
typedef float float4v __attribute__ ((ext_vector_type (4)));
typedef float float16v __attribute__ ((ext_vector_type (16)));
#define VKL_LDS __attribute__ ((address_space (3)))

constexpr int WBM = 256, WBN = 128, WBK = 64;
constexpr int WSTAGES = 3;
constexpr int WWAVES = 4;                       // 2 x 2
constexpr int WTN = WBN / 2 / 32;
constexpr int WROWB = WBK * 2;                  // bytes of a tile row


// element type of the dense kernels by their argument block: fp16 for the products
// with one plain epilogue, bf16 for those with segments
template <class Args> struct WideElem
{
  typedef half8 v8;
  static __device__ __forceinline__ float4v
  mfma (v8 a, v8 b, float4v c)
  {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16 (a, b, c, 0, 0, 0);
  }
};
template <> struct WideElem<GemmSegArgs>
{
  typedef bf8 v8;
  static __device__ __forceinline__ float4v
  mfma (v8 a, v8 b, float4v c)
  {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16 (a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ float16v
  mfma (v8 a, v8 b, float16v c)
  {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16 (a, b, c, 0, 0, 0);
  }
};

// Where a workgroup's output tile lies
struct WidePlace
{
  int m0, tn, zmat, ks; // first token row, tile of weight rows, matrix, part of the k range
  int half;             // (WideMix) of a tile that is cut by its columns
};
enum WideKind
{
  WIDE_NONE,
  WIDE_TILE,
  WIDE_HALF // of half the token rows
};

// The tiles of a launch, token-row tile fastest, then weight tile, matrix, part of the k
// range.  Workgroups go to the XCDs in turn: each XCD gets a contiguous range of tiles,
// so the weight tiles that they share stay in its L2.
//
// Tiles beyond the last whole round over the 256 compute units are cut in two where they
// fill at most half of a round: a round of 128-row tiles takes 0.6 of one of 256-row
// tiles.  Measured, us whole / cut: Q8_0 at 2048 rows 5120 x 5120 (1.25 rounds) 199 / 173,
// 5120 x 13824 506 / 429, at 3967 rows (2.5 rounds) 847 / 803, up/gate 13824 x 5120 (13.5)
// 1597 / 1556, at 512 rows up/gate 11008 x 4096 (1.34) 160 / 136; bf16 at 2048 rows 12544 x
// 4096 (3.06) 223 / 215.
struct WideGrid
{
  int tiles_m, tiles_n, nmat, ksplit;
  int whole; // tiles that are not cut

  static constexpr int kUnits = 256;
  __host__ __device__ int
  tiles () const
  {
    return tiles_m * tiles_n * nmat * ksplit;
  }
  __host__ WideGrid (int tm, int tn, int mats, int parts, bool cut)
      : tiles_m (tm), tiles_n (tn), nmat (mats), ksplit (parts)
  {
    const int rest = tiles () % kUnits;
    whole = cut && rest > 0 && rest <= kUnits / 2 ? tiles () - rest : tiles ();
  }
  // workgroups to launch: multiples of 8 of either kind
  __host__ __device__ int
  whole_groups () const
  {
    return (whole + 7) / 8 * 8;
  }
  __host__ int
  groups () const
  {
    return whole_groups () + (2 * (tiles () - whole) + 7) / 8 * 8;
  }
  template <int BM>
  __device__ __forceinline__ WideKind
  place (int M, WidePlace &at) const
  {
    const int first = whole_groups (), id = (int)blockIdx.x;
    const bool cut = id >= first;
    const int g = cut ? id - first : id, count = cut ? 2 * (tiles () - whole) : whole;
    const int per_xcd = (count + 7) / 8, j = g >> 3;
    const int i = (g & 7) * per_xcd + j;
    if (j >= per_xcd || i >= count)
      return WIDE_NONE;
    int t = cut ? whole + (i >> 1) : i;
    const int tm = t % tiles_m;
    t /= tiles_m;
    at.tn = t % tiles_n;
    t /= tiles_n;
    at.zmat = t % nmat;
    at.ks = t / nmat;
    at.m0 = tm * BM + (cut ? (i & 1) * (BM / 2) : 0);
    if (at.m0 >= M)
      return WIDE_NONE; // the empty half of the last tile
    return cut ? WIDE_HALF : WIDE_TILE;
  }
};

// Issue order of one quarter of a k-step: after product Q one fragment read
// (the first NR products) and an even share of the quarter's LQ loads.
template <int Q, int NP, int NR, int LQ> struct WideOrder
{
  static __device__ __forceinline__ void
  run ()
  {
    __builtin_amdgcn_sched_group_barrier (0x008, 1, 0); // one MFMA
    if constexpr (Q < NR)
      __builtin_amdgcn_sched_group_barrier (0x100, 1, 0); // one LDS read
    constexpr int nl = LQ * (Q + 1) / NP - LQ * Q / NP;
    if constexpr (nl > 0)
      __builtin_amdgcn_sched_group_barrier (0x020, nl, 0); // loads
    if constexpr (Q + 1 < NP)
      WideOrder<Q + 1, NP, NR, LQ>::run ();
  }
};

template <int V> struct WideInt
{
  static constexpr int value = V;
};

// The k-steps of a tile of ST stages whose loads are issued D steps ahead: step (kt, stage, left) for
// kt = 0 .. nk - 1.  left: how many k-steps stand behind it, D for D and more, where it issues the loads of
// kt + D; the last D steps issue none, so that no tile waits for loads that nothing reads (with stages
// for a whole compute unit, see deep64, us before / now, weights that no cache holds: 300 x 2048 x 2048
// 32-bit 28.2 / 25.8, 500 x 3072 x 2048 39.3 / 32.8, 128 x 8192 x 2048 bf16 18.2 / 17.0).  Their stage is
// a variable, which spares copies of them.
template <int D, int ST, int I = 0, class F>
__device__ __forceinline__ void
wide_steps_some (int kt, int n, F &step)
{
  if constexpr (I < ST)
    if (I < n)
      {
        step (kt + I, I, WideInt<D> ());
        wide_steps_some<D, ST, I + 1> (kt, n, step);
      }
}
template <int D, int ST, int I = 0, class F>
__device__ __forceinline__ void
wide_steps_round (int kt, F &step)
{
  if constexpr (I < ST)
    {
      step (kt + I, I, WideInt<D> ());
      wide_steps_round<D, ST, I + 1> (kt, step);
    }
}
template <int D, int ST, int LEFT, class F>
__device__ __forceinline__ void
wide_steps_last (int nk, int st, F &step)
{
  if (nk > LEFT)
    {
      step (nk - 1 - LEFT, st, WideInt<LEFT> ());
      st = st == ST - 1 ? 0 : st + 1;
    }
  if constexpr (LEFT > 0)
    wide_steps_last<D, ST, LEFT - 1> (nk, st, step);
}
// every one as if D stood behind it, for tiles without the registers for more copies of a step
template <int D, int ST, class F>
__device__ __forceinline__ void
wide_steps_alike (int nk, F &step)
{
  int kt = 0;
  for (; kt + ST <= nk; kt += ST)
    wide_steps_round<D, ST> (kt, step);
  wide_steps_some<D, ST> (kt, nk - kt, step);
}
template <int D, int ST, class F>
__device__ __forceinline__ void
wide_steps (int nk, F &step)
{
  int kt = 0;
  for (; kt + ST <= nk - D; kt += ST)
    wide_steps_round<D, ST> (kt, step);
  const int n = nk - D - kt > 0 ? nk - D - kt : 0; // 0 .. ST - 1
  wide_steps_some<D, ST> (kt, n, step);
  wide_steps_last<D, ST, D - 1> (nk, n, step);
}

// waits until at most V loads are in flight; LDS: and the wave's own LDS reads are back
template <int V, bool LDS>
__device__ __forceinline__ void
wait_loads ()
{
  constexpr int imm = (LDS ? 0x0070 : 0x0f70) | (V & 15) | ((V >> 4) << 14);
  __builtin_amdgcn_s_waitcnt (imm);
}

// Behind the k loop of every tile: no load may outlive the workgroup's LDS, and none may land where sums are
// parked.  A wave can wait for its own loads only, so each does so before the barrier behind which LDS is
// written by hand (tests/test_lds_loads.py follows the compiled code).  Tiles that load past the end
// (wide_steps_alike) have up to nine in flight here, the others none.
__device__ __forceinline__ void
land_all ()
{
  wait_loads<0, true> ();
}

// The products are formed transposed (the weights are the first operand): of a 32 x 32
// block lane l holds token row l%32, and register q output column 8 (q/4) + 4 (l/32) +
// q%4.  After exchanging half waves between the registers of two groups of four
// (v_permlane32_swap) a lane has eight neighbouring columns of its row.
//
// The epilogue takes that straight from the registers where it is simple: a wave's
// columns all there, in one segment, vector stores, nothing but an optional residual (or
// SiLU of the fused pair) on the way.  Everything else is parked in LDS (the k loop's
// stages are free by then) and walked row-wise in a short loop, eight neighbouring
// columns per lane.  Both are about latency and instruction fetch, with one wave per SIMD
// and code that runs once: the loop took 15 thousand cycles for a 256 x 128 tile (26 with
// segments) where the k loop takes 84 at K = 4096, and all cases unrolled as much.
// Straight, us per product at 2048 rows before / after: 4096 x 4096 fp16 71 / 66, bf16
// 69 / 60; bf16 8064 x 2048 82 / 63, 11008 x 4096 193 / 165; at 300 rows 8064 x 2048 21 / 16.
constexpr int kWideParkLd = 68; // floats per parked row: 16-byte aligned, rows 4 banks apart

// x, y -> the lower halves of both, the upper halves of both
__device__ __forceinline__ void
half_swap (float x, float y, float &lo, float &hi)
{
  const auto r = __builtin_amdgcn_permlane32_swap (__float_as_uint (x), __float_as_uint (y), false, false);
  lo = __uint_as_float (r[0]), hi = __uint_as_float (r[1]);
}

// Eight values of a simple epilogue
template <bool UPGATE, class Args> struct WideSimple;

template <bool UPGATE> struct WideSimple<UPGATE, GemmArgs>
{
  static constexpr int NR = 1; // 16-byte words of a residual
  const uint16_t *r;
  uint16_t *y;
  size_t ys;
  bool ok;

  // ncol: first of the wave's `n` columns
  __device__ __forceinline__
  WideSimple (const GemmArgs &a, int ncol, int n, int zmat, int vec, const float *part)
  {
    ok = vec && !part && ncol + n <= a.N
         && (UPGATE || a.nmat != 1 || (a.scale == 1.f && a.bias == 0.f && a.act == 0 && !a.y32));
    y = (UPGATE ? a.y[0] : pick3 (a.y[0], a.y[1], a.y[2], zmat)) + ncol, ys = a.ys;
    r = !UPGATE && a.nmat == 1 && a.residual ? a.residual + ncol : nullptr;
  }
  __device__ __forceinline__ void
  request (size_t m, int col, uint4 (&w)[NR]) const
  {
    w[0] = ldg4 (r + m * ys + col);
  }
  __device__ __forceinline__ void
  store (size_t m, int col, const float (&v)[8], const float (&g)[8], const uint4 *w) const
  {
    uint16_t h[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      h[e] = f2h (UPGATE ? silu (g[e]) * v[e] : v[e]);
    if (w)
      {
        const uint32_t rw[4] = { w->x, w->y, w->z, w->w };
#pragma unroll
        for (int e = 0; e < 8; ++e)
          h[e] = f2h (h2f (h[e]) + h2f ((uint16_t)(rw[e >> 1] >> ((e & 1) * 16))));
      }
    vkl_u32x4 pk;
    pk.x = h[0] | ((uint32_t)h[1] << 16), pk.y = h[2] | ((uint32_t)h[3] << 16);
    pk.z = h[4] | ((uint32_t)h[5] << 16), pk.w = h[6] | ((uint32_t)h[7] << 16);
    *(VKL_GLOBAL vkl_u32x4 *)(y + m * ys + col) = pk;
  }
};

template <bool UPGATE> struct WideSimple<UPGATE, GemmSegArgs>
{
  static constexpr int NR = 2;
  const float *r;
  char *y;
  size_t ys;
  int f32, relu2;
  bool ok;

  __device__ __forceinline__
  WideSimple (const GemmSegArgs &a, int ncol, int n, int, int, const float *part)
  {
    const SegCol c = seg_col (a, ncol); // (ncol is the same in all lanes)
    ok = !part && ncol + n <= a.N && c.whole && n <= c.n && c.cap <= 0.f
         && (c.act == VKL_ACT_NONE || c.act == VKL_ACT_RELU2);
    y = c.y, ys = c.ys, r = c.r, f32 = c.f32, relu2 = c.act == VKL_ACT_RELU2;
  }
  __device__ __forceinline__ void
  request (size_t m, int col, uint4 (&w)[NR]) const
  {
    w[0] = ldg4 (r + m * ys + col), w[1] = ldg4 (r + m * ys + col + 4);
  }
  __device__ __forceinline__ void
  store (size_t m, int col, float (&v)[8], const float (&)[8], const uint4 *w) const
  {
    typedef float f32x4 __attribute__ ((ext_vector_type (4)));
    if (relu2)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        v[e] = activate (VKL_ACT_RELU2, v[e]);
    if (f32)
      {
        f32x4 w0 = { v[0], v[1], v[2], v[3] }, w1 = { v[4], v[5], v[6], v[7] };
        if (w)
          w0 += __builtin_bit_cast (f32x4, w[0]), w1 += __builtin_bit_cast (f32x4, w[1]);
        float *o = (float *)y + m * ys + col;
        *(VKL_GLOBAL f32x4 *)o = w0;
        *(VKL_GLOBAL f32x4 *)(o + 4) = w1;
      }
    else
      {
        vkl_u32x4 pk;
        pk.x = f2bf (v[0]) | ((uint32_t)f2bf (v[1]) << 16), pk.y = f2bf (v[2]) | ((uint32_t)f2bf (v[3]) << 16);
        pk.z = f2bf (v[4]) | ((uint32_t)f2bf (v[5]) << 16), pk.w = f2bf (v[6]) | ((uint32_t)f2bf (v[7]) << 16);
        *(VKL_GLOBAL vkl_u32x4 *)((uint16_t *)y + m * ys + col) = pk;
      }
  }
};

// Sums of a part of the k range: eight neighbouring columns of row m from the registers to the dense rows that the
// reduction reads (rows of a multiple of eight values; others are parked).  The walk through LDS took 0.4 to 2.5 us of
// a launch, us through LDS / straight, weights that no cache holds: 600 x 2048 x 7552 38.2 / 36.7, 1500 x 2048 x 7552 64.0 /
// 61.6, 160 x 2048 x 2048 13.2 / 12.6, 32-bit 300 x 2048 x 5504 42.6 / 42.4.  (fp16 products, 77 x 4096 x 4096 and
// 11008, took the same, and keep the walk.)
__device__ __forceinline__ void
part_store8 (float *part, int M, int N, int m, int n, const float4v lo, const float4v hi)
{
  if (m >= M || n >= N)
    return;
  float *dst = part + (size_t)m * N + n;
  *(VKL_GLOBAL float4v *)dst = lo;
  *(VKL_GLOBAL float4v *)(dst + 4) = hi;
}

// TN: 32-column accumulators of a wave; mrow, ncol: the first row and output column of the
// wave's block
template <int TM, int TN>
__device__ __forceinline__ void
wide_epilogue (const GemmSegArgs &a, const float16v (&acc)[TM][TN], uint8_t *wide_lds, int wave, int lane, int mrow, int ncol,
               float *part)
{
  const WideSimple<false, GemmSegArgs> simple (a, ncol, TN * 32, 0, 1, part);
  if (simple.ok)
    {
      const int m0 = mrow + (lane & 31);
      auto walk = [&] (auto with) {
        constexpr bool RES = decltype (with)::value != 0;
        constexpr int NR = WideSimple<false, GemmSegArgs>::NR;
#pragma unroll
        for (int jn = 0; jn < TN; ++jn)
          {
            uint4 res[TM][2][NR];
            if (RES)
#pragma unroll
              for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int p = 0; p < 2; ++p)
                  simple.request ((size_t)min (m0 + i * 32, a.M - 1), jn * 32 + p * 16 + (lane >> 5) * 8, res[i][p]);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
              for (int p = 0; p < 2; ++p)
                {
                  float v[8], g[8];
#pragma unroll
                  for (int e = 0; e < 4; ++e)
                    {
                      half_swap (acc[i][jn][8 * p + e], acc[i][jn][8 * p + 4 + e], v[e], v[4 + e]);
                      g[e] = g[4 + e] = 0.f;
                    }
                  if (m0 + i * 32 < a.M)
                    simple.store ((size_t)(m0 + i * 32), jn * 32 + p * 16 + (lane >> 5) * 8, v, g, RES ? res[i][p] : nullptr);
                }
          }
      };
      if (simple.r)
        walk (WideInt<1> ());
      else
        walk (WideInt<0> ());
      return;
    }
  if (part && (a.N % 8) == 0)
    {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int jn = 0; jn < TN; ++jn)
#pragma unroll
          for (int p = 0; p < 2; ++p)
            {
              float4v lo, hi;
#pragma unroll
              for (int e = 0; e < 4; ++e)
                {
                  float x, y;
                  half_swap (acc[i][jn][8 * p + e], acc[i][jn][8 * p + 4 + e], x, y);
                  lo[e] = x, hi[e] = y;
                }
              part_store8 (part, a.M, a.N, mrow + i * 32 + (lane & 31), ncol + jn * 32 + p * 16 + (lane >> 5) * 8, lo, hi);
            }
      return;
    }
  // through LDS, 64 accumulator columns at a time
  constexpr int ROWS = TM * 32, LD = kWideParkLd;
  float *park = (float *)(wide_lds + wave * (ROWS * LD * 4));
  __builtin_amdgcn_s_barrier (); // every wave has read its last fragments
#pragma unroll
  for (int half = 0; half < TN / 2; ++half)
    {
#pragma unroll
      for (int c = 0; c < 2; ++c)
        {
          const int jn = 2 * half + c;
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int q = 0; q < 16; q += 4)
              *(float4 *)(park + (i * 32 + (lane & 31)) * LD + c * 32 + 2 * q + 4 * (lane >> 5))
                  = make_float4 (acc[i][jn][q], acc[i][jn][q + 1], acc[i][jn][q + 2], acc[i][jn][q + 3]);
        }
      // (a wave reads back only what it wrote itself: no barrier)
      constexpr int CPR = 8;                // lanes per row
      constexpr int RPI = 64 / CPR;         // rows per iteration
      const int er = lane / CPR, ec = (lane % CPR) * 8;
      const FinishRows<false, GemmSegArgs> fin (a, ncol + half * 64 + ec, 0, 1, part);
      for (int it = 0; it < ROWS / RPI; ++it)
        {
          const int row = it * RPI + er;
          uint4 res[2];
          fin.request (mrow + row, res);
          const float *pr = park + row * LD + ec;
          const float4 p0 = *(const float4 *)pr, p1 = *(const float4 *)(pr + 4);
          float v[8] = { p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w };
          const float g[8] = { 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f };
          fin.store (mrow + row, v, g, res);
        }
    }
}

// Epilogue through LDS (the k loop's stages are free by then) of the kernel for Q8_0
// weights, eight waves in a 2 x 4 grid (TM x 32 rows by 32 columns each; of the fused
// pair the waves 0, 1 of a row block hold up, 2, 3 gate): the BM x 128 tile is parked, and
// after a barrier all threads walk it row-wise, eight neighbouring columns per lane.
// Accumulator register q of lane l is row 8 (q/4) + 4 (l/32) + q%4, column l%32 of its
// 32 x 32 block.
constexpr int kWideTileLd = 132;

template <int BM, bool UPGATE, int TM>
__device__ __forceinline__ void
wide_epilogue_tile (const GemmArgs &a, const float16v (&acc)[TM][1], uint8_t *wide_lds, int wave, int lane,
                    int m0, int n0, int zmat, int vec, float *part)
{
  constexpr int LD = kWideTileLd;
  const int wm = wave >> 2, wn = wave & 3;
  __builtin_amdgcn_s_barrier (); // every wave has read its last fragments
  float *park = (float *)wide_lds;
  {
    float *pl = park + (wm * TM * 32 + (lane >> 5) * 4) * LD + wn * 32 + (lane & 31);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int q = 0; q < 16; ++q)
        pl[(i * 32 + (q >> 2) * 8 + (q & 3)) * LD] = acc[i][0][q];
  }
  __syncthreads ();
  constexpr int LPR = UPGATE ? 8 : 16;        // lanes per row
  constexpr int RPI = 8 * 64 / LPR;           // rows per iteration of the workgroup
  const int er = threadIdx.x / LPR, ec = (threadIdx.x % LPR) * 8;
  for (int it = 0; it < BM / RPI; ++it)
    {
      const int row = it * RPI + er;
      const float4 p0 = *(const float4 *)(park + row * LD + ec);
      const float4 p1 = *(const float4 *)(park + row * LD + ec + 4);
      float v[8] = { p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w };
      float g[8] = { 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f };
      if (UPGATE)
        {
          const float4 g0 = *(const float4 *)(park + row * LD + 64 + ec);
          const float4 g1 = *(const float4 *)(park + row * LD + 64 + ec + 4);
          g[0] = g0.x, g[1] = g0.y, g[2] = g0.z, g[3] = g0.w, g[4] = g1.x, g[5] = g1.y, g[6] = g1.z, g[7] = g1.w;
        }
      gemm_finish8<UPGATE> (a, v, g, m0 + row, n0 + ec, zmat, vec, part);
    }
}

template <int BM, int ST>
constexpr size_t
wide_lds_bf16 ()
{
  const size_t stages = (size_t)ST * (BM + WBN) * WROWB, park = (size_t)BM * 2 * kWideParkLd * 4;
  return stages > park ? stages : park;
}

// The planes of a 32-bit product (see there) leave a sum that is not finite where the
// product has such a value, where a weight is not finite (it meets zeros in the lower
// planes) and where split_planes_kernel marked a value that three planes do not hold.
// These sums are formed again by the 32-bit instructions, from x itself; the others stay.
// Bound by memory latency, sixteen values of k per round trip (about 45 us per block of 32 x
// 32 at K = 2048); products without such values pay 16 vector instructions per block (a
// prompt of 300 tokens, 4 layers of width 2048: 1000 -> 1004 us).
// mrow, ncol: the wave's first row and column.
template <int TM>
__device__ __forceinline__ void
wide_f32_again (const GemmSegArgs &a, float16v (&acc)[TM][WTN], int lane, int mrow, int ncol, int K)
{
  float t[TM][WTN], any = 0.f; // 0 unless one of the sums is not finite
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int jn = 0; jn < WTN; ++jn)
      {
        t[i][jn] = 0.f;
#pragma unroll
        for (int q = 0; q < 16; ++q)
          t[i][jn] = __builtin_fmaf (acc[i][jn][q], 0.f, t[i][jn]);
        any += t[i][jn];
      }
  if (__builtin_amdgcn_ballot_w64 (any != 0.f) == 0)
    return;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int jn = 0; jn < WTN; ++jn)
      {
        if (__builtin_amdgcn_ballot_w64 (t[i][jn] != 0.f) == 0)
          continue;
        const float *x = a.xf + (size_t)min (mrow + i * 32 + (lane & 31), a.M - 1) * a.xs + (lane >> 5) * 8;
        const uint16_t *w = a.wh[0] + (size_t)min (ncol + jn * 32 + (lane & 31), a.N - 1) * a.ws + (lane >> 5) * 8;
        float16v sum;
#pragma unroll
        for (int q = 0; q < 16; ++q)
          sum[q] = 0.f;
#pragma unroll 1
        for (int k = 0; k < K; k += 16)
          {
            const uint4 x0 = ldg4 (x + k), x1 = ldg4 (x + k + 4), w0 = ldg4 (w + k);
            const uint32_t xw[8] = { x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w };
            const uint32_t ww[4] = { w0.x, w0.y, w0.z, w0.w };
#pragma unroll
            for (int e = 0; e < 8; ++e)
              sum = __builtin_amdgcn_mfma_f32_32x32x2f32 (bf2f ((uint16_t)(ww[e >> 1] >> (16 * (e & 1)))),
                                                          __uint_as_float (xw[e]), sum, 0, 0, 0);
          }
#pragma unroll
        for (int q = 0; q < 16; ++q)
          acc[i][jn][q] = __builtin_fmaf (acc[i][jn][q], 0.f, 0.f) == 0.f ? acc[i][jn][q] : sum[q];
      }
}

// A BM x 128 tile by four waves of BM / 2 x 64, ST_ k-steps of it in LDS.  Of bf16 products 64 rows: three k-steps where
// two workgroups share a compute unit, six (144 KB) where each has one (deep64); and 128 and 256 rows in three, which they
// begin and end sooner than the eight waves of mix_tile (see launch_bf16_tiles).  Of 32-bit products 256 rows and their
// halves, in three.
// PLANES > 1: x holds PLANES values for every weight, in blocks of 64 (one k-step of
// each plane in turn): see the 32-bit product below.
template <int BM, int PLANES, int ST_>
__device__ __forceinline__ void
wide_bf16_tile (const GemmSegArgs &a, const WidePlace &at, int ksplit, float *ws)
{
  typedef WideElem<GemmSegArgs>::v8 v8;
  constexpr int TM = BM / 2 / 32;                    // 32-row accumulators per wave
  constexpr int STAGE_BYTES = (BM + WBN) * WROWB;
  constexpr int GPW = (BM + WBN) / 8 / WWAVES;       // 1 KiB load instructions per wave and k-step
  constexpr int AG = BM / 8 / WWAVES;                // of which rows of x
  extern __shared__ __align__ (16) uint8_t wide_lds[];
  const int ks = at.ks;
  const int nk_all = a.K / WBK;
  const int kbase = (int)((long)nk_all * ks / ksplit);
  const int nk = (int)((long)nk_all * (ks + 1) / ksplit) - kbase; // k-steps of this workgroup
  float *part = ksplit > 1 ? ws + (size_t)ks * a.M * a.N : nullptr;
  const int m0 = at.m0, n0 = at.tn * WBN;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane (threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  // Load addresses.  Instruction i of a wave covers tile rows 8g .. 8g+7 with
  // g = wave + 4 i (x for i < AG, then W); lane l fetches row 8g + l/8, and
  // LDS slot l%8 of that row receives chunk (l%8) ^ f(row), f(row) = (row & 7)
  // ^ ((row >> 3) & 1): 8 or 16 consecutive rows then hit different banks at
  // the same chunk.  Rows beyond M or N repeat the last row (never stored).
  const int lr = lane >> 3;
  const int chunk = (lane & 7) ^ lr ^ (wave & 1);
  const uint16_t *src[GPW];
#pragma unroll
  for (int i = 0; i < AG; ++i)
    {
      const int m = min (m0 + (wave + WWAVES * i) * 8 + lr, a.M - 1);
      src[i] = a.x + (size_t)m * (PLANES > 1 ? (size_t)a.K : a.xs) + chunk * 8 + (size_t)kbase * WBK;
    }
#pragma unroll
  for (int i = AG; i < GPW; ++i)
    {
      const int v = (wave + WWAVES * (i - AG)) * 8 + lr; // row of the weight tile
      src[i] = a.wh[0] + (size_t)min (n0 + v, a.N - 1) * a.ws + chunk * 8 + (PLANES > 1 ? 0 : (size_t)kbase * WBK);
    }

  // fragment reads: lane l holds row l%32 of a 32-row block, k = 16 ks + 8 (l/32) .. +7
  const int fsw = (lane & 7) ^ ((lane >> 3) & 1);
  uint32_t aoff[4], boff[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    {
      const int ko = ((2 * ks + (lane >> 5)) ^ fsw) << 4;
      aoff[ks] = (wm * (BM / 2) + (lane & 31)) * WROWB + ko;
      boff[ks] = BM * WROWB + (wn * 64 + (lane & 31)) * WROWB + ko;
    }
  constexpr int BJ = 32 * WROWB; // from a wave's first to its second column block

  float16v acc[TM][WTN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int jn = 0; jn < WTN; ++jn)
#pragma unroll
      for (int q = 0; q < 16; ++q)
        acc[i][jn][q] = 0.f;

  auto issue_part = [&] (int kt, int st, int i0, int i1) {
    const int kw = PLANES > 1 ? (kbase + kt) / PLANES : kt; // k-step of the weights
#pragma unroll
    for (int i = i0; i < i1; ++i)
      {
        const int g = i < AG ? wave + WWAVES * i : BM / 8 + wave + WWAVES * (i - AG);
        __builtin_amdgcn_global_load_lds ((const VKL_GLOBAL void *)(src[i] + (size_t)(i < AG ? kt : kw) * WBK),
                                          (VKL_LDS void *)(wide_lds + st * STAGE_BYTES + g * 1024), 16, 0, 0);
      }
  };
#pragma unroll
  for (int p = 0; p < ST_ - 1; ++p)
    if (p < nk)
      issue_part (p, p, 0, GPW);

  v8 af[2][TM], bf[2][WTN];
  // in the order the products need them
  auto read_frags = [&] (int st, int ks, int buf) {
    const uint8_t *sb = wide_lds + st * STAGE_BYTES;
    af[buf][0] = *(const v8 *)(sb + aoff[ks]);
#pragma unroll
    for (int jn = 0; jn < WTN; ++jn)
      bf[buf][jn] = *(const v8 *)(sb + boff[ks] + jn * BJ);
#pragma unroll
    for (int i = 1; i < TM; ++i)
      af[buf][i] = *(const v8 *)(sb + aoff[ks] + i * 32 * WROWB);
  };
  constexpr int LB1 = GPW / 3, LB2 = 2 * GPW / 3;
  constexpr int NR = TM + WTN, NP = TM * WTN;
  static_assert ((ST_ - 2) * GPW < 64, "");
  // One k-step.  On entry tile kt is in stage st and the fragments of its first quarter are on
  // their way into buffer 0.  (Stages of the loads are one fewer than those in LDS: DEEP.)
  constexpr int DEEP = ST_ - 1;
  auto step = [&] (int kt, int st, auto left) {
    constexpr int LEFT = decltype (left)::value;
    constexpr bool MORE = LEFT == DEEP;
    const int s1 = st == ST_ - 1 ? 0 : st + 1, sn = st == 0 ? ST_ - 1 : st - 1;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      {
        if (ks < 3)
          {
            read_frags (st, ks + 1, (ks + 1) & 1);
            // the loads of tile kt + ST - 1 go to the stage that was multiplied in the step
            // before (every wave has passed that step's barrier)
            if (MORE)
              issue_part (kt + DEEP, sn, ks == 0 ? 0 : ks == 1 ? LB1 : LB2, ks == 0 ? LB1 : ks == 1 ? LB2 : GPW);
          }
        else if (LEFT > 0)
          {
            // tile kt + 1 has landed (this wave's part; the barrier covers the
            // others') and this wave has read the last of tile kt
            wait_loads<(LEFT > 0 ? LEFT - 1 : 0) * GPW, true> ();
            __builtin_amdgcn_s_barrier ();
            __builtin_amdgcn_sched_barrier (0);
            read_frags (s1, 0, 0);
          }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int jn = 0; jn < WTN; ++jn)
            acc[i][jn] = WideElem<GemmSegArgs>::mfma (bf[ks & 1][jn], af[ks & 1][i], acc[i][jn]);
        if (ks == 0 && MORE)
          WideOrder<0, NP, NR, LB1>::run ();
        else if (ks == 1 && MORE)
          WideOrder<0, NP, NR, LB2 - LB1>::run ();
        else if (ks == 2 && MORE)
          WideOrder<0, NP, NR, GPW - LB2>::run ();
        else
          WideOrder<0, NP, NR, 0>::run ();
        __builtin_amdgcn_sched_barrier (0);
      }
  };
  if (nk < DEEP)
    wait_loads<0, false> ();
  else
    wait_loads<(DEEP - 1) * GPW, false> ();
  __builtin_amdgcn_s_barrier ();
  read_frags (0, 0, 0);
  __builtin_amdgcn_sched_barrier (0);
  wide_steps<DEEP, ST_> (nk, step);
  land_all ();

  if constexpr (PLANES > 1)
    if (!part) // (of parts the sum is looked at)
      wide_f32_again<TM> (a, acc, lane, m0 + wm * TM * 32, n0 + wn * 64, a.K / PLANES);
  wide_epilogue<TM, WTN> (a, acc, wide_lds, wave, lane, m0 + wm * TM * 32, n0 + wn * 64, part);
}

// The planes of a 32-bit operand (see there) in tiles of 64 rows: x holds three values for
// every weight, [plane 0 | plane 1 | plane 2] of 64 columns next to each other, and a k-step is
// 64 columns of the weights with those of all three planes.  Walked as a row of 3 K values, the
// weights came from the L2 and went through LDS three times: for 64 rows 72 KB into LDS and 144
// out of it per 64 columns, 1730 cycles at 128 bytes for 770 of products; now 40 + 80 KB.  Two
// stages are 80 KB, two workgroups to a compute unit, each of which multiplies where the other
// one waits; where there is one to a compute unit, four stages take its place.  Tiles of 128 rows
// (128 KB, one workgroup) were slower (800 x 16128 x 4096 362 us for
// 315); of 256 they do not fit, and those of wide_bf16_tile (144 + 288 KB for 3070 cycles of products)
// stay the better ones where they fill the chip (wide_plan_planes).  us before / now: 12 x 12288 x
// 4096 39.9 / 33.0, 300 x 2048 x 2048 27.8 / 25.2, 300 x 5504 x 2048 41.9 / 37.1, 300 x 12288 x 4096
// 120 / 96, 700 x 11008 x 4096 236 / 188.
constexpr int kPlanes = 3, kPlaneRows = 64;

template <int STAGES>
constexpr size_t
wide_lds_planes ()
{
  const size_t stages = (size_t)STAGES * (kPlanes * kPlaneRows + WBN) * WROWB, park = (size_t)kPlaneRows * 2 * kWideParkLd * 4;
  return stages > park ? stages : park;
}

template <int STAGES>
__global__ __launch_bounds__ (WWAVES * 64) void
gemm_wide_planes_kernel (const GemmSegArgs a, WideGrid grid, int ksplit, float *ws)
{
  WidePlace at;
  if (grid.place<kPlaneRows> (a.M, at) != WIDE_TILE)
    return;
  constexpr int BM = kPlaneRows;
  typedef WideElem<GemmSegArgs>::v8 v8;
  constexpr int TM = BM / 2 / 32;
  constexpr int A_BYTES = BM * WROWB, STAGE_BYTES = kPlanes * A_BYTES + WBN * WROWB;
  constexpr int AG = BM / 8 / WWAVES, BG = WBN / 8 / WWAVES, LOADS = kPlanes * AG + BG;
  extern __shared__ __align__ (16) uint8_t wide_lds[];
  const int ks = at.ks, nk_all = a.K / WBK / kPlanes;
  const int kbase = (int)((long)nk_all * ks / ksplit);
  const int nk = (int)((long)nk_all * (ks + 1) / ksplit) - kbase;
  float *part = ksplit > 1 ? ws + (size_t)ks * a.M * a.N : nullptr;
  const int m0 = at.m0, n0 = at.tn * WBN;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane (threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  // rows and chunks as in wide_bf16_tile
  const int lr = lane >> 3;
  const int chunk = (lane & 7) ^ lr ^ (wave & 1);
  const uint16_t *srca[AG], *srcb[BG];
#pragma unroll
  for (int i = 0; i < AG; ++i)
    srca[i] = a.x + (size_t)min (m0 + (wave + WWAVES * i) * 8 + lr, a.M - 1) * a.K + (size_t)kbase * kPlanes * WBK
              + chunk * 8;
#pragma unroll
  for (int i = 0; i < BG; ++i)
    srcb[i] = a.wh[0] + (size_t)min (n0 + (wave + WWAVES * i) * 8 + lr, a.N - 1) * a.ws + (size_t)kbase * WBK + chunk * 8;
  const int fsw = (lane & 7) ^ ((lane >> 3) & 1);
  uint32_t aoff[4], boff[4];
#pragma unroll
  for (int q = 0; q < 4; ++q)
    {
      const int ko = ((2 * q + (lane >> 5)) ^ fsw) << 4;
      aoff[q] = (wm * (BM / 2) + (lane & 31)) * WROWB + ko;
      boff[q] = kPlanes * A_BYTES + (wn * 64 + (lane & 31)) * WROWB + ko;
    }

  // the two lower planes' sums are kept apart: added to the large ones they would round those
  // two times more per sixteen products
  float16v acc[TM][WTN], low[TM][WTN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int jn = 0; jn < WTN; ++jn)
#pragma unroll
      for (int q = 0; q < 16; ++q)
        acc[i][jn][q] = 0.f, low[i][jn][q] = 0.f;

  // loads [i0, i1) of a k-step: the weights, then the planes
  auto issue = [&] (int kt, int st, int i0, int i1) {
#pragma unroll
    for (int i = i0; i < i1; ++i)
      {
        uint8_t *base = wide_lds + st * STAGE_BYTES;
        if (i < BG)
          __builtin_amdgcn_global_load_lds ((const VKL_GLOBAL void *)(srcb[i] + (size_t)kt * WBK),
                                            (VKL_LDS void *)(base + kPlanes * A_BYTES + (wave + WWAVES * i) * 1024), 16,
                                            0, 0);
        else
          {
            const int p = (i - BG) / AG, g = (i - BG) % AG;
            __builtin_amdgcn_global_load_lds (
                (const VKL_GLOBAL void *)(srca[g] + (size_t)kt * kPlanes * WBK + p * WBK),
                (VKL_LDS void *)(base + p * A_BYTES + (wave + WWAVES * g) * 1024), 16, 0, 0);
          }
      }
  };
  v8 af[2][kPlanes][TM], bf[2][WTN];
  auto read_frags = [&] (int st, int q, int buf) {
    const uint8_t *sb = wide_lds + st * STAGE_BYTES;
#pragma unroll
    for (int jn = 0; jn < WTN; ++jn)
      bf[buf][jn] = *(const v8 *)(sb + boff[q] + jn * 32 * WROWB);
#pragma unroll
    for (int p = 0; p < kPlanes; ++p)
#pragma unroll
      for (int i = 0; i < TM; ++i)
        af[buf][p][i] = *(const v8 *)(sb + aoff[q] + p * A_BYTES + i * 32 * WROWB);
  };
  constexpr int NP = kPlanes * TM * WTN, NR = kPlanes * TM + WTN;
  static_assert ((STAGES - 1) * LOADS < 64, "");
  // (of two stages the second one's loads come after the barrier)
  constexpr int FIRST = STAGES == 2 ? 1 : STAGES;
#pragma unroll
  for (int p = 0; p < FIRST; ++p)
    if (p < nk)
      issue (p, p, 0, LOADS);
  if (nk < FIRST)
    wait_loads<0, false> ();
  else
    wait_loads<(FIRST - 1) * LOADS, false> ();
  __builtin_amdgcn_s_barrier ();
  if (FIRST < STAGES && FIRST < nk)
    issue (FIRST, FIRST, 0, LOADS);
  read_frags (0, 0, 0);
  __builtin_amdgcn_sched_barrier (0);
  // One k-step: on entry tile kt is in stage st, the fragments of its first quarter are on
  // their way and the tiles behind it are on their way into the other stages.
  auto step = [&] (int kt, int st, auto left) {
    constexpr int LEFT = decltype (left)::value;
    constexpr bool MORE = LEFT == STAGES; // to load
#pragma unroll
    for (int q = 0; q < 4; ++q)
      {
        if (q < 3)
          read_frags (st, q + 1, (q + 1) & 1);
        else if (LEFT > 0)
          {
            // tile kt + 1 is there and nobody reads tile kt any more: its stage takes tile
            // kt + STAGES
            wait_loads<(MORE ? STAGES - 2 : LEFT > 0 ? LEFT - 1 : 0) * LOADS, true> ();
            __builtin_amdgcn_s_barrier ();
            __builtin_amdgcn_sched_barrier (0);
            read_frags (st == STAGES - 1 ? 0 : st + 1, 0, 0);
            if (MORE)
              issue (kt + STAGES, st, 0, LOADS);
          }
#pragma unroll
        for (int p = 0; p < kPlanes; ++p)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int jn = 0; jn < WTN; ++jn)
              {
                float16v &sum = p ? low[i][jn] : acc[i][jn];
                sum = WideElem<GemmSegArgs>::mfma (bf[q & 1][jn], af[q & 1][p][i], sum);
              }
        if (q == 3 && MORE)
          WideOrder<0, NP, NR, LOADS>::run ();
        else
          WideOrder<0, NP, NR, 0>::run ();
        __builtin_amdgcn_sched_barrier (0);
      }
  };
  wide_steps<STAGES, STAGES> (nk, step);
  land_all ();
  __builtin_amdgcn_s_barrier (); // every wave's fragments are read before the sums are parked

#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int jn = 0; jn < WTN; ++jn)
#pragma unroll
      for (int q = 0; q < 16; ++q)
        acc[i][jn][q] += low[i][jn][q];
  if (!part) // (of parts the sum is looked at)
    wide_f32_again<TM> (a, acc, lane, m0 + wm * TM * 32, n0 + wn * 64, a.K / kPlanes);
  wide_epilogue<TM, WTN> (a, acc, wide_lds, wave, lane, m0 + wm * TM * 32, n0 + wn * 64, part);
}

template <int BM, int PLANES, int ST>
__global__ __launch_bounds__ (WWAVES * 64) void
gemm_wide_bf16_kernel (const GemmSegArgs a, WideGrid grid, int ksplit, float *ws)
{
  WidePlace at;
  switch (grid.place<BM> (a.M, at))
    {
    case WIDE_NONE:
      return;
    case WIDE_TILE:
      return wide_bf16_tile<BM, PLANES, ST> (a, at, ksplit, ws);
    case WIDE_HALF:
      if constexpr (BM == WBM)
        return wide_bf16_tile<BM / 2, PLANES, ST> (a, at, ksplit, ws);
    }
}

// ---------------------------------------------------------------------------
// tiles of up to 256 x 256
// ---------------------------------------------------------------------------
constexpr int MWAVES = 8;

// What the tiles of gemm_mix_kernel take, us: of bm token rows and 256 columns, of 128 columns,
// and of half of that (by the rows of 256, by the columns of 128).  Fitted with wide_plan_bf16's other constants, see
// there, to the choice that they make.  By themselves (least squares, launch included) tiles of 256 x 256 take 1.30
// per k-step + 7.6, of 256 x 128 0.70 + 8.0, of 128 x 256 0.76 + 5.0, of 128 x 128 0.49 + 5.3 (one row of them 0.67 +
// 3.8), of 128 x 64 0.31 + 4.5.  Those last ones are charged with more: at 0.31 a product of 160 x 5504 x 2048 and its
// like would be in one part (15 us, in two 19.7), but it is held to be in parts (tests/test_gemm_f32.py).
struct MixTime
{
  double step, start, parked; // per k-step; per tile; more where its sums are parked in LDS
};
inline MixTime
mix_time (int bm, int kind, bool one_row, bool q8)
{
  // (Q8_0 weights: 256 rows only, and no parked sums to weigh; 511 launches of 256 to 2048 rows, none slower by more
  // than 2 % than without pairs.  With 2.20, 10; 1.30, 8; 0.70, 6 up/gate of 1300 to 2048 x 3072 x 1024 went into pairs:
  // 44.2 us, 41.4 without)
  constexpr MixTime tq8[3] = { { 2.26, 10.1, 0 }, { 1.30, 7.9, 0 }, { 0.71, 5.8, 0 } };
  if (q8)
    return tq8[kind];
  constexpr MixTime t256[3] = { { 1.41, 5.0, 15.5 }, { 0.69, 5.7, 8.3 }, { 0.53, 5.6, 4.4 } };
  // Fitted to the choice that they make among 460 bf16 products of 200 to 2048 rows, the other constants as they are: 1.5 %
  // faster in the mean for these tiles, which are in 70 of the plans, one of them 3 % slower than the plan before (the best
  // choice of all: 2.0 %).  448 others, 144 to 2200 rows, widths of 1024, 2048, 3072 and 4096: 1.7 % in the mean, up to 22; what was
  // slower is held back by kFew192 (and 528 x 2048 x 7552, 29.3 / 31.2, see kOddParts).
  constexpr MixTime t192[2] = { { 1.34, 6.97, 8.0 }, { 0.70, 3.63, 5.7 } };
  constexpr MixTime t128[3] = { { 0.70, 7.2, 7.7 }, { 0.49, 7.0, 3.0 }, { 0.52, 3.4, 0.51 } };
  // one row of tiles streams the weights
  constexpr MixTime t1[3] = { { 1.17, 7.6, 7.1 }, { 0.79, 7.0, 3.4 }, { 0.49, 5.1, 3.9 } };
  if (bm == 192)
    return t192[std::min (kind, 1)];
  return bm == WBM ? t256[kind] : one_row ? t1[kind] : t128[kind];
}

// When the compute units are done with tiles dealt in turn to whichever is free first.
struct MixSpan
{
  double at[4] = { 0, 0, 0, 0 };
  int units[4] = { WideGrid::kUnits, 0, 0, 0 }, n = 1; // each kind of tile adds at most one level
  double last = 0;

  void
  deal (int tiles, double time)
  {
    while (tiles > 0)
      {
        if (n == 1 && tiles >= units[0])
          {
            at[0] += tiles / units[0] * time, tiles %= units[0];
            last = at[0];
            continue;
          }
        int f = 0;
        for (int i = 1; i < n; ++i)
          if (at[i] < at[f])
            f = i;
        const double end = at[f] + time;
        const int take = tiles < units[f] ? tiles : units[f];
        last = end > last ? end : last, tiles -= take;
        int same = 0;
        while (same < n && at[same] != end)
          ++same;
        if (take == units[f] && same == n)
          at[f] = end; // the level moves
        else
          {
            if (same < n)
              units[same] += take;
            else
              at[n] = end, units[n++] = take;
            units[f] -= take;
            if (!units[f])
              --n, at[f] = at[n], units[f] = units[n];
          }
      }
  }
};

// The tiles of a launch: pairs of 128-column tiles as one of 256 columns, then tiles of 128
// columns, of which the last (few of 128 rows: all) may be cut in two.  Each kind is dealt to the XCDs
// in contiguous ranges of pairs, row tile fastest in groups of eight: the 32 pairs that an XCD
// multiplies at a time are then 8 x 4 and not 32 x 1, and share their rows in its L2 (8192 x
// 8192 x 8192 1023 us with 32 x 1, 823 with 8 x 4, 256 x 128 tiles).
//
// A tile of 256 columns takes less than two of 128 (every fragment that is read from LDS goes into
// twice the products; 0.95 of them by mix_time at K = 4096, of the tiles by themselves 0.86), but fewer of them fill a
// round over the 256 compute units.  So either no
// pair, as many as fill whole rounds, or all go into one tile, whichever is done first: 2048 x
// 12288 columns (1.5 rounds of pairs) 182 us with one round of pairs and 256 tiles, 198 without pairs,
// 211 of pairs alone; 1500 x 8064, K = 2048 59 / 59 / 55.
//
// 192 rows (bf16) are for products whose 256-row tiles fill a part of their last round only: one round of 192 x 256 takes
// 0.85 of one of 256 x 256.  us with tiles of 128 and 256 rows / with these, weights that no cache holds: 1500 x 7552 x 2048
// 57.4 / 48.8, 1500 x 2048 x 7552 (two parts) 61.4 / 57.1, 1500 x 4096 x 15104 181.9 / 165.7, 1152 x 4096 x 4096 55.4 / 49.5,
// 768 x 5504 x 2048 with GELU 0.83 of the time, 2048 x 5504 x 2048 0.90.  They are not cut.
//
// At most 128 tiles of 128 rows leave half the compute units idle while the others wait for weights: they are cut
// by their columns into twice as many of 128 x 64, with six stages of loads (whole / cut, us, fp16: 77 x 4096 x 11008 in four
// parts 34.0 / 27.2, 128 rows 38.7 / 31.9, 77 x 4096 x 4096 16.1 / 15.5).  The halves of more tiles would not all
// run at once.
struct WideMix
{
  int tiles_m, tiles_n, nmat, ksplit;
  int wide;  // pairs in one tile
  int whole; // tiles of 128 columns that are not cut

  __host__ __device__ int
  pairs () const
  {
    return tiles_m * (tiles_n / 2) * nmat * ksplit;
  }
  __host__ __device__ int
  narrow () const // tiles of 128 columns, cut or not
  {
    return tiles_m * tiles_n * nmat * ksplit - 2 * wide;
  }
  // bm: token rows of a tile, 256 (which may be cut by its rows), 192 or 128 (by its columns); steps: of the k range of a part;
  // park: how much of the time for parked sums a tile takes; us: the time of the launch's tiles
  __host__
  WideMix (int bm, int tm, int tn, int mats, int parts, double steps, double park, double *us = nullptr, bool q8 = false)
      : tiles_m (tm), tiles_n (tn), nmat (mats), ksplit (parts)
  {
    constexpr int U = WideGrid::kUnits;
    double t[3];
    for (int k = 0; k < 3; ++k)
      {
        const MixTime m = mix_time (bm, k, tm == 1, q8);
        t[k] = m.step * steps + m.start + park * m.parked;
      }
    const int options[3] = { 0, pairs () / U * U, pairs () };
    int best_wide = 0, best_whole = 0;
    double best = -1;
    for (int o = 0; o < 3; ++o)
      {
        if (o && options[o] == options[o - 1])
          continue;
        wide = options[o];
        const int rest = narrow () % U;
        whole = bm == WBM && wide % U == 0 && rest > 0 && rest <= U / 2 ? narrow () - rest : narrow ();
        if (bm == 128 && !q8 && narrow () <= U / 2)
          whole = 0;
        MixSpan span;
        span.deal (wide, t[0]);
        span.deal (whole, t[1]);
        span.deal (2 * (narrow () - whole), t[2]);
        if (best < 0 || span.last < best)
          best = span.last, best_wide = wide, best_whole = whole;
      }
    wide = best_wide, whole = best_whole;
    if (us)
      *us = best;
  }
  static __host__ __device__ int
  eight (int n)
  {
    return (n + 7) / 8 * 8;
  }
  __host__ int
  groups () const
  {
    return eight (wide) + eight (whole) + eight (2 * (narrow () - whole));
  }
  __device__ __forceinline__ void
  pair_at (int p, WidePlace &at, int BM) const
  {
    const int cols = tiles_n / 2, mats = tiles_m * cols * nmat, grp = 8 * cols * nmat;
    at.ks = p / mats;
    p -= at.ks * mats;
    const int g = p / grp, gm = min (8, tiles_m - 8 * g);
    p -= g * grp;
    at.m0 = (8 * g + p % gm) * BM;
    p /= gm;
    at.tn = 2 * (p % cols);
    at.zmat = p / cols;
  }
  // 0: nothing to do, 1: a pair, 2: one tile, 3: half a tile
  __device__ __forceinline__ int
  place (int M, int BM, WidePlace &at) const
  {
    const int g0 = eight (wide), g1 = g0 + eight (whole);
    int id = (int)blockIdx.x;
    const int kind = id < g0 ? 1 : id < g1 ? 2 : 3;
    id -= kind == 1 ? 0 : kind == 2 ? g0 : g1;
    const int count = kind == 1 ? wide : kind == 2 ? whole : 2 * (narrow () - whole);
    const int per_xcd = (count + 7) / 8, j = id >> 3;
    int i = (id & 7) * per_xcd + j;
    if (j >= per_xcd || i >= count)
      return 0;
    if (kind == 1)
      {
        pair_at (i, at, BM);
        return 1;
      }
    int half = 0;
    if (kind == 3)
      half = i & 1, i = whole + (i >> 1);
    const int left = 2 * (pairs () - wide);
    if (i < left)
      {
        pair_at (wide + (i >> 1), at, BM);
        at.tn += i & 1;
      }
    else
      {
        // the last column of an odd number
        i -= left;
        at.m0 = i % tiles_m * BM;
        i /= tiles_m;
        at.tn = tiles_n - 1, at.zmat = i % nmat, at.ks = i / nmat;
      }
    at.half = half;
    if (BM == WBM)
      at.m0 += half * (BM / 2);
    return at.m0 < M ? kind : 0;
  }
};

// Issue order of half a k-step: after each product an even share of its fragment reads and loads
template <int Q, int NP, int NR, int NL> struct MixOrder
{
  static __device__ __forceinline__ void
  run ()
  {
    __builtin_amdgcn_sched_group_barrier (0x008, 1, 0); // one MFMA
    constexpr int nr = NR * (Q + 1) / NP - NR * Q / NP, nl = NL * (Q + 1) / NP - NL * Q / NP;
    if constexpr (nr > 0)
      __builtin_amdgcn_sched_group_barrier (0x100, nr, 0); // LDS reads
    if constexpr (nl > 0)
      __builtin_amdgcn_sched_group_barrier (0x020, nl, 0); // loads
    if constexpr (Q + 1 < NP)
      MixOrder<Q + 1, NP, NR, NL>::run ();
  }
};

// acc[i][j]: 16 token rows by 16 weight rows; blocks 2 b and 2 b + 1 of a wave hold, in lane l,
// columns 8 (l / 16) .. + 3 and + 4 .. + 7 of its 32 columns b (see mix_tile): eight neighbours
// of token row l % 16.  Of the fused pair blocks 0, 1 are up and 2, 3 gate.
template <bool UPGATE, int TM, class Args>
__device__ __forceinline__ void
mix_epilogue (const Args &a, const float4v (&acc)[TM][4], uint8_t *wide_lds, int wave, int lane, int mrow, int ncol,
              int zmat, int vec, float *part)
{
  constexpr int NB = UPGATE ? 1 : 2; // 32-column blocks of outputs, each by itself
  if constexpr (std::is_same_v<Args, GemmSegArgs>)
    if (part && (a.N % 8) == 0)
      {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int b = 0; b < NB; ++b)
            part_store8 (part, a.M, a.N, mrow + i * 16 + (lane & 15), ncol + b * 32 + (lane >> 4) * 8, acc[i][2 * b], acc[i][2 * b + 1]);
        return;
      }
  bool parked = false;
#pragma unroll
  for (int b = 0; b < NB; ++b)
    {
      const WideSimple<UPGATE, Args> simple (a, ncol + b * 32, 32, zmat, vec, part);
      if (!simple.ok)
        {
          parked = true;
          continue;
        }
      const int m0 = mrow + (lane & 15), col = (lane >> 4) * 8;
      auto walk = [&] (auto with) {
        constexpr bool RES = decltype (with)::value != 0;
        constexpr int NR = WideSimple<UPGATE, Args>::NR;
        uint4 res[TM][NR];
        if (RES)
#pragma unroll
          for (int i = 0; i < TM; ++i)
            simple.request ((size_t)min (m0 + i * 16, a.M - 1), col, res[i]);
#pragma unroll
        for (int i = 0; i < TM; ++i)
          {
            float v[8], g[8];
#pragma unroll
            for (int e = 0; e < 4; ++e)
              {
                v[e] = acc[i][2 * b][e], v[4 + e] = acc[i][2 * b + 1][e];
                g[e] = UPGATE ? acc[i][2][e] : 0.f, g[4 + e] = UPGATE ? acc[i][3][e] : 0.f;
              }
            if (m0 + i * 16 < a.M)
              simple.store ((size_t)(m0 + i * 16), col, v, g, RES ? res[i] : nullptr);
          }
      };
      if (simple.r)
        walk (WideInt<1> ());
      else
        walk (WideInt<0> ());
    }
  if (!parked)
    return;
  __builtin_amdgcn_s_barrier (); // every wave (that is left) has read its last fragments
  // through LDS: a block of 32 columns of all rows, of the fused pair both blocks of 64 rows
  constexpr int PM = UPGATE && TM > 4 ? 4 : TM, ROWS = PM * 16, LD = UPGATE ? 68 : 36;
  float *park = (float *)(wide_lds + wave * (ROWS * LD * 4));
  constexpr int RPI = 16; // rows per iteration, four lanes each
  const int er = lane >> 2, ec = (lane & 3) * 8;
#pragma unroll
  for (int b = 0; b < NB; ++b)
    {
      if (WideSimple<UPGATE, Args> (a, ncol + b * 32, 32, zmat, vec, part).ok)
        continue;
      const FinishRows<UPGATE, Args> fin (a, ncol + b * 32 + ec, zmat, vec, part);
#pragma unroll
      for (int i0 = 0; i0 < TM; i0 += PM)
        {
#pragma unroll
          for (int i = 0; i < PM; ++i)
#pragma unroll
            for (int j = 0; j < (UPGATE ? 4 : 2); ++j)
              *(float4v *)(park + (i * 16 + (lane & 15)) * LD + (j >> 1) * 32 + (lane >> 4) * 8 + (j & 1) * 4)
                  = acc[i0 + i][2 * b + j];
          // (a wave reads back only what it wrote itself: no barrier)
#pragma unroll 1
          for (int it = 0; it < ROWS / RPI; ++it)
            {
              const int row = it * RPI + er, m = mrow + i0 * 16 + row;
              uint4 res[2];
              fin.request (m, res);
              const float *pr = park + row * LD + ec;
              const float4v p0 = *(const float4v *)pr, p1 = *(const float4v *)(pr + 4);
              float v[8] = { p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w };
              float g[8] = { 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f };
              if (UPGATE)
                {
                  const float4v g0 = *(const float4v *)(pr + 32), g1 = *(const float4v *)(pr + 36);
                  g[0] = g0.x, g[1] = g0.y, g[2] = g0.z, g[3] = g0.w, g[4] = g1.x, g[5] = g1.y, g[6] = g1.z, g[7] = g1.w;
                }
              fin.store (m, v, g, res);
            }
        }
    }
}

// A BM x BN tile by WM x WN waves of (BM / WM) x 64, ST k-steps of 64 in LDS: one workgroup
// of eight waves to a compute unit, so that one wave of a SIMD multiplies where the other one
// waits for a barrier or its fragments.
//
// Products of 16 x 16 x 32 (rather than 32 x 32 x 16) and 256 x 256 tiles: bound by the chip's
// power under matrix load (at 8192 x 8192 x 8192 matrix cores busy 71 % of the cycles at 1.81
// GHz, 56 % at 1.87 in 256 x 128 tiles of four waves with 32 x 32 x 16; the vendor library's kernel 88 %
// at 1.64), so less data per product out of LDS and L2 is what makes it faster.  The loads of a k-step are
// issued when its stage has just been read, not a quarter later: two stages of 64 KB are enough then.
// Of more than two stages each half of a k-step issues half of one (a burst of all in one half / halves, us:
// 300 x 16128 x 4096 bf16 62.2 / 56.6, 300 x 11008 x 4096 52.6 / 49.4, 700 x 11008 x 4096 85.5 / 80.1).
// Tried on the way, 4096 x 4096 x 4096, us: 107 as it is, 123 with 32 x 32 x 16, 147 with four waves
// of 128 x 128 (AGPR moves), 117 with raised wave priority around the products, 114 with four stages of
// 32 columns, 111 with two reads per product.
// Same call before / now, us, fp16, one box: 4096 x 4096 x 4096 132 / 110, 2048 x 12288 x 4096 191 / 174,
// 2048 x 22016 x 4096 366 / 318, 3967 x 5120 x 5120 256 / 192, 8192 x 8192 x 8192 1250 / 822, 300 x 4096 x
// 4096 28.8 / 27.2, 77 x 4096 x 4096 18.1 / 16.5, 2048 x 4096 x 4096 64.4 / 62.7.
template <int BM, int BN, int WM, int ST, bool UPGATE, class Args>
__device__ __forceinline__ void
mix_tile (const Args &a, const WidePlace &at, int vec, int ksplit, float *ws)
{
  typedef typename WideElem<Args>::v8 v8;
  constexpr int WN = MWAVES / WM, TM = BM / WM / 16, TN = 4;
  static_assert (BN / WN == 64 && BM % (MWAVES * 8) == 0 && BN % (MWAVES * 8) == 0, "");
  constexpr int STAGE_BYTES = (BM + BN) * WROWB;
  constexpr bool ALIKE = BM + BN > 256; // see wide_steps_alike
  constexpr int AG = BM / 8 / MWAVES, LOADS = (BM + BN) / 8 / MWAVES; // 1 KiB instructions per wave and k-step
  extern __shared__ __align__ (16) uint8_t wide_lds[];
  const int nk_all = a.K / WBK;
  const int kbase = (int)((long)nk_all * at.ks / ksplit);
  const int nk = (int)((long)nk_all * (at.ks + 1) / ksplit) - kbase;
  float *part = ksplit > 1 ? ws + (size_t)at.ks * a.M * a.N : nullptr;
  const int m0 = at.m0, n0 = (at.tn * WBN + (BN < WBN ? at.half * BN : 0)) / (UPGATE ? 2 : 1);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane (threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;

  // Load addresses.  Instruction i of a wave covers eight tile rows 8 g .. 8 g + 7, g = wave +
  // 8 i; slot l % 8 of row 8 g + l / 8 receives the row's chunk (l % 8) ^ f (row).  Sixteen
  // lanes read 16 bytes at a time, 0-3, 12-15, 20-27 and their complement of a half wave: of a
  // fragment eight rows at one chunk and eight others at the next.  With f = row / 2 of the
  // token rows, and of the weight rows, whose fragments are rows 8 (r / 4) + r % 4 (+ 4), bit 1
  // below bits 3 and 4, these lie in different banks (no conflicts by the counters; half of
  // the read cycles with the order of the 32 x 32 products).  Rows beyond M or N repeat the
  // last row (never stored).
  const int lr = lane >> 3;
  const int fa = (wave & 1) * 4 + (lane >> 4), fb = ((lr >> 1) & 1) | ((wave & 3) << 1);
  const uint16_t *src[LOADS];
#pragma unroll
  for (int i = 0; i < AG; ++i)
    src[i] = a.x + (size_t)min (m0 + (wave + MWAVES * i) * 8 + lr, a.M - 1) * a.xs + ((lane & 7) ^ fa) * 8
             + (size_t)kbase * WBK;
#pragma unroll
  for (int i = AG; i < LOADS; ++i)
    {
      const int v = (wave + MWAVES * (i - AG)) * 8 + lr;
      const int mat = UPGATE ? v / (BN / 2) : at.zmat;
      const int n = min (n0 + (UPGATE ? v % (BN / 2) : v), a.N - 1);
      src[i] = pick3 (a.wh[0], a.wh[1], a.wh[2], mat) + (size_t)n * a.ws + ((lane & 7) ^ fb) * 8 + (size_t)kbase * WBK;
    }
  // fragment reads: lane l holds row l % 16 of a fragment, k = 32 h + 8 (l / 16) .. + 7
  const int r = lane & 15, brow = (r >> 2) * 8 + (r & 3);
  const int ga = (r >> 1) & 7, gb = ((brow >> 1) & 1) | (((brow >> 3) & 3) << 1);
  uint32_t aoff[2], boff[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    {
      const int c = 4 * h + (lane >> 4);
      aoff[h] = (wm * (BM / WM) + r) * WROWB + ((c ^ ga) << 4);
      boff[h] = (BM + wn * (UPGATE ? 32 : 64) + brow) * WROWB + ((c ^ gb) << 4);
    }
  constexpr int BJ = (UPGATE ? BN / 2 : 32) * WROWB; // from a wave's first to its second 32 weight rows

  constexpr int EARLY = ST > 2 ? LOADS / 2 : LOADS;
  float4v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      acc[i][j] = float4v{ 0.f, 0.f, 0.f, 0.f };

  auto issue = [&] (int kt, int st, int i0, int i1) {
#pragma unroll
    for (int i = i0; i < i1; ++i)
      {
        const int g = i < AG ? wave + MWAVES * i : BM / 8 + wave + MWAVES * (i - AG);
        __builtin_amdgcn_global_load_lds ((const VKL_GLOBAL void *)(src[i] + (size_t)kt * WBK),
                                          (VKL_LDS void *)(wide_lds + st * STAGE_BYTES + g * 1024), 16, 0, 0);
      }
  };
#pragma unroll
  for (int p = 0; p < ST; ++p)
    if (ALIKE || p < nk)
      issue (p < nk ? p : nk - 1, p, 0, p < ST - 1 ? LOADS : EARLY);
  v8 af[2][TM], bf[2][TN];
  auto read_frags = [&] (int st, int h, int buf) {
    const uint8_t *sb = wide_lds + st * STAGE_BYTES;
#pragma unroll
    for (int j = 0; j < TN; ++j)
      bf[buf][j] = *(const v8 *)(sb + boff[h] + (j >> 1) * BJ + (j & 1) * 4 * WROWB);
#pragma unroll
    for (int i = 0; i < TM; ++i)
      af[buf][i] = *(const v8 *)(sb + aoff[h] + i * 16 * WROWB);
  };
  static_assert ((ST - 1) * LOADS < 64, "");
  // One k-step.  On entry tile kt is in stage st and the fragments of its first half are on
  // their way.  Between its halves tile kt + 1 has landed (this wave's part; the barrier covers
  // the others') and nobody reads tile kt any more, whose last fragments are in registers: its
  // stage takes tile kt + ST, a whole step and more before it is wanted (past the end, if at all, the
  // last tile again, which nothing reads, but which is still to land: land_all).
  auto step = [&] (int kt, int st, auto left) {
    constexpr int LEFT = decltype (left)::value;
    constexpr bool MORE = LEFT == ST; // to load
#pragma unroll
    for (int h = 0; h < 2; ++h)
      {
        if (h == 0)
          {
            read_frags (st, 1, 1);
            // the rest of tile kt + ST - 1
            if (EARLY < LOADS && LEFT >= ST - 1)
              issue (kt + ST - 1 < nk ? kt + ST - 1 : nk - 1, st == 0 ? ST - 1 : st - 1, EARLY, LOADS);
          }
        else if (LEFT > 0)
          {
            wait_loads<(MORE ? ST - 2 : LEFT > 0 ? LEFT - 1 : 0) * LOADS, true> ();
            __builtin_amdgcn_s_barrier ();
            __builtin_amdgcn_sched_barrier (0);
            if (MORE)
              issue (kt + ST < nk ? kt + ST : nk - 1, st, 0, EARLY);
            read_frags (st == ST - 1 ? 0 : st + 1, 0, 0);
          }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = WideElem<Args>::mfma (bf[h][j], af[h][i], acc[i][j]);
        if (h && MORE)
          MixOrder<0, TM * TN, TM + TN, EARLY>::run ();
        else if (!h && LEFT >= ST - 1)
          MixOrder<0, TM * TN, TM + TN, LOADS - EARLY>::run ();
        else
          MixOrder<0, TM * TN, TM + TN, 0>::run ();
        __builtin_amdgcn_sched_barrier (0);
      }
  };
  if (!ALIKE && nk < ST)
    wait_loads<0, false> ();
  else
    wait_loads<(ST - 2) * LOADS + EARLY, false> ();
  __builtin_amdgcn_s_barrier ();
  read_frags (0, 0, 0);
  __builtin_amdgcn_sched_barrier (0);
  if constexpr (ALIKE)
    wide_steps_alike<ST, ST> (nk, step);
  else
    wide_steps<ST, ST> (nk, step);
  land_all ();
  mix_epilogue<UPGATE, TM, Args> (a, acc, wide_lds, wave, lane, m0 + wm * (BM / WM), n0 + wn * (UPGATE ? 32 : 64), at.zmat,
                                  vec, part);
}

template <int BM>
constexpr size_t
mix_lds ()
{
  constexpr size_t wide = (size_t)(BM > 128 ? 2 : 3) * (BM + 256) * WROWB;
  constexpr size_t narrow = (size_t)(BM > 128 ? 3 : 4) * (BM + WBN) * WROWB;
  constexpr size_t park = (size_t)MWAVES * std::max (BM / 2 * 36, 64 * 68) * 4; // see mix_epilogue
  static_assert (BM > 128 || 6 * (BM + WBN / 2) * WROWB <= wide, "");
  return std::max (std::max (wide, narrow), park);
}

template <int BM, bool UPGATE, class Args>
__global__ __launch_bounds__ (MWAVES * 64) void
gemm_mix_kernel (const Args a, WideMix grid, int vec, int ksplit, float *ws)
{
  WidePlace at;
  switch (grid.place (a.M, BM, at))
    {
    case 1:
      return mix_tile<BM, 256, 2, (BM > 128 ? 2 : 3), UPGATE, Args> (a, at, vec, ksplit, ws);
    case 2:
      return mix_tile<BM, WBN, 4, (BM > 128 ? 3 : 4), UPGATE, Args> (a, at, vec, ksplit, ws);
    case 3:
      if constexpr (BM == WBM)
        return mix_tile<BM / 2, WBN, 4, 4, UPGATE, Args> (a, at, vec, ksplit, ws);
      else if constexpr (BM == 128)
        return mix_tile<BM, WBN / 2, 8, 6, UPGATE, Args> (a, at, vec, ksplit, ws);
    }
}

// ---------------------------------------------------------------------------
// planar Q8_0 weights
// ---------------------------------------------------------------------------
// Same tile, same staging.  The weight tile enters LDS as it lies in memory:
// 128 rows x 64 int8 (8 KiB, 16-byte chunks swizzled by (row >> 1) & 3) plus
// the two fp16 block scales of every row.  A wave converts the int8 fragments
// it reads to fp16 (exact integers) in registers, sums each block of 32 on the
// matrix core from a zero accumulator and applies the block's scale in fp32
// (acc = fma (part, d, acc)): the arithmetic of the tile kernel and of the
// reference shader.  That scaling costs as many vector-ALU cycles as the
// products cost matrix-core cycles, and it wants the block sums in ordinary
// registers: a workgroup is therefore EIGHT waves (two per SIMD, at most 256
// registers each, where the compiler keeps MFMA results out of the
// accumulation registers).  The unit of the schedule is a block (two MFMA
// k-slices): while block b is multiplied, the fragments of block b + 1 are
// read.  (LDS reads must not go through HIP's uint2/uint4 struct types here:
// the compiler takes reads of a struct type to alias the tiles that the
// direct-to-LDS loads still have in flight and waits for all of them.)
constexpr int QWAVES = 8;
// waves along N: 2 x 4 waves, 128 x 32 each (every weight fragment is converted by two
// waves), measured 5-12 % faster than 4 x 2, 64 x 64 each, on the 7B and 13B shapes
constexpr int WGN = 4;
// Three stages, laid out by kind (x tiles, then quants, then scales).
constexpr int QSTAGES = 3;
constexpr int QB_BYTES = WBN * WBK;
constexpr int QS_BYTES = WBN * 4; // two fp16 scales per row

template <int BM>
constexpr size_t
wide_lds_q8 ()
{
  const size_t stages = (size_t)QSTAGES * (BM * WROWB + QB_BYTES + QS_BYTES), park = (size_t)BM * kWideTileLd * 4;
  return stages > park ? stages : park;
}

// (a vector type, not HIP's uint2 struct: LDS reads of the struct type are
// taken to alias the tiles in flight and made to wait for all of them)
typedef uint32_t u32x2 __attribute__ ((ext_vector_type (2)));

__device__ __forceinline__ half8
q8_frag (u32x2 r)
{
  h16x2 a, b, c, d;
  i8x4_to_h2x2 (r.x, a, b);
  i8x4_to_h2x2 (r.y, c, d);
  half8 o;
  o[0] = a[0], o[1] = a[1], o[2] = b[0], o[3] = b[1];
  o[4] = c[0], o[5] = c[1], o[6] = d[0], o[7] = d[1];
  return o;
}

template <int BM, bool UPGATE>
__device__ __forceinline__ void
wide_q8_tile (const GemmArgs &a, const WidePlace &at, int vec, int ksplit, float *ws)
{
  constexpr int QTM = BM / (QWAVES / WGN) / 32; // 32-row accumulators per wave
  constexpr int QTN = 1;                        // 32-column accumulators per wave
  constexpr int QAG = BM / 8 / QWAVES;       // x load instructions per wave and k-step
  constexpr int QA_BYTES = BM * WROWB;
  constexpr int QB_BASE = QSTAGES * QA_BYTES;
  constexpr int QS_BASE = QB_BASE + QSTAGES * QB_BYTES;
  constexpr int QLOADS = QAG + 1 + 1;        // per wave and k-step: x, quants, scales
  extern __shared__ __align__ (16) uint8_t wide_lds[];
  const int ks = at.ks, zmat = at.zmat;
  const int nk_all = a.K / WBK;
  const int kbase = (int)((long)nk_all * ks / ksplit);
  const int nk = (int)((long)nk_all * (ks + 1) / ksplit) - kbase; // k-steps of this workgroup
  float *part = ksplit > 1 ? ws + (size_t)ks * a.M * a.N : nullptr;
  const int m0 = at.m0, n0 = at.tn * (UPGATE ? WBN / 2 : WBN);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane (threadIdx.x >> 6);
  const int wm = wave / WGN, wn = wave % WGN;

  // load addresses: x as in the fp16 kernel, instruction i of a wave covering
  // tile rows 8 g .. 8 g + 7 with g = wave + 8 i
  const int lr = lane >> 3;
  const int chunk = (lane & 7) ^ lr ^ (wave & 1);
  const uint8_t *src[QLOADS];
#pragma unroll
  for (int i = 0; i < QAG; ++i)
    {
      const int m = min (m0 + (wave + QWAVES * i) * 8 + lr, a.M - 1);
      src[i] = (const uint8_t *)(a.x + (size_t)m * a.xs + chunk * 8 + (size_t)kbase * WBK);
    }
  // quants: a wave's one instruction covers weight-tile rows 16 wave .. + 15;
  // lane l fetches chunk (l%4) ^ ((row >> 1) & 3) of row 16 wave + l/4
  {
    const int qr = lane >> 2;
    const int v = wave * 16 + qr;
    const int mat = UPGATE ? v >> 6 : zmat;
    const int n = min (UPGATE ? n0 + (v & 63) : n0 + v, a.N - 1);
    const uint8_t *w = mat == 0 ? a.wq[0] : (mat == 1 ? a.wq[1] : a.wq[2]);
    src[QAG] = w + (size_t)n * a.Kp + ((lane & 3) ^ ((qr >> 1) & 3)) * 16 + (size_t)kbase * WBK;
  }
  // scales: the two of a row are one dword; a wave fetches rows 64 (wave & 1)
  // + lane (four waves write each half, all the same values), so that every
  // wave counts the same number of loads
  {
    const int v = (wave & 1) * 64 + lane;
    const int mat = UPGATE ? v >> 6 : zmat;
    const int n = min (UPGATE ? n0 + (v & 63) : n0 + v, a.N - 1);
    const uint16_t *ds = mat == 0 ? a.wd[0] : (mat == 1 ? a.wd[1] : a.wd[2]);
    src[QAG + 1] = (const uint8_t *)(ds + (size_t)n * (a.Kp >> 5) + (size_t)kbase * 2);
  }

  // fragment reads
  const int fsw = (lane & 7) ^ ((lane >> 3) & 1);
  // (rows of the weight tile: for the fused pair 0 .. 63 are up, 64 .. 127 gate)
  const int brow = wn * 32 + (lane & 31);
  const int qsw = (lane >> 1) & 3;
  uint32_t aoff[4], qoff[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    {
      aoff[ks] = (wm * (QTM * 32) + (lane & 31)) * WROWB + (((2 * ks + (lane >> 5)) ^ fsw) << 4);
      qoff[ks] = QB_BASE + brow * WBK + ((ks ^ qsw) << 4) + (lane >> 5) * 8;
    }
  const uint32_t soff = QS_BASE + brow * 4;
  constexpr int BJR = UPGATE ? 64 : 32; // rows from a wave's first to its second column block

  float16v acc[QTM][QTN];
#pragma unroll
  for (int i = 0; i < QTM; ++i)
#pragma unroll
    for (int jn = 0; jn < QTN; ++jn)
#pragma unroll
      for (int q = 0; q < 16; ++q)
        acc[i][jn][q] = 0.f;

  auto issue = [&] (int kt, int st) {
#pragma unroll
    for (int i = 0; i < QAG; ++i)
      __builtin_amdgcn_global_load_lds ((const VKL_GLOBAL void *)(src[i] + (size_t)kt * WROWB),
                                        (VKL_LDS void *)(wide_lds + st * QA_BYTES + (wave + QWAVES * i) * 1024), 16,
                                        0, 0);
    __builtin_amdgcn_global_load_lds ((const VKL_GLOBAL void *)(src[QAG] + (size_t)kt * WBK),
                                      (VKL_LDS void *)(wide_lds + QB_BASE + st * QB_BYTES + wave * 1024), 16, 0, 0);
    __builtin_amdgcn_global_load_lds ((const VKL_GLOBAL void *)(src[QAG + 1] + (size_t)kt * 4),
                                      (VKL_LDS void *)(wide_lds + QS_BASE + st * QS_BYTES + (wave & 1) * 256), 4,
                                      0, 0);
  };
  issue (0, 0);
  issue (nk > 1 ? 1 : 0, 1);

  half8 af[2][2][QTM];  // [block buffer][k-slice of the block][row block]
  u32x2 bq[2][2][QTN];  // weight fragments as read (int8)
  float d[2][QTN];      // the scales of the tile's two blocks
  auto read_block = [&] (int st, int blk, int buf) {
    const int sa = st * QA_BYTES, sq = st * QB_BYTES;
#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2)
      {
        const int ks = 2 * blk + k2;
#pragma unroll
        for (int jn = 0; jn < QTN; ++jn)
          bq[buf][k2][jn] = *(const u32x2 *)(wide_lds + (qoff[ks] + sq) + jn * BJR * WBK);
#pragma unroll
        for (int i = 0; i < QTM; ++i)
          af[buf][k2][i] = *(const half8 *)(wide_lds + (aoff[ks] + sa) + i * 32 * WROWB);
      }
  };
  auto read_scales = [&] (int st) {
#pragma unroll
    for (int jn = 0; jn < QTN; ++jn)
      {
        const uint32_t sc = *(const uint32_t *)(wide_lds + (soff + st * QS_BYTES) + jn * BJR * 4);
        d[0][jn] = h2f ((uint16_t)(sc & 0xffff));
        d[1][jn] = h2f ((uint16_t)(sc >> 16));
        // (keeps the conversion out of the scaling products: as fp16 operands
        // they would become mixed-precision FMAs)
        asm volatile ("" : "+v"(d[0][jn]), "+v"(d[1][jn]));
      }
  };
  // The wave's four 32 x 32 blocks in turn, written so that the two MFMAs of one
  // stand before the sixteen scaling FMAs of the one before; the order within
  // a block is left to the compiler (pinned with scheduling barriers it ran
  // 7 % slower).
  auto multiply = [&] (int buf, const float (&dd)[QTN]) {
    half8 bfc[2][QTN];
#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
      for (int jn = 0; jn < QTN; ++jn)
        bfc[k2][jn] = q8_frag (bq[buf][k2][jn]);
    float16v part[2];
#pragma unroll
    for (int p = 0; p <= QTM * QTN; ++p)
      {
        if (p < QTM * QTN)
          {
            const int i = p / QTN, jn = p % QTN;
            float16v z;
#pragma unroll
            for (int e = 0; e < 16; ++e)
              z[e] = 0.f;
            z = __builtin_amdgcn_mfma_f32_32x32x16_f16 (af[buf][0][i], bfc[0][jn], z, 0, 0, 0);
            part[p & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16 (af[buf][1][i], bfc[1][jn], z, 0, 0, 0);
          }
        if (p > 0)
          {
            const int i = (p - 1) / QTN, jn = (p - 1) % QTN;
#pragma unroll
            for (int e = 0; e < 16; ++e)
              acc[i][jn][e] = __builtin_fmaf (part[(p - 1) & 1][e], dd[jn], acc[i][jn][e]);
          }
      }
  };
  // s_waitcnt: the loads of the newest tile may stay in flight; the one in the
  // loop also waits for the wave's own LDS reads
  constexpr int WAITVM = 0x0f70 | (QLOADS & 15) | ((QLOADS >> 4) << 14);
  __builtin_amdgcn_s_waitcnt (WAITVM);
  __builtin_amdgcn_s_barrier ();
  issue (nk > 2 ? 2 : nk - 1, 2);
  read_block (0, 0, 0);
  read_scales (0);
  __builtin_amdgcn_sched_barrier (0);
  // One k-step per turn.  On entry the fragments of block 0 of tile kt (stage
  // st = kt % 3) are in buffer 0, the scales of both its blocks in d, and the
  // loads of tiles kt + 1 and kt + 2 are in flight or done.  (One copy of the
  // step with the stage as a variable: unrolled by the stages, the
  // accumulators wander between sets of registers and the kernel spills.)
  int st = 0;
  for (int kt = 0; kt < nk; ++kt)
    {
      const int s1 = st == QSTAGES - 1 ? 0 : st + 1;
      float d1[QTN];
#pragma unroll
      for (int jn = 0; jn < QTN; ++jn)
        d1[jn] = d[1][jn];
      read_block (st, 1, 1);
      multiply (0, d[0]);
      __builtin_amdgcn_sched_barrier (0);
      // tile kt + 1 has landed (this wave's part; the barrier covers the
      // others') and this wave has read the last of tile kt: its stage takes
      // tile kt + 3 (past the end the last tile again, which nothing reads)
      __builtin_amdgcn_s_waitcnt (WAITVM & ~0x0f00);
      __builtin_amdgcn_s_barrier ();
      __builtin_amdgcn_sched_barrier (0);
      issue (kt + 3 < nk ? kt + 3 : nk - 1, st);
      read_block (s1, 0, 0);
      read_scales (s1);
      multiply (1, d1);
      __builtin_amdgcn_sched_barrier (0);
      st = s1;
    }
  __builtin_amdgcn_s_waitcnt (0x0f70); // no load may outlive the workgroup's LDS
  wide_epilogue_tile<BM, UPGATE, QTM> (a, acc, wide_lds, wave, lane, m0, n0, zmat, vec, part);
}

// A 256 x 256 tile of Q8_0 weights: eight waves of 128 x 64, three k-steps in LDS, products of
// 16 x 16 x 32, one for each block of a weight row, scaled in fp32 as above.
//
// Bound by the issue of vector instructions: 64 products, 256 scaling FMAs, 80 for the conversion
// of the weights and 20 more per wave and k-step fill 71 % of the cycles of a SIMD (matrix cores 37 %, LDS
// 20 %); a tile of 256 x 128 by the waves above spends as much on half of the products' reads.
// Each fragment of x is replaced by that of the next half step as soon as its four products are
// issued, so they need one set of registers.  The weight rows are dealt to fragments so that a
// lane ends with four neighbouring columns (of the fused pair two of up and of gate); the
// order of LDS is that of the fragments, its swizzle (row / 4) % 4.
// Same call before / now, us: 4096 x 4096 x 4096 181 / 154, 3967 rows: 13824 x 5120 768 / 668, 5120 x 13824 756 /
// 660, up/gate 13824 x 5120 1542 / 1325, three of 5120 x 5120 855 / 734; 1500 rows, up/gate 5120 x 5120 210 / 187; 1100 x
// 11008 x 4096 159 / 136.  Tried: 256 x 32 per wave (half the conversions) 151 for 153 at 4096 x 4096 x 4096,
// loads and reads dealt among the products 158, conversions of the next half step among them 153 to 162, the
// same with 256 x 128 tiles 186.
template <bool UPGATE>
__device__ __forceinline__ void
mix_q8_epilogue (const GemmArgs &a, const float4v (&acc)[8][4], uint8_t *wide_lds, int wave, int lane, int mrow, int ncol,
                 int zmat, int vec, float *part)
{
  constexpr int TM = 8, TN = 4, C = UPGATE ? 2 : 4; // columns of a lane
  const int row = (lane >> 4) * 4, col = (lane & 15) * C;
  const WideSimple<UPGATE, GemmArgs> simple (a, ncol, 16 * C, zmat, vec, part);
  if (simple.ok)
    {
      auto walk = [&] (auto with) {
        constexpr bool RES = decltype (with)::value != 0;
        constexpr int HALF = TM / 2;
#pragma unroll
        for (int i0 = 0; i0 < TM; i0 += HALF)
          {
            u32x2 res[HALF][4];
            if (RES)
#pragma unroll
              for (int i = 0; i < HALF; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                  res[i][e] = *(const VKL_GLOBAL u32x2 *)(simple.r + (size_t)min (mrow + (i0 + i) * 16 + row + e, a.M - 1) * simple.ys + col);
#pragma unroll
            for (int i = 0; i < HALF; ++i)
#pragma unroll
              for (int e = 0; e < 4; ++e)
                {
                  const int m = mrow + (i0 + i) * 16 + row + e;
                  uint16_t h[C];
#pragma unroll
                  for (int c = 0; c < C; ++c)
                    {
                      const float v = acc[i0 + i][c][e];
                      h[c] = f2h (UPGATE ? silu (acc[i0 + i][2 + c % 2][e]) * v : v);
                      if (RES)
                        h[c] = f2h (h2f (h[c]) + h2f ((uint16_t)(res[i][e][c / 2] >> ((c & 1) * 16))));
                    }
                  if (m < a.M)
                    {
                      uint16_t *o = simple.y + (size_t)m * simple.ys + col;
                      if constexpr (UPGATE)
                        *(VKL_GLOBAL uint32_t *)o = h[0] | ((uint32_t)h[1] << 16);
                      else
                        *(VKL_GLOBAL u32x2 *)o = u32x2{ h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16) };
                    }
                }
          }
      };
      if (simple.r)
        walk (WideInt<1> ());
      else
        walk (WideInt<0> ());
      return;
    }
  // through LDS, 64 rows of a wave at a time
  constexpr int PM = 4, ROWS = PM * 16, LD = kWideParkLd;
  float *park = (float *)(wide_lds + wave * (ROWS * LD * 4));
  __builtin_amdgcn_s_barrier (); // every wave (that is left) has read its last fragments
  constexpr int CPR = UPGATE ? 4 : 8, RPI = 64 / CPR; // lanes per row, rows per iteration
  const int er = lane / CPR, ec = (lane % CPR) * 8;
  const FinishRows<UPGATE, GemmArgs> fin (a, ncol + ec, zmat, vec, part);
#pragma unroll
  for (int i0 = 0; i0 < TM; i0 += PM)
    {
#pragma unroll
      for (int i = 0; i < PM; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int j = 0; j < TN; j += C)
            {
              float *dst = park + (i * 16 + row + e) * LD + (j / C) * 32 + col;
#pragma unroll
              for (int c = 0; c < C; ++c)
                dst[c] = acc[i0 + i][j + c][e];
            }
      // (a wave reads back only what it wrote itself: no barrier)
#pragma unroll 1
      for (int it = 0; it < ROWS / RPI; ++it)
        {
          const int r = it * RPI + er, m = mrow + i0 * 16 + r;
          uint4 res[2];
          fin.request (m, res);
          const float *pr = park + r * LD + ec;
          const float4v p0 = *(const float4v *)pr, p1 = *(const float4v *)(pr + 4);
          float v[8] = { p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w };
          float g[8] = { 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f };
          if (UPGATE)
            {
              const float4v g0 = *(const float4v *)(pr + 32), g1 = *(const float4v *)(pr + 36);
              g[0] = g0.x, g[1] = g0.y, g[2] = g0.z, g[3] = g0.w, g[4] = g1.x, g[5] = g1.y, g[6] = g1.z, g[7] = g1.w;
            }
          fin.store (m, v, g, res);
        }
    }
}

constexpr int kMixQ8Cols = 256;

constexpr size_t
mix_lds_q8 ()
{
  constexpr size_t wide = (size_t)QSTAGES * (WBM * WROWB + kMixQ8Cols * (WBK + 4)), park = (size_t)QWAVES * 64 * kWideParkLd * 4;
  return std::max (std::max (wide, park), wide_lds_q8<WBM> ());
}

template <bool UPGATE>
__device__ __forceinline__ void
mix_q8_tile (const GemmArgs &a, const WidePlace &at, int vec, int ksplit, float *ws)
{
  constexpr int BM = WBM, BN = kMixQ8Cols, WN = 4, TM = 8, TN = 4, ST = QSTAGES;
  constexpr int A_BYTES = BM * WROWB, Q_BYTES = BN * WBK, S_BYTES = BN * 4; // of a stage; laid out by kind
  constexpr int Q_BASE = ST * A_BYTES, S_BASE = Q_BASE + ST * Q_BYTES;
  constexpr int AG = BM / 8 / QWAVES, QG = BN / 16 / QWAVES, LOADS = AG + QG + 1; // per wave and k-step
  extern __shared__ __align__ (16) uint8_t wide_lds[];
  const int nk_all = a.K / WBK;
  const int kbase = (int)((long)nk_all * at.ks / ksplit);
  const int nk = (int)((long)nk_all * (at.ks + 1) / ksplit) - kbase;
  float *part = ksplit > 1 ? ws + (size_t)at.ks * a.M * a.N : nullptr;
  const int m0 = at.m0, n0 = at.tn * (UPGATE ? WBN / 2 : WBN);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane (threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;

  // load addresses: x as in mix_tile
  const int lr = lane >> 3, fa = (wave & 1) * 4 + (lane >> 4);
  const uint8_t *src[LOADS];
#pragma unroll
  for (int i = 0; i < AG; ++i)
    src[i] = (const uint8_t *)(a.x + (size_t)min (m0 + (wave + QWAVES * i) * 8 + lr, a.M - 1) * a.xs + ((lane & 7) ^ fa) * 8
                               + (size_t)kbase * WBK);
  // slot s of the tile holds, of wave s / 64, row s % 16 of fragment (s / 16) % 4: columns 4 (s % 16)
  // + fragment, of the fused pair 2 (s % 16) + fragment % 2 of up (fragments 0, 1) or gate
  auto weight = [&] (int s, int &n) {
    const int f = (s >> 4) & 3, r = s & 15;
    n = min (n0 + (UPGATE ? (s >> 6) * 32 + 2 * r + (f & 1) : (s >> 6) * 64 + 4 * r + f), a.N - 1);
    return UPGATE ? f >> 1 : at.zmat;
  };
  // quants: an instruction covers slots 16 g .. + 15, g = wave + 8 i; lane l fetches chunk (l % 4) ^
  // (slot / 4) % 4 of slot 16 g + l / 4
#pragma unroll
  for (int i = 0; i < QG; ++i)
    {
      const int s = (wave + QWAVES * i) * 16 + (lane >> 2);
      int n;
      const int mat = weight (s, n);
      src[AG + i] = pick3 (a.wq[0], a.wq[1], a.wq[2], mat) + (size_t)n * a.Kp + ((lane & 3) ^ ((s >> 2) & 3)) * 16 + (size_t)kbase * WBK;
    }
  // scales: the two of a row are one dword; a wave fetches 64 of the 256 rows (two waves the same)
  {
    int n;
    const int mat = weight ((wave & 3) * 64 + lane, n);
    src[AG + QG] = (const uint8_t *)(pick3 (a.wd[0], a.wd[1], a.wd[2], mat) + (size_t)n * (a.Kp >> 5) + (size_t)kbase * 2);
  }
  // fragment reads
  const int r = lane & 15;
  uint32_t aoff[2], qoff[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    {
      aoff[h] = (wm * (BM / 2) + r) * WROWB + (((4 * h + (lane >> 4)) ^ ((r >> 1) & 7)) << 4);
      qoff[h] = Q_BASE + (wn * 64 + r) * WBK + (((2 * h + (lane >> 5)) ^ ((r >> 2) & 3)) << 4) + ((lane >> 4) & 1) * 8;
    }
  const uint32_t soff = S_BASE + (wn * 64 + r) * 4;

  float4v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      acc[i][j] = float4v{ 0.f, 0.f, 0.f, 0.f };

  auto issue = [&] (int kt, int st) {
#pragma unroll
    for (int i = 0; i < AG; ++i)
      __builtin_amdgcn_global_load_lds ((const VKL_GLOBAL void *)(src[i] + (size_t)kt * WROWB),
                                        (VKL_LDS void *)(wide_lds + st * A_BYTES + (wave + QWAVES * i) * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < QG; ++i)
      __builtin_amdgcn_global_load_lds ((const VKL_GLOBAL void *)(src[AG + i] + (size_t)kt * WBK),
                                        (VKL_LDS void *)(wide_lds + Q_BASE + st * Q_BYTES + (wave + QWAVES * i) * 1024), 16, 0,
                                        0);
    __builtin_amdgcn_global_load_lds ((const VKL_GLOBAL void *)(src[AG + QG] + (size_t)kt * 4),
                                      (VKL_LDS void *)(wide_lds + S_BASE + st * S_BYTES + (wave & 3) * 256), 4, 0, 0);
  };
#pragma unroll
  for (int p = 0; p < ST; ++p)
    issue (p < nk ? p : nk - 1, p);

  half8 af[TM], bf[TN];
  u32x2 raw[TN];         // the next weight fragments as they lie
  uint32_t scales[TN];   // the next k-step's
  auto read_x = [&] (int st, int h, int i) { af[i] = *(const half8 *)(wide_lds + st * A_BYTES + aoff[h] + i * 16 * WROWB); };
  auto read_w = [&] (int st, int h) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
      raw[j] = *(const u32x2 *)(wide_lds + st * Q_BYTES + qoff[h] + j * 16 * WBK);
  };
  auto read_scales = [&] (int st) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
      scales[j] = *(const uint32_t *)(wide_lds + st * S_BYTES + soff + j * 16 * 4);
  };
  auto convert = [&] {
#pragma unroll
    for (int j = 0; j < TN; ++j)
      bf[j] = q8_frag (raw[j]);
  };
  // the products of half a k-step, each scaled behind the second one after it; the fragments of
  // x become those of half h of the k-step in stage st
  auto multiply = [&] (const float (&d)[TN], int st, int h) {
    constexpr int NP = TM * TN, BEHIND = 2;
    float4v sum[BEHIND + 1];
#pragma unroll
    for (int p = 0; p < NP + BEHIND; ++p)
      {
        if (p < NP)
          {
            sum[p % (BEHIND + 1)] = __builtin_amdgcn_mfma_f32_16x16x32_f16 (af[p / TN], bf[p % TN],
                                                                            float4v{ 0.f, 0.f, 0.f, 0.f }, 0, 0, 0);
            if (p % TN == TN - 1)
              read_x (st, h, p / TN);
          }
        if (p >= BEHIND)
          {
            const int q = p - BEHIND;
#pragma unroll
            for (int e = 0; e < 4; ++e)
              acc[q / TN][q % TN][e] = __builtin_fmaf (sum[q % (BEHIND + 1)][e], d[q % TN], acc[q / TN][q % TN][e]);
          }
      }
  };
  // s_waitcnt immediates as in mix_tile
  constexpr int V0 = (ST - 1) * LOADS, V1 = (ST - 2) * LOADS;
  constexpr int WAIT0 = 0x0f70 | (V0 & 15) | ((V0 >> 4) << 14), WAIT1 = 0x0070 | (V1 & 15) | ((V1 >> 4) << 14);
  __builtin_amdgcn_s_waitcnt (WAIT0);
  __builtin_amdgcn_s_barrier ();
#pragma unroll
  for (int i = 0; i < TM; ++i)
    read_x (0, 0, i);
  read_w (0, 0);
  read_scales (0);
  __builtin_amdgcn_sched_barrier (0);
  // One k-step per turn, as in mix_tile: between its halves tile kt + 1 has landed and the stage of
  // tile kt, whose last fragments are in registers, takes tile kt + 3.
  int st = 0;
  for (int kt = 0; kt < nk; ++kt)
    {
      const int s1 = st == ST - 1 ? 0 : st + 1;
      float d0[TN], d1[TN];
      convert ();
#pragma unroll
      for (int j = 0; j < TN; ++j)
        {
          d0[j] = h2f ((uint16_t)(scales[j] & 0xffff)), d1[j] = h2f ((uint16_t)(scales[j] >> 16));
          // (keeps the conversion out of the scaling products, see wide_q8_tile)
          asm volatile ("" : "+v"(d0[j]), "+v"(d1[j]));
        }
      read_w (st, 1);
      multiply (d0, st, 1);
      __builtin_amdgcn_sched_barrier (0);
      __builtin_amdgcn_s_waitcnt (WAIT1); // also for the wave's own LDS reads
      __builtin_amdgcn_s_barrier ();
      __builtin_amdgcn_sched_barrier (0);
      issue (kt + ST < nk ? kt + ST : nk - 1, st);
      convert ();
      read_w (s1, 0);
      read_scales (s1);
      multiply (d1, s1, 0);
      __builtin_amdgcn_sched_barrier (0);
      st = s1;
    }
  land_all (); // (up to three k-steps past the end)
  mix_q8_epilogue<UPGATE> (a, acc, wide_lds, wave, lane, m0 + wm * (BM / 2), n0 + wn * (UPGATE ? 32 : 64), at.zmat, vec, part);
}

template <bool UPGATE>
__global__ __launch_bounds__ (QWAVES * 64) void
gemm_mix_q8_kernel (const GemmArgs a, WideMix grid, int vec, int ksplit, float *ws)
{
  WidePlace at;
  switch (grid.place (a.M, WBM, at))
    {
    case 1:
      return mix_q8_tile<UPGATE> (a, at, vec, ksplit, ws);
    case 2:
      return wide_q8_tile<WBM, UPGATE> (a, at, vec, ksplit, ws);
    case 3:
      return wide_q8_tile<WBM / 2, UPGATE> (a, at, vec, ksplit, ws);
    }
}

// no pairs: tiles of 256 (or, the last, 128) rows and 128 columns, or of 128 rows.  (Beside the
// wide tile the compiler orders the k loop of these less well: 2048 x 4096 x 4096 99 us there, 93 here.)
template <int BM, bool UPGATE>
__global__ __launch_bounds__ (QWAVES * 64) void
gemm_wide_q8_kernel (const GemmArgs a, WideGrid grid, int vec, int ksplit, float *ws)
{
  WidePlace at;
  switch (grid.place<BM> (a.M, at))
    {
    case WIDE_NONE:
      return;
    case WIDE_TILE:
      return wide_q8_tile<BM, UPGATE> (a, at, vec, ksplit, ws);
    case WIDE_HALF:
      if constexpr (BM == WBM)
        return wide_q8_tile<BM / 2, UPGATE> (a, at, vec, ksplit, ws);
    }
}

// Which tile height and how many parts of the k range: the pair with the
// lowest estimated time, from a model fitted to measurements on the 7B shapes
// (microseconds: a round of 256-row tiles over the 256 compute units takes
// about 0.95 per k-step + 8, one of 128-row tiles 0.55 per k-step + 6; with Q8_0
// weights 1.35 and 0.90 per k-step, fitted on the 13B shapes at 3968 rows as
// well: every tile converts its weight fragments anew, so short tiles gain
// less there; a reduction launch 5 + its bytes at 2.5 TB/s).  The figures are older than the
// cut tiles of the last round (WideGrid), which is charged as a whole one except for the
// three fp16 matrices of one launch: their 2.25 rounds came out level with 4.5 of 128-row tiles,
// which took longer than the matrices apart (4096 x 4096, 1300 / 1500 rows: 1.07 / 1.12 of that;
// in 256-row tiles 0.91 / 0.94, 158 / 164 us).
// (The fp16 tiles have become faster since, those of 256 rows more than those of 128; the
// choices for the 7B and 13B shapes are held by tests/test_gemm_plan.py.)
// Below kWideMinGroups workgroups the tile kernel of vkl_gemm_mfma.hip does
// better.
constexpr int kWideMinRows = 128;
// From 65 rows on (where the tile kernel needs a second row of 64-row tiles) in
// one partly empty row of 128-row tiles: fp16 weights, the fused up/gate pair,
// and Q8_0 products with K up to 5120.  Measured at 80-127 rows: fp16 4096^2
// 20-23 -> 16-17 us, 12288 x 4096 41-43 -> 35-39, up/gate 62-67 -> 47-50 (13B
// 89-97 -> 65-70), down even; Q8_0 up/gate 84 -> 66 (13B 108 -> 92), 4096^2
// 27 -> 24.  Not the Q8_0 down product (K = 11008: 39 -> 42 us), and nothing
// below 65 rows (13B Q8_0 up/gate at 64 rows: 83 against 88 us).
constexpr int kWideMinRowsPartial = 65;
constexpr int kWideMinGroups = 88, kWideMinGroupsQ8 = 128;

struct WidePlan
{
  int bm;                  // token rows of a tile, 0: this form does not apply
  int ksplit;              // parts of the k range
  bool four_waves = false; // (bf16) tiles of 256 or 128 rows and 128 columns by four waves, see launch_bf16_tiles
};

long
wide_tiles (const GemmArgs &a, int bm)
{
  return (long)((a.M + bm - 1) / bm) * ((a.N + (a.upgate ? 63 : 127)) / (a.upgate ? 64 : 128))
         * (a.upgate ? 1 : a.nmat);
}

WidePlan
wide_plan (const GemmArgs &a)
{
  WidePlan none = { 0, 1 }, best = none;
  const int min_rows = a.wtype == 1 || a.upgate || a.K <= 5120 ? kWideMinRowsPartial : kWideMinRows;
  if ((a.wtype != 1 && a.wtype != 8) || a.batch > 1 || (a.K % WBK) != 0 || a.M < min_rows)
    return none;
  if (a.wtype == 8)
    {
      // whole k-steps of quants and scale pairs, aligned for 16- and 4-byte loads
      if (a.Kp != a.K)
        return none;
      for (int t = 0; t < (a.upgate ? 2 : a.nmat); ++t)
        if (((uintptr_t)a.wq[t] % 16) != 0 || ((uintptr_t)a.wd[t] % 4) != 0)
          return none;
    }
  const int nk = a.K / WBK;
  const size_t ws_bytes = a.workspace ? a.workspace_bytes : StreamScratch::bytes ();
  double best_cost = 0;
  for (int bm = 128; bm <= WBM; bm *= 2)
    for (int ks = 1; ks <= 4; ks *= 2)
      {
        // (a single row of 128-row tiles may be partly empty)
        if (a.M < bm && !(bm == 128 && a.M >= min_rows))
          continue;
        // parts only for one matrix with the plain epilogue, of at least 16
        // k-steps each, and as far as the scratch holds them
        if (ks > 1
            && (a.upgate || a.nmat != 1 || nk / ks < 16 || (size_t)ks * a.M * a.N * sizeof (float) > ws_bytes))
          continue;
        const long groups = wide_tiles (a, bm) * ks;
        if (groups < (a.wtype == 8 ? kWideMinGroupsQ8 : kWideMinGroups))
          continue;
        const double per_step = a.wtype == 8 ? (bm == WBM ? 1.35 : 0.90) : (bm == WBM ? 0.95 : 0.55);
        const double round = per_step * nk / ks + (bm == WBM ? 8 : 6);
        const double reduce = ks > 1 ? 5 + (double)ks * a.M * a.N * sizeof (float) / 2.5e6 : 0;
        const long rest = groups % WideGrid::kUnits;
        const bool cut = bm == WBM && a.wtype == 1 && a.nmat == 3 && rest > 0 && rest <= WideGrid::kUnits / 2;
        const double last = cut ? 0.55 * nk + 6 : rest > 0 ? round : 0;
        const double cost = (double)(groups / WideGrid::kUnits) * round + last + reduce;
        if (!best.bm || cost < best_cost)
          best = { bm, ks }, best_cost = cost;
      }
  return best;
}
} // namespace

bool
gemm_wide_supported (const GemmArgs &a)
{
  return wide_plan (a).bm != 0;
}

void
gemm_wide_choice (const GemmArgs &a, int *tile_rows, int *ksplit)
{
  const WidePlan p = wide_plan (a);
  *tile_rows = p.bm, *ksplit = p.bm ? p.ksplit : 1;
}

// The time of the tiles by mix_time.  Q8_0 in tiles of 128 rows, which that does not know, takes 0.65 of 256 rows (us of one round: 2048 wide
// 27.6 / 42.2, 1024 wide 16.7 / 25.5).
double
gemm_wide_us (const GemmArgs &a)
{
  const WidePlan p = wide_plan (a);
  if (!p.bm)
    return 0;
  const int tiles_m = (a.M + p.bm - 1) / p.bm, tiles_n = (a.N + (a.upgate ? 63 : 127)) / (a.upgate ? 64 : 128), mats = a.upgate ? 1 : a.nmat;
  const double steps = (double)(a.K / WBK) / p.ksplit;
  if (a.wtype == 8 && p.bm == 128)
    {
      const MixTime t = mix_time (WBM, 1, false, true);
      return (wide_tiles (a, p.bm) * p.ksplit + WideGrid::kUnits - 1) / WideGrid::kUnits * 0.65 * (t.step * steps + t.start);
    }
  double us = 0;
  WideMix (p.bm, tiles_m, tiles_n, mats, p.ksplit, steps, 0, &us, a.wtype == 8);
  return us;
}

size_t
gemm_wide_workspace_bytes (const GemmArgs &a)
{
  const WidePlan p = wide_plan (a);
  return p.bm && p.ksplit > 1 ? (size_t)p.ksplit * a.M * a.N * sizeof (float) : 0;
}

int
gemm_wide_launch (const GemmArgs &a, hipStream_t s, GemmNorm *norm)
{
  constexpr size_t m256 = mix_lds<256> (), m128 = mix_lds<128> ();
  constexpr size_t qmix = mix_lds_q8 (), q256 = wide_lds_q8<256> (), q128 = wide_lds_q8<128> ();
  constexpr int NK = 10;
  static LdsLimit limits[NK];
  const void *const kernels[NK]
      = { (const void *)gemm_mix_kernel<256, false, GemmArgs>, (const void *)gemm_mix_kernel<256, true, GemmArgs>,
          (const void *)gemm_mix_kernel<128, false, GemmArgs>, (const void *)gemm_mix_kernel<128, true, GemmArgs>,
          (const void *)gemm_mix_q8_kernel<false>, (const void *)gemm_mix_q8_kernel<true>,
          (const void *)gemm_wide_q8_kernel<256, false>, (const void *)gemm_wide_q8_kernel<256, true>,
          (const void *)gemm_wide_q8_kernel<128, false>, (const void *)gemm_wide_q8_kernel<128, true> };
  const size_t need[NK] = { m256, m256, m128, m128, qmix, qmix, q256, q256, q128, q128 };
  for (int i = 0; i < NK; ++i)
    if (int e = limits[i].raise (kernels[i], need[i]))
      return e;
  const WidePlan plan = wide_plan (a);
  const int bm = plan.bm;
  int ksplit = plan.ksplit;
  if (!bm)
    return (int)hipErrorInvalidValue;
  StreamScratch own;
  float *ws = nullptr;
  if (ksplit > 1 && !(ws = a.workspace ? a.workspace : own.take (s)))
    ksplit = 1;
  const int tiles_m = (a.M + bm - 1) / bm;
  const int tiles_n = (a.N + (a.upgate ? 63 : 127)) / (a.upgate ? 64 : 128);
  const bool q8 = a.wtype == 8;
  const WideGrid tiles (tiles_m, tiles_n, a.upgate ? 1 : a.nmat, ksplit, bm == WBM);
  const WideMix mix (bm, tiles_m, tiles_n, a.upgate ? 1 : a.nmat, ksplit, (double)(a.K / WBK) / ksplit, 0, nullptr, q8);
  const bool pairs = !q8 || (bm == WBM && mix.wide > 0);
  const dim3 grid ((unsigned)(pairs ? mix.groups () : tiles.groups ()));
  const dim3 block ((q8 ? QWAVES : MWAVES) * 64);
  // 16-byte accesses to the outputs (and the residual) where their rows allow it
  int vec = (a.ys % 8) == 0 && (!a.residual || ((uintptr_t)a.residual % 16) == 0)
            && (!a.y32 || ((a.N % 4) == 0 && ((uintptr_t)a.y32 % 16) == 0));
  for (int t = 0; t < (a.upgate ? 1 : a.nmat); ++t)
    vec = vec && ((uintptr_t)a.y[t] % 16) == 0;
  if (q8 && pairs)
    {
      if (a.upgate)
        gemm_mix_q8_kernel<true><<<grid, block, qmix, s>>> (a, mix, vec, ksplit, ws);
      else
        gemm_mix_q8_kernel<false><<<grid, block, qmix, s>>> (a, mix, vec, ksplit, ws);
    }
  else if (q8 && bm == 256)
    {
      if (a.upgate)
        gemm_wide_q8_kernel<256, true><<<grid, block, q256, s>>> (a, tiles, vec, ksplit, ws);
      else
        gemm_wide_q8_kernel<256, false><<<grid, block, q256, s>>> (a, tiles, vec, ksplit, ws);
    }
  else if (q8)
    {
      if (a.upgate)
        gemm_wide_q8_kernel<128, true><<<grid, block, q128, s>>> (a, tiles, vec, ksplit, ws);
      else
        gemm_wide_q8_kernel<128, false><<<grid, block, q128, s>>> (a, tiles, vec, ksplit, ws);
    }
  else if (bm == 256)
    {
      if (a.upgate)
        gemm_mix_kernel<256, true, GemmArgs><<<grid, block, m256, s>>> (a, mix, vec, ksplit, ws);
      else
        gemm_mix_kernel<256, false, GemmArgs><<<grid, block, m256, s>>> (a, mix, vec, ksplit, ws);
    }
  else if (a.upgate)
    gemm_mix_kernel<128, true, GemmArgs><<<grid, block, m128, s>>> (a, mix, vec, ksplit, ws);
  else
    gemm_mix_kernel<128, false, GemmArgs><<<grid, block, m128, s>>> (a, mix, vec, ksplit, ws);
  if (ksplit > 1)
    return gemm_reduce_parts (a, ws, ksplit, a.M, s, norm);
  return (int)hipGetLastError ();
}

// ---------------------------------------------------------------------------
// bf16 operands, output columns in segments
// ---------------------------------------------------------------------------
namespace
{
// wide_f32_again for sums of parts: v the sums of E columns from n on of row m, in every
// lane of a wave others.  The wave forms the sums of a lane that has one that is not finite
// together, 512 values of k at a time.
template <int E>
__device__ __forceinline__ void
seg_f32_again (const GemmSegArgs &a, float (&v)[E], int m, int n, int lane, int K)
{
  float t = 0.f;
#pragma unroll
  for (int e = 0; e < E; ++e)
    t = __builtin_fmaf (v[e], 0.f, t);
  uint64_t bad = __builtin_amdgcn_ballot_w64 (t != 0.f);
#pragma unroll 1
  while (bad)
    {
      const int who = __builtin_ctzll (bad);
      bad &= bad - 1;
      const float *x = a.xf + (size_t)__builtin_amdgcn_readlane (m, who) * a.xs;
      const int n0 = __builtin_amdgcn_readlane (n, who);
      float sum[E];
#pragma unroll
      for (int e = 0; e < E; ++e)
        sum[e] = 0.f;
#pragma unroll 1
      for (int k = lane * 8; k < K; k += 64 * 8)
        {
          const uint4 x0 = ldg4 (x + k), x1 = ldg4 (x + k + 4);
          const uint32_t xw[8] = { x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w };
#pragma unroll
          for (int e = 0; e < E; ++e)
            {
              const uint4 w0 = ldg4 (a.wh[0] + (size_t)min (n0 + e, a.N - 1) * a.ws + k);
              const uint32_t ww[4] = { w0.x, w0.y, w0.z, w0.w };
#pragma unroll
              for (int j = 0; j < 8; ++j)
                sum[e] = __builtin_fmaf (__uint_as_float (xw[j]), bf2f ((uint16_t)(ww[j >> 1] >> (16 * (j & 1)))), sum[e]);
            }
        }
#pragma unroll
      for (int e = 0; e < E; ++e)
        {
#pragma unroll
          for (int d = 32; d > 0; d >>= 1)
            sum[e] += __shfl_xor (sum[e], d, 64);
          if (lane == who && __builtin_fmaf (v[e], 0.f, 0.f) != 0.f)
            v[e] = sum[e];
        }
    }
}

// adds the parts of a split k range in order and applies the segments' epilogue; the
// values of four parts are requested at a time.  PLANES: a product of planes.
constexpr int kSegReduce = 64; // threads: few values, spread over many compute units
template <bool PLANES>
__global__ __launch_bounds__ (kSegReduce) void
wide_reduce_seg_kernel (const GemmSegArgs a, const float *ws, int parts)
{
  const int n8 = (a.N + 7) / 8;
  const size_t all = (size_t)a.M * n8;
  size_t i = (size_t)blockIdx.x * kSegReduce + threadIdx.x;
  const bool live = i < all;
  if (!PLANES && !live)
    return;
  i = live ? i : all - 1;
  const int m = (int)(i / n8), n = (int)(i % n8) * 8;
  const size_t at = (size_t)m * a.N, part = (size_t)a.M * a.N;
  float v[8], g[8];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    v[e] = 0.f, g[e] = 0.f;
  if ((a.N % 8) == 0)
    for (int p0 = 0; p0 < parts; p0 += 4)
      {
        float4 x[4][2];
#pragma unroll
        for (int p = 0; p < 4; ++p)
          {
            const float *src = ws + (size_t)min (p0 + p, parts - 1) * part + at + n;
            x[p][0] = __builtin_bit_cast (float4, ldg4 (src)), x[p][1] = __builtin_bit_cast (float4, ldg4 (src + 4));
          }
#pragma unroll
        for (int p = 0; p < 4; ++p)
          if (p0 + p < parts)
            {
              v[0] += x[p][0].x, v[1] += x[p][0].y, v[2] += x[p][0].z, v[3] += x[p][0].w;
              v[4] += x[p][1].x, v[5] += x[p][1].y, v[6] += x[p][1].z, v[7] += x[p][1].w;
            }
      }
  else
    for (int p = 0; p < parts; ++p)
      {
        const float *src = ws + (size_t)p * part + at;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          v[e] += ldg (src + min (n + e, a.N - 1));
      }
  if (PLANES)
    {
      seg_f32_again (a, v, m, n, (int)threadIdx.x, a.K / kPlanes);
      if (!live)
        return;
    }
  gemm_finish8<false> (a, v, g, m, n, 0, 0, nullptr);
}

// As wide_plan, with every row count allowed and, where the tiles are few, up to 16 parts
// of at least 4 k-steps: with few token rows the workgroups exist to stream the weights.
// The model is the time of the tiles (WideMix) and that of the reduction.  Tiles of 64 rows have two workgroups to a
// compute unit, or where each gets one at most six stages of loads (deep64).  Where a segment's sums are parked in LDS a
// tile takes longer (MixTime), which parts leave to the reduction.
// The constants are fitted to the choice they make among all plans of 646 bf16 products, each with and without GELU,
// 2 to 2200 rows, 512 to 16128 columns, K = 512 to 15104, weights that no cache holds: 1.6 % slower than the best plan in
// the mean, and in 7 of the 1292 more than 2.5 % (at most 5) slower than the plans of tiles of four waves alone that they
// replaced.  Constants fitted to the mean only, without any tiles of four waves above 64 rows, were 3.3 % off and slower
// in 119, us then / now: 33 x 16128 x 4096 35.2 / 31.3, 128 x 4096 x 11008 33.0 / 31.3,
// 160 x 4096 x 4096 21.3 / 20.0, 1500 x 5504 x 2048 52.3 / 42.7, 1100 x 2048 x 5504 48.4 / 42.0, 160 x 8064 x 2048 with GELU
// 23.1 / 19.0.
// Beyond 128 rows, tiles of 64 in one part where each compute unit gets one at most and no sums are parked: us
// without / with them 512 x 2048 x 2048 19.5 / 15.4, 300 x 2048 x 2048 18.0 / 15.5, 200 x 8192 x 2048 20.9 / 15.7.
// With GELU they would gain as much (600 x 2048 x 2048 21.5 / 19.1), and up to 192 rows with more
// than 128 tiles (192 x 5504 x 2048 20.6 / 17.5), but a product of either kind is held to be in
// parts (tests/test_gemm_f32.py), which these tiles are not.
// (a tile's waves walk 64 parked rows at a time)
double
mix_park (const GemmSegArgs &a)
{
  bool parked = false; // see WideSimple
  for (int i = 0; i < a.nseg; ++i)
    parked = parked || !a.seg[i].vec || a.seg[i].cap > 0.f || (a.seg[i].act != VKL_ACT_NONE && a.seg[i].act != VKL_ACT_RELU2);
  return parked ? std::min (1.0, a.M / 64.0) : 0;
}

// whether every compute unit gets one tile at most, which then may have all of its LDS
bool
one_round (const GemmSegArgs &a, int bm, int ksplit)
{
  return (long)((a.M + bm - 1) / bm) * ((a.N + WBN - 1) / WBN) * ksplit <= WideGrid::kUnits;
}
constexpr int kDeep64 = 6, kDeepPlanes = 4; // stages of 64-row tiles then

// (a tile of fewer k-steps would wait for all of them before its first product: 33 x 3072 x 1024 in four parts 10.0 us
// with six stages, 9.7 with three)
bool
deep64 (const GemmSegArgs &a, int ksplit)
{
  return one_round (a, 64, ksplit) && a.K / WBK / ksplit >= kDeep64 - 1;
}

// 256 x 128 tiles that leave a quarter of the compute units and more without one and are full of rows (see launch_bf16_tiles)
bool
four256 (const GemmSegArgs &a, int ksplit, int tiles, double park)
{
  return ksplit == 1 && park == 0 && tiles > WideGrid::kUnits / 2 && tiles <= WideGrid::kUnits * 3 / 4 && a.K / WBK <= 64
         && a.M >= (a.M + WBM - 1) / WBM * (WBM / 8 * 7);
}

// Parts that are no power of two fill the compute units where powers leave a quarter to a half of them idle (us, without / with:
// 1200 x 4096 x 15104 177 / 141, 600 x 4096 x 15104 96 / 87, 1200 x 2048 x 7552 58.9 / 49.6, 300 x 4096 x 11008 50.6 / 47.2).
// They are taken where they promise 4 % (of 391 products of 131 to 2100 rows none of 150 rows and more got more than 5 %
// slower than by the parts before them, the mean is 0.989 of the time; with 8 % promised 0.990), by tiles of 128, 192 and 256 rows, and
// from 144 rows on: below, the model takes tiles of few rows for faster than they are (131 x 4096 x 11008 38.0 / 43.1, 77 x 12576 x
// 4096 30.0 / 36.5).  192 rows take five or three parts in one of 300 products: powers of two and other tiles / these, 366 x 3072 x
// 11264 46.6 / 40.8, 288 x 3072 x 8192 34.1 / 31.2, 528 x 2048 x 7552 36.0 / 31.7 (which 128 rows in three parts do in 30.2).
constexpr double kOddParts = 0.96;
constexpr int kOddRows = 144;

// A last row of 256-row tiles that holds at most 64 rows takes less than the model says.  Tiles of 192 rows that leave a quarter of the
// compute units without one have to promise 2.5 % there: us, 256 rows / 192, 555 x 7680 x 5120 57.0 / 61.1, 2074 x 2048 x
// 7552 79.7 / 82.3, 2078 x 2048 x 5504 65.0 / 64.8, 1298 x 3072 x 8192 85.0 / 80.9; more tiles of 192 rows stay faster (1049 x 4096
// x 4096 49.7 / 45.6, 1049 x 5120 x 5120 64.5 / 60.4).  2833 products of 144 to 2300 rows, all whose tiles are not those of powers of two
// and 64, 128 and 256 rows, take 0.886 of the time with those, and none is more than 2 % slower.
constexpr int kShortRows = 64;
constexpr double kFew192 = 0.975;

WidePlan
wide_plan_bf16 (const GemmSegArgs &a, size_t scratch)
{
  // 64-row tiles, one and two workgroups per compute unit: one or two rows of them stream the
  // weights, more share them in the L2; the reduction; 128-row tiles by four waves
  const bool few = a.M <= 128;
  const double one64 = few ? 0.57 : 0.42, first64 = few ? 1.69 : 3.0, two64 = few ? 0.75 : 1.07, round64 = few ? 6.5 : 2.48;
  const double park64 = few ? 3.5 : 5.9, shallow64 = few ? 1.0 : 0.5, reduce0 = few ? 6.3 : 3.7, rate = few ? 3.0e6 : 1.9e6;
  const double step4 = few ? 0.76 : 0.54, start4 = few ? 5.5 : 3.9;
  WidePlan best = { 0, 1 };
  double best_cost = 0;
  const int nk = a.K / WBK, tiles_n = (a.N + WBN - 1) / WBN;
  const double parked = mix_park (a);
  for (int bm = 64; bm <= WBM; bm += 64)
    for (int ks = 1; ks <= 16; ++ks)
      {
        const bool odd = (ks & (ks - 1)) != 0; // no power of two
        if (odd && (a.M < kOddRows || bm == 64))
          continue;
        const int tiles_m = (a.M + bm - 1) / bm, tiles = tiles_m * tiles_n * ks;
        if (a.M < bm && bm > 128)
          continue;
        if (bm == 64 && !few && (tiles > WideGrid::kUnits || ks > 4 || (ks == 1 && (parked > 0 || (a.M <= 192 && tiles > 128)))))
          continue;
        // (parts that fill the compute units four times gain nothing)
        if (ks > 1
            && (nk / ks < 4 || (size_t)ks * a.M * a.N * sizeof (float) > scratch || tiles > 4 * 2 * WideGrid::kUnits))
          continue;
        const double steps = (double)nk / ks, park = ks == 1 ? parked : 0;
        double cost = 0;
        if (bm == 64)
          {
            const double p = ks == 1 && parked > 0 ? std::min (1.0, a.M / 32.0) * park64 : 0;
            const int two = tiles / (2 * WideGrid::kUnits), rest = tiles % (2 * WideGrid::kUnits);
            const double round = two64 * steps + round64 + p;
            cost = two * round;
            if (rest > 0)
              cost += rest <= WideGrid::kUnits ? one64 * steps + first64 + p : round;
            if (tiles <= WideGrid::kUnits && !deep64 (a, ks))
              cost += shallow64;
          }
        else
          WideMix (bm, tiles_m, tiles_n, 1, ks, steps, park, &cost);
        const double reduce = ks > 1 ? reduce0 + (double)ks * a.M * a.N * sizeof (float) / rate : 0;
        const bool few192 = best.bm == 192 && best.ksplit == 1 && (a.M + 191) / 192 * tiles_n <= WideGrid::kUnits * 3 / 4;
        const bool short256 = bm == WBM && ks == 1 && tiles_m * bm - a.M >= bm - kShortRows;
        const double promise = odd ? kOddParts : few192 && short256 ? 1 / kFew192 : 1.0;
        if (!best.bm || cost + reduce < promise * best_cost)
          best = { bm, ks, bm == WBM && four256 (a, ks, tiles, park) }, best_cost = cost + reduce;
        if (bm != 128 || tiles <= WideGrid::kUnits / 2 || park > 0)
          continue;
        cost = (tiles + WideGrid::kUnits - 1) / WideGrid::kUnits * (step4 * steps + start4);
        if (cost + reduce < (odd ? kOddParts : 1.0) * best_cost)
          best = { bm, ks, true }, best_cost = cost + reduce;
      }
  return best;
}

// The tiles of a product of planes: 64 rows in up to 16 parts of the k range (one and two
// workgroups to a compute unit, as above), or wide_bf16_tile's 256 rows, the last of which may be
// cut.  Fitted to 160 products of 2 to 2048 rows in 1 to 16 parts and 151 of 192 to 2048 rows in
// both forms, all in two stages (four take 0.8 to 0.95 of that where a compute unit has one tile, in one
// part or several): 0.5 % slower than the best plan in the mean, 7 at worst; without 256 rows 2.5 % and 22
// (2048 x 8064 x 2048 187 us with them, 229 without; 512 x 16128 x 4096 175, 199).
// Three, five, six and seven parts are taken where they promise 8 %: of 204 products of 2 to 532 rows (weights that no cache
// holds) 0.988 of the time in the mean, none more than 2.2 % slower; us, powers of two / now: 300 x 2048 x 5504 42.7 / 36.3, 300 x 4096 x
// 4096 54.7 / 45.7, 300 x 4096 x 11008 110.2 / 94.8, 181 x 6416 x 2048 35.4 / 30.3.  With 4 % promised seven were 2 to 6 % slower, and so are nine and
// more parts.
constexpr double kOddPlanes = 0.92;
constexpr int kOddPlaneParts = 7;

WidePlan
wide_plan_planes (const GemmSegArgs &a, size_t scratch)
{
  const int nk = a.K / WBK / kPlanes, tiles_n = (a.N + WBN - 1) / WBN;
  WidePlan best = { kPlaneRows, 1 };
  double best_cost = 0;
  for (int ks = 1; ks <= 16; ++ks)
    {
      const bool odd = (ks & (ks - 1)) != 0; // no power of two
      if (odd && ks > kOddPlaneParts)
        continue;
      if (ks > 1 && (nk / ks < 4 || (size_t)ks * a.M * a.N * sizeof (float) > scratch))
        continue;
      const int tiles = (a.M + kPlaneRows - 1) / kPlaneRows * tiles_n * ks;
      const int two = tiles / (2 * WideGrid::kUnits), rest = tiles % (2 * WideGrid::kUnits);
      const double steps = (double)nk / ks, round = 1.14 * steps + 6.4;
      double cost = two * round + (ks > 1 ? 4.2 + (double)ks * a.M * a.N * sizeof (float) / 3.8e6 : 0);
      if (rest > 0)
        cost += rest <= WideGrid::kUnits ? 0.935 * steps + 1.6 : round;
      if (ks == 1 || cost < (odd ? kOddPlanes : 1.0) * best_cost)
        best.ksplit = ks, best_cost = cost;
    }
  if (a.M >= WBM)
    {
      const WideGrid tiles ((a.M + WBM - 1) / WBM, tiles_n, 1, 1, true);
      const int whole = (tiles.whole + WideGrid::kUnits - 1) / WideGrid::kUnits;
      if (whole * (1.97 * nk + 9.6) + (tiles.whole < tiles.tiles () ? 1.44 * nk + 6.6 : 0) < best_cost)
        best = { WBM, 1 };
    }
  return best;
}

WideMix
mix_tiles (const GemmSegArgs &a, int bm, int ksplit)
{
  return WideMix (bm, (a.M + bm - 1) / bm, (a.N + WBN - 1) / WBN, 1, ksplit, (double)(a.K / WBK) / ksplit,
                  ksplit == 1 ? mix_park (a) : 0);
}

// ws: scratch for the parts of the k range, whose sums the caller adds
template <int BM>
int
launch_mix_parts (const GemmSegArgs &a, int ksplit, float *ws, hipStream_t s)
{
  static LdsLimit limit;
  constexpr size_t lds = mix_lds<BM> ();
  const auto kernel = gemm_mix_kernel<BM, false, GemmSegArgs>;
  if (int e = limit.raise ((const void *)kernel, lds))
    return e;
  const WideMix tiles = mix_tiles (a, BM, ksplit);
  kernel<<<dim3 ((unsigned)tiles.groups ()), dim3 (MWAVES * 64), lds, s>>> (a, tiles, 1, ksplit, ws);
  return (int)hipGetLastError ();
}

template <int BM, int ST, int PLANES = 1>
int
launch_wide_parts (const GemmSegArgs &a, int ksplit, float *ws, hipStream_t s)
{
  static LdsLimit limit;
  constexpr size_t lds = wide_lds_bf16<BM, ST> ();
  const auto kernel = gemm_wide_bf16_kernel<BM, PLANES, ST>;
  if (int e = limit.raise ((const void *)kernel, lds))
    return e;
  const WideGrid tiles ((a.M + BM - 1) / BM, (a.N + WBN - 1) / WBN, 1, ksplit, BM == WBM);
  kernel<<<dim3 ((unsigned)tiles.groups ()), dim3 (WWAVES * 64), lds, s>>> (a, tiles, ksplit, ws);
  return (int)hipGetLastError ();
}

// The tiles of a bf16 product.  128 rows by four waves take 0.52 per k-step + 3.6 us, by eight 0.46 + 5.0: the shorter the
// k range of a tile, the better.  They are weighed where more than 128 tiles leave none to be cut and no sums are parked
// (us, eight / four waves: 650 x 3072 x 1024 11.6 / 10.6, 77 x 4096 x 11008 in eight parts 29.2 / 27.9, 160 x 4096 x 4096 in
// four 23.3 / 20.0; parked 10 to 15 % slower).
// 256 rows by four waves are level with eight over most of one round of tiles, and slower with more tiles, longer k ranges
// and parked sums.  What is left to them (four256) takes 0.965 to 1.014 of the time, 0.986 in the mean of 18: 700 x 8064 x 2048
// 31.4 / 30.3, 750 x 5504 x 2048 30.6 / 29.9, 512 x 12288 x 4096 57.3 / 55.8; with more tiles or tiles less full of rows
// 0.98 to 1.03.
int
launch_bf16_tiles (const GemmSegArgs &a, const WidePlan &p, float *ws, hipStream_t s)
{
  if (p.bm == WBM)
    return p.four_waves ? launch_wide_parts<WBM, WSTAGES> (a, p.ksplit, ws, s) : launch_mix_parts<WBM> (a, p.ksplit, ws, s);
  if (p.bm == 192)
    return launch_mix_parts<192> (a, p.ksplit, ws, s);
  if (p.bm == 128)
    return p.four_waves ? launch_wide_parts<128, WSTAGES> (a, p.ksplit, ws, s) : launch_mix_parts<128> (a, p.ksplit, ws, s);
  return deep64 (a, p.ksplit) ? launch_wide_parts<64, kDeep64> (a, p.ksplit, ws, s)
                              : launch_wide_parts<64, WSTAGES> (a, p.ksplit, ws, s);
}

// the tiles of a product of planes
template <int STAGES>
int
launch_planes_parts (const GemmSegArgs &a, int ksplit, float *ws, hipStream_t s)
{
  static LdsLimit limit;
  constexpr size_t lds = wide_lds_planes<STAGES> ();
  if (int e = limit.raise ((const void *)gemm_wide_planes_kernel<STAGES>, lds))
    return e;
  const WideGrid tiles ((a.M + kPlaneRows - 1) / kPlaneRows, (a.N + WBN - 1) / WBN, 1, ksplit, false);
  gemm_wide_planes_kernel<STAGES><<<dim3 ((unsigned)tiles.groups ()), dim3 (WWAVES * 64), lds, s>>> (a, tiles, ksplit, ws);
  return (int)hipGetLastError ();
}

int
launch_planes_tiles (const GemmSegArgs &a, const WidePlan &p, float *ws, hipStream_t s)
{
  return p.bm == WBM                               ? launch_wide_parts<WBM, WSTAGES, kPlanes> (a, 1, nullptr, s)
         : one_round (a, kPlaneRows, p.ksplit) ? launch_planes_parts<kDeepPlanes> (a, p.ksplit, ws, s)
                                                   : launch_planes_parts<2> (a, p.ksplit, ws, s);
}

template <bool PLANES>
int
launch_reduce_seg (const GemmSegArgs &a, int ksplit, const float *ws, hipStream_t s)
{
  if (ksplit > 1)
    {
      const size_t total = (size_t)a.M * ((a.N + 7) / 8);
      wide_reduce_seg_kernel<PLANES><<<dim3 ((unsigned)((total + kSegReduce - 1) / kSegReduce)), dim3 (kSegReduce), 0, s>>> (a, ws, ksplit);
    }
  return (int)hipGetLastError ();
}

// a product of planes and, if it is in parts, their sum; ws: scratch for the parts
int
launch_planes (const GemmSegArgs &a, size_t bytes, float *ws, hipStream_t s)
{
  const WidePlan p = wide_plan_planes (a, bytes);
  if (int e = launch_planes_tiles (a, p, ws, s))
    return e;
  return launch_reduce_seg<true> (a, p.ksplit, ws, s);
}

// ---------------------------------------------------------------------------
// 32-bit activations on the bf16 matrix cores
// ---------------------------------------------------------------------------
// An fp32 value is the sum of three bf16 values (its 24 significant bits, eight at
// a time), and a product of two bf16 values is exact in fp32: x W^T is the product
// of three planes of x with the same weights, summed in the same fp32 accumulator,
// without any rounding that the 32-bit matrix instructions would not do (they add
// one product at a time, these sixteen before they round).  The matrix cores do
// three such products in a fifth of the time of one in fp32.  Against 64 bits the
// result is closer than that of the 32-bit instructions: relative error 1.3e-7 to 4e-7
// (1.6e-7 to 7e-7 where the lower planes share the first one's accumulators) instead
// of 8e-7 to 1.4e-6 over K = 2048 to 7552.
//
// What this does not hold for: an infinite weight meets zeros in the lower planes, and
// of values below 2^-110 the last bits lie below the smallest bf16 number, 2^-133 (the
// matrix cores take numbers below the smallest normal one as they are).  Such a value gets
// a NaN for its third plane, and sums that are not finite are formed again by the 32-bit
// instructions (wide_f32_again; sums of parts of a split k range by seg_f32_again).
//
// Planes lie in blocks of 64 columns, [plane 0 | plane 1 | plane 2] of a block next to
// each other: one k-step of gemm_wide_planes_kernel, three of wide_bf16_tile, which walks
// them as one row of 3 K values and takes every k-step of the weights three times.

// the planes of one value
__device__ __forceinline__ void
split_value (uint32_t in, uint32_t (&p)[kPlanes])
{
  // truncation: no plane overflows, and each remainder is exact.  Infinities and
  // NaN go into the first plane alone.  A last remainder (of the smallest values)
  // marks the third.
  const bool finite = (in & 0x7f800000u) != 0x7f800000u;
  const float v = __uint_as_float (in);
  p[0] = finite ? in >> 16 : (uint32_t)f2bf (v);
  const float r = finite ? v - __uint_as_float (in & 0xffff0000u) : 0.f;
  p[1] = __float_as_uint (r) >> 16;
  const uint32_t last = __float_as_uint (r - __uint_as_float (__float_as_uint (r) & 0xffff0000u));
  p[2] = (last & 0xffffu) ? 0x7fc0u : last >> 16;
}

__global__ __launch_bounds__ (256) void
split_planes_kernel (const float *x, size_t xs, int M, int K, uint16_t *out)
{
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  const int k8 = K / 8;
  if (i >= (size_t)M * k8)
    return;
  const int m = (int)(i / k8), c = (int)(i % k8) * 8;
  const float *src = x + (size_t)m * xs + c;
  const uint4 w0 = ldg4 (src), w1 = ldg4 (src + 4);
  const uint32_t in[8] = { w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w };
  uint32_t p[kPlanes][8];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    {
      uint32_t one[kPlanes];
      split_value (in[e], one);
#pragma unroll
      for (int q = 0; q < kPlanes; ++q)
        p[q][e] = one[q];
    }
  uint16_t *dst = out + (size_t)m * kPlanes * K + (size_t)(c / WBK) * kPlanes * WBK + c % WBK;
#pragma unroll
  for (int q = 0; q < kPlanes; ++q)
    {
      vkl_u32x4 pk;
      pk.x = p[q][0] | (p[q][1] << 16), pk.y = p[q][2] | (p[q][3] << 16);
      pk.z = p[q][4] | (p[q][5] << 16), pk.w = p[q][6] | (p[q][7] << 16);
      *(VKL_GLOBAL vkl_u32x4 *)(dst + q * WBK) = pk;
    }
}
} // namespace

int
gemm_wide_bf16_launch (const GemmSegArgs &a, hipStream_t s)
{
  WidePlan p = wide_plan_bf16 (a, StreamScratch::bytes ());
  StreamScratch own;
  float *ws = nullptr;
  if (p.ksplit > 1 && !(ws = own.take (s)))
    p.ksplit = 1;
  if (int e = launch_bf16_tiles (a, p, ws, s))
    return e;
  return launch_reduce_seg<false> (a, p.ksplit, ws, s);
}

namespace
{
// whether the 32-bit instructions would take longer than planes
bool
planes_pay (const GemmSegArgs &a)
{
  // Short rows of few values are over in the time of two more launches.  Measured, us,
  // 32-bit instructions / planes: K = 256, N = 2048, 300 rows 10 / 16, 4000 rows 48 / 36;
  // K = 512, N = 512, 1000 rows 15.5 / 20; K = 768, N = 128, 1 row 20 / 13; K = 2048,
  // N = 2048, 1 row 47 / 14, 2000 rows 162 / 60; K = 2048, N = 8064, 300 rows 121 / 48;
  // K = 5504, N = 2048, 300 rows 161 / 42; K = 4096, N = 11008, 2000 rows 1530 / 570.
  if (a.K <= 512 && (size_t)a.M * a.N * a.K <= (size_t)1 << 30)
    return false;
  // Where their 64 x 64 tiles just fill the compute units once, the 32-bit instructions need
  // 2.2 us + 23 ns per value of K for up to a million outputs; planes of many outputs, which take
  // several parts of the k range then, do not get below that while K is small (300 x 2048
  // outputs, K = 576 17.3 / 19.7, 77 x 8064 17.7 / 20.0, 400 x 2048, K = 640 18.7 / 22.7, 768 21.3 /
  // 23.4, 896 24.3 / 24.2, 256 x 4096, K = 768 21.4 / 25.2; fewer outputs, 130 x 2048, K = 640
  // 18.1 / 15.1).
  const size_t outputs = (size_t)a.M * a.N, tiles = (size_t)((a.M + 63) / 64) * ((a.N + 63) / 64);
  return !(tiles <= 256 && ((a.K <= 640 && outputs >= 600000) || (a.K <= 768 && outputs >= 800000)));
}

// nothing is allocated while the stream is captured
bool
capturing (hipStream_t s)
{
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing (s, &capture) != hipSuccess)
    {
      (void)hipGetLastError (); // (the default stream while another one is captured)
      return true;
    }
  return capture != hipStreamCaptureStatusNone;
}

// rows whose planes half of the scratch holds
size_t
plane_rows (int K)
{
  return StreamScratch::bytes () / 2 / ((size_t)kPlanes * K * sizeof (uint16_t));
}

// the rows that are multiplied at a time
int
portion_rows (const GemmSegArgs &a)
{
  const size_t most = plane_rows (a.K);
  return most >= (size_t)a.M ? a.M : (int)(most / WBM * WBM);
}

void
launch_split (const float *x, size_t xs, int M, int K, float *ws, hipStream_t s)
{
  const size_t total = (size_t)M * (K / 8);
  split_planes_kernel<<<dim3 ((unsigned)((total + 255) / 256)), dim3 (256), 0, s>>> (x, xs, M, K, (uint16_t *)ws);
}

// a with the planes of its x in ws
GemmSegArgs
with_planes (const GemmSegArgs &a, float *ws)
{
  GemmSegArgs b = a;
  b.x = (const uint16_t *)ws, b.K = kPlanes * a.K;
  return b;
}
} // namespace

bool
gemm_wide_f32_launch (const GemmSegArgs &a, hipStream_t s, int &err)
{
  if (!planes_pay (a) || capturing (s))
    return false;
  // the planes of as many rows as half of the scratch holds at a time, the parts of
  // a split k range behind them
  const size_t half = StreamScratch::bytes () / 2;
  const int rows = portion_rows (a);
  StreamScratch own;
  float *ws = rows > 0 ? own.take (s) : nullptr;
  if (!ws)
    return false;
  for (int m0 = 0; m0 < a.M; m0 += rows)
    {
      GemmSegArgs b = with_planes (a, ws);
      b.M = a.M - m0 < rows ? a.M - m0 : rows, b.xf = a.xf + (size_t)m0 * a.xs;
      launch_split (b.xf, a.xs, b.M, a.K, ws, s);
      for (int i = 0; i < a.nseg; ++i)
        {
          b.seg[i].y = (char *)a.seg[i].y + (size_t)m0 * a.seg[i].ys * (a.seg[i].f32 ? 4 : 2);
          if (a.seg[i].residual)
            b.seg[i].residual = a.seg[i].residual + (size_t)m0 * a.seg[i].ys;
        }
      if ((err = launch_planes (b, half, ws + half / sizeof (float), s)))
        return true;
    }
  return true;
}

// ---------------------------------------------------------------------------
// between two products: the sum into the residual rows and its norm
// ---------------------------------------------------------------------------
// A launch costs 4.5 to 5 us behind another one whatever it does, so one does what three did:
// it adds the parts of a product and the residual row (wide_reduce_seg_kernel), norms the row
// (rmsnorm_f32_kernel) and, in 32 bits, writes the planes that the next product reads
// (split_planes_kernel).  A workgroup has one row in registers; the sums and the norm are formed in
// the order of those kernels, bit for bit.  us before / now: 300 rows of 2048 in four parts 15.4 / 6.1,
// in bf16 (1500 rows, two parts) 15.0 / 11.2.
namespace
{
struct RowNorm
{
  const float *w;
  float eps;
  int Wp; // values of a row of h, zeros beyond N
  void *h;
  size_t hs;
  int f32;
  uint16_t *planes; // optional: rows of 3 Wp
};

// NV: float4 of a row per thread.  a: the product, one segment; parts 0: its sum stands in y.
template <int NV, bool PLANES>
__global__ __launch_bounds__ (256) void
sum_norm_kernel (const GemmSegArgs a, const float *ws, int parts, const RowNorm r)
{
  __shared__ float red[4];
  const int m = blockIdx.x, tid = threadIdx.x;
  float *y = (float *)a.seg[0].y + (size_t)m * a.seg[0].ys;
  const size_t at = (size_t)m * a.N, part = (size_t)a.M * a.N;
  float v[NV][4];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j)
    {
      // (N is a multiple of 4: a load is all inside or all padding)
      const int c = (tid + j * 256) * 4, cc = min (c, a.N - 4);
      const float4v res = __builtin_bit_cast (float4v, ldg4 (y + cc));
      if (parts > 0)
        {
          float t[4] = { 0.f, 0.f, 0.f, 0.f };
          for (int p0 = 0; p0 < parts; p0 += 4)
            {
              float4v x[4];
#pragma unroll
              for (int p = 0; p < 4; ++p)
                x[p] = __builtin_bit_cast (float4v, ldg4 (ws + (size_t)min (p0 + p, parts - 1) * part + at + cc));
#pragma unroll
              for (int p = 0; p < 4; ++p)
                if (p0 + p < parts)
#pragma unroll
                  for (int e = 0; e < 4; ++e)
                    t[e] += x[p][e];
            }
          if (PLANES)
            seg_f32_again<4> (a, t, m, cc, tid & 63, a.K / kPlanes);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            v[j][e] = t[e] + res[e];
          if (c < a.N)
            *(VKL_GLOBAL float4v *)(y + c) = float4v{ v[j][0], v[j][1], v[j][2], v[j][3] };
        }
      else
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[j][e] = res[e];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        {
          v[j][e] = c < a.N ? v[j][e] : 0.f;
          ss = __builtin_fmaf (v[j][e], v[j][e], ss);
        }
    }
  const float alpha = 1.0f / sqrtf (group_sum (ss, red) / (float)a.N + r.eps);
#pragma unroll
  for (int j = 0; j < NV; ++j)
    {
      const int c = (tid + j * 256) * 4;
      if (c >= r.Wp)
        continue;
      const float4v w = __builtin_bit_cast (float4v, ldg4 (r.w + min (c, a.N - 4)));
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        o[e] = v[j][e] * alpha * w[e];
      const size_t to = (size_t)m * r.hs + c;
      if (r.f32)
        *(VKL_GLOBAL float4v *)((float *)r.h + to) = float4v{ o[0], o[1], o[2], o[3] };
      else
        stg ((unsigned long long *)((uint16_t *)r.h + to),
             (unsigned long long)f2bf (o[0]) | ((unsigned long long)f2bf (o[1]) << 16)
                 | ((unsigned long long)f2bf (o[2]) << 32) | ((unsigned long long)f2bf (o[3]) << 48));
      if (r.planes)
        {
          uint32_t p[4][kPlanes];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            split_value (__float_as_uint (o[e]), p[e]);
          uint16_t *dst = r.planes + (size_t)m * kPlanes * r.Wp + (size_t)(c / WBK) * kPlanes * WBK + c % WBK;
#pragma unroll
          for (int q = 0; q < kPlanes; ++q)
            stg ((unsigned long long *)(dst + q * WBK),
                 (unsigned long long)(p[0][q] | (p[1][q] << 16)) | ((unsigned long long)(p[2][q] | (p[3][q] << 16)) << 32));
        }
    }
}

template <bool PLANES>
int
launch_sum_norm (const GemmSegArgs &a, const float *ws, int parts, const RowNorm &r, hipStream_t s)
{
  const dim3 grid ((unsigned)a.M), block (256);
  if (r.Wp <= 1024)
    sum_norm_kernel<1, PLANES><<<grid, block, 0, s>>> (a, ws, parts, r);
  else if (r.Wp <= 2048)
    sum_norm_kernel<2, PLANES><<<grid, block, 0, s>>> (a, ws, parts, r);
  else if (r.Wp <= 4096)
    sum_norm_kernel<4, PLANES><<<grid, block, 0, s>>> (a, ws, parts, r);
  else
    sum_norm_kernel<8, PLANES><<<grid, block, 0, s>>> (a, ws, parts, r);
  return (int)hipGetLastError ();
}

constexpr int kSumNormWidth = 8192;

// y += x W^T (add null: nothing is added), h = norm (y), the product of h; the arguments are
// checked.  False where no launch would be saved (nothing has been launched then).
bool
add_norm_project (const GemmSegArgs *add, const GemmSegArgs &rows, RowNorm r, const GemmSegArgs &next, hipStream_t s, int &err)
{
  const GemmSegArgs &y = add ? *add : rows;
  if (r.Wp > kSumNormWidth || (y.N % 8) != 0 || (y.seg[0].ys % 4) != 0 || (r.hs % 4) != 0 || ((uintptr_t)y.seg[0].y % 16) != 0
      || ((uintptr_t)r.w % 16) != 0 || ((uintptr_t)r.h % 16) != 0 || capturing (s))
    return false;
  StreamScratch own;
  if (!r.f32)
    {
      // only parts are added here: a sum without parts is formed by the tiles
      const WidePlan p = add ? wide_plan_bf16 (*add, StreamScratch::bytes ()) : WidePlan{ 0, 1 };
      float *ws = p.ksplit > 1 ? own.take (s) : nullptr;
      if (!ws)
        return false;
      if ((err = launch_bf16_tiles (*add, p, ws, s)))
        return true;
      err = launch_sum_norm<false> (*add, ws, p.ksplit, r, s);
      own.give ();
      if (!err)
        err = gemm_wide_bf16_launch (next, s);
      return true;
    }
  // planes of all rows at once, of both products or the next one
  const bool first = add && planes_pay (*add) && plane_rows (add->K) >= (size_t)add->M;
  if ((add && !first) || !planes_pay (next) || plane_rows (next.K) < (size_t)next.M)
    return false;
  float *ws = own.take (s);
  if (!ws)
    return false;
  const size_t half = StreamScratch::bytes () / 2;
  float *parts = ws + half / sizeof (float);
  r.planes = (uint16_t *)ws; // (those of the first product have been read by then)
  int n = 0;
  if (add)
    {
      launch_split (add->xf, add->xs, add->M, add->K, ws, s);
      const GemmSegArgs b = with_planes (*add, ws);
      const WidePlan p = wide_plan_planes (b, half);
      if ((err = launch_planes_tiles (b, p, parts, s)))
        return true;
      n = p.ksplit > 1 ? p.ksplit : 0;
      err = launch_sum_norm<true> (b, parts, n, r, s);
    }
  else
    err = launch_sum_norm<false> (rows, nullptr, 0, r, s);
  if (!err)
    err = launch_planes (with_planes (next, ws), half, parts, s);
  return true;
}

// the arguments of a product, checked
int
seg_args (const void *x, int xtype, size_t xs, const void *w, int M, int N, int K, const vkl_out_seg *segs, int nseg,
          GemmSegArgs &a)
{
  VKL_CHECK_ARG (x && w && segs && M > 0 && N > 0 && K > 0 && (K % 64) == 0 && xs >= (size_t)K);
  VKL_CHECK_ARG (nseg > 0 && nseg <= kGemmSegs && (xtype == VKL_TYPE_F32 || xtype == VKL_TYPE_BF16));
  VKL_CHECK_ARG ((xs % 8) == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0);
  a = {};
  if (xtype == VKL_TYPE_F32)
    a.xf = (const float *)x;
  else
    a.x = (const uint16_t *)x;
  a.xs = xs, a.M = M, a.N = N, a.K = K, a.Kp = K, a.wtype = 1, a.batch = 1, a.nmat = 1, a.scale = 1.f;
  a.wh[0] = a.wh[1] = a.wh[2] = (const uint16_t *)w;
  a.ws = (size_t)K;
  a.nseg = nseg;
  int end = 0;
  for (int i = 0; i < nseg; ++i)
    {
      const vkl_out_seg &o = segs[i];
      VKL_CHECK_ARG (o.y && o.n > 0 && o.n0 >= end && (o.n0 % 8) == 0 && o.n0 + o.n <= N && o.ys >= (size_t)o.n);
      VKL_CHECK_ARG (i > 0 || o.n0 == 0);
      VKL_CHECK_ARG (o.act >= VKL_ACT_NONE && o.act <= VKL_ACT_GELU);
      VKL_CHECK_ARG (o.type == VKL_TYPE_F32 || (o.type == VKL_TYPE_BF16 && !o.residual));
      GemmSeg &g = a.seg[i];
      g.n0 = o.n0, g.n = o.n, g.y = o.y, g.ys = o.ys, g.f32 = o.type == VKL_TYPE_F32;
      g.act = o.act, g.residual = o.residual, g.cap = o.cap;
      g.vec = (o.ys % 8) == 0 && ((uintptr_t)o.y % 16) == 0 && (!o.residual || ((uintptr_t)o.residual % 16) == 0);
      end = o.n0 + o.n;
    }
  return 0;
}

int
project (const GemmSegArgs &a, hipStream_t s)
{
  return a.xf ? gemm_f32_launch (a, s) : gemm_wide_bf16_launch (a, s);
}
} // namespace
} // namespace vkl

extern "C" int
vkl_project_bf16w (const void *x, int xtype, size_t xs, const void *w, int M, int N, int K,
                   const vkl_out_seg *segs, int nseg, void *stream)
{
  vkl::GemmSegArgs a;
  if (int e = vkl::seg_args (x, xtype, xs, w, M, N, K, segs, nseg, a))
    return e;
  return vkl::project (a, (hipStream_t)stream);
}

extern "C" int
vkl_project_plan (int xtype, int M, int N, int K, int otype, int act, vkl_project_plan_t *out)
{
  using namespace vkl;
  VKL_CHECK_ARG (out);
  // (addresses that fit, which nothing follows)
  void *any = (void *)(uintptr_t)16;
  const vkl_out_seg seg = { 0, N, any, (size_t)(N > 0 ? N : 0), otype, act, nullptr, 0.f };
  GemmSegArgs a;
  if (int e = seg_args (any, xtype, (size_t)(K > 0 ? K : 0), any, M, N, K, &seg, 1, a))
    return e;
  const bool f32 = xtype == VKL_TYPE_F32;
  *out = { 0, 1, 0, 0, 1 };
  WidePlan p;
  if (f32)
    {
      a.M = portion_rows (a);
      if (!planes_pay (a) || a.M <= 0)
        return 0;
      p = wide_plan_planes (with_planes (a, nullptr), StreamScratch::bytes () / 2);
      out->planes = kPlanes;
    }
  else
    p = wide_plan_bf16 (a, StreamScratch::bytes ());
  out->tile_rows = p.bm, out->ksplit = p.ksplit;
  out->four_waves = f32 || p.bm == 64 || p.four_waves;
  if (!out->four_waves)
    out->pairs = mix_tiles (a, p.bm, p.ksplit).wide;
  return 0;
}

extern "C" int
vkl_add_norm_project_bf16w (const vkl_add_norm_project *p, int type, int M, void *stream)
{
  VKL_CHECK_ARG (p && p->y && p->norm && p->h && p->W > 0 && p->Wp >= p->W && p->ys >= (size_t)p->W && p->hs >= (size_t)p->Wp);
  const vkl_out_seg back = { 0, p->W, p->y, p->ys, VKL_TYPE_F32, VKL_ACT_NONE, p->y, 0.f };
  vkl::GemmSegArgs add = {}, rows = {}, next;
  if (p->x)
    if (int e = vkl::seg_args (p->x, type, p->xs, p->w, M, p->W, p->K, &back, 1, add))
      return e;
  if (int e = vkl::seg_args (p->h, type, p->hs, p->w_next, M, p->N, p->Wp, p->segs, p->nseg, next))
    return e;
  rows.M = M, rows.N = p->W, rows.seg[0].y = p->y, rows.seg[0].ys = p->ys;
  const vkl::RowNorm r = { p->norm, p->eps, p->Wp, p->h, p->hs, type == VKL_TYPE_F32, nullptr };
  hipStream_t s = (hipStream_t)stream;
  int err = 0;
  if (vkl::add_norm_project (p->x ? &add : nullptr, rows, r, next, s, err))
    return err;
  if (p->x)
    if (int e = vkl::project (add, s))
      return e;
  if (int e = vkl_rmsnorm_f32 (p->y, p->ys, nullptr, M, p->W, p->norm, p->eps, p->h, type, p->hs, p->Wp, stream))
    return e;
  return vkl::project (next, s);
}

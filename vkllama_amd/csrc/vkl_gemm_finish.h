// Shared epilogue of the prompt GEMM kernels that walk their results row-wise,
// eight neighbouring output columns per lane.
#ifndef VKL_GEMM_FINISH_H
#define VKL_GEMM_FINISH_H
#include "vkl_act.h"
#include "vkl_common.h"
#include "vkl_gemm.h"

namespace vkl
{
// One of three pointers.  (Opaque values: a select of values that come from memory may
// become a load from a selected address, and an index that varies puts the kernel's whole
// argument block in scratch.)
template <class T>
__device__ __forceinline__ T *
pick3 (T *p0, T *p1, T *p2, int i)
{
  asm ("" : "+s"(p0), "+s"(p1), "+s"(p2));
  return i == 0 ? p0 : (i == 1 ? p1 : p2);
}

// Eight neighbouring outputs of row m from column ncol0 on: v the fp32 sums (for
// the fused pair: up; g: gate), then scale, bias, activation, rounding,
// residual, the stores.
// pre: the residual's eight values, requested ahead (see FinishRows)
template <bool UPGATE>
__device__ __forceinline__ void
gemm_finish8 (const GemmArgs &a, float (&v)[8], const float (&g)[8], int m, int ncol0, int zmat, int vec,
              float *part, const uint4 *pre = nullptr)
{
  if (!UPGATE && part)
    {
      // one part of a split k range: the raw sums, dense [M, N] fp32; the
      // reduction kernel adds the parts in order and applies the rest
      if (m >= a.M || ncol0 >= a.N)
        return;
      float *dst = part + (size_t)m * a.N + ncol0;
      if ((a.N % 4) == 0 && ncol0 + 8 <= a.N)
        {
          typedef float f32x4 __attribute__ ((ext_vector_type (4)));
          f32x4 w0 = { v[0], v[1], v[2], v[3] }, w1 = { v[4], v[5], v[6], v[7] };
          *(VKL_GLOBAL f32x4 *)dst = w0;
          *(VKL_GLOBAL f32x4 *)(dst + 4) = w1;
        }
      else
        for (int e = 0; e < 8 && ncol0 + e < a.N; ++e)
          dst[e] = v[e];
      return;
    }
  uint16_t *y = UPGATE ? a.y[0] : pick3 (a.y[0], a.y[1], a.y[2], zmat);
  const bool plain = a.nmat != 1; // one of three fused outputs: no scale, activation, residual
  if (UPGATE)
    {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        v[e] = silu (g[e]) * v[e];
    }
  else if (!plain)
    {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        v[e] = v[e] * a.scale + a.bias;
      if (a.act == 1)
        {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            v[e] = silu (v[e]);
        }
    }
  if (m >= a.M || ncol0 >= a.N)
    return;
  uint16_t h[8];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    h[e] = f2h (v[e]);
  const size_t o = (size_t)m * a.ys + ncol0;
  const bool res = !UPGATE && !plain && a.residual;
  float *y32 = !UPGATE && !plain && a.y32 ? a.y32 + (size_t)m * a.N + ncol0 : nullptr;
  if (vec && ncol0 + 8 <= a.N)
    {
      if (res)
        {
          const uint4 rv = pre ? *pre : ldg4 (a.residual + o);
          const uint32_t rw[4] = { rv.x, rv.y, rv.z, rv.w };
#pragma unroll
          for (int e = 0; e < 8; ++e)
            h[e] = f2h (h2f (h[e]) + h2f ((uint16_t)(rw[e >> 1] >> ((e & 1) * 16))));
        }
      vkl_u32x4 pk;
      pk.x = h[0] | ((uint32_t)h[1] << 16), pk.y = h[2] | ((uint32_t)h[3] << 16);
      pk.z = h[4] | ((uint32_t)h[5] << 16), pk.w = h[6] | ((uint32_t)h[7] << 16);
      *(VKL_GLOBAL vkl_u32x4 *)(y + o) = pk;
      if (y32)
        {
          typedef float f32x4 __attribute__ ((ext_vector_type (4)));
          f32x4 w0 = { h2f (h[0]), h2f (h[1]), h2f (h[2]), h2f (h[3]) };
          f32x4 w1 = { h2f (h[4]), h2f (h[5]), h2f (h[6]), h2f (h[7]) };
          *(VKL_GLOBAL f32x4 *)y32 = w0;
          *(VKL_GLOBAL f32x4 *)(y32 + 4) = w1;
        }
      return;
    }
  // ragged end of a row, or operands that are not 16-byte aligned
  for (int e = 0; e < 8 && ncol0 + e < a.N; ++e)
    {
      uint16_t he = h[e];
      if (res)
        he = f2h (h2f (he) + h2f (ldg (a.residual + o + e)));
      y[o + e] = he;
      if (y32)
        y32[e] = h2f (he);
    }
}
// Where a product with segments puts the eight columns from ncol0 (a multiple of 8) on:
// segments start at multiples of 8, so all eight belong to one.  A kernel that walks
// the rows of one column group looks this up once.
struct SegCol
{
  char *y;        // the group's first value of row 0
  const float *r; // residual, likewise
  size_t ys;
  float cap;
  int f32, act, n; // n: columns that are written
  bool whole;      // all eight, with vector accesses
};

__device__ __forceinline__ SegCol
seg_col (const GemmSegArgs &a, int ncol0)
{
  SegCol c = {};
#pragma unroll
  for (int i = 0; i < kGemmSegs; ++i)
    if (i < a.nseg && ncol0 >= a.seg[i].n0)
      {
        const GemmSeg &sg = a.seg[i];
        const int at = ncol0 - sg.n0;
        c.y = (char *)sg.y + (size_t)at * (sg.f32 ? 4 : 2);
        c.r = sg.residual ? sg.residual + at : nullptr;
        c.ys = sg.ys, c.cap = sg.cap, c.f32 = sg.f32, c.act = sg.act;
        c.n = sg.n - at, c.whole = sg.vec && at + 8 <= sg.n;
      }
  return c;
}

// v the sums of row m; pre: the residual's eight values, requested ahead
__device__ __forceinline__ void
seg_finish8 (const SegCol &c, float (&v)[8], int m, const uint4 *pre)
{
  typedef float f32x4 __attribute__ ((ext_vector_type (4)));
  if (c.act != VKL_ACT_NONE)
    activate8 (c.act, v);
  if (c.cap > 0.f)
#pragma unroll
    for (int e = 0; e < 8; ++e)
      v[e] = c.cap * tanhf (v[e] / c.cap);
  if (c.f32)
    {
      float *y = (float *)c.y + (size_t)m * c.ys;
      const float *r = c.r ? c.r + (size_t)m * c.ys : nullptr;
      if (c.whole)
        {
          f32x4 w0 = { v[0], v[1], v[2], v[3] }, w1 = { v[4], v[5], v[6], v[7] };
          if (r)
            {
              w0 += pre ? __builtin_bit_cast (f32x4, pre[0]) : *(const VKL_GLOBAL f32x4 *)r;
              w1 += pre ? __builtin_bit_cast (f32x4, pre[1]) : *(const VKL_GLOBAL f32x4 *)(r + 4);
            }
          *(VKL_GLOBAL f32x4 *)y = w0;
          *(VKL_GLOBAL f32x4 *)(y + 4) = w1;
        }
      else
        for (int e = 0; e < 8 && e < c.n; ++e)
          y[e] = r ? r[e] + v[e] : v[e];
    }
  else
    {
      uint16_t *y = (uint16_t *)c.y + (size_t)m * c.ys;
      uint16_t h[8];
#pragma unroll
      for (int e = 0; e < 8; ++e)
        h[e] = f2bf (v[e]);
      if (c.whole)
        {
          vkl_u32x4 pk;
          pk.x = h[0] | ((uint32_t)h[1] << 16), pk.y = h[2] | ((uint32_t)h[3] << 16);
          pk.z = h[4] | ((uint32_t)h[5] << 16), pk.w = h[6] | ((uint32_t)h[7] << 16);
          *(VKL_GLOBAL vkl_u32x4 *)y = pk;
        }
      else
        for (int e = 0; e < 8 && e < c.n; ++e)
          y[e] = h[e];
    }
}

template <bool UPGATE>
__device__ __forceinline__ void
gemm_finish8 (const GemmSegArgs &a, float (&v)[8], const float (&)[8], int m, int ncol0, int, int, float *part)
{
  typedef float f32x4 __attribute__ ((ext_vector_type (4)));
  if (m >= a.M || ncol0 >= a.N)
    return;
  if (part)
    {
      // (N is a multiple of 8 here or the tail is written one by one)
      float *dst = part + (size_t)m * a.N + ncol0;
      if ((a.N % 8) == 0)
        {
          f32x4 w0 = { v[0], v[1], v[2], v[3] }, w1 = { v[4], v[5], v[6], v[7] };
          *(VKL_GLOBAL f32x4 *)dst = w0;
          *(VKL_GLOBAL f32x4 *)(dst + 4) = w1;
        }
      else
        for (int e = 0; e < 8 && ncol0 + e < a.N; ++e)
          dst[e] = v[e];
      return;
    }
  seg_finish8 (seg_col (a, ncol0), v, m, nullptr);
}

// The epilogue of rows that a lane walks in one column group: what does not depend on
// the row is looked up once, and the residual of the next rows is requested before
// the rows are finished (a residual may lie in the output's own rows, so the compiler
// cannot move a request above a store).
template <bool UPGATE, class Args> struct FinishRows;

template <bool UPGATE> struct FinishRows<UPGATE, GemmArgs>
{
  const GemmArgs &a;
  int ncol0, zmat, vec;
  float *part;
  bool ahead;

  __device__ __forceinline__
  FinishRows (const GemmArgs &args, int n, int z, int v, float *p)
      : a (args), ncol0 (n), zmat (z), vec (v), part (p),
        ahead (!UPGATE && !p && v && args.nmat == 1 && args.residual && n + 8 <= args.N)
  {
  }
  __device__ __forceinline__ void
  request (int m, uint4 (&r)[2]) const
  {
    if (ahead)
      r[0] = ldg4 (a.residual + (size_t)min (m, a.M - 1) * a.ys + ncol0);
  }
  __device__ __forceinline__ void
  store (int m, float (&v)[8], const float (&g)[8], const uint4 (&r)[2]) const
  {
    gemm_finish8<UPGATE> (a, v, g, m, ncol0, zmat, vec, part, ahead ? r : nullptr);
  }
};

template <bool UPGATE> struct FinishRows<UPGATE, GemmSegArgs>
{
  const GemmSegArgs &a;
  int ncol0;
  float *part;
  SegCol c;
  bool ahead;

  __device__ __forceinline__
  FinishRows (const GemmSegArgs &args, int n, int, int, float *p)
      : a (args), ncol0 (n), part (p), c (seg_col (args, n)), ahead (!p && n < args.N && c.whole && c.r && c.f32)
  {
  }
  __device__ __forceinline__ void
  request (int m, uint4 (&r)[2]) const
  {
    if (ahead)
      {
        const float *src = c.r + (size_t)min (m, a.M - 1) * c.ys;
        r[0] = ldg4 (src), r[1] = ldg4 (src + 4);
      }
  }
  __device__ __forceinline__ void
  store (int m, float (&v)[8], const float (&g)[8], const uint4 (&r)[2]) const
  {
    if (part)
      gemm_finish8<UPGATE> (a, v, g, m, ncol0, 0, 0, part);
    else if (m < a.M && ncol0 < a.N)
      seg_finish8 (c, v, m, ahead ? r : nullptr);
  }
};
} // namespace vkl
#endif

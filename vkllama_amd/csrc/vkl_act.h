// Activations of the products of decoder stacks.
#ifndef VKL_ACT_H
#define VKL_ACT_H
#include "../../include/vkl_stack.h"
#include "vkl_common.h"

namespace vkl
{
// x Phi (x), Phi the normal distribution: 1 - h for x >= 0 and h below, h = erfc (|x| / sqrt 2) / 2 as e^(-x^2/2) t P (t), t = 1 /
// (1 + 0.43 |x| / sqrt 2).  P is the polynomial whose largest relative error over |x| < 17 is least (2.1e-7; Chebyshev
// fit of e^(z^2) erfc (z) / t).  Against 64 bits over |x| < 9: absolute error 3.8e-7, relative 7e-7 above -3 and 2.1e-6 above -6; with
// 1 + erff (x / sqrt 2), which cancels below zero, 4.5e-7, 1.1e-5 and 1.  Two dozen instructions in place of erff's two
// branches, of which a wave takes both: us of a product with GELU, erff / this: 2048 x
// 5504 x 2048 60.0 / 55.3, 600 rows 23.3 / 21.9, 2048 x 11008 x 4096 178.5 / 173.
__device__ __forceinline__ float
gelu (float x)
{
  const float z = fabsf (x) * 0.70710678118654752440f;
  const float t = __builtin_amdgcn_rcpf (__builtin_fmaf (z, 0.43f, 1.0f));
  float p = 0.07187054459355813f;
  p = __builtin_fmaf (p, t, -0.30266294766022617f);
  p = __builtin_fmaf (p, t, 0.37034016398068037f);
  p = __builtin_fmaf (p, t, -0.07337288084714394f);
  p = __builtin_fmaf (p, t, 0.2403002471567231f);
  p = __builtin_fmaf (p, t, 0.2069291065001833f);
  p = __builtin_fmaf (p, t, 0.24406096646819633f);
  p = __builtin_fmaf (p, t, 0.24253482856151803f);
  const float h = 0.5f * (p * t) * __builtin_amdgcn_exp2f (x * x * -0.72134752044448170368f);
  return x * (x >= 0.f ? 1.0f - h : h);
}

// what a product stores for a sum (VKL_ACT_...)
__device__ __forceinline__ float
activate (int act, float v)
{
  if (act == VKL_ACT_SILU)
    return silu (v);
  if (act == VKL_ACT_RELU2)
    {
      v = fmaxf (v, 0.f);
      return v * v;
    }
  if (act == VKL_ACT_GELU)
    return gelu (v);
  return v;
}

// the same for eight, with one look at `act`
__device__ __forceinline__ void
activate8 (int act, float (&v)[8])
{
  if (act == VKL_ACT_SILU)
    {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        v[e] = activate (VKL_ACT_SILU, v[e]);
    }
  else if (act == VKL_ACT_RELU2)
    {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        v[e] = activate (VKL_ACT_RELU2, v[e]);
    }
  else if (act == VKL_ACT_GELU)
    {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        v[e] = activate (VKL_ACT_GELU, v[e]);
    }
}
} // namespace vkl
#endif

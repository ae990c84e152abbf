// Activations of the products of decoder stacks.
#ifndef VKL_ACT_H
#define VKL_ACT_H
#include "../../include/vkl_stack.h"
#include "vkl_common.h"

namespace vkl
{
// what a product stores for a sum (VKL_ACT_...)
// GELU with erff, of whose two branches a wave takes both (us of a product with GELU, 2048 x 5504 x 2048: 60.0).  A polynomial for
// the normal distribution's tail took 55.3, but twice to five times erff's error against 64 bits between -1.5 and 1 (relative, around
// zero 4.5e-7 / 1.2e-7).
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
    return 0.5f * v * (1.0f + erff (v * 0.70710678118654752440f));
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

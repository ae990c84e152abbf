// Q8_0: host quantiser, GGUF-block <-> planar repack, embedding gather.
#include "../../include/vkl_hip.h"
#include "vkl_common.h"
#include <math.h>
#include <string.h>

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static inline uint16_t
host_f32_to_f16_rne (float f)
{
  return __builtin_bit_cast (uint16_t, (_Float16)f);
}

static inline float
host_f16_to_f32 (uint16_t h)
{
  return (float)__builtin_bit_cast (_Float16, h);
}

extern "C" size_t
vkl_q8_0_row_bytes (size_t K)
{
  return (K + 31) / 32 * 34;
}

// Follows src/core/quants.h:35-96: amax over the block, scale = amax/127,
// inverse = 127/amax (0 when the block is all zero), q = roundf(x*inverse),
// tail padded with zeros.  The scale is stored as fp16 (RNE) in front of the
// 32 quants, the block the reference's shaders read.
extern "C" void
vkl_quantize_q8_0_h (const float *src, size_t n, uint8_t *dst)
{
  const size_t nb = (n + 31) / 32;
  for (size_t b = 0; b < nb; ++b)
    {
      const size_t start = b * 32;
      const size_t end = start + 32 < n ? start + 32 : n;
      float amax = fabsf (src[start]);
      for (size_t i = start; i < end; ++i)
        amax = fmaxf (amax, fabsf (src[i]));
      const float scale = amax / 127.0f;
      const float inv = scale > 0 ? 127.0f / amax : 0.0f;
      const uint16_t h = host_f32_to_f16_rne (scale);
      memcpy (dst, &h, 2);
      int8_t *q = (int8_t *)(dst + 2);
      for (size_t i = 0; i < 32; ++i)
        q[i] = start + i < n ? (int8_t)roundf (src[start + i] * inv) : 0;
      dst += 34;
    }
}

extern "C" void
vkl_dequantize_q8_0_h (const uint8_t *src, size_t n, float *dst)
{
  const size_t nb = (n + 31) / 32;
  for (size_t b = 0; b < nb; ++b)
    {
      uint16_t h;
      memcpy (&h, src + b * 34, 2);
      const float d = host_f16_to_f32 (h);
      const int8_t *q = (const int8_t *)(src + b * 34 + 2);
      for (size_t i = 0; i < 32 && b * 32 + i < n; ++i)
        dst[b * 32 + i] = (float)q[i] * d;
    }
}

// ---------------------------------------------------------------------------
// repack
// ---------------------------------------------------------------------------
// One thread per block.  Raw blocks are only 2-byte aligned, so they are read
// and written as 17 ushorts; the planar side is 32-byte aligned.
__global__ void
q8_pack_kernel (const uint16_t *__restrict__ raw, uint32_t *__restrict__ q,
                uint16_t *__restrict__ d, size_t nblocks)
{
  const size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nblocks)
    return;
  const uint16_t *src = raw + b * 17;
  d[b] = src[0];
  uint32_t *dst = q + b * 8;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    dst[i] = (uint32_t)src[1 + 2 * i] | ((uint32_t)src[2 + 2 * i] << 16);
}

__global__ void
q8_unpack_kernel (const uint32_t *__restrict__ q,
                  const uint16_t *__restrict__ d, uint16_t *__restrict__ raw,
                  size_t nblocks)
{
  const size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nblocks)
    return;
  uint16_t *dst = raw + b * 17;
  dst[0] = d[b];
  const uint32_t *src = q + b * 8;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    {
      const uint32_t w = src[i];
      dst[1 + 2 * i] = (uint16_t)(w & 0xffffu);
      dst[2 + 2 * i] = (uint16_t)(w >> 16);
    }
}

extern "C" int
vkl_q8_0_pack (const void *raw, void *planar, size_t rows, size_t K,
               void *stream)
{
  VKL_CHECK_ARG (raw && planar);
  const size_t nb = (K + 31) / 32, nblocks = rows * nb;
  if (nblocks == 0)
    return 0;
  VKL_CHECK_ARG ((nblocks + 255) / 256 <= 0x7fffffffu);
  uint8_t *p = (uint8_t *)planar;
  q8_pack_kernel<<<dim3 ((unsigned)((nblocks + 255) / 256)), dim3 (256), 0,
                   (hipStream_t)stream>>> (
      (const uint16_t *)raw, (uint32_t *)p, (uint16_t *)(p + nblocks * 32),
      nblocks);
  return vkl_launch_status ();
}

extern "C" int
vkl_q8_0_unpack (const void *planar, void *raw, size_t rows, size_t K,
                 void *stream)
{
  VKL_CHECK_ARG (raw && planar);
  const size_t nb = (K + 31) / 32, nblocks = rows * nb;
  if (nblocks == 0)
    return 0;
  VKL_CHECK_ARG ((nblocks + 255) / 256 <= 0x7fffffffu);
  const uint8_t *p = (const uint8_t *)planar;
  q8_unpack_kernel<<<dim3 ((unsigned)((nblocks + 255) / 256)), dim3 (256), 0,
                     (hipStream_t)stream>>> (
      (const uint32_t *)p, (const uint16_t *)(p + nblocks * 32),
      (uint16_t *)raw, nblocks);
  return vkl_launch_status ();
}

// ---------------------------------------------------------------------------
// embedding
// ---------------------------------------------------------------------------
// One thread per eight neighbouring values of a token's row, 16-byte stores: out =
// fp16(float(q) * float(d)).  HBM-bound: with a thread per block of 32 and 2-byte stores
// 3967 rows of 5120 values (62 MB) took 159 us, with one per fp16 value 2048 rows of 4096
// took 38; their prompts 13630 -> 13445 and 2307 -> 2277 us.  VEC: rows are multiples of eight values, 16-byte aligned.
__device__ __forceinline__ uint32_t
known_token (const uint32_t *toks, uint32_t t, uint32_t VH, uint32_t unk)
{
  const uint32_t tok = toks[t];
  return tok >= VH ? unk : tok;
}

template <bool VEC>
__global__ __launch_bounds__ (256) void
embed_q8_kernel (const uint8_t *__restrict__ q, const uint16_t *__restrict__ d,
                 uint32_t VH, uint32_t VW, uint32_t nb,
                 const uint32_t *__restrict__ toks, uint32_t unk,
                 uint16_t *__restrict__ out)
{
  const uint32_t c = (blockIdx.x * 256 + threadIdx.x) * 8, t = blockIdx.y;
  if (c >= VW)
    return;
  const size_t row = (size_t)known_token (toks, t, VH, unk) * nb;
  const float scale = vkl::h2f (d[row + (c >> 5)]);
  const uint2 w2 = *(const uint2 *)(q + row * 32 + c);
  const uint32_t w[2] = { w2.x, w2.y };
  uint16_t h[8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    h[i] = vkl::f2h ((float)(int8_t)(w[i >> 2] >> (8 * (i & 3))) * scale);
  uint16_t *o = out + (size_t)t * VW + c;
  if (VEC)
    *(uint4 *)o = make_uint4 (h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16), h[4] | ((uint32_t)h[5] << 16),
                              h[6] | ((uint32_t)h[7] << 16));
  else
    for (uint32_t i = 0; i < 8 && c + i < VW; ++i)
      o[i] = h[i];
}

template <bool VEC>
__global__ __launch_bounds__ (256) void
embed_f16_kernel (const uint16_t *__restrict__ table, uint32_t VH, uint32_t VW,
                  const uint32_t *__restrict__ toks, uint32_t unk,
                  uint16_t *__restrict__ out)
{
  const uint32_t c = (blockIdx.x * 256 + threadIdx.x) * 8, t = blockIdx.y;
  if (c >= VW)
    return;
  const uint16_t *src = table + (size_t)known_token (toks, t, VH, unk) * VW + c;
  uint16_t *o = out + (size_t)t * VW + c;
  if (VEC)
    *(uint4 *)o = *(const uint4 *)src;
  else
    for (uint32_t i = 0; i < 8 && c + i < VW; ++i)
      o[i] = src[i];
}

extern "C" int
vkl_embed_q8_0 (const void *table_planar, uint32_t VH, uint32_t VW,
                const uint32_t *toks, uint32_t n, uint32_t unk, void *out,
                void *stream)
{
  VKL_CHECK_ARG (table_planar && toks && out && VH > 0 && VW > 0);
  VKL_CHECK_ARG (unk < VH && n <= 65535);
  if (n == 0)
    return 0;
  const uint32_t nb = (VW + 31) / 32;
  const uint8_t *p = (const uint8_t *)table_planar;
  const dim3 grid ((VW + 2047) / 2048, n);
  const auto kernel = (VW % 8) == 0 && ((uintptr_t)out % 16) == 0 ? embed_q8_kernel<true> : embed_q8_kernel<false>;
  kernel<<<grid, dim3 (256), 0, (hipStream_t)stream>>> (p, (const uint16_t *)(p + (size_t)VH * nb * 32), VH, VW, nb, toks,
                                                        unk, (uint16_t *)out);
  return vkl_launch_status ();
}

extern "C" int
vkl_embed_f16 (const void *table, uint32_t VH, uint32_t VW,
               const uint32_t *toks, uint32_t n, uint32_t unk, void *out,
               void *stream)
{
  VKL_CHECK_ARG (table && toks && out && VH > 0 && VW > 0);
  VKL_CHECK_ARG (unk < VH && n <= 65535);
  if (n == 0)
    return 0;
  const dim3 grid ((VW + 2047) / 2048, n);
  const auto kernel = (VW % 8) == 0 && (((uintptr_t)out | (uintptr_t)table) % 16) == 0 ? embed_f16_kernel<true> : embed_f16_kernel<false>;
  kernel<<<grid, dim3 (256), 0, (hipStream_t)stream>>> ((const uint16_t *)table, VH, VW, toks, unk, (uint16_t *)out);
  return vkl_launch_status ();
}

// mlp_net.hpp -- device code shared by the fused predictor kernels
// (mlp.hip, mlp_features.hip, mlp_infer.hip): bf16 conversion and the hidden
// layers' activation.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace hps
{
  typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
  typedef float  f32x16 __attribute__((ext_vector_type(16)));
  typedef float  f32x4 __attribute__((ext_vector_type(4)));

  __device__ __forceinline__ uint16_t f2bf(float f)
  {
    // round to nearest even
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
  }
  __device__ __forceinline__ float bf2f(uint16_t b)
  {
    return __uint_as_float(((uint32_t)b) << 16);
  }

  // tanh for the hidden layers (the result is rounded to bf16, relative
  // spacing 2^-8): 1 - 2 / (exp(2 x) + 1) with the hardware exponential and
  // reciprocal, whose absolute error of about 2e-7 is a relative error below
  // 5e-6 for |x| >= 2^-4, and x - x^3 / 3 below that (2 x^4 / 15 < 2.1e-6).
  // Both sides are formed without a branch: a wave meets both.
  __device__ __forceinline__ float tanh_fast(float x)
  {
    const float small = x * (1.0f - 0.333333333f * (x * x));
    const float e     = __builtin_amdgcn_exp2f(2.885390082f * x); // 2 log2(e) x
    const float large = 1.0f - 2.0f * __builtin_amdgcn_rcpf(e + 1.0f);
    return fabsf(x) < 0.0625f ? small : large;
  }

  // widths of the built network: 272 stencil features -> 3 x 128 -> 4
  constexpr int NET_IN = 272, NET_H = 128, NET_OUT = 4;
} // namespace hps

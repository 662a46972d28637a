// BF16 matrix-core types and rounding of the scorer inside the search (v_mfma_f32_32x32x8_bf16).
#pragma once
#include "velo_common.cuh"

namespace velo {
namespace mlp {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ uint16_t to_bf16(float f)
{
  const uint32_t b = __float_as_uint(f);
  return static_cast<uint16_t>((b + 0x7FFFu + ((b >> 16) & 1u)) >> 16);
}
__device__ __forceinline__ float from_bf16(uint16_t h) { return __uint_as_float(static_cast<uint32_t>(h) << 16); }

__device__ __forceinline__ f32x16 zero16()
{
  f32x16 z;
#pragma unroll
  for (unsigned v = 0; v < 16; ++v) z[v] = 0.f;
  return z;
}

} // namespace mlp
} // namespace velo

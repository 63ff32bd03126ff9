// zh_field.h -- the cell hash of fractal_noise.frag, shared by the noise kernel
// (zh_field.hip) and the interpreter (zh_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace zh {

// pcg4d (Jarzynski and Olano, "Hash Functions for GPU Rendering", JCGT 9(3),
// 2020): an LCG step per lane, then two rounds of cross-lane multiply-adds
// around a 16-bit xorshift; wrapping 32-bit arithmetic.
__device__ __forceinline__ uint4 pcg4d(uint4 v) {
  v.x = v.x * 1664525u + 1013904223u;
  v.y = v.y * 1664525u + 1013904223u;
  v.z = v.z * 1664525u + 1013904223u;
  v.w = v.w * 1664525u + 1013904223u;
  v.x += v.y * v.w; v.y += v.z * v.x; v.z += v.x * v.y; v.w += v.y * v.z;
  v.x ^= v.x >> 16; v.y ^= v.y >> 16; v.z ^= v.z >> 16; v.w ^= v.w >> 16;
  v.x += v.y * v.w; v.y += v.z * v.x; v.z += v.x * v.y; v.w += v.y * v.z;
  return v;
}

// The corner value of a cell: pcg4d of (cell, 0, 0) over 2^32 - 1 (as f32,
// that is 2^32), each lane a channel.
__device__ __forceinline__ float4 cell_value(uint32_t sx, uint32_t sy) {
  const uint4 h = pcg4d(make_uint4(sx, sy, 0u, 0u));
  const float k = 4294967295.0f;
  return make_float4((float)h.x / k, (float)h.y / k, (float)h.z / k, (float)h.w / k);
}

// f32 floor as the shader's ivec2(floor(.)) cell index, saturated to int32.
__device__ __forceinline__ uint32_t cell_index(float f) {
  return (uint32_t)(int32_t)fminf(fmaxf(f, -2147483648.0f), 2147483520.0f);
}

}  // namespace zh

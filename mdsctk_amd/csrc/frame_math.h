// Small FP64 device helpers shared by the kernel sources: wave sums and the
// eigenvectors of the 3x3 and 4x4 symmetric matrices of a frame.
#pragma once

#include <hip/hip_runtime.h>

namespace mdsctk {

// One atom's coordinates: a single 12-byte load per lane.
struct F3 {
  float x, y, z;
};

__device__ __forceinline__ double wave_sum_d(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

__device__ __forceinline__ unsigned short bf16_rne(float v) {
  unsigned u = __float_as_uint(v);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ double bf16_val(unsigned short h) {
  return (double)__uint_as_float(((unsigned)h) << 16);
}

}  // namespace mdsctk

// blkval.hpp -- device helpers of the block kernels: entries of stored matrix blocks as doubles, and a
// wave's largest value with its index.
#pragma once

#include <hip/hip_runtime.h>

namespace exa {

// Block entries as doubles: FP64 / FP32 storage, or BF16 kept as the upper 16 bits of an FP32
// (unsigned short storage)
template <typename T>
__device__ __forceinline__ double blk_val(T x) { return static_cast<double>(x); }
template <>
__device__ __forceinline__ double blk_val<unsigned short>(unsigned short x) {
  return static_cast<double>(__uint_as_float(static_cast<unsigned int>(x) << 16));
}

// (v, i) of the wave's largest v, ties to the smaller i, on every lane
__device__ inline void argmax_wave(double& v, int& i) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    double ov = __shfl_xor(v, off);
    int oi = __shfl_xor(i, off);
    if (ov > v || (ov == v && oi < i)) { v = ov; i = oi; }
  }
}

}  // namespace exa

// blkval.hpp -- entries of stored matrix blocks as doubles.
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

}  // namespace exa

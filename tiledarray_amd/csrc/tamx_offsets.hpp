// Source offsets of the general limb split's rows and k (host and device).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace tamx {
namespace split {

// Offset of index x over n modes (extents ext, strides str, the last
// fastest), zero for x past the `count` indices they have: blocks reach past
// a tile's end, and a tile without rows or k has modes of extent zero, which
// nothing divides by.
__host__ __device__ inline int64_t mixed_radix_offset(int x, int count, int n, const int32_t* ext,
                                                      const int64_t* str) {
  if (x >= count) return 0;
  int64_t off = 0;
  for (int d = n - 1; d > 0; --d) {
    const int e = ext[d];
    const int q = x / e;
    off += (int64_t)(x - q * e) * str[d];
    x = q;
  }
  return off + (int64_t)x * str[0];
}

}  // namespace split
}  // namespace tamx

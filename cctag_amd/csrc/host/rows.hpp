// Image rows in memory.
#pragma once

#include <cstddef>

namespace cctagx {

// Whether `height` rows of `width` bytes, `stride` apart, lie within
// `capacity` (at least width * height) bytes from the first on; without a
// product, which could wrap for a stride that is no distance at all.
inline bool rows_fit(size_t capacity, size_t width, size_t height, size_t stride) {
  return height <= 1 || stride <= (capacity - width) / (height - 1);
}

}  // namespace cctagx

// Byte offsets of rows inside a raw buffer resource (32-bit offsets).
#pragma once

#include <stdint.h>

namespace q4nx {

// An offset that lies outside every resource of less than 2 GiB, also with the bytes of one
// row added to it.
constexpr uint32_t kOutOfRange = 0x80000000u;

// Offset of row r of a batch of `rows`, `pitch` bytes apart, rows * pitch < 2^31. A row past the
// batch gets kOutOfRange: r * pitch would wrap for a large pitch and land between the rows.
constexpr uint32_t row_offset(int r, int rows, uint32_t pitch) {
  return r < rows ? (uint32_t)r * pitch : kOutOfRange;
}

}  // namespace q4nx

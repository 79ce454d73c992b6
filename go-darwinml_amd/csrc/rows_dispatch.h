// Host rules of the row kernels' dispatch (k_rows.hip).
#pragma once
#include <stdint.h>

namespace ghip {

// Blocks of 16 bytes (vec elements) that a row of n elements may touch, rows following
// each other from `off` elements into a block.
constexpr int64_t row_blocks(int64_t n, int vec, int off) {
  return n % vec == 0 ? (off + n + vec - 1) / vec  // every row starts at the same offset
                      : (n + 2 * vec - 2) / vec;   // at any offset
}

}  // namespace ghip

// Dispatch rules that are arithmetic on sizes and alignments alone: plain C++, so that a test can hold
// them against what the kernels behind them assume, without a GPU.
#pragma once

#include <stdint.h>

namespace cti {

// Whether the ragged kernel may read a table of `rows` rows of `dim` elements of `elem_bytes`, `row_bytes`
// apart from `base` on, with buffer loads: rows of at least one 16-byte chunk, every chunk 4-byte aligned
// (the last one ends with the row, so the row's own length counts beside the base and the stride; it also
// keeps the table's end, where loads past a bag go, a whole number of words away), and no offset from the
// end on, by up to a row, wrapping around 32 bits.
inline bool ragged_buffer_loads(uint64_t base, int64_t rows, int64_t row_bytes, int64_t dim, int elem_bytes) {
  const int64_t len = dim * elem_bytes;
  const int64_t span = (rows - 1) * row_bytes + len;
  return len >= 16 && base % 4 == 0 && row_bytes % 4 == 0 && len % 4 == 0 && span + len < (int64_t{1} << 32);
}

}  // namespace cti

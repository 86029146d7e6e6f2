// How the rows of a training batch are divided into slices for the weight gradients (plain C++, so that
// it can be checked without a GPU).
#pragma once
#include <algorithm>
#include <cstddef>

namespace fos {

// rows per slice: 512, so that 65,536 rows give each of the 256 CUs work, and more where there would be
// over 256 slices (whose partials the last pass reads); a multiple of the 32 rows staged at a time
constexpr size_t SLICE_ROWS = 512, SLICES = 256, SLICE_STEP = 32;

inline size_t slice_rows(size_t n) {
  return std::max(SLICE_ROWS, ((n + SLICES - 1) / SLICES + SLICE_STEP - 1) / SLICE_STEP * SLICE_STEP);
}

inline size_t slice_count(size_t n) { return (n + slice_rows(n) - 1) / slice_rows(n); }

// The most slices of any batch of up to n rows: what a workspace for n rows has to hold.  slice_count itself
// falls where the rows per slice grow (131,072 rows: 256 slices, 131,073: 241).
inline size_t slice_room(size_t n) { return std::min(SLICES, (n + SLICE_ROWS - 1) / SLICE_ROWS); }

}  // namespace fos

// How the long role of the push cuts a row into column slices, which columns its loader lanes read, and where a slice's columns
// lie in LDS.  Plain constexpr functions: the kernel and a host program can both call them.
#pragma once
#include <cstdint>

namespace hctr {

// Columns per slice of rows of more than 32 floats: kSliceColumns, or kGiantSlice for the longest runs.  (Rows of up to 16 or
// 32 floats are one slice of as many columns.)
#ifndef HCTR_GIANT_SLICE
#define HCTR_GIANT_SLICE 32
#endif
constexpr uint32_t kSliceColumns = 64, kGiantSlice = HCTR_GIANT_SLICE;
static_assert(kSliceColumns % kGiantSlice == 0, "tiers of the long role");

// True: every long run is cut into slices of kGiantSlice columns, because the last slice of kSliceColumns would be half empty.
constexpr bool narrow_slices(uint32_t width) {
  const uint32_t over = width % kSliceColumns;
  return over && over <= kSliceColumns / 2;
}

// the column a lane that is due at column c < width really starts at, where rows travel in overlapping vectors of four
constexpr uint32_t overlapped_col(uint32_t c, uint32_t width) { return c < width - 4 ? c : width - 4; }

// Where the slice's column `place`, column `col` of the row, lies in a slice whose lanes store their four columns where they are
// due: the last lane of a row holds columns width - 4 to width - 1, also if it is due at the last of these only.
constexpr uint32_t overlapped_place(uint32_t place, uint32_t col, uint32_t width) {
  const uint32_t due = col / 4 * 4;
  return due + 4 > width ? place + (due + 4 - width) : place;
}

} // namespace hctr

// How the long role of the push cuts a row into column slices, and which columns its loader lanes read.  Plain constexpr
// functions: the kernel, the host's choice of a kernel and a host program can all call them.
#pragma once
#include <cstdint>

namespace hctr {

constexpr uint32_t kSliceColumns = 64; // at most

// Columns per slice where rows travel in overlapping vectors of four, from `cs` of them (a multiple of four) down: the last
// lane of a row starts at column width - 4 (kOdd4 in kernels.h) and has to stay inside its slice, so slices get narrower
// until the last one holds four columns at least -- if one of 8 to 64 columns will do (slices_hold_overlap).
constexpr uint32_t overlap_slice(uint32_t width, uint32_t cs) {
  while (cs > 8 && width % cs != 0 && width % cs < 4) cs -= 4;
  return cs;
}

// False for the widths that leave one to three columns whatever the slice: 2882880 k + 1, 2 and 3 (2882880 is the least
// common multiple of 8, 12, .. 64).
constexpr bool slices_hold_overlap(uint32_t width) {
  const uint32_t whole = (width + 3) / 4 * 4;
  const uint32_t last = width % overlap_slice(width, whole < kSliceColumns ? whole : kSliceColumns);
  return last == 0 || last >= 4;
}

// the column a lane that is due at column c < width really starts at, where rows travel in overlapping vectors of four
constexpr uint32_t overlapped_col(uint32_t c, uint32_t width) { return c < width - 4 ? c : width - 4; }

} // namespace hctr

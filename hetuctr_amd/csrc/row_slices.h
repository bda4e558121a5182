// How the long role of the push cuts a row into column slices, which columns its loader lanes read, and where a slice's columns
// lie in LDS.  Plain constexpr functions: the kernel and a host program can both call them.
#pragma once
#include <cstdint>

namespace hctr {

// Columns per slice of rows of more than 32 floats: kSliceColumns, or kGiantSlice for the longest runs (narrow_classes).  (Rows of up to 16 or
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

// How many of the leading length classes of a batch's long runs (class c: 2^(17-c) rows and more) are cut into slices of
// kGiantSlice columns, where not all of them are; rows: of the batch's long runs, which `blocks` blocks share.  A slice of 32
// columns costs a block 3.4 ns per row, one of 64 columns 6: narrow slices are more work, but a run is through in little more
// than half the time, which counts where it is longer than half a block's share of the work (where the row is one slice
// of less than 64 columns, and less is won, than four thirds of it), and has 4096 rows.
// The push in us with the line at 16384 rows whatever the batch, at 4096, and by this rule: 64 floats, Zipf 1.05, 426 k keys
// 54.8, 43.5, 44.1; 1.04 M 122.8, 86.8, 92.2; 8.5 M pooled by tens, Zipf 1.4, 427, 436, 426; 128 floats, 1.04 M keys 160.3, 149.1,
// 148.8; 100 floats, 5.2 M 970, 1017, 895; 37 floats, Zipf 1.4, 1.04 M 129.5, 137.5, 129.0, 639 k pooled by threes, 1.2, 55.4, 46.4,
// 44.9.  Down to 256 rows, 37 floats, 195 k keys take 35.2 instead of 25.0; from the whole share on 128 floats, 1.04 M keys
// 161.8; from half of it on 37 floats, 1.04 M keys 138.3.
constexpr int narrow_classes(uint32_t width, uint64_t rows, uint32_t blocks) {
  const uint64_t share = rows * ((width + kSliceColumns - 1) / kSliceColumns) / blocks;
  int c = 0;
  while (c < 6 && (width < kSliceColumns ? (3ull << 17 >> c) >= 4 * share : (2ull << 17 >> c) >= share)) c++;
  return c;
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

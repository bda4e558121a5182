"""The column slices of the push's long role (hetuctr_amd/csrc/row_slices.h), for every row width a table accepts."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hetuctr_amd", "csrc")

# What the kernel does with the functions: lane l of slice s is due at s * cs + 4 l, reads four floats from where it really
# starts, and puts them at (start - s * cs) of an LDS row of `cs` floats.  Every slice before the last two is a whole one.
PROGRAM = r"""
#include <cstdio>
#include "row_slices.h"
using namespace hctr;
static const char *check(uint32_t w, bool overlap) {
  const uint32_t whole = (w + 3) / 4 * 4, most = whole < kSliceColumns ? whole : kSliceColumns;
  const uint32_t cs = overlap ? overlap_slice(w, most) : most, slices = (w + cs - 1) / cs;
  for (uint32_t s = slices > 2 ? slices - 2 : 0; s < slices; s++) {
    const uint32_t first = s * cs;
    uint64_t loaded = 0; // by place in the slice
    for (uint32_t l = 0; l * 4 < cs; l++) {
      const uint32_t due = first + l * 4;
      if (due >= w) continue;
      const uint32_t col = overlap ? overlapped_col(due, w) : due;
      if (col < first || col - first + 4 > cs) return "a lane stores outside its LDS row";
      if (col + 4 > w) return "a lane reads past the row";
      loaded |= 15ull << (col - first);
    }
    for (uint32_t c = first; c < w && c < first + cs; c++)
      if (!(loaded >> (c - first) & 1)) return "a column of the slice is not loaded";
  }
  return nullptr;
}
int main() {
  const uint32_t widest = 1u << 24; // what a table accepts
  int single = 0; // widths whose rows move one float per lane
  for (uint32_t w = 4; w < widest; w++) {
    const char *bad = slices_hold_overlap(w) ? check(w, true) : nullptr;
    if (!slices_hold_overlap(w)) single++;
    if (!bad && w % 4 == 0) bad = check(w, false);
    if (bad) return printf("width %u: %s\n", w, bad), 1;
  }
  return printf("ok %d\n", single), 0;
}
"""


def test_every_width_stays_inside_its_slice(tmp_path):
    src, exe = tmp_path / "slices.cpp", tmp_path / "slices"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I" + CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert (out.returncode, out.stdout) == (0, "ok 15\n"), out.stdout

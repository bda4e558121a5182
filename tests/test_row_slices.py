"""The column slices of the push's long role (hetuctr_amd/csrc/row_slices.h), for every row width a table accepts."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hetuctr_amd", "csrc")

# What the kernel does with the functions: lane l of slice s is due at s * cs + 4 l, reads four floats from where it really
# starts (lanes due behind the row read its first four) and puts them at 4 l of an LDS row of `cs` floats; the lane that sums
# column c of the row, place c - s * cs of the slice, reads where overlapped_place() says.  Every slice before the last two is
# a whole one.
PROGRAM = r"""
#include <cstdio>
#include "row_slices.h"
using namespace hctr;
static const char *check(uint32_t w, uint32_t cs) {
  const uint32_t slices = (w + cs - 1) / cs;
  for (uint32_t s = slices > 2 ? slices - 2 : 0; s < slices; s++) {
    const uint32_t first = s * cs;
    uint32_t holds[kSliceColumns]; // column of the row, by place in LDS
    for (uint32_t l = 0; l * 4 < cs; l++) {
      const uint32_t due = first + l * 4, col = due < w ? overlapped_col(due, w) : 0;
      if (col + 4 > w) return "a lane reads past the row";
      for (uint32_t k = 0; k < 4; k++) holds[l * 4 + k] = col + k;
    }
    for (uint32_t c = first; c < w && c < first + cs; c++) {
      const uint32_t at = overlapped_place(c - first, c, w);
      if (at >= cs) return "a summing lane reads outside its LDS row";
      if (holds[at] != c) return "a summing lane reads another column";
    }
  }
  return nullptr;
}
int main() {
  const uint32_t widest = 1u << 24; // what a table accepts
  int wide = 0;                     // widths with slices of kSliceColumns
  for (uint32_t w = 4; w < widest; w++) {
    const char *bad = nullptr;
    if (w <= 16) {
      bad = check(w, 16);
    } else if (w <= 32) {
      bad = check(w, 32);
    } else {
      bad = check(w, kGiantSlice);
      if (!narrow_slices(w)) {
        wide++;
        if (!bad) bad = check(w, kSliceColumns);
        if (w % kSliceColumns && w % kSliceColumns <= kSliceColumns / 2) bad = "the last slice is half empty";
      }
    }
    if (bad) return printf("width %u: %s\n", w, bad), 1;
  }
  return printf("ok %d\n", wide), 0;
}
"""


def test_every_width_stays_inside_its_slice(tmp_path):
    src, exe = tmp_path / "slices.cpp", tmp_path / "slices"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I" + CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    # half of the widths below 2^24, without 0
    assert (out.returncode, out.stdout) == (0, "ok %d\n" % (2 ** 23 - 1)), out.stdout


def test_the_longest_runs_are_cut_narrower_where_they_outlast_a_block_s_share(tmp_path):
    # the rule in python: classes down to 4096 rows whose runs are half a block's share long at least (four thirds of it, where a row is
    # one slice of less than 64 columns)
    src, exe = tmp_path / "classes.cpp", tmp_path / "classes"
    src.write_text(r"""
#include <cstdio>
#include <initializer_list>
#include "row_slices.h"
using namespace hctr;
int main() {
  for (uint32_t w : {33u, 48u, 63u, 64u, 65u, 128u, 1000u, 1u << 24})
    for (int e = 0; e < 34; e++)
      for (uint64_t rows : {1ull << e, (1ull << e) - 1, 3ull << e}) printf("%u %llu %d\n", w, (unsigned long long)rows, narrow_classes(w, rows, 128));
}
""")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I" + CSRC, str(src), "-o", str(exe)], check=True)
    lines = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, check=True).stdout.split("\n")[:-1]
    assert len(lines) == 8 * 34 * 3
    for line in lines:
        w, rows, got = map(int, line.split())
        share = rows * -(-w // 64) // 128
        want = [c for c in range(6) if (3 * 2 ** (17 - c) >= 4 * share if w < 64 else 2 * 2 ** (17 - c) >= share)]
        assert got == len(want), line

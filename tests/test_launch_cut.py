"""How a launch's blocks are shared out among the shards it serves (hetuctr_amd/csrc/launch_cut.h)."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hetuctr_amd", "csrc")

# Records of 0 blocks to millions, in every place: every block of a launch must find its record and number, no block may be left
# over, and a launch must stay below 2^32 threads (a record that cannot goes alone).
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "launch_cut.h"
using namespace hctr;
constexpr int M = 8;
static const char *check(const std::vector<uint32_t> &need, uint32_t threads, uint32_t each, int launches_expected) {
  int launches = 0;
  for (int i = 0; i < (int)need.size();) {
    BlockCut<M> cut;
    for (auto &f : cut.first) f = 12345; // what the launch before left there
    const int m = cut_blocks(cut, (int)need.size() - i, threads, each, [&](int k) { return need[i + k]; });
    if (m < 1 || m > M) return "a launch serves no record, or too many";
    uint64_t sum = 0;
    for (int k = 0; k < m; k++) {
      const uint32_t n = need[i + k];
      if (cut.blocks[k] != n) return "a record has not the blocks it needs";
      for (uint32_t b : {0u, 1u, n / 2, n - 1})
        if (b < n) {
          uint32_t block = (uint32_t)sum + b;
          if ((int)record_of(cut, block) != k || block != b) return "a block finds another record";
        }
      sum += n;
    }
    if (cut.total != sum) return "blocks without a record";
    if (m > 1 && (sum + (uint64_t)each * m) * threads >= (1ull << 32)) return "too many threads";
    i += m;
    launches++;
  }
  return launches_expected && launches != launches_expected ? "another number of launches" : nullptr;
}
int main() {
  srand(1);
  const uint32_t sizes[] = {0, 0, 1, 2, 7, 300, 53248, 2000000};
  for (int t = 0; t < 200000; t++) {
    std::vector<uint32_t> need(1 + rand() % 20);
    for (auto &n : need) n = sizes[rand() % 8];
    const uint32_t threads = rand() % 2 ? 256 : 512, each = rand() % 2 ? 0 : 384;
    if (const char *bad = check(need, threads, each, 0)) return puts(bad), 1;
  }
  // one large batch and seven tiny ones: 8 x the largest would be 2^33 threads, their sum is a launch
  if (const char *bad = check({2100000, 9, 9, 9, 9, 9, 9, 9}, 512, 384, 1)) return puts(bad), 1;
  // eight of 2^30 threads each: three to a launch; and single ones at and beyond the limit go alone
  if (const char *bad = check(std::vector<uint32_t>(8, 1u << 21), 512, 384, 3)) return puts(bad), 1;
  if (const char *bad = check({1u << 23, 5, (1u << 23) - 1, 0}, 512, 0, 3)) return puts(bad), 1;
  return puts("ok"), 0;
}
"""


def test_every_block_finds_its_record(tmp_path):
    src, exe = tmp_path / "cut.cpp", tmp_path / "cut"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I" + CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert (out.returncode, out.stdout) == (0, "ok\n"), out.stdout

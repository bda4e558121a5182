// How the blocks of one launch are shared out among the records (shards) it serves.  Plain constexpr functions: the kernels,
// their launchers and a host program can all call them.
#pragma once
#include <cstdint>

namespace hctr {

// Record k has blocks first[k] .. first[k + 1): as many as its own batch needs.  (Cut for the largest batch times the records
// instead, a launch for one large batch beside seven small ones is seven eighths idle blocks, and may exceed the 2^32 threads
// a launch can have where a launch per record did not.)
template <int M> struct BlockCut {
  uint32_t first[M + 1] = {};
  constexpr uint32_t blocks(int k) const { return first[k + 1] - first[k]; }
  constexpr uint32_t total() const { return first[M]; }
};

// the record block `block` of the launch works for; `block` becomes its number among that record's blocks
template <int M> constexpr int record_of(const BlockCut<M> &cut, uint32_t &block) {
  int k = 0;
  for (int i = 1; i < M; i++) k += block >= cut.first[i] ? 1 : 0;
  block -= cut.first[k];
  return k;
}

// Blocks of `threads` threads for the records that need need(0), need(1), .. of them, need(count - 1) the last: as many records
// as one launch takes (M, and fewer than 2^32 threads in all; the first one goes in whatever it needs, alone it is for the
// runtime to accept or refuse).  `each`: blocks a record gets on top of those.  Returns how many records went in.
template <int M, typename F> constexpr int cut_blocks(BlockCut<M> &cut, int count, uint32_t threads, uint32_t each, F &&need) {
  uint64_t total = 0;
  int m = 0;
  for (; m < count && m < M; m++) {
    const uint64_t with = total + need(m);
    if (m > 0 && (with + (uint64_t)each * (m + 1)) * threads >= (1ull << 32)) break;
    total = with;
    cut.first[m + 1] = (uint32_t)total;
  }
  for (int k = m; k < M; k++) cut.first[k + 1] = cut.first[m];
  return m;
}

} // namespace hctr

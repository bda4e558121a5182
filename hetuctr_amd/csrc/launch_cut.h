// How the blocks of one launch are shared out among the records (shards) it serves.  Plain constexpr functions: the kernels,
// their launchers and a host program can all call them.
#pragma once
#include <cstdint>

namespace hctr {

// Record k has blocks first[k] .. first[k] + blocks[k) of the launch, as many as its own batch needs.  (Cut for the largest batch
// times the records instead, a launch for one large batch beside seven small ones is seven eighths idle blocks, and may
// exceed the 2^32 threads a launch can have where a launch per record did not.  Eight shards, one batch of 1.7 M keys x 128
// floats and seven of 1000: a step takes 1313 us, cut for the largest 2149, with a launch per shard 1360; four shards of 426 k
// keys each 1035 .. 1042 and 1038 .. 1043.)
template <int M> struct BlockCut {
  uint32_t first[M] = {};
  uint32_t blocks[M] = {};
  uint32_t total = 0;
};
constexpr uint32_t kNoStart = 0x7fffffffu; // a start behind every block

// The record that block `block` of the launch works for; `block` becomes its number among that record's blocks.  Always inline: a
// call that is left standing until late makes the compiler copy the kernel's records to scratch memory (a push of 306 us
// took 4150).
template <int M> [[gnu::always_inline]] constexpr uint32_t record_of(const BlockCut<M> &cut, uint32_t &block) {
  uint32_t k = 0; // starts that do not lie behind the block (the sign of start - 1 - block: scalar arithmetic throughout)
  for (int i = 1; i < M; i++) k += (cut.first[i] - 1 - block) >> 31;
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
    const uint64_t n = need(m);
    if (m > 0 && (total + n + (uint64_t)each * (m + 1)) * threads >= (1ull << 32)) break;
    cut.first[m] = (uint32_t)total;
    cut.blocks[m] = (uint32_t)n;
    total += n;
  }
  for (int k = m; k < M; k++) cut.first[k] = kNoStart, cut.blocks[k] = 0;
  cut.total = (uint32_t)total;
  return m;
}

} // namespace hctr

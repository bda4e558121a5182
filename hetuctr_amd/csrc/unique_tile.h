// What the index keeps per unique key, written by a block for one tile of the sorted keys: shared by the unique pass of
// large batches (one block per tile) and by the single-block index of small ones.
#pragma once
#include "kernels.h"

namespace hctr {

constexpr int kUBlock = 512; // threads of such a block

// Position j = base + k * kUBlock + thread of the sorted order holds key[k] (j < n); edge[k]: the key before it on lane 0 of
// a wave (anything at j = 0).  s: this thread's share of the unique keys before the tile.  Every load and store is coalesced
// across the wave.  Contains barriers: every thread of the block calls it.
template <typename K, int ITEMS>
__device__ __forceinline__ void emit_unique_tile(const K (&key)[ITEMS], const K (&edge)[ITEMS], uint32_t s, uint32_t base,
                                                 uint32_t n, int id_bits, int nrank, const slot_t *__restrict__ slot,
                                                 const BatchView &b, uint32_t *__restrict__ u_copy) {
  constexpr int NW = kUBlock / kWave;
  __shared__ uint32_t sm[NW + 1];
  __shared__ uint32_t wsum[ITEMS * NW + 1];
  const unsigned lane = lane_id();
  const int w = threadIdx.x / kWave;
  K pk[ITEMS];
  bool head[ITEMS];
  uint32_t before[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; k++) {
    const uint32_t j = base + k * kUBlock + threadIdx.x;
    const bool valid = j < n;
    const K up = (K)__shfl_up(key[k], 1, kWave);
    pk[k] = lane == 0 ? edge[k] : up;
    head[k] = valid && (j == 0 || key[k] != pk[k]);
    const uint64_t m = __ballot(head[k]);
    before[k] = __popcll(m & ((1ull << lane) - 1ull));
    if (lane == 0) wsum[k * NW + w] = __popcll(m);
  }
  // the directory lookups of the heads travel while the ranks are worked out
  const K id_mask = (K)(((uint64_t)1 << id_bits) - 1);
  slot_t off[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; k++) off[k] = head[k] ? slot[(uint64_t)(key[k] & id_mask)] : kNoSlot;
  uint32_t prefix;
  block_exclusive_scan<kUBlock>(s, sm, prefix); // unique ranks before this tile
  if (threadIdx.x < kWave) { // the wave totals, in item order, by one wave
    uint32_t run = 0;
    for (int i0 = 0; i0 < ITEMS * NW; i0 += kWave) {
      const bool in = i0 + (int)lane < ITEMS * NW;
      const uint32_t v = in ? wsum[i0 + lane] : 0u;
      const uint32_t inc = wave_inclusive_scan(v);
      if (in) wsum[i0 + lane] = run + inc - v;
      run += __shfl(inc, kWave - 1, kWave);
    }
  }
  __syncthreads();
  K *ukey = (K *)b.ukey;
#pragma unroll
  for (int k = 0; k < ITEMS; k++) {
    const uint32_t j = base + k * kUBlock + threadIdx.x;
    if (j >= n) continue;
    const uint32_t rank = prefix + wsum[k * NW + w] + before[k] + (head[k] ? 1u : 0u) - 1u;
    const int r = (int)(key[k] >> id_bits);
    if (head[k]) {
      ukey[rank] = key[k];
      b.run_start[rank] = j;
      b.uoff[rank] = off[k];
      const int r_prev = j == 0 ? -1 : (int)(pk[k] >> id_bits);
      for (int i = r_prev + 1; i <= r; i++) b.bucket_lo[i] = rank;
    }
    b.rank_sorted[j] = rank;
    if (j == n - 1) {
      const uint32_t U = rank + 1;
      *b.d_U = U;
      if (u_copy) *u_copy = U;
      b.run_start[U] = n;
      for (int i = r + 1; i <= nrank; i++) b.bucket_lo[i] = U;
    }
  }
}

} // namespace hctr

// Key preprocess of one batch after the sort: unique keys, run starts, inverse index, owner buckets,
// resident offsets; and the push plan of the previous batch.
// Reference: csrc/core/preprocess.cu:11-182 (kernels generate_sort_kv, write_sort_result,
// preprocess_batch_data, compute_idx_map, block_cvt_offset_to_shape, decide_update and the
// cub RunLengthEncode / ExclusiveSum calls between them).
#include <algorithm>

#include "kernels.h"
#include "radix_sort.h"
#include "run_lists.h"
#include "tile_sort.h"
#include "unique_tile.h"

namespace hctr {
namespace {

constexpr int kBlock = 256;
constexpr int kItems = 8;
constexpr int kTile = kBlock * kItems; // 2048: scan_blocks(n) sizes the scratch

// ids -> sort keys (owner << id_bits | id; they are the batch's copy of the ids as well), the range check, the reset
// of the batch's run counters, and the per-tile counts of the first sort pass' digit: a block works on one sort tile, so the sort
// needs no counting launch of its own for that pass.  This is the one kernel that reads the caller's buffer: the
// call may return when it has said that it has them all (ReadSignal), or is through.
template <typename K, int ITEMS, int M> // M: records of the launch
__global__ __launch_bounds__(kSortBlock) void make_keys(Records<KeyShard, M> shards, int id_bits, int dbits) {
  uint32_t tile, tiles;
  const KeyShard &S = my_record(shards, tile, tiles);
  const index_t *__restrict__ keys = S.ids;
  const uint32_t n = S.n;
  const uint64_t id_max = S.t.id_max;
  const int nrank = S.t.nrank;
  const worker_t *__restrict__ root = S.t.root;
  K *__restrict__ comp = (K *)S.comp_keys;
  uint32_t *__restrict__ err = S.err, *__restrict__ nlong = S.nlong, *__restrict__ counts = S.sort_counts;
  const bool ids32 = S.ids32;
  __shared__ uint32_t h[kSortMaxBins];
  const uint32_t nb = 1u << dbits, mask = nb - 1;
  if (counts)
    for (uint32_t i = threadIdx.x; i < nb; i += kSortBlock) h[i] = 0;
  if (tile == 0 && threadIdx.x < kRunCounters && nlong) nlong[threadIdx.x] = 0; // counters of this batch
  const uint32_t base = tile * (ITEMS * kSortBlock);
  uint64_t id[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; k++) {
    const uint32_t i = base + k * kSortBlock + threadIdx.x;
    // the caller's ids are read here and nowhere else (ids32: as narrowed on their way from pageable host memory)
    id[k] = i >= n ? 0 : ids32 ? (uint64_t)load_once(&((const uint32_t *)keys)[i]) : (uint64_t)load_once(&keys[i]);
  }
  __syncthreads();
  bool bad = false;
#pragma unroll
  for (int k = 0; k < ITEMS; k++) {
    const uint32_t i = base + k * kSortBlock + threadIdx.x;
    if (i < n && id[k] >= id_max) { // also catches negative ids
      bad = true;
      id[k] = 0;
    }
  }
  uint64_t owner[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; k++) owner[k] = nrank > 1 ? root[id[k]] : 0;
#pragma unroll
  for (int k = 0; k < ITEMS; k++) {
    const uint32_t i = base + k * kSortBlock + threadIdx.x;
    if (i < n) store_key(comp + i, (K)((owner[k] << id_bits) | id[k]), S.read);
  }
  tell_ids_read(S.read, tiles, bad, err);
#pragma unroll
  for (int k = 0; k < ITEMS; k++) {
    const uint32_t i = base + k * kSortBlock + threadIdx.x;
    const K c = (K)((owner[k] << id_bits) | id[k]);
    if (counts) count_digit(h, (uint32_t)c & mask, i < n);
  }
  if (!counts) return; // the keys alone: another sort counts for itself
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < nb; i += kSortBlock) counts[(size_t)tile * nb + i] = h[i];
}

// The unique pass works on tiles of kUTile sorted positions; position j of a tile is handled by thread (j % kUBlock)
// in round (j / kUBlock): every load and store below is coalesced across the wave.
#ifndef HCTR_UNIQUE_ITEMS
#define HCTR_UNIQUE_ITEMS 8
#endif
constexpr int kUItems = HCTR_UNIQUE_ITEMS, kUTile = kUBlock * kUItems;
inline unsigned unique_tiles(uint32_t n) { return div_up(n, kUTile); }

// Heads (sorted positions that hold another key than the position before) are counted per chunk of sorted positions,
// in a form that needs no look at a neighbouring chunk: the heads of a chunk other than its first position, and the
// chunk's first and last key.  The last launch of the tile-sorted passes leaves these three per chunk (tile_sort.h);
// after the other sort head_count makes them, one chunk per tile of the unique pass.
template <typename K>
__global__ __launch_bounds__(kUBlock) void head_count(const K *__restrict__ sk, uint32_t n,
                                                      uint32_t *__restrict__ inner, K *__restrict__ first,
                                                      K *__restrict__ last) {
  __shared__ uint32_t sm[kUBlock / kWave + 1];
  const uint32_t base = blockIdx.x * kUTile;
  const unsigned lane = lane_id();
  K key[kUItems], edge[kUItems];
#pragma unroll
  for (int k = 0; k < kUItems; k++) {
    const uint32_t j = base + k * kUBlock + threadIdx.x;
    key[k] = j < n ? sk[j] : (K)0;
    edge[k] = (lane == 0 && j < n && j > base) ? sk[j - 1] : (K)0; // the key before a wave's first position
  }
  uint32_t c = 0;
#pragma unroll
  for (int k = 0; k < kUItems; k++) {
    const uint32_t j = base + k * kUBlock + threadIdx.x;
    const K up = (K)__shfl_up(key[k], 1, kWave);
    const K pk = lane == 0 ? edge[k] : up;
    c += (j < n) && j > base && key[k] != pk;
  }
  uint32_t total;
  block_exclusive_scan<kUBlock>(c, sm, total);
  if (threadIdx.x == 0) {
    inner[blockIdx.x] = total;
    first[blockIdx.x] = key[0];
    last[blockIdx.x] = sk[min(base + kUTile, n) - 1];
  }
}

// One block per tile of ITEMS * kUBlock sorted positions; position j of a tile is handled by thread (j % kUBlock) in
// round (j / kUBlock).  chunk: sorted positions per entry of the head counts (a divisor of the tile).
template <typename K, int ITEMS, int M>
__global__ __launch_bounds__(kUBlock) void unique_emit(Records<UniqueShard, M> shards, int id_bits, uint32_t chunk) {
  uint32_t tile, tiles;
  const UniqueShard &S = my_record(shards, tile, tiles);
  const K *__restrict__ sk = (const K *)S.sorted_keys;
  const uint32_t n = S.b.n;
  const uint32_t *__restrict__ head_inner = S.heads.inner;
  const K *__restrict__ head_first = (const K *)S.heads.first, *__restrict__ head_last = (const K *)S.heads.last;
  constexpr uint32_t kTileU = ITEMS * kUBlock;
  const uint32_t base = tile * kTileU;
  const unsigned lane = lane_id();
  // everything that comes from memory first: the keys of the tile, the key before every wave's first position and the
  // head counts of the chunks before the tile
  K key[ITEMS], edge[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; k++) {
    const uint32_t j = base + k * kUBlock + threadIdx.x;
    key[k] = j < n ? sk[j] : (K)0;
    edge[k] = (lane == 0 && j < n && j > 0) ? sk[j - 1] : (K)0;
  }
  uint32_t s = 0;
  const uint32_t chunks_before = base / chunk;
  for (uint32_t i = threadIdx.x; i < chunks_before; i += kUBlock)
    s += head_inner[i] + ((i == 0 || head_first[i] != head_last[i - 1]) ? 1u : 0u);
  emit_unique_tile<K, ITEMS>(key, edge, s, base, n, id_bits, S.t.nrank, S.t.slot, S.b, S.u_copy);
}

// The inverse index in batch order (the reference's d_idx_map).  The hot path works in sorted order
// (sorted_arg + rank_sorted are the same mapping, grouped by key) and never reads this array; it is
// materialised on request.
__global__ __launch_bounds__(kBlock) void scatter_idx_map(BatchView b) {
  const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
  if (j < b.n) b.idx_map[b.sorted_arg[j]] = b.rank_sorted[j];
}

// the run lists of a batch by a launch of their own (run_lists.h), for a batch no gather builds them for
__global__ __launch_bounds__(kRunListBlock) void list_long_runs(BatchView b) {
  __shared__ uint32_t cnt[kRunLists], base[kRunLists];
  list_runs_chunk(b, blockIdx.x, cnt, base);
}

// ---- push plan, three launches for all shards of a group ----------------------------------------------------------
typedef Records<PlanShard, kShardsPerLaunch> PlanShards;
typedef Records<BucketShard, kShardsPerLaunch> BucketShards;

// need[u] of one tile of unique keys and the tile's sum
template <typename K>
__global__ __launch_bounds__(kBlock) void plan_decide(PlanShards shards, int id_bits) {
  __shared__ uint32_t sm[kBlock / kWave + 1];
  uint32_t tile, tiles;
  const PlanShard &S = my_record(shards, tile, tiles);
  const uint32_t U = *S.b.d_U;
  if (tile * kTile >= U) return; // the grid is cut for the batches' keys
  uint32_t c = 0;
#pragma unroll
  for (int k = 0; k < kItems; k++) {
    const uint32_t u = tile * kTile + k * kBlock + threadIdx.x;
    if (u >= U) continue;
    const int r = (int)(((const K *)S.b.ukey)[u] >> id_bits);
    const slot_t o = S.b.uoff[u];
    const version_t cnt = (version_t)(S.b.run_start[u + 1] - S.b.run_start[u]);
    uint32_t nd;
    if (r == S.t.rank) nd = 0;
    else if (o == kNoSlot) nd = 1;
    else nd = (S.t.upd[o] + cnt <= S.t.push_bound) ? 0 : 1;
    S.need[u] = nd;
    c += nd;
  }
  uint32_t total;
  block_exclusive_scan<kBlock>(c, sm, total);
  if (threadIdx.x == 0) S.block_sums[tile] = total;
}

__global__ __launch_bounds__(kBlock) void plan_scan(PlanShards shards) {
  __shared__ uint32_t sm[kBlock / kWave + 1];
  uint32_t tile, tiles;
  const PlanShard &S = my_record(shards, tile, tiles);
  const uint32_t U = *S.b.d_U;
  if (tile * kTile >= U) return;
  uint32_t s = 0;
  for (uint32_t i = threadIdx.x; i < tile; i += kBlock) s += S.block_sums[i];
  uint32_t prefix;
  block_exclusive_scan<kBlock>(s, sm, prefix);
  const uint32_t j0 = tile * kTile + threadIdx.x * kItems;
  uint32_t v[kItems], c = 0;
#pragma unroll
  for (int k = 0; k < kItems; k++) {
    v[k] = (j0 + k < U) ? S.need[j0 + k] : 0u;
    c += v[k];
  }
  uint32_t total;
  uint32_t run = prefix + block_exclusive_scan<kBlock>(c, sm, total);
  const bool last = (tile + 1) * kTile >= U;
#pragma unroll
  for (int k = 0; k < kItems; k++) {
    if (j0 + k < U) S.prefix[j0 + k] = run;
    run += v[k];
  }
  if (last && threadIdx.x == kBlock - 1) *S.total = run;
}

__global__ void plan_counts(PlanShards shards, int nrank) {
  const PlanShard &S = shards.s[blockIdx.x];
  const int d = threadIdx.x;
  if (d > nrank) return;
  uint64_t c = 0;
  if (d < nrank) {
    const uint32_t U = *S.b.d_U;
    const uint32_t lo = S.b.bucket_lo[d], hi = S.b.bucket_lo[d + 1];
    const uint32_t a = lo >= U ? *S.total : S.prefix[lo];
    const uint32_t e = hi >= U ? *S.total : S.prefix[hi];
    c = U ? (uint64_t)(e - a) : 0;
  }
  S.cnt_out[d] = c;
  S.host_out[d] = c; // pinned host memory: the caller sizes the push buffers from it, no copy in between
}

__global__ void bucket_sizes(BucketShards shards, int nrank) {
  const BucketShard &S = shards.s[blockIdx.x];
  const int d = threadIdx.x;
  if (d > nrank) return;
  const uint64_t c = d == nrank ? 0 : (uint64_t)(S.bucket_lo[d + 1] - S.bucket_lo[d]);
  S.cnt_out[d] = c;
  S.host_out[d] = c; // pinned host memory, like the number of unique keys beside it
  if (d == 0) *S.host_U = *S.d_U;
}

} // namespace

void launch_make_keys(hipStream_t s, const KeyLayout &kl, const KeyShard *shards, int count) {
  const int dbits = sort_first_digit_bits(kl.total_bits);
  auto make = [&](int k) {
    HCTR_CHECK(!shards[k].ids32 || shards[k].t.id_max <= 0xffffffffull, "internal: narrowed ids and a table of 2^32 rows or more");
    HCTR_CHECK(sort_tile(shards[k].n) == sort_tile(shards[0].n), "internal: batches of one launch differ in shape");
    return shards[k];
  };
  auto blocks = [&](int k) { return (uint32_t)sort_tiles(shards[k].n); };
  launch_one_or_records<KeyShard>(count, kSortBlock, make, blocks, [&](const auto &p, int) {
    constexpr int M = sizeof p.s / sizeof p.s[0];
    const dim3 grid = grid_of(p);
#define CALL(I)                                                                                                     \
  do {                                                                                                              \
    if (kl.wide) hipLaunchKernelGGL((make_keys<uint64_t, I, M>), grid, dim3(kSortBlock), 0, s, p, kl.id_bits, dbits); \
    else hipLaunchKernelGGL((make_keys<uint32_t, I, M>), grid, dim3(kSortBlock), 0, s, p, kl.id_bits, dbits);       \
  } while (0)
    HCTR_SORT_ITEMS_DISPATCH(shards[0].n, CALL);
#undef CALL
    HCTR_HIP(hipGetLastError());
  });
}

void launch_unique(hipStream_t s, const KeyLayout &kl, const UniqueShard *shards, int count, bool count_heads) {
  HCTR_CHECK(!count_heads || count == 1, "internal: heads are counted for one batch at a time");
  const HeadChunks &heads = shards[0].heads;
  // the tile of the pass: that of the sort that left the head counts, or kUTile when they are counted here
  const int items = count_heads ? kUItems : (int)(heads.chunk / kWave);
  const uint32_t chunk = count_heads ? (uint32_t)kUTile : heads.chunk;
  auto make = [&](int k) {
    HCTR_CHECK(shards[k].heads.chunk == heads.chunk, "internal: batches of one launch differ in shape");
    return shards[k];
  };
  auto blocks = [&](int k) { return div_up(shards[k].b.n, (size_t)items * kUBlock); };
  launch_one_or_records<UniqueShard>(count, kUBlock, make, blocks, [&](const auto &p, int) {
    constexpr int M = sizeof p.s / sizeof p.s[0];
    const dim3 grid = grid_of(p);
#define EMIT(K, I) hipLaunchKernelGGL((unique_emit<K, I, M>), grid, dim3(kUBlock), 0, s, p, kl.id_bits, chunk)
#define EMIT_K(K)                                                                                          \
  do {                                                                                                     \
    if (count_heads)                                                                                       \
      hipLaunchKernelGGL(head_count<K>, grid, dim3(kUBlock), 0, s, (const K *)p.s[0].sorted_keys, p.s[0].b.n, heads.inner, \
                         (K *)heads.first, (K *)heads.last);                                              \
    switch (items) {                                                                                       \
      case 2: EMIT(K, 2); break;                                                                           \
      case 4: EMIT(K, 4); break;                                                                           \
      case 8: EMIT(K, 8); break;                                                                           \
      case 13: EMIT(K, 13); break;                                                                         \
      case 16: EMIT(K, 16); break;                                                                         \
      default: throw Error("hetuCTR: internal: no unique pass for this tile shape");                       \
    }                                                                                                      \
  } while (0)
    if (kl.wide) EMIT_K(uint64_t);
    else EMIT_K(uint32_t);
#undef EMIT_K
#undef EMIT
    HCTR_HIP(hipGetLastError());
  });
}

void launch_idx_map(hipStream_t s, const BatchView &b) {
  if (!b.n) return;
  hipLaunchKernelGGL(scatter_idx_map, dim3(div_up(b.n, kBlock)), dim3(kBlock), 0, s, b);
  HCTR_HIP(hipGetLastError());
}

void launch_list_long_runs(hipStream_t s, const BatchView &b) { // the class counters were zeroed by make_keys
  if (!b.n) return;
  hipLaunchKernelGGL(list_long_runs, dim3(div_up(b.n, kRunListBlock)), dim3(kRunListBlock), 0, s, b);
  HCTR_HIP(hipGetLastError());
}

void launch_plans(hipStream_t s, const KeyLayout &kl, const PlanShard *shards, int count) {
  auto make = [&](int k) { return shards[k]; };
  auto blocks = [&](int k) { return div_up(shards[k].b.n, kTile); };
  launch_records<PlanShard, kShardsPerLaunch>(count, kBlock, make, blocks, [&](const PlanShards &p, int m) {
    const dim3 grid = grid_of(p);
    if (kl.wide) hipLaunchKernelGGL(plan_decide<uint64_t>, grid, dim3(kBlock), 0, s, p, kl.id_bits);
    else hipLaunchKernelGGL(plan_decide<uint32_t>, grid, dim3(kBlock), 0, s, p, kl.id_bits);
    hipLaunchKernelGGL(plan_scan, grid, dim3(kBlock), 0, s, p);
    const int nrank = p.s[0].t.nrank;
    hipLaunchKernelGGL(plan_counts, dim3(m), dim3(nrank + 1), 0, s, p, nrank);
    HCTR_HIP(hipGetLastError());
  });
}

void launch_bucket_sizes(hipStream_t s, int nrank, const BucketShard *shards, int count) {
  auto make = [&](int k) { return shards[k]; };
  launch_records<BucketShard, kShardsPerLaunch>(count, nrank + 1, make, [](int) { return 1u; }, [&](const BucketShards &p, int m) {
    hipLaunchKernelGGL(bucket_sizes, dim3(m), dim3(nrank + 1), 0, s, p, nrank);
    HCTR_HIP(hipGetLastError());
  });
}

} // namespace hctr

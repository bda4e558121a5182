// Pull side and owner side of a step: version lookup for the query, applying pushed rows, deciding which
// queried rows are outdated, packing the rows to return, refreshing cached rows and the final gather of
// every key's row into the caller's output.
// Reference: csrc/core/generate_query.cu:91-106, csrc/core/handle_query.cu:7-116,
// csrc/core/writeback.cu:8-56.
#include <algorithm>

#include "kernels.h"
#include "run_lists.h"

namespace hctr {
namespace {

constexpr int kBlock = 256;
static_assert(kBlock == kRunListBlock, "the gather's blocks list runs chunk by chunk");
typedef float floatx4 __attribute__((ext_vector_type(4)));

// Rows travel in vectors of kCols<VEC> columns per lane: 4 (the width is a multiple of four and every pointer 16-byte
// aligned), kOdd4 (any other width from 4 on: see kernels.h) or 1.
template <int VEC> struct RowVec;
template <> struct RowVec<4> { typedef floatx4 T; };
template <> struct RowVec<kOdd4> { typedef floatx4 T __attribute__((aligned(4))); };
template <> struct RowVec<1> { typedef float T; };
// row[0 .. kCols) = v, without the columns the lane before writes too
template <int VEC> __device__ __forceinline__ void store_own(embed_t *row, typename RowVec<VEC>::T v, uint32_t shared) {
  typedef typename RowVec<VEC>::T V;
  if constexpr (VEC == kOdd4) {
    if (shared) {
#pragma unroll
      for (uint32_t k = 1; k < 4; k++)
        if (k >= shared) row[k] = v[k];
      return;
    }
  }
  *(V *)row = v;
}

// The queries of a step (csrc/core/generate_query.cu:91-106): per unique key its id and the version of the local copy
// (invalid if the key is not cached here), written where the key's owner reads its queries: place u + delta[owner]
// of a receive area all owners share.
// (This and the other kernels of a shard's own batch: see kShardsPerLaunch.)
typedef Records<PullShard, kShardsPerLaunch> PullShards;
template <typename K>
__global__ __launch_bounds__(kBlock) void build_queries(PullShards shards, int id_bits) {
  uint32_t block, blocks;
  const PullShard &S = my_record(shards, block, blocks);
  const BatchView &c = S.b;
  const uint32_t u = block * kBlock + threadIdx.x;
  if (u >= c.n || u >= *c.d_U) return;
  const slot_t o = c.uoff[u];
  const K key = ((const K *)c.ukey)[u];
  const uint32_t pos = u + S.delta[(uint32_t)(key >> id_bits)];
  S.q_idx[pos] = (index_t)(key & (K)(((uint64_t)1 << id_bits) - 1));
  // (of rows the shard owns none: no owner asks whether its own copy is outdated, and it may be moving the version just now)
  S.q_ver[pos] = o != kNoSlot && (uint32_t)o < S.t.n_cached ? S.t.ver[o] : kInvalidVersion;
}

// ---- owner side: every kernel below serves ALL shards of a loopback group in one launch (blockIdx.y = shard), the
// way the shards' GPUs would work side by side; with one shard per process the grid is one row high.
//
// Received pushes (csrc/core/handle_query.cu:106-116 applies them source by source, in rank order).  The rows that hit
// one target must be added in source order, so a target's rows all go to one block: every source's segment of the
// receive buffer is ascending in id (it is a slice of the sender's sorted unique keys), block b takes the ids
// between two splitters drawn from the longest segment, finds that id range in every other segment by binary search,
// and walks the sources in order with a barrier between them.  Inside a source ids are distinct, so its rows are
// applied in parallel, kAhead rows per group of LPR lanes at a time.
//
// A search is done by kProbes lanes at once, which cut what is left into kProbes + 1 pieces per round, and both ends of all ranges
// are searched for side by side: 3 or 4 dependent loads for segments of 5 k rows where one lane per source, one end after the
// other, took 24.  (Four shards of 53 k keys: 20.9 -> 17.2 us.)
constexpr uint32_t kProbes = 16;
// first position in [lo, hi) whose id is >= x; the kProbes neighbouring lanes of a group call it with the same arguments
__device__ __forceinline__ uint32_t lower_bound_id(const index_t *__restrict__ a, uint32_t lo, uint32_t hi, index_t x) {
  const uint32_t probe = threadIdx.x % kProbes, shift = threadIdx.x % kWave / kProbes * kProbes;
  while (lo < hi) {
    const uint32_t n = hi - lo, step = n <= kProbes ? 1 : (n - 1) / (kProbes + 1) + 1, at = (probe + 1) * step - 1;
    const bool below = at < n && a[lo + at] < x;
    const uint32_t c = __popc((uint32_t)(__ballot(below) >> shift) & ((1u << kProbes) - 1)); // ids ascend: the first c probes
    if (c < kProbes) hi = min(hi, lo + (c + 1) * step - 1);
    lo += c * step;
  }
  return lo;
}
#ifndef HCTR_APPLY_AHEAD
#define HCTR_APPLY_AHEAD 2
#endif
#ifndef HCTR_APPLY_BATCHES
#define HCTR_APPLY_BATCHES 1
#endif
// Rows of one source a group works on together (distinct ids, hence distinct targets), and batches of that many rows
// per group and block.  Small blocks measured fastest: the kernel is a stream of independent read-modify-writes, and
// what limits it is how evenly the blocks spread over the chip, not the loads one wave keeps in flight.
constexpr int kApplyAhead = HCTR_APPLY_AHEAD;
constexpr int kApplyBatches = HCTR_APPLY_BATCHES;
// The slot of an id the shard owns, kNoSlot for any other id.  Slots below n_cached hold the cached copies of rows
// other shards own, so the slot alone tells (no look at the owner table).
__device__ __forceinline__ slot_t owned_slot(const slot_t *__restrict__ slot, uint64_t id, uint64_t id_max, uint32_t n_cached) {
  if (id >= id_max) return kNoSlot;
  const slot_t o = slot[id];
  return (o != kNoSlot && (uint32_t)o >= n_cached) ? o : kNoSlot;
}
template <int VEC, int LPR>
__global__ __launch_bounds__(kBlock) void apply_remote_all(const OwnerShard *__restrict__ shards, int nsrc,
                                                           uint32_t rows_per_block) {
  typedef typename RowVec<VEC>::T V;
  constexpr int kGroups = kBlock / LPR;
  const OwnerShard &S = shards[blockIdx.y];
  if (blockIdx.x >= S.push_blocks) return;
  const index_t *__restrict__ rg_idx = S.rg_idx;
  const version_t *__restrict__ rg_cnt = S.rg_cnt;
  const embed_t *__restrict__ rg_val = S.rg_val;
  const slot_t *__restrict__ slot = S.t.slot;
  embed_t *__restrict__ emb = S.t.emb;
  version_t *__restrict__ ver = S.t.ver;
  const uint64_t id_max = S.t.id_max;
  const uint32_t n_cached = S.t.n_cached, W = S.t.width;
  __shared__ uint32_t lo[256], hi[256];
  const int longest = S.longest;
  const uint32_t big_lo = S.rg_seg[longest], big_hi = S.rg_seg[longest + 1];
  const uint32_t first = big_lo + blockIdx.x * rows_per_block, last = first + rows_per_block;
  for (int q = threadIdx.x / kProbes; q < 2 * nsrc; q += kBlock / kProbes) { // lower and upper end for every source
    const int s = q / 2;
    const bool upper = q % 2;
    const uint32_t a = S.rg_seg[s], b = S.rg_seg[s + 1], at = upper ? last : first;
    uint32_t end;
    if (s == longest) end = min(at, big_hi);           // the splitters are this segment's own rows
    else if (upper && last >= big_hi) end = b;         // the last block ends above every id
    else if (!upper && blockIdx.x == 0) end = a;       // block 0 starts below every id
    else end = lower_bound_id(rg_idx, a, b, rg_idx[at]);
    if (threadIdx.x % kProbes == 0) (upper ? hi : lo)[s] = end;
  }
  __syncthreads();
  const uint32_t gl = threadIdx.x % LPR;
  constexpr int kAhead = kApplyAhead;
  bool bad = false;
  for (int s = 0; s < nsrc; s++) {
    const uint32_t end = hi[s];
    for (uint32_t k0 = lo[s] + threadIdx.x / LPR; k0 < end; k0 += kGroups * kAhead) {
      slot_t o[kAhead];
      uint64_t id[kAhead];
#pragma unroll
      for (int a = 0; a < kAhead; a++) id[a] = (uint64_t)rg_idx[min(k0 + a * kGroups, end - 1)];
#pragma unroll
      for (int a = 0; a < kAhead; a++) {
        o[a] = owned_slot(slot, id[a], id_max, n_cached);
        if (k0 + a * kGroups >= end) o[a] = kNoSlot;
        else if (o[a] == kNoSlot) bad = true;
      }
      if (gl == 0) {
#pragma unroll
        for (int a = 0; a < kAhead; a++)
          if (o[a] != kNoSlot) ver[o[a]] += load_once(rg_cnt + k0 + a * kGroups);
      }
      for (uint32_t c = gl * kCols<VEC>; c < W; c += LPR * kCols<VEC>) {
        const uint32_t col = lane_col<VEC>(c, W);
        V cur[kAhead], add[kAhead];
#pragma unroll
        for (int a = 0; a < kAhead; a++) {
          if (o[a] == kNoSlot) continue;
          cur[a] = *(const V *)(emb + (size_t)o[a] * W + col);
          add[a] = __builtin_nontemporal_load((const V *)(rg_val + (size_t)(k0 + a * kGroups) * W + col)); // read once: keep it out of the caches
        }
#pragma unroll
        for (int a = 0; a < kAhead; a++)
          if (o[a] != kNoSlot) store_own<VEC>(emb + (size_t)o[a] * W + col, cur[a] + add[a], c - col);
      }
    }
    __syncthreads(); // the next source may push to the same rows
  }
  if (bad && gl == 0) atomicOr(S.err, 2u);
}

// Owner side of the pull (csrc/core/handle_query.cu:7-78) in three launches; the first two work on tiles of kBlock
// received queries, one query per thread.
// decide_count: the outdated flag of every query (pull rule, self-exempt, :47-54) and the number of flags per tile.
// scan_positions: a tile's flags scanned behind the tiles before it -> position of every flagged query among the
// returned rows (:56-57, :74-75), and the first returned row of every requester's segment (:59-61) written both to
// device memory, where place_returns reads it, and to the host.
// pack_rows: version and row of every flagged query packed at its position (:24-40), from the list of their slots
// that scan_positions leaves.
// One block.  Thread d, owner: its queries per requester in rank order (rq_seg), their number, the tiles of its flag
// scan; then the owners' pieces of the area in rank order; thread s, requester: what it adds to a unique key's rank
// per owner (query_delta), and what owner d adds to the place of one of s' queries to get the place of its flag in
// s' array (got_delta: s' flags stand in owner order).  Up to kPlaceLds shards the matrix of counts is fetched into LDS
// by all threads at once (one memory round trip instead of one per entry and thread).
constexpr int kPlaceLds = 48;
struct PlaceSources { // of the first kPlaceLds shards: where their counts lie, and whether they ask at all
  const uint64_t *send_cnt[kPlaceLds];
  uint32_t n_keys[kPlaceLds];
};
__global__ __launch_bounds__(kBlock) void place_queries(OwnerShard *shards, int R, QueryArea area, PlaceSources src) {
  __shared__ uint32_t sm[kBlock / kWave + 1];
  __shared__ uint32_t base[kBlock];
  __shared__ uint32_t cnt[kPlaceLds * kPlaceLds];  // [requester][owner] unique keys asked for
  __shared__ uint32_t segm[kPlaceLds * kPlaceLds]; // [owner][requester] first query of the requester at the owner
  const int t = threadIdx.x;
  const bool in_lds = R <= kPlaceLds;
  if (in_lds) {
    for (int i = t; i < R * R; i += kBlock) {
      const int s = i / R, d = i % R;
      cnt[i] = src.n_keys[s] ? (uint32_t)src.send_cnt[s][d] : 0u;
    }
    __syncthreads();
  }
  auto asked = [&](int s, int d) -> uint32_t { // unique keys requester s asks owner d for
    if (in_lds) return cnt[s * R + d];
    return shards[s].n_keys ? (uint32_t)shards[s].send_cnt[d] : 0u;
  };
  uint32_t Q = 0;
  if (t < R) {
    OwnerShard &D = shards[t];
    for (int s = 0; s < R; s++) {
      D.rq_seg[s] = Q;
      if (in_lds) segm[t * R + s] = Q;
      Q += asked(s, t);
    }
    D.rq_seg[R] = Q;
    D.q = Q;
    D.query_tiles = max(1u, (Q + kBlock - 1) / kBlock); // one tile even without queries: the segment table is written
  }
  uint32_t total;
  const uint32_t lo = block_exclusive_scan<kBlock>(Q, sm, total);
  base[t] = lo;
  if (t < R) {
    OwnerShard &D = shards[t];
    D.rq_idx = area.idx + lo;
    D.rq_ver = area.ver + lo;
    D.outdated = area.outdated + lo;
    D.q_slot = area.q_slot + lo;
    D.ret_slot = area.ret_slot + lo;
  }
  __syncthreads(); // rq_seg of every owner is written (global memory, this block), base[] too
  if (t < R) {
    uint32_t ulo = 0; // unique keys of requester t that belong to the owners before d
    for (int d = 0; d < R; d++) {
      const uint32_t seg = in_lds ? segm[d * R + t] : shards[d].rq_seg[t];
      // (place in the area) - (rank among the requester's unique keys), modulo 2^32 like the sum the kernel forms
      area.query_delta[(size_t)t * R + d] = base[d] + seg - ulo;
      shards[d].got_delta[t] = ulo - seg;
      ulo += asked(t, d);
    }
  }
}

__global__ __launch_bounds__(kBlock) void decide_count(const OwnerShard *__restrict__ shards, int nseg) {
  const OwnerShard &S = shards[blockIdx.y];
  if (blockIdx.x >= S.query_tiles) return;
  const TableView &t = S.t;
  __shared__ uint32_t wcnt[kBlock / kWave];
  __shared__ uint32_t sseg[258];
  for (int i = threadIdx.x; i <= nseg; i += kBlock) sseg[i] = S.rq_seg[i];
  __syncthreads();
  // the grid is cut from a guess (the number of queries is known on the device only): a block takes every gridDim.x-th tile
  for (uint32_t tile = blockIdx.x; tile < S.query_tiles; tile += gridDim.x) {
    const uint32_t k = tile * kBlock + threadIdx.x;
    uint32_t flag = 0;
    if (k < S.q) {
      const slot_t o = owned_slot(t.slot, (uint64_t)S.rq_idx[k], t.id_max, t.n_cached);
      S.q_slot[k] = o;
      // the requester: the segment of the receive buffer the query lies in (segments may be empty)
      uint32_t lo = 0, hi = nseg - 1;
      while (lo < hi) { // the first segment that ends behind k
        const uint32_t mid = (lo + hi) / 2;
        if (sseg[mid + 1] <= k) lo = mid + 1;
        else hi = mid;
      }
      if (o == kNoSlot) {
        atomicOr(S.err, 4u);
      } else {
        const version_t local = S.rq_ver[k], global = t.ver[o];
        const bool from_self = lo == (uint32_t)t.rank;
        const bool out = local == kInvalidVersion || local + t.pull_bound < global;
        flag = (out && !from_self) ? 1u : 0u;
      }
      S.outdated[k] = flag;
      shards[lo].got[k + S.got_delta[lo]] = flag; // the requester reads it from its own array
    }
    const uint64_t m = __ballot(flag != 0);
    if (lane_id() == 0) wcnt[threadIdx.x / kWave] = __popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t c = 0;
      for (int i = 0; i < kBlock / kWave; i++) c += wcnt[i];
      S.tile_cnt[tile] = c;
    }
    __syncthreads(); // wcnt is rewritten for the next tile
  }
}

__global__ __launch_bounds__(kBlock) void scan_positions(const OwnerShard *__restrict__ shards, int nseg) {
  const OwnerShard &S = shards[blockIdx.y];
  __shared__ uint32_t sm[kBlock / kWave + 1];
  __shared__ uint32_t excl[kBlock + 1]; // position of every query of the tile among the returned rows; [kBlock]: after it
  const uint32_t q = S.q;
  for (uint32_t tile = blockIdx.x; tile < S.query_tiles; tile += gridDim.x) { // as in decide_count
    const uint32_t tile_lo = tile * kBlock, k = tile_lo + threadIdx.x;
    const uint32_t f = k < q ? S.outdated[k] : 0u;
    uint32_t s = 0;
    for (uint32_t i = threadIdx.x; i < tile; i += kBlock) s += S.tile_cnt[i];
    uint32_t before;
    block_exclusive_scan<kBlock>(s, sm, before); // flagged queries in the tiles before this one
    uint32_t total;
    const uint32_t pos = before + block_exclusive_scan<kBlock>(f, sm, total);
    if (f) S.ret_slot[pos] = S.q_slot[k]; // the rows to return, in the order they go back
    excl[threadIdx.x] = pos;
    if (threadIdx.x == 0) excl[kBlock] = before + total;
    __syncthreads();
    // the first returned row of a requester's segment is the position of the segment's first query
    const bool last_tile = tile == S.query_tiles - 1;
    for (int g = threadIdx.x; g <= nseg; g += kBlock) {
      const uint32_t start = S.rq_seg[g];
      uint32_t v = ~0u;
      if (start >= tile_lo && start < tile_lo + kBlock && start < q) v = excl[start - tile_lo];
      else if (last_tile && start >= q) v = excl[kBlock]; // segments that start at the end: the total
      if (v != ~0u) {
        S.seg_dev[g] = v;
        S.seg_host[g] = v;
      }
    }
    if (last_tile && threadIdx.x == 0) S.seg_host[257] = *S.err;
    __syncthreads(); // excl is rewritten for the next tile
  }
}

// What comes back per unique key of the step, in two roles over tiles of kRTile keys.  They need the owners' flags only, so they
// share the launches of place_returns and pack_rows, the flags and offsets being requested before the number of unique keys is
// here.  (In launches of their own behind pack_rows they took 14 us and two gaps of a step of four shards of 53 k keys.  Beside the
// owners' work remote_emit still takes what it took -- with 1.7 M keys the two launches 44 + 14 us, the one 60 -- so the gaps
// are what is gained: two steps 355 -> 337 us in one pair, 364 -> 347 in another, where runs differ by up to 10 %.)
//  count_returned  returned rows per tile, and the counts of the step: keys cached and fresh enough, not stored here, cached
//                  and refreshed; and whether an owned row came back as outdated (it never may)
//  remote_emit     ret_i[u] = index of u's row among the returned rows (exclusive scan of the flags; a tile adds up the
//                  sums of the tiles before it itself); src_row[u] = where the gather finds the row: the resident offset,
//                  or (top bit set) that index.  The last tile adds up the counts of all tiles and hands them to the host
//                  (pinned memory).
// The counts were added up by device-scope atomics of every block of remote_emit, with a fence in front of the ticket that
// named the last block.
constexpr uint32_t kReturnedRow = 0x80000000u;
constexpr int kRItems = 8, kRTile = kBlock * kRItems; // 2048 keys: the tile scan_blocks() sizes the scratch for
struct TileCounts {
  uint32_t returned, fresh, absent, refreshed; // top bit of the last: an owned row came back
};
constexpr uint32_t kOwnedCame = 0x80000000u;
// the block's totals of four counts (top bit of the fourth: or), for its first thread; sm: 5 words that read zero
__device__ __forceinline__ void block_totals(TileCounts &c, uint32_t *sm) {
  uint32_t came = c.refreshed & kOwnedCame;
  c.refreshed &= ~kOwnedCame;
  for (int d = 32; d; d >>= 1) {
    c.returned += __shfl_down(c.returned, d);
    c.fresh += __shfl_down(c.fresh, d);
    c.absent += __shfl_down(c.absent, d);
    c.refreshed += __shfl_down(c.refreshed, d);
    came |= __shfl_down(came, d);
  }
  __syncthreads(); // the zeros
  if (threadIdx.x % kWave == 0) {
    atomicAdd(&sm[0], c.returned);
    atomicAdd(&sm[1], c.fresh);
    atomicAdd(&sm[2], c.absent);
    atomicAdd(&sm[3], c.refreshed); // at most 2^31 - 1 keys
    atomicOr(&sm[4], came);
  }
  __syncthreads();
  c = TileCounts{sm[0], sm[1], sm[2], sm[3] | sm[4]};
}
__device__ __forceinline__ void count_returned(const PullShards &shards, uint32_t tile) {
  __shared__ uint32_t sm[5];
  const PullShard &S = shards.s[record_of(shards.cut, tile)];
  const uint32_t *__restrict__ got = S.a.got;
  uint32_t g[kRItems];
  slot_t o[kRItems];
#pragma unroll
  for (int k = 0; k < kRItems; k++) { // neighbouring threads count neighbouring keys; requested before U is here
    const uint32_t j = min(tile * kRTile + k * kBlock + threadIdx.x, S.b.n - 1);
    g[k] = got[j];
    o[k] = S.b.uoff[j];
  }
  const uint32_t U = *S.b.d_U; // the grid is cut for the batches' keys: the host has not seen the number of unique ones
  if (tile * kRTile >= U) return;
  if (threadIdx.x < 5) sm[threadIdx.x] = 0;
  TileCounts c = {0, 0, 0, 0};
  uint32_t came = 0;
#pragma unroll
  for (int k = 0; k < kRItems; k++) {
    if (tile * kRTile + k * kBlock + threadIdx.x >= U) continue;
    c.returned += g[k];
    if (o[k] == kNoSlot) c.absent++;
    else if ((uint32_t)o[k] >= S.t.n_cached) came |= g[k] ? kOwnedCame : 0u;
    else if (g[k]) c.refreshed++;
    else c.fresh++;
  }
  c.refreshed |= came;
  block_totals(c, sm);
  if (threadIdx.x == 0) ((TileCounts *)S.tile_counts)[tile] = c;
}
__device__ __forceinline__ void remote_emit(const PullShards &shards, uint32_t tile) {
  __shared__ uint32_t sm[kBlock / kWave + 1], tot[5];
  const PullShard &S = shards.s[record_of(shards.cut, tile)];
  const BatchView &c = S.b;
  const uint32_t *__restrict__ got = S.a.got;
  const TileCounts *__restrict__ counts = (const TileCounts *)S.tile_counts;
  uint32_t *__restrict__ ret_i = S.a.ret_i, *__restrict__ src_row = S.a.src_row;
  const uint32_t j0 = tile * kRTile + threadIdx.x * kRItems;
  uint32_t g[kRItems], mine = 0;
  slot_t o[kRItems];
#pragma unroll
  for (int k = 0; k < kRItems; k++) { // requested before U is here
    g[k] = got[min(j0 + k, c.n - 1)];
    o[k] = c.uoff[min(j0 + k, c.n - 1)];
  }
  uint32_t s = 0;
  for (uint32_t i = threadIdx.x; i < tile; i += kBlock) s += counts[i].returned; // (past the last tile: not used)
  const uint32_t U = *c.d_U;
  const uint32_t tiles = (U + kRTile - 1) / kRTile; // of the grid's blocks (cut for the batch's keys) these have work
  if (tile >= tiles) return;
  uint32_t prefix;
  block_exclusive_scan<kBlock>(s, sm, prefix); // its total: returned rows in the tiles before this one
#pragma unroll
  for (int k = 0; k < kRItems; k++) mine += j0 + k < U ? g[k] : 0u;
  uint32_t total;
  uint32_t run = prefix + block_exclusive_scan<kBlock>(mine, sm, total);
#pragma unroll
  for (int k = 0; k < kRItems; k++) {
    if (j0 + k < U) {
      ret_i[j0 + k] = run;
      src_row[j0 + k] = o[k] == kNoSlot ? (kReturnedRow | run) : (uint32_t)o[k];
    }
    run += g[k];
  }
  if (tile == tiles - 1) {
    if (threadIdx.x < 5) tot[threadIdx.x] = 0;
    TileCounts sum = {0, 0, 0, 0};
    for (uint32_t i = threadIdx.x; i < tiles; i += kBlock) {
      const TileCounts n = counts[i];
      sum.fresh += n.fresh, sum.absent += n.absent;
      sum.refreshed = (sum.refreshed + (n.refreshed & ~kOwnedCame)) | (n.refreshed & kOwnedCame);
    }
    block_totals(sum, tot);
    if (threadIdx.x == 0) {
      S.host_stats[0] = sum.fresh;
      S.host_stats[1] = sum.absent;
      S.host_stats[2] = sum.refreshed & ~kOwnedCame;
      S.host_stats[3] = sum.refreshed & kOwnedCame ? 8u : 0u;
    }
  }
}

// Where the rows an owner returns stand in the requesters' buffers: a requester's rows arrive in owner order
// (csrc/core/all2all.cu:89-130), and how many rows an owner returns to a requester is only known on the device.
// Thread (owner d, requester s): ret_delta of d for s = rows the owners before d return to s, minus the start of s'
// segment in d's own return order.
// place_blocks of the launch's blocks do this, the others count_returned.
__global__ __launch_bounds__(kBlock) void place_returns(const OwnerShard *__restrict__ shards, int nrank, PullShards pulls, uint32_t place_blocks) {
  if (blockIdx.x >= place_blocks) {
    count_returned(pulls, blockIdx.x - place_blocks);
    return;
  }
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (uint32_t)nrank * nrank) return;
  const int d = i / nrank, s = i % nrank;
  uint32_t before = 0;
  for (int e = 0; e < d; e++) before += shards[e].seg_dev[s + 1] - shards[e].seg_dev[s];
  shards[d].ret_delta[s] = before - shards[d].seg_dev[s];
}

// kPackAhead rows to return per group of LPR lanes (two, four of many rows); which rows, scan_positions has listed.  A row goes straight into
// the buffers of the shard that asked for it (in one process a plain device address, between GPUs peer memory).
// Four where that leaves kPackBlocks blocks at least: what a block does before its first row -- two tables, a barrier, the list --
// is then shared by more rows (rows of 128 floats, 16 k for each of seven owners: 58.6 -> 47.7 us); a small launch is as long as its
// longest block (rows of 32 floats, four owners of 5 k: 8.2 us with two, 10.4 with four).  Two and four on either side of the line:
// four owners that all ask, 106 k keys of 64 floats each 36.2 and 31.6, eight, 53 k of 128 68.6 and 62.5 (four is taken); one of four asking,
// 426 k of 128, 18.1 and 15.9, both of two, 426 k of 32, 35.7 and 24.2 (two is): in the middle the line could be lower.
constexpr uint32_t kPackBlocks = 4096;
// The launch has a row of blocks per owner, the first pack_blocks of which do this; the rows behind them do remote_emit.
template <int VEC, int LPR, int kPackAhead>
__global__ __launch_bounds__(kBlock) void pack_rows(const OwnerShard *__restrict__ shards, int nseg, PullShards pulls, uint32_t pack_blocks) {
  if (blockIdx.y >= (uint32_t)nseg) {
    const uint32_t block = (blockIdx.y - nseg) * gridDim.x + blockIdx.x;
    if (block < pulls.cut.total) remote_emit(pulls, block);
    return;
  }
  if (blockIdx.x >= pack_blocks) return;
  typedef typename RowVec<VEC>::T V;
  constexpr int kGroups = kBlock / LPR;
  __shared__ uint32_t sseg[258], sdelta[257];
  const OwnerShard &S = shards[blockIdx.y];
  for (int i = threadIdx.x; i <= nseg; i += kBlock) sseg[i] = S.seg_dev[i];
  for (int i = threadIdx.x; i < nseg; i += kBlock) sdelta[i] = S.ret_delta[i];
  __syncthreads();
  const uint32_t total = sseg[nseg]; // rows this shard returns: known on the device only, the grid is cut for the most
  const embed_t *__restrict__ emb = S.t.emb;
  const uint32_t gl = threadIdx.x % LPR, W = S.t.width;
  for (uint32_t k0 = blockIdx.x * (kGroups * kPackAhead) + threadIdx.x / LPR; k0 < total; k0 += pack_blocks * (kGroups * kPackAhead)) {
  slot_t o[kPackAhead];
#pragma unroll
  for (int a = 0; a < kPackAhead; a++) o[a] = k0 + a * kGroups < total ? S.ret_slot[k0 + a * kGroups] : kNoSlot;
  // the requester of every row: the segment of the return order it lies in (segments may be empty)
  embed_t *dst_val[kPackAhead];
  version_t *dst_ver[kPackAhead];
#pragma unroll
  for (int a = 0; a < kPackAhead; a++) {
    const uint32_t k = min(k0 + a * kGroups, total - 1);
    uint32_t lo = 0, hi = nseg - 1;
    while (lo < hi) { // the first segment that ends behind k
      const uint32_t mid = (lo + hi) / 2;
      if (sseg[mid + 1] <= k) lo = mid + 1;
      else hi = mid;
    }
    const uint32_t row = k + sdelta[lo];
    dst_val[a] = shards[lo].in_val + (size_t)row * W;
    dst_ver[a] = shards[lo].in_ver + row;
  }
  if (gl == 0) {
#pragma unroll
    for (int a = 0; a < kPackAhead; a++)
      if (o[a] != kNoSlot) *dst_ver[a] = S.t.ver[o[a]];
  }
  for (uint32_t c = gl * kCols<VEC>; c < W; c += LPR * kCols<VEC>) {
    const uint32_t col = lane_col<VEC>(c, W);
    V v[kPackAhead];
#pragma unroll
    for (int a = 0; a < kPackAhead; a++)
      if (o[a] != kNoSlot) v[a] = *(const V *)(emb + (size_t)o[a] * W + col);
#pragma unroll
    for (int a = 0; a < kPackAhead; a++)
      if (o[a] != kNoSlot) __builtin_nontemporal_store(v[a], (V *)(dst_val[a] + col)); // read next by another shard's kernels
  }
  }
}


// The cached rows that came back, in one of three ways.  What bounds them: a chain of three loads (flags, where the row came
// back, the row), and where many rows came back the memory.
//  * A group of LPR lanes per unique key, up to kRefreshEachBlocks blocks of those: they run at once, and nothing is as short.
//  * A wave looks at the flags of `flags` unique keys, one per lane, lists those that have something to do and copies their rows, a
//    group per row, kRefreshAhead rows on their way at a time: at as many keys as its groups copy in one go, where most
//    rows come back (in the step before they did) or ...
//  * ... at kWave keys, where few do and that makes kRefreshSparseBlocks blocks at least: most of the work is then to look.
// us on an MI355X, four shards, by unique keys of each shard; none / three quarters of them came back into a cached row:
//     rows of 32 floats       first way      second        third       | of 128: first       second          third
//     3.7 k / 2.3 k           2.4 /  4.5     2.8 /  5.3    2.8 /  6.8  |    3.8 /   5.7     2.3 /   6.6    2.7 /  14.1
//      25 k / 15.5 k          3.2 /  7.3     2.5 /  7.2    2.5 /  8.6  |    7.6 /  17.3     3.9 /  15.5    4.2 /  22.3
//     125 k / 78 k            9.1 / 21.5     4.9 / 19.1    4.3 / 21.6  |   28.2 /  73.9    12.2 /  65.6    4.6 /  76.7
//     500 k / 310 k          28.4 / 80.1    13.5 / 71.4    9.0 / 73.5  |  103.7 / 295.4    39.4 / 278.4    9.3 / 289.1
// Half of them: the second way 41.0, the third 44.0 (78 k, 128 floats), 45.0 and 44.5 (310 k, 32 floats); a quarter: 30.7 and 28.2,
// 33.6 and 28.8.  A group per key that goes on to the next key, four in a row, took 16.5 / 70.6 us (78 k, 128 floats)
// and 55.3 / 274.8 (310 k).
constexpr uint32_t kRefreshAhead = 4;
constexpr uint64_t kRefreshEachBlocks = 1536, kRefreshSparseBlocks = 512;
template <int VEC, int LPR>
__global__ __launch_bounds__(kBlock) void refresh_each(PullShards shards) {
  typedef typename RowVec<VEC>::T V;
  uint32_t block, blocks;
  const PullShard &S = my_record(shards, block, blocks);
  const TableView &t = S.t;
  const BatchView &b = S.b;
  const PullArgs &a = S.a;
  constexpr uint32_t kGroups = kBlock / LPR;
  const uint32_t U = *b.d_U, gl = threadIdx.x % LPR, W = t.width;
  for (uint32_t u = block * kGroups + threadIdx.x / LPR; u < U; u += blocks * kGroups) {
    const slot_t o = b.uoff[u];
    const bool got = a.got[u] != 0;
    if (!got || o == kNoSlot || (uint32_t)o >= t.n_cached) continue; // (an owned row that came back is reported by remote_emit)
    const uint32_t k = a.ret_i[u];
    if (gl == 0) t.ver[o] = a.in_ver[k];
    for (uint32_t c = gl * kCols<VEC>; c < W; c += LPR * kCols<VEC>) {
      const uint32_t col = lane_col<VEC>(c, W);
      *(V *)(t.emb + (size_t)o * W + col) =
          *(const V *)(a.in_val + (size_t)k * W + col) + *(const V *)(t.pend + (size_t)o * W + col);
    }
  }
}

template <int VEC, int LPR>
__global__ __launch_bounds__(kBlock) void refresh(PullShards shards, uint32_t flags) {
  typedef typename RowVec<VEC>::T V;
  __shared__ uint2 todo[kBlock]; // {resident offset, returned row}, kWave of every wave
  uint32_t block, blocks;
  const PullShard &S = my_record(shards, block, blocks);
  const TableView &t = S.t;
  const BatchView &b = S.b;
  const PullArgs &a = S.a;
  constexpr uint32_t kGroups = kWave / LPR; // of a wave
  const uint32_t U = *b.d_U, lane = threadIdx.x % kWave, gl = lane % LPR, W = t.width;
  uint2 *const mine = todo + threadIdx.x / kWave * kWave;
  for (uint32_t u0 = (block * kBlock + threadIdx.x) / kWave * flags; u0 < U; u0 += blocks * (kBlock / kWave) * flags) {
    const uint32_t u = u0 + lane, at = min(u, U - 1);
    const slot_t o = b.uoff[at];
    const bool work = lane < flags && u < U && a.got[at] != 0 && o != kNoSlot && (uint32_t)o < t.n_cached; // (an owned row that came back is reported by remote_emit)
    const uint64_t all = __ballot(work);
    if (!all) continue;
    if (work) {
      const uint32_t k = a.ret_i[u];
      t.ver[o] = a.in_ver[k];
      mine[__popcll(all & (((uint64_t)1 << lane) - 1))] = make_uint2((uint32_t)o, k);
    }
    // a wave's LDS operations are done in its own order; the fences keep the compiler from moving them
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t rows = __popcll(all);
    for (uint32_t r = lane / LPR; r < rows; r += kGroups * kRefreshAhead) {
      uint2 w[kRefreshAhead];
#pragma unroll
      for (uint32_t k = 0; k < kRefreshAhead; k++) w[k] = mine[min(r + k * kGroups, rows - 1)];
      for (uint32_t c = gl * kCols<VEC>; c < W; c += LPR * kCols<VEC>) {
        const uint32_t col = lane_col<VEC>(c, W);
        V in[kRefreshAhead], pend[kRefreshAhead];
#pragma unroll
        for (uint32_t k = 0; k < kRefreshAhead; k++) {
          in[k] = *(const V *)(a.in_val + (size_t)w[k].y * W + col);
          pend[k] = *(const V *)(t.pend + (size_t)w[k].x * W + col);
        }
#pragma unroll
        for (uint32_t k = 0; k < kRefreshAhead; k++)
          if (r + k * kGroups < rows) *(V *)(t.emb + (size_t)w[k].x * W + col) = in[k] + pend[k];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier(); // the list is written again for the next keys
  }
}

// Gather in SORTED order: one group per kRows consecutive sorted positions.  Duplicates of a key are adjacent,
// so a table row is fetched from HBM once and re-read from cache for its other occurrences; every output row is
// written whole, once, with non-temporal stores, at the batch position sorted_arg names.
#ifndef HCTR_GATHER_ROWS
#define HCTR_GATHER_ROWS 8
#endif
constexpr int kRows = HCTR_GATHER_ROWS;
// kStream: dst is written with nontemporal stores (a compile-time choice: merged into one store by the compiler, a
// run-time one loses the hint)
template <int VEC, int LPR, bool kLocalOnly, bool kStream>
__device__ __forceinline__ void gather_rows(const TableView &t, const BatchView &b, const PullArgs &a, uint32_t block,
                                            uint32_t blocks) {
  typedef typename RowVec<VEC>::T V;
  constexpr int kGroups = kBlock / LPR;
  const uint32_t n = b.n, W = t.width;
  if (block < a.list_chunks) { // the batch's run lists for its push one step later, before the block's own rows
    __shared__ uint32_t cnt[kRunLists], base[kRunLists];
    for (uint32_t chunk = block; chunk < a.list_chunks; chunk += blocks) list_runs_chunk(b, chunk, cnt, base);
  }
  const uint32_t j0 = (block * kGroups + threadIdx.x / LPR) * kRows;
  if (j0 >= n) return;
  const uint32_t gl = threadIdx.x % LPR;
  const embed_t *src[kRows];
  embed_t *dst[kRows];
#pragma unroll
  for (int k = 0; k < kRows; k++) {
    const uint32_t j = min(j0 + k, n - 1);
    const uint32_t u = b.rank_sorted[j];
    const uint32_t i = b.sorted_arg[j];
    if (kLocalOnly) {
      src[k] = t.emb + (size_t)b.uoff[u] * W;
    } else {
      const uint32_t r = a.src_row[u];
      src[k] = (r & kReturnedRow) ? a.in_val + (size_t)(r & ~kReturnedRow) * W : t.emb + (size_t)r * W;
    }
    dst[k] = a.dst + (size_t)i * W;
  }
  for (uint32_t c = gl * kCols<VEC>; c < W; c += LPR * kCols<VEC>) {
    const uint32_t col = lane_col<VEC>(c, W);
    V v[kRows];
#pragma unroll
    for (int k = 0; k < kRows; k++) v[k] = *(const V *)(src[k] + col);
#pragma unroll
    for (int k = 0; k < kRows; k++)
      if (j0 + k < n) {
        if (kStream) __builtin_nontemporal_store(v[k], (V *)(dst[k] + col));
        else *(V *)(dst[k] + col) = v[k];
      }
  }
}

template <int VEC, int LPR, bool kStream>
__global__ __launch_bounds__(kBlock) void gather(TableView t, BatchView b, PullArgs a) {
  gather_rows<VEC, LPR, true, kStream>(t, b, a, blockIdx.x, gridDim.x);
}
template <int VEC, int LPR, bool kStream>
__global__ __launch_bounds__(kBlock) void gather_group(PullShards shards) {
  uint32_t block, blocks;
  const PullShard &S = my_record(shards, block, blocks);
  gather_rows<VEC, LPR, false, kStream>(S.t, S.b, S.a, block, blocks);
}

// Gather in BATCH order straight from the batch's keys, for one shard: dst[i] = emb[slot[id of position i]].  It needs
// nothing of the batch's index (sort, unique pass), so a step whose index is longer than its push -- a small batch --
// does not wait for it; what it gives up is the order in which the duplicates of a key are adjacent, which only matters
// once the rows of a batch no longer fit the caches.
template <int VEC, int LPR, typename K, bool kStream>
__global__ __launch_bounds__(kBlock) void gather_direct(TableView t, const K *__restrict__ keys, int id_bits, uint32_t n,
                                                        embed_t *__restrict__ dst_rows) {
  typedef typename RowVec<VEC>::T V;
  constexpr int kGroups = kBlock / LPR;
  const uint32_t W = t.width;
  const uint32_t i0 = (blockIdx.x * kGroups + threadIdx.x / LPR) * kRows;
  if (i0 >= n) return;
  const uint32_t gl = threadIdx.x % LPR;
  const K id_mask = (K)(((uint64_t)1 << id_bits) - 1);
  const embed_t *src[kRows];
#pragma unroll
  for (int k = 0; k < kRows; k++) {
    const uint32_t i = min(i0 + k, n - 1);
    src[k] = t.emb + (size_t)t.slot[(uint64_t)(keys[i] & id_mask)] * W; // one shard: every id is resident
  }
  for (uint32_t c = gl * kCols<VEC>; c < W; c += LPR * kCols<VEC>) {
    const uint32_t col = lane_col<VEC>(c, W);
    V v[kRows];
#pragma unroll
    for (int k = 0; k < kRows; k++) v[k] = *(const V *)(src[k] + col);
#pragma unroll
    for (int k = 0; k < kRows; k++)
      if (i0 + k < n) {
        V *d = (V *)(dst_rows + (size_t)(i0 + k) * W + col);
        if (kStream) __builtin_nontemporal_store(v[k], d);
        else *d = v[k];
      }
  }
}

// Sum-pooled lookups: one group of LPR lanes per bag of `bag` consecutive batch positions.  The rows of the bag are requested
// kPoolAhead at a time and added in position order (fp32, starting from the first row), so a bag costs one output
// row instead of `bag`.
// Where the rows lie, the lanes of the group find out together, a position each (row_of), and hand each other: looked up by every
// lane for itself, bags of ten took 40 load instructions of which ten fetched something new, and rows past the end of a bag were
// read again to fill the last round.  852 k bags of ten rows of 64 floats, Zipf 1.4: 217 -> 152 us, 14 TB/s out of the caches; 12
// rows ahead 160, 16 rows 174 (fewer waves fit).
constexpr int kPoolAhead = 8;
template <int VEC, int LPR, typename RowOf, typename RowAt>
__device__ __forceinline__ void pool_bag(uint32_t W, uint32_t i0, uint32_t bag, embed_t *__restrict__ dst, RowOf &&row_of, RowAt &&row_at) {
  typedef typename RowVec<VEC>::T V;
  constexpr int kPer = LPR < kPoolAhead ? kPoolAhead / LPR : 1, kFound = LPR * kPer; // positions per lane, of the group
  const uint32_t gl = threadIdx.x % LPR;
  for (uint32_t c0 = 0; c0 < W; c0 += LPR * kCols<VEC>) {
    const uint32_t due = c0 + gl * kCols<VEC>;
    const bool active = due < W;
    const uint32_t col = active ? lane_col<VEC>(due, W) : 0u; // a lane behind the row reads its first columns, and finds rows
    V acc;
    for (uint32_t h0 = 0; h0 < bag; h0 += kFound) {
      uint32_t row[kPer];
#pragma unroll
      for (int j = 0; j < kPer; j++) row[j] = row_of(i0 + min(h0 + j * LPR + gl, bag - 1));
// Not unrolled: that took 82 registers with 32 lanes, 116 with 64, and half the waves fitted (213 k bags of eight rows of 160 floats
// 139 us, as a loop 98; of 128 floats 73 and 66).
#pragma unroll 1
      for (int r = 0; r < kFound; r += kPoolAhead) { // once, where a lane has several positions
        const uint32_t h = h0 + r;
        if (h >= bag) break;
        const uint32_t n = min(bag - h, (uint32_t)kPoolAhead);
        V v[kPoolAhead];
        auto fetch = [&](int k) { v[k] = *(const V *)(row_at((uint32_t)__shfl((int)row[k / LPR], kPer > 1 ? k % LPR : r + k, LPR)) + col); };
        if (n == kPoolAhead) {
#pragma unroll
          for (int k = 0; k < kPoolAhead; k++) fetch(k);
        } else {
#pragma unroll
          for (int k = 0; k < kPoolAhead - 1; k++)
            if ((uint32_t)k < n) fetch(k);
        }
        if (h == 0) acc = v[0];
        else acc = acc + v[0];
#pragma unroll
        for (int k = 1; k < kPoolAhead; k++)
          if ((uint32_t)k < n) acc = acc + v[k];
      }
    }
    if (active) __builtin_nontemporal_store(acc, (V *)(dst + col));
  }
}

// In batch order, through the inverse index of the batch.
template <int VEC, int LPR, bool kLocalOnly>
__global__ __launch_bounds__(kBlock) void gather_pooled(TableView t, BatchView batch, PullArgs a, uint32_t bag,
                                                        uint32_t n_bags) {
  constexpr int kGroups = kBlock / LPR;
  if (blockIdx.x < a.list_chunks) { // the batch's run lists, as in gather
    __shared__ uint32_t cnt[kRunLists], base[kRunLists];
    for (uint32_t chunk = blockIdx.x; chunk < a.list_chunks; chunk += gridDim.x) list_runs_chunk(batch, chunk, cnt, base);
  }
  const uint32_t b = blockIdx.x * kGroups + threadIdx.x / LPR;
  if (b >= n_bags) return;
  const uint32_t W = t.width;
  pool_bag<VEC, LPR>(W, b * bag, bag, a.dst + (size_t)b * W,
                     [&](uint32_t i) -> uint32_t { return kLocalOnly ? (uint32_t)batch.uoff[batch.idx_map[i]] : a.src_row[batch.idx_map[i]]; },
                     [&](uint32_t r) -> const embed_t * {
                       if (kLocalOnly) return t.emb + (size_t)r * W;
                       return (r & kReturnedRow) ? a.in_val + (size_t)(r & ~kReturnedRow) * W : t.emb + (size_t)r * W;
                     });
}

// The same for one shard from the batch's keys in batch order (as gather_direct): a bag's positions are consecutive in
// the batch, so this order costs no locality the other would have, and nothing of the batch's index is needed.
template <int VEC, int LPR, typename K>
__global__ __launch_bounds__(kBlock) void gather_pooled_direct(TableView t, const K *__restrict__ keys, int id_bits,
                                                               embed_t *__restrict__ dst_rows, uint32_t bag, uint32_t n_bags) {
  constexpr int kGroups = kBlock / LPR;
  const uint32_t b = blockIdx.x * kGroups + threadIdx.x / LPR;
  if (b >= n_bags) return;
  const uint32_t W = t.width;
  const K id_mask = (K)(((uint64_t)1 << id_bits) - 1);
  pool_bag<VEC, LPR>(W, b * bag, bag, dst_rows + (size_t)b * W,
                     [&](uint32_t i) -> uint32_t { return (uint32_t)t.slot[(uint64_t)(keys[i] & id_mask)]; },
                     [&](uint32_t r) -> const embed_t * { return t.emb + (size_t)r * W; });
}

// plain 16-byte-lane copy of known size: the yardstick the HBM byte counters are scaled with
__global__ __launch_bounds__(kBlock) void plain_copy(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t n16) {
  const size_t stride = (size_t)gridDim.x * kBlock;
  for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n16; i += stride) dst[i] = src[i];
}

inline int lanes_for(uint32_t width, int vec) {
  const uint32_t per = vec == 1 ? 1 : 4, lanes = (width + per - 1) / per;
  return lanes <= 4 ? 4 : lanes <= 8 ? 8 : lanes <= 16 ? 16 : lanes <= 32 ? 32 : 64;
}

// expands F<VEC, LPR>(args...) over the (VEC, LPR) pairs; rows that move one float per lane have less than four
#define HCTR_DISPATCH_ROW(vec, lpr, CALL)         \
  do {                                            \
    if ((vec) == 4) HCTR_DISPATCH_LPR(4, lpr, CALL); \
    else if ((vec) == kOdd4) HCTR_DISPATCH_LPR(kOdd4, lpr, CALL); \
    else CALL(1, 4);                              \
  } while (0)
#define HCTR_DISPATCH_LPR(V, lpr, CALL) \
  do {                                  \
    switch (lpr) {                      \
      case 4: CALL(V, 4); break;        \
      case 8: CALL(V, 8); break;        \
      case 16: CALL(V, 16); break;      \
      case 32: CALL(V, 32); break;      \
      default: CALL(V, 64); break;      \
    }                                   \
  } while (0)

} // namespace

template <typename Blocks, typename F> static void for_shards(const PullShard *shards, int count, Blocks &&blocks, F &&f) {
  launch_records<PullShard, kShardsPerLaunch>(count, kBlock, [&](int k) { return shards[k]; }, [&](int k) { return blocks(shards[k]); }, f);
}

void launch_build_queries(hipStream_t s, const KeyLayout &kl, const PullShard *shards, int count) {
  // grids for the batches' keys: the kernel reads the numbers of unique ones itself
  for_shards(shards, count, [](const PullShard &o) { return div_up(o.b.n, kBlock); }, [&](const PullShards &p, int) {
    const dim3 grid = grid_of(p);
    if (kl.wide) hipLaunchKernelGGL(build_queries<uint64_t>, grid, dim3(kBlock), 0, s, p, kl.id_bits);
    else hipLaunchKernelGGL(build_queries<uint32_t>, grid, dim3(kBlock), 0, s, p, kl.id_bits);
    HCTR_HIP(hipGetLastError());
  });
}

size_t query_tiles(uint32_t q) { return std::max<size_t>(1, div_up(q, kBlock)); }

uint32_t owner_push_rows_per_block(uint32_t width) {
  const int lpr = lanes_for(width, row_vec(width, nullptr));
  return kApplyBatches * kApplyAhead * (kBlock / lpr);
}

void launch_place_queries(hipStream_t s, OwnerShard *shards_dev, const OwnerShard *shards_host, int nsrc,
                          const QueryArea &area) {
  HCTR_CHECK(nsrc <= kBlock, "internal: more shards than the placing block has threads");
  PlaceSources src;
  for (int i = 0; i < kPlaceLds; i++) {
    src.send_cnt[i] = i < nsrc ? shards_host[i].send_cnt : nullptr;
    src.n_keys[i] = i < nsrc ? shards_host[i].n_keys : 0;
  }
  hipLaunchKernelGGL(place_queries, dim3(1), dim3(kBlock), 0, s, shards_dev, nsrc, area, src);
  HCTR_HIP(hipGetLastError());
}

// Grids of kernels whose work is known on the device only are cut from a guess (what the step before had, and some)
// and never beyond the most there can be; the kernels stride over what there is.
static uint32_t guessed_blocks(uint32_t guess, uint32_t most, uint32_t per_block) {
  const uint64_t g = (uint64_t)guess + guess / 4 + 4 * per_block;
  return std::max(1u, div_up(std::min<uint64_t>(g, most), per_block));
}

void launch_apply_pushes(hipStream_t s, const OwnerShard *shards_dev, int nshards, int nsrc, uint32_t width, uint32_t push_blocks) {
  if (!push_blocks) return;
  const int vec = row_vec(width, nullptr);
  const int lpr = lanes_for(width, vec);
  const uint32_t rpb = owner_push_rows_per_block(width);
#define CALL(V, L) \
  hipLaunchKernelGGL((apply_remote_all<V, L>), dim3(push_blocks, nshards), dim3(kBlock), 0, s, shards_dev, nsrc, rpb)
  HCTR_DISPATCH_ROW(vec, lpr, CALL);
#undef CALL
  HCTR_HIP(hipGetLastError());
}

void launch_owner_side(hipStream_t s, const OwnerShard *shards_dev, int nshards, int nsrc, uint32_t width, uint32_t queries_max,
                       uint32_t queries_guess, const PullShard *pulls, int npulls) {
  const uint32_t tiles = guessed_blocks(queries_guess, queries_max, kBlock);
  const int vec = row_vec(width, nullptr);
  const int lpr = lanes_for(width, vec);
  hipLaunchKernelGGL(decide_count, dim3(tiles, nshards), dim3(kBlock), 0, s, shards_dev, nsrc);
  hipLaunchKernelGGL(scan_positions, dim3(tiles, nshards), dim3(kBlock), 0, s, shards_dev, nsrc);
  // the launches of several groups of requesters, the first of them with the owners' work
  auto with_requesters = [&](bool owners, auto &&launch) {
    // for the batches' keys; the kernels read how many are unique
    for_shards(pulls, npulls, [](const PullShard &o) { return div_up(o.b.n, kRTile); }, [&](const PullShards &p, int) {
      launch(p, owners);
      owners = false;
    });
    if (owners) launch(PullShards{}, true); // nobody asked
  };
  with_requesters(queries_max != 0, [&](const PullShards &p, bool owners) {
    const uint32_t place_blocks = owners ? div_up((uint32_t)(nsrc * nsrc), kBlock) : 0u;
    hipLaunchKernelGGL(place_returns, dim3(place_blocks + p.cut.total), dim3(kBlock), 0, s, shards_dev, nsrc, p, place_blocks);
  });
  with_requesters(queries_max != 0, [&](const PullShards &p, bool owners) {
    auto blocks = [&](int ahead) { return owners ? guessed_blocks(queries_guess, queries_max, ahead * (kBlock / lpr)) : 0u; };
    const bool four = (uint64_t)blocks(4) * nshards >= kPackBlocks;
    const uint32_t pack = blocks(four ? 4 : 2);
    const uint32_t across = std::max(pack, 64u); // few rows to pack: few idle blocks, and few rows of requesters
    const dim3 grid(across, nshards + div_up(p.cut.total, across));
#define CALL(V, L)                                                                                             \
  do {                                                                                                         \
    if (four) hipLaunchKernelGGL((pack_rows<V, L, 4>), grid, dim3(kBlock), 0, s, shards_dev, nsrc, p, pack);    \
    else hipLaunchKernelGGL((pack_rows<V, L, 2>), grid, dim3(kBlock), 0, s, shards_dev, nsrc, p, pack);         \
  } while (0)
    HCTR_DISPATCH_ROW(vec, lpr, CALL);
#undef CALL
  });
  HCTR_HIP(hipGetLastError());
}

void launch_refresh(hipStream_t s, const PullShard *shards, int count) {
  if (!count) return;
  const uint32_t width = shards[0].t.width;
  const int vec = row_vec(width, nullptr), lpr = lanes_for(width, vec);
  auto blocks_of = [&](const PullShard &o, uint32_t keys) { return guessed_blocks(o.unique_guess, o.b.n, keys); }; // keys per block
  uint64_t unique = 0, refreshed = 0, each_blocks = 0, sparse_blocks = 0;
  for (int k = 0; k < count; k++) {
    unique += shards[k].unique_guess;
    refreshed += shards[k].refreshed_guess;
    each_blocks += blocks_of(shards[k], kBlock / lpr);
    sparse_blocks += blocks_of(shards[k], kBlock);
  }
  const bool each = each_blocks <= kRefreshEachBlocks;
  const bool sparse = 2 * refreshed < unique && sparse_blocks >= kRefreshSparseBlocks;
  const uint32_t flags = sparse ? kWave : std::min<uint32_t>(kWave, kRefreshAhead * (kWave / lpr));
  auto blocks = [&](const PullShard &o) { return blocks_of(o, each ? kBlock / lpr : kBlock / kWave * flags); };
  for_shards(shards, count, blocks, [&](const PullShards &p, int) {
#define CALL(V, L)                                                                            \
  do {                                                                                        \
    if (each) hipLaunchKernelGGL((refresh_each<V, L>), grid_of(p), dim3(kBlock), 0, s, p);    \
    else hipLaunchKernelGGL((refresh<V, L>), grid_of(p), dim3(kBlock), 0, s, p, flags);       \
  } while (0)
    HCTR_DISPATCH_ROW(vec, lpr, CALL);
#undef CALL
    HCTR_HIP(hipGetLastError());
  });
}

void launch_gather_group(hipStream_t s, const PullShard *shards, int count) {
  if (!count) return;
  const uint32_t width = shards[0].t.width;
  const uint32_t rows = kRows * (kBlock / lanes_for(width, row_vec(width, nullptr))); // of a block, whatever its vectors
  for_shards(shards, count, [&](const PullShard &o) { return div_up(o.b.n, rows); }, [&](const PullShards &p, int m) {
    int vec = 4;
    bool stream = true;
    for (int k = 0; k < m; k++) { // one kernel for all: vectors that suit every output, the common kind of stores
      if (row_vec(width, p.s[k].a.dst) != 4) vec = row_vec(width, p.s[k].a.dst);
      stream = stream && p.s[k].a.stream_stores;
    }
    const int lpr = lanes_for(width, vec);
#define CALL(V, L)                                                                                             \
  do {                                                                                                         \
    if (stream) hipLaunchKernelGGL((gather_group<V, L, true>), grid_of(p), dim3(kBlock), 0, s, p);    \
    else hipLaunchKernelGGL((gather_group<V, L, false>), grid_of(p), dim3(kBlock), 0, s, p);          \
  } while (0)
    HCTR_DISPATCH_ROW(vec, lpr, CALL);
#undef CALL
    HCTR_HIP(hipGetLastError());
  });
}

void launch_gather(hipStream_t s, const TableView &t, const BatchView &cur, const PullArgs &a) {
  if (!cur.n) return;
  HCTR_CHECK(t.nrank == 1, "internal: the gather of local rows is for one shard");
  const int vec = row_vec(t.width, a.dst);
  const int lpr = lanes_for(t.width, vec);
#define CALL(V, L)                                                                                               \
  do {                                                                                                           \
    const unsigned blocks = div_up(div_up(cur.n, kRows), kBlock / L);                                            \
    if (a.stream_stores) hipLaunchKernelGGL((gather<V, L, true>), dim3(blocks), dim3(kBlock), 0, s, t, cur, a);  \
    else hipLaunchKernelGGL((gather<V, L, false>), dim3(blocks), dim3(kBlock), 0, s, t, cur, a);                 \
  } while (0)
  HCTR_DISPATCH_ROW(vec, lpr, CALL);
#undef CALL
  HCTR_HIP(hipGetLastError());
}

void launch_gather_direct(hipStream_t s, const TableView &t, const KeyLayout &kl, const void *keys, uint32_t n, embed_t *dst,
                          bool stream_stores) {
  if (!n) return;
  HCTR_CHECK(t.nrank == 1, "internal: the gather from the keys is for one shard");
  const int vec = row_vec(t.width, dst);
  const int lpr = lanes_for(t.width, vec);
#define CALL(V, L)                                                                                                    \
  do {                                                                                                                \
    const unsigned blocks = div_up(n, (kBlock / L) * kRows);                                                          \
    if (kl.wide && stream_stores) hipLaunchKernelGGL((gather_direct<V, L, uint64_t, true>), dim3(blocks), dim3(kBlock), 0, s, t, (const uint64_t *)keys, kl.id_bits, n, dst); \
    else if (kl.wide) hipLaunchKernelGGL((gather_direct<V, L, uint64_t, false>), dim3(blocks), dim3(kBlock), 0, s, t, (const uint64_t *)keys, kl.id_bits, n, dst); \
    else if (stream_stores) hipLaunchKernelGGL((gather_direct<V, L, uint32_t, true>), dim3(blocks), dim3(kBlock), 0, s, t, (const uint32_t *)keys, kl.id_bits, n, dst); \
    else hipLaunchKernelGGL((gather_direct<V, L, uint32_t, false>), dim3(blocks), dim3(kBlock), 0, s, t, (const uint32_t *)keys, kl.id_bits, n, dst); \
  } while (0)
  HCTR_DISPATCH_ROW(vec, lpr, CALL);
#undef CALL
  HCTR_HIP(hipGetLastError());
}

void launch_gather_pooled_direct(hipStream_t s, const TableView &t, const KeyLayout &kl, const void *keys, uint32_t n,
                                 embed_t *dst, uint32_t bag) {
  if (!n) return;
  HCTR_CHECK(t.nrank == 1, "internal: the gather from the keys is for one shard");
  const uint32_t n_bags = n / bag;
  const int vec = row_vec(t.width, dst);
  const int lpr = lanes_for(t.width, vec);
#define CALL(V, L)                                                                                                    \
  do {                                                                                                                \
    const unsigned blocks = div_up(n_bags, kBlock / L);                                                               \
    if (kl.wide) hipLaunchKernelGGL((gather_pooled_direct<V, L, uint64_t>), dim3(blocks), dim3(kBlock), 0, s, t, (const uint64_t *)keys, kl.id_bits, dst, bag, n_bags); \
    else hipLaunchKernelGGL((gather_pooled_direct<V, L, uint32_t>), dim3(blocks), dim3(kBlock), 0, s, t, (const uint32_t *)keys, kl.id_bits, dst, bag, n_bags); \
  } while (0)
  HCTR_DISPATCH_ROW(vec, lpr, CALL);
#undef CALL
  HCTR_HIP(hipGetLastError());
}

void launch_gather_pooled(hipStream_t s, const TableView &t, const BatchView &cur, const PullArgs &a, uint32_t bag) {
  if (!cur.n) return;
  const uint32_t n_bags = cur.n / bag;
  const int vec = row_vec(t.width, a.dst);
  const int lpr = lanes_for(t.width, vec);
  const bool local_only = a.got == nullptr;
#define CALL(V, L)                                                                                                  \
  do {                                                                                                              \
    const unsigned blocks = div_up(n_bags, kBlock / L);                                                             \
    if (local_only) hipLaunchKernelGGL((gather_pooled<V, L, true>), dim3(blocks), dim3(kBlock), 0, s, t, cur, a, bag, n_bags); \
    else hipLaunchKernelGGL((gather_pooled<V, L, false>), dim3(blocks), dim3(kBlock), 0, s, t, cur, a, bag, n_bags);  \
  } while (0)
  HCTR_DISPATCH_ROW(vec, lpr, CALL);
#undef CALL
  HCTR_HIP(hipGetLastError());
}

void launch_plain_copy(hipStream_t s, const void *src, void *dst, size_t bytes) {
  hipLaunchKernelGGL(plain_copy, dim3(256 * 16), dim3(kBlock), 0, s, (const uint4 *)src, (uint4 *)dst, bytes / 16);
  HCTR_HIP(hipGetLastError());
}

} // namespace hctr

// Host-callable launchers of the hot-path kernels.  Each one only enqueues work on `stream`.
// Reference stages are cited where the launcher is defined.
#pragma once
#include "common.h"
#include "launch_cut.h"
#include "row_slices.h"

namespace hctr {

// The sort key of a batch position: (owner << id_bits) | id.  Its order is the reference's
// id + kEmbeddingIDMax*owner (csrc/core/preprocess.cu:17): owner first, id second.
struct KeyLayout {
  int id_bits;    // bits of an id
  int total_bits; // id_bits + bits of an owner
  bool wide;      // 64-bit sort keys (total_bits > 32)
  int max_digit_bits = 0; // widest digit of the tile-sorted passes (0: the most the sort takes); narrower for tests
};

// Device-side view of one preprocessed batch (the reference's PreprocessData,
// csrc/core/preprocess_struct.h:7-24, with 32-bit positions and ranks).
struct BatchView {
  uint32_t n;                // keys in the batch (host-known)
  uint32_t *sorted_arg;      // [n]   positions grouped by unique key, stable   (d_sorted_arg)
  uint32_t *rank_sorted;     // [n]   unique rank of sorted position j
  uint32_t *idx_map;         // [n]   unique rank of position i, filled on request only    (d_idx_map)
  void *ukey;                // [U]   sort key of unique rank u: id and owner   (d_unique_idx, d_root)
  uint32_t *run_start;       // [U+1] first sorted position of rank u           (d_run_length)
  slot_t *uoff;              // [U]   resident offset of rank u or -1           (d_offset)
  uint32_t *bucket_lo;       // [R+1] first rank owned by each shard            (u_shape before :131)
  uint32_t *d_U;             // [1]   number of unique keys                     (unique_size)
  uint4 *long_list;          // [kLongBuckets][long_cap] runs longer than kLongRun by length class: {unique rank, first sorted position, length, resident offset}
  uint32_t *d_nlong;         // [kRunCounters] entries per class of long runs, then counters of the push
  uint32_t long_cap;         // capacity of one class
  uint32_t *med_list;        // [d_nlong[kMedCount]] unique ranks with kTinyRun < run length <= kLongRun (any order)
};

// d_nlong layout: [0, kLongBuckets) long runs per class, then the number of medium runs and the ticket counters of
// the long role
constexpr int kLongBuckets = 12;
constexpr int kMedCount = kLongBuckets, kTicketBase = kLongBuckets + 1, kTicketLanes = 16,
              kRunCounters = kTicketBase + 2 * kTicketLanes;

// A run of equal keys longer than this is summed by a whole block that streams its gradient rows through
// LDS; shorter runs are summed by a small group of lanes.
#ifndef HCTR_LONG_RUN
#define HCTR_LONG_RUN 128
#endif
constexpr uint32_t kLongRun = HCTR_LONG_RUN;
#ifndef HCTR_TINY_RUN
#define HCTR_TINY_RUN 8
#endif
constexpr uint32_t kTinyRun = HCTR_TINY_RUN; // runs up to this length are summed by the group that owns their rank
// Long runs are listed by length class (class 0 = longest) so that the push can start the longest chains first.
inline size_t long_list_capacity(uint32_t n) { return n / (kLongRun + 1) + 1; }
inline size_t med_list_capacity(uint32_t n) { return n / (kTinyRun + 1) + 1; }
__host__ __device__ inline int long_bucket(uint32_t len) {
  // class c holds lengths in [2^(17-c), 2^(18-c)), the first everything from 2^17 up, the last everything below 256
  int c = 0;
  for (uint32_t lim = 1u << 17; c < kLongBuckets - 1 && len < lim; lim >>= 1) c++;
  return c;
}

struct TableView {
  int rank, nrank;
  uint64_t id_max;
  uint32_t width;
  uint32_t n_stored, n_cached;   // kStorageMax, kNonLocalStorageMax
  float neg_lr;
  version_t pull_bound, push_bound;
  const worker_t *root;          // [id_max]
  const slot_t *slot;            // [id_max]  id -> resident offset or -1
  embed_t *emb;                  // [n_stored][width]
  version_t *ver;                // [n_stored]
  embed_t *pend;                 // [n_cached][width]
  version_t *upd;                // [n_cached]
};

// How many columns of a row a lane moves at a time, as a template argument of the row kernels:
//   4      16-byte vectors: the width is a multiple of four and the caller's pointer 16-byte aligned,
//   kOdd4  vectors of four floats at any 4-byte address (gfx950 loads and stores them in one instruction): every other
//          width from four on, and rows at pointers that are not 16-byte aligned.  The last lane of a row starts at
//          column W - 4, so it shares up to three columns with the lane before: both read them, and where a row is
//          updated in place only the lane before writes them,
//   1      rows of less than four floats.
// Against one float per lane (what every width but multiples of four took before), rows of 37 floats, 195 k keys of 39
// Zipf fields on an MI355X: a training step 148 -> 86 us (the push alone was 103 us of
// the 148).
constexpr int kOdd4 = -4;
template <int VEC> constexpr uint32_t kCols = VEC < 0 ? (uint32_t)-VEC : (uint32_t)VEC;
inline int row_vec(uint32_t width, const void *p) {
  return width < 4 ? 1 : (width % 4 == 0 && (uintptr_t)p % 16 == 0) ? 4 : kOdd4;
}
// the column a lane that is due at column c < width really starts at
template <int VEC> __device__ __forceinline__ uint32_t lane_col(uint32_t c, uint32_t width) {
  return VEC == kOdd4 ? overlapped_col(c, width) : c;
}

// Kernels of a step that every shard of a loopback group launches alike serve up to kShardsPerLaunch shards with one
// launch: the records travel as kernel arguments, and a block finds its own from where the records' blocks start.  (A
// launch costs a small batch more than its work: one launch per shard and kernel made a step of four shards of 53 k keys 73
// launches and 365 us; one for all, 22 and 183 us.)
constexpr int kShardsPerLaunch = 8;
// the records of one launch: one by itself, or up to kShardsPerLaunch
template <typename S, int M> struct Records {
  S s[M];
  BlockCut<M> cut;
};
// the record this block works for; block, blocks: its number among that record's blocks, and how many they are
template <typename S, int M>
__device__ __forceinline__ const S &my_record(const Records<S, M> &r, uint32_t &block, uint32_t &blocks) {
  block = blockIdx.x;
  if constexpr (M == 1) {
    blocks = gridDim.x;
    return r.s[0];
  } else {
    const uint32_t k = record_of(r.cut, block);
    blocks = r.cut.blocks[k];
    return r.s[k];
  }
}
// f(records, how many of them) for records make(0) .. make(count - 1) in pieces of one launch each, of blocks(k) blocks of
// `threads` threads for record k; the launch's grid is grid_of(records)
template <typename S, int M, typename Make, typename Blocks, typename F>
void launch_records(int count, uint32_t threads, Make &&make, Blocks &&blocks, F &&f) {
  for (int i = 0; i < count;) {
    Records<S, M> p = {};
    const int m = cut_blocks(p.cut, count - i, threads, 0, [&](int k) { return blocks(i + k); });
    for (int k = 0; k < m; k++) p.s[k] = make(i + k);
    if (p.cut.total) f(p, m);
    i += m;
  }
}
template <typename R> dim3 grid_of(const R &records) { return dim3(records.cut.total); }
// ... with kernels of their own for a single record
template <typename S, typename Make, typename Blocks, typename F>
void launch_one_or_records(int count, uint32_t threads, Make &&make, Blocks &&blocks, F &&f) {
  if (count == 1) launch_records<S, 1>(count, threads, make, blocks, f);
  else launch_records<S, kShardsPerLaunch>(count, threads, make, blocks, f);
}

// ---- preprocess ---------------------------------------------------------------------------------
// How the kernel that reads the caller's ids tells the host that it has, before the kernel ends: every block counts itself
// in *count once its ids are in registers and its sort keys have reached memory, and the last one puts the count back to
// zero and stores seq << 1 | (an id was out of range) in *word, which lies in pinned memory and is polled.  A launch and
// the wait for it then take 8.3 us for 52 blocks of a batch and 9.7 for 191, where an event behind the kernel takes 11.8;
// the count is one atomic per block, served one after the other, and eats that up between 256 and 416 blocks.
// There is no release in this: what makes the keys visible is what gfx950 does with the instructions, not the memory model.  A
// store at agent scope (sc1) writes through the XCD's cache, s_waitcnt vmcnt(0) returns when such stores are done, the barrier
// orders every wave's wait before the count, and the kernel that reads the keys begins with an acquire of its own launch.  A
// release would write back the whole cache of the XCD once per block.  A port to another chip has to put one there.
constexpr uint32_t kReadSignalBlocks = 256;
struct ReadSignal {
  uint32_t *count = nullptr, *word = nullptr; // word == nullptr: nobody polls
  uint32_t seq = 0;
};
// The sort key of one position.  Where somebody polls, a kernel on another stream may read the keys before this one has
// ended: the store then goes through to memory, and tell_ids_read() waits for it.
template <typename K> __device__ __forceinline__ void store_key(K *p, K v, const ReadSignal &r) {
  if (r.word) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = v;
}
// bad: this thread found an id out of range; err: where that is reported if nobody polls.  Every thread of the block calls it,
// having used every id it loaded and stored its keys.
__device__ __forceinline__ void tell_ids_read(const ReadSignal &r, uint32_t blocks, bool bad, uint32_t *err) {
  if (!r.word) {
    if (bad) atomicOr(err, 1u);
    return;
  }
  __builtin_amdgcn_s_waitcnt(0); // this wave's keys are in memory
  const uint32_t add = __syncthreads_or(bad) ? 0x10001u : 1u;
  if (threadIdx.x != 0) return;
  const uint32_t seen = __hip_atomic_fetch_add(r.count, add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + add;
  if ((seen & 0xffffu) != blocks) return;
  __hip_atomic_store(r.count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(r.word, r.seq << 1 | (seen >> 16 ? 1u : 0u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ids -> sort keys; flags ids outside [0, id_max) in *err (and sorts them as id 0)
// comp_keys is the batch's copy of the ids as well (the reference's d_idx); nlong (optional) is zeroed;
// sort_counts: the sort's scratch, which receives the per-tile counts of the first pass' digit
// ids32: `keys` points to 32-bit ids (narrowed on their way from pageable host memory; one that did not fit is
// 0xffffffff, which the range check flags like the id it stands for)
struct KeyShard {
  TableView t;
  const index_t *ids;
  uint32_t n;
  void *comp_keys;
  uint32_t *err, *nlong, *sort_counts;
  bool ids32;
  ReadSignal read;
};
// (batches of one tile shape)
void launch_make_keys(hipStream_t s, const KeyLayout &kl, const KeyShard *shards, int count);
// sorted keys -> everything per unique key + inverse index.  heads: the head counts per chunk of sorted positions that
// the last launch of the tile-sorted passes left (count_heads false), or storage for them (count_heads true: a launch
// of its own counts them first, one chunk per tile of the unique pass).
// u_copy (optional) receives the number of unique keys as well (b.d_U always does)
struct UniqueShard;
void launch_unique(hipStream_t s, const KeyLayout &kl, const UniqueShard *shards, int count, bool count_heads);

// batch-order inverse index from sorted_arg and rank_sorted (introspection; the hot path does not need it)
void launch_idx_map(hipStream_t s, const BatchView &b);
// the run lists of the batch (run_lists.h) by a launch of their own, after launch_unique; the gather builds them on its
// way when PullArgs::list_chunks is set
void launch_list_long_runs(hipStream_t s, const BatchView &b);
inline uint32_t run_list_chunks(uint32_t n) { return (n + 255) / 256; } // enough for any number of unique keys <= n

// Push plan of a batch (csrc/core/preprocess.cu:148-182) for every record: need[u] in {0,1}, prefix[u] = pushed rows before
// u, *total their number, and pushed rows per owner: prefix[lo[d+1]] - prefix[lo[d]] in cnt_out[0..nrank] and, pinned host
// memory, host_out.
struct PlanShard {
  TableView t;
  BatchView b;
  uint32_t *need, *prefix, *total, *block_sums; // block_sums: scan_blocks(n) + 1 words
  uint64_t *cnt_out, *host_out;
};
void launch_plans(hipStream_t s, const KeyLayout &kl, const PlanShard *shards, int count);
// unique keys per owner of every record's batch, in cnt_out[0..nrank] and host_out, and their number in host_U
struct BucketShard {
  const uint32_t *bucket_lo, *d_U;
  uint64_t *cnt_out, *host_out;
  uint32_t *host_U;
};
void launch_bucket_sizes(hipStream_t s, int nrank, const BucketShard *shards, int count);

// Division of a batch position by the bag size of sum-pooled lookups without a divide instruction: for any 32-bit
// n and bag >= 2, n / bag == (((n - q) >> 1) + q) >> shift with q = high word of n * magic (the "round up, add back"
// form of division by an invariant integer).  bag == 1 leaves positions alone (no shifts, magic 0).
struct BagDiv {
  uint32_t bag = 1, magic = 0, half = 0, shift = 0;
  BagDiv() = default;
  explicit BagDiv(uint32_t d) : bag(d) {
    if (d < 2) return; // magic 0 and no shifts: the formula below returns n
    half = 1;
    int lg = 31;
    while (!((d >> lg) & 1u)) lg--; // floor(log2 d)
    if ((d & (d - 1)) == 0) {         // a power of two: q is 0 and the two shifts make up log2(d)
      magic = 0;
      shift = (uint32_t)lg - 1;
      return;
    }
    const uint64_t num = (uint64_t)1 << (32 + lg);
    uint64_t m = num / d;
    const uint64_t rem = num - m * d;
    m = (m + m) & 0xffffffffull;
    const uint64_t twice = rem + rem;
    if (twice >= d) m += 1;
    magic = (uint32_t)(m + 1);
    shift = (uint32_t)lg;
  }
  // straight-line code for every bag size (a branch here would sit inside the load pipelines of the push)
  __host__ __device__ __forceinline__ uint32_t operator()(uint32_t n) const {
#ifdef __HIP_DEVICE_COMPILE__
    const uint32_t q = __umulhi(n, magic);
#else
    const uint32_t q = (uint32_t)(((uint64_t)n * magic) >> 32);
#endif
    return (((n - q) >> half) + q) >> shift;
  }
};

// ---- push: segment-sum of gradients by unique key + fused SGD ----------------------------------------
struct PushArgs {
  const embed_t *grad;       // [n_prev / bag][width]
  BagDiv bag;                // bag size of sum-pooled lookups (1: none): position i reads gradient row i / bag
  const uint32_t *need;      // [U_prev] or nullptr when nrank == 1
  const uint32_t *prefix;    // [U_prev] push slot
  index_t *g_idx;            // push buffers
  version_t *g_cnt;
  embed_t *g_val;
};
// pos[u] = prefix[u] + delta[owner of unique key u] for the n_unique unique keys of every record's batch: the place of a
// pushed row in a receive area shared by all owners, from its place in the shard's own plan (delta: nrank words in device
// memory)
struct PlaceShard {
  const void *ukey;
  uint32_t n_unique;
  const uint32_t *prefix, *delta;
  uint32_t *pos;
};
void launch_place_rows(hipStream_t s, const KeyLayout &kl, const PlaceShard *shards, int count);
// the pushes of every record's batch (one shard's, or those of the shards of a group, all with the same bag size)
struct PushShard {
  TableView t;
  BatchView b;
  PushArgs a;
  uint32_t n_unique;         // number of unique keys of the batch (host copy)
};
void launch_push(hipStream_t s, const KeyLayout &kl, const PushShard *shards, int count);

// ---- query / owner side / pull -------------------------------------------------------------------------
// Owner side of a step: applying the received pushes (per target row in source order) and serving the received
// queries (outdated flags, positions of the rows to return, rows packed, first returned row of every requester).
// One entry per shard of the group; one set of launches serves them all.
struct OwnerShard {
  TableView t;
  // received pushes, sources concatenated in rank order; rg_seg[0..nsrc]: first row of every source
  const index_t *rg_idx;
  const version_t *rg_cnt;
  const embed_t *rg_val;
  uint32_t rg_seg[258];
  int longest;               // the source with the most rows
  uint32_t push_blocks;      // blocks the push kernel needs for this shard (rows of `longest` / rows per block)
  // Received queries; rq_seg[0..nsrc]: first query of every requester; [rq_seg[rank], rq_seg[rank + 1]) are its own.
  // How many unique keys every shard asks every owner for is known on the device only (the host does not wait for the
  // index of the current batches): send_cnt / n_keys are filled in on the host, and place_queries -- a launch in front
  // of the query kernels -- cuts the group's receive area from them and writes rq_idx .. ret_slot and got_delta below.
  const uint64_t *send_cnt;  // [nsrc] unique keys of THIS shard's current batch per owner (written by its index)
  uint32_t n_keys;           // keys of this shard's current batch; 0: the shard asks for nothing (send_cnt is stale)
  const index_t *rq_idx;
  const version_t *rq_ver;
  uint32_t rq_seg[258];
  uint32_t q, query_tiles;
  uint32_t *outdated, *tile_cnt;
  slot_t *q_slot;            // slot of every received query (kNoSlot: not owned here)
  slot_t *ret_slot;          // slots of the rows to return, in return order
  // The returned rows are written straight into the requesters' buffers.  in_ver / in_val: THIS shard's buffers as a
  // requester (an owner finds its requester s in entry s of the array of shards); ret_delta[s]: what an owner adds to
  // the place of a row in its own return order to get the row's place in requester s' buffers, where the rows of all
  // owners stand in owner order.
  version_t *in_ver;
  embed_t *in_val;
  uint32_t *ret_delta;       // [nsrc]
  // The flag of every received query goes straight to its requester as well: got = THIS shard's flags as a requester
  // (one per unique key, owners in rank order); got_delta[s]: what an owner adds to the place of a query in its receive
  // buffer to get the place of the flag in requester s' array (written by place_queries).
  uint32_t *got;
  uint32_t got_delta[257];
  uint32_t *err;             // the shard's error word
  uint32_t *seg_dev;         // [0..nsrc] first returned row of every requester's segment, device copy
  uint32_t *seg_host;        // the same in memory the host reads; [257] = error flags
};
size_t query_tiles(uint32_t q);                       // tile_cnt needs this many words + 1
uint32_t owner_push_rows_per_block(uint32_t width);   // rows of the longest source one block of the push kernel takes
// The receive area of the queries of a step, shared by all owners of the group: every array holds one entry per unique
// key of all current batches at most (`capacity`).  launch_place_queries cuts it: one piece per owner, inside it one per
// requester, both in rank order (csrc/core/all2all.cu:18-46), from the counts the shards' index kernels left on the
// device, and writes into every shard's record where its piece lies, and into query_delta[s * nsrc + d] what requester
// s adds to the rank of a unique key owned by d to get the key's place in the area.
struct QueryArea {
  index_t *idx;
  version_t *ver;
  uint32_t *outdated;
  slot_t *q_slot, *ret_slot;
  uint32_t *query_delta;     // [nsrc * nsrc]
};
// (shards_host: the records as the host filled them in, for the addresses of the counts)
void launch_place_queries(hipStream_t s, OwnerShard *shards_dev, const OwnerShard *shards_host, int nsrc,
                          const QueryArea &area);
// shards_dev: the array in device memory.  nshards == nsrc: every shard of the group is in the array, in rank order (an
// owner looks its requesters up there).
// The received pushes; push_blocks: the most blocks a shard's need.  Nothing of it depends on the batches that are current: it
// does not wait for their index.
void launch_apply_pushes(hipStream_t s, const OwnerShard *shards_dev, int nshards, int nsrc, uint32_t width, uint32_t push_blocks);
// The received queries, behind launch_apply_pushes; queries_max: no shard receives more queries than this; queries_guess: what the busiest shard probably receives (the grids are cut
// from it; what a shard does receive, the kernels read from the records and stride over).
// pulls: the requesters; their launches' share is the index of every returned row per unique key (a.ret_i), where the gather
// reads each key's row (a.src_row) and the counts of the step.
struct PullShard;
void launch_owner_side(hipStream_t s, const OwnerShard *shards_dev, int nshards, int nsrc, uint32_t width, uint32_t queries_max, uint32_t queries_guess, const PullShard *pulls, int npulls);
// requester: refresh cached rows that came back, then gather every key's row into dst
struct PullArgs {
  const uint32_t *got;       // [U] or nullptr: nothing came back (nrank == 1)
  uint32_t *ret_i;           // [U] index into the returned rows (written by launch_owner_side)
  uint32_t *src_row;         // [U] where the gather reads a key's row (written by launch_owner_side): offset or returned row
  const version_t *in_ver;
  const embed_t *in_val;
  embed_t *dst;              // [n][width]
  bool stream_stores;        // write dst with nontemporal stores (see Shard::write_back)
  uint32_t list_chunks;      // the gather also builds the batch's run lists (run_lists.h): chunks of unique ranks, else 0
};
// One shard of a loopback group as the kernels on its own batch see it; the launches below serve all records.
struct PullShard {
  TableView t;
  BatchView b;               // n != 0
  PullArgs a;
  // queries: id and local version of every unique key of the batch, written to place (unique rank + delta[owner of the
  // key]) of q_idx / q_ver (delta: nrank words in device memory)
  const uint32_t *delta;
  index_t *q_idx;
  version_t *q_ver;
  // refresh: scratch of 4 * scan_blocks(n) words; four words the device can write (hit / miss / refreshed counts of the step,
  // error bits)
  uint32_t *tile_counts, *host_stats;
  // what the step before had: unique keys (the grid of the refresh is cut from it; how many there are the kernels read), cached
  // rows that came back
  uint32_t unique_guess, refreshed_guess;
};
void launch_build_queries(hipStream_t s, const KeyLayout &kl, const PullShard *shards, int count);
// The refresh of the cached rows that came back.
void launch_refresh(hipStream_t s, const PullShard *shards, int count);
// every key's row into a.dst (may be null: nothing to gather), and the run lists of the batch (a.list_chunks)
void launch_gather_group(hipStream_t s, const PullShard *shards, int count);
// one shard, every row local
void launch_gather(hipStream_t s, const TableView &t, const BatchView &cur, const PullArgs &a);
// one shard: dst[i] = row of the id in keys[i] (the batch's sort keys in batch order), for all n positions; needs
// nothing of the batch's index
void launch_gather_direct(hipStream_t s, const TableView &t, const KeyLayout &kl, const void *keys, uint32_t n, embed_t *dst,
                          bool stream_stores);
// the same for bags of `bag` consecutive positions, one summed output row per bag (n a multiple of bag)
void launch_gather_pooled_direct(hipStream_t s, const TableView &t, const KeyLayout &kl, const void *keys, uint32_t n,
                                 embed_t *dst, uint32_t bag);
// sum-pooled lookups: dst[b] = the rows of positions b * bag .. b * bag + bag - 1 added up in that order
// (cur.idx_map must be filled: launch_idx_map)
void launch_gather_pooled(hipStream_t s, const TableView &t, const BatchView &cur, const PullArgs &a, uint32_t bag);

// ---- init -------------------------------------------------------------------------------------------------
void launch_init_values(hipStream_t s, embed_t *out, size_t len, int type, float a, float b, unsigned seed);
void launch_fill_i64(hipStream_t s, version_t *p, size_t n, version_t v);
void launch_fill_i32(hipStream_t s, int32_t *p, size_t n, int32_t v);
void launch_build_directory(hipStream_t s, const index_t *store_ids, uint32_t n_stored, slot_t *slot);
void launch_plain_copy(hipStream_t s, const void *src, void *dst, size_t bytes); // bytes % 16 == 0
// keys_out[r * fields + f] = log[rows[r] * fields + f]; a row number outside [0, n_samples) sets bit 0 of *err
void launch_sample_rows(hipStream_t s, const index_t *log, uint64_t n_samples, uint32_t fields, const index_t *rows,
                        uint64_t n_rows, index_t *keys_out, uint32_t *err);

} // namespace hctr

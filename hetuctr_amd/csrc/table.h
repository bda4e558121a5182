// Host-side state of one shard (the reference's HetuTable, csrc/core/hetu_gpu_table.h:21-144) and of the
// in-process loopback group that stands in for the NCCL communicator.
#pragma once
#include <condition_variable>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/hetuctr_hip.h"
#include "host_copy.h"
#include "kernels.h"
#include "radix_sort.h"
#include "tile_sort.h"

namespace hctr {

// growable device allocation; contents are NOT kept when it grows
struct DeviceBuf {
  void *p = nullptr;
  size_t bytes = 0;
  DeviceBuf() = default;
  DeviceBuf(const DeviceBuf &) = delete;
  DeviceBuf &operator=(const DeviceBuf &) = delete;
  DeviceBuf(DeviceBuf &&o) noexcept : p(o.p), bytes(o.bytes) { o.p = nullptr; o.bytes = 0; }
  DeviceBuf &operator=(DeviceBuf &&o) noexcept {
    if (this != &o) {
      release();
      p = o.p;
      bytes = o.bytes;
      o.p = nullptr;
      o.bytes = 0;
    }
    return *this;
  }
  ~DeviceBuf() { release(); }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
  }
  bool reserve(size_t want) { // true: a new allocation was made
    if (want <= bytes) return false;
    release();
    size_t grow = want + want / 8; // headroom so that slowly growing batches do not reallocate every step
    HCTR_HIP(hipMalloc(&p, grow));
    bytes = grow;
    return true;
  }
  template <typename T> T *as() const { return (T *)p; }
};

// per-batch buffers: the reference's PreprocessData (csrc/core/preprocess_struct.h:7-24)
struct Batch {
  uint32_t n = 0;   // keys
  uint32_t U = 0;   // unique keys (host copy, valid after the preprocess call returned)
  bool idx_map_valid = false;
  bool cleared = false; // the device side reads as an empty batch (U = 0, no buckets, no runs) since clear()
  bool planned = false; // the push plan (need, prefix, push_cnt) has been computed for the batch as it stands
  int early_sort_steps = 0; // three-launch passes: the launches that preprocess enqueues before it returns
  bool lists_ready = true;  // the run lists of the batch's push have been built (or the batch is empty)
  bool tile_sorted = false; // indexed by the tile-sorted passes (tile_sort.h)
  bool one_block = false;   // indexed by one block in one launch (tile_sort.h)
  bool direct_gather = false; // one shard, small batch: the step's gather works from `comp` in batch order and does not
                              // wait for the index (the run lists are then built while the next preprocess waits for
                              // its ids, or in front of the batch's push)
  bool keys_made = false;   // the ids are read by a kernel that makes the sort keys alone; else by the first launch of the
                            // tile-sorted passes.  Either leaves the sort keys in comp
  // comp: the batch's sort keys in batch order (id and owner of every position); staged: ids that arrived in
  // pageable host memory, on their way to the key kernel
  DeviceBuf comp, staged, sorted_arg, rank_sorted, idx_map, ukey, run_start, uoff, bucket_lo, dU, long_list, dnlong, med_list;
  DeviceBuf need, prefix, plan_total; // push plan per unique key: pushed or not, position among the pushed rows; their number
  std::vector<uint64_t> send_cnt, recv_cnt;       // queries per owner / per requester
  std::vector<uint64_t> push_cnt, pushrecv_cnt;   // pushed rows per owner / per source
  void reserve(uint32_t n_keys, int nrank, bool wide);
  bool holds(uint32_t n_keys, int nrank, bool wide) const; // reserve() would not allocate
  void clear(hipStream_t s, int nrank); // make the device side an empty batch; does nothing if it already is
  void drop(); // an empty batch to the host, whatever its buffers hold (they may be half made)
  BatchView view() const;
};

// What the host reads back after a preprocess call: written by kernels into one device block (DevStat) and
// copied with ONE transfer into the pinned HostMirror.  A single shard only needs the first 16 bytes.
struct DevStat {
  uint32_t U;
  uint32_t err;
  uint32_t push_total;
  uint32_t read_count; // ReadSignal::count: zero between the launches that use it
  uint64_t send_cnt[257];
  uint64_t push_cnt[257];
};
struct HostMirror {
  DevStat st;
  uint32_t stats[4];
  uint32_t ret_seg[258];
  // written by the kernel that reads the caller's ids when preprocess returns early (no copy): an id out of range, or
  // the two at once (ReadSignal)
  uint32_t key_err, ids_read;
  uint32_t key_err_known; // where the kernel's range check reports what the host has found already
};

class Group;

// launches of the sort that a deferred preprocess enqueues itself: the column scan and the scatter of the first pass
// and the count of the second (the first count comes from the key kernel); with the tile-sorted passes, the first of
// the launches that follow the key kernel
#ifndef HCTR_EARLY_SORT_STEPS
#define HCTR_EARLY_SORT_STEPS 4
#endif
#ifndef HCTR_EARLY_TILE_PASSES
#define HCTR_EARLY_TILE_PASSES 1
#endif
constexpr int kEarlySortSteps = HCTR_EARLY_SORT_STEPS, kEarlyTilePasses = HCTR_EARLY_TILE_PASSES;
// ... and where the run lists of the batch before are built meanwhile, the column scan alone.  The push follows those lists
// within a few microseconds, and a scatter launched early would be holding the CUs then, two blocks each: the long runs'
// blocks, which start first, would land two by two on the few it leaves, and the push of 4.16 M keys of 16 floats, Zipf 1.4
// (508 blocks of the scatter on 512 places), takes 391 us instead of 269.  Two training steps with the scatter early and
// behind the push: those 1116 and 865 us (903 with the lists in front of the push), 1.6 M keys 410 and 393, 2.6 M 586 and
// 569; pooled, 64 floats, 4.15 M keys 1013 and 832, 8.4 M 1584 and 1598 (no difference: runs differ by 2 %); keys held in 64
// bits, one block per CU, 2 M 701 and 497, 3 M 772 and 688, with exponent 1.05 741 and 760.  A push that follows without
// such lists comes a little later; 3 M keys of 32 floats are 4 % slower this way.
constexpr int kEarlySortStepsBesideLists = 2;
// One shard: a batch whose output rows take up to this many bytes is gathered in batch order straight from its keys
// (Batch::direct_gather).  Measured on an MI355X with 512-byte rows: 107 k keys 78 us per step against 92 with the gather
// in sorted order behind the index, 426 k keys 165 against 174, 852 k keys 316 against 279 -- in batch order the
// duplicates of a key are not adjacent, and from about the size of the last-level cache (256 MB) on the rows of a batch
// no longer stay cached between them.
#ifndef HCTR_DIRECT_GATHER_BYTES
#define HCTR_DIRECT_GATHER_BYTES (256ull << 20)
#endif

// stages whose device time can be measured separately (HIP events on the group's stream)
enum Stage { S_KEYS = 0, S_SORT, S_UNIQUE, S_PLAN, S_PUSH, S_QUERY, S_EXCHANGE, S_OWNER, S_REFRESH, S_GATHER, S_COUNT };
const char *stage_name(int s);

class Shard {
 public:
  Shard(const hctr_config &cfg, const uint8_t *root_arr, const int64_t *storage_arr, size_t n_storage,
        unsigned seed, std::shared_ptr<Group> group);
  ~Shard();

  hctr_config cfg;
  std::string ip;
  std::shared_ptr<Group> group;
  KeyLayout kl;
  TableView tv;
  size_t n_owned = 0;

  // ---- stages, each only enqueues on the group's stream (names follow hetu_gpu_table.h:82-97) ----
  void swap_batches() { std::swap(cur, prev); }
  void check_batch(const int64_t *keys, size_t n) const; // refuses what no batch can be
  void preprocess_index(const int64_t *keys, size_t n) {
    ingest_keys(keys, n);
    index_batch();
  }
  // the caller's ids -> device copy and sort keys; flag: where the range check reports (default: the device word)
  // scratch_area (default: the shard's own growable buffers): the index scratch of this batch is cut out of it
  void ingest_keys(const int64_t *keys, size_t n, uint32_t *flag = nullptr, void *scratch_area = nullptr);
  // sort, unique, run lists of the ingested batch; u_out: where the number of unique keys goes besides the batch's
  // own device word (default: the device block that is read back after the call)
  void index_batch(uint32_t *u_out = nullptr, int part = 0);
  // the host's part of ingest_keys, without its launch (Group::launch_keys)
  void prepare_keys(const int64_t *keys, size_t n, uint32_t *flag, void *scratch_area = nullptr);
  TileSortShard tile_sort_record() const;
  HeadChunks heads() const;
  const index_t *ids_ = nullptr; // of the prepared batch: where the key kernel reads them, and whether as 32-bit words
  bool narrowed_ = false;
  uint32_t *key_flag_ = nullptr; // ... and where it reports a key out of range
  ReadSignal read_;              // ... or how it says that it has read them all
  bool wait_ids_read(hipStream_t on); // waits for that, if it does say so; true: a key was out of range
  // One shard, ids narrowed on their way through pinned memory: the caller's buffer is free and the ids' range known when they
  // are staged, so preprocess waits for no kernel (ids_bad_ is what it reports).  Whoever reads the sort keys outside the index
  // stream waits first: a step's gather from the keys (keys_unread_).
  bool staged_ = false, ids_bad_ = false, keys_unread_ = false;
  void wait_keys();
  TileSortBuffers tile_sort_buffers() const; // the index scratch as the tile-sorted passes take it
  HostStager stager;                         // ids that arrive in pageable host memory go through its pinned buffer
  bool pooled_from_keys = true;   // HETUCTR_POOLED_FROM_KEYS=0: pooled gathers of one shard go through the inverse index
  uint32_t direct_gather_max = 0; // keys: HCTR_DIRECT_GATHER_BYTES / bytes of a row, or HETUCTR_DIRECT_GATHER_MAX
  int tile_sort_mode = 1;                    // HETUCTR_TILE_SORT: 0 no batch takes the tile-sorted passes, 1 those of up
                                             // to kTileSortMaxKeys keys (up to kOneBlockKeys: one block does it all), 2
                                             // every batch whose tiles they can hold
  bool plan_record(Batch &b, PlanShard &o); // this shard's part of a launch of plans; false: b is empty, nothing to plan
  void enqueue_readback_preprocess();
  void finish_preprocess();                 // after the stream sync: mirrors -> host fields, error checks
  // the same in two halves, for a preprocess whose push plan and index run on different streams
  void finish_plan(Batch &b); // takes the counts over into b once they are there
  void finish_index();
  void check_key_error();                   // raises if the ingested batch held a key outside [0, length)
  // the push of a step in two halves, so that a group can place every shard's pushed rows before any push kernel runs
  void begin_push(const float *grad, uint32_t bag = 1);  // which batch is pushed (none on an inference step), checks
  void list_runs();
  bool push_record(PushShard &o);                        // what the push kernel needs of this shard; false: nothing
  // handleGradient + handleQuery: what the group's owner-side launches need of this shard (queries_max: no shard
  // receives more queries than this)
  void fill_owner_args(OwnerShard &o, uint64_t queries_max);
  void finish_handle_query();               // after the step: return counts and error flags from the pinned block
  // several shards: what the query, refresh and gather launches need of this one (delta: see QueryArea::query_delta)
  bool pull_record(PullShard &o, float *dst, uint32_t bag, const uint32_t *delta);
  PullArgs pull_args(float *dst) const;
  uint32_t take_list_chunks();
  void forget_lists();
  void gather_bags(const PullArgs &a, uint32_t bag);
  void write_back(float *dst, uint32_t bag = 1); // one shard
  bool direct_now(uint32_t bag) const; // this step's gather works from the keys and does not wait for the index
  void finish_push_pull();

  size_t fetch(int which, void *host_out, size_t cap);
  // rows, versions, pending gradients and update counters to / from one file (checkpoint.hip)
  void save(const char *path);
  void load(const char *path);

  Batch cur, prev;
  bool prev_active = false; // false: inference step or no previous batch, nothing is pushed
  DeviceBuf root, slot, emb, ver, pend, upd, store_ids;
  // scratch shared by the stages
  DeviceBuf ktmp0, ktmp1, vtmp0, vtmp1, sortws, block_sums, headws, dstat;
  // where the index stages of the current batch find their scratch: the buffers above or pieces of the static array
  struct ScratchPtrs {
    void *ktmp0 = nullptr, *ktmp1 = nullptr;
    uint32_t *vtmp0 = nullptr, *vtmp1 = nullptr, *sortws = nullptr, *block_sums = nullptr, *headws = nullptr;
  } sp;
  DeviceBuf plan_sums, query_sums; // query_sums: flags per tile of received queries // plan_sums: scan scratch of the push plan (the index has block_sums to itself)
  DevStat *dst_ = nullptr; // == dstat.p
  uint32_t read_seq_ = 0;
  uint32_t *err_ptr() const { return &dst_->err; }
  // send side
  const float *push_grad_ = nullptr; // arguments of the push between begin_push and push_record
  uint32_t push_bag_ = 1;
  bool trains_ = false;              // the last push_pull came with a gradient
  // receive side (owner role)
  DeviceBuf src_row, ret_seg_dev;
  std::vector<uint64_t> rq_seg, rg_seg, ret_seg; // R+1 prefix offsets per source / requester
  uint64_t rg_base = 0;      // first row of this shard's piece of the group's receive area for pushed rows
  uint64_t rq_base = 0;      // first query of its piece of the receive area for queries (rq_seg, rq_base: the host's
                             // copy of what place_queries computed on the device, made when the step is over)
  DeviceBuf push_pos;        // place of every unique key's pushed row in that area (plan position + distance)
  // requester side of the return
  DeviceBuf got, ret_i, in_ver, in_val;
  HostMirror *mirror = nullptr;
  long long last_stats[6] = {0, 0, 0, 0, 0, 0};
  float last_pre_ms = 0.f, last_pp_ms = 0.f, last_push_ms = 0.f;
  bool u_cleared = false;    // the device-side copy of the number of unique keys reads as zero

 private:
  void reserve_batch_scratch(uint32_t n);
  void use_scratch_area(void *area, uint32_t n);
};

// The entry point that allocates nothing takes batches of up to kNoAllocMaxKeys keys; kNoAllocScratchBytes is what
// the index of such a batch needs with 64-bit sort keys (sort ping-pong buffers, per-tile digit tables, scan sums, head
// counts per chunk), every piece rounded up to 256 bytes.
constexpr size_t kNoAllocMaxKeys = 262144;
constexpr size_t index_scratch_round(size_t b) { return (b + 255) / 256 * 256; }
// words of digit tables either sort of a batch of n keys needs
constexpr inline size_t index_table_words(size_t n) {
  const size_t a = sort_scratch_words(n), b = tile_sort_possible(n) ? tile_sort_table_words(n) : 0;
  return a > b ? a : b;
}
// bytes of index scratch a batch of n keys needs (n >= 1)
constexpr inline size_t index_scratch_bytes(uint32_t n, bool wide) {
  const size_t m = n < 1 ? 1 : n, ks = wide ? 8 : 4;
  return 2 * index_scratch_round(m * ks) + 2 * index_scratch_round(m * 4) + index_scratch_round(index_table_words(m) * 4) +
         index_scratch_round((scan_blocks(m) + 2) * 4) + index_scratch_round(head_chunk_words(m) * 4);
}
// An upper bound of index_scratch_bytes over all n <= kNoAllocMaxKeys that needs no loop: the tables of the smallest
// tile shape (or of the most tiles the tile-sorted passes take) and the head counts of the smallest chunk at the largest n.
constexpr size_t kNoAllocScratchBytes =
    2 * (kNoAllocMaxKeys * 8) + 2 * (kNoAllocMaxKeys * 4) +
    (kNoAllocMaxKeys / (kSortBlock * kSortItemsSmall) + 8) * kSortMaxBins * 4 + (kNoAllocMaxKeys / 2048 + 3) * 4 +
    (kNoAllocMaxKeys / 128 + 1) * 5 * 4 + 64 + 8 * 256;
static_assert((kTileSortMaxTiles + 7) / 8 * 8 <= kNoAllocMaxKeys / (kSortBlock * kSortItemsSmall) + 8, "tables of the tile-sorted passes");
// the sizes where the tile shape of a sort changes, and the largest batch: changed tile constants fail here
static_assert(index_scratch_bytes((uint32_t)kSortSmallUpTo, true) <= kNoAllocScratchBytes &&
                  index_scratch_bytes((uint32_t)kSortSmallUpTo + 1, true) <= kNoAllocScratchBytes &&
                  index_scratch_bytes((uint32_t)(2 * kTileSortMaxTiles * kSortBlock), true) <= kNoAllocScratchBytes &&
                  index_scratch_bytes((uint32_t)(2 * kTileSortMaxTiles * kSortBlock) + 1, true) <= kNoAllocScratchBytes &&
                  index_scratch_bytes((uint32_t)kNoAllocMaxKeys, true) <= kNoAllocScratchBytes,
              "the static scratch of the entry point that allocates nothing is too small");

// All shards of one loopback group live in one process on one device and share one stream.  The group
// carries the collective calls: every shard's thread deposits its arguments, the last one to arrive runs the
// step for all shards, the others wait for it.
class Group {
 public:
  Group(int nrank, int device_id, std::string key);
  ~Group();
  const int nrank;
  const int device_id;
  const std::string key;
  hipStream_t stream = nullptr;          // the stream the stages enqueue on (see StreamSwitch)
  hipEvent_t ev0 = nullptr, ev1 = nullptr, ev_pre0 = nullptr, ev_pre1 = nullptr; // call timing: of push_pull, of preprocess
  // Single shard: preprocess enqueues its work on a second stream and returns once the caller's ids are consumed;
  // sorting and deduplicating them has no dependence on the pending gradient push, so the next push_pull starts the
  // push on the main stream right away and only the gather waits for both.
  hipStream_t index_stream = nullptr;
  hipEvent_t ev_index = nullptr, ev_keys = nullptr, ev_push = nullptr, ev_pushed = nullptr, ev_plan = nullptr;
  bool defer_index = false;              // the mode is on (HETUCTR_DEFER_INDEX != 0)
  bool index_pending = false;            // a batch's index is enqueued and nobody has waited for it yet
  bool index_rest_pending = false;       // single shard: preprocess enqueued only the first launches of the index
  void enqueue_index_rest();
  void enqueue_index_all(int part);             // enqueues the others
  // the same stage of several shards' batches, one launch for all whose batches have the same shape
  void launch_keys(Shard *const *shards, size_t count);
  void index_batches(Shard *const *shards, size_t count, uint32_t *u_out, int part);
  void enqueue_bucket_sizes(bool empty);
  // enqueues the push plans of one batch of each of the shards; the counts reach the host when the stream has run it
  void plan_batches(const std::vector<Shard *> &shards, Batch Shard::*which);
  void flush_index();                    // waits for a pending index and takes its results over
  // owner-side arguments of every shard: pinned staging and the device copy the kernels read (owner_host: the records behind
  // the distances of the pushed rows in one staging area, because both go to the device in front of the push)
  OwnerShard *owner_host = nullptr;
  DeviceBuf owner_dev, ret_delta_dev;    // ret_delta_dev: nrank words per owner, see OwnerShard::ret_delta
  uint64_t fill_owners();
  void apply_pushes();
  void owner_side(uint64_t queries_max, const std::vector<PullShard> &pulls);
  // Where every shard's pushed rows go: one receive area for the whole group (ids, counts, rows), cut into one piece
  // per owner and, inside it, per source; sized from the plans before any push kernel runs.  Every sender gets, per
  // owner, the distance between a row's place in its own plan and its place in the area (nrank words per sender).
  uint64_t place_pushes(); // and fills the owners' records; returns the most queries there can be
  DeviceBuf rg_idx_all, rg_cnt_all, rg_val_all, push_delta_dev;
  uint32_t *push_delta_host = nullptr;   // pinned staging of the distances and, owner_offset() bytes in, of the records
  size_t owner_offset() const { return ((size_t)nrank * nrank * sizeof(uint32_t) + 255) / 256 * 256; }
  bool pushes_placed_ = false;           // the step has pushed rows: push_delta_dev holds its distances and records
  // The same for the queries of a step: one receive area (ids, versions, and what the owners keep per query), nrank
  // distances per requester.  How many queries go where is known on the device only: reserve_queries() sizes the area
  // for the most there can be, launch_place_queries (behind the upload of the owners' records) cuts it.
  uint64_t reserve_queries();
  QueryArea query_area();
  void note_query_places(); // rq_seg / rq_base of every shard from the counts the host has once the step is over
  uint32_t queries_guess_ = 0; // queries the busiest owner received in the step before
  bool queries_seen_ = false;
  DeviceBuf rq_idx_all, rq_ver_all, rq_outdated_all, rq_slot_all, rq_ret_all, query_delta_dev;
  bool time_calls = false;               // bracket the two calls with events (hctr_call_timing)
  bool pre_timed_ = false;               // the events of the last preprocess are recorded and nobody has asked for the time
  std::vector<Shard *> members;
  double wait_seconds = 120.0;
  void sync_stream();
  bool wait_ids_read(); // waits until the callers' ids have been read; true: a key was out of range

  // per-stage device time, accumulated over calls while stage_timing is on
  bool stage_timing = false;
  double stage_ms[S_COUNT] = {};
  long long stage_calls[S_COUNT] = {};
  struct StageMark { int stage; hipEvent_t a, b; };
  std::vector<StageMark> marks;          // of the call in flight
  std::vector<hipEvent_t> event_pool;
  hipEvent_t take_event();
  void collect_marks();                  // after a stream sync
  void set_defer_index(bool on);         // switches the early return of preprocess; waits for a pending index first
  void set_call_timing(bool on);         // events around the two calls; the times of earlier calls are forgotten
  void take_pre_time();                  // last_pre_ms of every shard, waiting for the kernels of the call if need be
  void set_stage_timing(bool on);        // resets the accumulators; waits for a pending index under the group's lock

  void join(Shard *s);
  void leave(Shard *s);
  bool complete() const;

  // lock-step bodies (one caller)
  void preprocess_all(const int64_t *const *keys, const size_t *n);
  void preprocess_noalloc(const int64_t *keys, size_t n);
  void *noalloc_scratch = nullptr;       // device address of this GPU's static scratch array
  // bag > 1: sum-pooled lookups, grads and dsts hold one row per bag of `bag` consecutive keys
  void push_pull_all(const float *const *grads, float *const *dsts, size_t bag = 1);
  // per-shard entry points: rendezvous of nrank callers
  void preprocess_one(int rank, const int64_t *keys, size_t n);
  void push_pull_one(int rank, const float *grad, float *dst, size_t bag = 1);

 private:
  void exchange_shapes();
  void push_pull_steps(const float *const *grads, float *const *dsts, uint32_t bag); // the body of push_pull_all
  void preprocess_steps(const int64_t *const *keys, const size_t *n, bool &taken); // the body of preprocess_all
  void stop_work();
  void finish_lists();
  bool lists_running_ = false; // a preprocess has launched the run lists of the previous batch on the main stream
  bool index_joining_ = false; // push_pull has taken a pending index over and not yet read its results
  template <typename F> void collective(int rank, int op, F &&run_all);
  std::mutex mu_;
  std::condition_variable cv_;
  int arrived_ = 0, pending_op_ = 0;
  uint64_t generation_ = 0;
  std::string failure_;
  std::vector<const int64_t *> a_keys_;
  std::vector<size_t> a_n_;
  std::vector<const float *> a_grad_;
  std::vector<float *> a_dst_;
  std::vector<size_t> a_bag_;
};

// brackets the launches of one stage with two events when stage timing is on
struct StageScope {
  Group &g;
  int idx = -1;
  StageScope(Group &grp, int stage) : g(grp) {
    if (!g.stage_timing) return;
    Group::StageMark m{stage, g.take_event(), g.take_event()};
    HCTR_HIP(hipEventRecord(m.a, g.stream));
    g.marks.push_back(m);
    idx = (int)g.marks.size() - 1;
  }
  ~StageScope() {
    if (idx >= 0) (void)hipEventRecord(g.marks[idx].b, g.stream);
  }
};

// makes the stages enqueue on another stream for the lifetime of the object
struct StreamSwitch {
  Group &g;
  hipStream_t saved;
  StreamSwitch(Group &grp, hipStream_t s) : g(grp), saved(grp.stream) { g.stream = s; }
  ~StreamSwitch() { g.stream = saved; }
};

std::shared_ptr<Group> find_or_create_group(int nrank, int device_id, const std::string &ip, int port);

} // namespace hctr

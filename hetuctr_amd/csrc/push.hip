// Gradient push: deterministic segment-sum of the gradient rows of every unique key of the previous
// batch, fused with the SGD write-back to the table, the hot-row cache, the pending-gradient store,
// the version / update counters and the push buffer.
// Reference: csrc/core/generate_query.cu:8-89 (gradient_reduction_kernel, gradient_index_kernel).
//
// Summation order: the reference adds the gradient rows of one key serially, in ascending batch position,
// then multiplies once by -lr and adds once to the row.  fp32 addition is not associative, so any other
// order differs from it in the last bits by an amount that grows with the number of duplicates.  Here
// every run of equal keys is summed by ONE chain of additions per column, in exactly that order: sums are
// bit-identical to the reference's order (compiled without fused multiply-add contraction), for any skew.
// "Bit-identical" is against that non-contracted restatement on the CPU: the reference itself is built by nvcc,
// whose default may fuse `sum *= -lr; dest += sum` (generate_query.cu:37-39) into one multiply-add, so against a
// CUDA build the last rounding of an updated value can differ by one ulp.  The contract against the reference is
// its own tolerance, 1e-5 relative.
//
// One launch, three ranges of blocks, one per class of run length (the long chains are dispatched first and the
// other blocks fill the machine behind them):
//  * long (> kLongRun duplicates): bundles of runs are streamed by whole blocks, one column slice at a time.  Six
//    loader waves keep 16 vectors of gradient rows in flight per lane and stage them through two LDS slots; one wave
//    adds the staged rows in order, one column per lane, and one draws the work and applies the sums.  The serial chain
//    costs one add per duplicate.
//    The longest runs are started first and cut into narrower slices, i.e. fed by more blocks.
//  * medium (kTinyRun < duplicates <= kLongRun): one group of LPR lanes per run, kBatch rows in flight.
//  * short (<= kTinyRun): a group of LPR lanes (LPR*VEC floats = one row) owns a few consecutive unique keys
//    and sums their runs, all first loads of the group issued together.
#include <algorithm>
#include <type_traits>
#include "kernels.h"

namespace hctr {

// tuning knobs (overridable at compile time for experiments)
#ifndef HCTR_TILE_BATCH
#define HCTR_TILE_BATCH 8
#endif
#ifndef HCTR_LONG_BLOCKS
#define HCTR_LONG_BLOCKS 128
#endif
#ifndef HCTR_MED_BLOCKS
#define HCTR_MED_BLOCKS 512
#endif
constexpr int kPushBlock = 512;

constexpr int kBatch = HCTR_TILE_BATCH;   // short role: gradient rows in flight per group past the first two
constexpr int kInFlight = 16;             // long role: rows in flight per loader thread
constexpr int kSlice = kSliceColumns;     // long role: columns per block
constexpr int kLongBlocks = HCTR_LONG_BLOCKS;
constexpr int kMedBlocks = HCTR_MED_BLOCKS;

namespace {

__device__ __forceinline__ uint32_t div_up_dev(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

#ifndef HCTR_GRAD_NT
#define HCTR_GRAD_NT 1
#endif
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 f32x4_any __attribute__((aligned(4))); // at any 4-byte address
// the vectors of a row as they lie in memory (never a template argument: that drops the alignment from the type)
template <int VEC> struct RowMem { typedef f32x4 M; };
template <> struct RowMem<kOdd4> { typedef f32x4_any M; };
// The gradient row of batch position `pos`: the position itself, or with sum-pooled bags of `bag` consecutive
// positions the row of the position's bag (every key of a bag receives the bag's gradient).
// kPooled is a compile-time switch: the plain push must not pay for the division in its load pipelines.
template <bool kPooled> __device__ __forceinline__ uint32_t grad_row(uint32_t pos, const BagDiv &bag) {
  return kPooled ? bag(pos) : pos;
}

// The columns a lane moves at a time (see kOdd4 in kernels.h).  T: as the lane computes with them, a
// vector f32x4 or the four floats of a float4.  The medium role takes the latter: its two batches of vectors, each held in
// four registers in a row, left one register too few, and a push with scratch memory took a batch of 53 k keys 22.2 us
// instead of 20.4.  The short role takes vectors: 8.5 M uniform keys are pushed in 1027 us, with float4 in 1064.
template <typename T4, int VEC> struct Vec4 {
  typedef T4 T;
  typedef typename RowMem<VEC>::M M;
  static_assert(alignof(M) == (VEC == kOdd4 ? 4 : 16), "what the compiler may take for granted of a row's address");
  static __device__ __forceinline__ T zero() { return T{0.f, 0.f, 0.f, 0.f}; }
  static __device__ __forceinline__ void add(T &a, const T &b) { a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w; }
  static __device__ __forceinline__ T scale(const T &a, float s) { return T{a.x * s, a.y * s, a.z * s, a.w * s}; }
  static __device__ __forceinline__ T load(const float *p) { return of(*(const M *)p); }
  static __device__ __forceinline__ T load_once(const float *p) { return of(__builtin_nontemporal_load((const M *)p)); }
  static __device__ __forceinline__ void store_all(float *p, const T &a) { *(M *)p = to(a); }
  static __device__ __forceinline__ void store_all_away(float *p, const T &a) { __builtin_nontemporal_store(to(a), (M *)p); }

 private:
  // (by value: a reference to a row's vector would promise more alignment than it has)
  static __device__ __forceinline__ T of(f32x4 v) { return T{v.x, v.y, v.z, v.w}; }
  static __device__ __forceinline__ f32x4 to(const T &a) { return f32x4{a.x, a.y, a.z, a.w}; }
};
template <int VEC, typename T4 = f32x4> struct Vec;
template <typename T4> struct Vec<4, T4> : Vec4<T4, 4> {
  typedef Vec4<T4, 4> B;
  static __device__ __forceinline__ void store(float *p, const T4 &a, uint32_t) { B::store_all(p, a); }
  // a store past the caches: for rows another shard's kernel reads next
  static __device__ __forceinline__ void store_away(float *p, const T4 &a, uint32_t) { B::store_all_away(p, a); }
};
template <typename T4> struct Vec<kOdd4, T4> : Vec4<T4, kOdd4> {
  typedef Vec4<T4, kOdd4> B;
  // without the first `shared` columns, which the lane before writes (and, in a row of more than one round of the
  // group, may have updated before this lane reads them: what it computes for them is dropped)
  static __device__ __forceinline__ void store(float *p, const T4 &a, uint32_t shared) {
    if (!shared) {
      B::store_all(p, a);
    } else {
      if (shared < 2) p[1] = a.y;
      if (shared < 3) p[2] = a.z;
      p[3] = a.w;
    }
  }
  static __device__ __forceinline__ void store_away(float *p, const T4 &a, uint32_t shared) {
    if (!shared) {
      B::store_all_away(p, a);
    } else {
      if (shared < 2) __builtin_nontemporal_store(a.y, p + 1);
      if (shared < 3) __builtin_nontemporal_store(a.z, p + 2);
      __builtin_nontemporal_store(a.w, p + 3);
    }
  }
};
template <typename T4> struct Vec<1, T4> {
  typedef float T;
  static __device__ __forceinline__ T zero() { return 0.f; }
  static __device__ __forceinline__ void add(T &a, const T &b) { a += b; }
  static __device__ __forceinline__ T scale(const T &a, float s) { return a * s; }
  static __device__ __forceinline__ T load(const float *p) { return *p; }
  static __device__ __forceinline__ T load_once(const float *p) { return __builtin_nontemporal_load(p); }
  static __device__ __forceinline__ void store_all(float *p, const T &a) { *p = a; }
  static __device__ __forceinline__ void store(float *p, const T &a, uint32_t) { *p = a; }
  static __device__ __forceinline__ void store_away(float *p, const T &a, uint32_t) { __builtin_nontemporal_store(a, p); }
};

// A gradient row is read exactly once per step: it is loaded past the caches.  With sum-pooled bags (kPooled) a row
// is read once per key of its bag, so there it is loaded the ordinary way and the repeats hit the cache; and so it is
// in the long role (kAgain) where it shares its lines with its neighbours, see push_block.
template <typename R, bool kAgain> __device__ __forceinline__ typename R::T grad_load(const embed_t *p) { // R: a Vec
  return HCTR_GRAD_NT && !kAgain ? R::load_once(p) : R::load(p);
}

// The version / update counters of unique rank u and its entry among the pushed rows (gradient_index_kernel,
// generate_query.cu:51-83).  type: the update type of generate_query.cu:18-25; q: the row's place among the pushed rows.
template <typename K>
__device__ __forceinline__ void move_counters(const TableView &t, int id_bits, const BatchView &p, const PushArgs &a,
                                              uint32_t u, slot_t o, int type, uint32_t q) {
  version_t cnt = (version_t)(p.run_start[u + 1] - p.run_start[u]);
  if (type == 1) t.ver[o] += cnt;
  else if (type >= 2) {
    version_t up = t.upd[o] + cnt;
    if (type == 2) {
      cnt = up;
      up = 0;
      t.ver[o] += cnt;
    }
    t.upd[o] = up;
  }
  if (type == 0 || type == 2) { // the rows the plan marks as pushed
    a.g_idx[q] = (index_t)(((const K *)p.ukey)[u] & (K)(((uint64_t)1 << id_bits) - 1));
    a.g_cnt[q] = cnt;
  }
}

// Applies the finished sum of unique rank u (already multiplied by -lr) to column(s) `col`.  Update types as in
// generate_query.cu:18-25.  The counters of the row move in the last blocks of the launch.
template <typename R, typename K> // R: a Vec
__device__ __forceinline__ void apply_row(const TableView &t, int id_bits, const BatchView &p, const PushArgs &a,
                                          uint32_t u, typename R::T s, uint32_t col, uint32_t shared = 0) {
  typedef typename R::T V;
  const slot_t o = p.uoff[u];
  const uint32_t W = t.width;
  if (t.nrank == 1) { // every key is owned and resident: type 1 only
    embed_t *e = t.emb + (size_t)o * W + col;
    V cur = R::load(e);
    R::add(cur, s);
    R::store(e, cur, shared);
    return;
  }
  const bool need = a.need[u] != 0;
  const int type = o == kNoSlot ? 0 : ((uint32_t)o >= t.n_cached ? 1 : (need ? 2 : 3));
  const uint32_t q = a.prefix[u];
  if (type != 0) {
    embed_t *e = t.emb + (size_t)o * W + col;
    V cur = R::load(e);
    R::add(cur, s);
    R::store(e, cur, shared);
  } else {
    R::store_away(a.g_val + (size_t)q * W + col, s, shared);
  }
  if (type >= 2) {
    embed_t *g = t.pend + (size_t)o * W + col;
    V pg = R::load(g);
    R::add(pg, s);
    if (type == 2) {
      R::store_away(a.g_val + (size_t)q * W + col, pg, shared);
      pg = R::zero();
    }
    R::store(g, pg, shared);
  }
}

// ---- short role ----------------------------------------------------------------------------------------
// A group of LPR lanes owns kRunsPerGroup consecutive unique ranks and sums every run among them that is not
// long.  Everything the group needs first is requested before anything is waited for: the run bounds and
// resident offsets, then the destination rows, the first two gradient-row indices of every run and those
// gradient rows.  Nine runs out of ten are finished by that; longer ones continue eight rows at a time.
// Three runs per group: alone the kernel is 1 % faster with two, next to the index kernels of the following batch on the
// second stream it is 3 % faster with three (blocks that live longer lose less to what is scheduled beside them); from
// four on registers spill.
#ifndef HCTR_RUNS_PER_GROUP
#define HCTR_RUNS_PER_GROUP 3
#endif
constexpr int kRunsPerGroup = HCTR_RUNS_PER_GROUP;
constexpr int kHead = 2; // occurrences per run fetched up front
constexpr int kTail = 6; // occurrences per step after those

template <int VEC, int LPR, typename K, bool kSingle, bool kPooled>
__device__ __forceinline__ void short_role(const TableView &t, int id_bits, const BatchView &p, const PushArgs &a,
                                           uint32_t block, uint32_t U) {
  typedef typename Vec<VEC>::T V;
  constexpr int G = kRunsPerGroup;
  constexpr int kGroups = kPushBlock / LPR;
  const uint32_t W = t.width, n = p.n;
  const uint32_t u0 = (block * kGroups + threadIdx.x / LPR) * G;
  if (u0 >= U) return;
  const uint32_t gl = threadIdx.x % LPR;
  const uint32_t *__restrict__ run_start = p.run_start;
  const uint32_t *__restrict__ sorted_arg = p.sorted_arg;
  const embed_t *__restrict__ grad = a.grad;
  uint32_t rs[G + 1];
  slot_t off[G];
#pragma unroll
  for (int i = 0; i <= G; i++) rs[i] = run_start[min(u0 + i, U)];
#pragma unroll
  for (int i = 0; i < G; i++) off[i] = p.uoff[min(u0 + i, U - 1)];
  // several shards: the update type of every run (generate_query.cu:18-25) and its place among the pushed rows
  int type[G];
  uint32_t q[G];
  if (!kSingle) {
    uint32_t nd[G];
#pragma unroll
    for (int i = 0; i < G; i++) {
      nd[i] = a.need[min(u0 + i, U - 1)];
      q[i] = a.prefix[min(u0 + i, U - 1)];
    }
#pragma unroll
    for (int i = 0; i < G; i++)
      type[i] = off[i] == kNoSlot ? 0 : ((uint32_t)off[i] >= t.n_cached ? 1 : (nd[i] ? 2 : 3));
  }
  const float neg_lr = t.neg_lr;

  for (uint32_t c0 = 0; c0 < W; c0 += LPR * kCols<VEC>) {
    const uint32_t due = c0 + gl * kCols<VEC>, col = lane_col<VEC>(due, W), shared = due - col;
    const bool active = due < W;
    uint32_t len[G];
    bool mine[G];
    V e[G], pg[G];
    uint32_t si[G][kHead];
    V v[G][kHead];
#pragma unroll
    for (int i = 0; i < G; i++) {
      len[i] = rs[i + 1] - rs[i];
      mine[i] = u0 + i < U && len[i] <= kTinyRun && active;
    }
    // the rows the sums will be added to are requested before the gradient rows, not after the sums are done
#pragma unroll
    for (int i = 0; i < G; i++) {
      e[i] = Vec<VEC>::zero();
      if (mine[i] && (kSingle || type[i] != 0)) e[i] = Vec<VEC>::load(t.emb + (size_t)off[i] * W + col);
    }
    if (!kSingle) {
#pragma unroll
      for (int i = 0; i < G; i++) {
        pg[i] = Vec<VEC>::zero();
        if (mine[i] && type[i] >= 2) pg[i] = Vec<VEC>::load(t.pend + (size_t)off[i] * W + col);
      }
    }
#pragma unroll
    for (int i = 0; i < G; i++)
#pragma unroll
      for (int k = 0; k < kHead; k++) si[i][k] = grad_row<kPooled>(sorted_arg[min(rs[i] + k, n - 1)], a.bag);
#pragma unroll
    for (int i = 0; i < G; i++)
#pragma unroll
      for (int k = 0; k < kHead; k++) {
        v[i][k] = Vec<VEC>::zero();
        if (mine[i] && (uint32_t)k < len[i]) v[i][k] = grad_load<Vec<VEC>, kPooled>(grad + (size_t)si[i][k] * W + col);
      }
    V acc[G];
#pragma unroll
    for (int i = 0; i < G; i++) { // heads of all runs first: their registers are free before the tails start
      acc[i] = Vec<VEC>::zero();  // the reference starts every sum from 0
#pragma unroll
      for (int k = 0; k < kHead; k++)
        if (mine[i] && (uint32_t)k < len[i]) Vec<VEC>::add(acc[i], v[i][k]);
    }
#pragma unroll
    for (int i = 0; i < G; i++) {
      if (!mine[i]) continue;
      // the rest of the run (at most kTinyRun - kHead rows), in order, kTail rows at a time
      for (uint32_t j = rs[i] + kHead; j < rs[i + 1]; j += kTail) {
        uint32_t sj[kTail];
        V x[kTail];
#pragma unroll
        for (int k = 0; k < kTail; k++) sj[k] = grad_row<kPooled>(sorted_arg[min(j + k, rs[i + 1] - 1)], a.bag);
#pragma unroll
        for (int k = 0; k < kTail; k++) x[k] = grad_load<Vec<VEC>, kPooled>(grad + (size_t)sj[k] * W + col);
#pragma unroll
        for (int k = 0; k < kTail; k++)
          if (j + k < rs[i + 1]) Vec<VEC>::add(acc[i], x[k]);
      }
      const V scaled = Vec<VEC>::scale(acc[i], neg_lr);
      if (kSingle) {
        V r = e[i];
        Vec<VEC>::add(r, scaled);
        Vec<VEC>::store(t.emb + (size_t)off[i] * W + col, r, shared); // the version counters move in the last blocks of the launch
      } else {
        // the same updates as apply_row(), with the rows already here
        if (type[i] != 0) {
          V r = e[i];
          Vec<VEC>::add(r, scaled);
          Vec<VEC>::store(t.emb + (size_t)off[i] * W + col, r, shared);
        } else {
          Vec<VEC>::store_away(a.g_val + (size_t)q[i] * W + col, scaled, shared);
        }
        if (type[i] >= 2) {
          V g = pg[i];
          Vec<VEC>::add(g, scaled);
          if (type[i] == 2) {
            Vec<VEC>::store_away(a.g_val + (size_t)q[i] * W + col, g, shared);
            g = Vec<VEC>::zero();
          }
          Vec<VEC>::store(t.pend + (size_t)off[i] * W + col, g, shared);
        }
      }
    }
  }
}

// ---- medium role ---------------------------------------------------------------------------------------
// Runs between kTinyRun and kLongRun occurrences: one group of LPR lanes per run of the list (groups stride
// over it).  The group first copies the run's gradient-row indices into LDS with one coalesced load, so that no
// later load waits for an index; then two batches of kBatch gradient rows are kept in flight while the rows are
// added in order.
template <int VEC, int LPR, typename K, bool kSingle, bool kPooled>
__device__ __forceinline__ void medium_role(const TableView &t, int id_bits, const BatchView &p, const PushArgs &a,
                                            uint32_t *lds_idx, uint32_t block, uint32_t nblocks) {
  typedef Vec<VEC, float4> R;
  typedef typename R::T V;
  constexpr int kGroups = kPushBlock / LPR;
  const uint32_t W = t.width;
  const uint32_t gl = threadIdx.x % LPR;
  uint32_t *my_idx = lds_idx + (threadIdx.x / LPR) * kLongRun; // this group's slice of the index staging area
  const uint32_t n_med = p.d_nlong[kMedCount];
  const uint32_t *__restrict__ sorted_arg = p.sorted_arg;
  const embed_t *__restrict__ grad = a.grad;
  const float neg_lr = t.neg_lr;
  for (uint32_t item = block * kGroups + threadIdx.x / LPR; item < n_med; item += nblocks * kGroups) {
    const uint32_t u = p.med_list[item];
    const uint32_t lo = p.run_start[u], hi = p.run_start[u + 1];
    const uint32_t len = hi - lo; // <= kLongRun
    const slot_t off = p.uoff[u];
    for (uint32_t q = gl; q < len; q += LPR) my_idx[q] = grad_row<kPooled>(sorted_arg[lo + q], a.bag);
    // a group never spans waves: the LDS writes above are ordered before the reads below in hardware; the
    // fence keeps the compiler from moving them
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (uint32_t c0 = 0; c0 < W; c0 += LPR * kCols<VEC>) {
      const uint32_t due = c0 + gl * kCols<VEC>, col = lane_col<VEC>(due, W), shared = due - col;
      const bool active = due < W;
      const embed_t *gcol = grad + (active ? col : 0);
      V e = R::zero();
      if (kSingle && active) e = R::load(t.emb + (size_t)off * W + col);
      V acc = R::zero();
      V xa[kBatch], xb[kBatch];
      auto fetch = [&](V(&x)[kBatch], uint32_t q0) { // rows q0 .. q0+kBatch-1 of the run (clamped to its end)
#pragma unroll
        for (int k = 0; k < kBatch; k++) x[k] = grad_load<R, kPooled>(gcol + (size_t)my_idx[min(q0 + k, len - 1)] * W);
      };
      auto add = [&](const V(&x)[kBatch], uint32_t q0) {
#pragma unroll
        for (int k = 0; k < kBatch; k++)
          if (q0 + k < len) R::add(acc, x[k]);
      };
      fetch(xa, 0);
      for (uint32_t q = 0; q < len; q += 2 * kBatch) {
        if (q + kBatch < len) fetch(xb, q + kBatch);
        add(xa, q);
        if (q + 2 * kBatch < len) fetch(xa, q + 2 * kBatch);
        if (q + kBatch < len) add(xb, q + kBatch);
      }
      if (!active) continue;
      const V scaled = R::scale(acc, neg_lr);
      if (kSingle) {
        R::add(e, scaled);
        R::store(t.emb + (size_t)off * W + col, e, shared); // versions: bump_versions
      } else {
        apply_row<R, K>(t, id_bits, p, a, u, scaled, col, shared);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier(); // the staging area is rewritten for the next run
  }
}

// ---- long role -----------------------------------------------------------------------------------------
// A block works on ONE column slice (CS columns) of a bundle of long runs at a time and treats the bundle as one
// stream of chunks, so that the loads of the next run are in flight while the current one is summed.  Runs are
// listed by length class, longest first; a bundle is 1..kTable runs of one class holding at least ~2048
// occurrences.  Tickets (bundle, slice) are handed out through one counter per group of blocks that share slices.
//
// Fast path (slices of 16, 32 or 64 columns, CSC).  One wave sums, one draws the tickets and applies the sums, the other six
// ("loaders") move gradient rows global -> registers -> LDS.
//  * The lanes of the summing wave are kSets sets of one lane per column of the slice, and a chunk is 96 rows for each set.  The
//    wave reads a chunk in two halves of 12 x 16 bytes per lane, four rows of the lane's column at a time, and adds one half
//    while the next one is on its way.  A sum never leaves its wave (it goes from set to set by a swap of lanes).
//  * For that, four neighbouring rows of a column lie side by side in LDS.  A loader lane has just these rows (four columns of
//    four neighbouring rows of the chunk) in its registers and stores one column of them at a time; where a column lies in a
//    group of rows (column_slot) makes both sides touch every bank equally often.
//  * The waves never meet at a barrier.  Loaders count the parts of a chunk they have written, the summing wave the chunks it has
//    read, and whoever needs a slot full or empty looks at the count.
//  * The rows the sums are added to (with several shards also the plan's words and the pending rows) are requested by the wave that
//    draws, when a bundle begins, and are there when its sums arrive.  It draws the next ticket kDrawAhead chunks before a bundle
//    ends: drawn at its beginning, tickets lay with the blocks that had the longest runs while others ran out of work.
// What bounds it: the chain.  Adds alone take 4.3 cycles per row, the 24 reads of a chunk of 192 rows 6 to 12 cycles each, the
// counts about 150 per chunk; 7.4 cycles per row in all at 2.3 GHz, 2.5 more where the rows come from HBM and not from the
// last-level cache.  Two waves that took turns at reading and adding, with a barrier per chunk, took 7.6 and 9.9; what is gained
// beyond the chain is the end of the launch, where blocks now finish together.  The push of 8.5 M keys of 64 floats, Zipf 1.4:
// pooled by tens 480 -> 425 us, plain 624 -> 565; of 1.7 M keys of 128 floats 247 -> 240.  Steps of the first two
// 7 and 6 % shorter, of the last within their spread (2 %) the same, of 195 k keys of 37 floats 5 %.  Measured without gain: one read between every few adds (14 cycles each), a raised
// priority for the summing wave, 20 instead of 16 vectors in flight, 192 blocks, barriers instead of counts.
// Generic path (CSC 0; rows of less than four floats): seven loader waves and one that reads and adds, eight rows at a time,
// three slots.
constexpr int kTable = 16;      // runs per bundle at most
constexpr int kHalfGroups = 12; // groups of four rows a lane of the summing wave holds of half a chunk
constexpr int kSlotVectors = 2 * kHalfGroups * kWave; // 16-byte vectors of a slot of the ring: a chunk, whatever the slice
constexpr int kSlotsFast = 2, kSlotsGeneric = 3; // LDS slots
// Chunks before the end of a bundle at which the next ticket is drawn.  4, 16 and 64: the push of 195 k keys of 37 floats, Zipf 1.4, 23.8,
// 23.3 and 27.4 us, of 1.04 M of 64 floats, 1.1, 96, 93 and 95, of 5.3 M of 17 floats, 1.2, 539, 538 and 539.
constexpr uint32_t kDrawAhead = 16;
// the value of the lanes 16 / 32 below (up) or above (!up), for the lanes of the other half of a pair of halves
template <int D, bool up> __device__ __forceinline__ float from_half(float x) {
  const uint32_t v = __float_as_uint(x);
  if constexpr (D == 32) return __uint_as_float(__builtin_amdgcn_permlane32_swap(v, v, false, false)[up ? 0 : 1]);
  else return __uint_as_float(__builtin_amdgcn_permlane16_swap(v, v, false, false)[up ? 0 : 1]);
}
// The sets of a summing wave in the order in which they hold the rows of the first half of a chunk; the second half goes back.
// Neighbours differ in one bit, so that a swap of halves of the wave moves a sum on.
__host__ __device__ constexpr uint32_t set_at(uint32_t t, bool second, int sets) {
  const uint32_t k = second ? sets - 1 - t : t;
  return k ^ (k >> 1);
}

// This wave's LDS operations are done.  A barrier waits for them by itself, but where it is the first thing in a loop the compiler
// of ROCm 7.2 drops that wait, having seen nothing outstanding in front of the loop: what comes around the loop is
// outstanding.  (tests/test_kernel_resources.py looks for such barriers in every kernel.)
__device__ __forceinline__ void lds_done() { __builtin_amdgcn_s_waitcnt(0xc07f); } // lgkmcnt(0), nothing else

// the value of lane Q of the quad
template <int Q> __device__ __forceinline__ uint64_t of_quad(uint64_t v) {
  constexpr int kPerm = Q * 0x55;
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, kPerm, 0xf, 0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), kPerm, 0xf, 0xf, true);
  return (uint64_t)hi << 32 | lo;
}
// a value that is the same in every lane, moved to a scalar register
__device__ __forceinline__ uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

// Counts in LDS that the waves of a block poll instead of meeting at a barrier.  What a count stands for is done when it moves
// (the caller waits for its LDS operations first), and what follows it is not begun before it is seen.
__device__ __forceinline__ uint32_t peek(const uint32_t *count) { return __hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
__device__ __forceinline__ void wait_until(const uint32_t *count, uint32_t at_least) {
  while ((int)(uni(peek(count)) - at_least) < 0) __builtin_amdgcn_s_sleep(1);
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ void tell(uint32_t *count, uint32_t value) {
  asm volatile("" ::: "memory");
  if (threadIdx.x % kWave == 0) __hip_atomic_store(count, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void tell_add(uint32_t *count) {
  asm volatile("" ::: "memory");
  if (threadIdx.x % kWave == 0) (void)__hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// the number of long runs of class c, of which lane c has it
__device__ __forceinline__ uint32_t count_of(uint32_t counts, int c) { return (uint32_t)__builtin_amdgcn_readlane((int)counts, c); }

// log2 of the runs per bundle: classes halve in length -- one run of 2048 or more, 2 of 1024.., 4, 8, 16; `shrink` halves that
// (down to single runs) for batches with few long runs
__device__ __forceinline__ int bundle_log(int cls, int shrink) { return max(min(cls - 6, 4) - shrink, 0); }
static_assert(kTable == 1 << 4, "the most runs per bundle");

// CSC: columns per slice if known at compile time, else 0; kAgain: the lines a gradient row lies in are read again
template <int VEC, typename K, int CSC, bool kPooled, bool kAgain>
__device__ __forceinline__ void long_role(const TableView &t, int id_bits, const BatchView &p, const PushArgs &a,
                                          float *lds, uint4 *tables, uint32_t *shared, float *sums,
                                          uint32_t counts, int c_lo, int c_hi, uint32_t bidx, uint32_t nblk, uint32_t *counters) {
  typedef typename Vec<VEC>::T V;
  constexpr uint32_t C = kCols<VEC>;
  constexpr uint32_t kOthers = CSC ? 2 : 1; // waves that do not load
  constexpr int kLoaders = kPushBlock - kOthers * kWave;
  const uint32_t W = t.width;
  static_assert((CSC == 0) == (VEC == 1), "the generic path is for rows of less than four floats, one slice each");
  const uint32_t CS = CSC ? (uint32_t)CSC : W;
  const uint32_t lanes = CSC ? CS / C : W <= 2 ? W : 4; // loader lanes per row slice, a power of two
  constexpr int kSets = CSC ? kWave / CSC : 1;
  constexpr int kRPT = CSC ? 4 : 2;        // rows per loader thread and chunk
  constexpr int kDepth = kInFlight / kRPT; // chunks in flight per loader thread
  const uint32_t CR = kLoaders / lanes * kRPT; // rows per chunk
  constexpr uint32_t kHalfRows = 4 * kHalfGroups * kSets;
  static_assert(!CSC || 2 * kHalfRows == kLoaders / (CSC / C) * kRPT, "a chunk of the fast path is whole loads");
  const uint32_t slices = (W + CS - 1) / CS;
  const float neg_lr = t.neg_lr;
  const uint32_t wave = uni(threadIdx.x / kWave);
  const uint32_t *__restrict__ sorted_arg = p.sorted_arg;

  // tickets of this block's group: (bundle, slice) with the bundle changing slowest, so the longest runs go first
  const uint32_t share = min(min(slices, nblk), (uint32_t)kTicketLanes);
  const uint32_t lane_id = bidx % share;
  const uint32_t n_sl = (slices - lane_id + share - 1) / share; // slices lane_id, lane_id + share, ...
  const uint32_t group_blocks = (nblk - lane_id + share - 1) / share; // blocks drawing from this counter
  // Lane c looks after class c of the runs.  (In scalar registers, twelve of them, some of the loaders' were spilled.)
  const int class_of_lane = threadIdx.x % kWave;
  counts = class_of_lane >= c_lo && class_of_lane < c_hi ? counts : 0u;
  if (!__ballot(counts != 0)) return;
  // A block streams a bundle at the pace its rows in flight allow (a few ns per occurrence), whatever the other
  // blocks do: a small batch, whose long runs make fewer tickets than there are blocks to draw them, gets smaller
  // bundles until every block has work or every bundle is a single run.  Every block computes the same value.
  uint32_t nbundles, of_class; // bundles; of this lane's class
  int shrink = 0;
  for (;;) {
    const int lg = bundle_log(class_of_lane, shrink);
    of_class = (counts + (1u << lg) - 1) >> lg;
    nbundles = 0;
#pragma unroll
    for (int c = 0; c < kLongBuckets; c++) nbundles += count_of(of_class, c);
    if (shrink == 4 || nbundles * slices >= 2 * nblk) break;
    shrink++;
  }
  const uint32_t tickets = nbundles * n_sl;

  // one wave draws a ticket and leaves its bundle in set `to`: descriptors of the runs (one lane per run, which keeps its own
  // in `mine`), number of runs, chunks and the slice
  auto draw = [&](uint32_t to, uint4 &mine) {
    const uint32_t lane = threadIdx.x % kWave;
    uint32_t tk = 0;
    if (lane == 0) tk = atomicAdd(counters + lane_id, 1u);
    tk = (uint32_t)__builtin_amdgcn_readfirstlane((int)tk);
    if (tk >= tickets) {
      // Every block of the group draws exactly one ticket past the end.  The block that draws the last of them
      // knows that nobody will touch the counter again in this launch and puts it back to zero, so that the same
      // batch can be pushed again (push_pull twice without a preprocess in between applies the gradient twice,
      // csrc/core/hetu_gpu_table.cu:9-41).
      if (lane == 0 && tk == tickets + group_blocks - 1) atomicExch(counters + lane_id, 0u);
      if (lane == 0) shared[to * 4] = 0;
      return;
    }
    uint32_t bundle = tk / n_sl;
    int cls = 0;
    uint32_t run0 = 0, runs = 0;
    asm volatile("" : "+v"(of_class)); // asked anew, not kept in scalar registers
#pragma unroll
    for (int c = 0; c < kLongBuckets; c++) {
      const uint32_t nb = count_of(of_class, c);
      if (!runs) {
        if (bundle < nb) {
          const int lg = bundle_log(c, shrink);
          cls = c;
          run0 = bundle << lg;
          runs = min(1u << lg, count_of(counts, c) - run0);
        } else {
          bundle -= nb;
        }
      }
    }
    uint32_t chunks = 0;
    if (lane < runs) {
      mine = p.long_list[(size_t)cls * p.long_cap + run0 + lane]; // rank, first position, length, offset
      chunks = (mine.z + CR - 1) / CR;
      tables[to * kTable + lane] = mine;
    }
#pragma unroll
    for (int d = kTable / 2; d; d >>= 1) chunks += __shfl_down(chunks, d);
    if (lane == 0) {
      shared[to * 4] = runs;
      shared[to * 4 + 1] = chunks;
      shared[to * 4 + 2] = lane_id + (tk % n_sl) * share;
    }
  };

  // Whole rounds run without a condition inside: with one, the compiler must assume that loads may have been
  // skipped and waits for nearly everything in flight before each use.
  auto rounds = [&](uint32_t G, auto &&step) {
    uint32_t g0 = 0;
    for (; g0 + kDepth <= G; g0 += kDepth) {
#pragma unroll
      for (int k = 0; k < kDepth; k++) step(k);
    }
#pragma unroll
    for (int k = 0; k < kDepth; k++)
      if (g0 + k < G) step(k); // uniform over the block: all waves make the same number of barriers
  };

  __syncthreads(); // of the runs before these
  if constexpr (CSC != 0) {
    f32x4 *const ring = (f32x4 *)lds;
    constexpr uint32_t kColVecs = CSC / 4; // column vectors of a row slice
    // Where in a group of four rows the vector of column 4 * v + k of the slice lies: neighbours in v side by side, and the k turned
    // by the group's number where the group is shorter than a round of all banks.
    auto column_slot = [](uint32_t v, uint32_t k, uint32_t group) { return (k ^ (group & (kSets - 1))) * kColVecs + v; };
    // the column of the slice that lane position `pl` of a set sums
    auto column_of = [](uint32_t pl) { return pl % kColVecs * 4 + pl / kColVecs; };
    // What the waves tell each other, all of it counted from the start of the role: bundles drawn, bundles summed, bundles whose sums
    // have been fetched, chunks read, and per slot the loader waves that have written their part of a chunk there.  (One count for both slots would not do: a wave may
    // be done with the next chunk while another is not with this one.)  Bundle number b is in set b % 2, chunk number c in
    // slot c % 2.
    uint32_t *const drawn = shared + 8, *const summed = shared + 9, *const fetched = shared + 10, *const taken = shared + 11,
                   *const written = shared + 12;
    constexpr uint32_t kLoaderWaves = kLoaders / kWave;
    auto all_wrote = [](uint32_t chunk) { return (chunk / 2 + 1) * kLoaderWaves; };
    if (threadIdx.x < 6) shared[8 + threadIdx.x] = 0;
    lds_done();
    __syncthreads();
    if (wave % 4) {
      // ---------------- loaders ----------------
      uint32_t lt = threadIdx.x - (wave < 4 ? 1 : 2) * kWave; // loader thread number
      asm volatile("" : "+v"(lt)); // what follows from it is worked out here and takes no registers of the other waves
      const uint32_t group = lt / kColVecs, my_lane = lt % kColVecs; // the group of four rows of a chunk, the column vector
      uint32_t slot_of[4];
#pragma unroll
      for (uint32_t k = 0; k < 4; k++) slot_of[k] = group * CSC + column_slot(my_lane, k, group);
      // Every quad of lanes works out where its group's four rows lie, one row per lane: in every lane for itself that kept the
      // loaders' SIMDs busy longer than the adds take.
      const uint32_t my_row = group * 4 + lt % 4;
      uint32_t idx[kDepth];
      V val[kDepth][kRPT];
      // The cursor of the index stage, 2 * kDepth chunks ahead of the LDS stage.  Loads are unconditional, so that kDepth chunks stay
      // in flight per thread: positions past the end of a run re-read its last row (never summed), and so do the chunks past the
      // end of the bundle.
      uint32_t runs = 0, run = 0, clo = 0, len = 0, first = 0, at = 0; // at: chunks written, in all bundles
      const uint4 *table = tables;
      const embed_t *base = a.grad;
      auto open_run = [&]() {
        const uint4 m = table[run];
        clo = uni(m.y), len = uni(m.z), first = 0;
      };
      auto read_index = [&](int k) {
        const uint32_t from = min(first, len - 1), last = min(CR, len - from) - 1;
        idx[k] = sorted_arg[clo + from + min(my_row, last)];
        first += CR;
        if (first >= len) {
          if (run + 1 < runs) run++, open_run();
          else first = len;
        }
      };
      auto find_rows = [&](int k, const embed_t *(&from)[kRPT]) { // (the bag of a position where it is read would wait for it)
        const uint64_t off = (uint64_t)grad_row<kPooled>(idx[k], a.bag) * (W * 4);
        from[0] = (const embed_t *)((const char *)base + of_quad<0>(off));
        from[1] = (const embed_t *)((const char *)base + of_quad<1>(off));
        from[2] = (const embed_t *)((const char *)base + of_quad<2>(off));
        from[3] = (const embed_t *)((const char *)base + of_quad<3>(off));
      };
      auto read_rows = [&](int k, const embed_t *const (&from)[kRPT]) {
#pragma unroll
        for (int q = 0; q < kRPT; q++) val[k][q] = grad_load<Vec<VEC>, kAgain>(from[q]);
      };
      for (uint32_t bundle = 0;; bundle++) {
        wait_until(drawn, bundle + 1);
        const uint32_t cur = bundle & 1, G = uni(shared[cur * 4 + 1]);
        runs = uni(shared[cur * 4]);
        if (!runs) break;
        const uint32_t due = uni(shared[cur * 4 + 2]) * CSC + my_lane * C; // first column of this lane's vector
        base = a.grad + (due < W ? lane_col<VEC>(due, W) : 0u);
        table = tables + cur * kTable, run = 0;
        open_run();
#pragma unroll
        for (int k = 0; k < kDepth; k++) read_index(k);
#pragma unroll
        for (int k = 0; k < kDepth; k++) {
          const embed_t *from[kRPT];
          find_rows(k, from);
          read_rows(k, from);
          read_index(k); // in the order of the rounds below: the compiler waits for what either way into them has in flight
        }
        // val[k] holds the chunk that is written next and idx[k] the row indices of the one kDepth behind it
        rounds(G, [&](int k) {
          const embed_t *from[kRPT];
          find_rows(k, from);
          wait_until(taken, at - 1); // the chunk that was in this slot has been read (before the first two: -1 and 0)
          f32x4 *sp = ring + (at & 1) * kSlotVectors;
#pragma unroll
          for (int c = 0; c < 4; c++) sp[slot_of[c]] = f32x4{val[k][0][c], val[k][1][c], val[k][2][c], val[k][3][c]};
          read_rows(k, from);
          lds_done();
          tell_add(written + (at & 1)); // this wave's part of the chunk is in its slot
          at++;
          read_index(k);
        });
      }
    } else if (wave == 0) {
      // ---------------- the summing wave: rows strictly in order ----------------
      uint32_t lane = threadIdx.x % kWave;
      asm volatile("" : "+v"(lane)); // what follows from it is worked out here and takes no registers of the loaders
      const uint32_t set = lane / CSC, pl = lane % CSC;
      // where this lane's rows of either half start, and the t-th set of each
      uint32_t turn = 0;
#pragma unroll
      for (uint32_t k = 0; k < (uint32_t)kSets; k++)
        if (set_at(k, false, kSets) == set) turn = k;
      const uint32_t base0 = turn * (kHalfGroups * CSC), base1 = (kHalfGroups * kSets + (kSets - 1 - turn) * kHalfGroups) * CSC;
      typedef f32x4 Half[kHalfGroups];
      auto add4 = [](const f32x4 &v, float &acc) { acc += v[0], acc += v[1], acc += v[2], acc += v[3]; };
      auto pass = [](auto from, auto second, float &acc) { // the sum goes on to the next set
        constexpr bool kSecond = decltype(second)::value;
        constexpr uint32_t s = set_at(decltype(from)::value, kSecond, kSets), to = set_at(decltype(from)::value + 1, kSecond, kSets);
        acc = from_half<(s ^ to) * CSC, (s < to)>(acc);
      };
      // adds the n rows of half a chunk; returns the set that then holds the sum
      auto add_half = [&](auto second, const Half &x, uint32_t n, const f32x4 &rest, float &acc) -> uint32_t {
        auto pass_on = [&](auto from) { pass(from, second, acc); };
        auto add_set = [&]() {
#pragma unroll
          for (int i = 0; i < kHalfGroups; i++) add4(x[i], acc);
        };
        auto add_first = [&](uint32_t m) { // the first m < 4 * kHalfGroups rows of the set; the last m % 4 lie apart
#pragma unroll
          for (int i = 0; i < kHalfGroups - 1; i++)
            if (m >= 4u * (i + 1)) add4(x[i], acc);
          if (m % 4 > 0) acc += rest[0];
          if (m % 4 > 1) acc += rest[1];
          if (m % 4 > 2) acc += rest[2];
        };
        constexpr uint32_t kSetRows = 4 * kHalfGroups;
        uint32_t done = 0; // sets whose rows have all been added
        if (n >= kSetRows) {
          add_set(), done = 1;
          if constexpr (kSets > 1) {
            if (n >= 2 * kSetRows) {
              pass_on(std::integral_constant<uint32_t, 0>()), add_set(), done = 2;
              if constexpr (kSets > 2) {
                if (n >= 3 * kSetRows) {
                  pass_on(std::integral_constant<uint32_t, 1>()), add_set(), done = 3;
                  if (n == 4 * kSetRows) pass_on(std::integral_constant<uint32_t, 2>()), add_set(), done = 4;
                }
              }
            }
          }
        }
        const uint32_t over = n - done * kSetRows;
        if (over) {
          if constexpr (kSets > 1) {
            if (done == 1) pass_on(std::integral_constant<uint32_t, 0>());
            if constexpr (kSets > 2) {
              if (done == 2) pass_on(std::integral_constant<uint32_t, 1>());
              if (done == 3) pass_on(std::integral_constant<uint32_t, 2>());
            }
          }
          add_first(over);
          done++;
        }
        return set_at(done - 1, decltype(second)::value, kSets);
      };
      uint32_t at_chunk = 0; // chunks read, in all bundles
      for (uint32_t bundle = 0;; bundle++) {
        wait_until(drawn, bundle + 1);
        const uint32_t cur = bundle & 1;
        const uint32_t runs = uni(shared[cur * 4]), G = uni(shared[cur * 4 + 1]), slice = uni(shared[cur * 4 + 2]);
        if (!runs) break;
        const uint4 *table = tables + cur * kTable;
        // Where the lane's column lies: where it is due, but for the columns of the last lane of a row at any address, which starts
        // at column W - 4.
        const uint32_t place = column_of(pl), mycol = slice * CSC + place;
        const uint32_t at = VEC == kOdd4 && mycol < W ? overlapped_place(place, mycol, W) : place;
        uint32_t col[kSets]; // in the groups of number 0, 1, ... mod kSets
#pragma unroll
        for (uint32_t k = 0; k < (uint32_t)kSets; k++) col[k] = column_slot(at / 4, at % 4, k);
        auto read_half = [&](Half &x, const f32x4 *sp) {
          const f32x4 *from[kSets];
#pragma unroll
          for (int k = 0; k < kSets; k++) {
            uint32_t first = (uint32_t)(sp - ring) + col[k];
            asm volatile("" : "+v"(first)); // one address and 12 offsets, not 12 addresses kept in registers for the next time
            from[k] = ring + first;
          }
#pragma unroll
          for (int i = 0; i < kHalfGroups; i++) x[i] = from[i % kSets][i * CSC];
        };
        // a whole half is added from x while the next one is read into y
        auto add_reading = [&](auto second, const Half &x, Half &y, const f32x4 *sp, float &acc, auto &&late) {
          auto one_set = [&](auto turn) {
            constexpr int t = decltype(turn)::value;
#pragma unroll
            for (int i = 0; i < kHalfGroups; i++) {
              add4(x[i], acc);
              if (t * kHalfGroups + i + 1 == kSets * kHalfGroups * 3 / 4) { // what was read has come by now
                asm volatile("" : "+v"(acc));
                late();
                __builtin_amdgcn_sched_barrier(0);
              }
            }
            if constexpr (t + 1 < kSets) pass(turn, second, acc);
          };
          read_half(y, sp);
          __builtin_amdgcn_sched_barrier(0);
          one_set(std::integral_constant<uint32_t, 0>());
          if constexpr (kSets > 1) one_set(std::integral_constant<uint32_t, 1>());
          if constexpr (kSets > 2) one_set(std::integral_constant<uint32_t, 2>()), one_set(std::integral_constant<uint32_t, 3>());
          asm volatile("" : "+v"(acc)); // the adds stay in front of what follows
          __builtin_amdgcn_sched_barrier(0);
        };
        Half x0, x1;
        f32x4 rest = {0.f, 0.f, 0.f, 0.f};
        float acc = 0.f; // the reference starts every sum from 0
        uint32_t j = 0, left = uni(table[0].z); // the run, and its rows that have not been read
        uint32_t n1 = 0, j1 = 0;  // rows of the second half that wait in x1, and their run ...
        bool ends1 = false;       // ... which they end
        auto finish = [&](uint32_t run, uint32_t holder) { // the sum of a run is complete
          if (set == holder) sums[run * CSC + pl] = acc;
          acc = 0.f;
        };
        auto slot = [&]() { return ring + (at_chunk & 1) * kSlotVectors; };
        auto chunk_taken = [&]() { // both halves are in registers, or will be in a moment
          at_chunk++;
          lds_done();
          tell(taken, at_chunk);
        };
        wait_until(fetched, bundle); // the sums of the bundle before (this one's first rows are on their way)
        const uint32_t end = at_chunk + G;
        while (at_chunk != end) {
          if (n1 == kHalfRows && !ends1) { // whole chunks that follow a whole one
            const uint32_t whole = left / CR;
            uint32_t seen = peek(written + (at_chunk & 1));
            for (uint32_t k = 0; k < whole; k++) {
              if ((int)(uni(seen) - all_wrote(at_chunk)) < 0) wait_until(written + (at_chunk & 1), all_wrote(at_chunk));
              asm volatile("" ::: "memory");
              const f32x4 *sp = slot();
              add_reading(std::true_type(), x1, x0, sp + base0, acc, []() {});
              add_reading(std::false_type(), x0, x1, sp + base1, acc, [&]() {
                chunk_taken(); // the loaders have to fill the slot before the chunk after the next is due
                seen = peek(written + (at_chunk & 1)); // here when the next chunk is due
              });
            }
            left -= whole * CR;
            if (!left) {
              ends1 = true;
              if (j + 1 < runs) left = uni(table[++j].z);
            }
            if (at_chunk == end) break;
          }
          wait_until(written + (at_chunk & 1), all_wrote(at_chunk));
          const f32x4 *sp = slot();
          const uint32_t rows = min(CR, left), n0 = min(rows, kHalfRows);
          read_half(x0, sp + base0);
          __builtin_amdgcn_sched_barrier(0);
          if (n1) {
            const uint32_t holder = add_half(std::true_type(), x1, n1, rest, acc);
            if (ends1) finish(j1, holder);
          }
          __builtin_amdgcn_sched_barrier(0);
          const uint32_t last_group = min(rows / 4, CR / 4 - 1); // of which the chunk may have less than four rows
          rest = sp[last_group * CSC + column_slot(at / 4, at % 4, last_group)];
          read_half(x1, sp + base1);
          __builtin_amdgcn_sched_barrier(0);
          const uint32_t holder = add_half(std::false_type(), x0, n0, rest, acc);
          n1 = rows - n0, j1 = j, ends1 = rows == left;
          if (ends1 && !n1) finish(j, holder);
          left -= rows;
          if (!left && j + 1 < runs) left = uni(table[++j].z);
          chunk_taken();
        }
        if (n1) finish(j1, add_half(std::true_type(), x1, n1, rest, acc));
        lds_done();
        tell(summed, bundle + 1);
      }
    } else {
      // ---------------- the wave that draws the tickets and applies the sums ----------------
      uint32_t lane = threadIdx.x % kWave;
      asm volatile("" : "+v"(lane));
      const uint32_t set = lane / CSC, pl = lane % CSC;
      constexpr int kRuns = kTable / kSets; // runs per set: number j * kSets + set of the bundle
      const bool direct = t.nrank == 1;     // every key is owned and resident; the version counters move elsewhere
      uint4 next = {0, 0, 0, 0};
      draw(0, next);
      lds_done();
      tell(drawn, 1);
      uint32_t end = 0; // chunks of the bundles up to this one
      for (uint32_t bundle = 0;; bundle++) {
        const uint32_t cur = bundle & 1;
        const uint32_t runs = uni(shared[cur * 4]), slice = uni(shared[cur * 4 + 2]);
        if (!runs) break;
        end += uni(shared[cur * 4 + 1]);
        const uint4 mine = next; // of run `lane` of the bundle
        const uint32_t mycol = slice * CSC + column_of(pl);
        const bool col_ok = mycol < W;
        // the rows the sums will be added to, all of them at once; they are here long before the sums
        uint32_t need = 0, q = 0;
        if (!direct && lane < runs) need = a.need[mine.x], q = a.prefix[mine.x];
        float row[kRuns], pend[kRuns];
        auto off_of = [&](int j) { return (slot_t)__shfl((int)mine.w, j * kSets + set); };
        auto works = [&](int j) { return col_ok && j * kSets + set < runs; };
        auto type_of = [&](int j) { // the update type of generate_query.cu:18-25
          const slot_t o = off_of(j);
          const bool nd = __shfl((int)need, j * kSets + set) != 0;
          return direct ? 1 : o == kNoSlot ? 0 : ((uint32_t)o >= t.n_cached ? 1 : (nd ? 2 : 3));
        };
#pragma unroll
        for (int j = 0; j < kRuns; j++) {
          row[j] = 0.f;
          const slot_t o = off_of(j);
          if (works(j) && (direct || o != kNoSlot)) row[j] = t.emb[(size_t)o * W + mycol];
        }
        if (!direct) {
#pragma unroll
          for (int j = 0; j < kRuns; j++) {
            pend[j] = 0.f;
            const slot_t o = off_of(j);
            if (works(j) && o != kNoSlot && (uint32_t)o < t.n_cached) pend[j] = t.pend[(size_t)o * W + mycol];
          }
        }
        // The next ticket is drawn when this bundle is nearly through: drawn at once, it would lie here while blocks with shorter
        // bundles run out of work.
        wait_until(taken, end - min(end, kDrawAhead));
        draw(cur ^ 1, next);
        lds_done();
        tell(drawn, bundle + 2);
        wait_until(summed, bundle + 1);
        float sum[kRuns];
#pragma unroll
        for (int j = 0; j < kRuns; j++) sum[j] = sums[(j * kSets + set) * CSC + pl];
        lds_done();
        tell(fetched, bundle + 1);
#pragma unroll
        for (int j = 0; j < kRuns; j++) {
          const slot_t o = off_of(j);
          const int type = type_of(j);
          const uint32_t at = (uint32_t)__shfl((int)q, j * kSets + set);
          if (!works(j)) continue;
          const float scaled = sum[j] * neg_lr;
          if (type != 0) t.emb[(size_t)o * W + mycol] = row[j] + scaled;
          else Vec<1>::store_away(a.g_val + (size_t)at * W + mycol, scaled, 0);
          if (type >= 2) {
            float g = pend[j] + scaled;
            if (type == 2) {
              Vec<1>::store_away(a.g_val + (size_t)at * W + mycol, g, 0);
              g = 0.f;
            }
            t.pend[(size_t)o * W + mycol] = g;
          }
        }
      }
    }
    lds_done();
  } else {
    // cursor of a loader's index stage, 2 * kDepth chunks ahead of its LDS stage; past the end of the stream it stays on the
    // last run
    uint32_t bundle_set = 0, J = 0, cj = 0, first = 0; // the run, and the first row of the next chunk in it
    uint32_t clo = 0, len = 1;
    auto open_run = [&]() {
      const uint4 m = tables[bundle_set * kTable + cj];
      clo = uni(m.y), len = uni(m.z), first = 0;
    };
    // read(positions of the next chunk, its last row): loads are unconditional, so that kDepth chunks stay in flight per thread, and
    // rows past the end of a run re-read its last one (never summed)
    auto next_chunk = [&](auto &&read) {
      const uint32_t from = min(first, len - 1), last = min(CR, len - from) - 1;
      read(sorted_arg + clo + from, last);
      first += CR;
      if (first >= len) {
        if (cj + 1 < J) {
          cj++;
          open_run();
        } else {
          first = len;
        }
      }
    };
    auto open_cursor = [&](uint32_t set, uint32_t runs) {
      bundle_set = set, J = runs, cj = 0;
      open_run();
    };
    uint4 mine;
    if (wave == 0) draw(0, mine);
    __syncthreads();
    for (uint32_t cur = 0;; cur ^= 1) {
      const uint4 *table = tables + cur * kTable;
      const uint32_t runs = uni(shared[cur * 4]), G = uni(shared[cur * 4 + 1]), slice = uni(shared[cur * 4 + 2]);
      if (!runs) break;
      if (wave == 0) draw(cur ^ 1, mine); // while the loaders wait for the first rows of this bundle
      const uint32_t slot_floats = CR * CS;
      if (wave != 0) {
        const uint32_t lt = threadIdx.x - kWave, my_row = lt / lanes, my_lane = lt % lanes, step = kLoaders / lanes;
        const bool in_slice = my_lane < CS && my_row < step;
        const uint32_t col = slice * CS + my_lane;
        const embed_t *gbase = a.grad + (in_slice && col < W ? col : 0u); // lanes outside the slice read column 0
        uint32_t idx[kDepth][kRPT];
        V val[kDepth][kRPT];
        auto read_index = [&](int k) {
          next_chunk([&](const uint32_t *pos, uint32_t last) {
#pragma unroll
            for (int q = 0; q < kRPT; q++) idx[k][q] = pos[min(q * step + my_row, last)];
          });
        };
        auto row_load = [&](uint32_t pos) -> V { // (the bag of a position where it is read would wait for it)
          return grad_load<Vec<VEC>, kAgain>((const embed_t *)((const char *)gbase + (uint64_t)grad_row<kPooled>(pos, a.bag) * (W * 4)));
        };
        // val[k] holds chunk k and idx[k] the row indices of chunk k + kDepth
        open_cursor(cur, runs);
#pragma unroll
        for (int k = 0; k < kDepth; k++) read_index(k);
#pragma unroll
        for (int k = 0; k < kDepth; k++)
#pragma unroll
          for (int q = 0; q < kRPT; q++) val[k][q] = row_load(idx[k][q]);
#pragma unroll
        for (int k = 0; k < kDepth; k++) read_index(k);
        uint32_t slot = 0;
        rounds(G, [&](int k) {
          float *sp = lds + slot * slot_floats;
          slot = slot + 1 == kSlotsGeneric ? 0 : slot + 1;
#pragma unroll
          for (int q = 0; q < kRPT; q++) {
            if (in_slice) Vec<VEC>::store_all(sp + (q * step + my_row) * CS + my_lane, val[k][q]);
            val[k][q] = row_load(idx[k][q]); // chunk + kDepth
          }
          read_index(k); // chunk + 2 * kDepth
          lds_done();
          __syncthreads(); // barrier of this chunk
        });
      } else {
        const uint32_t place = threadIdx.x % kWave, mycol = slice * CS + place;
        const bool col_ok = place < CS && mycol < W;
        const bool direct = t.nrank == 1;
        if (direct) { // the table rows the sums are added to, for every run of the bundle at once and parked in LDS
          float rows[kTable];
#pragma unroll
          for (uint32_t j = 0; j < kTable; j++) {
            rows[j] = 0.f;
            if (j < runs && col_ok) rows[j] = t.emb[(size_t)table[j].w * W + mycol];
          }
#pragma unroll
          for (uint32_t j = 0; j < kTable; j++) sums[j * kWave + place] = rows[j];
        }
        uint32_t slot = 0;
        for (uint32_t j = 0; j < runs; j++) {
          const uint4 m = table[j];
          float acc = 0.f; // the reference starts every sum from 0
          for (uint32_t c = 0; c * CR < m.z; c++) {
            lds_done();
            __syncthreads(); // barrier of this chunk
            const float *sp = lds + slot * slot_floats + place;
            slot = slot + 1 == kSlotsGeneric ? 0 : slot + 1;
            if (place < CS) {
              const uint32_t rows = min(CR, m.z - c * CR);
              uint32_t r = 0;
              for (; r + 8 <= rows; r += 8) {
                float x[8];
#pragma unroll
                for (int q = 0; q < 8; q++) x[q] = sp[(r + q) * CS];
#pragma unroll
                for (int q = 0; q < 8; q++) acc += x[q];
              }
              for (; r < rows; r++) acc += sp[r * CS];
            }
          }
          if (col_ok) { // the sum of run j of the bundle is complete
            const float scaled = acc * neg_lr;
            if (direct) t.emb[(size_t)m.w * W + mycol] = sums[j * kWave + place] + scaled;
            else apply_row<Vec<1>, K>(t, id_bits, p, a, m.x, scaled, mycol);
          }
        }
      }
      __syncthreads(); // everybody is done with the table and the ring
    }
  }
}

// all roles in one launch: the long chains start first, medium and short blocks fill the machine behind them, the
// version counters of a single shard come last
template <int VEC, int LPR, typename K, bool kSingle, bool kPooled>
__device__ __forceinline__ void push_block(const TableView &t, int id_bits, const BatchView &p, const PushArgs &a, uint32_t U,
                                           uint32_t block) {
  // one LDS area for whichever role the block plays: the row ring of the long role or the index staging of the
  // medium role (one slice of kLongRun indices per group)
  constexpr int kRingWords = VEC == 1 ? kSlotsGeneric * 2 * kPushBlock : kSlotsFast * kSlotVectors * 4;
  constexpr int kStageWords = (kPushBlock / LPR) * (int)kLongRun;
  __shared__ __align__(16) float lds[kRingWords > kStageWords ? kRingWords : kStageWords];
  __shared__ uint4 run_table[2 * kTable];
  __shared__ uint32_t run_totals[4 * 4];
  __shared__ float sums[kTable * kWave]; // long role: the sums of a bundle's runs (generic path: the rows they are added to)
  if (block < kLongBlocks) {
    // Every block first takes tickets of the longest runs, which are cut into narrower column slices so that more
    // blocks feed each of them (the blocks of a saturated memory system get equal shares of it, and a chain
    // advances with the share of the block that feeds it), then tickets of the other long runs.
    uint32_t *tk = p.d_nlong + kTicketBase;
    uint32_t counts = p.d_nlong[min(threadIdx.x % kWave, (uint32_t)kLongBuckets - 1)]; // long runs by length class, one per lane
    auto runs = [&](auto csc, auto again, int c_lo, int c_hi, uint32_t *counters) {
      long_role<VEC, K, decltype(csc)::value, kPooled, kPooled || decltype(again)::value>(t, id_bits, p, a, lds, run_table, run_totals, sums, counts, c_lo, c_hi, block, kLongBlocks, counters);
    };
    if constexpr (VEC == 1) {
      runs(std::integral_constant<int, 0>(), std::false_type(), 0, kLongBuckets, tk);
    } else if constexpr (LPR <= 8) { // rows of up to 16 or 32 floats
      // A row that is no whole line shares one with its neighbour, whose key is often the same one (several ids per field), and a
      // lane reads neighbours in four loads: they are to find the line in the cache.  Loaded past it / not, 5.3 M keys of 18 ids
      // per field, Zipf 1.2, the push alone on an MI355X: 12 floats 449 / 373 us, 17 floats 540 / 446, 31 floats 702 / 636; 3 ids
      // per field, 24 floats, 1.6 M keys 124 / 97; one id per field, 20 floats, 2.6 M keys 158 / 132.  Of 32 floats,
      // which are a line, 432 / 439, and two steps 1370 / 1411: their rows push out what the gather reads.
      constexpr int kLineFloats = 32;
      if (LPR * 4 == kLineFloats && t.width == kLineFloats && !kPooled)
        runs(std::integral_constant<int, LPR * 4>(), std::false_type(), 0, kLongBuckets, tk);
      else runs(std::integral_constant<int, LPR * 4>(), std::true_type(), 0, kLongBuckets, tk);
    } else {
      uint64_t rows = 0; // of all long runs, roughly: by the middle of their classes
#pragma unroll
      for (int c = 0; c < kLongBuckets; c++) rows += (uint64_t)count_of(counts, c) * (3u << 16 >> c);
      const int narrow = narrow_slices(t.width) ? kLongBuckets : narrow_classes(t.width, rows, kLongBlocks);
      asm volatile("" : "+v"(counts)); // read again from here on, not kept in twelve scalar registers
      runs(std::integral_constant<int, kGiantSlice>(), std::false_type(), 0, narrow, tk);
      if (narrow < kLongBuckets) runs(std::integral_constant<int, kSlice>(), std::false_type(), narrow, kLongBuckets, tk + kTicketLanes);
    }
  } else if (block < kLongBlocks + kMedBlocks) { // medium runs take long per block: they start early
    medium_role<VEC, LPR, K, kSingle, kPooled>(t, id_bits, p, a, (uint32_t *)lds, block - kLongBlocks, kMedBlocks);
  } else {
    constexpr int kGroups = kPushBlock / LPR;
    const uint32_t short_blocks = div_up_dev(U, kGroups * kRunsPerGroup);
    const uint32_t b = block - kLongBlocks - kMedBlocks;
    if (b < short_blocks) {
      short_role<VEC, LPR, K, kSingle, kPooled>(t, id_bits, p, a, b, U);
    } else {
      // The counters of every unique key, one thread per key, in the last blocks of the grid: they depend on the
      // batch's index and plan only, not on the sums.
      const uint32_t u = (b - short_blocks) * kPushBlock + threadIdx.x;
      if (u < U) {
        if (kSingle) {
          // Single shard: every key is owned, so the only counter is the row version, which grows by the number of
          // duplicates (generate_query.cu:68-69).  Nontemporal: a counter line is touched once per step; left in the
          // cache it is written back in the middle of the gather that follows.
          version_t *vp = &t.ver[p.uoff[u]];
          const version_t v = __builtin_nontemporal_load(vp) + (version_t)(p.run_start[u + 1] - p.run_start[u]);
          __builtin_nontemporal_store(v, vp);
        } else {
          const slot_t o = p.uoff[u];
          const bool need = a.need[u] != 0;
          const int type = o == kNoSlot ? 0 : ((uint32_t)o >= t.n_cached ? 1 : (need ? 2 : 3));
          move_counters<K>(t, id_bits, p, a, u, o, type, a.prefix[u]);
        }
      }
    }
  }
}

#ifndef HCTR_PUSH_WAVES
#define HCTR_PUSH_WAVES 4
#endif
#define HCTR_PUSH_BOUNDS __launch_bounds__(kPushBlock) __attribute__((amdgpu_waves_per_eu(HCTR_PUSH_WAVES, 8)))
template <int VEC, int LPR, typename K, bool kPooled>
__global__ HCTR_PUSH_BOUNDS void push_fused(TableView t, int id_bits, BatchView p, PushArgs a, uint32_t U) {
  push_block<VEC, LPR, K, true, kPooled>(t, id_bits, p, a, U, blockIdx.x);
}
// The pushes of the shards of a group in one launch.  First come the blocks that every shard has (its chains, its medium runs
// and as many more as the smallest batch needs), neighbouring blocks being the same block of different shards, so that every
// shard's long chains start first; behind them the rest of the larger batches, a shard after the other.
typedef Records<PushShard, kShardsPerLaunch> PushShards; // cut: of the rest
constexpr uint32_t kEachBlocks = kLongBlocks + kMedBlocks;
template <int VEC, int LPR, typename K, bool kPooled>
__global__ HCTR_PUSH_BOUNDS void push_group(PushShards shards, uint32_t count, uint32_t common, int id_bits) {
  uint32_t block = blockIdx.x, k;
  if (block < common * count) {
    k = block % count;
    block /= count;
  } else {
    block -= common * count;
    k = record_of(shards.cut, block);
    block += common;
  }
  const PushShard &S = shards.s[k];
  push_block<VEC, LPR, K, false, kPooled>(S.t, id_bits, S.b, S.a, S.n_unique, block);
}

typedef Records<PlaceShard, kShardsPerLaunch> PlaceShards;
template <typename K> __global__ __launch_bounds__(256) void place_rows(PlaceShards shards, int id_bits) {
  uint32_t block, blocks;
  const PlaceShard &S = my_record(shards, block, blocks);
  const uint32_t u = block * 256 + threadIdx.x;
  if (u < S.n_unique) S.pos[u] = S.prefix[u] + S.delta[(uint32_t)(((const K *)S.ukey)[u] >> id_bits)];
}

template <int VEC, int LPR, typename K, bool kPooled>
void launch_push_t(hipStream_t st, int id_bits, PushShards &shards, int count) {
  // short runs, and the counters of every unique key
  auto need = [](const PushShard &S) { return div_up(S.n_unique, (kPushBlock / LPR) * kRunsPerGroup) + div_up(S.n_unique, kPushBlock); };
  const PushShard &S = shards.s[0];
  if (S.t.nrank == 1) {
    hipLaunchKernelGGL((push_fused<VEC, LPR, K, kPooled>), dim3(kEachBlocks + need(S)), dim3(kPushBlock), 0, st, S.t, id_bits, S.b, S.a, S.n_unique);
    return;
  }
  for (int i = 0; i < count;) { // nearly always one launch
    const int m = cut_blocks(shards.cut, count - i, kPushBlock, kEachBlocks, [&](int k) { return need(shards.s[i + k]); });
    if (i) std::copy(shards.s + i, shards.s + i + m, shards.s);
    const uint32_t least = *std::min_element(shards.cut.blocks, shards.cut.blocks + m), common = kEachBlocks + least;
    cut_blocks(shards.cut, m, kPushBlock, common, [&](int k) { return need(shards.s[k]) - least; });
    hipLaunchKernelGGL((push_group<VEC, LPR, K, kPooled>), dim3(common * m + shards.cut.total), dim3(kPushBlock), 0, st, shards, (uint32_t)m, common, id_bits);
    i += m;
  }
}

template <int VEC, typename K, bool kPooled>
void launch_push_p(hipStream_t st, int id_bits, PushShards &shards, int count) {
  if constexpr (VEC == 1) { // rows of less than four floats
    launch_push_t<VEC, 4, K, kPooled>(st, id_bits, shards, count);
  } else {
    const uint32_t lanes = (shards.s[0].t.width + kCols<VEC> - 1) / kCols<VEC>;
    if (lanes <= 4) launch_push_t<VEC, 4, K, kPooled>(st, id_bits, shards, count);
    else if (lanes <= 8) launch_push_t<VEC, 8, K, kPooled>(st, id_bits, shards, count);
    else if (lanes <= 16) launch_push_t<VEC, 16, K, kPooled>(st, id_bits, shards, count);
    else if (lanes <= 32) launch_push_t<VEC, 32, K, kPooled>(st, id_bits, shards, count);
    else launch_push_t<VEC, 64, K, kPooled>(st, id_bits, shards, count);
  }
}

template <int VEC, typename K>
void launch_push_k(hipStream_t st, int id_bits, PushShards &shards, int count) {
  if (shards.s[0].a.bag.bag > 1) launch_push_p<VEC, K, true>(st, id_bits, shards, count);
  else launch_push_p<VEC, K, false>(st, id_bits, shards, count);
}

} // namespace

void launch_place_rows(hipStream_t s, const KeyLayout &kl, const PlaceShard *shards, int count) {
  auto make = [&](int k) { return shards[k]; };
  auto need = [&](int k) { return div_up(shards[k].n_unique, 256); };
  launch_records<PlaceShard, kShardsPerLaunch>(count, 256, make, need, [&](const PlaceShards &p, int) {
    const dim3 grid = grid_of(p);
    if (kl.wide) hipLaunchKernelGGL(place_rows<uint64_t>, grid, dim3(256), 0, s, p, kl.id_bits);
    else hipLaunchKernelGGL(place_rows<uint32_t>, grid, dim3(256), 0, s, p, kl.id_bits);
    HCTR_HIP(hipGetLastError());
  });
}

void launch_push(hipStream_t s, const KeyLayout &kl, const PushShard *shards, int count) {
  for (int i = 0; i < count;) {
    PushShards p = {};
    int m = 0, vec = 4;
    for (; i < count && m < kShardsPerLaunch; i++) {
      if (!shards[i].b.n || !shards[i].n_unique) continue;
      p.s[m++] = shards[i];
      const int v = row_vec(shards[i].t.width, shards[i].a.grad);
      if (v != 4) vec = v; // vectors that suit every shard's gradient
    }
    if (!m) break;
#define PUSH(VEC)                                                       \
  do {                                                                  \
    if (kl.wide) launch_push_k<VEC, uint64_t>(s, kl.id_bits, p, m);     \
    else launch_push_k<VEC, uint32_t>(s, kl.id_bits, p, m);             \
  } while (0)
    switch (vec) {
      case 4: PUSH(4); break;
      case kOdd4: PUSH(kOdd4); break;
      default: PUSH(1); break;
    }
#undef PUSH
    HCTR_HIP(hipGetLastError());
  }
}

} // namespace hctr

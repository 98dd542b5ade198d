// batch.hip -- many frusta over many object groups in one persistent launch,
// and the plain per-view form of the same work.
//
// Reference: cull(group, result, viewProjection) (dp/culling/Manager.h:139),
// one call per (view, group) in the reference (dp/culling/cpu/src/ManagerImpl.cpp:467-518).
//
// Work decomposition: a group is split into tiles of 64*K objects.  A work item
// is (tile, slice of the frusta paired with the tile's group).  A wave owns one
// item at a time: every lane builds what the quick test needs of its K objects
// once (one read of each object's matrix and box), then the wave takes the item's
// frusta in runs of sixteen: the lanes hold four rows of each of the run's views,
// the matrix cores contract them with the lanes' objects, and each (frustum, 64
// objects) result is one lane mask, a 64-bit mask word.  No two items write the
// same mask word, so no atomics touch the output.
//
// What bounds it: with many frusta per object, instruction issue and what does not
// overlap it: a frustum and 64 objects take 7 matrix and 16 vector instructions (48
// vector instructions with the quick test's products on the vector unit, 190 when
// each pair took the exact test).  500,003 objects x 32 frusta: 109 us with the
// exact test, 35 with the quick test, 26 with its products on the matrix cores, of
// which 9 are reading the objects and 11 the instructions, and 68 where the quick test
// decides nothing (kDenseLanes); 64 frusta over 64 groups of 2,097,152 objects: 40 ->
// 35 us, 5.3 TB/s, bound by reading the objects, those of undecided pairs twice.
//
// Schedule: items are sorted by cost (frusta x objects) on the host, and the
// persistent grid walks them round-robin (wave w takes w, w+W, ...), which
// bounds the load imbalance by the cost of one item.  Objects are not loaded
// ahead of the item that is tested: without the 22 registers that takes, six
// waves run per SIMD, and hide the loads themselves.
#include <algorithm>
#include <cstddef>
#include <cstring>
#include <numeric>
#include <vector>

#include "batch_types.hpp"
#include "cull_math.hpp"
#include "internal.hpp"

#pragma clang fp contract(off)

namespace dpc {
namespace {

struct WorkItem {
  uint64_t first_object;
  uint32_t count;       // objects in the tile (<= 64*K)
  uint32_t tile_word;   // mask word of the tile's first object, relative to its group
  uint32_t pair_begin;  // slice of the pair table
  uint32_t pair_count;
  uint32_t scene;       // entry of the scene table
  uint32_t pad;
};
static_assert(sizeof(WorkItem) == 32, "WorkItem layout");


struct ViewTile {
  uint64_t first_object;
  uint64_t mask_word;
  uint32_t count;
  uint32_t scene;
  uint64_t pad;
};
static_assert(sizeof(ViewTile) == 32, "ViewTile layout");

// Device copy of a dpc_scene_desc (same layout).
struct SceneDev {
  const float4* box_a;
  const float2* box_b;
  const uint32_t* xform;
  const float4* planes;
  uint64_t ld;
  uint64_t n_objects;
};
static_assert(sizeof(SceneDev) == 48 && sizeof(SceneDev) == sizeof(dpc_scene_desc), "SceneDev layout");

__device__ __forceinline__ void load_vp(const float* __restrict__ vps, uint32_t frustum, Mat16& vp)
{
#pragma unroll
  for (int c = 0; c < 16; ++c) vp.m[c] = vps[16 * static_cast<size_t>(frustum) + c];
}

// Pairs (object, frustum) that the quick test left undecided wait in LDS, one
// queue per wave, until its entries nearly fill the wave: then each lane takes
// one of them through the exact test.  A few lanes in a thousand are undecided,
// which would otherwise send every third wave through the exact test for the
// sake of one lane.  The mask words they belong to wait with them and are stored
// once, complete.
struct QueueEntry {
  uint32_t object_lo;
  uint32_t object_hi;  // bits 0-15; bits 16-23: which of the waiting words; bits 24-29: the object's bit in it
  uint32_t frustum;
  uint32_t scene;
};
struct QueueWord {
  unsigned long long bits;
  uint64_t index;  // word of the mask buffer
};
template <int K>
struct Queue {
  static constexpr uint32_t kCapacity = kWave * K;  // any one (frustum, work item) fits when it is empty
  QueueEntry entry[kCapacity];
  QueueWord word[kCapacity];
};

// The exact test of the queue's n entries, then the stores of its n_words words.
template <int K>
__device__ __forceinline__ void drain(Queue<K>& queue, uint32_t n, uint32_t n_words, uint32_t lane,
                                      const SceneDev* __restrict__ scenes, const float* __restrict__ vps,
                                      unsigned long long* __restrict__ masks)
{
  wave_lds_order();
  for (uint32_t q0 = 0; q0 < n; q0 += kWave) {
    const bool on = q0 + lane < n;
    const QueueEntry e = queue.entry[on ? q0 + lane : q0];
    const SceneDev sc = scenes[e.scene];
    const size_t object = (static_cast<size_t>(e.object_hi & 0xFFFFu) << 32) | e.object_lo;
    const Slot slot = make_slot(object, object + 1, sc.xform, sc.ld);
    const RawObj raw = load_raw(sc.box_a, sc.box_b, sc.planes, sc.ld, slot.i, slot.m);
    Mat16 m;
    load_vp(vps, e.frustum, m);
    if (on & obb_visible(obb_of(raw), m.m))
      __hip_atomic_fetch_or(&queue.word[(e.object_hi >> 16) & 0xFFu].bits, 1ull << (e.object_hi >> 24),
                            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
  }
  wave_lds_order();
  for (uint32_t w = lane; w < n_words; w += kWave) masks[queue.word[w].index] = queue.word[w].bits;
  wave_lds_order();
}

// What a wave keeps of the work item it tests.
template <int K>
struct TileObjects {
  QuickObj quick[K];
  unsigned long long tested[K];  // lanes that hold an object with a matrix
  unsigned long long always[K];  // lanes whose object is visible whatever the frustum (matrix index outside the array)
};

// The loads of a work item's objects, and what the wave keeps of them.
template <int K>
__device__ __forceinline__ void load_objects(const SceneDev* __restrict__ scenes, const WorkItem& item, uint32_t lane,
                                             Slot (&slot)[K], RawObj (&raw)[K])
{
  const SceneDev sc = scenes[item.scene];
  const size_t end = item.first_object + item.count;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    slot[k] = make_slot(item.first_object + lane + kWave * k, end, sc.xform, sc.ld);
    raw[k] = load_raw(sc.box_a, sc.box_b, sc.planes, sc.ld, slot[k].i, slot[k].m);
  }
}

template <int K>
__device__ __forceinline__ void quick_objects(const Slot (&slot)[K], const RawObj (&raw)[K], TileObjects<K>& t)
{
#pragma unroll
  for (int k = 0; k < K; ++k) {
    t.quick[k] = quick_of(obb_of(raw[k]));
    t.tested[k] = ballot(slot[k].valid & !slot[k].bad_matrix);
    t.always[k] = ballot(slot[k].valid & slot[k].bad_matrix);
  }
}

// The entries of a work item's list that a wave's lanes hold: lane 4 f + i that of
// frustum p0 + f (the last one again past the end).
__device__ __forceinline__ KPair load_pairs(const KPair* __restrict__ pairs, const WorkItem& item, uint32_t p0,
                                            uint32_t lane)
{
  const uint32_t p = p0 + lane / 4 % kQuickRun;
  return pairs[item.pair_begin + (p < item.pair_count ? p : item.pair_count - 1)];
}

template <int Lane>
__device__ __forceinline__ uint32_t lane_of(uint32_t v)
{
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), Lane));
}

// `to` with the wave-uniform v in one lane.
template <int Lane>
__device__ __forceinline__ uint32_t set_lane(uint32_t v, uint32_t to)
{
  asm("v_writelane_b32 %0, %1, %2" : "+v"(to) : "s"(v), "n"(Lane));
  return to;
}

// A run of kQuickRun frusta (at most) of a work item's list.
template <int K>
struct Run {
  uint32_t todo, again;   // bit f: frustum f is to be tested; is left for when the queue is empty
  uint32_t queued[K];     // bit f: word k of frustum f waits in the queue
  uint32_t lo[K], hi[K];  // lane 4 f: word k of frustum f
};

// Where the quick test decides little (boxes as large as what a view sees; object
// matrices with a projective part, of which it decides nothing), the queue costs more
// than testing every pair exactly: an undecided pair reads its object and its view
// again, alone (500,003 objects x 32 frusta, nothing decided: 136 us, with every pair
// tested exactly 66).  A full queue therefore ends a run: a frustum that leaves more
// than kDenseLanes objects of 64 undecided goes to the exact test as a whole, with
// those after it, where the words that wait were as dense (68 us; a third of the
// matrices projective, 19 a word: 82 -> 68, and 112 with the line at 24 lanes; with it
// at 8, boxes of which a word leaves 8 undecided: 41 -> 58).  The question is asked of a
// full queue only: asked at every undecided word it cost the ordinary scene 8 %.
constexpr uint32_t kDenseLanes = 16;
constexpr uint32_t kExact = 1u << 31;
// After an item of whose list less than a quarter was done before that, a wave takes
// this many items through the exact test without trying the quick one (68.4 us; with
// every item tried 70.7, with one in eight 68.4).
constexpr uint32_t kExactItems = 3;

// Tests the wave's objects against frustum F of a run.  A word with undecided
// objects goes to the queue; without room for them the frustum and those after it
// are left (kExact: to the exact test).
template <int F, int K>
__device__ __forceinline__ void test_frustum(Run<K>& run, const WorkItem& item, const TileObjects<K>& t,
                                             const QuickRows& rows, const KPair& pair, uint32_t lane, Queue<K>& queue,
                                             uint32_t& waiting, uint32_t& words)
{
  if (!((run.todo >> F) & 1)) return;
  unsigned long long bits[K], open[K], any = 0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const QuickResult<unsigned long long> r = quick_wave<F>(t.quick[k], rows);
    bits[k] = (r.visible & t.tested[k]) | t.always[k];
    open[k] = t.tested[k] & ~(r.visible | r.culled);
    any |= open[k];
    run.lo[k] = set_lane<4 * F>(static_cast<uint32_t>(bits[k]), run.lo[k]);
    run.hi[k] = set_lane<4 * F>(static_cast<uint32_t>(bits[k] >> 32), run.hi[k]);
  }
  if (__builtin_expect(any == 0, 1)) return;
  uint32_t n_open = 0;
#pragma unroll
  for (int k = 0; k < K; ++k) n_open += static_cast<uint32_t>(__builtin_popcountll(open[k]));
  if (waiting + n_open > Queue<K>::kCapacity) {
    run.again = run.todo & (~0u << F);
    if (n_open > kDenseLanes * K && waiting > kDenseLanes * words) run.again |= kExact;
    run.todo = 0;
    return;
  }
  const uint32_t frustum = lane_of<4 * F>(pair.frustum);
  const uint64_t word = static_cast<uint64_t>(lane_of<4 * F>(static_cast<uint32_t>(pair.mask_word >> 32))) << 32 |
                        lane_of<4 * F>(static_cast<uint32_t>(pair.mask_word));
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (open[k] == 0) continue;
    if (__builtin_amdgcn_inverse_ballot_w64(open[k])) {
      const uint64_t object = item.first_object + lane + kWave * k;
      const uint32_t at = waiting + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(open[k] >> 32),
                                                              __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(open[k]), 0u));
      queue.entry[at] = QueueEntry{static_cast<uint32_t>(object),
                                   static_cast<uint32_t>(object >> 32) | (words << 16) | (lane << 24), frustum, item.scene};
    }
    queue.word[words] = QueueWord{bits[k], word + item.tile_word + k};  // (every lane the same)
    run.queued[k] |= 1u << F;
    waiting += static_cast<uint32_t>(__builtin_popcountll(open[k]));
    ++words;
  }
}

// (A matrix instruction names the view it reads, so each frustum of a run has code
// of its own.)
template <int F, int K>
__device__ __forceinline__ void test_run(Run<K>& run, const WorkItem& item, const TileObjects<K>& t,
                                         const QuickRows& rows, const KPair& pair, uint32_t lane, Queue<K>& queue,
                                         uint32_t& waiting, uint32_t& words)
{
  if constexpr (F < static_cast<int>(kQuickRun)) {
    test_frustum<F, K>(run, item, t, rows, pair, lane, queue, waiting, words);
    test_run<F + 1, K>(run, item, t, rows, pair, lane, queue, waiting, words);
  }
}

// Tests a work item against its frusta, kQuickRun at a time, one mask word per
// frustum and 64 objects.  Words that the quick test (quick_cull.hpp) decides whole
// are stored together, a run's in one instruction; the others wait in the queue.
// pair: the first run's entries of the item's list.  view_of(p0, p, frustum) gives
// the lane the QuickView of the item's p-th frustum, in the run from p0 on.  Returns
// how many of the list's frusta are done: where not all are, the next ones are left to
// test_exact.
template <int K, class ViewOf>
__device__ __forceinline__ uint32_t test_frusta(const WorkItem& item, const TileObjects<K>& t, KPair pair, uint32_t lane,
                                                const KPair* __restrict__ pairs, const SceneDev* __restrict__ scenes,
                                                const float* __restrict__ vps, unsigned long long* __restrict__ masks,
                                                Queue<K>& queue, uint32_t& waiting, uint32_t& words, ViewOf&& view_of)
{
  uint32_t p0 = 0;
  for (;;) {
    const uint32_t left = item.pair_count - p0;
    uint32_t n = left < kQuickRun ? left : kQuickRun;
    const QuickRows rows = quick_rows(view_of(p0, p0 + min(lane / 4 % kQuickRun, n - 1), pair.frustum), lane % 4);
    const KPair next = load_pairs(pairs, item, p0 + kQuickRun, lane);
    Run<K> run = {};
    run.todo = (1u << n) - 1;
    for (;;) {
      test_run<0, K>(run, item, t, rows, pair, lane, queue, waiting, words);
      if (run.again == 0) break;
      if (run.again & kExact) {
        n = static_cast<uint32_t>(__builtin_ctz(run.again));
        break;
      }
      drain<K>(queue, waiting, words, lane, scenes, vps, masks);
      waiting = words = 0;
      run.todo = run.again;
      run.again = 0;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      // (a work item holds at least one object: the first word is always stored)
      if (k != 0 && static_cast<uint32_t>(kWave * k) >= item.count) break;
      if (lane % 4 == 0 && lane / 4 < n && !((run.queued[k] >> (lane / 4)) & 1))
        masks[pair.mask_word + item.tile_word + k] = static_cast<unsigned long long>(run.hi[k]) << 32 | run.lo[k];
    }
    p0 += n;
    if (p0 >= item.pair_count || n < kQuickRun) break;
    pair = next;
  }
  return p0;
}

// The exact test of a work item's objects against the frusta [first, end) of its list,
// each in scalar registers.  The objects are read again: kept across the quick test they
// would take the registers of a wave per SIMD.
template <int K>
__device__ __forceinline__ void test_exact(WorkItem item, uint32_t first, uint32_t end, uint32_t lane,
                                           const KPair* __restrict__ pairs, const SceneDev* __restrict__ scenes,
                                           const float* __restrict__ vps, unsigned long long* __restrict__ masks)
{
  // (as new values: the scene and addresses of the first read would otherwise be kept)
  asm volatile("" : "+s"(item.scene), "+s"(item.first_object), "+v"(lane));
  Slot slot[K];
  RawObj raw[K];
  load_objects<K>(scenes, item, lane, slot, raw);
  Obb o[K];
#pragma unroll
  for (int k = 0; k < K; ++k) o[k] = obb_of(raw[k]);
  for (uint32_t p = first; p < end; ++p) {
    const KPair pair = pairs[item.pair_begin + p];
    Mat16 m;
    load_vp(vps, pair.frustum, m);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const unsigned long long bits = ballot(slot_visible(slot[k], obb_visible(o[k], m.m)));
      if (k == 0 || static_cast<uint32_t>(kWave * k) < item.count) masks[pair.mask_word + item.tile_word + k] = bits;
    }
  }
}

// Where a wave finds the QuickViews of its frusta: about a hundred instructions
// with three square roots would go into each use.  The batched kernel keeps those
// of all frusta of a launch in LDS, computed once per workgroup (Table: at most
// kTableViews frusta, 12 KB); without, and in the serving kernel, a wave keeps those
// of 64 frusta of its list, one per lane.
constexpr uint32_t kTableViews = 128;
constexpr uint32_t kBatchWaves = 4;  // waves of a workgroup, at most

__device__ __forceinline__ void list_views(const KPair* __restrict__ list, uint32_t count,
                                           const float* __restrict__ vps, uint32_t lane, QuickView* views)
{
  wave_lds_order();
  if (lane < count) {
    Mat16 m;
    load_vp(vps, list[lane].frustum, m);
    views[lane] = quick_view(m.m);
  }
  wave_lds_order();
}

// The second launch bound keeps the 24 waves per CU of the default grid resident
// (80 registers; at 95, and five waves per SIMD, 2,097,152 objects took 37.7 us
// against 33.8), and has the matrix instructions' results in ordinary registers:
// without one they are copied from the accumulation registers.
template <int K, bool Table>
__global__ __launch_bounds__(256, K == 1 ? (Table ? 6 : 5) : K == 2 ? 4 : 2) void cull_batch_kernel(const WorkItem* __restrict__ items, uint32_t n_items,
                                                         const KPair* __restrict__ pairs,
                                                         const SceneDev* __restrict__ scenes,
                                                         const float* __restrict__ vps, uint32_t n_frusta,
                                                         unsigned long long* __restrict__ masks)
{
  __shared__ QuickView table[Table ? kTableViews : kBatchWaves * kWave];
  __shared__ Queue<K> queues[kBatchWaves];
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t waves_per_block = blockDim.x / kWave;
  const uint32_t n_waves = gridDim.x * waves_per_block;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  uint32_t it = blockIdx.x * waves_per_block + wave;
  uint32_t waiting = 0, words = 0;
  for (bool first = true;; first = false) {
    WorkItem item = items[it < n_items ? it : 0];  // (n_items >= 1)
    Slot slot[K];
    RawObj raw[K];
    load_objects<K>(scenes, item, lane, slot, raw);
    const KPair pair = load_pairs(pairs, item, 0, lane);
    if (first) {  // the table is built while the first objects are in flight
      if (Table) {
        uint32_t f = threadIdx.x;
        asm volatile("" : "+v"(f));  // (the comparison stays here, not in registers of the whole loop)
        for (; f < n_frusta; f += blockDim.x) {
          Mat16 m;
          load_vp(vps, f, m);
          table[f] = quick_view(m.m);
        }
        lds_barrier();
      }
      if (it >= n_items) return;  // (a wave without an item helped with the table)
    }
    TileObjects<K> objects;
    quick_objects<K>(slot, raw, objects);
    auto view_of = [&](uint32_t p0, uint32_t p, uint32_t f) -> const QuickView& {
      if (Table) return table[f];
      if (p0 % kWave == 0)
        list_views(pairs + item.pair_begin + p0, item.pair_count - p0, vps, lane, &table[wave * kWave]);
      return table[wave * kWave + p % kWave];
    };
    uint32_t done =
        test_frusta<K>(item, objects, pair, lane, pairs, scenes, vps, masks, queues[wave], waiting, words, view_of);
    if (__builtin_expect(done < item.pair_count, 0)) {
      // (the next items here too: asked for at each item, they cost a short launch 0.1 us)
      for (uint32_t more = done * 4 < item.pair_count ? kExactItems : 0;; --more) {
        test_exact<K>(item, done, item.pair_count, lane, pairs, scenes, vps, masks);
        if (more == 0 || it + n_waves >= n_items) break;
        it += n_waves;
        item = items[it];
        done = 0;
      }
    }
    it += n_waves;
    if (it >= n_items) break;
  }
  drain<K>(queues[wave], waiting, words, lane, scenes, vps, masks);
}

// ---- serving form -----------------------------------------------------------
// One entry per request of a serving batch: the whole scene is tested against
// the request's frusta (pairs[pair_begin .. +pair_count)).  Work is split without
// a per-batch item list: the (tile, frustum) pairs of all entries, in order, are
// divided equally over the waves, and a wave walks its run tile by tile.  A tile
// may be shared by several waves, each of which reads its objects: whole tiles per
// wave left small scenes to few waves and large batches with one tile more on some
// (203 tiles x 13 frusta: 14 -> 8.4 us; seven scenes of 9,058 tiles in all x 17 to
// 32: 57 -> 39 us; 6,250 tiles x 20: 40 -> 32 us).

constexpr uint32_t kServeViews = 64;  // frusta of a request, at most (dpc_server_submit)

// A request of this many frusta or fewer takes the exact test: each of its tiles' object
// bounds, for which the quick test reads the objects first, would serve one or two words
// (quick -> exact: 10,000 x 1 6.1 -> 4.2 us, x 2 7.1 -> 4.2; 200,000 x 1 7.8 -> 5.7, x 2
// 9.2 -> 7.3; 1,000,000 x 1 19.0 -> 17.5, x 2 20.8 -> 21.0).  Of four frusta the quick
// test takes as long up to 100,000 objects (6.1 to 8.2 us, exact 5.3 to 8.0) and less
// beyond (500,000 17.3 -> 15.1 us, 1,000,000 29.1 -> 22.4).
constexpr uint32_t kFewFrusta = 2;
static_assert(kServeViews <= kWave, "one lane per frustum");

// A wave's current entry: its fields in the lanes of one register, each read where it
// is used (as scalars beside the loop's state they spill: 4 scenes of 500,003 objects,
// 32 views each, 282 -> 291 us a tick).
struct EntryLanes {
  uint32_t v;  // lane l: word l % 8 of the ServeEntry
  __device__ __forceinline__ uint32_t get(size_t offset) const
  {
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), static_cast<int>(offset / 4)));
  }
  __device__ __forceinline__ uint32_t pair_begin() const { return get(offsetof(ServeEntry, pair_begin)); }
  __device__ __forceinline__ uint32_t pair_count() const { return get(offsetof(ServeEntry, pair_count)); }
  __device__ __forceinline__ uint32_t tiles() const { return get(offsetof(ServeEntry, tiles)); }
};
static_assert(sizeof(ServeEntry) == 32, "eight words");

__device__ __forceinline__ EntryLanes entry_lanes(const ServeEntry* __restrict__ entries, uint32_t a, uint32_t lane)
{
  return {reinterpret_cast<const uint32_t*>(&entries[a])[lane % 8]};
}

// The part of an entry's tile that a wave tests: `count` frusta from the entry's
// frustum `first` on.
template <int K>
__device__ __forceinline__ WorkItem serve_item(const EntryLanes& e, uint32_t tile, uint32_t first, uint32_t count)
{
  WorkItem w;
  w.first_object = static_cast<uint64_t>(tile) * (kWave * K);
  const uint64_t objects = static_cast<uint64_t>(e.get(offsetof(ServeEntry, objects) + 4)) << 32 |
                           e.get(offsetof(ServeEntry, objects));
  const uint64_t left = objects - w.first_object;
  w.count = static_cast<uint32_t>(left < static_cast<uint64_t>(kWave * K) ? left : static_cast<uint64_t>(kWave * K));
  w.tile_word = tile * K;
  w.pair_begin = e.pair_begin() + first;
  w.pair_count = count;
  w.scene = e.get(offsetof(ServeEntry, scene));
  w.pad = 0;
  return w;
}

// The kernel's LDS, and the workgroups of it that a CU holds: its 160 KB are given out
// in units of 1280 bytes, so of 32 KB four fit, not five (hipOccupancyMaxActiveBlocks-
// PerMultiprocessor says five; a fifth takes as long as of 33,280 bytes).
template <int K>
struct ServeLds {
  Queue<K> queues[kBatchWaves];
  QuickView views[kBatchWaves][kServeViews];  // of each wave's current entry
};
constexpr uint32_t lds_blocks(size_t bytes) { return static_cast<uint32_t>(160 * 1024 / ((bytes + 1279) / 1280 * 1280)); }
static_assert(lds_blocks(32000) == 5 && lds_blocks(32768) == 4, "units of 1280 bytes");
template <int K>
constexpr uint32_t kServeBlocks = lds_blocks(sizeof(ServeLds<K>));
static_assert(kServeBlocks<1> == 4 && kServeBlocks<2> == 4, "launch_serve's times are of four");

template <int K>
__global__ __launch_bounds__(256, 4) void cull_serve_kernel(const ServeEntry* __restrict__ entries, uint32_t n_entries,
                                                         uint64_t total_cost, const KPair* __restrict__ pairs,
                                                         const SceneDev* __restrict__ scenes,
                                                         const float* __restrict__ vps,
                                                         unsigned long long* __restrict__ masks)
{
  __shared__ ServeLds<K> lds;
  auto& queues = lds.queues;
  auto& views = lds.views;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t waves_per_block = blockDim.x / kWave;
  const uint64_t W = static_cast<uint64_t>(gridDim.x) * waves_per_block;
  const uint32_t block_wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint64_t wave = static_cast<uint64_t>(blockIdx.x) * waves_per_block + block_wave;
  const uint64_t c0 = total_cost * wave / W, c1 = total_cost * (wave + 1) / W;
  if (c0 >= c1) return;
  // the entry of pair c0: the last that begins there or before (its cost is not 0)
  uint32_t a = 0;
  for (uint32_t base = 0; base < n_entries; base += kWave) {
    const uint32_t k = base + lane;
    a += __popcll(ballot(entries[k < n_entries ? k : 0].cost_begin <= c0 && k < n_entries));
  }
  a = __builtin_amdgcn_readfirstlane(a - 1);
  uint32_t left = static_cast<uint32_t>(c1 - c0);  // (at most a few tiles' frusta: c1 - c0 is total_cost / W)
  uint32_t tile = static_cast<uint32_t>((c0 - entries[a].cost_begin) / entries[a].pair_count);
  uint32_t first = static_cast<uint32_t>((c0 - entries[a].cost_begin) % entries[a].pair_count);
  EntryLanes e = entry_lanes(entries, a, lane);
  bool viewed = false;
  uint32_t waiting = 0, words = 0, exact = 0;
  for (;;) {
    const uint32_t listed = e.pair_count(), rest = listed - first, count = rest < left ? rest : left;
    const WorkItem item = serve_item<K>(e, tile, first, count);
    uint32_t done = 0, end = count;
    if (__builtin_expect(exact != 0, 0)) {
      --exact;
    } else if (listed > kFewFrusta) {
      Slot slot[K];
      RawObj raw[K];
      load_objects<K>(scenes, item, lane, slot, raw);
      const KPair pair = load_pairs(pairs, item, 0, lane);
      if (!viewed) {  // the entry's QuickViews, one per lane, while its first objects are in flight
        list_views(pairs + e.pair_begin(), e.pair_count(), vps, lane, views[block_wave]);
        viewed = true;
      }
      TileObjects<K> objects;
      quick_objects<K>(slot, raw, objects);
      const QuickView* const list = &views[block_wave][first];
      done = test_frusta<K>(item, objects, pair, lane, pairs, scenes, vps, masks, queues[block_wave], waiting, words,
                            [&](uint32_t, uint32_t p, uint32_t) -> const QuickView& { return list[p]; });
      // (what is left, to the end of the run: what the list's later views see may be decided again)
      end = min(done / kQuickRun * kQuickRun + kQuickRun, count);
      if (done * 4 < end) exact = kExactItems;
    }
    if (__builtin_expect(done < end, 0)) test_exact<K>(item, done, end, lane, pairs, scenes, vps, masks);
    left -= end;
    if (left == 0) break;
    first += end;
    asm volatile("" : "+v"(e.v));  // (as a new value: what was read of it would otherwise be kept)
    if (first < e.pair_count()) continue;
    first = 0;
    for (++tile; tile >= e.tiles(); tile = 0) {  // (pairs are left: an entry with tiles follows)
      e = entry_lanes(entries, ++a, lane);
      viewed = false;
    }
  }
  drain<K>(queues[block_wave], waiting, words, lane, scenes, vps, masks);
}

// Plain per-view launch: one wave per 64-object tile, the frustum by value.
__global__ __launch_bounds__(256) void cull_tiles_kernel(const ViewTile* __restrict__ tiles, uint32_t n_tiles,
                                                         const SceneDev* __restrict__ scenes, Mat16 vp,
                                                         unsigned long long* __restrict__ masks)
{
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t t = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave);
  if (t >= n_tiles) return;
  const ViewTile tile = tiles[t];
  const SceneDev sc = scenes[tile.scene];
  const Slot sl = make_slot(tile.first_object + lane, tile.first_object + tile.count, sc.xform, sc.ld);
  const bool vis = slot_visible(sl, obb_visible(obb_of(load_raw(sc.box_a, sc.box_b, sc.planes, sc.ld, sl.i, sl.m)), vp.m));
  const unsigned long long bits = __ballot(vis);
  if (lane == 0) masks[tile.mask_word] = bits;
}

}  // namespace
}  // namespace dpc

struct dpc_batch_plan {
  dpc_batch_config cfg;
  uint32_t n_frusta = 0;
  uint64_t mask_words = 0;
  uint64_t tests = 0;
  uint32_t n_items = 0;
  dpc::WorkItem* d_items = nullptr;
  dpc::KPair* d_pairs = nullptr;
  // groups read by at least one pair, for validating bound scenes
  std::vector<dpc_group_range> used_groups;
  uint32_t n_scenes_needed = 0;
  dpc::SceneDev* d_scenes = nullptr;
  uint32_t n_scenes_bound = 0;
  // per-view form
  std::vector<uint32_t> view_tile_begin;  // n_frusta + 1
  dpc::ViewTile* d_view_tiles = nullptr;
  int device = 0;
};

using namespace dpc;

namespace {

int validate_config(const dpc_batch_config& c)
{
  if (c.objects_per_lane != 1 && c.objects_per_lane != 2 && c.objects_per_lane != 4)
    return set_error(DPC_ERR_INVALID_ARGUMENT, "batch config: objects_per_lane must be 1, 2 or 4");
  if (c.block_threads != 64 && c.block_threads != 128 && c.block_threads != 256)
    return set_error(DPC_ERR_INVALID_ARGUMENT, "batch config: block_threads must be 64, 128 or 256");
  if (c.waves_per_cu == 0 || c.waves_per_cu > 64)
    return set_error(DPC_ERR_INVALID_ARGUMENT, "batch config: waves_per_cu must be 1..64");
  return DPC_OK;
}

void free_plan(dpc_batch_plan* p)
{
  if (!p) return;
  if (p->d_items) (void)hipFree(p->d_items);
  if (p->d_pairs) (void)hipFree(p->d_pairs);
  if (p->d_view_tiles) (void)hipFree(p->d_view_tiles);
  if (p->d_scenes) (void)hipFree(p->d_scenes);
  delete p;
}

}  // namespace

extern "C" {

int dpc_batch_plan_create(const dpc_group_range* groups, size_t n_groups, const dpc_cull_pair* pairs, size_t n_pairs,
                          uint32_t n_frusta, const dpc_batch_config* cfg, dpc_batch_plan** out)
{
  if (!out) return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_batch_plan_create: null output");
  *out = nullptr;
  if ((n_groups && !groups) || (n_pairs && !pairs))
    return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_batch_plan_create: null groups/pairs");
  dpc_batch_config c{1, 256, 24, 0};
  if (cfg) c = *cfg;
  int rc = validate_config(c);
  if (rc) return rc;
  for (size_t k = 0; k < n_pairs; ++k) {
    if (pairs[k].frustum >= n_frusta || pairs[k].group >= n_groups)
      return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_batch_plan_create: pair %zu names frustum %u / group %u out of range",
                       k, pairs[k].frustum, pairs[k].group);
  }
  for (size_t g = 0; g < n_groups; ++g)
    if (groups[g].count > 0xFFFFFFFFull)
      return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_batch_plan_create: group %zu has more than 2^32 objects", g);

  auto* plan = new dpc_batch_plan();
  plan->cfg = c;
  plan->n_frusta = n_frusta;
  (void)hipGetDevice(&plan->device);
  const uint64_t cus = static_cast<uint64_t>(std::max(device_cu_count(), 1));

  // Pairs grouped by group, frusta ascending within a group.
  std::vector<uint32_t> order(n_pairs);
  std::iota(order.begin(), order.end(), 0u);
  std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) {
    if (pairs[a].group != pairs[b].group) return pairs[a].group < pairs[b].group;
    return pairs[a].frustum < pairs[b].frustum;
  });
  std::vector<KPair> kp(n_pairs);
  std::vector<uint64_t> group_pair_begin(n_groups + 1, 0);
  for (size_t k = 0; k < n_pairs; ++k) {
    const dpc_cull_pair& p = pairs[order[k]];
    kp[k] = KPair{p.frustum, 0u, p.mask_word_offset};
    group_pair_begin[p.group + 1]++;
  }
  for (size_t g = 0; g < n_groups; ++g) group_pair_begin[g + 1] += group_pair_begin[g];

  const uint64_t tile_objects = static_cast<uint64_t>(kWave) * c.objects_per_lane;
  if (!cfg) {
    // Where the tiles alone would leave the device idle, lists are split into
    // slices of a length that gives about five work items per CU, of two views at
    // least (79 tiles x 64 views: 10.3 us in slices of 32, 6.0 of 4, 6.3 of 2; 625 x
    // 13: 6.8 us in slices of 16, 6.5 of 8, 6.8 of 4; 313 x 4: 5.2 us unsplit, 4.9 in
    // slices of 2, 5.1 of 1).  With eight tiles per CU a slice's second read of the
    // objects costs more than it gives (2,344 x 6: 7.6 us unsplit, 9.6 in slices of
    // 4); lists are then cut only after 16 views, so that the last items of a long
    // launch are short (1,563 x 64: 15.7 us in slices of 16, 16.2 of 32).
    uint64_t tiles = 0, tile_pairs = 0;
    for (size_t g = 0; g < n_groups; ++g) {
      const uint64_t n = group_pair_begin[g + 1] - group_pair_begin[g];
      const uint64_t t = (groups[g].count + tile_objects - 1) / tile_objects;
      tiles += n ? t : 0;
      tile_pairs += n * t;
    }
    c.max_frusta_per_item =
        tiles >= 8 * cus ? 16u : static_cast<uint32_t>(std::clamp<uint64_t>((tile_pairs + 5 * cus - 1) / (5 * cus), 2, 16));
  }
  std::vector<WorkItem> items;
  for (size_t g = 0; g < n_groups; ++g) {
    const uint64_t pb = group_pair_begin[g], pe = group_pair_begin[g + 1];
    if (pb == pe || groups[g].count == 0) continue;
    const uint64_t most = c.max_frusta_per_item ? c.max_frusta_per_item : pe - pb;
    const uint64_t slices = (pe - pb + most - 1) / most;
    const uint64_t chunk = (pe - pb + slices - 1) / slices;
    for (uint64_t t0 = 0; t0 < groups[g].count; t0 += tile_objects) {
      const uint32_t cnt = static_cast<uint32_t>(std::min<uint64_t>(tile_objects, groups[g].count - t0));
      for (uint64_t q = pb; q < pe; q += chunk) {
        WorkItem w{};
        w.scene = groups[g].scene;
        w.first_object = groups[g].first_object + t0;
        w.count = cnt;
        w.tile_word = static_cast<uint32_t>(t0 / kWave);
        w.pair_begin = static_cast<uint32_t>(q);
        w.pair_count = static_cast<uint32_t>(std::min<uint64_t>(chunk, pe - q));
        items.push_back(w);
      }
    }
  }
  // Largest items first (cost = frusta x 64-object words); lists of one length are
  // in that order already.
  const auto larger = [](const WorkItem& a, const WorkItem& b) {
    const uint64_t ca = static_cast<uint64_t>(a.pair_count) * ((a.count + 63) / 64);
    const uint64_t cb = static_cast<uint64_t>(b.pair_count) * ((b.count + 63) / 64);
    return ca > cb;
  };
  if (!std::is_sorted(items.begin(), items.end(), larger)) std::stable_sort(items.begin(), items.end(), larger);
  if (items.size() > 0xFFFFFFFFull) {
    free_plan(plan);
    return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_batch_plan_create: too many work items");
  }
  plan->n_items = static_cast<uint32_t>(items.size());

  // Per-view tiles: frustum-major, 64 objects per tile.
  std::vector<std::vector<ViewTile>> per_view(n_frusta);
  std::vector<uint64_t> view_words(n_frusta, 0);
  uint64_t all_words = 0;
  for (size_t k = 0; k < n_pairs; ++k) {
    const uint64_t words = (groups[pairs[k].group].count + 63) / 64;
    view_words[pairs[k].frustum] += words;
    all_words += words;
  }
  for (uint32_t f = 0; f < n_frusta; ++f) per_view[f].reserve(view_words[f]);
  for (size_t k = 0; k < n_pairs; ++k) {
    const dpc_cull_pair& p = pairs[k];
    const dpc_group_range& g = groups[p.group];
    const uint64_t words = (g.count + 63) / 64;
    plan->mask_words = std::max(plan->mask_words, p.mask_word_offset + words);
    plan->tests += g.count;
    for (uint64_t w = 0; w < words; ++w) {
      ViewTile vt{};
      vt.first_object = g.first_object + 64 * w;
      vt.mask_word = p.mask_word_offset + w;
      vt.count = static_cast<uint32_t>(std::min<uint64_t>(64, g.count - 64 * w));
      vt.scene = g.scene;
      per_view[p.frustum].push_back(vt);
    }
  }
  std::vector<ViewTile> flat;
  flat.reserve(all_words);
  plan->view_tile_begin.assign(n_frusta + 1, 0);
  for (uint32_t f = 0; f < n_frusta; ++f) {
    plan->view_tile_begin[f] = static_cast<uint32_t>(flat.size());
    flat.insert(flat.end(), per_view[f].begin(), per_view[f].end());
  }
  plan->view_tile_begin[n_frusta] = static_cast<uint32_t>(flat.size());
  {
    std::vector<bool> used(n_groups, false);
    for (size_t k = 0; k < n_pairs; ++k) used[pairs[k].group] = true;
    for (size_t g = 0; g < n_groups; ++g) {
      if (!used[g] || groups[g].count == 0) continue;
      plan->used_groups.push_back(groups[g]);
      plan->n_scenes_needed = std::max(plan->n_scenes_needed, groups[g].scene + 1);
    }
  }

  hipError_t e = hipSuccess;
  if (!items.empty()) {
    e = hipMalloc(&plan->d_items, items.size() * sizeof(WorkItem));
    if (e == hipSuccess)
      e = hipMemcpy(plan->d_items, items.data(), items.size() * sizeof(WorkItem), hipMemcpyHostToDevice);
  }
  if (e == hipSuccess && !kp.empty()) {
    e = hipMalloc(&plan->d_pairs, kp.size() * sizeof(KPair));
    if (e == hipSuccess) e = hipMemcpy(plan->d_pairs, kp.data(), kp.size() * sizeof(KPair), hipMemcpyHostToDevice);
  }
  if (e == hipSuccess && !flat.empty()) {
    e = hipMalloc(&plan->d_view_tiles, flat.size() * sizeof(ViewTile));
    if (e == hipSuccess)
      e = hipMemcpy(plan->d_view_tiles, flat.data(), flat.size() * sizeof(ViewTile), hipMemcpyHostToDevice);
  }
  if (e != hipSuccess) {
    free_plan(plan);
    return hip_fail(e, "dpc_batch_plan_create: upload");
  }
  *out = plan;
  return DPC_OK;
}

int dpc_batch_plan_destroy(dpc_batch_plan* plan)
{
  free_plan(plan);
  return DPC_OK;
}

int dpc_batch_plan_info(const dpc_batch_plan* plan, uint64_t* mask_words, uint64_t* tests, uint64_t* work_items)
{
  if (!plan) return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_batch_plan_info: null plan");
  if (mask_words) *mask_words = plan->mask_words;
  if (tests) *tests = plan->tests;
  if (work_items) *work_items = plan->n_items;
  return DPC_OK;
}

}  // extern "C"

namespace {
int check_bound(const dpc_batch_plan* plan, size_t mask_words, const char* who)
{
  if (!plan) return set_error(DPC_ERR_INVALID_ARGUMENT, "%s: null plan", who);
  if (plan->n_scenes_bound < plan->n_scenes_needed)
    return set_error(DPC_ERR_STATE, "%s: the plan reads %u scenes but %u are bound (dpc_batch_plan_bind)", who,
                     plan->n_scenes_needed, plan->n_scenes_bound);
  if (mask_words < plan->mask_words)
    return set_error(DPC_ERR_INVALID_ARGUMENT, "%s: mask buffer holds %zu words, the pairs need %llu", who,
                     mask_words, static_cast<unsigned long long>(plan->mask_words));
  return DPC_OK;
}
}  // namespace

extern "C" {

int dpc_batch_plan_bind(dpc_batch_plan* plan, const dpc_scene_desc* scenes, size_t n_scenes)
{
  if (!plan) return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_batch_plan_bind: null plan");
  if (n_scenes && !scenes) return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_batch_plan_bind: null scene table");
  if (n_scenes < plan->n_scenes_needed)
    return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_batch_plan_bind: the plan reads %u scenes, %zu given",
                     plan->n_scenes_needed, n_scenes);
  for (size_t k = 0; k < n_scenes; ++k) {
    const dpc_scene_desc& d = scenes[k];
    if (d.n_objects && (!d.box_a || !d.box_b || !d.planes || !aligned(d.box_a, 16) || !aligned(d.box_b, 8) ||
                        !aligned(d.planes, 16)))
      return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_batch_plan_bind: scene %zu has a null or misaligned array", k);
  }
  for (const dpc_group_range& g : plan->used_groups) {
    const dpc_scene_desc& d = scenes[g.scene];
    if (g.first_object + g.count > d.n_objects)
      return set_error(DPC_ERR_INVALID_ARGUMENT,
                       "dpc_batch_plan_bind: a group reaches object %llu of scene %u, which holds %llu",
                       static_cast<unsigned long long>(g.first_object + g.count), g.scene,
                       static_cast<unsigned long long>(d.n_objects));
    if (!d.xform && d.ld < g.first_object + g.count)
      return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_batch_plan_bind: scene %u has no indices and ld < objects",
                       g.scene);
  }
  std::vector<SceneDev> table(n_scenes);
  for (size_t k = 0; k < n_scenes; ++k) {
    table[k].box_a = reinterpret_cast<const float4*>(scenes[k].box_a);
    table[k].box_b = reinterpret_cast<const float2*>(scenes[k].box_b);
    table[k].xform = scenes[k].xform;
    table[k].planes = reinterpret_cast<const float4*>(scenes[k].planes);
    table[k].ld = scenes[k].ld;
    table[k].n_objects = scenes[k].n_objects;
  }
  if (n_scenes > plan->n_scenes_bound || !plan->d_scenes) {
    if (plan->d_scenes) (void)hipFree(plan->d_scenes);
    plan->d_scenes = nullptr;
    plan->n_scenes_bound = 0;
    DPC_HIP_TRY(hipMalloc(&plan->d_scenes, std::max<size_t>(n_scenes, 1) * sizeof(SceneDev)), "hipMalloc scenes");
  }
  if (n_scenes)
    DPC_HIP_TRY(hipMemcpy(plan->d_scenes, table.data(), n_scenes * sizeof(SceneDev), hipMemcpyHostToDevice),
                "upload scene table");
  plan->n_scenes_bound = static_cast<uint32_t>(n_scenes);
  return DPC_OK;
}

int dpc_cull_batch(const dpc_batch_plan* plan, const float* d_vps, uint64_t* d_masks, size_t mask_words,
                   void* stream)
{
  if (int rc = check_bound(plan, mask_words, "dpc_cull_batch")) return rc;
  if (plan->n_items == 0) return DPC_OK;
  if (!d_vps || !d_masks || !aligned(d_masks, 8) || !aligned(d_vps, 4))
    return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_cull_batch: null or misaligned frusta/masks");
  const dpc_batch_config& c = plan->cfg;
  const uint32_t waves_per_block = c.block_threads / kWave;
  uint64_t blocks = static_cast<uint64_t>(device_cu_count()) * c.waves_per_cu / waves_per_block;
  const uint64_t needed = (plan->n_items + waves_per_block - 1) / waves_per_block;
  if (blocks > needed) blocks = needed;
  if (blocks == 0) blocks = 1;
  const dim3 grid(static_cast<unsigned>(blocks)), block(c.block_threads);
  auto* m = reinterpret_cast<unsigned long long*>(d_masks);
  hipStream_t s = as_stream(stream);
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, block, 0, s, plan->d_items, plan->n_items, plan->d_pairs, plan->d_scenes, d_vps,
                       plan->n_frusta, m);
  };
  const bool table = plan->n_frusta <= kTableViews;
  switch (c.objects_per_lane) {
    case 1:
      table ? launch(cull_batch_kernel<1, true>) : launch(cull_batch_kernel<1, false>);
      break;
    case 2:
      table ? launch(cull_batch_kernel<2, true>) : launch(cull_batch_kernel<2, false>);
      break;
    default:
      table ? launch(cull_batch_kernel<4, true>) : launch(cull_batch_kernel<4, false>);
      break;
  }
  return check_launch("cull_batch_kernel");
}

}  // extern "C"

namespace dpc {
// Launches one serving batch (see ServeEntry).  d_entries/d_pairs/d_vps/d_masks
// live on the device; total_cost and n_entries come from the host copy.
// Copy-out of a serving batch's masks: blockIdx.y = the request, threads take
// consecutive 64-bit words (a wave writes 512 contiguous bytes per store).
// The destinations are pinned host memory, which device stores reach directly.
__global__ __launch_bounds__(256) void copy_out_kernel(const CopyOut* __restrict__ copies, const char* __restrict__ arena)
{
  const CopyOut c = copies[blockIdx.y];
  const auto* src = reinterpret_cast<const unsigned long long*>(arena + c.src_offset);
  for (uint64_t w = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x; w < c.words;
       w += static_cast<uint64_t>(gridDim.x) * 256)
    c.dst[w] = src[w];
}

int launch_copy_out(const void* d_copies, uint32_t n, const char* d_arena, uint64_t max_words, void* stream_handle)
{
  if (n == 0 || max_words == 0) return DPC_OK;
  if (n > 65535) return set_error(DPC_ERR_INVALID_ARGUMENT, "launch_copy_out: more than 65535 ranges");
  // enough blocks per range for its words, at most 64 (then each thread loops)
  const uint64_t per = (max_words + 255) / 256;
  const unsigned bx = static_cast<unsigned>(per < 64 ? per : 64);
  hipLaunchKernelGGL(copy_out_kernel, dim3(bx, n), dim3(256), 0, as_stream(stream_handle),
                     static_cast<const CopyOut*>(d_copies), d_arena);
  return check_launch("copy_out_kernel");
}

int launch_serve(const void* d_entries, uint32_t n_entries, uint64_t total_cost, uint64_t tiles, const void* d_pairs,
                 const void* d_scenes, const float* d_vps, uint64_t* d_masks, uint32_t objects_per_lane,
                 uint32_t waves_per_cu, void* stream_handle)
{
  hipStream_t stream = as_stream(stream_handle);
  if (n_entries == 0 || total_cost == 0) return DPC_OK;
  const uint32_t waves_per_block = 4;
  // A small batch is split into runs of a length that gives about five waves per CU,
  // as a batch plan's lists are (dpc_batch_plan_create); a large one into as many
  // runs as the device holds waves: with a workgroup per CU more, a fifth of the equal
  // runs starts when the others end (1,000,003 objects x 32 views of which the quick
  // test decides nothing: 307 us a tick, 282 without; ordinary 168 to 175, 168).  Up to
  // that number each tile has a wave: with less than 16 frusta a run of 16 pairs passes
  // over several tiles, and a wave has one tile's objects in flight at a time (500,000
  // objects x 1 17.4 -> 13.1 us, 1,000,000 x 1 26.4 -> 18.9, x 4 22.6 -> 22.4).  Runs of
  // one pair are for batches that take the exact test; the quick test reads the objects
  // for two at least (10,000 x 2 5.6 -> 4.2 us).
  const uint64_t cus = device_cu_count();
  const uint32_t held = waves_per_block * (objects_per_lane == 2 ? kServeBlocks<2> : kServeBlocks<1>);
  uint64_t waves = cus * (waves_per_cu ? waves_per_cu : held);
  const uint64_t run =
      std::clamp<uint64_t>((total_cost + 5 * cus - 1) / (5 * cus), total_cost <= kFewFrusta * tiles ? 1 : 2, 16);
  waves = std::min(waves, std::max(total_cost / run, tiles));
  if (waves == 0) waves = 1;
  const uint64_t blocks = (waves + waves_per_block - 1) / waves_per_block;
  const auto* e = static_cast<const ServeEntry*>(d_entries);
  const auto* p = static_cast<const KPair*>(d_pairs);
  const auto* sc = static_cast<const SceneDev*>(d_scenes);
  auto* m = reinterpret_cast<unsigned long long*>(d_masks);
  switch (objects_per_lane) {
    case 2:
      hipLaunchKernelGGL(cull_serve_kernel<2>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, e, n_entries,
                         total_cost, p, sc, d_vps, m);
      break;
    default:
      hipLaunchKernelGGL(cull_serve_kernel<1>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, e, n_entries,
                         total_cost, p, sc, d_vps, m);
      break;
  }
  return check_launch("cull_serve_kernel");
}
}  // namespace dpc

extern "C" {

int dpc_cull_per_view(const dpc_batch_plan* plan, const float* h_vps, uint64_t* d_masks, size_t mask_words,
                      void* stream)
{
  if (int rc = check_bound(plan, mask_words, "dpc_cull_per_view")) return rc;
  if (!h_vps || !d_masks || !aligned(d_masks, 8))
    return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_cull_per_view: null or misaligned frusta/masks");
  auto* m = reinterpret_cast<unsigned long long*>(d_masks);
  hipStream_t s = as_stream(stream);
  for (uint32_t f = 0; f < plan->n_frusta; ++f) {
    const uint32_t t0 = plan->view_tile_begin[f], t1 = plan->view_tile_begin[f + 1];
    if (t0 == t1) continue;
    Mat16 vp;
    std::memcpy(vp.m, h_vps + 16 * static_cast<size_t>(f), sizeof vp.m);
    const uint32_t n = t1 - t0;
    const unsigned blocks = (n + 3) / 4;
    hipLaunchKernelGGL(cull_tiles_kernel, dim3(blocks), dim3(256), 0, s, plan->d_view_tiles + t0, n, plan->d_scenes,
                       vp, m);
    int rc = check_launch("cull_tiles_kernel");
    if (rc) return rc;
  }
  return DPC_OK;
}

}  // extern "C"

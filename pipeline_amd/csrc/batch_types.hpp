// batch_types.hpp -- device-visible descriptor layouts shared by the batched
// kernels (batch.hip) and the host code that fills them (host/Serving.cpp).
#pragma once
#include <cstdint>

namespace dpc {

// One (frustum, group) pair of a batch: the frustum's index in the batch's
// matrix array and the first 64-bit mask word of its result.
struct KPair {
  uint32_t frustum;
  uint32_t pad;
  uint64_t mask_word;
};
static_assert(sizeof(KPair) == 16, "KPair layout");

// One request of a serving batch: the whole scene against pairs
// [pair_begin, pair_begin + pair_count).  cost_begin = sum of tiles * pair_count
// over the earlier entries (the kernel splits the total cost evenly over waves).
struct ServeEntry {
  uint32_t scene;
  uint32_t pair_begin;
  uint32_t pair_count;
  uint32_t tiles;  // ceil(objects / (64 * objects_per_lane))
  uint64_t cost_begin;
  uint64_t objects;
};
static_assert(sizeof(ServeEntry) == 32, "ServeEntry layout");

// Launches one serving batch; every pointer is device memory.  total_cost is the sum of
// the entries' tiles times frusta, tiles that of their tiles.
int launch_serve(const void* d_entries, uint32_t n_entries, uint64_t total_cost, uint64_t tiles, const void* d_pairs,
                 const void* d_scenes, const float* d_vps, uint64_t* d_masks, uint32_t objects_per_lane,
                 uint32_t waves_per_cu, void* stream);

// Scatters count delta matrices (16 floats each, row-major) into row planes,
// reading the indices and matrices from pinned host memory (device-visible
// pointers) with system-coherent loads; no copy is needed before it.  At most
// kMaxHostScatter matrices into at most kMaxHostScatterLd slots (32-bit byte
// offsets).
constexpr uint32_t kMaxHostScatter = 1u << 25;
constexpr uint32_t kMaxHostScatterLd = (1u << 26) - 1;
int launch_scatter_host(float* d_planes, size_t ld, const uint32_t* idx, const float* src, size_t count,
                        void* stream);

// One packed delta of a batch's arena (byte offsets, 16-byte aligned): count
// indices; matrix k as three 16-byte rows, (row i's x y z, row 3's component i)
// for i = 0, 1, 2; and the last columns (m[3], m[7], m[11], m[15]) as 16 bytes
// each, or, with tails 0, 0 0 0 1 for every matrix.  Its matrices go to `planes`
// (row planes of ld slots); every value is moved as its bits.
struct StageJob {
  float* planes;
  uint64_t ld;
  uint32_t idx, packed, tails;
  uint32_t count;
};
static_assert(sizeof(StageJob) == 32, "StageJob layout");

// Scatters the n jobs' deltas out of an arena of `bytes` bytes (below 2^31), in one
// launch; the jobs travel by value in its arguments, at most kStageJobs.  With
// d_arena set the arena lies in pinned host memory and its first desc_bytes bytes
// (a multiple of 16) are copied to d_arena as well: a batch's whole upload in one
// launch.  With d_arena null it is device memory, and the deltas are scattered only.
constexpr uint32_t kStageJobs = 64;
int launch_stage(const char* arena, uint64_t bytes, char* d_arena, uint64_t desc_bytes, const StageJob* jobs, uint32_t n,
                 void* stream);

// One request's masks to its caller's buffer in pinned host memory: `words`
// 64-bit words from byte offset src_offset of the batch arena to dst (the
// buffer's device-visible address).
struct CopyOut {
  uint64_t src_offset;
  uint64_t words;
  uint64_t* dst;
  uint64_t pad;
};
static_assert(sizeof(CopyOut) == 32, "CopyOut layout");

// Copies n CopyOut ranges (d_copies: device memory) out of the arena in one
// launch; the device writes the callers' pinned buffers itself, in 512-byte
// wave-wide stores, instead of a DMA transfer per request.
int launch_copy_out(const void* d_copies, uint32_t n, const char* d_arena, uint64_t max_words, void* stream);

}  // namespace dpc

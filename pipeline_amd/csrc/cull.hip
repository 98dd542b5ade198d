// cull.hip -- single-frustum culling, layout conversion, matrix deltas,
// group bounding box and result diff.
//
// Reference path: dp::culling::cpu::ManagerImpl::cull
// (dp/culling/cpu/src/ManagerImpl.cpp:467-518), GroupCPU::updateOBBs (:114-162),
// ManagerBitSet::calculateBoundingBox (dp/culling/src/ManagerBitSet.cpp:268-306)
// and ResultBitSet::updateChanged (dp/culling/src/ResultBitSet.cpp:61-108).
#include <algorithm>
#include <atomic>
#include <cfloat>
#include <mutex>
#include <type_traits>

#include "cull_math.hpp"
#include "cull_shape.hpp"
#include "internal.hpp"
#include "batch_types.hpp"

#pragma clang fp contract(off)

namespace dpc {
namespace {

constexpr unsigned kCullThreads = 256;  // persistent streaming form
constexpr unsigned kIndexedThreads = 512;  // plain form with an index array
constexpr unsigned kPlainThreads = 1024;  // plain form without an index array
constexpr unsigned kSmallThreads = 64;    // ... of short calls (flat_cull_threads)

// With Diff (the cull of Manager::cull, which the result diff follows), the
// wave that stores mask word w also stores the number of bits in which it
// differs from old[w] (bits below n only) as count[w], one byte per word:
// the write pass of the diff then needs no counting launch of its own.
__device__ __forceinline__ uint8_t changed_in_word(unsigned long long old_bits, unsigned long long new_bits, size_t w,
                                                   size_t n)
{
  unsigned long long x = old_bits ^ new_bits;
  const size_t tail = n & 63;
  if (tail && w == (n >> 6)) x &= (~0ull) >> (64 - tail);
  return static_cast<uint8_t>(__popcll(x));
}

// Plain form: one object per lane, one 64-object tile per wave, a grid that
// covers all tiles.  The object's four matrix rows come from four row planes,
// so every load of the wave is one contiguous 1 KiB (rows, box_a) or 512 B
// (box_b) segment; the visibility bits leave as one ballot word per wave.
// Without an index array every box and matrix is read once per launch, so
// they are loaded as streaming data, in blocks of 1024 threads or of one wave
// (flat_cull_threads); with one (matrices shared by several objects, e.g. the
// leaves of a transform tree), plain cached loads in 512-thread blocks measured
// fastest (19.3 us against 19.5-19.7 us with 256 threads for the 2.37M objects of
// a 1M-node tree; long calls take two tiles per wave, below).
template <bool Indexed, bool Diff, unsigned Threads>
__global__ __launch_bounds__(Threads) void cull_kernel(const float4* __restrict__ box_a,
                                                            const float2* __restrict__ box_b,
                                                            const uint32_t* __restrict__ xform, size_t n,
                                                            const float4* __restrict__ planes, size_t ld, Mat16 vp,
                                                            unsigned long long* __restrict__ mask,
                                                            const unsigned long long* __restrict__ old,
                                                            uint8_t* __restrict__ count)
{
  const size_t i = static_cast<size_t>(blockIdx.x) * Threads + threadIdx.x;
  const bool writer = (threadIdx.x & (kWave - 1)) == 0 && i < n;  // lane 0 of a wave holding objects
  const unsigned long long old_bits = Diff && writer ? old[i >> 6] : 0ull;  // loaded with the objects
  const Slot s = make_slot(i, n, Indexed ? xform : nullptr, ld);
  const RawObj r = Indexed ? load_raw(box_a, box_b, planes, ld, s.i, s.m)
                           : load_raw_stream<true>(box_a, box_b, planes, ld, s.i, s.m);
  const bool vis = slot_visible(s, obb_visible(obb_of(r), vp.m));
  const unsigned long long bits = __ballot(vis);
  if (writer) {
    mask[i >> 6] = bits;
    if (Diff) count[i >> 6] = changed_in_word(old_bits, bits, i >> 6, n);
  }
}

// The same, two adjacent tiles per wave (launch_cull: where): both tiles' indices,
// then both tiles' boxes and rows are in flight together, and half as many waves
// start and end.
constexpr unsigned kPairThreads = 256;

template <bool Diff>
__global__ __launch_bounds__(kPairThreads) void cull_pair_kernel(const float4* __restrict__ box_a,
                                                                 const float2* __restrict__ box_b,
                                                                 const uint32_t* __restrict__ xform, size_t n,
                                                                 const float4* __restrict__ planes, size_t ld, Mat16 vp,
                                                                 unsigned long long* __restrict__ mask,
                                                                 const unsigned long long* __restrict__ old,
                                                                 uint8_t* __restrict__ count)
{
  const unsigned lane = threadIdx.x & (kWave - 1);
  const size_t first = (static_cast<size_t>(blockIdx.x) * kPairThreads + (threadIdx.x & ~(kWave - 1u))) * 2 + lane;
  Slot s[2];
  RawObj r[2];
  unsigned long long old_bits[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const size_t i = first + kWave * k;
    old_bits[k] = Diff && lane == 0 && i < n ? old[i >> 6] : 0ull;
    s[k] = make_slot(i, n, xform, ld);
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) r[k] = load_raw(box_a, box_b, planes, ld, s[k].i, s[k].m);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const size_t i = first + kWave * k;
    const unsigned long long bits = __ballot(slot_visible(s[k], obb_visible(obb_of(r[k]), vp.m)));
    if (lane == 0 && i < n) {
      mask[i >> 6] = bits;
      if (Diff) count[i >> 6] = changed_in_word(old_bits[k], bits, i >> 6, n);
    }
  }
}

// Streaming form: a persistent grid in which every wave walks tiles t, t+W,
// t+2W, ... with two register sets: while one tile is tested, the loads of the
// next one are in flight.  Every wave runs the same number of steps (tiles past
// the end load clamped indices and store nothing), so all loads are
// unconditional and the wait before each compute covers only that tile's loads.
template <bool Indexed, bool Diff>
__device__ __forceinline__ void stream_fetch(const float4* __restrict__ box_a, const float2* __restrict__ box_b,
                                             const uint32_t* __restrict__ xform, size_t n,
                                             const float4* __restrict__ planes, size_t ld, size_t tile, unsigned lane,
                                             const unsigned long long* __restrict__ old, Slot& s, RawObj& r,
                                             unsigned long long& old_bits)
{
  s = make_slot(tile * kWave + lane, n, Indexed ? xform : nullptr, ld);
  r = load_raw(box_a, box_b, planes, ld, s.i, s.m);
  old_bits = Diff && lane == 0 && tile * kWave < n ? old[tile] : 0ull;
  // keep the loads issued here, ahead of the test of the previous tile (the
  // scheduler would otherwise sink them below it to shorten register lifetimes)
  __builtin_amdgcn_sched_barrier(0);
}

template <bool Diff>
__device__ __forceinline__ void stream_test(const Slot& s, const RawObj& r, const Mat16& vp, size_t tile, size_t n,
                                            size_t n_tiles, unsigned lane, unsigned long long* __restrict__ mask,
                                            unsigned long long old_bits, uint8_t* __restrict__ count)
{
  const bool vis = slot_visible(s, obb_visible(obb_of(r), vp.m));
  const unsigned long long bits = __ballot(vis);
  if (lane == 0 && tile < n_tiles) {
    mask[tile] = bits;
    if (Diff) count[tile] = changed_in_word(old_bits, bits, tile, n);
  }
}

template <bool Indexed, bool Diff>
__global__ __launch_bounds__(kCullThreads) void cull_stream_kernel(const float4* __restrict__ box_a,
                                                                   const float2* __restrict__ box_b,
                                                                   const uint32_t* __restrict__ xform, size_t n,
                                                                   const float4* __restrict__ planes, size_t ld,
                                                                   Mat16 vp, unsigned long long* __restrict__ mask,
                                                                   const unsigned long long* __restrict__ old,
                                                                   uint8_t* __restrict__ count)
{
  const unsigned lane = threadIdx.x & (kWave - 1);
  const size_t waves_per_block = blockDim.x / kWave;
  const size_t W = static_cast<size_t>(gridDim.x) * waves_per_block;
  const size_t n_tiles = (n + kWave - 1) / kWave;
  const size_t steps = (n_tiles + W - 1) / W;  // the same for every wave
  size_t t = static_cast<size_t>(blockIdx.x) * waves_per_block + threadIdx.x / kWave;
  Slot sa, sb;
  RawObj ra, rb;
  unsigned long long oa, ob;
  stream_fetch<Indexed, Diff>(box_a, box_b, xform, n, planes, ld, t, lane, old, sa, ra, oa);
  for (size_t k = 0; k < steps; k += 2) {
    stream_fetch<Indexed, Diff>(box_a, box_b, xform, n, planes, ld, t + W, lane, old, sb, rb, ob);
    stream_test<Diff>(sa, ra, vp, t, n, n_tiles, lane, mask, oa, count);
    if (k + 1 >= steps) break;
    stream_fetch<Indexed, Diff>(box_a, box_b, xform, n, planes, ld, t + 2 * W, lane, old, sa, ra, oa);
    stream_test<Diff>(sb, rb, vp, t + W, n, n_tiles, lane, mask, ob, count);
    t += 2 * W;
  }
}

// Row planes <- AoS matrices with a byte stride.  One thread per (matrix, row).
__global__ void from_aos_kernel(const char* __restrict__ aos, size_t stride, size_t count, float4* __restrict__ planes,
                                size_t ld)
{
  const size_t t = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= count * 4) return;
  const size_t k = t >> 2, r = t & 3;
  const float* src = reinterpret_cast<const float*>(aos + k * stride) + 4 * r;
  planes[r * ld + k] = make_float4(src[0], src[1], src[2], src[3]);
}

__global__ void to_aos_kernel(const float4* __restrict__ planes, size_t ld, const uint32_t* __restrict__ slot,
                              size_t count, char* __restrict__ aos, size_t stride)
{
  const size_t t = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= count * 4) return;
  const size_t k = t >> 2, r = t & 3;
  const size_t s = slot ? static_cast<size_t>(slot[k]) : k;
  float* dst = reinterpret_cast<float*>(aos + k * stride) + 4 * r;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  if (s < ld) v = planes[r * ld + s];
  dst[0] = v.x;
  dst[1] = v.y;
  dst[2] = v.z;
  dst[3] = v.w;
}

__global__ void scatter_kernel(float4* __restrict__ planes, size_t ld, const uint32_t* __restrict__ idx,
                               const float4* __restrict__ src, size_t count)
{
  const size_t t = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= count * 4) return;
  const size_t k = t >> 2, r = t & 3;
  const size_t s = idx[k];
  if (s < ld) planes[r * ld + s] = src[k * 4 + r];
}

// The same scatter with the delta read straight from pinned host memory:
// system-coherent 16-byte buffer loads (sc0 sc1: they see the host's writes
// and are not kept in device caches), so no copy precedes it.  A small grid
// strides over the rows: enough loads in flight to fill PCIe, few waves
// holding CUs while they wait on it.
constexpr int kSystemCoherent = 17;  // buffer load cache policy: sc0 | sc1
constexpr int kRawBuffer = 0x00020000;
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void scatter_host_kernel(float4* __restrict__ planes, uint32_t ld, const uint32_t* idx,
                                                           const float* src, uint32_t count)
{
  const __amdgpu_buffer_rsrc_t ri =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(idx), 0, count * 4u, kRawBuffer);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src), 0, count * 64u, kRawBuffer);
  // the four row planes as one buffer (ld <= kMaxHostScatterLd keeps it below 4 GB)
  const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(planes, 0, ld * 64u, kRawBuffer);
  const uint32_t rows = count * 4u;
  for (uint32_t t = blockIdx.x * 256u + threadIdx.x; t < rows; t += gridDim.x * 256u) {
    const uint32_t k = t >> 2, r = t & 3u;
    // both loads issue before either is waited for; the store is issued on
    // every path (an index outside the planes gets an offset the hardware drops)
    const uint32_t s = __builtin_amdgcn_raw_buffer_load_b32(ri, k * 4u, 0, kSystemCoherent);
    const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(rs, t * 16u, 0, kSystemCoherent);
    __builtin_amdgcn_raw_buffer_store_b128(v, rp, s < ld ? (r * ld + s) * 16u : 0xFFFFFFF0u, 0, 0);
  }
}

// A batch's deltas out of its arena (launch_stage), and from pinned host memory
// its descriptors too.  The work is cut into units of one wave: kStageChunk
// 16-byte chunks of the descriptors first, then 64 matrices of a job each (192
// chunks: three coalesced loads per lane, through LDS to the lane of their
// matrix, which stores one 16-byte row to each plane).
//
// What bounds it: PCIe, where the arena is on the host, and the chain of a batch's
// launches, where it is small.  After a DMA copy the first scatter waited 15 to
// 60 us for the copy's signal, and eight scatters of 5 us followed each other; one
// launch that reads the host's arena itself has neither.  One request for each of
// 16 scenes: 428 to 436 us a tick with a copy and scatters, 382 to 396 with this.
constexpr uint32_t kStageChunk = 192;
// 16 workgroups of 13 KB in flight fill PCIe (1 MB: 32 us with 16, 37 with 64 or
// more, of which 11 are a launch and its completion).
constexpr uint32_t kStageHostBlocks = 16;

struct StageJobs {
  StageJob job[kStageJobs];
  uint32_t first_unit[kStageJobs];
  uint32_t n, units, desc_units, desc_chunks;
};

template <bool Host>
__global__ __launch_bounds__(256) void stage_kernel(const char* arena, uint32_t bytes, u32x4_t* __restrict__ d_arena,
                                                    StageJobs jobs)
{
  __shared__ u32x4_t lds[4][kStageChunk];
  constexpr int policy = Host ? kSystemCoherent : 0;
  const __amdgpu_buffer_rsrc_t src =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(arena), 0, static_cast<int>(bytes), kRawBuffer);
  const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64u);
  uint32_t j = 0;
  for (uint32_t u = blockIdx.x * 4u + wave; u < jobs.units; u += gridDim.x * 4u) {
    if (u < jobs.desc_units) {
      const uint32_t c = u * kStageChunk + lane;
      const u32x4_t v0 = __builtin_amdgcn_raw_buffer_load_b128(src, c * 16u, 0, policy);
      const u32x4_t v1 = __builtin_amdgcn_raw_buffer_load_b128(src, (c + 64u) * 16u, 0, policy);
      const u32x4_t v2 = __builtin_amdgcn_raw_buffer_load_b128(src, (c + 128u) * 16u, 0, policy);
      if (c < jobs.desc_chunks) d_arena[c] = v0;
      if (c + 64u < jobs.desc_chunks) d_arena[c + 64u] = v1;
      if (c + 128u < jobs.desc_chunks) d_arena[c + 128u] = v2;
      continue;
    }
    while (j + 1 < jobs.n && jobs.first_unit[j + 1] <= u) ++j;
    const StageJob job = jobs.job[j];
    const uint32_t base = (u - jobs.first_unit[j]) * 64u, k = base + lane;
    // (loads past the job's end read what follows in the arena, or zero past that)
    const uint32_t s = __builtin_amdgcn_raw_buffer_load_b32(src, job.idx + k * 4u, 0, policy);
    const uint32_t at = job.packed + base * 48u + lane * 16u;
    const u32x4_t v0 = __builtin_amdgcn_raw_buffer_load_b128(src, at, 0, policy);
    const u32x4_t v1 = __builtin_amdgcn_raw_buffer_load_b128(src, at + 1024u, 0, policy);
    const u32x4_t v2 = __builtin_amdgcn_raw_buffer_load_b128(src, at + 2048u, 0, policy);
    u32x4_t w = {0u, 0u, 0u, 0x3f800000u};  // the bits of 0.0f, 0.0f, 0.0f, 1.0f
    if (job.tails) w = __builtin_amdgcn_raw_buffer_load_b128(src, job.tails + k * 16u, 0, policy);
    lds[wave][lane] = v0;
    lds[wave][lane + 64u] = v1;
    lds[wave][lane + 128u] = v2;
    wave_lds_order();
    const u32x4_t a = lds[wave][3 * lane], b = lds[wave][3 * lane + 1], c = lds[wave][3 * lane + 2];
    wave_lds_order();
    if (k < job.count && s < job.ld) {
      u32x4_t* const planes = reinterpret_cast<u32x4_t*>(job.planes);
      planes[s] = u32x4_t{a.x, a.y, a.z, w.x};
      planes[job.ld + s] = u32x4_t{b.x, b.y, b.z, w.y};
      planes[2 * job.ld + s] = u32x4_t{c.x, c.y, c.z, w.z};
      planes[3 * job.ld + s] = u32x4_t{a.w, b.w, c.w, w.w};
    }
  }
}

__global__ void gather_u32_kernel(const uint32_t* __restrict__ table, size_t table_len,
                                  const uint32_t* __restrict__ idx, size_t n, uint32_t* __restrict__ out)
{
  const size_t k = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const size_t i = idx[k];
  out[k] = i < table_len ? table[i] : 0xFFFFFFFFu;
}

__global__ void boxes_kernel(const float* __restrict__ lu, size_t n, float4* __restrict__ box_a,
                             float2* __restrict__ box_b)
{
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float* b = lu + 6 * i;
  // ManagerBitSet.cpp:102-103: lowerLeft = (lower, 1), extent = (upper - lower, 0).
  box_a[i] = make_float4(b[0], b[1], b[2], b[3] - b[0]);
  box_b[i] = make_float2(b[4] - b[1], b[5] - b[2]);
}

// ---- group bounding box -----------------------------------------------------
// Box4f::update (dp/math/Boxnt.h:245-258) keeps the running value unless the new
// point is strictly smaller (lower) / larger (upper).  That is "leftmost extremum"
// selection, which is associative over ordered ranges: combining a range with the
// range that follows it, left operand first, reproduces the sequential scan bit for
// bit (including which of +0/-0 survives and that NaN never enters).
struct __align__(8) Box6 {  // (8-byte aligned: a partial box loads as three dwordx2)
  float lo[3], hi[3];
};

__device__ __forceinline__ void box_take(Box6& acc, const float4& p)
{
  if (acc.lo[0] > p.x) acc.lo[0] = p.x;
  if (acc.hi[0] < p.x) acc.hi[0] = p.x;
  if (acc.lo[1] > p.y) acc.lo[1] = p.y;
  if (acc.hi[1] < p.y) acc.hi[1] = p.y;
  if (acc.lo[2] > p.z) acc.lo[2] = p.z;
  if (acc.hi[2] < p.z) acc.hi[2] = p.z;
}

__device__ __forceinline__ Box6 box_empty()
{
  Box6 b;
  for (int c = 0; c < 3; ++c) {
    b.lo[c] = FLT_MAX;
    b.hi[c] = -FLT_MAX;
  }
  return b;
}

constexpr unsigned kBoxThreads = 256;
constexpr unsigned kBoxWavesPerBlock = kBoxThreads / kWave;
constexpr unsigned kBoxWavesPerCu = 16;

// Box4f::update's comparison: the running value unless the other is strictly lower
// (higher); a NaN never enters.
__device__ __forceinline__ float lower(float a, float b) { return b < a ? b : a; }
__device__ __forceinline__ float higher(float a, float b) { return b > a ? b : a; }

// The minimum and maximum instructions themselves, for the eight corners of an
// object: of a number and a NaN the number, and denormals kept, like the
// comparisons above.  (fminf may not assume what is true here, that no operand is
// a signalling NaN, and takes two more instructions.)  Only the sign of a zero
// may differ from the first of equal values.  Their results go to comparisons
// only: an instruction that reads another lane's register needs distance from
// the write, which the compiler does not see in here.
__device__ __forceinline__ float vmin(float a, float b)
{
  float r;
  asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float vmax(float a, float b)
{
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float vmin3(float a, float b, float c)
{
  float r;
  asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float vmax3(float a, float b, float c)
{
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float vmin8(const float (&v)[8])
{
  return vmin(vmin3(vmin3(v[0], v[1], v[2]), v[3], v[4]), vmin3(v[5], v[6], v[7]));
}
__device__ __forceinline__ float vmax8(const float (&v)[8])
{
  return vmax(vmax3(vmax3(v[0], v[1], v[2]), v[3], v[4]), vmax3(v[5], v[6], v[7]));
}

// The sign of a zero extremum.  Folding objects in index order with strict
// comparisons keeps the first of equal values (the reference's sequential
// Box4f::update, Boxnt.h:245-258), and equal values differ only where both are
// zeros.  An extremum of zero therefore has the sign of the first zero among the
// points (in a coordinate whose lowest value is zero every zero is the lowest), so
// the values are folded without regard to order and the first zero is kept beside
// them: its place in the order, and its sign in bit 0 (kNoZero: none).
constexpr uint32_t kNoZero = 0xFFFFFFFFu;

// A value's bits with the sign of the first zero where it is a zero.
__device__ __forceinline__ float with_zero_sign(float v, uint32_t zero)
{
  return v == 0.0f && zero != kNoZero ? __uint_as_float((zero & 1u) << 31) : v;
}

// One step of a wave reduction by data-parallel primitives: each lane takes the
// value of another, or its own where the pattern gives it none.
template <int Ctrl, int RowMask>
__device__ __forceinline__ uint32_t dpp_from(uint32_t v)
{
  return __builtin_amdgcn_update_dpp(v, v, Ctrl, RowMask, 0xf, false);
}

template <class Op>
__device__ __forceinline__ uint32_t wave_fold(uint32_t v, Op&& op)  // the result: in lane 63
{
  v = op(v, dpp_from<0x111, 0xf>(v));  // row_shr:1
  v = op(v, dpp_from<0x112, 0xf>(v));  // row_shr:2
  v = op(v, dpp_from<0x114, 0xf>(v));  // row_shr:4
  v = op(v, dpp_from<0x118, 0xf>(v));  // row_shr:8
  v = op(v, dpp_from<0x142, 0xa>(v));  // row_bcast:15 into rows 1 and 3
  v = op(v, dpp_from<0x143, 0xc>(v));  // row_bcast:31 into rows 2 and 3
  return __builtin_amdgcn_readlane(static_cast<int>(v), kWave - 1);
}
__device__ __forceinline__ float wave_min(float v)
{
  return __uint_as_float(wave_fold(__float_as_uint(v), [](uint32_t a, uint32_t b) {
    return __float_as_uint(lower(__uint_as_float(a), __uint_as_float(b)));
  }));
}
__device__ __forceinline__ float wave_max(float v)
{
  return __uint_as_float(wave_fold(__float_as_uint(v), [](uint32_t a, uint32_t b) {
    return __float_as_uint(higher(__uint_as_float(a), __uint_as_float(b)));
  }));
}
__device__ __forceinline__ uint32_t wave_first(uint32_t v)
{
  return wave_fold(v, [](uint32_t a, uint32_t b) { return a < b ? a : b; });
}

// One object's inputs to the bounding box: its box and its matrix's rows (row
// index clamped to 0 when it lies outside the array; such an object is skipped).
struct BoxIn {
  float4 a;
  float2 b;
  float4 r0, r1, r2, r3;
};

__device__ __forceinline__ BoxIn load_box_in(const float4* __restrict__ box_a, const float2* __restrict__ box_b,
                                             const float4* __restrict__ planes, size_t ld, size_t i, size_t m)
{
  const size_t c = m < ld ? m : 0;
  BoxIn d;
  d.a = box_a[i];
  d.b = box_b[i];
  d.r0 = planes[c];
  d.r1 = planes[ld + c];
  d.r2 = planes[2 * ld + c];
  d.r3 = planes[3 * ld + c];
  return d;
}

// Each wave scans one contiguous chunk of objects, lane l taking objects
// begin + l, begin + l + 64, ... (coalesced loads): a lane folds its objects'
// corners into its running box, the wave its lanes', thread 0 the workgroup's four
// waves' (consecutive chunks), and one partial per workgroup is stored, in index
// order of the chunks.
//
// What bounds it: reading the objects.  Beside that, minima and maxima of values
// take 36 instructions per object and 80 per wave, where an extremum with its
// object's index took 120 and, through LDS permutes, 430.  A call over 2,400,000
// objects in the order of their matrices: 29.4 -> 25.9 us (104 MB; the cull that
// reads the same takes 24.0); 600,011: 13.9 -> 11.3.
//
// With matrices in no order each row is a 128-byte line of its own, shared only
// with other objects' rows of the same plane.  A wave that finds its first 64
// matrices in 32 lines or more therefore takes up to three rounds at once, row by
// row: all waves read one plane at a time, and of a plane, unlike of four, an XCD's
// L2 holds a good part (600,011 objects over 200,003 matrices, 3.2 MB a plane: 46 %
// of the reads hit instead of 28 %, 40.0 -> 33.2 us; 400,000: 25.7 -> 20.4; 250,000,
// a round per wave: 14.7 -> 13.8; 2,400,000: 171 -> 163).  In order, where the reads
// share their lines, that waits more often (2,400,000 objects: 29.4 us against 25.9;
// 250,000: 10.1 against 8.4), so those waves keep two sets of inputs in turn.
template <bool Indexed>
__global__ __launch_bounds__(kBoxThreads) void bbox_partial_kernel(const float4* __restrict__ box_a,
                                                                   const float2* __restrict__ box_b,
                                                                   const uint32_t* __restrict__ xform, size_t n,
                                                                   const float4* __restrict__ planes, size_t ld,
                                                                   size_t chunk, Box6* __restrict__ partial)
{
  // wave-uniform in scalar registers, so the loop below branches on scalars
  const size_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * kBoxWavesPerBlock + threadIdx.x / kWave);
  const unsigned lane = threadIdx.x & (kWave - 1);
  const size_t begin = wave * chunk;
  size_t end = begin + chunk;
  if (end > n) end = n;
  Box6 acc = box_empty();
  uint32_t zero[3] = {kNoZero, kNoZero, kNoZero};
  // Round k takes object begin + lane + 64k.  The loads are clamped and
  // unconditional and run ahead of the folds, in two register sets that take
  // turns (no copies, which would wait for the loads): the box and matrix rows
  // of round k + 1 and the matrix index of round k + 2 are in flight while round
  // k is folded.
  const size_t count = end > begin ? end - begin : 0;
  const size_t rounds = (count + kWave - 1) / kWave;  // the same on every lane of the wave
  auto object_of = [&](size_t k) -> size_t {
    const size_t i = begin + lane + k * kWave;
    return i < end ? i : begin;  // (begin < end whenever rounds > 0)
  };
  auto matrix_of = [&](size_t i) -> size_t { return Indexed ? static_cast<size_t>(xform[i]) : i; };
  // Folds an object (index i, matrix m, inputs d) into the lane's box.  A lane past
  // the chunk's end has the chunk's first object, which changes nothing; an object
  // whose matrix index is outside the array adds nothing.
  auto fold_obb = [&](const Obb& o, size_t i) {
    // ManagerBitSet.cpp:282-294: v0 = lower * M, x/y/z = extent[k] * row k, same add tree as the cull.
    float4 v[8];
    v[0] = o.p;
    v[1] = add4(o.p, o.ex);
    v[2] = add4(o.p, o.ey);
    v[3] = add4(v[1], o.ey);
    v[4] = add4(o.p, o.ez);
    v[5] = add4(v[1], o.ez);
    v[6] = add4(v[2], o.ez);
    v[7] = add4(v[3], o.ez);
    const float x[8] = {v[0].x, v[1].x, v[2].x, v[3].x, v[4].x, v[5].x, v[6].x, v[7].x};
    const float y[8] = {v[0].y, v[1].y, v[2].y, v[3].y, v[4].y, v[5].y, v[6].y, v[7].y};
    const float z[8] = {v[0].z, v[1].z, v[2].z, v[3].z, v[4].z, v[5].z, v[6].z, v[7].z};
    const float lo[3] = {vmin8(x), vmin8(y), vmin8(z)}, hi[3] = {vmax8(x), vmax8(y), vmax8(z)};
    for (int c = 0; c < 3; ++c) {
      acc.lo[c] = lower(acc.lo[c], lo[c]);
      acc.hi[c] = higher(acc.hi[c], hi[c]);
    }
    const bool zeros = (lo[0] == 0.0f) | (hi[0] == 0.0f) | (lo[1] == 0.0f) | (hi[1] == 0.0f) | (lo[2] == 0.0f) |
                       (hi[2] == 0.0f);
    if (zeros) {
      const uint32_t at = static_cast<uint32_t>(i - begin) << 1;
      for (int c = 0; c < 3; ++c) {
        if (zero[c] != kNoZero) continue;
        const float(&p)[8] = c == 0 ? x : c == 1 ? y : z;
        for (int q = 8; q-- > 0;)
          if (p[q] == 0.0f) zero[c] = at | (__float_as_uint(p[q]) >> 31);
      }
    }
  };
  auto fold = [&](const BoxIn& d, size_t i, size_t m) {
    if (m < ld) fold_obb(make_obb(d.a, d.b, d.r0, d.r1, d.r2, d.r3), i);
  };
  size_t done = 0;  // rounds
  // K rounds of scattered matrices, row by row
  auto fold_rows = [&](auto rounds_at_once) {
    constexpr int K = decltype(rounds_at_once)::value;
    size_t m[K];
    float4 ba[K], row[K];
    float2 bb[K];
    Obb o[K];
    for (int k = 0; k < K; ++k) {
      const size_t i = object_of(done + k);
      m[k] = matrix_of(i);
      ba[k] = box_a[i];
      bb[k] = box_b[i];
    }
    auto load_row = [&](int r) {
      for (int k = 0; k < K; ++k) row[k] = planes[r * ld + (m[k] < ld ? m[k] : 0)];
    };
    // (the next row's address waits for this row's arithmetic: the compiler would
    // issue all the loads at once)
    auto wait_row = [&] {
      for (int k = 0; k < K; ++k) asm volatile("" : "+v"(m[k]) : "v"(o[k].p.x));
    };
    // make_obb row by row: the same products and sums in the same order
    load_row(0);
    for (int k = 0; k < K; ++k) {
      o[k].p = scale4(ba[k].x, row[k]);
      o[k].ex = scale4(ba[k].w, row[k]);
    }
    wait_row();
    load_row(1);
    for (int k = 0; k < K; ++k) {
      o[k].p = add4(o[k].p, scale4(ba[k].y, row[k]));
      o[k].ey = scale4(bb[k].x, row[k]);
    }
    wait_row();
    load_row(2);
    for (int k = 0; k < K; ++k) {
      o[k].p = add4(o[k].p, scale4(ba[k].z, row[k]));
      o[k].ez = scale4(bb[k].y, row[k]);
    }
    wait_row();
    load_row(3);
    for (int k = 0; k < K; ++k) {
      o[k].p = add4(o[k].p, row[k]);
      if (m[k] < ld) fold_obb(o[k], object_of(done + k));
    }
    done += K;
  };
  bool scattered = false;
  if (Indexed && rounds) {
    const uint32_t line = static_cast<uint32_t>(matrix_of(object_of(0)) / 8);
    scattered = __popcll(ballot(line != dpp_from<0x138, 0xf>(line))) >= kWave / 2;  // (wave_shr:1)
  }
  if (scattered) {
    while (done + 3 <= rounds) fold_rows(std::integral_constant<int, 3>{});
    if (done + 2 == rounds) fold_rows(std::integral_constant<int, 2>{});
    if (done + 1 == rounds) fold_rows(std::integral_constant<int, 1>{});
  } else if (rounds) {
    size_t ia = object_of(0), ma = matrix_of(ia);
    BoxIn a = load_box_in(box_a, box_b, planes, ld, ia, ma);
    size_t in = object_of(1), mn = matrix_of(in);  // the next round's object and matrix index
    BoxIn b;
    size_t ib = 0, mb = 0;
    for (size_t k = 0; k < rounds; k += 2) {
      // round k is in a; load round k + 1 into b and the index of round k + 2
      ib = in;
      mb = mn;
      in = object_of(k + 2);
      mn = matrix_of(in);
      b = load_box_in(box_a, box_b, planes, ld, ib, mb);
      __builtin_amdgcn_sched_barrier(0);  // keep these loads ahead of the fold
      fold(a, ia, ma);
      if (k + 1 >= rounds) break;
      // round k + 1 is in b; load round k + 2 into a and the index of round k + 3
      ia = in;
      ma = mn;
      in = object_of(k + 3);
      mn = matrix_of(in);
      a = load_box_in(box_a, box_b, planes, ld, ia, ma);
      __builtin_amdgcn_sched_barrier(0);
      fold(b, ib, mb);
    }
  }
  __shared__ Box6 waves[kBoxWavesPerBlock];
  Box6 box;
  for (int c = 0; c < 3; ++c) {
    box.lo[c] = wave_min(acc.lo[c]);
    box.hi[c] = wave_max(acc.hi[c]);
    if (ballot(zero[c] != kNoZero)) {
      const uint32_t first = wave_first(zero[c]);
      box.lo[c] = with_zero_sign(box.lo[c], first);
      box.hi[c] = with_zero_sign(box.hi[c], first);
    }
  }
  if (lane == 0) waves[threadIdx.x / kWave] = box;
  lds_barrier();
  if (threadIdx.x != 0) return;
  Box6 all = waves[0];
  for (unsigned w = 1; w < kBoxWavesPerBlock; ++w)
    for (int c = 0; c < 3; ++c) {
      all.lo[c] = lower(all.lo[c], waves[w].lo[c]);
      all.hi[c] = higher(all.hi[c], waves[w].hi[c]);
    }
  partial[blockIdx.x] = all;
}

constexpr unsigned kBoxFinalThreads = 256;

// One workgroup folds the partial boxes, which are in index order of their chunks:
// thread t takes partials t, t + 256, ... (coalesced loads, four per round issued
// together), each wave then folds its lanes and thread 0 the four waves.  A zero
// extremum has the sign that the first partial with that zero has.
__global__ __launch_bounds__(kBoxFinalThreads) void bbox_final_kernel(const Box6* __restrict__ partial,
                                                                      size_t n_partial, float* __restrict__ out6)
{
  constexpr unsigned kWaves = kBoxFinalThreads / kWave;
  __shared__ Box6 waves[kWaves];
  __shared__ uint32_t zeros[kWaves][6];
  const unsigned t = threadIdx.x, lane = t & (kWave - 1);
  Box6 run = box_empty();
  uint32_t zero[6] = {kNoZero, kNoZero, kNoZero, kNoZero, kNoZero, kNoZero};  // of lo, then of hi
  // four partials per thread and round, all loaded before any is folded (a
  // clamped index past the end loads the last partial again, which changes nothing)
  constexpr unsigned kU = 4;
  for (size_t k0 = t; k0 < n_partial; k0 += kU * kBoxFinalThreads) {
    Box6 b[kU];
#pragma unroll
    for (unsigned u = 0; u < kU; ++u) {
      const size_t k = k0 + u * kBoxFinalThreads;
      b[u] = partial[k < n_partial ? k : n_partial - 1];
    }
#pragma unroll
    for (unsigned u = 0; u < kU; ++u) {
      const size_t k = k0 + u * kBoxFinalThreads;
      const uint32_t at = static_cast<uint32_t>(k < n_partial ? k : n_partial - 1) << 1;
      for (int c = 0; c < 3; ++c) {
        run.lo[c] = lower(run.lo[c], b[u].lo[c]);
        run.hi[c] = higher(run.hi[c], b[u].hi[c]);
        if (b[u].lo[c] == 0.0f) zero[c] = min(zero[c], at | (__float_as_uint(b[u].lo[c]) >> 31));
        if (b[u].hi[c] == 0.0f) zero[3 + c] = min(zero[3 + c], at | (__float_as_uint(b[u].hi[c]) >> 31));
      }
    }
  }
  for (int c = 0; c < 3; ++c) {
    run.lo[c] = wave_min(run.lo[c]);
    run.hi[c] = wave_max(run.hi[c]);
  }
  for (int c = 0; c < 6; ++c) zero[c] = ballot(zero[c] != kNoZero) ? wave_first(zero[c]) : kNoZero;
  if (lane == 0) {
    waves[t / kWave] = run;
    for (int c = 0; c < 6; ++c) zeros[t / kWave][c] = zero[c];
  }
  lds_barrier();
  if (t != 0) return;
  Box6 acc = waves[0];
  for (unsigned w = 1; w < kWaves; ++w)
    for (int c = 0; c < 3; ++c) {
      acc.lo[c] = lower(acc.lo[c], waves[w].lo[c]);
      acc.hi[c] = higher(acc.hi[c], waves[w].hi[c]);
    }
  for (int c = 0; c < 3; ++c) {
    uint32_t zl = zeros[0][c], zh = zeros[0][3 + c];
    for (unsigned w = 1; w < kWaves; ++w) {
      zl = min(zl, zeros[w][c]);
      zh = min(zh, zeros[w][3 + c]);
    }
    acc.lo[c] = with_zero_sign(acc.lo[c], zl);
    acc.hi[c] = with_zero_sign(acc.hi[c], zh);
  }
  // return Box3f(lower.xyz, upper.xyz): Boxnt(p0, p1) runs init(), update(p0), update(p1)
  // (dp/math/Boxnt.h:213-219), which turns the empty box into (-FLT_MAX, +FLT_MAX).
  Box6 r = box_empty();
  box_take(r, make_float4(acc.lo[0], acc.lo[1], acc.lo[2], 0.f));
  box_take(r, make_float4(acc.hi[0], acc.hi[1], acc.hi[2], 0.f));
  for (int c = 0; c < 3; ++c) {
    out6[c] = r.lo[c];
    out6[3 + c] = r.hi[c];
  }
}

size_t bbox_waves(size_t n)
{
  // kBoxWavesPerCu waves per CU of partials at most, at least 64 objects each.
  size_t waves = (n + kWave - 1) / kWave;
  const size_t cap = static_cast<size_t>(device_cu_count()) * kBoxWavesPerCu;
  if (waves > cap) waves = cap;
  if (waves == 0) waves = 1;
  waves = (waves + kBoxWavesPerBlock - 1) / kBoxWavesPerBlock * kBoxWavesPerBlock;
  return waves;
}

// ---- result diff --------------------------------------------------------------
constexpr unsigned kDiffThreads = 256;  // one 64-bit word per thread

__device__ __forceinline__ unsigned long long diff_word(const unsigned long long* old_w,
                                                        const unsigned long long* new_w, size_t w, size_t n_words,
                                                        size_t n_bits)
{
  if (w >= n_words) return 0ull;
  unsigned long long x = old_w[w] ^ new_w[w];
  const size_t tail = n_bits & 63;
  if (w == n_words - 1 && tail) x &= (~0ull) >> (64 - tail);
  return x;
}

// diff_word without a branch: both words are loaded (from a clamped index)
// on every lane, so the loads of a kernel's later steps can be issued before
// anything waits for these.
__device__ __forceinline__ unsigned long long diff_word_clamped(const unsigned long long* old_w,
                                                                const unsigned long long* new_w, size_t w,
                                                                size_t n_words, size_t n_bits,
                                                                unsigned long long& new_bits)
{
  const size_t c = w < n_words ? w : n_words - 1;  // n_words >= 1 wherever a diff kernel runs
  new_bits = new_w[c];
  unsigned long long x = old_w[c] ^ new_bits;
  const size_t tail = n_bits & 63;
  const unsigned long long keep = (tail && c == n_words - 1) ? (~0ull) >> (64 - tail) : ~0ull;
  return w < n_words ? (x & keep) : 0ull;
}

// Inclusive scan over a wave (data-parallel primitives: within rows of 16 lanes,
// then the last lane of each half row pair, then of the lower half).
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v)
{
  v += __builtin_amdgcn_update_dpp(0u, v, 0x111, 0xf, 0xf, true);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0u, v, 0x112, 0xf, 0xf, true);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0u, v, 0x114, 0xf, 0xf, true);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0u, v, 0x118, 0xf, 0xf, true);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0u, v, 0x142, 0xa, 0xf, true);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0u, v, 0x143, 0xc, 0xf, true);  // row_bcast:31 into rows 2 and 3
  return v;
}

// Position of this thread's first of `count` entries: every thread's `before`
// together, and the counts of the threads before it; *total: all of both.  One
// barrier: each wave leaves its two sums in LDS (lds: 2 * Threads / 64 words) and
// adds up all waves' itself.
template <unsigned Threads>
__device__ __forceinline__ uint32_t block_position(uint32_t count, uint32_t before, uint32_t* lds, uint32_t* total)
{
  constexpr unsigned kWaves = Threads / kWave;
  static_assert(kWaves <= 16, "one row of lanes holds the waves' sums");
  const unsigned lane = threadIdx.x & (kWave - 1);
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t scan = wave_inclusive_scan(count);
  const uint32_t sum = wave_inclusive_scan(before);
  if (lane == kWave - 1) {
    lds[wave] = scan;
    lds[kWaves + wave] = sum;
  }
  lds_barrier();
  const uint32_t c = lane < kWaves ? lds[lane] : 0u;
  const uint32_t b = lane < kWaves ? lds[kWaves + lane] : 0u;
  const uint32_t to_here = wave_inclusive_scan(b + (lane < wave ? c : 0u));
  const uint32_t all = wave_inclusive_scan(b + c);
  *total = __builtin_amdgcn_readlane(static_cast<int>(all), kWave - 1);
  return __builtin_amdgcn_readlane(static_cast<int>(to_here), kWave - 1) + scan - count;
}

__global__ __launch_bounds__(kDiffThreads) void diff_count_kernel(const unsigned long long* __restrict__ old_w,
                                                                  const unsigned long long* __restrict__ new_w,
                                                                  size_t n_words, size_t n_bits,
                                                                  uint32_t* __restrict__ block_count)
{
  __shared__ uint32_t lds[2 * kDiffThreads / kWave];
  const size_t w = static_cast<size_t>(blockIdx.x) * kDiffThreads + threadIdx.x;
  const uint32_t c = __popcll(diff_word(old_w, new_w, w, n_words, n_bits));
  uint32_t total;
  block_position<kDiffThreads>(c, 0u, lds, &total);
  if (threadIdx.x == 0) block_count[blockIdx.x] = total;
}

// Single block: exclusive scan of block counts in place; writes the grand total.
__global__ __launch_bounds__(kDiffThreads) void diff_scan_kernel(uint32_t* __restrict__ block_count, size_t n_blocks,
                                                                 uint32_t* __restrict__ d_count)
{
  __shared__ uint32_t lds[2 * kDiffThreads / kWave];
  uint32_t carry = 0;
  for (size_t base = 0; base < n_blocks; base += kDiffThreads) {
    const size_t k = base + threadIdx.x;
    const uint32_t v = k < n_blocks ? block_count[k] : 0u;
    uint32_t total;
    const uint32_t ex = block_position<kDiffThreads>(v, 0u, lds, &total);
    if (k < n_blocks) block_count[k] = carry + ex;
    carry += total;
    lds_barrier();  // (the next round overwrites what this one has read)
  }
  if (threadIdx.x == 0) *d_count = carry;
}

__global__ __launch_bounds__(kDiffThreads) void diff_write_kernel(unsigned long long* __restrict__ old_w,
                                                                  const unsigned long long* __restrict__ new_w,
                                                                  size_t n_words, size_t n_bits,
                                                                  const uint32_t* __restrict__ block_offset,
                                                                  uint32_t* __restrict__ out, int update_old)
{
  __shared__ uint32_t lds[2 * kDiffThreads / kWave];
  const size_t w = static_cast<size_t>(blockIdx.x) * kDiffThreads + threadIdx.x;
  unsigned long long x = diff_word(old_w, new_w, w, n_words, n_bits);
  uint32_t total;
  uint32_t pos = block_offset[blockIdx.x] + block_position<kDiffThreads>(__popcll(x), 0u, lds, &total);
  while (x) {
    const unsigned b = __ffsll(static_cast<long long>(x)) - 1;
    out[pos++] = static_cast<uint32_t>(w * 64 + b);
    x &= x - 1;
  }
  if (update_old && w < n_words) old_w[w] = new_w[w];
}

// The write pass for at most kDiffDirectBlocks blocks: each block sums the
// counts of the blocks before it itself (no separate scan launch); the last
// block writes the grand total.
constexpr size_t kDiffDirectBlocks = 1024;

__global__ __launch_bounds__(kDiffThreads) void diff_write_direct_kernel(unsigned long long* __restrict__ old_w,
                                                                         const unsigned long long* __restrict__ new_w,
                                                                         size_t n_words, size_t n_bits,
                                                                         const uint32_t* __restrict__ block_count,
                                                                         uint32_t* __restrict__ out, int update_old,
                                                                         uint32_t* __restrict__ d_count)
{
  __shared__ uint32_t lds[2 * kDiffThreads / kWave];
  // this thread's words first: their loads are then in flight with those of the counts
  const size_t w = static_cast<size_t>(blockIdx.x) * kDiffThreads + threadIdx.x;
  unsigned long long new_bits;
  unsigned long long x = diff_word_clamped(old_w, new_w, w, n_words, n_bits, new_bits);
  // this thread's share of the counts of blocks [0, blockIdx.x): clamped loads, all issued at once
  constexpr unsigned kCountsPerThread = kDiffDirectBlocks / kDiffThreads;
  uint32_t v[kCountsPerThread];
#pragma unroll
  for (unsigned q = 0; q < kCountsPerThread; ++q) {
    const unsigned k = threadIdx.x + q * kDiffThreads;
    v[q] = block_count[k < blockIdx.x ? k : 0u];
  }
  uint32_t before = 0;
#pragma unroll
  for (unsigned q = 0; q < kCountsPerThread; ++q) before += threadIdx.x + q * kDiffThreads < blockIdx.x ? v[q] : 0u;
  uint32_t total;
  uint32_t pos = block_position<kDiffThreads>(__popcll(x), before, lds, &total);
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *d_count = total;
  while (x) {
    const unsigned b = __ffsll(static_cast<long long>(x)) - 1;
    out[pos++] = static_cast<uint32_t>(w * 64 + b);
    x &= x - 1;
  }
  if (update_old && w < n_words) old_w[w] = new_bits;
}

// The write pass after a cull that stored one change count per mask word
// (cull_kernel / cull_stream_kernel with Diff): each block of kDiffFusedThreads
// words adds up the counts of the words before its own, sixteen bytes per
// thread and load, and then writes as diff_write_direct_kernel.  For at most
// kDiffFusedWords mask words (2^22 objects): every thread then needs at most
// kDiffFusedWords / 16 / kDiffFusedThreads = 4 loads of counts, issued at once.
constexpr unsigned kDiffFusedThreads = 1024;
constexpr size_t kDiffFusedWords = 65536;

__device__ __forceinline__ uint32_t byte_sum(uint32_t v, uint32_t acc) { return __builtin_amdgcn_sad_u8(v, 0u, acc); }

__global__ __launch_bounds__(kDiffFusedThreads) void diff_write_fused_kernel(unsigned long long* __restrict__ old_w,
                                                                             const unsigned long long* __restrict__ new_w,
                                                                             size_t n_words, size_t n_bits,
                                                                             const uint4* __restrict__ word_count,
                                                                             uint32_t* __restrict__ out, int update_old,
                                                                             uint32_t* __restrict__ d_count)
{
  __shared__ uint32_t lds[2 * kDiffFusedThreads / kWave];
  // this thread's words first: their loads are then in flight with those of the counts
  const size_t w = static_cast<size_t>(blockIdx.x) * kDiffFusedThreads + threadIdx.x;
  unsigned long long new_bits;
  unsigned long long x = diff_word_clamped(old_w, new_w, w, n_words, n_bits, new_bits);
  // this thread's share of the counts of words [0, kDiffFusedThreads * blockIdx.x), clamped loads
  constexpr unsigned kChunksPerThread = kDiffFusedWords / 16 / kDiffFusedThreads;
  const size_t chunks = static_cast<size_t>(blockIdx.x) * (kDiffFusedThreads / 16);
  uint4 c[kChunksPerThread];
#pragma unroll
  for (unsigned q = 0; q < kChunksPerThread; ++q) {
    const size_t k = threadIdx.x + static_cast<size_t>(q) * kDiffFusedThreads;
    c[q] = word_count[k < chunks ? k : 0];
  }
  uint32_t before = 0;
#pragma unroll
  for (unsigned q = 0; q < kChunksPerThread; ++q) {
    const uint32_t part = byte_sum(c[q].w, byte_sum(c[q].z, byte_sum(c[q].y, byte_sum(c[q].x, 0u))));
    before += threadIdx.x + static_cast<size_t>(q) * kDiffFusedThreads < chunks ? part : 0u;
  }
  uint32_t total;
  uint32_t pos = block_position<kDiffFusedThreads>(__popcll(x), before, lds, &total);
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *d_count = total;
  while (x) {
    const unsigned b = __ffsll(static_cast<long long>(x)) - 1;
    if (pos < n_bits) out[pos] = static_cast<uint32_t>(w * 64 + b);  // (always, when the counts match the masks)
    ++pos;
    x &= x - 1;
  }
  if (update_old && w < n_words) old_w[w] = new_bits;
}

unsigned grid_for(size_t work, unsigned per_block)
{
  return static_cast<unsigned>((work + per_block - 1) / per_block);
}

std::atomic<uint32_t> g_cull_waves_per_cu{0};  // the plain form (measured fastest on gfx950)

dpc_cull_config current_cull_config()
{
  dpc_cull_config c;
  c.waves_per_cu = g_cull_waves_per_cu.load(std::memory_order_relaxed);
  return c;
}

// Argument checks of the single-frustum cull (what: the caller's name).
int check_cull_args(const float* d_box_a, const float* d_box_b, const uint32_t* d_xform, size_t n_objects,
                    const float* d_planes, size_t ld, const float* vp, const uint64_t* d_mask, const char* what)
{
  if (!d_box_a || !d_box_b || !d_planes || !d_mask || !vp)
    return set_error(DPC_ERR_INVALID_ARGUMENT, "%s: null pointer argument", what);
  if (!aligned(d_box_a, 16) || !aligned(d_planes, 16) || !aligned(d_box_b, 8) || !aligned(d_mask, 8))
    return set_error(DPC_ERR_INVALID_ARGUMENT, "%s: misaligned device pointer", what);
  if (!d_xform && ld < n_objects)
    return set_error(DPC_ERR_INVALID_ARGUMENT, "%s: %zu objects without indices need ld >= n (ld=%zu)", what,
                     n_objects, ld);
  if (ld == 0) return set_error(DPC_ERR_INVALID_ARGUMENT, "%s: no matrices (ld = 0)", what);
  return DPC_OK;
}

// The cull's launch in the tuned shape; with Diff, also the per-word change
// counts against d_old (count: one byte per mask word).
template <bool Diff>
int launch_cull(const float* d_box_a, const float* d_box_b, const uint32_t* d_xform, size_t n_objects,
                const float* d_planes, size_t ld, const float* vp, uint64_t* d_mask, const uint64_t* d_old,
                uint8_t* count, void* stream)
{
  Mat16 m;
  for (int k = 0; k < 16; ++k) m.m[k] = vp[k];
  const auto* a = reinterpret_cast<const float4*>(d_box_a);
  const auto* b = reinterpret_cast<const float2*>(d_box_b);
  const auto* p = reinterpret_cast<const float4*>(d_planes);
  auto* out = reinterpret_cast<unsigned long long*>(d_mask);
  const auto* old = reinterpret_cast<const unsigned long long*>(d_old);
  const dpc_cull_config cfg = current_cull_config();
  const size_t tiles = (n_objects + kWave - 1) / kWave;
  hipStream_t s = as_stream(stream);
  if (cfg.waves_per_cu == 0) {
    // Two tiles per wave where three objects or more share a matrix and the call is
    // long: a tile then reads 40 to 45 bytes an object and waits for latency more than
    // for memory (2,372,871 objects with 4 to a matrix: 19.9 -> 18.5 us; 4,900,000:
    // 44.1 -> 39.2, with 7 41.6 -> 35.8; 1,500,000 with 4: 13.0 -> 12.7).  Shorter
    // calls lose by the waves they no longer have (700,000 with 4: 8.2 -> 8.4 us;
    // 400,000: 5.8 -> 6.3), and with a matrix to each object or two memory is the
    // bound (4,900,000: 72.8 -> 75.2 with one, 50.4 -> 50.8 with two).
    if (d_xform && n_objects >= 1'400'000 && n_objects / 3 >= ld) {
      hipLaunchKernelGGL((cull_pair_kernel<Diff>), dim3(grid_for((n_objects + 1) / 2, kPairThreads)), dim3(kPairThreads), 0,
                         s, a, b, d_xform, n_objects, p, ld, m, out, old, count);
      return check_launch("cull_pair_kernel");
    }
    const auto launch = [&](auto kernel, unsigned threads) {
      hipLaunchKernelGGL(kernel, dim3(grid_for(n_objects, threads)), dim3(threads), 0, s, a, b, d_xform, n_objects, p, ld, m,
                         out, old, count);
    };
    // (with an index array workgroups of 512, whose loads wait for the indices first: two
    // frames over 500,000 objects, 4 to a matrix, 19.5 us against 20.0 with one wave each;
    // not measured below 500,000)
    if (d_xform)
      launch(cull_kernel<true, Diff, kIndexedThreads>, kIndexedThreads);
    else if (n_objects <= 100'000 ||  // (less than half a row: not worth asking for the device)
             flat_cull_threads(n_objects, static_cast<uint32_t>(std::max(device_cu_count(), 1)), Diff) == kSmallThreads)
      launch(cull_kernel<false, Diff, kSmallThreads>, kSmallThreads);
    else
      launch(cull_kernel<false, Diff, kPlainThreads>, kPlainThreads);
  } else {
    const size_t waves_per_block = kCullThreads / kWave;
    size_t blocks = static_cast<size_t>(device_cu_count()) * cfg.waves_per_cu / waves_per_block;
    const size_t needed = (tiles + waves_per_block - 1) / waves_per_block;
    if (blocks > needed) blocks = needed;
    if (blocks == 0) blocks = 1;
    if (d_xform)
      hipLaunchKernelGGL((cull_stream_kernel<true, Diff>), dim3(static_cast<unsigned>(blocks)), dim3(kCullThreads), 0,
                         s, a, b, d_xform, n_objects, p, ld, m, out, old, count);
    else
      hipLaunchKernelGGL((cull_stream_kernel<false, Diff>), dim3(static_cast<unsigned>(blocks)), dim3(kCullThreads),
                         0, s, a, b, d_xform, n_objects, p, ld, m, out, old, count);
  }
  return check_launch("cull_kernel");
}

}  // namespace
}  // namespace dpc

using namespace dpc;

extern "C" {

int dpc_cull(const float* d_box_a, const float* d_box_b, const uint32_t* d_xform, size_t n_objects,
             const float* d_planes, size_t ld, const float vp[16], uint64_t* d_mask, void* stream)
{
  if (n_objects == 0) return DPC_OK;
  if (int rc = check_cull_args(d_box_a, d_box_b, d_xform, n_objects, d_planes, ld, vp, d_mask, "dpc_cull")) return rc;
  return launch_cull<false>(d_box_a, d_box_b, d_xform, n_objects, d_planes, ld, vp, d_mask, nullptr, nullptr, stream);
}

int dpc_cull_get_config(dpc_cull_config* cfg)
{
  if (!cfg) return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_cull_get_config: null output");
  *cfg = current_cull_config();
  return DPC_OK;
}

int dpc_cull_set_config(const dpc_cull_config* cfg)
{
  if (!cfg || cfg->waves_per_cu > 64)
    return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_cull_set_config: waves_per_cu must be 0..64");
  g_cull_waves_per_cu.store(cfg->waves_per_cu, std::memory_order_relaxed);
  return DPC_OK;
}

int dpc_matrices_from_aos(const void* d_aos, size_t stride_bytes, size_t count, float* d_planes, size_t ld,
                          void* stream)
{
  if (count == 0) return DPC_OK;
  if (!d_aos || !d_planes) return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_matrices_from_aos: null pointer");
  if (stride_bytes < 64 || stride_bytes % 4 || !aligned(d_aos, 4) || !aligned(d_planes, 16) || ld < count)
    return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_matrices_from_aos: bad stride/alignment/ld");
  hipLaunchKernelGGL(from_aos_kernel, dim3(grid_for(count * 4, 256)), dim3(256), 0, as_stream(stream),
                     static_cast<const char*>(d_aos), stride_bytes, count, reinterpret_cast<float4*>(d_planes), ld);
  return check_launch("from_aos_kernel");
}

int dpc_matrices_to_aos(const float* d_planes, size_t ld, const uint32_t* d_slot, size_t count, void* d_aos,
                        size_t stride_bytes, void* stream)
{
  if (count == 0) return DPC_OK;
  if (!d_aos || !d_planes) return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_matrices_to_aos: null pointer");
  if (stride_bytes < 64 || stride_bytes % 4 || !aligned(d_aos, 4) || !aligned(d_planes, 16))
    return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_matrices_to_aos: bad stride/alignment");
  if (!d_slot && ld < count) return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_matrices_to_aos: ld < count");
  hipLaunchKernelGGL(to_aos_kernel, dim3(grid_for(count * 4, 256)), dim3(256), 0, as_stream(stream),
                     reinterpret_cast<const float4*>(d_planes), ld, d_slot, count, static_cast<char*>(d_aos),
                     stride_bytes);
  return check_launch("to_aos_kernel");
}

int dpc_matrices_scatter(float* d_planes, size_t ld, const uint32_t* d_idx, const float* d_src, size_t count,
                         void* stream)
{
  if (count == 0) return DPC_OK;
  if (!d_planes || !d_idx || !d_src) return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_matrices_scatter: null pointer");
  if (!aligned(d_planes, 16) || !aligned(d_src, 16))
    return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_matrices_scatter: misaligned pointer");
  hipLaunchKernelGGL(scatter_kernel, dim3(grid_for(count * 4, 256)), dim3(256), 0, as_stream(stream),
                     reinterpret_cast<float4*>(d_planes), ld, d_idx, reinterpret_cast<const float4*>(d_src), count);
  return check_launch("scatter_kernel");
}

}  // extern "C"

namespace dpc {

int launch_scatter_host(float* d_planes, size_t ld, const uint32_t* idx, const float* src, size_t count,
                        void* stream)
{
  if (count == 0) return DPC_OK;
  if (count > kMaxHostScatter || ld > kMaxHostScatterLd)
    return set_error(DPC_ERR_INVALID_ARGUMENT, "launch_scatter_host: %zu matrices into %zu slots exceed %u into %u",
                     count, ld, kMaxHostScatter, kMaxHostScatterLd);
  // 64 workgroups (256 CUs hold 4x more): ~16k rows of 16 B in flight, well above PCIe's bandwidth-latency product
  const unsigned grid = std::min<unsigned>(grid_for(count * 4, 256), 64u);
  hipLaunchKernelGGL(scatter_host_kernel, dim3(grid), dim3(256), 0, as_stream(stream),
                     reinterpret_cast<float4*>(d_planes), static_cast<uint32_t>(ld), idx, src, static_cast<uint32_t>(count));
  return check_launch("scatter_host_kernel");
}

int launch_stage(const char* arena, uint64_t bytes, char* d_arena, uint64_t desc_bytes, const StageJob* jobs, uint32_t n,
                 void* stream)
{
  if (!arena || (n && !jobs) || n > kStageJobs || bytes >= (1ull << 31) || desc_bytes > bytes || desc_bytes % 16 ||
      !aligned(arena, 16) || !aligned(d_arena, 16) || (desc_bytes && !d_arena))
    return set_error(DPC_ERR_INVALID_ARGUMENT, "launch_stage: bad argument");
  for (uint32_t k = 0; k < n; ++k) {
    const StageJob& j = jobs[k];
    if (!j.planes || !aligned(j.planes, 16) || j.idx % 4 || j.packed % 16 || j.tails % 16 ||
        j.idx + 4ull * j.count > bytes || j.packed + 48ull * j.count > bytes ||
        (j.tails && j.tails + 16ull * j.count > bytes))
      return set_error(DPC_ERR_INVALID_ARGUMENT, "launch_stage: bad job");
  }
  StageJobs args;
  args.desc_chunks = static_cast<uint32_t>(desc_bytes / 16);
  args.desc_units = (args.desc_chunks + kStageChunk - 1) / kStageChunk;
  args.n = 0;
  args.units = args.desc_units;
  for (uint32_t k = 0; k < n; ++k) {
    if (jobs[k].count == 0) continue;
    args.job[args.n] = jobs[k];
    args.first_unit[args.n++] = args.units;
    args.units += (jobs[k].count + 63) / 64;
  }
  if (args.units == 0) return DPC_OK;
  const uint32_t most = d_arena ? kStageHostBlocks : 8u * static_cast<uint32_t>(device_cu_count());
  const dim3 grid(std::min((args.units + 3) / 4, most));
  if (d_arena)
    hipLaunchKernelGGL(stage_kernel<true>, grid, dim3(256), 0, as_stream(stream), arena, static_cast<uint32_t>(bytes),
                       reinterpret_cast<u32x4_t*>(d_arena), args);
  else
    hipLaunchKernelGGL(stage_kernel<false>, grid, dim3(256), 0, as_stream(stream), arena, static_cast<uint32_t>(bytes),
                       nullptr, args);
  return check_launch("stage_kernel");
}

}  // namespace dpc

extern "C" {

int dpc_gather_u32(const uint32_t* d_table, size_t table_len, const uint32_t* d_idx, size_t n, uint32_t* d_out,
                   void* stream)
{
  if (n == 0) return DPC_OK;
  if (!d_idx || !d_out || (table_len && !d_table))
    return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_gather_u32: null pointer");
  hipLaunchKernelGGL(gather_u32_kernel, dim3(grid_for(n, 256)), dim3(256), 0, as_stream(stream), d_table, table_len,
                     d_idx, n, d_out);
  return check_launch("gather_u32_kernel");
}

int dpc_boxes_from_lower_upper(const float* d_lower_upper, size_t n, float* d_box_a, float* d_box_b, void* stream)
{
  if (n == 0) return DPC_OK;
  if (!d_lower_upper || !d_box_a || !d_box_b || !aligned(d_box_a, 16) || !aligned(d_box_b, 8))
    return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_boxes_from_lower_upper: bad pointer");
  hipLaunchKernelGGL(boxes_kernel, dim3(grid_for(n, 256)), dim3(256), 0, as_stream(stream), d_lower_upper, n,
                     reinterpret_cast<float4*>(d_box_a), reinterpret_cast<float2*>(d_box_b));
  return check_launch("boxes_kernel");
}

size_t dpc_bbox_workspace(size_t n_objects) { return bbox_waves(n_objects) / kBoxWavesPerBlock * sizeof(Box6); }

int dpc_bbox(const float* d_box_a, const float* d_box_b, const uint32_t* d_xform, size_t n_objects,
             const float* d_planes, size_t ld, float* d_out6, void* d_workspace, void* stream)
{
  if (!d_out6 || !d_workspace || !aligned(d_workspace, 8))
    return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_bbox: null output/workspace (or workspace not 8-byte aligned)");
  if (n_objects && (!d_box_a || !d_box_b || !d_planes || !aligned(d_box_a, 16) || !aligned(d_box_b, 8) ||
                    !aligned(d_planes, 16)))
    return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_bbox: bad object/matrix pointer");
  if (n_objects && !d_xform && ld < n_objects)
    return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_bbox: objects without indices need ld >= n");
  const size_t waves = bbox_waves(n_objects);
  size_t chunk = (n_objects + waves - 1) / waves;
  chunk = (chunk + kWave - 1) / kWave * kWave;
  if (chunk == 0) chunk = kWave;
  auto* partial = static_cast<Box6*>(d_workspace);
  const dim3 grid(static_cast<unsigned>(waves / kBoxWavesPerBlock));
  if (d_xform)
    hipLaunchKernelGGL(bbox_partial_kernel<true>, grid, dim3(kBoxThreads), 0, as_stream(stream),
                       reinterpret_cast<const float4*>(d_box_a), reinterpret_cast<const float2*>(d_box_b), d_xform,
                       n_objects, reinterpret_cast<const float4*>(d_planes), ld, chunk, partial);
  else
    hipLaunchKernelGGL(bbox_partial_kernel<false>, grid, dim3(kBoxThreads), 0, as_stream(stream),
                       reinterpret_cast<const float4*>(d_box_a), reinterpret_cast<const float2*>(d_box_b), d_xform,
                       n_objects, reinterpret_cast<const float4*>(d_planes), ld, chunk, partial);
  int rc = check_launch("bbox_partial_kernel");
  if (rc) return rc;
  hipLaunchKernelGGL(bbox_final_kernel, dim3(1), dim3(kBoxFinalThreads), 0, as_stream(stream), partial,
                     waves / kBoxWavesPerBlock, d_out6);
  return check_launch("bbox_final_kernel");
}

size_t dpc_result_diff_workspace(size_t n_bits)
{
  const size_t n_words = (n_bits + 63) / 64;
  const size_t blocks = (n_words + kDiffThreads - 1) / kDiffThreads;
  return (blocks ? blocks : 1) * sizeof(uint32_t);
}

}  // extern "C"

namespace dpc {
namespace {

// Argument checks shared by both result-diff entry points (what: the caller's name).
int check_result_diff_args(const uint64_t* d_old, const uint64_t* d_new, size_t n_bits,
                           const uint32_t* d_changed_idx, const uint32_t* d_count, const char* what)
{
  if (!d_count) return set_error(DPC_ERR_INVALID_ARGUMENT, "%s: null count", what);
  if (n_bits == 0) return DPC_OK;
  if (!d_old || !d_new || !d_changed_idx || !aligned(d_old, 8) || !aligned(d_new, 8))
    return set_error(DPC_ERR_INVALID_ARGUMENT, "%s: bad mask pointer", what);
  if (n_bits > 0xFFFFFFFFull) return set_error(DPC_ERR_INVALID_ARGUMENT, "%s: more than 2^32 bits", what);
  return DPC_OK;
}

// The result diff's launches, with counts = one u32 per block of kDiffThreads
// mask words (every one written by diff_count_kernel before it is read).
int launch_result_diff(uint64_t* d_old, const uint64_t* d_new, size_t n_bits, uint32_t* d_changed_idx,
                       uint32_t* d_count, int update_old, uint32_t* counts, void* stream)
{
  if (n_bits == 0) return dpc_fill_u32(d_count, 0u, 1, stream);
  const size_t n_words = (n_bits + 63) / 64;
  const unsigned blocks = grid_for(n_words, kDiffThreads);
  auto* o = reinterpret_cast<unsigned long long*>(d_old);
  auto* nw = reinterpret_cast<const unsigned long long*>(d_new);
  hipLaunchKernelGGL(diff_count_kernel, dim3(blocks), dim3(kDiffThreads), 0, as_stream(stream), o, nw, n_words, n_bits,
                     counts);
  int rc = check_launch("diff_count_kernel");
  if (rc) return rc;
  if (blocks <= kDiffDirectBlocks) {
    hipLaunchKernelGGL(diff_write_direct_kernel, dim3(blocks), dim3(kDiffThreads), 0, as_stream(stream), o, nw,
                       n_words, n_bits, counts, d_changed_idx, update_old, d_count);
    return check_launch("diff_write_direct_kernel");
  }
  hipLaunchKernelGGL(diff_scan_kernel, dim3(1), dim3(kDiffThreads), 0, as_stream(stream), counts,
                     static_cast<size_t>(blocks), d_count);
  rc = check_launch("diff_scan_kernel");
  if (rc) return rc;
  hipLaunchKernelGGL(diff_write_kernel, dim3(blocks), dim3(kDiffThreads), 0, as_stream(stream), o, nw, n_words, n_bits,
                     counts, d_changed_idx, update_old);
  return check_launch("diff_write_kernel");
}

}  // namespace
}  // namespace dpc

// ---- allocation-free result diff ----------------------------------------------
// The per-block counts of dpc_result_diff_noalloc live in this array, one copy
// per device, which the library holds until the process ends (256 KiB: 65,536
// blocks of 256 mask words, i.e. up to 2^30 bits).  Host code never passes the
// array's name to a kernel (on the host it is only a stand-in): it looks up
// each device's address once with hipGetSymbolAddress and passes that.
static_assert(DPC_RESULT_DIFF_NOALLOC_MAX_BITS % (64ull * 256ull) == 0, "whole blocks of 256 mask words");
static __device__ __align__(256) uint32_t scratch[DPC_RESULT_DIFF_NOALLOC_MAX_BITS / (64ull * 256ull)];

namespace dpc {
namespace {

constexpr int kScratchDevices = 64;
std::mutex g_scratch_mutex;
uint32_t* g_scratch_ptr[kScratchDevices] = {};  // per device, looked up on its first call

// The current device's copy of the scratch array (no allocation: a fixed table
// of per-device addresses, filled on each device's first call).
int scratch_of_current_device(uint32_t** ptr, const char* what)
{
  int dev = 0;
  DPC_HIP_TRY(hipGetDevice(&dev), "hipGetDevice");
  if (dev < 0 || dev >= kScratchDevices)
    return set_error(DPC_ERR_INVALID_ARGUMENT, "%s: device %d is beyond the %d devices served", what, dev,
                     kScratchDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    if (!p) return set_error(DPC_ERR_HIP, "%s: hipGetSymbolAddress returned no address", what);
    g_scratch_ptr[dev] = static_cast<uint32_t*>(p);
  }
  *ptr = g_scratch_ptr[dev];
  return DPC_OK;
}

}  // namespace
}  // namespace dpc

extern "C" {

int dpc_result_diff(uint64_t* d_old, const uint64_t* d_new, size_t n_bits, uint32_t* d_changed_idx, uint32_t* d_count,
                    int update_old, void* d_workspace, void* stream)
{
  if (!d_workspace) return set_error(DPC_ERR_INVALID_ARGUMENT, "dpc_result_diff: null workspace");
  const int rc = check_result_diff_args(d_old, d_new, n_bits, d_changed_idx, d_count, "dpc_result_diff");
  if (rc) return rc;
  return launch_result_diff(d_old, d_new, n_bits, d_changed_idx, d_count, update_old,
                            static_cast<uint32_t*>(d_workspace), stream);
}

int dpc_result_diff_noalloc(uint64_t* d_old, const uint64_t* d_new, size_t n_bits, uint32_t* d_changed_idx,
                            uint32_t* d_count, int update_old, void* stream)
{
  int rc = check_result_diff_args(d_old, d_new, n_bits, d_changed_idx, d_count, "dpc_result_diff_noalloc");
  if (rc) return rc;
  if (n_bits > DPC_RESULT_DIFF_NOALLOC_MAX_BITS)
    return set_error(DPC_ERR_INVALID_ARGUMENT,
                     "dpc_result_diff_noalloc: %zu bits exceed the %llu its fixed scratch serves (use dpc_result_diff)",
                     n_bits, static_cast<unsigned long long>(DPC_RESULT_DIFF_NOALLOC_MAX_BITS));
  uint32_t* counts = nullptr;
  rc = scratch_of_current_device(&counts, "dpc_result_diff_noalloc");
  if (rc) return rc;
  return launch_result_diff(d_old, d_new, n_bits, d_changed_idx, d_count, update_old, counts, stream);
}

size_t dpc_cull_diff_workspace(size_t n_objects)
{
  const size_t words = (n_objects + 63) / 64;
  const size_t counts = (words + 15) / 16 * 16;  // one byte per mask word, read sixteen at a time
  const size_t diff = dpc_result_diff_workspace(n_objects);
  return counts > diff ? counts : diff;
}

int dpc_cull_diff(const float* d_box_a, const float* d_box_b, const uint32_t* d_xform, size_t n_objects,
                  const float* d_planes, size_t ld, const float vp[16], uint64_t* d_mask, uint64_t* d_old,
                  uint32_t* d_changed_idx, uint32_t* d_count, int update_old, void* d_workspace, void* stream)
{
  const char* what = "dpc_cull_diff";
  int rc = check_result_diff_args(d_old, d_mask, n_objects, d_changed_idx, d_count, what);
  if (rc) return rc;
  if (n_objects == 0) return dpc_fill_u32(d_count, 0u, 1, stream);
  if ((rc = check_cull_args(d_box_a, d_box_b, d_xform, n_objects, d_planes, ld, vp, d_mask, what))) return rc;
  if (!d_workspace || !aligned(d_workspace, 16))
    return set_error(DPC_ERR_INVALID_ARGUMENT, "%s: null or misaligned workspace", what);
  if (d_old == d_mask) return set_error(DPC_ERR_INVALID_ARGUMENT, "%s: the old and new masks are one buffer", what);
  const size_t n_words = (n_objects + 63) / 64;
  if (n_words > kDiffFusedWords) {  // the prefix sums would grow quadratically: count in a launch of its own
    rc = launch_cull<false>(d_box_a, d_box_b, d_xform, n_objects, d_planes, ld, vp, d_mask, nullptr, nullptr, stream);
    if (rc) return rc;
    return launch_result_diff(d_old, d_mask, n_objects, d_changed_idx, d_count, update_old,
                              static_cast<uint32_t*>(d_workspace), stream);
  }
  auto* counts = static_cast<uint8_t*>(d_workspace);
  rc = launch_cull<true>(d_box_a, d_box_b, d_xform, n_objects, d_planes, ld, vp, d_mask, d_old, counts, stream);
  if (rc) return rc;
  const size_t blocks = (n_words + kDiffFusedThreads - 1) / kDiffFusedThreads;
  hipLaunchKernelGGL(diff_write_fused_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kDiffFusedThreads), 0,
                     as_stream(stream), reinterpret_cast<unsigned long long*>(d_old),
                     reinterpret_cast<const unsigned long long*>(d_mask), n_words, n_objects,
                     reinterpret_cast<const uint4*>(counts), d_changed_idx, update_old, d_count);
  return check_launch("diff_write_fused_kernel");
}

}  // extern "C"

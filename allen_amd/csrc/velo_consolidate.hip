// Track consolidation, the simplified VELO Kalman fit, the device prefix sum and fills.
//
//   k_copy_track_hit_number   VeloCopyTrackHitNumber.cu:49-78
//   k_consolidate_tracks      VeloConsolidateTracks.cu:120-192 (one thread per track hit)
//   k_kalman_filter           VeloKalmanFilter.cu:335-418, VeloKalmanFilter.cuh:25-158 (one thread per track)
//   k_create_velo_views       VeloConsolidateTracks.cu:11-46 (Allen's view objects, byte for byte)
//   k_clusters_views          MaskedVeloClustering.cu:519-522, DecodeRetinaClusters.cu:331-346
//   k_consolidate_and_fit     the three above in one launch (whole sequence; one workgroup per event)
//   k_scan_events, k_track_offsets  the whole sequence's offsets from per-event totals
//   k_scan_*                  replaces host_prefix_sum_t (HostPrefixSum.cpp:76-107) by a device scan
#include "velo_amd.h"
#include "velo_common.cuh"
#include "velo_kernels.h"

#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>

namespace velo {

// ---------------------------------------------------------------------------------------
// Prefix sum: out[0] = 0, out[i+1] = in[0] + ... + in[i] (u32 wrap), in three passes:
// per-tile sums, a scan of the tile sums, then per-tile scans seeded with their offset.
// Sizes up to one_pass_items run as a single workgroup (a launch instead of three).
constexpr unsigned scan_block = 1024;
constexpr unsigned scan_items = 4;
constexpr unsigned scan_tile = scan_block * scan_items;
constexpr unsigned one_pass_max = 32 * scan_block;

__device__ __forceinline__ uint32_t block_scan_1024(uint32_t v, uint32_t* scratch, uint32_t* total)
{
  return block_exclusive_scan(v, scratch, total);
}

__global__ void __launch_bounds__(scan_block)
  k_scan_tile_sums(const uint32_t* in, unsigned n, uint32_t* tile_sums)
{
  __shared__ uint32_t scratch[scan_block / wave_size + 1];
  const size_t base = (size_t) blockIdx.x * scan_tile;
  uint32_t s = 0;
#pragma unroll
  for (unsigned k = 0; k < scan_items; ++k) {
    const size_t i = base + (size_t) k * scan_block + threadIdx.x;
    if (i < n) s += in[i];
  }
  uint32_t total;
  block_scan_1024(s, scratch, &total);
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

// Exclusive scan of `n` values in place by one workgroup (n_tiles is small).
__global__ void __launch_bounds__(scan_block) k_scan_small_inplace(uint32_t* v, unsigned n)
{
  __shared__ uint32_t scratch[scan_block / wave_size + 1];
  uint32_t carry = 0;
  for (unsigned c = 0; c < n; c += scan_block) {
    const unsigned i = c + threadIdx.x;
    const uint32_t x = i < n ? v[i] : 0u;
    uint32_t total;
    const uint32_t e = block_scan_1024(x, scratch, &total);
    if (i < n) v[i] = carry + e;
    carry += total;
  }
}

// Per-tile scan: thread t owns items [t*scan_items, (t+1)*scan_items) of its tile (contiguous, so the
// prefix within a thread is a short serial sum).
__global__ void __launch_bounds__(scan_block)
  k_scan_tiles(const uint32_t* in, unsigned n, uint32_t* out, const uint32_t* tile_offsets)
{
  __shared__ uint32_t scratch[scan_block / wave_size + 1];
  const size_t base = (size_t) blockIdx.x * scan_block * scan_items + (size_t) threadIdx.x * scan_items;
  uint32_t v[scan_items];
  uint32_t s = 0;
#pragma unroll
  for (unsigned k = 0; k < scan_items; ++k) {
    const size_t i = base + k;
    v[k] = i < n ? in[i] : 0u;
    s += v[k];
  }
  uint32_t total;
  uint32_t run = block_scan_1024(s, scratch, &total) + (tile_offsets ? tile_offsets[blockIdx.x] : 0u);
  if (blockIdx.x == 0 && threadIdx.x == 0) out[0] = 0;
#pragma unroll
  for (unsigned k = 0; k < scan_items; ++k) {
    const size_t i = base + k;
    run += v[k];
    if (i < n) out[i + 1] = run;
  }
}

// Prefix over n arrays of equal length (per event, say) by one workgroup of 1024: wave w takes a
// contiguous range, sums it, and scans it again from the sum of the waves before. emit(i, k,
// inclusive prefix) is called for every item and array. Every read is a whole wave's line.
template<unsigned n, typename F>
__device__ __forceinline__ void
scan_by_waves(const uint32_t* const (&in)[n], unsigned n_events, uint32_t (&scratch)[n][scan_block / wave_size], F&& emit)
{
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / wave_size), l = lane_id();
  const unsigned range = (n_events + scan_block - 1) / scan_block * wave_size;
  const unsigned begin = min(wave * range, n_events), end = min(begin + range, n_events);
  uint32_t sum[n];
#pragma unroll
  for (unsigned k = 0; k < n; ++k) sum[k] = 0;
  for (unsigned i = begin + l; i < end; i += wave_size)
#pragma unroll
    for (unsigned k = 0; k < n; ++k) sum[k] += in[k][i];
#pragma unroll
  for (unsigned k = 0; k < n; ++k) {
    const uint32_t inc = wave_inclusive_scan(sum[k]);
    if (l == wave_size - 1) scratch[k][wave] = inc;
  }
  __syncthreads();
  uint32_t carry[n];
#pragma unroll
  for (unsigned k = 0; k < n; ++k) {
    const uint32_t t = l < scan_block / wave_size ? scratch[k][l] : 0u;
    carry[k] = __builtin_amdgcn_readlane(wave_inclusive_scan(t) - t, wave);
  }
  for (unsigned i0 = begin; i0 < end; i0 += wave_size) {
    const unsigned i = i0 + l;
#pragma unroll
    for (unsigned k = 0; k < n; ++k) {
      const uint32_t inc = wave_inclusive_scan(i < end ? in[k][i] : 0u);
      if (i < end) emit(i, k, carry[k] + inc);
      carry[k] += __builtin_amdgcn_readlane(inc, wave_size - 1);
    }
  }
}

// A prefix sum of up to one_pass_max items by one workgroup: wave w takes a contiguous range, a line
// per read, all of them in flight at once and before any write (in and out may overlap). 13 000
// items: 5.9 us; with 32 consecutive items per thread, whose reads went over the L1's lines
// eight times, 15.5 us, and 27 us for 26 000.
constexpr unsigned one_pass_items = one_pass_max / scan_block;
__global__ void __launch_bounds__(scan_block) k_scan_one(const uint32_t* in, unsigned n, uint32_t* out)
{
  __shared__ uint32_t scratch[scan_block / wave_size];
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / wave_size), l = lane_id();
  const unsigned lines = (n + scan_block - 1) / scan_block; // per wave
  const unsigned begin = wave * lines * wave_size;
  uint32_t v[one_pass_items], sum = 0;
#pragma unroll
  for (unsigned k = 0; k < one_pass_items; ++k) {
    const unsigned i = begin + k * wave_size + l;
    v[k] = k < lines && i < n ? in[i] : 0u;
  }
#pragma unroll
  for (unsigned k = 0; k < one_pass_items; ++k) sum += v[k];
  const uint32_t inc = wave_inclusive_scan(sum);
  if (l == wave_size - 1) scratch[wave] = inc;
  uint32_t total;
  uint32_t carry = block_wave_prefix(scratch, &total);
  if (threadIdx.x == 0) out[0] = 0;
#pragma unroll
  for (unsigned k = 0; k < one_pass_items; ++k) {
    const unsigned i = begin + k * wave_size + l;
    if (k >= lines) continue;
    const uint32_t run = wave_inclusive_scan(v[k]);
    if (i < n) out[i + 1] = carry + run;
    carry += __builtin_amdgcn_readlane(run, wave_size - 1);
  }
}

size_t prefix_sum_scratch_words(unsigned n) { return (n + scan_tile - 1) / scan_tile; }

hipError_t launch_prefix_sum(const uint32_t* in, unsigned n, uint32_t* out, uint32_t* scratch, hipStream_t s)
{
  const unsigned tiles = (n + scan_tile - 1) / scan_tile;
  if (tiles <= 1) {
    hipLaunchKernelGGL(k_scan_tiles, dim3(1), dim3(scan_block), 0, s, in, n, out, nullptr);
    return hipGetLastError();
  }
  if (n <= one_pass_max) {
    hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(scan_block), 0, s, in, n, out);
    return hipGetLastError();
  }
  if (!scratch) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_scan_tile_sums, dim3(tiles), dim3(scan_block), 0, s, in, n, scratch);
  hipLaunchKernelGGL(k_scan_small_inplace, dim3(1), dim3(scan_block), 0, s, scratch, tiles);
  hipLaunchKernelGGL(k_scan_tiles, dim3(tiles), dim3(scan_block), 0, s, in, n, out, scratch);
  return hipGetLastError();
}

// Tile sums of the allocation-free prefix sum: one u32 per scan tile, room for
// prefix_sum_static_max_items items (256 KiB per device, held until the process ends). Every
// launch writes all the tile sums it reads, so nothing needs clearing between calls; calls that
// overlap on one device share the array and race.
constexpr unsigned prefix_sum_static_max_tiles = prefix_sum_static_max_items / scan_tile;
static_assert(prefix_sum_static_max_items % scan_tile == 0, "whole tiles");
static __device__ __align__(256) uint32_t scratch[prefix_sum_static_max_tiles];

namespace {
std::mutex g_scratch_mutex;
std::map<int, uint32_t*> g_scratch_ptr; // device -> address of its copy of `scratch`
} // namespace

// The device address of the current device's `scratch`, looked up once per device (the array's
// name is a host-side stand-in and is never passed to a kernel).
static hipError_t static_scratch(uint32_t** ptr)
{
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  auto it = g_scratch_ptr.find(dev);
  if (it != g_scratch_ptr.end()) {
    *ptr = it->second;
    return hipSuccess;
  }
  void* p = nullptr;
  e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return e;
  if (!p) return hipErrorInvalidSymbol;
  g_scratch_ptr.emplace(dev, static_cast<uint32_t*>(p));
  *ptr = static_cast<uint32_t*>(p);
  return hipSuccess;
}

hipError_t prefix_sum_static_init()
{
  uint32_t* p = nullptr;
  return static_scratch(&p);
}

hipError_t launch_prefix_sum_static(const uint32_t* in, unsigned n, uint32_t* out, hipStream_t s)
{
  if (n > prefix_sum_static_max_items) return hipErrorInvalidValue;
  uint32_t* p = nullptr;
  const hipError_t e = static_scratch(&p);
  if (e != hipSuccess) return e;
  return launch_prefix_sum(in, n, out, p, s);
}

__global__ void k_fill_u32(uint32_t* p, size_t n, uint32_t value)
{
  for (size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t) gridDim.x * blockDim.x)
    p[i] = value;
}
__global__ void k_fill_u8(uint8_t* p, size_t n, uint8_t value)
{
  for (size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t) gridDim.x * blockDim.x)
    p[i] = value;
}

hipError_t launch_fill_u32(uint32_t* p, size_t n, uint32_t value, hipStream_t s)
{
  if (!n) return hipSuccess;
  const unsigned grid = (unsigned) std::min<size_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(k_fill_u32, dim3(grid), dim3(256), 0, s, p, n, value);
  return hipGetLastError();
}
hipError_t launch_fill_u8(uint8_t* p, size_t n, uint8_t value, hipStream_t s)
{
  if (!n) return hipSuccess;
  const unsigned grid = (unsigned) std::min<size_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(k_fill_u8, dim3(grid), dim3(256), 0, s, p, n, value);
  return hipGetLastError();
}

namespace {
std::mutex g_query_mutex;
std::map<std::tuple<int, const void*, unsigned, size_t>, unsigned> g_resident; // (device, kernel, block, lds)
std::map<int, int> g_max_lds;                                                   // device -> bytes
} // namespace

int device_max_lds_per_block()
{
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  std::lock_guard<std::mutex> lock(g_query_mutex);
  auto it = g_max_lds.find(dev);
  if (it != g_max_lds.end()) return it->second;
  int v = 0;
  if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) return 0;
  g_max_lds.emplace(dev, v);
  return v;
}

unsigned device_resident_blocks(const void* kernel, unsigned block, size_t dyn_lds)
{
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  const auto key = std::make_tuple(dev, kernel, block, dyn_lds);
  std::lock_guard<std::mutex> lock(g_query_mutex);
  auto it = g_resident.find(key);
  if (it != g_resident.end()) return it->second;
  int cus = 0, per_cu = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, static_cast<int>(block), dyn_lds) != hipSuccess ||
      cus <= 0 || per_cu <= 0)
    return 0;
  const unsigned v = static_cast<unsigned>(cus) * static_cast<unsigned>(per_cu);
  g_resident.emplace(key, v);
  return v;
}

// ---------------------------------------------------------------------------------------
// Whole-sequence scans: every count belongs to an event, so the offsets follow from the events'
// totals, which the kernels that make the counts add up on the way.

// Events in descending order of their hit count (buckets of 32 hits, order within a bucket
// unspecified), for launching search_by_triplet largest events first: with every event in
// flight at once, the largest event sets the duration of the launch. Results do not depend on
// the order. One workgroup of 1024 threads.
constexpr unsigned order_buckets = 1024;
template<typename F>
__device__ __forceinline__ void
order_events(unsigned n, F&& hits_of, uint32_t (&bucket)[order_buckets], uint32_t* scratch, uint32_t* order)
{
  static_assert(order_buckets == scan_block, "a bucket per thread");
  bucket[threadIdx.x] = 0;
  __syncthreads();
  const auto key = [&](unsigned e) { return order_buckets - 1 - min(hits_of(e) >> 5, order_buckets - 1); }; // descending
  for (unsigned e = threadIdx.x; e < n; e += blockDim.x) atomicAdd(&bucket[key(e)], 1u);
  __syncthreads();
  uint32_t total;
  const uint32_t ex = block_exclusive_scan(bucket[threadIdx.x], scratch, &total);
  bucket[threadIdx.x] = ex;
  __syncthreads();
  for (unsigned e = threadIdx.x; e < n; e += blockDim.x) order[atomicAdd(&bucket[key(e)], 1u)] = e;
}

__global__ void __launch_bounds__(scan_block) k_order_events_by_hits(
  const uint32_t* offsets_estimated_input_size,
  const uint32_t* number_of_events,
  uint32_t* order)
{
  __shared__ uint32_t bucket[order_buckets];
  __shared__ uint32_t scratch[scan_block / wave_size];
  order_events(
    number_of_events[0],
    [&](unsigned e) {
      return offsets_estimated_input_size[(e + 1) * n_module_pairs] - offsets_estimated_input_size[e * n_module_pairs];
    },
    bucket, scratch, order);
}

hipError_t launch_order_events_by_hits(
  const uint32_t* offsets_estimated_input_size,
  const uint32_t* number_of_events,
  uint32_t* order,
  hipStream_t s)
{
  hipLaunchKernelGGL(
    k_order_events_by_hits, dim3(1), dim3(scan_block), 0, s, offsets_estimated_input_size, number_of_events, order);
  return hipGetLastError();
}

// The offsets of a.per_event counts per event (26 module pairs, or a retina slot each), about
// scan_tile of them per workgroup: a workgroup starts from the sum of the totals of the events
// before its own, so one launch does what a scan in three launches did, or one workgroup with 32
// strided items per thread (27 us for the 26 000 counts of 1000 events). Two more workgroups,
// where asked for, scan the candidates and order the events meanwhile.
__global__ void __launch_bounds__(scan_block) k_scan_events(const EventScanLaunch a, unsigned events_per_block, unsigned scan_blocks)
{
  __shared__ uint32_t scratch[1][scan_block / wave_size];
  __shared__ uint32_t bucket[order_buckets];
  unsigned b = blockIdx.x;
  if (b >= scan_blocks) {
    if (a.candidates && b == scan_blocks) {
      const uint32_t* const in[1] = {a.candidates};
      if (threadIdx.x == 0) a.candidates_offsets[0] = 0;
      scan_by_waves<1>(in, a.n_events, scratch, [&](unsigned e, unsigned, uint32_t v) { a.candidates_offsets[e + 1] = v; });
    }
    else {
      order_events(a.n_events, [&](unsigned e) { return a.totals[e]; }, bucket, scratch[0], a.order);
    }
    return;
  }
  const unsigned first = b * events_per_block;
  const unsigned last = min(first + events_per_block, a.n_events);
  uint32_t before = 0;
  for (unsigned e = threadIdx.x; e < first; e += scan_block) before += a.totals[e];
  uint32_t base;
  block_exclusive_scan(before, scratch[0], &base);
  const size_t begin = (size_t) first * a.per_event, end = (size_t) last * a.per_event;
  if (b == 0 && threadIdx.x == 0) a.offsets[0] = 0;
  for (size_t c = begin; c < end; c += scan_tile) {
    // Thread t owns scan_items consecutive counts.
    const size_t i = c + (size_t) threadIdx.x * scan_items;
    uint32_t v[scan_items] = {};
    if (i + scan_items <= end) {
      __builtin_memcpy(v, a.counts + i, sizeof(v));
    }
    else {
      for (unsigned k = 0; k < scan_items; ++k)
        if (i + k < end) v[k] = a.counts[i + k];
    }
    uint32_t s = 0;
#pragma unroll
    for (unsigned k = 0; k < scan_items; ++k) s += v[k];
    uint32_t total;
    uint32_t run = base + block_exclusive_scan(s, scratch[0], &total);
#pragma unroll
    for (unsigned k = 0; k < scan_items; ++k) {
      run += v[k];
      if (i + k < end) a.offsets[i + k + 1] = run;
    }
    base += total;
  }
}

hipError_t launch_scan_events(const EventScanLaunch& a, hipStream_t s)
{
  if (!a.n_events) return hipSuccess;
  const unsigned events_per_block = std::max(scan_tile / a.per_event, 1u);
  const unsigned blocks = (a.n_events + events_per_block - 1) / events_per_block;
  hipLaunchKernelGGL(
    k_scan_events, dim3(blocks + (a.candidates ? 1 : 0) + (a.order ? 1 : 0)), dim3(scan_block), 0, s, a, events_per_block,
    blocks);
  return hipGetLastError();
}

// Offsets of the events' tracks, kept three-hit tracks, all tracks and track hits, by one workgroup.
__global__ void __launch_bounds__(scan_block) k_track_offsets(const TrackOffsetsLaunch a)
{
  __shared__ uint32_t scratch[3][scan_block / wave_size];
  const uint32_t* const in[3] = {a.number_of_velo_tracks, a.number_of_three_hit_tracks, a.event_track_hits};
  if (threadIdx.x == 0)
    a.offsets_velo_tracks[0] = a.offsets_three_hit[0] = a.offsets_all_velo_tracks[0] = a.event_hit_offsets[0] = 0;
  uint32_t tracks = 0;
  scan_by_waves<3>(in, a.n_events, scratch, [&](unsigned e, unsigned k, uint32_t v) {
    if (k == 0) {
      a.offsets_velo_tracks[e + 1] = v;
      tracks = v;
    }
    else if (k == 1) {
      a.offsets_three_hit[e + 1] = v;
      a.offsets_all_velo_tracks[e + 1] = tracks + v;
    }
    else {
      a.event_hit_offsets[e + 1] = v;
    }
  });
}

hipError_t launch_track_offsets(const TrackOffsetsLaunch& a, hipStream_t s)
{
  if (!a.n_events) return hipSuccess;
  hipLaunchKernelGGL(k_track_offsets, dim3(1), dim3(scan_block), 0, s, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------------
// K7 (grid = number of events).
__global__ void k_copy_track_hit_number(
  const TrackHits* tracks_all,
  const uint32_t* offsets_velo_tracks,
  const uint32_t* offsets_estimated_input_size,
  const uint32_t* offsets_three_hit,
  uint32_t* velo_track_hit_number,
  uint32_t* offsets_all_velo_tracks)
{
  const unsigned e = blockIdx.x;
  const TrackHits* tracks = tracks_all + track_offset(offsets_estimated_input_size, e);
  const unsigned n_tracks = offsets_velo_tracks[e + 1] - offsets_velo_tracks[e];
  const unsigned n_three = offsets_three_hit[e + 1] - offsets_three_hit[e];
  uint32_t* out = velo_track_hit_number + offsets_velo_tracks[e] + offsets_three_hit[e];
  for (unsigned i = threadIdx.x; i < n_tracks; i += blockDim.x) out[i] = tracks[i].hitsNum;
  for (unsigned i = threadIdx.x; i < n_three; i += blockDim.x) out[n_tracks + i] = 3;
  if (threadIdx.x == 0) {
    offsets_all_velo_tracks[e + 1] = offsets_velo_tracks[e + 1] + offsets_three_hit[e + 1];
    if (e == 0) offsets_all_velo_tracks[0] = 0;
  }
}

// K8: one thread per (track, hit); the event's tracks are [main tracks][filtered 3-hit tracks].
constexpr unsigned consolidate_lds_tracks = 2047; // tracks of an event whose offsets are staged in LDS
constexpr unsigned consolidate_lds_hits = 4096;    // track hits of an event mapped to their tracks in LDS

__global__ void k_consolidate_tracks(
  const uint32_t* event_list,
  const uint32_t* number_of_events,
  const uint32_t* offsets_all_velo_tracks,
  const TrackHits* tracks_all,
  const uint32_t* offsets_velo_track_hit_number,
  const char* sorted_container,
  const uint32_t* offsets_estimated_input_size,
  const TrackletHits* three_hit_output_all,
  const uint32_t* offsets_three_hit,
  char* velo_track_hits,
  uint8_t* accepted)
{
  const unsigned e = event_list ? event_list[blockIdx.x] : blockIdx.x;
  const unsigned n_events = number_of_events[0];
  const unsigned total_clusters = offsets_estimated_input_size[n_module_pairs * n_events];
  const unsigned total_tracks = offsets_all_velo_tracks[n_events];
  const unsigned total_hits = offsets_velo_track_hit_number[total_tracks];
  const Clusters in {const_cast<char*>(sorted_container), total_clusters};
  const Clusters out {velo_track_hits, total_hits};
  const unsigned hit_offset = offsets_estimated_input_size[e * n_module_pairs];
  const unsigned toff = track_offset(offsets_estimated_input_size, e);
  const unsigned t0 = offsets_all_velo_tracks[e];
  const unsigned n_total = offsets_all_velo_tracks[e + 1] - t0;
  const unsigned n_main = n_total - (offsets_three_hit[e + 1] - offsets_three_hit[e]);
  const unsigned h_begin = offsets_velo_track_hit_number[t0];
  const unsigned h_end = offsets_velo_track_hit_number[t0 + n_total];
  for (unsigned i = threadIdx.x; i < n_total; i += blockDim.x)
    if (accepted) accepted[t0 + i] = 1;
  // The event's slice of the hit-number offsets, in LDS when it fits. With it, every track
  // writes (track, position in the track) for each of its hits into an LDS map (one thread per
  // track), so a hit reads its track in one LDS access; otherwise each hit finds its track by a
  // binary search over the offsets.
  __shared__ uint32_t s_off[consolidate_lds_tracks + 1];
  __shared__ uint16_t s_map[consolidate_lds_hits];
  const bool in_lds = n_total <= consolidate_lds_tracks;
  const bool mapped = in_lds && h_end - h_begin <= consolidate_lds_hits;
  if (in_lds)
    for (unsigned i = threadIdx.x; i <= n_total; i += blockDim.x) s_off[i] = offsets_velo_track_hit_number[t0 + i];
  __syncthreads();
  if (mapped) {
    static_assert(consolidate_lds_tracks < (1u << 11) && max_track_size <= 32, "(track, position) in 16 bits");
    for (unsigned t = threadIdx.x; t < n_total; t += blockDim.x) {
      const unsigned a = s_off[t] - h_begin, b = s_off[t + 1] - h_begin;
      for (unsigned j = a; j < b; ++j) s_map[j] = static_cast<uint16_t>((t << 5) | (j - a));
    }
    __syncthreads();
  }
  const uint32_t* off = in_lds ? s_off : offsets_velo_track_hit_number + t0;
  for (unsigned h = h_begin + threadIdx.x; h < h_end; h += blockDim.x) {
    unsigned lo, k;
    if (mapped) {
      const unsigned m = s_map[h - h_begin];
      lo = m >> 5;
      k = m & 31u;
    }
    else {
      lo = 0;
      unsigned hi = n_total;
      while (hi - lo > 1) {
        const unsigned mid = (lo + hi) / 2;
        if (off[mid] <= h) lo = mid;
        else hi = mid;
      }
      k = h - off[lo];
    }
    const unsigned hit = lo < n_main ? tracks_all[toff + lo].hits[k] : three_hit_output_all[toff + lo - n_main].hits[k];
    const size_t src = (size_t) hit_offset + hit;
    // All four fields are read before any is written (the output may not alias the input, but
    // the compiler cannot know that and would otherwise wait out each read in turn).
    const uint32_t id = in.ids()[src];
    const float x = in.xyz()[3 * src], y = in.xyz()[3 * src + 1], z = in.xyz()[3 * src + 2];
    out.ids()[h] = id;
    out.xyz()[3 * (size_t) h] = x;
    out.xyz()[3 * (size_t) h + 1] = y;
    out.xyz()[3 * (size_t) h + 2] = z;
  }
}

// ---------------------------------------------------------------------------------------
// K9
struct KState {
  float x, y, z, tx, ty;
  float c00, c20, c22, c11, c31, c33;
};

// FP64 covariance fallback (no reference counterpart): the FP32 update (1 - gain_p) * pp_pred
// loses about kappa * 2^-24 of relative accuracy, kappa = 1 + w * pp_pred (about 1e7 on a
// track's first step). Above kappa = 100 the step's covariance prediction and update run in
// FP64 from the stored FP32 covariance, the update as (1 - gain_p) = inv / w, and the three
// terms are rounded to FP32; the state update keeps the reference's FP32 arithmetic.
constexpr float kalman_kappa_limit_minus_one = 99.f;

// One coordinate's filter step to the hit at z_hit with measurement m and weight w: position
// p, slope t and their covariance (pp, pt, tt) are predicted over dz and updated with the gain
// (the reference's expression order, VeloKalmanFilter.cuh:25-60).
template<bool fp64_fallback>
__device__ __forceinline__ void
filter_step(float z, float z_hit, float m, float w, float& p, float& t, float& pp, float& pt, float& tt)
{
  const float dz = z_hit - z;
  const float p_pred = p + dz * t;
  const float dz_tt = dz * tt;
  const float pt_pred = pt + dz_tt;
  const float dz_pt = dz * pt;
  const float pp_pred = pp + 2 * dz_pt + dz * dz_tt;
  const float tt_pred = tt;
  const float inv = 1.0f / ((1.0f / w) + pp_pred);
  const float gain_p = pp_pred * inv;
  const float gain_t = pt_pred * inv;
  const float res = m - p_pred;
  p = p_pred + gain_p * res;
  t = t + gain_t * res;
  if (fp64_fallback && pp_pred * w > kalman_kappa_limit_minus_one) {
    const double dzd = dz, c00 = pp, c20 = pt, c22 = tt;
    const double pt_d = c20 + dzd * c22;
    const double pp_d = c00 + 2.0 * (dzd * c20) + dzd * (dzd * c22);
    const double tt_d = c22;
    const double iw = 1.0 / static_cast<double>(w);
    const double inv_d = 1.0 / (iw + pp_d);
    pp = static_cast<float>(pp_d * iw * inv_d);
    pt = static_cast<float>(pt_d * iw * inv_d);
    tt = static_cast<float>(tt_d - pt_d * pt_d * inv_d);
    return;
  }
  pp = (1 - gain_p) * pp_pred;
  pt = (1 - gain_p) * pt_pred;
  tt = tt_pred - gain_t * pt_pred;
}

// The coordinates of a track's first two and last two hits (0, 1, nh - 2, nh - 1; nh >= 2),
// read together before the fits.
struct TrackEnds {
  float f[3], f1[3], l1[3], l[3];
};

// A hit's coordinates, and how a fit reads the hits of its track: consecutive coordinates in memory,
// or by the track's hit indices from the event's hits (both may be in LDS). The index is signed: an
// unsigned one may wrap, so every hit's address would be computed anew (drop-in fit of 5000 one-vertex
// events: 63 us, 68 with unsigned ones).
struct Xyz {
  float c[3];
};
struct PackedHits {
  const float* xyz;
  __device__ __forceinline__ Xyz operator()(int i) const { return {xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2]}; }
};
struct GatheredHits {
  const uint16_t* index;
  const float* xyz;
  __device__ __forceinline__ Xyz operator()(int i) const
  {
    const unsigned h = 3u * index[i];
    return {xyz[h], xyz[h + 1], xyz[h + 2]};
  }
};

template<bool upstream, bool fp64_fallback, typename H>
__device__ __forceinline__ KState
simplified_fit(const H& hits, unsigned nh, const TrackEnds& te, float at_tx, float at_ty, const float* beamline, bool backward)
{
  const int direction = (backward ? 1 : -1) * (upstream ? 1 : -1);
  const float layer_noise = 1e-8f + 7e-6f * (at_tx * at_tx + at_ty * at_ty);
  int first = 0;
  int last = static_cast<int>(nh) - 1;
  int step = 1;
  const bool reverse = (te.l[2] - te.f[2]) * direction < 0;
  if (reverse) {
    const int t = first;
    first = last;
    last = t;
    step = -1;
  }
  KState s;
  s.x = reverse ? te.l[0] : te.f[0];
  s.y = reverse ? te.l[1] : te.f[1];
  s.z = reverse ? te.l[2] : te.f[2];
  s.tx = at_tx;
  s.ty = at_ty;
  s.c00 = param_w_inverted;
  s.c11 = param_w_inverted;
  s.c20 = 0.f;
  s.c31 = 0.f;
  s.c22 = 1.f;
  s.c33 = 1.f;
  // The next hit's coordinates are read while the current step computes (each step waits for
  // nothing but its own arithmetic).
  float nx = reverse ? te.l1[0] : te.f1[0], ny = reverse ? te.l1[1] : te.f1[1], nz = reverse ? te.l1[2] : te.f1[2];
  for (int i = first + step; i != last + step; i += step) {
    const float hx = nx, hy = ny, hz = nz;
    if (i + step != last + step) {
      const Xyz next = hits(i + step);
      nx = next.c[0];
      ny = next.c[1];
      nz = next.c[2];
    }
    s.c22 += layer_noise;
    s.c33 += layer_noise;
    filter_step<fp64_fallback>(s.z, hz, hx, param_w, s.x, s.tx, s.c00, s.c20, s.c22);
    filter_step<fp64_fallback>(s.z, hz, hy, param_w, s.y, s.ty, s.c11, s.c31, s.c33);
    s.z = hz;
  }
  s.c22 += layer_noise;
  s.c33 += layer_noise;
  float delta_z = 0.f;
  if constexpr (upstream) {
    delta_z = (s.tx * (beamline[0] - s.x) + s.ty * (beamline[1] - s.y)) / (s.tx * s.tx + s.ty * s.ty);
  }
  else {
    delta_z = z_end_velo - s.z;
  }
  s.x = s.x + s.tx * delta_z;
  s.y = s.y + s.ty * delta_z;
  s.z = s.z + delta_z;
  const float dz2 = delta_z * delta_z;
  s.c00 += dz2 * s.c22 + 2.f * delta_z * s.c20;
  s.c11 += dz2 * s.c33 + 2.f * delta_z * s.c31;
  s.c20 += s.c22 * delta_z;
  s.c31 += s.c33 * delta_z;
  return s;
}

__device__ __forceinline__ void store_state(float* base, unsigned total_tracks, unsigned i, const KState& s)
{
  float* st = base + 6 * (size_t) i;
  st[0] = s.x;
  st[1] = s.y;
  st[2] = s.z;
  st[3] = s.tx;
  st[4] = s.ty;
  float* cv = base + 6 * (size_t) total_tracks + 8 * (size_t) i;
  cv[0] = s.c00;
  cv[1] = s.c20;
  cv[2] = s.c22;
  cv[3] = s.c11;
  cv[4] = s.c31;
  cv[5] = s.c33;
}

// One track: linear_fit, the upstream fit to the beamline and the downstream fit to the end of
// the VELO (VeloKalmanFilter.cu:384-399).
template<typename H>
__device__ __forceinline__ void fit_track(
  const H& hits,
  unsigned nh,
  unsigned t,
  unsigned total_tracks,
  const float* bl,
  uint8_t* is_backward,
  float* beamline_states,
  float* endvelo_states,
  unsigned fp64_fallback)
{
  TrackEnds te;
  {
    const Xyz f = hits(0), f1 = hits(1), l1 = hits(nh - 2), l = hits(nh - 1);
#pragma unroll
    for (unsigned c = 0; c < 3; ++c) {
      te.f[c] = f.c[c];
      te.f1[c] = f1.c[c];
      te.l1[c] = l1.c[c];
      te.l[c] = l.c[c];
    }
  }
  __builtin_amdgcn_sched_barrier(0); // the four hits' loads are in flight together
  // linear_fit (VeloKalmanFilter.cu:335-355)
  const float fx = te.f[0], fy = te.f[1], fz = te.f[2];
  const float lx = te.l[0], ly = te.l[1], lz = te.l[2];
  const float ltx = (lx - fx) / (lz - fz);
  const float lty = (ly - fy) / (lz - fz);
  const float ldz = (ltx * (bl[0] - lx) + lty * (bl[1] - ly)) / (ltx * ltx + lty * lty);
  const float lin_z = lz + ldz;
  const bool backward = lin_z > fz;
  is_backward[t] = backward;
  if (fp64_fallback) {
    const KState b = simplified_fit<true, true>(hits, nh, te, ltx, lty, bl, backward);
    const KState v = simplified_fit<false, true>(hits, nh, te, b.tx, b.ty, bl, backward);
    store_state(beamline_states, total_tracks, t, b);
    store_state(endvelo_states, total_tracks, t, v);
  }
  else {
    const KState b = simplified_fit<true, false>(hits, nh, te, ltx, lty, bl, backward);
    const KState v = simplified_fit<false, false>(hits, nh, te, b.tx, b.ty, bl, backward);
    store_state(beamline_states, total_tracks, t, b);
    store_state(endvelo_states, total_tracks, t, v);
  }
}

// KalmanStates view of event e (VeloKalmanFilter.cu:370-374).
__device__ __forceinline__ void write_states_view(
  velo_kalman_states_view* views, const float* states, const uint32_t* offsets_all_velo_tracks, unsigned e,
  unsigned n_events)
{
  velo_kalman_states_view v;
  v.base_pointer = reinterpret_cast<const char*>(states);
  v.offset = offsets_all_velo_tracks[e];
  v.size = offsets_all_velo_tracks[e + 1] - offsets_all_velo_tracks[e];
  v.total_number_of_tracks = offsets_all_velo_tracks[n_events];
  v.pad_ = 0;
  views[e] = v;
}

// One workgroup per listed event, one thread per track. views: the tracks and their hits come
// through the event's Tracks view (Track -> Hits -> the consolidated container), as the
// reference reads them; otherwise from the hit-number offsets and the container.
template<bool views>
__global__ void k_kalman_filter(
  const uint32_t* event_list,
  const uint32_t* number_of_events,
  const uint32_t* offsets_all_velo_tracks,
  const uint32_t* offsets_velo_track_hit_number,
  const char* velo_track_hits,
  const velo_tracks_view* tracks_view,
  const float* beamline,
  uint8_t* is_backward,
  float* beamline_states,
  float* endvelo_states,
  velo_kalman_states_view* beamline_states_view,
  velo_kalman_states_view* endvelo_states_view,
  unsigned fp64_fallback)
{
  const unsigned e = event_list ? event_list[blockIdx.x] : blockIdx.x;
  const unsigned n_events = number_of_events[0];
  const unsigned total_tracks = offsets_all_velo_tracks[n_events];
  const float bl[2] = {beamline[0], beamline[1]};
  if (threadIdx.x == 0) {
    if (beamline_states_view)
      write_states_view(beamline_states_view, beamline_states, offsets_all_velo_tracks, e, n_events);
    if (endvelo_states_view)
      write_states_view(endvelo_states_view, endvelo_states, offsets_all_velo_tracks, e, n_events);
  }
  if constexpr (views) {
    const velo_tracks_view tv = tracks_view[e];
    for (unsigned i = threadIdx.x; i < tv.size; i += blockDim.x) {
      const velo_track_view tr = tv.track[i];
      const velo_hits_view h = *tr.hits;
      if (tr.number_of_hits < 2) continue;
      const float* xyz = reinterpret_cast<const float*>(h.base_pointer) + h.total_number_of_hits +
                         3 * (size_t) (h.offset + tr.offset);
      fit_track(PackedHits {xyz}, tr.number_of_hits, tv.offset + i, total_tracks, bl, is_backward, beamline_states,
                endvelo_states, fp64_fallback);
    }
  }
  else {
    const unsigned total_hits = offsets_velo_track_hit_number[total_tracks];
    const float* xyz_all = reinterpret_cast<const float*>(velo_track_hits) + total_hits;
    for (unsigned t = offsets_all_velo_tracks[e] + threadIdx.x; t < offsets_all_velo_tracks[e + 1];
         t += blockDim.x) {
      const unsigned h0 = offsets_velo_track_hit_number[t];
      const unsigned nh = offsets_velo_track_hit_number[t + 1] - h0;
      if (nh < 2) continue; // every VELO track has >= 3 hits
      fit_track(PackedHits {xyz_all + 3 * (size_t) h0}, nh, t, total_tracks, bl, is_backward, beamline_states, endvelo_states,
                fp64_fallback);
    }
  }
}

// Copies `words` 32-bit words (from any 2-byte boundary) to 16-byte aligned LDS by the workgroup, 16
// bytes a lane, four of those in flight (one at a time, every pass waits out a memory round trip).
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_unaligned __attribute__((aligned(2)));
typedef uint32_t u32_unaligned __attribute__((aligned(2)));
__device__ __forceinline__ void copy_to_lds(uint32_t* to, const void* from, unsigned words)
{
  const auto* src = static_cast<const u32x4_unaligned*>(from);
  const unsigned quads = words / 4;
  for (unsigned q0 = threadIdx.x; q0 < quads; q0 += 4 * blockDim.x) {
    u32x4 v[4];
#pragma unroll
    for (unsigned k = 0; k < 4; ++k) v[k] = src[min(q0 + k * blockDim.x, quads - 1)];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (unsigned k = 0; k < 4; ++k)
      if (q0 + k * blockDim.x < quads) reinterpret_cast<u32x4*>(to)[q0 + k * blockDim.x] = v[k];
  }
  const unsigned w = 4 * quads + threadIdx.x;
  if (w < words) to[w] = static_cast<const u32_unaligned*>(from)[w];
}

// K7, K8 and K9 of one event by one workgroup (whole-sequence path): the tracks' hit numbers and
// offsets from the event's hit offset, the consolidated hits, and both fits of every track. The
// event's coordinates (nearly all of its hits end in tracks) and its tracks, 256 at a time, are
// copied to LDS in whole lines, so the fits wait for no memory: a load in their chain of steps
// would also wait for every store issued before it. Sixteen lanes copy a track's hits, so that
// neighbouring lanes write neighbouring slots, four tracks read before the first is written. Bound by the divisions of the fits' chains, and
// with many events in flight by the bytes (about 50 KB an event). Events with more hits than the
// LDS holds read the coordinates from the container.
constexpr unsigned fit_block = 256;
constexpr unsigned fit_copy_lanes = 16;
constexpr unsigned fit_lds_hits = 1920; // with the tracks 37 KB: four workgroups a CU, so 1000 events are in flight at once
struct FitChunk {
  const TrackHits* tracks; // in LDS
  const uint32_t* first;   // in LDS
  unsigned n;
  unsigned t0;             // number of the first track
  unsigned total_tracks;
};
template<bool fp64_fallback>
__device__ __forceinline__ void copy_and_fit(
  const TrackFitLaunch& a, const FitChunk& f, const uint32_t* ids, const float* xyz, const Clusters& out, const float* bl)
{
  const unsigned tid = threadIdx.x;
  constexpr unsigned groups = fit_block / fit_copy_lanes, batch = 4;
  for (unsigned j = tid % fit_copy_lanes; j < max_track_size; j += fit_copy_lanes) {
    for (unsigned g0 = tid / fit_copy_lanes; g0 < f.n; g0 += batch * groups) {
      uint32_t id[batch];
      Xyz p[batch];
      bool has[batch];
#pragma unroll
      for (unsigned k = 0; k < batch; ++k) {
        const unsigned g = min(g0 + k * groups, f.n - 1);
        has[k] = g0 + k * groups < f.n && j < f.tracks[g].hitsNum;
        const unsigned h = f.tracks[g].hits[has[k] ? j : 0u];
        id[k] = ids[h];
        p[k] = {xyz[3 * h], xyz[3 * h + 1], xyz[3 * h + 2]};
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (unsigned k = 0; k < batch; ++k) {
        if (!has[k]) continue;
        const size_t at = (size_t) f.first[g0 + k * groups] + j;
        out.ids()[at] = id[k];
        out.xyz()[3 * at] = p[k].c[0];
        out.xyz()[3 * at + 1] = p[k].c[1];
        out.xyz()[3 * at + 2] = p[k].c[2];
      }
    }
  }
  if (tid < f.n && f.tracks[tid].hitsNum >= 2) // every VELO track has >= 3 hits
    fit_track(GatheredHits {f.tracks[tid].hits, xyz}, f.tracks[tid].hitsNum, f.t0 + tid, f.total_tracks, bl, a.is_backward,
              reinterpret_cast<float*>(a.beamline_states), reinterpret_cast<float*>(a.endvelo_states), fp64_fallback);
}

template<bool fp64_fallback>
__global__ void __launch_bounds__(fit_block) k_consolidate_and_fit(const TrackFitLaunch a)
{
  __shared__ __align__(16) float s_xyz[3 * fit_lds_hits];
  __shared__ __align__(16) TrackHits s_tracks[fit_block]; // a chunk of tracks
  __shared__ uint32_t s_first[fit_block];   // their first hits' slots
  __shared__ uint32_t s_scan[fit_block / wave_size];
  const unsigned e = blockIdx.x, tid = threadIdx.x;
  const uint32_t* est = a.offsets_estimated_input_size;
  const unsigned total_clusters = est[n_module_pairs * a.n_events];
  const unsigned hit_offset = est[e * n_module_pairs];
  const unsigned n_hits = est[(e + 1) * n_module_pairs] - hit_offset;
  const unsigned toff = track_offset(est, e);
  const unsigned t0 = a.offsets_all_velo_tracks[e];
  const unsigned n_total = a.offsets_all_velo_tracks[e + 1] - t0;
  const unsigned n_main = n_total - (a.offsets_three_hit[e + 1] - a.offsets_three_hit[e]);
  const unsigned total_tracks = a.offsets_all_velo_tracks[a.n_events];
  const unsigned total_hits = a.event_hit_offsets[a.n_events];
  const float bl[2] = {a.beamline[0], a.beamline[1]};
  const Clusters in {const_cast<char*>(a.sorted_container), total_clusters};
  const Clusters out {a.velo_track_hits, total_hits};
  const uint32_t* ids = in.ids() + hit_offset;
  const float* xyz = in.xyz() + 3 * (size_t) hit_offset;
  const TrackHits* tracks = static_cast<const TrackHits*>(a.tracks) + toff;
  const TrackletHits* three = static_cast<const TrackletHits*>(a.three_hit_tracks_output) + toff;
  const bool staged = a.lds_hits && n_hits <= fit_lds_hits;
  if (staged) copy_to_lds(reinterpret_cast<uint32_t*>(s_xyz), xyz, 3 * n_hits);
  unsigned slot = a.event_hit_offsets[e];
  for (unsigned c = 0; c < n_total; c += fit_block) {
    const unsigned i = c + tid;
    // The chunk's tracks in words, from a 2-byte boundary (an odd number of tracks leaves half a word,
    // the last one's number of hits), kept three-hit tracks after them.
    const unsigned n_copy = min(fit_block, n_main - min(n_main, c));
    copy_to_lds(reinterpret_cast<uint32_t*>(s_tracks), tracks + c, sizeof(TrackHits) * n_copy / 4);
    if (tid == 0 && n_copy % 2) s_tracks[n_copy - 1].hitsNum = tracks[c + n_copy - 1].hitsNum;
    if (i >= n_main && i < n_total) {
      const TrackletHits t = three[i - n_main];
      s_tracks[tid].hits[0] = t.hits[0];
      s_tracks[tid].hits[1] = t.hits[1];
      s_tracks[tid].hits[2] = t.hits[2];
      s_tracks[tid].hitsNum = 3;
    }
    __syncthreads();
    const unsigned nh = i < n_total ? s_tracks[tid].hitsNum : 0u;
    uint32_t chunk_hits;
    const unsigned first = slot + block_exclusive_scan(nh, s_scan, &chunk_hits);
    slot += chunk_hits;
    s_first[tid] = first;
    if (i < n_total) {
      a.velo_track_hit_number[t0 + i] = nh;
      a.offsets_velo_track_hit_number[t0 + i] = first;
      a.accepted_velo_tracks[t0 + i] = 1;
    }
    __syncthreads();
    // Two copies of the code: a read that may go to LDS or to memory would be a generic (flat) one.
    const FitChunk f {s_tracks, s_first, min(fit_block, n_total - c), t0 + c, total_tracks};
    if (staged) copy_and_fit<fp64_fallback>(a, f, ids, s_xyz, out, bl);
    else copy_and_fit<fp64_fallback>(a, f, ids, xyz, out, bl);
    __syncthreads(); // the chunk's tracks have been read
  }
  if (e + 1 == a.n_events && tid == 0) a.offsets_velo_track_hit_number[total_tracks] = total_hits;
}

hipError_t launch_consolidate_and_fit(const TrackFitLaunch& a, hipStream_t s)
{
  if (!a.n_events) return hipSuccess;
  if (a.fp64_fallback) hipLaunchKernelGGL(k_consolidate_and_fit<true>, dim3(a.n_events), dim3(fit_block), 0, s, a);
  else hipLaunchKernelGGL(k_consolidate_and_fit<false>, dim3(a.n_events), dim3(fit_block), 0, s, a);
  return hipGetLastError();
}

// create_velo_views (VeloConsolidateTracks.cu:11-46): event e's Hits and Tracks views and one
// Track view per track; the first workgroup also writes the multi-event view and its address.
__global__ void k_create_velo_views(
  const uint32_t* number_of_events,
  const uint32_t* offsets_all_velo_tracks,
  const uint32_t* offsets_velo_track_hit_number,
  const char* velo_track_hits,
  velo_hits_view* hits_view,
  velo_track_view* track_view,
  velo_tracks_view* tracks_view,
  velo_multi_event_tracks_view* multi_view,
  const velo_multi_event_tracks_view** imec)
{
  const unsigned n_events = number_of_events[0];
  const unsigned e = blockIdx.x;
  const unsigned first_track = offsets_all_velo_tracks[e];
  const unsigned n_tracks = offsets_all_velo_tracks[e + 1] - first_track;
  const uint32_t* hit_offsets = offsets_velo_track_hit_number + first_track;
  const unsigned first_hit = hit_offsets[0];
  for (unsigned i = threadIdx.x; i < n_tracks; i += blockDim.x) {
    velo_track_view t;
    t.hits = hits_view + e;
    t.track_index = i;
    t.track_container_offset = first_track;
    t.offset = hit_offsets[i] - first_hit;
    t.number_of_hits = hit_offsets[i + 1] - hit_offsets[i];
    track_view[first_track + i] = t;
  }
  if (threadIdx.x == 0) {
    velo_hits_view h;
    h.base_pointer = velo_track_hits;
    h.offset = first_hit;
    h.size = offsets_velo_track_hit_number[first_track + n_tracks] - first_hit;
    h.total_number_of_hits = offsets_velo_track_hit_number[offsets_all_velo_tracks[n_events]];
    h.pad_ = 0;
    hits_view[e] = h;
    velo_tracks_view ts;
    ts.track = track_view + first_track;
    ts.size = n_tracks;
    ts.offset = first_track;
    tracks_view[e] = ts;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    velo_multi_event_tracks_view m;
    m.type_id = VELO_TYPE_ID_VELO_TRACKS;
    m.pad_ = 0;
    m.container = tracks_view;
    m.number_of_events = n_events;
    m.pad2_ = 0;
    *multi_view = m;
    imec[0] = multi_view;
  }
}

// The Velo::Clusters view of each listed event (one thread per list entry); with zero_all every
// entry is cleared first by the same threads (the reference's memset of the retina decoding's
// views, DecodeRetinaClusters.cu:442; a single workgroup keeps the clear before the writes).
__global__ void k_clusters_views(
  const uint32_t* event_list,
  unsigned n_list,
  unsigned n_events,
  unsigned zero_all,
  const uint32_t* number_of_events,
  const uint32_t* totals,
  unsigned totals_stride,
  char* container,
  velo_clusters_view* views)
{
  if (zero_all) {
    for (unsigned i = threadIdx.x; i < n_events; i += blockDim.x) {
      velo_clusters_view z;
      z.base_pointer = nullptr;
      z.total_number_of_hits = 0;
      z.offset = 0;
      views[i] = z;
    }
    __syncthreads();
  }
  const unsigned total = totals[(size_t) totals_stride * number_of_events[0]];
  for (unsigned i = threadIdx.x; i < n_list; i += blockDim.x) {
    velo_clusters_view v;
    v.base_pointer = container;
    v.total_number_of_hits = total;
    v.offset = 0;
    views[event_list ? event_list[i] : i] = v;
  }
}

hipError_t launch_copy_track_hit_number(const CopyHitNumberLaunch& a, hipStream_t s)
{
  if (!a.n_events) return hipSuccess;
  hipLaunchKernelGGL(
    k_copy_track_hit_number, dim3(a.n_events), dim3(256), 0, s, reinterpret_cast<const TrackHits*>(a.tracks),
    a.offsets_velo_tracks, a.offsets_estimated_input_size, a.offsets_three_hit, a.velo_track_hit_number,
    a.offsets_all_velo_tracks);
  return hipGetLastError();
}

hipError_t launch_consolidate_tracks(const ConsolidateLaunch& a, hipStream_t s)
{
  if (!a.n_list) return hipSuccess;
  hipLaunchKernelGGL(
    k_consolidate_tracks, dim3(a.n_list), dim3(256), 0, s, a.event_list, a.number_of_events, a.offsets_all_velo_tracks,
    reinterpret_cast<const TrackHits*>(a.tracks), a.offsets_velo_track_hit_number, a.sorted_container,
    a.offsets_estimated_input_size, reinterpret_cast<const TrackletHits*>(a.three_hit_tracks_output),
    a.offsets_three_hit, a.velo_track_hits, a.accepted_velo_tracks);
  return hipGetLastError();
}

hipError_t launch_kalman_filter(const KalmanLaunch& a, hipStream_t s)
{
  if (!a.n_list) return hipSuccess;
  auto* bsv = static_cast<velo_kalman_states_view*>(a.beamline_states_view);
  auto* esv = static_cast<velo_kalman_states_view*>(a.endvelo_states_view);
  const auto* tv = static_cast<const velo_tracks_view*>(a.tracks_view);
  if (tv)
    hipLaunchKernelGGL(
      k_kalman_filter<true>, dim3(a.n_list), dim3(256), 0, s, a.event_list, a.number_of_events,
      a.offsets_all_velo_tracks, a.offsets_velo_track_hit_number, a.velo_track_hits, tv, a.beamline, a.is_backward,
      reinterpret_cast<float*>(a.beamline_states), reinterpret_cast<float*>(a.endvelo_states), bsv, esv,
      a.fp64_fallback);
  else
    hipLaunchKernelGGL(
      k_kalman_filter<false>, dim3(a.n_list), dim3(256), 0, s, a.event_list, a.number_of_events,
      a.offsets_all_velo_tracks, a.offsets_velo_track_hit_number, a.velo_track_hits, tv, a.beamline, a.is_backward,
      reinterpret_cast<float*>(a.beamline_states), reinterpret_cast<float*>(a.endvelo_states), bsv, esv,
      a.fp64_fallback);
  return hipGetLastError();
}

hipError_t launch_create_velo_views(const VeloViewsLaunch& a, hipStream_t s)
{
  if (!a.n_events) return hipSuccess;
  hipLaunchKernelGGL(
    k_create_velo_views, dim3(a.n_events), dim3(256), 0, s, a.number_of_events, a.offsets_all_velo_tracks,
    a.offsets_velo_track_hit_number, a.velo_track_hits, static_cast<velo_hits_view*>(a.hits_view),
    static_cast<velo_track_view*>(a.track_view), static_cast<velo_tracks_view*>(a.tracks_view),
    static_cast<velo_multi_event_tracks_view*>(a.multi_event_tracks_view),
    static_cast<const velo_multi_event_tracks_view**>(a.imec_velo_tracks));
  return hipGetLastError();
}

hipError_t launch_clusters_views(const ClustersViewLaunch& a, hipStream_t s)
{
  if (!a.n_list && !a.zero_all) return hipSuccess;
  hipLaunchKernelGGL(
    k_clusters_views, dim3(1), dim3(1024), 0, s, a.event_list, a.n_list, a.n_events, unsigned(a.zero_all),
    a.number_of_events, a.totals, a.totals_stride, a.container, static_cast<velo_clusters_view*>(a.views));
  return hipGetLastError();
}

} // namespace velo

// Super-pixel decoding, masked clustering and phi sort for gfx950.
//
//   k_number_of_candidates   VeloCalculateNumberOfCandidates.cu:10-48   one wave per event
//   k_bank_index             VeloCalculateNumberOfCandidates.cu:35-43   last-writer-wins in CPU order
//   k_estimate_input_size    EstimateInputSize.cu:10-239                one workgroup per event
//   k_masked_clustering      MaskedVeloClustering.cu:131-576            one workgroup per event
//   k_sort_by_phi            SortByPhi.cu:49-153                        one wave per module pair
//   k_bank_directory, k_estimate_mp, k_cluster_mp
//                            the same for the whole sequence: the banks of every module pair,
//                            then one wave per module pair for K2, and for K3 and K4 together
//
// The cluster arithmetic (pattern lookup, 64-bit mask growth, centroid, local->global
// transform, hit_phi_16) is evaluated exactly as in the reference with fp contraction off.
#include "velo_common.cuh"
#include "velo_kernels.h"

namespace velo {

constexpr unsigned max_banks_per_mp = 8; // v2/v3: 8 sensors per module pair; v4: 4 sensor pairs

// ---------------------------------------------------------------------------------------
// Bit tricks of MaskedVeloClustering.cu:21-84.
__device__ __forceinline__ uint64_t make_8con_mask(uint64_t c)
{
  return c | ((c & 0x7FFF7FFF7FFF7FFFull) << 1) | ((c & 0xFFFEFFFEFFFEFFFEull) << 15) | (c << 16) |
         ((c & 0xFFFCFFFCFFFCFFFCull) << 17) | ((c & 0xFFFEFFFEFFFEFFFEull) >> 1) |
         ((c & 0x7FFF7FFF7FFF7FFFull) >> 15) | (c >> 16) | ((c & 0x3FFF3FFF3FFF3FFFull) >> 17);
}
__device__ __forceinline__ uint64_t mask_east(uint64_t c)
{
  const uint64_t m = c >> 48;
  return m | ((m & 0x7FFF7FFF7FFF7FFFull) << 1) | (m >> 1);
}
__device__ __forceinline__ uint64_t mask_west(uint64_t c)
{
  const uint64_t m = c << 48;
  return m | (m << 1) | ((m & 0xFFFEFFFEFFFEFFFEull) >> 1);
}

struct Grown {
  uint64_t pixels;
  uint32_t x, y, n;
};

__device__ __forceinline__ Grown grow_cluster(uint64_t pixel_map, uint64_t start, unsigned col_lower, unsigned row_lower)
{
  uint64_t cur = 0, next = start;
  while (cur != next) {
    cur = next;
    next = pixel_map & make_8con_mask(cur);
  }
  const unsigned n = __popcll(cur);
  const unsigned x = col_lower * n + __popcll(cur & 0x00000000FFFF0000ull) + __popcll(cur & 0x0000FFFF00000000ull) * 2 +
                     __popcll(cur & 0xFFFF000000000000ull) * 3;
  // Sum of the row offsets r (bit r of each 16-bit column) by bit planes of r. The reference sums
  // r = 1..14; a pixel at r = 15 makes every caller drop the cluster, so the sums agree wherever
  // they are used.
  const unsigned y = row_lower * n + __popcll(cur & 0xAAAAAAAAAAAAAAAAull) + 2 * __popcll(cur & 0xCCCCCCCCCCCCCCCCull) +
                     4 * __popcll(cur & 0xF0F0F0F0F0F0F0F0ull) + 8 * __popcll(cur & 0xFF00FF00FF00FF00ull);
  return {cur, x, y, n};
}

// Global position and LHCbID of a cluster (MaskedVeloClustering.cu:192-225,459-494).
struct ClusterOut {
  uint32_t id;
  float x, y, z;
  int16_t phi;
};

// A cluster before it is placed: its id holds sensor (bits 18-27), column and row of its pixel
// (cx = bits 8-17, cy = bits 0-7), fx and fy the fractions.
struct ClusterSeed {
  uint32_t id;
  float fx, fy;
};

// The index of a seed's sensor in the geometry.
template<int version>
__device__ __forceinline__ uint32_t seed_sensor(const ClusterSeed& s)
{
  return (s.id >> 18) & (version == 2 || version == 3 ? 0x1FFu : 0x3FFu);
}

__device__ __forceinline__ ClusterOut place_cluster(const Geometry& g, uint32_t sensor, const ClusterSeed& s)
{
  const float* ltg = g.ltg + 12 * sensor;
  const unsigned cx = (s.id >> 8) & 0x3FFu, cy = s.id & 0xFFu;
  // Every geometry load is issued before the first is used (the scheduler would otherwise wait
  // out several memory round trips one after another).
  float m[12];
#pragma unroll
  for (unsigned k = 0; k < 12; ++k) m[k] = ltg[k];
  const float lx = g.local_x[cx], pitch = g.x_pitch[cx];
  __builtin_amdgcn_sched_barrier(0);
  const float local_x = lx + s.fx * pitch;
  const float local_y = (cy + 0.5f + s.fy) * pixel_size;
  ClusterOut c;
  c.id = s.id;
  c.x = m[0] * local_x + m[1] * local_y + m[9];
  c.y = m[3] * local_x + m[4] * local_y + m[10];
  c.z = m[6] * local_x + m[7] * local_y + m[11];
  c.phi = hit_phi_16(c.x, c.y);
  return c;
}

// One or two clusters of an isolated SP from the pattern table (MaskedVeloClustering.cu:165-286).
// Returns the number written into s0, s1.
template<int version>
__device__ __forceinline__ unsigned isolated_sp_clusters(
  const uint8_t* sp_patterns,
  const float* sp_fx,
  const float* sp_fy,
  uint32_t source,
  uint32_t sp_word,
  ClusterSeed& s0,
  ClusterSeed& s1)
{
  constexpr bool v23 = (version == 2 || version == 3);
  const uint32_t sensor_bit = (sp_word >> 23) & 1u;
  const uint32_t sensor_index = v23 ? source : (((source & 0x1FFu) << 1) | sensor_bit);
  const uint32_t sp_addr = (sp_word & 0x007FFF00u) >> 8;
  const uint32_t sp_row = sp_addr & 0x3Fu;
  const uint32_t sp_col = sp_addr >> 6;
  const uint32_t sp = sp_word & 0xFFu;
  const uint32_t idx = sp_patterns[sp];
  auto seed = [&](uint32_t row, uint32_t col, unsigned k) {
    const uint32_t cx = sp_col * 2 + col;
    const uint32_t cy = sp_row * 4 + row;
    return ClusterSeed {lhcb_id_of(sensor_index, sp_col >> 7, cx & 0xFFu, cy), sp_fx[sp * 2 + k], sp_fy[sp * 2 + k]};
  };
  s0 = seed(idx & 0x03u, (idx >> 2) & 1u, 0);
  if (!(idx & 8)) return 1;
  s1 = seed((idx >> 4) & 3u, (idx >> 6) & 1u, 1);
  return 2;
}

// Candidate pixels of a non-isolated SP (EstimateInputSize.cu:104-204), in two steps:
// Neighbours collects in the 18-bit neighbourhood what the other SP words of the bank
// contribute, candidates_final() applies the candidate mask. The neighbour scan keeps the
// reference's behaviour: every word of the bank, of either sensor and isolated or not,
// contributes (EstimateInputSize.cu:111-141).
__device__ __forceinline__ uint32_t neighbourhood_init(uint32_t sp_word)
{
  const uint32_t sp = sp_word & 0xFFu;
  return (sp & 0x0F) | ((sp & 0xF0) << 2);
}

// The pixels that other words of the bank add to an SP's neighbourhood: the OR of the words at the five
// addresses that matter, in three masks whose bits don't collide. Fourteen instructions a word.
struct Neighbours {
  uint32_t top, top_right, right, bot_right, bot; // addresses; all ones: outside the SP grid
  uint32_t column = 0, side = 0, corner = 0;
  __device__ __forceinline__ Neighbours(uint32_t sp_addr)
  {
    constexpr uint32_t outside = 0xFFFFFFFFu;
    const uint32_t row = sp_addr & 0x3Fu;
    const bool up = row < 63u, down = row > 0u, east = sp_addr < (511u << 6);
    top = up ? sp_addr + 1u : outside;
    bot = down ? sp_addr - 1u : outside;
    right = east ? sp_addr + 64u : outside;
    top_right = up && east ? sp_addr + 65u : outside;
    bot_right = down && east ? sp_addr + 63u : outside;
  }
  __device__ __forceinline__ void add(uint32_t other)
  {
    const uint32_t address = (other >> 8) & 0x7FFFu;
    uint32_t mask = address == top ? 0x11u : 0u;
    mask = address == bot ? 0x80u : mask;
    mask = address == bot_right ? 0x08u : mask;
    column |= other & mask;
    side |= other & (address == right ? 0x0Fu : 0u);
    corner |= other & (address == top_right ? 0x01u : 0u);
  }
  __device__ __forceinline__ uint32_t pixels() const
  {
    return ((column & 0x01u) << 4) | ((column & 0x10u) << 6) | (corner << 16) | (side << 12) | ((column & 0x08u) << 8) |
           ((column & 0x80u) >> 2);
  }
};

// Returns a 2-bit mask: bit0 = first candidate (pixels 0,1,4,5), bit1 = second; the pixel
// numbers are returned in *p0, *p1.
__device__ __forceinline__ unsigned candidates_final(uint32_t pixels, unsigned* p0, unsigned* p1)
{
  const uint32_t inside = pixels & 0x3CF;
  const uint32_t mask = (inside << 1) | (inside << 5) | (inside << 6) | (inside << 7);
  const uint32_t working = mask & (~pixels);
  const uint32_t cand = ((working >> 1) & (working >> 5) & (working >> 6) & (working >> 7)) & pixels;
  const uint32_t consolidated = (cand & 0x0F) | ((cand >> 2) & 0xF0);
  const uint32_t first = consolidated & 0x33;
  const uint32_t second = consolidated & 0xCC;
  unsigned m = 0;
  if (first) {
    *p0 = __clz(first) - 24;
    m |= 1;
  }
  if (second) {
    *p1 = __clz(second) - 24;
    m |= 2;
  }
  return m;
}

__device__ __forceinline__ unsigned isolated_cluster_count(uint32_t sp)
{
  const bool pattern_0 = (sp & 0x88) && !(sp & 0x44) && (sp & 0x33);
  const bool pattern_1 = (sp & 0xCC) && !(sp & 0x22) && (sp & 0x11);
  return (pattern_0 | pattern_1) ? 2 : 1;
}

// rest_of_clusters (MaskedVeloClustering.cu:290-496) for one candidate pixel, in two steps:
// window_acc() ORs one other SP word of the bank into the 5-column x 4-row SP window around the
// candidate's SP (pa[c]: one SP column, rows bottom to top, 16 bits per pixel column), and
// masked_cluster_final() grows the cluster and applies the precedence and window-edge rules.
struct Window {
  uint32_t pa0, pa1, pa2, pa3, pa4;
};

template<int version>
__device__ __forceinline__ void
window_acc(int32_t sp_row_lower, int32_t sp_col_lower, uint32_t sensor_number, uint32_t other, Window& w)
{
  if constexpr (version > 3) {
    if (((other >> 23) & 1u) != (sensor_number & 1u)) return;
  }
  if (other & 0x80000000u) return;
  const uint32_t oaddr = (other & 0x007FFF00u) >> 8;
  const int32_t rr = static_cast<int32_t>(oaddr & 0x3Fu) - sp_row_lower;
  const int32_t rc = static_cast<int32_t>(oaddr >> 6) - sp_col_lower;
  if (rr >= 0 && rr <= 3 && rc >= 0 && rc <= 4) {
    const uint32_t osp = other & 0xFFu;
    const uint32_t bits = ((osp & 0x0Fu) << (4 * rr)) | ((osp & 0xF0u) << (12 + 4 * rr));
    w.pa0 |= rc == 0 ? bits : 0u;
    w.pa1 |= rc == 1 ? bits : 0u;
    w.pa2 |= rc == 2 ? bits : 0u;
    w.pa3 |= rc == 3 ? bits : 0u;
    w.pa4 |= rc == 4 ? bits : 0u;
  }
}

__device__ __forceinline__ bool masked_cluster_final(
  uint32_t sp_word,
  uint32_t sensor_number,
  uint32_t starting_pixel_location,
  const Window& pa,
  ClusterSeed* out)
{
  const uint32_t sp_addr = (sp_word & 0x007FFF00u) >> 8;
  const int32_t sp_row = sp_addr & 0x3Fu;
  const int32_t sp_col = sp_addr >> 6;
  const int32_t row_lower_limit = (sp_row - 2) * 4;
  const int32_t col_lower_limit = (sp_col - 3) * 2;
  const uint32_t rel_row = starting_pixel_location & 0x3u;
  const uint32_t rel_col = starting_pixel_location < 4;
  const uint32_t col = sp_col * 2 + rel_col;
  const uint64_t starting_pixel = ((uint64_t)(0x01u << (11 - rel_row)) << (16 * (col & 0x01))) << 32;
  const uint64_t pixel_map = (((uint64_t) pa.pa3) << 32) | pa.pa2;
  const Grown cl = grow_cluster(pixel_map, starting_pixel, col_lower_limit + 4, row_lower_limit);
  const uint64_t precedence = (mask_east(cl.pixels) & pa.pa4) | (cl.pixels & (starting_pixel ^ (0ull - starting_pixel)));
  bool keep = precedence == 0 && !(cl.pixels & 0x8000800080008000ull) && !(cl.pixels & 0x0001000100010001ull);
  if (!keep) return false;
  unsigned x = cl.x, y = cl.y, n = cl.n;
  if (cl.pixels & 0xFFFFull) {
    const uint64_t west_map = (((uint64_t) pa.pa1) << 32) | pa.pa0;
    const uint64_t west_start = mask_west(cl.pixels) & west_map;
    const Grown ext = grow_cluster(west_map, west_start, col_lower_limit, row_lower_limit);
    x += ext.x;
    y += ext.y;
    n += ext.n;
    keep = !(ext.pixels & 0x8000800080008000ull) && !(ext.pixels & 0xFFFFull);
  }
  if (!keep) return false;
  // Their integer parts are the quotients of the integers: n is at most 128 pixels and a quotient below
  // 2^10, so one that is no integer lies at least 2^-7 from one, and rounding moves it by 2^-14 at most.
  const float qx = x / static_cast<float>(n), qy = y / static_cast<float>(n);
  const unsigned cx = static_cast<unsigned>(qx);
  const unsigned cy = static_cast<unsigned>(qy);
  const float fx = qx - cx;
  const float fy = qy - cy;
  *out = ClusterSeed {lhcb_id_of(sensor_number, cx >> 8, cx & 0xFFu, cy), fx, fy};
  return true;
}

// The whole of rest_of_clusters for the SP at `sp_index` of a bank whose words are `words`.
template<int version>
__device__ __forceinline__ bool masked_cluster(
  const uint32_t* words,
  unsigned n_sp,
  unsigned sp_index,
  uint32_t sensor_number,
  uint32_t starting_pixel_location,
  ClusterSeed* out)
{
  const uint32_t sp_word = words[sp_index];
  const uint32_t sp_addr = (sp_word & 0x007FFF00u) >> 8;
  const int32_t sp_row_lower = static_cast<int32_t>(sp_addr & 0x3Fu) - 2;
  const int32_t sp_col_lower = static_cast<int32_t>(sp_addr >> 6) - 3;
  Window w {0, 0, 0, 0, 0};
  for (unsigned k = 0; k < n_sp; ++k) window_acc<version>(sp_row_lower, sp_col_lower, sensor_number, words[k], w);
  return masked_cluster_final(sp_word, sensor_number, starting_pixel_location, w, out);
}

__device__ __forceinline__ void store_cluster(const Clusters& c, unsigned i, const ClusterOut& o)
{
  c.ids()[i] = o.id;
  c.xyz()[3 * (size_t) i] = o.x;
  c.xyz()[3 * (size_t) i + 1] = o.y;
  c.xyz()[3 * (size_t) i + 2] = o.z;
  c.phis()[i] = o.phi;
}

// ---------------------------------------------------------------------------------------
// K1: one wave per event sums the SP words of its VELO banks.
template<int version>
__global__ void k_number_of_candidates(
  const char* raw,
  const uint32_t* offsets,
  const uint32_t* sizes,
  const uint32_t* types,
  unsigned mep,
  const uint32_t* event_list,
  unsigned n_list,
  unsigned event_start,
  uint32_t* number_of_candidates)
{
  const unsigned waves = blockDim.x / wave_size;
  const unsigned ev_idx = blockIdx.x * waves + threadIdx.x / wave_size;
  if (ev_idx >= n_list) return;
  const unsigned event_number = event_list ? event_list[ev_idx] : ev_idx;
  const RawEvent ev(raw, offsets, sizes, types, mep, event_number + event_start);
  uint32_t n = 0;
  for (unsigned b = lane_id(); b < ev.n_banks; b += wave_size) {
    const RawBank bank = raw_bank<version>(ev, b);
    if (is_velo_bank(bank.type)) n += bank_n_sp<version>(bank);
  }
#pragma unroll
  for (unsigned d = 32; d > 0; d >>= 1) n += __shfl_xor(n, d, wave_size);
  if (lane_id() == 0) number_of_candidates[event_number] = 2 * n;
}

// dev_velo_bank_index as the CPU target leaves it: events of CPU block 0 (ev_idx = 0, G, 2G, ...)
// write in order and the last write of each entry wins. Walk those events backwards and keep the
// first value seen per entry; stop once every sensor has one.
struct BankIndexShared {
  int best[n_sensors];
  uint8_t written[n_sensors];
  unsigned n_written;
};
template<int version>
__device__ __forceinline__ void bank_index_block(
  const char* raw,
  const uint32_t* offsets,
  const uint32_t* sizes,
  const uint32_t* types,
  unsigned mep,
  const uint32_t* event_list,
  unsigned n_list,
  unsigned event_start,
  unsigned cpu_grid,
  uint32_t* bank_index,
  BankIndexShared& sh)
{
  int(&best)[n_sensors] = sh.best;
  uint8_t(&written)[n_sensors] = sh.written;
  unsigned& n_written = sh.n_written;
  for (unsigned i = threadIdx.x; i < n_sensors; i += blockDim.x) written[i] = 0;
  if (threadIdx.x == 0) n_written = 0;
  __syncthreads();
  if (n_list == 0) return;
  const unsigned last = ((n_list - 1) / cpu_grid) * cpu_grid;
  for (int ev_idx = last; ev_idx >= 0; ev_idx -= cpu_grid) {
    for (unsigned i = threadIdx.x; i < n_sensors; i += blockDim.x) best[i] = -1;
    __syncthreads();
    const unsigned event_number = event_list ? event_list[ev_idx] : ev_idx;
    const RawEvent ev(raw, offsets, sizes, types, mep, event_number + event_start);
    for (unsigned b = threadIdx.x; b < ev.n_banks; b += blockDim.x) {
      const RawBank bank = raw_bank<version>(ev, b);
      const uint32_t pair = bank.sourceID & 0x1FFu;
      // Entries beyond the 208 sensors would be written out of bounds by the reference;
      // they are skipped here.
      if constexpr (version > 3) {
        if ((pair << 1) < n_sensors) atomicMax(&best[pair << 1], (int) b);
        if (((pair << 1) | 1u) < n_sensors) atomicMax(&best[(pair << 1) | 1u], (int) b);
      }
      else {
        if (pair < n_sensors) atomicMax(&best[pair], (int) b);
      }
    }
    __syncthreads();
    for (unsigned i = threadIdx.x; i < n_sensors; i += blockDim.x) {
      if (best[i] >= 0 && !written[i]) {
        bank_index[i] = best[i];
        written[i] = 1;
        atomicAdd(&n_written, 1u);
      }
    }
    __syncthreads();
    if (n_written >= n_sensors) break;
  }
}

template<int version>
__global__ void k_bank_index(
  const char* raw,
  const uint32_t* offsets,
  const uint32_t* sizes,
  const uint32_t* types,
  unsigned mep,
  const uint32_t* event_list,
  unsigned n_list,
  unsigned event_start,
  unsigned cpu_grid,
  uint32_t* bank_index)
{
  __shared__ BankIndexShared sh;
  bank_index_block<version>(raw, offsets, sizes, types, mep, event_list, n_list, event_start, cpu_grid, bank_index, sh);
}

// Bank directory of the whole-sequence path: one wave per event reads the bank headers once
// and writes, per (event, module pair), the module pair's banks in bank order (at most 8) as
// {first SP word (index into the raw buffer in 32-bit words), SP words, sourceID}, plus their
// number. Also writes dev_number_of_candidates (2 x SP words of the VELO banks), what later
// launches of the run start from, and (the last workgroup) dev_velo_bank_index.
template<int version>
__global__ void k_bank_directory(
  const char* raw,
  const uint32_t* offsets,
  const uint32_t* sizes,
  const uint32_t* types,
  unsigned mep,
  unsigned n_events,
  uint32_t* number_of_candidates,
  BankEntry* directory,
  uint32_t* directory_count,
  uint32_t* event_totals,
  uint32_t* number_of_events,
  uint32_t* status,
  unsigned cpu_grid,
  uint32_t* bank_index)
{
  if (blockIdx.x + 1 == gridDim.x) {
    __shared__ BankIndexShared sh;
    if (threadIdx.x == 0) {
      number_of_events[0] = n_events;
      status[0] = 0;
    }
    bank_index_block<version>(raw, offsets, sizes, types, mep, nullptr, n_events, 0, cpu_grid, bank_index, sh);
    return;
  }
  constexpr bool v23 = (version == 2 || version == 3);
  const unsigned waves = blockDim.x / wave_size;
  const unsigned e = blockIdx.x * waves + threadIdx.x / wave_size;
  if (e >= n_events) return;
  const RawEvent ev(raw, offsets, sizes, types, mep, e);
  uint32_t total = 0;
  unsigned my_count = 0; // lane m: banks of module pair m so far
  for (unsigned base = 0; base < ev.n_banks; base += wave_size) {
    const unsigned b = base + lane_id();
    unsigned mp = n_module_pairs;
    RawBank bank;
    if (b < ev.n_banks) {
      bank = raw_bank<version>(ev, b);
      if (is_velo_bank(bank.type)) {
        total += bank_n_sp<version>(bank);
        const uint32_t pair = bank.sourceID & 0x1FFu;
        mp = v23 ? pair / 8 : (pair << 1) / 8;
      }
    }
    // One round per module pair present in this chunk: its banks take the next ranks in bank
    // order (lane order within the chunk).
    for (uint64_t todo = __ballot(mp < n_module_pairs); todo;) {
      const unsigned m = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(mp), __ffsll(static_cast<unsigned long long>(todo)) - 1));
      const uint64_t bal = __ballot(mp == m);
      const unsigned before = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(my_count), static_cast<int>(m)));
      if (mp == m) {
        const unsigned rank = before + __popcll(bal & lanes_below_mask());
        if (rank < max_banks_per_mp) {
          BankEntry en;
          en.word_offset = static_cast<uint32_t>((reinterpret_cast<const char*>(bank.word) - raw) / 4);
          en.n_sp = bank_n_sp<version>(bank);
          en.source = bank.sourceID;
          en.pad = 0;
          directory[(static_cast<size_t>(e) * n_module_pairs + m) * max_banks_per_mp + rank] = en;
        }
      }
      if (lane_id() == m) my_count += __popcll(bal);
      todo &= ~bal;
    }
  }
#pragma unroll
  for (unsigned d = 32; d > 0; d >>= 1) total += __shfl_xor(total, d, wave_size);
  if (lane_id() < n_module_pairs) directory_count[e * n_module_pairs + lane_id()] = min(my_count, max_banks_per_mp);
  if (lane_id() == 0) {
    number_of_candidates[e] = 2 * total;
    event_totals[e] = 0;
  }
}

// Banks of an event as one wave sees them: lane l holds the header of its l-th bank, so the
// dependent reads of the headers (offset, source, count) take one round trip each for up to 64
// banks, not for every bank.
struct BankHeader {
  uint32_t pair, n_sp;
  const uint32_t* word;
  bool velo;
};
template<int version>
__device__ __forceinline__ BankHeader bank_header(const RawEvent& ev, unsigned b)
{
  BankHeader h {0, 0, nullptr, false};
  if (b < ev.n_banks) {
    const RawBank bank = raw_bank<version>(ev, b);
    h.velo = is_velo_bank(bank.type);
    h.pair = bank.sourceID & 0x1FFu;
    h.n_sp = bank_n_sp<version>(bank);
    h.word = bank.word;
  }
  return h;
}
__device__ __forceinline__ BankHeader lane_header(const BankHeader& h, unsigned lane)
{
  const uint64_t p = reinterpret_cast<uint64_t>(h.word);
  BankHeader r;
  r.pair = __builtin_amdgcn_readlane(h.pair, lane);
  r.n_sp = __builtin_amdgcn_readlane(h.n_sp, lane);
  r.word = reinterpret_cast<const uint32_t*>(
    static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<uint32_t>(p), lane))) |
    static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<uint32_t>(p >> 32), lane))) << 32);
  r.velo = __builtin_amdgcn_readlane(h.velo, lane) != 0;
  return r;
}

// Pixels that the words held by the wave's lanes (n of them, lane k the k-th) add to each lane's
// neighbourhood: what Neighbours does with every word, from a difference of SP addresses
// (column << 6 | row). The word is the same in all lanes, so taking it apart is scalar work and
// costs the lanes 16 instructions a word. The pixels of the row above or below a lane at the edge
// of its column, which the difference takes from the next column, are masked out at the end.
__device__ __forceinline__ uint32_t neighbours_of_lanes(uint32_t words, unsigned n, uint32_t sp_addr)
{
  uint32_t pixels = 0;
  for (unsigned k = 0; k < n; ++k) {
    const uint32_t other = __builtin_amdgcn_readlane(words, k);
    const uint32_t osp = other & 0xFFu;
    const uint32_t d = ((other & 0x007FFF00u) >> 8) - sp_addr;
    pixels |= d == 1u ? (osp & 0x01) << 4 | (osp & 0x10) << 6 : 0u;
    pixels |= d == 65u ? (osp & 0x01) << 16 : 0u;
    pixels |= d == 64u ? (osp & 0x0F) << 12 : 0u;
    pixels |= d == 63u ? (osp & 0x08) << 8 : 0u;
    pixels |= d == 0xFFFFFFFFu ? (osp & 0x80) >> 2 : 0u;
  }
  const uint32_t row = sp_addr & 0x3Fu;
  if (row == 63u) pixels &= ~((1u << 4) | (1u << 10) | (1u << 16));
  if (row == 0u) pixels &= ~((1u << 11) | (1u << 5));
  return pixels;
}

// K2: one workgroup per event; wave w takes banks w, w+W, ...; lanes take SP words. Bound by the
// latency of a bank (its words, then the scan over them): 16 waves share an event's 104 or 208
// banks, and the words a lane is compared with come from the other lanes' registers instead of
// memory. 500 pile-up events: 118 us, 410 us before.
constexpr unsigned estimate_block = 1024;
template<int version>
__global__ void __launch_bounds__(estimate_block) k_estimate_input_size(
  const char* raw,
  const uint32_t* offsets,
  const uint32_t* sizes,
  const uint32_t* types,
  unsigned mep,
  const uint32_t* event_list,
  unsigned event_start,
  const uint32_t* candidates_offsets,
  uint32_t* estimated_input_size,
  uint32_t* module_candidate_num,
  uint32_t* cluster_candidates)
{
  __shared__ uint32_t est[n_module_pairs];
  __shared__ uint32_t n_cand;
  const unsigned event_number = event_list ? event_list[blockIdx.x] : blockIdx.x;
  for (unsigned i = threadIdx.x; i < n_module_pairs; i += blockDim.x) est[i] = 0;
  if (threadIdx.x == 0) n_cand = 0;
  __syncthreads();
  uint32_t* cands = cluster_candidates + candidates_offsets[event_number];
  const RawEvent ev(raw, offsets, sizes, types, mep, event_number + event_start);
  const unsigned waves = blockDim.x / wave_size, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / wave_size);
  const unsigned l = lane_id();
  for (unsigned b0 = wave; b0 < ev.n_banks; b0 += waves * wave_size) {
    const BankHeader headers = bank_header<version>(ev, b0 + waves * l);
    const unsigned n_mine = min(wave_size, (ev.n_banks - b0 + waves - 1) / waves);
    for (unsigned i = 0; i < n_mine; ++i) {
      const BankHeader bank = lane_header(headers, i);
      const unsigned mp = (version == 2 || version == 3) ? bank.pair / 8 : (bank.pair << 1) / 8;
      if (!bank.velo || mp >= n_module_pairs) continue; // mp: a sourceID outside the 208 sensors
      uint32_t count = 0;
      for (unsigned s0 = 0; s0 < bank.n_sp; s0 += wave_size) {
        const unsigned s = s0 + l;
        const uint32_t w = s < bank.n_sp ? bank.word[s] : 0x80000000u;
        const bool isolated = w & 0x80000000u;
        const uint32_t sp_addr = (w & 0x007FFF00u) >> 8;
        unsigned m = 0, p0 = 0, p1 = 0;
        if (__ballot(!isolated)) {
          uint32_t pixels = neighbourhood_init(w);
          for (unsigned t0 = 0; t0 < bank.n_sp; t0 += wave_size) {
            const uint32_t others = t0 == s0 ? w : t0 + l < bank.n_sp ? bank.word[t0 + l] : 0u;
            pixels |= neighbours_of_lanes(others, min(wave_size, bank.n_sp - t0), sp_addr);
          }
          if (!isolated) m = candidates_final(pixels, &p0, &p1);
        }
        const uint64_t b0s = __ballot(m & 1), b1s = __ballot(m & 2);
        const unsigned n_new = __popcll(b0s) + __popcll(b1s);
        if (n_new) {
          uint32_t slot = 0;
          if (l == 0) slot = atomicAdd(&n_cand, n_new);
          slot = __builtin_amdgcn_readfirstlane(slot) + rank_below(b0s) + rank_below(b1s);
          const uint32_t sensor_number =
            (version == 2 || version == 3) ? bank.pair : ((bank.pair << 1) | ((w >> 23) & 0x1u));
          if (m & 1) cands[slot++] = (s << 11) | (sensor_number << 3) | p0;
          if (m & 2) cands[slot] = (s << 11) | (sensor_number << 3) | p1;
        }
        const bool one = isolated && s < bank.n_sp;
        count += n_new + __popcll(__ballot(one)) + __popcll(__ballot(one && isolated_cluster_count(w & 0xFFu) == 2));
      }
      if (l == 0 && count) atomicAdd(&est[mp], count);
    }
  }
  __syncthreads();
  for (unsigned i = threadIdx.x; i < n_module_pairs; i += blockDim.x)
    estimated_input_size[event_number * n_module_pairs + i] = est[i];
  if (threadIdx.x == 0) module_candidate_num[event_number] = n_cand;
}

// K3: one workgroup per event. Phase 1 takes isolated SPs of all banks, phase 2 the candidates. Bound by
// the latency of a wave's banks and candidates one after the other, so up to 512 events, which are all in
// flight, get 16 waves each (500 pile-up events: 70 us; 78 with 8 waves, 124 with 4, 117 before).
// With more of them waves that wait for their event's last ones are lost to other events: 8 waves up to
// 2048 events, or beyond for crowded ones (2000 one-vertex events: 125 us; 183 with 16, 143
// with 4 and before; 5000 at nu = 30: 1406, 1749, 1625 and 1566), else 4 (10 000 one-vertex events: 532 us;
// 915 with 16, 586 with 8, 535 before).
constexpr unsigned max_masked_block = 1024;
static unsigned masked_block(unsigned n_events, unsigned mean_hits)
{
  if (n_events <= 512) return max_masked_block;
  return n_events <= 2048 || mean_hits > crowded_hits ? 512 : 256;
}
template<int version>
__global__ void __launch_bounds__(max_masked_block) k_masked_clustering(
  const char* raw,
  const uint32_t* offsets,
  const uint32_t* sizes,
  const uint32_t* types,
  unsigned mep,
  const uint32_t* event_list,
  unsigned event_start,
  const uint32_t* number_of_events,
  const uint32_t* offsets_estimated_input_size,
  const uint32_t* module_candidate_num,
  const uint32_t* cluster_candidates,
  const uint32_t* candidates_offsets,
  const uint32_t* bank_index,
  const Geometry* geometry,
  const uint8_t* sp_patterns,
  const float* sp_fx,
  const float* sp_fy,
  uint32_t* module_cluster_num,
  char* cluster_container)
{
  __shared__ uint32_t count[n_module_pairs];
  const unsigned event_number = event_list ? event_list[blockIdx.x] : blockIdx.x;
  const unsigned n_events = number_of_events[0];
  const Clusters clusters {cluster_container, offsets_estimated_input_size[n_module_pairs * n_events]};
  const uint32_t* mp_start = offsets_estimated_input_size + event_number * n_module_pairs;
  for (unsigned i = threadIdx.x; i < n_module_pairs; i += blockDim.x) count[i] = 0;
  __syncthreads();
  const Geometry& g = *geometry;
  const RawEvent ev(raw, offsets, sizes, types, mep, event_number + event_start);
  const unsigned waves = blockDim.x / wave_size;
  for (unsigned b = threadIdx.x / wave_size; b < ev.n_banks; b += waves) {
    const RawBank bank = raw_bank<version>(ev, b);
    if (!is_velo_bank(bank.type)) continue;
    const unsigned n_sp = bank_n_sp<version>(bank);
    const uint32_t pair = bank.sourceID & 0x1FFu;
    const unsigned mp = (version == 2 || version == 3) ? pair / 8 : (pair << 1) / 8;
    if (mp >= n_module_pairs) continue;
    for (unsigned s = lane_id(); s < n_sp; s += wave_size) {
      const uint32_t w = bank.word[s];
      if (!(w & 0x80000000u)) continue;
      ClusterSeed s0, s1;
      const unsigned n = isolated_sp_clusters<version>(sp_patterns, sp_fx, sp_fy, bank.sourceID, w, s0, s1);
      const ClusterOut c0 = place_cluster(g, seed_sensor<version>(s0), s0);
      ClusterOut c1;
      if (n > 1) c1 = place_cluster(g, seed_sensor<version>(s1), s1);
      const unsigned slot = atomicAdd(&count[mp], n);
      const unsigned cap = mp_start[mp + 1] - mp_start[mp];
      if (slot < cap) store_cluster(clusters, mp_start[mp] + slot, c0);
      if (n > 1 && slot + 1 < cap) store_cluster(clusters, mp_start[mp] + slot + 1, c1);
    }
  }
  __syncthreads();
  const unsigned n_cand = module_candidate_num[event_number];
  const uint32_t* cands = cluster_candidates + candidates_offsets[event_number];
  for (unsigned i = threadIdx.x; i < n_cand; i += blockDim.x) {
    const uint32_t cand = cands[i];
    const uint32_t sensor_number = (cand >> 3) & 0xFFu;
    if (sensor_number >= n_sensors) continue;
    const RawBank bank = raw_bank<version>(ev, bank_index[sensor_number]);
    ClusterSeed c;
    if (masked_cluster<version>(bank.word, bank_n_sp<version>(bank), cand >> 11, sensor_number, cand & 7u, &c)) {
      const unsigned mp = sensor_number / 8;
      const unsigned slot = atomicAdd(&count[mp], 1u);
      const ClusterOut placed = place_cluster(g, sensor_number, c);
      if (mp < n_module_pairs && slot < mp_start[mp + 1] - mp_start[mp]) store_cluster(clusters, mp_start[mp] + slot, placed);
    }
  }
  __syncthreads();
  for (unsigned i = threadIdx.x; i < n_module_pairs; i += blockDim.x)
    module_cluster_num[event_number * n_module_pairs + i] = min(count[i], mp_start[i + 1] - mp_start[i]);
}

// (phi, id) as one unsigned 64-bit key: phi (signed) in the high word, offset to unsigned. Key
// order is the sort's (phi, id) order (SortByPhi.cu:90-125), and distinct clusters of a module
// pair have distinct ids, so the rank of a cluster is the number of keys below its own.
__device__ __forceinline__ uint64_t phi_id_key(int16_t phi, uint32_t id)
{
  return (static_cast<uint64_t>(static_cast<uint16_t>(phi) ^ 0x8000u) << 32) | id;
}

// K4: one wave per (module pair, event). A cluster's rank is the number of clusters in the phi buckets
// before its own and of those in its own with a smaller key, which it finds by their list; module pairs
// of more than sort_lds_cap clusters add up such ranks over tiles of them. Equal keys (a word twice
// in a bank) share a rank, and the slot they leave takes the container's first cluster, as the zero
// that its entry of the permutation holds says. 500 pile-up events: 11 us (37 with 256 lanes that
// compared every two); 600 events of up to 960 clusters a module pair: 117 us (617, and 1190 where one
// wave compared every two from memory).
constexpr unsigned sort_lds_cap = 512;
__global__ void __launch_bounds__(wave_size) k_sort_by_phi(
  const uint32_t* event_list,
  const uint32_t* number_of_events,
  const uint32_t* offsets_estimated_input_size,
  const uint32_t* module_cluster_num,
  const char* cluster_container,
  char* sorted_container,
  uint32_t* hit_permutation)
{
  constexpr unsigned none = 0xFFFFu; // ends a bucket's list
  __shared__ uint64_t s_key[sort_lds_cap];
  __shared__ uint16_t s_next[sort_lds_cap];
  __shared__ uint8_t s_taken[sort_lds_cap];
  __shared__ uint32_t s_newest[wave_size], s_before[wave_size];
  const unsigned mp = blockIdx.x, l = threadIdx.x;
  const unsigned event_number = event_list ? event_list[blockIdx.y] : blockIdx.y;
  const unsigned total = offsets_estimated_input_size[n_module_pairs * number_of_events[0]];
  const Clusters in {const_cast<char*>(cluster_container), total};
  const Clusters out {sorted_container, total};
  const unsigned start = offsets_estimated_input_size[event_number * n_module_pairs + mp];
  const unsigned n = module_cluster_num[event_number * n_module_pairs + mp];
  const auto key_of = [&](unsigned i) { return phi_id_key(in.phis()[start + i], in.ids()[start + i]); };
  // Clusters [t0, t0 + tn) to LDS, in lists by the bucket of their phi.
  const auto enter_tile = [&](unsigned t0, unsigned tn) {
    s_newest[l] = none;
    s_before[l] = 0;
    __syncthreads();
    for (unsigned i = l; i < tn; i += wave_size) {
      const uint64_t key = key_of(t0 + i);
      const unsigned bucket = static_cast<unsigned>(key >> 42);
      s_key[i] = key;
      s_taken[i] = 0;
      atomicAdd(&s_before[bucket], 1u);
      s_next[i] = static_cast<uint16_t>(atomicExch(&s_newest[bucket], i));
    }
    __syncthreads();
    const uint32_t count = s_before[l], before = wave_inclusive_scan(count) - count;
    __syncthreads();
    s_before[l] = before;
    __syncthreads();
  };
  // The tile's clusters below `key`.
  const auto below = [&](uint64_t key) {
    const unsigned bucket = static_cast<unsigned>(key >> 42);
    unsigned rank = s_before[bucket];
    for (unsigned j = s_newest[bucket]; j != none;) {
      const uint64_t other = s_key[j];
      j = s_next[j];
      rank += other < key;
    }
    return rank;
  };
  if (n <= sort_lds_cap) {
    enter_tile(0, n);
    const auto write = [&](size_t slot, size_t from, uint64_t key, float x, float y, float z) {
      hit_permutation[slot] = static_cast<uint32_t>(from);
      out.ids()[slot] = static_cast<uint32_t>(key);
      out.phis()[slot] = static_cast<int16_t>(static_cast<uint16_t>(key >> 32) ^ 0x8000u);
      out.xyz()[3 * slot] = x;
      out.xyz()[3 * slot + 1] = y;
      out.xyz()[3 * slot + 2] = z;
    };
    for (unsigned i = l; i < n; i += wave_size) {
      const float* xyz = in.xyz() + 3 * (size_t)(start + i);
      const float x = xyz[0], y = xyz[1], z = xyz[2];
      const uint64_t key = s_key[i];
      const unsigned rank = below(key);
      s_taken[rank] = 1;
      write(start + rank, start + i, key, x, y, z);
    }
    __syncthreads();
    for (unsigned i = l; i < n; i += wave_size)
      if (!s_taken[i]) write(start + i, 0, phi_id_key(in.phis()[0], in.ids()[0]), in.xyz()[0], in.xyz()[1], in.xyz()[2]);
    return;
  }
  // The sum over the tiles is kept where the sorted container will have an id.
  for (unsigned t0 = 0; t0 < n; t0 += sort_lds_cap) {
    const bool last = n - t0 <= sort_lds_cap;
    __syncthreads(); // the tile before has been read
    enter_tile(t0, min(sort_lds_cap, n - t0));
    for (unsigned i = l; i < n; i += wave_size) {
      const unsigned rank = (t0 ? out.ids()[start + i] : 0u) + below(key_of(i));
      if (last) hit_permutation[start + rank] = start + i;
      else out.ids()[start + i] = rank;
    }
  }
  __threadfence_block();
  __syncthreads();
  for (unsigned i = l; i < n; i += wave_size) {
    const unsigned src = hit_permutation[start + i];
    out.ids()[start + i] = in.ids()[src];
    out.phis()[start + i] = in.phis()[src];
    out.xyz()[3 * (size_t)(start + i)] = in.xyz()[3 * (size_t) src];
    out.xyz()[3 * (size_t)(start + i) + 1] = in.xyz()[3 * (size_t) src + 1];
    out.xyz()[3 * (size_t)(start + i) + 2] = in.xyz()[3 * (size_t) src + 2];
  }
}

// ---------------------------------------------------------------------------------------
// Host launchers.
template<int version>
static hipError_t launch_candidates_v(const CandidatesLaunch& a, hipStream_t s)
{
  const unsigned waves = 4;
  const unsigned grid = (a.n_list + waves - 1) / waves;
  const unsigned cpu_grid = (a.n_list + a.block_dim_x - 1) / a.block_dim_x;
  if (!grid) return hipSuccess;
  if (a.directory) {
    if (a.event_list || a.event_start || !a.event_totals || !a.number_of_events || !a.status) return hipErrorInvalidValue;
    hipLaunchKernelGGL(
      k_bank_directory<version>, dim3(grid + 1), dim3(waves * wave_size), 0, s, a.raw, a.offsets, a.sizes, a.types, unsigned(a.mep),
      a.n_list, a.number_of_candidates, static_cast<BankEntry*>(a.directory), a.directory_count, a.event_totals,
      a.number_of_events, a.status, cpu_grid, a.bank_index);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(
    k_number_of_candidates<version>, dim3(grid), dim3(waves * wave_size), 0, s, a.raw, a.offsets, a.sizes, a.types, unsigned(a.mep),
    a.event_list, a.n_list, a.event_start, a.number_of_candidates);
  hipLaunchKernelGGL(
    k_bank_index<version>, dim3(1), dim3(256), 0, s, a.raw, a.offsets, a.sizes, a.types, unsigned(a.mep), a.event_list, a.n_list,
    a.event_start, cpu_grid, a.bank_index);
  return hipGetLastError();
}

hipError_t launch_number_of_candidates(const CandidatesLaunch& a, hipStream_t s)
{
  switch (a.version) {
  case 2: return launch_candidates_v<2>(a, s);
  case 3: return launch_candidates_v<3>(a, s);
  default: return launch_candidates_v<4>(a, s);
  }
}

hipError_t launch_estimate_input_size(const EstimateLaunch& a, hipStream_t s)
{
  if (!a.n_list) return hipSuccess;
#define VELO_LAUNCH_EST(V)                                                                                          \
  hipLaunchKernelGGL(                                                                                               \
    k_estimate_input_size<V>, dim3(a.n_list), dim3(estimate_block), 0, s, a.raw, a.offsets, a.sizes, a.types, unsigned(a.mep), a.event_list,    \
    a.event_start, a.candidates_offsets, a.estimated_input_size, a.module_candidate_num, a.cluster_candidates)
  switch (a.version) {
  case 2: VELO_LAUNCH_EST(2); break;
  case 3: VELO_LAUNCH_EST(3); break;
  default: VELO_LAUNCH_EST(4); break;
  }
#undef VELO_LAUNCH_EST
  return hipGetLastError();
}

hipError_t launch_masked_clustering(const MaskedClusteringLaunch& a, hipStream_t s)
{
  if (!a.n_list) return hipSuccess;
#define VELO_LAUNCH_MC(V)                                                                                           \
  hipLaunchKernelGGL(                                                                                               \
    k_masked_clustering<V>, dim3(a.n_list), dim3(masked_block(a.n_list, a.mean_hits)), 0, s, a.raw, a.offsets, a.sizes, a.types, unsigned(a.mep), a.event_list,      \
    a.event_start, a.number_of_events, a.offsets_estimated_input_size, a.module_candidate_num, a.cluster_candidates, \
    a.candidates_offsets, a.bank_index, reinterpret_cast<const Geometry*>(a.geometry), a.sp_patterns, a.sp_fx,       \
    a.sp_fy, a.module_cluster_num, a.cluster_container)
  switch (a.version) {
  case 2: VELO_LAUNCH_MC(2); break;
  case 3: VELO_LAUNCH_MC(3); break;
  default: VELO_LAUNCH_MC(4); break;
  }
#undef VELO_LAUNCH_MC
  return hipGetLastError();
}

hipError_t launch_sort_by_phi(const SortLaunch& a, hipStream_t s)
{
  if (!a.n_list) return hipSuccess;
  hipLaunchKernelGGL(
    k_sort_by_phi, dim3(n_module_pairs, a.n_list), dim3(wave_size), 0, s, a.event_list, a.number_of_events,
    a.offsets_estimated_input_size, a.module_cluster_num, a.cluster_container, a.sorted_container, a.hit_permutation);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------------
// Whole-sequence clustering, one wave per (event, module pair), no block barriers.
//
//   k_estimate_mp   the K2 estimate of one module pair; also records, for every non-isolated
//                   SP word, its candidate pixels in one byte indexed by the word's position in
//                   the raw buffer (bit0/bit1: first/second candidate, bits 2-4 and 5-7: pixels)
//   k_cluster_mp    K3 + K4 of one module pair: isolated SPs through the pattern table, the
//                   recorded candidates through the masked clustering window (each bank's
//                   non-isolated words sorted by sensor, column and row, so a window reads one
//                   run of them), clusters appended with wave ballots, then ranked by (phi, id)
//                   and written sorted
//
// Each wave works in its own LDS slice; a module pair larger than the slice runs tile by tile.
// Two waves to a workgroup: a finished wave keeps its LDS until its workgroup ends, and module pairs
// differ (20 000 one-vertex events: 665 + 940 us with two, 692 + 978 with four, 660 + 941 with one).
namespace mp {
constexpr unsigned waves_per_block = 2;
constexpr unsigned hash_bits = 10;  // estimate: (bank, SP address) table of a module pair,
constexpr unsigned hash_slots = 1u << hash_bits; // more slots than words, so an empty slot ends every probe
constexpr unsigned table_words = 704; // most words that enter it
constexpr uint32_t hash_empty = 0xFFFFFFFFu; // an empty slot; keys have 18 bits, so no slot of a key is all ones
constexpr uint32_t hash_no_key = 0x01000000u; // a lookup key that matches no slot (nor an empty one)
constexpr unsigned hash_min_bank = 12; // largest bank (words) above which the table beats the scan (measured)
static_assert(hash_slots > table_words, "hash table load");

// Banks of one module pair (at most 8), kept in the wave's LDS slice while it is worked on in tiles.
// Bank k's words start at base + word_offset[k].
struct Banks {
  const uint32_t* base;
  unsigned n;
  uint32_t start[max_banks_per_mp + 1];
  uint32_t source[max_banks_per_mp];
  uint32_t word_offset[max_banks_per_mp];
  __device__ __forceinline__ const uint32_t* word(unsigned k) const { return base + word_offset[k]; }
};

__device__ __forceinline__ void wave_sync_lds()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The bank directory record of one (event, module pair) as this lane holds it: lanes 0-7 load
// one entry each, every lane the number of entries; both loads are issued together, without
// waiting, so a wave can fetch the next item's record while it works on the current one.
struct DirFetch {
  BankEntry en;
  unsigned nb;
};

__device__ __forceinline__ DirFetch fetch_dir(const BankEntry* directory, const uint32_t* directory_count, unsigned idx)
{
  DirFetch f;
  f.en = BankEntry {0, 0, 0, 0};
  const unsigned l = lane_id();
  if (l < max_banks_per_mp) f.en = directory[static_cast<size_t>(idx) * max_banks_per_mp + l];
  f.nb = min(directory_count[idx], max_banks_per_mp);
  return f;
}

// The banks of one module pair from its directory record.
__device__ __forceinline__ void load_banks(const char* raw, const DirFetch& f, Banks& B)
{
  const unsigned nb = f.nb;
  const unsigned l = lane_id();
  const BankEntry en = l < nb ? f.en : BankEntry {0, 0, 0, 0};
  const uint32_t inc = wave_inclusive_scan(l < nb ? en.n_sp : 0u);
  if (l < nb) {
    B.start[l] = inc - en.n_sp;
    B.source[l] = en.source;
    B.word_offset[l] = en.word_offset;
  }
  if (l == 0) {
    B.n = nb;
    B.base = reinterpret_cast<const uint32_t*>(raw);
  }
  if (l == nb) B.start[nb] = inc - (l < nb ? en.n_sp : 0u);
  wave_sync_lds();
}

// The bank holding position w of a list laid out bank after bank (starts[k]: bank k's first
// position): the starts are non-decreasing, so the last bank starting at or before w is the
// number of banks after the first that do (all starts read at once, one LDS round trip).
__device__ __forceinline__ unsigned bank_at(const uint32_t* starts, unsigned n, unsigned w)
{
  unsigned bi = 0;
#pragma unroll
  for (unsigned k = 1; k < max_banks_per_mp; ++k) bi += (k < n && starts[k] <= w) ? 1u : 0u;
  return bi;
}
__device__ __forceinline__ unsigned bank_of(const Banks& B, unsigned w) { return bank_at(B.start, B.n, w); }
} // namespace mp

namespace mp {
// Word `w` of the module pair (flattened over its banks), from global memory.
__device__ __forceinline__ uint32_t word_at(const Banks& B, unsigned w)
{
  const unsigned bi = bank_of(B, w);
  return B.word(bi)[w - B.start[bi]];
}

// Copies words [t0, t0 + n) of the module pair into the wave's LDS slice.
__device__ __forceinline__ void load_words(const Banks& B, unsigned t0, unsigned n, uint32_t* lw)
{
  wave_sync_lds();
  for (unsigned i = lane_id(); i < n; i += wave_size) lw[i] = word_at(B, t0 + i);
  wave_sync_lds();
}

// Calls f(word) for every word of the flattened range [lo, hi), tile by tile through the slice
// (wave-uniform tile loop, per-lane ranges; eight LDS reads in flight at a time).
template<typename F>
__device__ __forceinline__ void
for_words(const Banks& B, unsigned n_words, uint32_t* lw, unsigned tile, bool active, unsigned lo, unsigned hi, F&& f)
{
  for (unsigned t0 = 0; t0 < n_words; t0 += tile) {
    const unsigned tn = min(tile, n_words - t0);
    load_words(B, t0, tn, lw);
    if (!active) continue;
    unsigned k = max(lo, t0) - t0;
    const unsigned end = min(hi, t0 + tn) - t0;
    if (hi <= t0) continue;
    for (; k + 8 <= end; k += 8) {
      uint32_t v[8];
#pragma unroll
      for (unsigned u = 0; u < 8; ++u) v[u] = lw[k + u];
#pragma unroll
      for (unsigned u = 0; u < 8; ++u) f(v[u]);
    }
    for (; k < end; ++k) f(lw[k]);
  }
}

// Slot of a (bank, SP address) key in a table of 2^bits slots: multiplicative hashing.
__device__ __forceinline__ unsigned hash_slot(uint32_t key, unsigned bits) { return (key * 2654435761u) >> (32 - bits); }
} // namespace mp

// What one wave of k_estimate_mp holds in LDS: 5.5 KB, so that 28 waves fit a CU.
namespace mp {
struct alignas(16) EstimateLds {
  static constexpr unsigned word_cap = 336;
  uint32_t table[hash_slots];
  uint4 bank[max_banks_per_mp]; // word offset less the words before the bank, first word, end
  uint32_t words[word_cap];
  // A module pair that is worked on in tiles has its banks where the table would be.
  __device__ __forceinline__ Banks& banks() { return *reinterpret_cast<Banks*>(table); }
};
static_assert(max_banks_per_mp * hash_min_bank <= EstimateLds::word_cap, "words of small banks");
} // namespace mp

// K2 of one module pair (idx = event * 26 + module pair) by one wave. The neighbourhood of a
// non-isolated SP is what the reference collects by scanning every word of its bank: the SP
// bytes of the words at five neighbouring addresses, OR-ed (EstimateInputSize.cu:111-141). OR-ing is
// order-free and a word at another address adds nothing, so three ways give the same:
//  - banks that are all small: the scan, from LDS;
//  - larger ones: the words are first entered in a hash table keyed by (bank, SP address) whose
//    value is the OR of their SP bytes (one word per slot: key << 8 | value), and each SP looks its
//    five neighbours up. A scan costs a wave 17 instructions for each word of its largest bank, the
//    table about 200;
//  - more words than the table takes: the scan, tile by tile.
// Bound by VALU issue. 20 000 one-vertex events: 482 us (692 with 27 instructions for each word that is
// compared and module pairs of more than 384 words in tiles), 2000 stress events: 104 us (200).
// Scans of banks of up to 10, 16 and 24 words: 480, 486 and 520 us.
__device__ __forceinline__ void estimate_item(
  const char* raw,
  const mp::DirFetch& f,
  unsigned idx,
  mp::EstimateLds& L,
  uint32_t* estimated_input_size,
  uint32_t* event_totals,
  uint8_t* sp_flags)
{
  const unsigned l = lane_id();
  const unsigned n_sp = l < f.nb ? f.en.n_sp : 0u;
  const unsigned inc = wave_inclusive_scan(n_sp), first = inc - n_sp; // words before this lane's bank
  const unsigned n_words = __builtin_amdgcn_readlane(inc, max_banks_per_mp - 1);
  unsigned largest_bank = 0;
  for (unsigned k = 0; k < f.nb; ++k) largest_bank = max(largest_bank, static_cast<unsigned>(__builtin_amdgcn_readlane(n_sp, k)));
  const bool scan = largest_bank <= mp::hash_min_bank;
  const bool table = !scan && n_words <= mp::table_words;
  // Table of eight times as many slots as words, 256 to 1024: the wave waits for its longest probe,
  // so the probes must stay short everywhere.
  const unsigned bits = min(mp::hash_bits, max(8u, 32u - __clz(8 * n_words - 1)));
  const unsigned hmask = (1u << bits) - 1;
  const uint32_t* raw_words = reinterpret_cast<const uint32_t*>(raw);
  // The number of the bank holding word w: the banks after the first that start at or before it.
  auto bank_of = [&](unsigned w) {
    unsigned bi = 0;
    for (unsigned j = 1; j < f.nb; ++j) bi += w >= static_cast<unsigned>(__builtin_amdgcn_readlane(first, j));
    return bi;
  };
  mp::wave_sync_lds();
  if (l < f.nb) L.bank[l] = make_uint4(f.en.word_offset - first, first, inc, 0);
  if (table)
    for (unsigned h = 4 * l; h <= hmask; h += 4 * wave_size)
      *reinterpret_cast<uint4*>(L.table + h) = make_uint4(mp::hash_empty, mp::hash_empty, mp::hash_empty, mp::hash_empty);
  mp::wave_sync_lds();
  if (scan || table) {
    for (unsigned base = 0; base < n_words; base += wave_size) {
      const unsigned w = base + l;
      const unsigned bi = bank_of(w); // by the whole wave: it reads other lanes' registers
      if (w >= n_words) continue;
      const uint32_t word = raw_words[L.bank[bi].x + w];
      if (w < mp::EstimateLds::word_cap) L.words[w] = word;
      if (scan) continue;
      const uint32_t key = (bi << 15) | ((word & 0x007FFF00u) >> 8);
      for (unsigned h = mp::hash_slot(key, bits);; h = (h + 1) & hmask) {
        const uint32_t old = atomicCAS(&L.table[h], mp::hash_empty, (key << 8) | (word & 0xFFu));
        if (old == mp::hash_empty) break;
        if ((old >> 8) == key) {
          atomicOr(&L.table[h], word & 0xFFu);
          break;
        }
      }
    }
  }
  else mp::load_banks(raw, f, L.banks());
  mp::wave_sync_lds();
  uint32_t count = 0;
  for (unsigned base = 0; base < n_words; base += wave_size) {
    const unsigned w = base + l;
    const bool active = w < n_words;
    const unsigned bi = bank_of(w);
    const uint4 bank = L.bank[bi];
    uint32_t sp_word = 0;
    if (active) {
      if ((scan || table) && w < mp::EstimateLds::word_cap) sp_word = L.words[w];
      else sp_word = raw_words[bank.x + w];
    }
    const bool isolated = (sp_word & 0x80000000u) != 0, non = active && !isolated;
    const uint32_t sp_addr = (sp_word >> 8) & 0x7FFFu;
    Neighbours around(sp_addr);
    uint32_t pixels = neighbourhood_init(sp_word);
    if (table) {
      if (non) {
        // The five first probes are issued together, then the rare longer probes.
        const uint32_t kb = bi << 15;
        const uint32_t address[5] = {around.top, around.top_right, around.right, around.bot_right, around.bot};
        uint32_t key[5], got[5], v[5];
        unsigned h[5];
#pragma unroll
        for (unsigned k = 0; k < 5; ++k) {
          const bool valid = address[k] != 0xFFFFFFFFu;
          key[k] = valid ? (kb | address[k]) : mp::hash_no_key;
          h[k] = mp::hash_slot(key[k], bits);
          got[k] = valid ? L.table[h[k]] : mp::hash_empty;
        }
#pragma unroll
        for (unsigned k = 0; k < 5; ++k)
          while ((got[k] >> 8) != key[k] && got[k] != mp::hash_empty) {
            h[k] = (h[k] + 1) & hmask;
            got[k] = L.table[h[k]];
          }
#pragma unroll
        for (unsigned k = 0; k < 5; ++k) v[k] = (got[k] >> 8) == key[k] ? got[k] : 0u;
        around.column = (v[0] & 0x11u) | (v[3] & 0x08u) | (v[4] & 0x80u);
        around.corner = v[1] & 0x01u;
        around.side = v[2] & 0x0Fu;
      }
    }
    else if (scan) {
      if (non) // four words at a time; the last is taken again where fewer are left
        for (unsigned k = bank.y; k < bank.z; k += 4) {
          uint32_t v[4];
#pragma unroll
          for (unsigned u = 0; u < 4; ++u) v[u] = L.words[min(k + u, bank.z - 1)];
#pragma unroll
          for (unsigned u = 0; u < 4; ++u) around.add(v[u]);
        }
    }
    else {
      mp::for_words(L.banks(), n_words, L.words, mp::EstimateLds::word_cap, non, bank.y, bank.z,
                    [&](uint32_t other) { around.add(other); });
    }
    pixels |= around.pixels();
    unsigned clusters = 0;
    if (isolated) {
      clusters = isolated_cluster_count(sp_word & 0xFFu);
    }
    else if (active) {
      unsigned p0 = 0, p1 = 0;
      const unsigned mk = candidates_final(pixels, &p0, &p1);
      clusters = __popc(mk);
      sp_flags[bank.x + w] = static_cast<uint8_t>(mk | (p0 << 2) | (p1 << 5));
    }
    count += __popcll(__ballot(clusters > 0)) + __popcll(__ballot(clusters > 1)); // one or two a word
  }
  if (l == 0) {
    estimated_input_size[idx] = count;
    atomicAdd(event_totals + idx / n_module_pairs, count);
  }
}

// Resident grid: each wave takes items idx, idx + stride, ... and fetches the next item's
// bank directory record before working on the current one.
template<int version>
__global__ void __launch_bounds__(mp::waves_per_block* wave_size) k_estimate_mp(
  const char* raw,
  const BankEntry* directory,
  const uint32_t* directory_count,
  unsigned n_events,
  uint32_t* estimated_input_size,
  uint32_t* event_totals,
  uint8_t* sp_flags)
{
  __shared__ mp::EstimateLds s_lds[mp::waves_per_block];
  const unsigned wave = threadIdx.x / wave_size;
  const unsigned n_items = n_events * n_module_pairs;
  const unsigned stride = gridDim.x * mp::waves_per_block;
  unsigned idx = blockIdx.x * mp::waves_per_block + wave;
  if (idx >= n_items) return;
  mp::DirFetch cur = mp::fetch_dir(directory, directory_count, idx);
  for (; idx < n_items; idx += stride) {
    mp::DirFetch next = cur;
    if (idx + stride < n_items) next = mp::fetch_dir(directory, directory_count, idx + stride);
    estimate_item(raw, cur, idx, s_lds[wave], estimated_input_size, event_totals, sp_flags);
    cur = next;
  }
}

// What one wave of k_cluster_mp holds in LDS: 5.6 KB, so that 28 waves fit a CU.
namespace mp {
constexpr unsigned non_isolated_cap = 256; // non-isolated SP words of a module pair
constexpr unsigned cluster_cap = 192;      // its clusters; more of them go through global memory
// The ranking's memory for `cap` clusters: each phi bucket's newest cluster and their number, the keys,
// each cluster's successor in its bucket.
constexpr unsigned rank_bytes(unsigned cap) { return 2 * 4 * wave_size + 10 * cap; }
struct ClusterLds {
  // The non-isolated words (then the list of candidates), the sorted ones, and the sort's keys (then
  // the candidates' windows). Once the seeds are found, the ranking keys take this memory.
  static constexpr unsigned window_words = 5 * wave_size;
  uint64_t work[(2 * non_isolated_cap + window_words) / 2];
  float xyz[3 * cluster_cap];           // a seed's fx, fy and id, then the placed cluster's x, y, z
  uint2 bank[max_banks_per_mp];         // word offset less the words before the bank, source
  uint32_t non_start[max_banks_per_mp + 1]; // non-isolated words before each bank
  __device__ __forceinline__ uint32_t* words() { return reinterpret_cast<uint32_t*>(work); }
  __device__ __forceinline__ uint32_t* sorted() { return words() + non_isolated_cap; }
  __device__ __forceinline__ uint32_t* keys() { return words() + 2 * non_isolated_cap; }
  // A module pair that is worked on in tiles has its banks where the sort's keys would be.
  static constexpr unsigned tile = 2 * non_isolated_cap;
  __device__ __forceinline__ Banks& banks() { return *reinterpret_cast<Banks*>(keys()); }
  // Most clusters that are ranked with nothing else in the slice, and in tiles of keys alone.
  static constexpr unsigned rank_cap = (4 * (2 * non_isolated_cap + window_words + 3 * cluster_cap) - rank_bytes(0)) / 10;
  static constexpr unsigned key_tile = (2 * non_isolated_cap + window_words + 3 * cluster_cap) / 2;
};
static_assert(non_isolated_cap <= ClusterLds::window_words && non_isolated_cap <= 256, "sort keys");
static_assert(sizeof(ClusterLds::work) >= rank_bytes(cluster_cap) && cluster_cap % 2 == 0, "ranking");
static_assert(sizeof(Banks) <= 4 * ClusterLds::window_words && non_isolated_cap % 2 == 0, "banks");
static_assert(offsetof(ClusterLds, xyz) == sizeof(ClusterLds::work), "the ranking reaches into xyz");
} // namespace mp

// The number of keys[0 .. n) below `key` (eight reads in flight at a time).
__device__ __forceinline__ unsigned keys_below(const uint64_t* keys, unsigned n, uint64_t key)
{
  unsigned below = 0, j = 0;
  for (; j + 8 <= n; j += 8) {
    uint64_t v[8];
#pragma unroll
    for (unsigned u = 0; u < 8; ++u) v[u] = keys[j + u];
#pragma unroll
    for (unsigned u = 0; u < 8; ++u) below += v[u] < key;
  }
  for (; j < n; ++j) below += keys[j] < key;
  return below;
}

struct ClusterArgs {
  const char* raw;
  const BankEntry* directory;
  const uint32_t* directory_count;
  const uint32_t* offsets_estimated_input_size;
  const uint8_t* sp_flags;
  const Geometry* geometry;
  const uint8_t* sp_patterns;
  const float* sp_fx;
  const float* sp_fy;
  uint32_t* module_cluster_num;
  char* sorted_container;
  char* unsorted_scratch;
};

// K3 + K4 of one module pair (idx = event * 26 + module pair) by one wave.
//
// Every word is read once. An isolated word becomes one or two seeds through the pattern table; the
// non-isolated ones are kept, and sorted within their bank by (sensor, SP column, SP row) (v2/v3: the
// bank is the sensor, bit 23 cleared), each with its candidate byte in bits 24-31. A candidate's
// window then takes only the words of its bank and sensor in SP columns col - 3 .. col + 1, a run
// found by binary search, instead of every word of the bank; OR-ing the window is order-free, so the
// windows are the scan's. The candidates form one list and each lane grows one of them. The seeds of
// all words are placed together, so that the transform and phi run with full lanes, and ranked by
// (phi, id).
//
// Bound by VALU issue, and by the largest module pair where there are few events. 20 000 one-vertex
// events: 806 us (1155 with a sort of all words, windows in registers, each cluster placed where it was
// found and ranked against all others); 1000 pile-up events: 48 us (82); 8 of them: 14 us (27). Two
// module pairs to a wave, which fills the lanes better, needs more LDS and lost more by the fewer
// waves that then fit a CU: 1066 against 980 us.
template<int version>
struct ClusterItem {
  static constexpr bool v23 = (version == 2 || version == 3);
  const ClusterArgs& a;
  mp::ClusterLds& L;
  const unsigned total, idx, start, estimate;
  const bool in_lds;
  unsigned n = 0; // clusters so far
  static constexpr uint32_t none = 0xFFFFu; // ends a bucket's list

  __device__ __forceinline__ ClusterItem(const ClusterArgs& args, mp::ClusterLds& lds, unsigned total_clusters, unsigned item) :
    a(args), L(lds), total(total_clusters), idx(item), start(a.offsets_estimated_input_size[item]),
    estimate(a.offsets_estimated_input_size[item + 1] - start), in_lds(estimate <= mp::cluster_cap)
  {}

  __device__ __forceinline__ void keep_seed(unsigned slot, const ClusterSeed& s)
  {
    if (slot >= estimate) return;
    if (in_lds) {
      float* at = L.xyz + 3 * slot;
      at[0] = s.fx;
      at[1] = s.fy;
      at[2] = __uint_as_float(s.id);
    }
    else {
      const Clusters scratch {a.unsorted_scratch, total};
      const size_t at = start + slot;
      scratch.ids()[at] = s.id;
      scratch.xyz()[3 * at] = s.fx;
      scratch.xyz()[3 * at + 1] = s.fy;
    }
  }

  // Appends k (0, 1 or 2) seeds of each lane. The order in which they are appended does not reach the
  // output: the clusters are ranked by their distinct (phi, id) keys.
  __device__ __forceinline__ void emit(unsigned k, const ClusterSeed& s0, const ClusterSeed& s1)
  {
    const uint64_t one = __ballot(k > 0), two = __ballot(k > 1);
    const unsigned slot = n + rank_below(one) + rank_below(two);
    if (k > 0) keep_seed(slot, s0);
    if (k > 1) keep_seed(slot + 1, s1);
    n += __popcll(one) + __popcll(two);
  }

  // The module pair's seeds with its non-isolated words in the slice. False, with nothing written but
  // scratch, if they don't fit.
  __device__ __forceinline__ bool seeds(const mp::DirFetch& f)
  {
    constexpr uint32_t field = v23 ? 0x7FFFu : 0xFFFFu;
    const unsigned l = lane_id();
    const unsigned inc = wave_inclusive_scan(l < f.nb ? f.en.n_sp : 0u);
    const unsigned first = l < f.nb ? inc - f.en.n_sp : inc; // words before this lane's bank
    const unsigned n_words = __builtin_amdgcn_readlane(inc, max_banks_per_mp - 1);
    if (l < f.nb) L.bank[l] = make_uint2(f.en.word_offset - first, f.en.source);
    mp::wave_sync_lds();
    const uint32_t* raw_words = reinterpret_cast<const uint32_t*>(a.raw);
    uint32_t* words = L.words();
    uint32_t* sorted = L.sorted();
    uint32_t* keys = L.keys();
    unsigned n_non = 0, non_before = 0; // non_before: those before this lane's bank
    for (unsigned base = 0; base < n_words; base += wave_size) {
      const unsigned w = base + l;
      // The number of the bank holding word w: the banks after the first that start at or before it.
      unsigned bi = 0;
      for (unsigned j = 1; j < f.nb; ++j) bi += w >= static_cast<unsigned>(__builtin_amdgcn_readlane(first, j));
      const uint2 bank = L.bank[bi];
      const bool active = w < n_words;
      uint32_t word = 0, flags = 0;
      if (active) {
        word = raw_words[bank.x + w];
        flags = a.sp_flags[bank.x + w]; // written for non-isolated words
      }
      const bool isolated = active && (word & 0x80000000u), non = active && !isolated;
      ClusterSeed s0, s1;
      unsigned n_seeds = 0;
      if (isolated) n_seeds = isolated_sp_clusters<version>(a.sp_patterns, a.sp_fx, a.sp_fy, bank.y, word, s0, s1);
      emit(n_seeds, s0, s1);
      const uint64_t nons = __ballot(non);
      const unsigned slot = n_non + rank_below(nons);
      const unsigned to_bank = first > base ? min(first - base, wave_size) : 0u;
      non_before += __popcll(nons & (to_bank >= wave_size ? ~0ull : (1ull << to_bank) - 1));
      n_non += __popcll(nons);
      if (n_non > mp::non_isolated_cap) return false;
      if (non) {
        // Distinct for distinct words: bank, sensor, column and row, then the slot.
        keys[slot] = (bi << 24) | (((word >> 8) & field) << 8) | slot;
        words[slot] = (word & (v23 ? 0x007FFFFFu : 0x00FFFFFFu)) | (flags << 24);
      }
    }
    if (l < f.nb) L.non_start[l] = non_before;
    if (l == f.nb) L.non_start[l] = n_non;
    mp::wave_sync_lds(); // keys and words written
    // Ranks within the bank; the candidates of the sorted words, as (word, bank, which). The list
    // takes the place of the words: 64 (r + 1) of these have been read after round r, and the list
    // holds at most 128 (r + 1) entries of half a word.
    uint16_t* candidates = reinterpret_cast<uint16_t*>(words);
    unsigned n_cand = 0;
    for (unsigned base = 0; base < n_non; base += wave_size) {
      const unsigned slot = base + l;
      unsigned at = 0;
      uint32_t word = 0;
      if (slot < n_non) {
        const uint32_t key = keys[slot];
        word = words[slot];
        const unsigned bi = key >> 24;
        const unsigned from = L.non_start[bi], to = L.non_start[bi + 1];
        unsigned rank = 0, j = from;
        for (; j + 4 <= to; j += 4) {
          uint32_t v[4];
#pragma unroll
          for (unsigned u = 0; u < 4; ++u) v[u] = keys[j + u];
#pragma unroll
          for (unsigned u = 0; u < 4; ++u) rank += v[u] < key ? 1u : 0u;
        }
        for (; j < to; ++j) rank += keys[j] < key ? 1u : 0u;
        at = (from + rank) | (bi << 8);
        sorted[from + rank] = word;
      }
      const uint64_t firsts = __ballot(word & (1u << 24)), seconds = __ballot(word & (2u << 24));
      unsigned c = n_cand + rank_below(firsts) + rank_below(seconds);
      n_cand += __popcll(firsts) + __popcll(seconds);
      mp::wave_sync_lds(); // this round's words have been read
      if (word & (1u << 24)) candidates[c++] = static_cast<uint16_t>(at);
      if (word & (2u << 24)) candidates[c] = static_cast<uint16_t>(at | 0x1000u);
    }
    mp::wave_sync_lds(); // the list and the sorted words written; the keys are free
    uint32_t* window = keys + l; // SP column c of this lane's window at [64 c]
    for (unsigned base = 0; base < n_cand; base += wave_size) {
      bool keep = false;
      ClusterSeed s, unused;
      if (base + l < n_cand) {
        const unsigned e = candidates[base + l];
        const unsigned bi = (e >> 8) & 7u, at = e & 255u;
        const uint32_t word = sorted[at];
        const unsigned end = L.non_start[bi + 1];
        unsigned lo = L.non_start[bi], hi = at;
        const uint32_t pair = L.bank[bi].y & 0x1FFu;
#pragma unroll
        for (unsigned c = 0; c < 5; ++c) window[wave_size * c] = 0;
        const uint32_t key = (word >> 8) & 0xFFFFu;
        const uint32_t sensor = key & 0x8000u;
        const uint32_t col = (key >> 6) & 0x1FFu;
        const uint32_t lower = sensor | ((max(col, 3u) - 3u) << 6);
        const uint32_t upper = sensor + min((col + 2u) << 6, 0x8000u);
        while (lo < hi) { // the first word at or above `lower`; the candidate's own is
          const unsigned mid = (lo + hi) >> 1;
          if (((sorted[mid] >> 8) & 0xFFFFu) < lower) lo = mid + 1;
          else hi = mid;
        }
        const uint32_t row_lower = (key & 0x3Fu) - 2u, col_lower = (key >> 6) - 3u;
        for (unsigned j = lo; j < end; ++j) {
          const uint32_t o = sorted[j];
          const uint32_t address = (o >> 8) & 0xFFFFu;
          if (address >= upper) break;
          const uint32_t row = (address & 0x3Fu) - row_lower;
          // Four rows of two pixel columns, 16 bits apart, into the word's SP column: an LDS OR each
          // costs the VALU half of what selecting one of five registers does.
          if (row < 4u)
            atomicOr(window + wave_size * ((address >> 6) - col_lower),
                     ((o & 0x0Fu) | ((o & 0xF0u) << 12)) << (4 * row));
        }
        const Window win {window[0], window[wave_size], window[2 * wave_size], window[3 * wave_size], window[4 * wave_size]};
        keep = masked_cluster_final(word & 0x00FFFFFFu, v23 ? pair : ((pair << 1) | (sensor >> 15)),
                                    (e & 0x1000u) ? word >> 29 : (word >> 26) & 7u, win, &s);
      }
      emit(keep ? 1u : 0u, s, unused);
    }
    return true;
  }

  // The seeds of a module pair with too many words for the slice: every word in place by its
  // isolated bit, and every SP with candidates scans its bank, tile by tile through the slice.
  __device__ __forceinline__ void seeds_in_tiles(const mp::DirFetch& f)
  {
    n = 0;
    mp::Banks& B = L.banks();
    mp::wave_sync_lds();
    mp::load_banks(a.raw, f, B);
    const unsigned n_words = B.start[B.n];
    for (unsigned base = 0; base < n_words; base += wave_size) {
      const unsigned w = base + lane_id();
      const bool active = w < n_words;
      const unsigned bi = active ? mp::bank_of(B, w) : 0;
      const size_t at = active ? B.word_offset[bi] + (w - B.start[bi]) : 0;
      const uint32_t sp_word = active ? B.base[at] : 0x80000000u;
      uint32_t flags = 0;
      ClusterSeed s0, s1;
      unsigned k = 0;
      if (active) {
        if (sp_word & 0x80000000u)
          k = isolated_sp_clusters<version>(a.sp_patterns, a.sp_fx, a.sp_fy, B.source[bi], sp_word, s0, s1);
        else flags = a.sp_flags[at];
      }
      emit(k, s0, s1);
      const uint32_t pair = B.source[bi] & 0x1FFu;
      const uint32_t sensor_number = v23 ? pair : ((pair << 1) | ((sp_word >> 23) & 0x1u));
      const uint32_t sp_addr = (sp_word & 0x007FFF00u) >> 8;
      const int32_t sp_row_lower = static_cast<int32_t>(sp_addr & 0x3Fu) - 2;
      const int32_t sp_col_lower = static_cast<int32_t>(sp_addr >> 6) - 3;
      Window win {0, 0, 0, 0, 0};
      // Both candidates of an SP share its window.
      mp::for_words(B, n_words, L.words(), mp::ClusterLds::tile, (flags & 3) != 0, B.start[bi], B.start[bi + 1],
                    [&](uint32_t other) { window_acc<version>(sp_row_lower, sp_col_lower, sensor_number, other, win); });
#pragma nounroll
      for (unsigned which = 0; which < 2; ++which) {
        const bool candidate = (flags >> which) & 1u;
        const bool keep = candidate && masked_cluster_final(
                                         sp_word & 0x00FFFFFFu, sensor_number, (flags >> (2 + 3 * which)) & 7u, win, &s0);
        emit(keep ? 1u : 0u, s0, s1);
      }
    }
  }

  // Places the seeds and writes them in the order of their keys.
  __device__ __forceinline__ void finish()
  {
    const Clusters out {a.sorted_container, total};
    n = min(n, estimate);
    if (lane_id() == 0) a.module_cluster_num[idx] = n;
    mp::wave_sync_lds(); // seeds written, windows read
    if (n <= mp::ClusterLds::rank_cap) {
      // 64 buckets of phi: a cluster's rank is the number of clusters in the buckets before its own and
      // of those in its own with a smaller key, which it finds by their list. Against every key it
      // would be n comparisons of 64 bits: 228 clusters took 13 us, four rounds over all keys.
      const unsigned l = lane_id();
      const unsigned cap = in_lds ? mp::cluster_cap : mp::ClusterLds::rank_cap;
      uint32_t* newest = L.words();
      uint32_t* counts = newest + wave_size;
      uint64_t* keys = L.work + wave_size;
      uint16_t* next = reinterpret_cast<uint16_t*>(keys + cap);
      const Clusters scratch {a.unsorted_scratch, total};
      newest[l] = none;
      counts[l] = 0;
      if (!in_lds) __threadfence_block();
      mp::wave_sync_lds();
      for (unsigned i = l; i < n; i += wave_size) {
        float* at = in_lds ? L.xyz + 3 * i : nullptr;
        ClusterSeed s;
        if (in_lds) s = ClusterSeed {__float_as_uint(at[2]), at[0], at[1]};
        else s = ClusterSeed {scratch.ids()[start + i], scratch.xyz()[3 * (size_t)(start + i)], scratch.xyz()[3 * (size_t)(start + i) + 1]};
        const ClusterOut c = place_cluster(*a.geometry, seed_sensor<version>(s), s);
        const uint64_t key = phi_id_key(c.phi, c.id);
        const unsigned bucket = static_cast<unsigned>(key >> 42);
        keys[i] = key;
        atomicAdd(counts + bucket, 1u);
        next[i] = static_cast<uint16_t>(atomicExch(newest + bucket, i));
        if (in_lds) {
          at[0] = c.x;
          at[1] = c.y;
          at[2] = c.z;
        }
        else store_cluster(scratch, start + i, c);
      }
      if (!in_lds) __threadfence_block();
      mp::wave_sync_lds();
      const unsigned count = counts[l], before = wave_inclusive_scan(count) - count;
      mp::wave_sync_lds();
      counts[l] = before;
      mp::wave_sync_lds();
      for (unsigned i = l; i < n; i += wave_size) {
        const uint64_t key = keys[i];
        const unsigned bucket = static_cast<unsigned>(key >> 42);
        unsigned rank = counts[bucket];
        for (unsigned j = newest[bucket]; j != none;) {
          const uint64_t other = keys[j];
          j = next[j];
          rank += other < key;
        }
        ClusterOut c;
        c.id = static_cast<uint32_t>(key);
        c.phi = static_cast<int16_t>(static_cast<uint16_t>(key >> 32) ^ 0x8000u);
        if (in_lds) {
          c.x = L.xyz[3 * i];
          c.y = L.xyz[3 * i + 1];
          c.z = L.xyz[3 * i + 2];
        }
        else {
          const float* at = scratch.xyz() + 3 * (size_t)(start + i);
          c.x = at[0];
          c.y = at[1];
          c.z = at[2];
        }
        store_cluster(out, start + rank, c);
      }
      return;
    }
    // Too many clusters for that: they sit in the scratch container; rank them against
    // tiles of (phi, id) staged through the slice.
    uint64_t* keys = L.work;
    const Clusters scratch {a.unsorted_scratch, total};
    __threadfence_block();
    for (unsigned i = lane_id(); i < n; i += wave_size) {
      const size_t at = start + i;
      const ClusterSeed s {scratch.ids()[at], scratch.xyz()[3 * at], scratch.xyz()[3 * at + 1]};
      store_cluster(scratch, start + i, place_cluster(*a.geometry, seed_sensor<version>(s), s));
    }
    __threadfence_block();
    unsigned tile = ~0u; // the one whose keys are in the slice
    for (unsigned i0 = 0; i0 < n; i0 += wave_size) {
      const unsigned i = i0 + lane_id();
      const bool mine = i < n;
      ClusterOut c;
      if (mine) {
        c.id = scratch.ids()[start + i];
        c.phi = scratch.phis()[start + i];
        c.x = scratch.xyz()[3 * (size_t)(start + i)];
        c.y = scratch.xyz()[3 * (size_t)(start + i) + 1];
        c.z = scratch.xyz()[3 * (size_t)(start + i) + 2];
      }
      unsigned rank = 0;
      for (unsigned t0 = 0; t0 < n; t0 += mp::ClusterLds::key_tile) {
        const unsigned tn = min(mp::ClusterLds::key_tile, n - t0);
        if (t0 != tile) {
          mp::wave_sync_lds();
          for (unsigned j = lane_id(); j < tn; j += wave_size)
            keys[j] = phi_id_key(scratch.phis()[start + t0 + j], scratch.ids()[start + t0 + j]);
          mp::wave_sync_lds();
          tile = t0;
        }
        if (mine) rank += keys_below(keys, tn, phi_id_key(c.phi, c.id));
      }
      if (mine) store_cluster(out, start + rank, c);
    }
  }
};

template<int version>
__device__ __forceinline__ void
cluster_item(const ClusterArgs& a, mp::ClusterLds& L, unsigned total, unsigned idx, const mp::DirFetch& f)
{
  ClusterItem<version> item(a, L, total, idx);
  if (!item.seeds(f)) item.seeds_in_tiles(f);
  item.finish();
}

// One wave per module pair (loop = false, the default), or a resident grid (loop = true) whose waves
// take items idx, idx + stride, ... and fetch the next item's bank directory record before
// working on the current one.
template<int version, bool loop>
__global__ void __launch_bounds__(mp::waves_per_block* wave_size, 6) k_cluster_mp(ClusterArgs a, unsigned n_events)
{
  __shared__ mp::ClusterLds s_lds[mp::waves_per_block];
  const unsigned wave = threadIdx.x / wave_size;
  const unsigned n_items = n_events * n_module_pairs;
  const unsigned stride = gridDim.x * mp::waves_per_block;
  unsigned idx = blockIdx.x * mp::waves_per_block + wave;
  if (idx >= n_items) return;
  const unsigned total = a.offsets_estimated_input_size[n_items];
  mp::DirFetch cur = mp::fetch_dir(a.directory, a.directory_count, idx);
  if constexpr (!loop) {
    cluster_item<version>(a, s_lds[wave], total, idx, cur);
    return;
  }
  for (; idx < n_items; idx += stride) {
    mp::DirFetch next = cur;
    if (idx + stride < n_items) next = mp::fetch_dir(a.directory, a.directory_count, idx + stride);
    cluster_item<version>(a, s_lds[wave], total, idx, cur);
    cur = next;
  }
}

// One wave per item, or (resident) at most the blocks that stay resident, whose waves loop
// over the items. One wave per item balances uneven module pairs better (the dispatcher starts
// a new wave wherever one ends), and is the default.
static unsigned mp_grid(const void* kernel, unsigned n_items, bool resident)
{
  const unsigned need = (n_items + mp::waves_per_block - 1) / mp::waves_per_block;
  if (!resident) return need;
  const unsigned blocks = device_resident_blocks(kernel, mp::waves_per_block * wave_size, 0);
  return blocks ? min(need, blocks) : need;
}

hipError_t launch_estimate_mp(const EstimateMpLaunch& a, hipStream_t s)
{
  if (!a.n_events) return hipSuccess;
  const unsigned v = a.version == 2 || a.version == 3 ? a.version : 4;
  const void* kernel = v == 2 ? reinterpret_cast<const void*>(&k_estimate_mp<2>)
                     : v == 3 ? reinterpret_cast<const void*>(&k_estimate_mp<3>)
                              : reinterpret_cast<const void*>(&k_estimate_mp<4>);
  const unsigned grid = mp_grid(kernel, a.n_events * n_module_pairs, a.resident_grid);
#define VELO_LAUNCH_EMP(V)                                                                                          \
  hipLaunchKernelGGL(                                                                                               \
    k_estimate_mp<V>, dim3(grid), dim3(mp::waves_per_block * wave_size), 0, s, a.raw,                               \
    static_cast<const BankEntry*>(a.directory), a.directory_count, a.n_events, a.estimated_input_size,            \
    a.event_totals, a.sp_flags)
  switch (a.version) {
  case 2: VELO_LAUNCH_EMP(2); break;
  case 3: VELO_LAUNCH_EMP(3); break;
  default: VELO_LAUNCH_EMP(4); break;
  }
#undef VELO_LAUNCH_EMP
  return hipGetLastError();
}

hipError_t launch_cluster_mp(const ClusterMpLaunch& a, hipStream_t s)
{
  if (!a.n_events) return hipSuccess;
  const unsigned v = a.version == 2 || a.version == 3 ? a.version : 4;
  const void* kernel = v == 2 ? reinterpret_cast<const void*>(&k_cluster_mp<2, true>)
                     : v == 3 ? reinterpret_cast<const void*>(&k_cluster_mp<3, true>)
                              : reinterpret_cast<const void*>(&k_cluster_mp<4, true>);
  const unsigned grid = mp_grid(kernel, a.n_events * n_module_pairs, a.resident_grid);
  const ClusterArgs args {a.raw, static_cast<const BankEntry*>(a.directory), a.directory_count,
                          a.offsets_estimated_input_size, a.sp_flags, reinterpret_cast<const Geometry*>(a.geometry),
                          a.sp_patterns, a.sp_fx, a.sp_fy, a.module_cluster_num, a.sorted_container, a.unsorted_scratch};
#define VELO_LAUNCH_CMP(V, L)                                                                                       \
  hipLaunchKernelGGL((k_cluster_mp<V, L>), dim3(grid), dim3(mp::waves_per_block * wave_size), 0, s, args, a.n_events)
  switch (v * 2 + (a.resident_grid ? 1 : 0)) {
  case 4: VELO_LAUNCH_CMP(2, false); break;
  case 5: VELO_LAUNCH_CMP(2, true); break;
  case 6: VELO_LAUNCH_CMP(3, false); break;
  case 7: VELO_LAUNCH_CMP(3, true); break;
  case 8: VELO_LAUNCH_CMP(4, false); break;
  default: VELO_LAUNCH_CMP(4, true); break;
  }
#undef VELO_LAUNCH_CMP
  return hipGetLastError();
}

} // namespace velo

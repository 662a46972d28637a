// search_by_triplet and the three-hit filter for gfx950.
//
//   k_search_by_triplet     SearchByTriplet.cu:110-609   one workgroup per event
//   k_three_hit_filter      ThreeHitTracksFilter.cu:48-169
//
// The reference appends seeds, tracks to follow, promoted tracks and three-hit tracks with
// atomicAdd, so its GPU output order depends on scheduling. Here every append is an ordered
// compaction (wave ballot + popcount, then a prefix over the waves of the block) over the
// items in the order the CPU target visits them (h1 index order in seeding, ring order in
// forwarding). Ring slots, track numbers and three-hit slots therefore land exactly where the
// CPU target puts them, and everything downstream is bit-identical.
//
// The event's hits (x, y, z, phi, used) live in LDS when they fit the per-launch budget;
// a larger event runs the same code on the global containers.
#include "velo_common.cuh"
#include "velo_kernels.h"
#include "velo_mfma.cuh"

namespace velo {

// LDS bytes per hit of the full layout: x, y, z (f32), then phi (i16) and flags in one word.
constexpr unsigned search_bytes_per_hit = 16;
// The mixed layout keeps phi (i16) and a flags byte.
constexpr unsigned mixed_bytes_per_hit = 3;
// Default capacity of the list of unused hits of the previous module pair used by seeding
// (a launch parameter, at most 1024); a larger module pair takes the pendulum walk.
constexpr unsigned unused_list_cap = 1024;
// Number of tracks to follow kept in LDS, the last positions of the ring (which is written through
// to HBM and holds all max_tracks_to_follow): a power of two, 64 to 512 where the caller sets it and
// 512 or 1024 where the launch chooses. A forwarding step reads the ring and the tracks back from HBM when
// its entries and those it writes exceed the window: at 512 positions that was the largest events,
// which set the length of a launch.
constexpr unsigned ring_window = 1024;
constexpr unsigned max_ring_window_knob = 512;
static_assert(max_tracks_to_follow % ring_window == 0, "window positions follow ring positions");

// A window entry: the ring's entry and what forwarding reads of its track, in 8 bytes. last2: the
// track's last two hits (low and high 16 bits). A seed (bit_seed) holds its tracklet's number in
// 11 bits and its first hit in the 16 above; a track its number in 20 bits (an event has fewer
// than 22 300 track slots; larger numbers stand for "beyond them") and its number of hits in the
// 5 above. Both hold the skipped modules where the ring's entries do.
constexpr unsigned seed_first_pos = 11, track_hits_pos = 20;
constexpr uint32_t window_track_number = (1u << track_hits_pos) - 1;
static_assert(max_tracks_to_follow == 1u << seed_first_pos && max_track_size < 32 && skipped_pos == 28, "window entry");
__device__ __forceinline__ uint2 window_seed(uint32_t full, unsigned first, unsigned last2)
{
  return make_uint2(full | (first << seed_first_pos), last2);
}
__device__ __forceinline__ uint2 window_track(uint32_t skipped, uint32_t number, unsigned n_hits, unsigned last2)
{
  return make_uint2(skipped | min(number, window_track_number) | (n_hits << track_hits_pos), last2);
}

// The waves that work on the event: all of the workgroup's, or the first few of them (the others
// have ended, and the hardware's barriers do not wait for them). A team of one wave takes the
// barriers as well: one costs it ten cycles, and a branch around it kept its condition in scalar
// registers that were spilled (20 000 events: 1640 us, 1660 with the branch).
struct Team {
  unsigned waves, lanes, wave; // wave: this wave's number
  __device__ __forceinline__ void sync() const { __syncthreads(); }
  static __device__ __forceinline__ void wave_fence()
  {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
};

// Up to three 0/1 flags scanned at once over the team. Exclusive ranks in r[], totals in t[]
// (wave-uniform, in scalar registers: they come from ballots and lane reads only).
// One barrier: consecutive scans must alternate between two scratch buffers (a scan's reads of
// its buffer are ordered before the next scan's barrier, hence before the reuse two scans on).
struct Scan3 {
  uint32_t r[3];
  uint32_t t[3];
};
template<unsigned n>
__device__ __forceinline__ Scan3 team_flag_scan(const Team& team, bool f0, bool f1, bool f2, uint2* scratch)
{
  const bool f[3] = {f0, f1, f2};
  Scan3 s;
#pragma unroll
  for (unsigned k = 0; k < 3; ++k) {
    s.r[k] = s.t[k] = 0;
    if (k >= n) continue;
    const uint64_t b = __ballot(f[k]);
    s.r[k] = rank_below(b);
    s.t[k] = __popcll(b);
  }
  if (team.waves == 1) return s;
  // Per wave: the first two counts as 16 bits each (at most 1024), the third in a word of its own.
  if (lane_id() == 0) scratch[team.wave] = make_uint2(s.t[0] | (s.t[1] << 16), s.t[2]);
  __syncthreads();
  const uint2 c = scratch[min(lane_id(), team.waves - 1)];
  uint32_t tot01 = 0, tot2 = 0, before01 = 0, before2 = 0;
  for (unsigned w = 0; w < team.waves; ++w) {
    if (w == team.wave) {
      before01 = tot01;
      before2 = tot2;
    }
    tot01 += __builtin_amdgcn_readlane(c.x, w);
    if constexpr (n > 2) tot2 += __builtin_amdgcn_readlane(c.y, w);
  }
  s.r[0] += before01 & 0xFFFFu;
  s.r[1] += before01 >> 16;
  s.r[2] += before2;
  s.t[0] = tot01 & 0xFFFFu;
  s.t[1] = tot01 >> 16;
  s.t[2] = tot2;
  return s;
}

struct ModulePairData {
  unsigned hit_start;
  unsigned hit_num;
  float z[2];
  unsigned table; // offset of the module pair's phi bucket table, or no_phi_table
};

// Phi bucket tables of an event's module pairs (LDS, u8 entries, module pairs of at most 255
// hits): entry b < phi_buckets is the first position whose phi lies in bucket b or above, entry
// phi_buckets the number of hits. 128 buckets: a window of the default tolerance then reads about
// a third of a hit more than it holds (a module pair has some 40 hits), for 3.4 KB of LDS.
constexpr unsigned phi_buckets = 128;
constexpr unsigned phi_bucket_shift = 9;
constexpr unsigned phi_table_stride = phi_buckets + 2; // even, so that two entries can be written at once
constexpr unsigned phi_tables_bytes = (n_module_pairs * phi_table_stride + 15) & ~15u;
constexpr unsigned no_phi_table = 0xFFFFFFFFu;
// A module pair whose phis are not in order: retina words of one pixel that differ only in their
// fractions share a sorting key and so a slot, and the slot left over among the module pair's hits
// holds whatever was there (one module pair in a few thousand events). Tables and runs need
// order, so such a module pair is searched as irregular_search states.
constexpr unsigned irregular_phis = 0xFFFFFFFEu;
__device__ __forceinline__ unsigned phi_bucket(int16_t phi)
{
  return static_cast<unsigned>(static_cast<uint16_t>(phi) ^ 0x8000u) >> phi_bucket_shift;
}

// Per-hit flags of the LDS layouts: bit 0 = used (dev_hit_used), bit 1 = module parity of
// the hit's sensor, ((id >> 18) & 0xFF) / 4 % 2.
constexpr uint8_t flag_used = 1, flag_odd = 2;

struct Hit {
  float x, y, z;
  int16_t phi;
  bool used, odd;
};

// Hits of one event in LDS, 16 bytes each: x, y, z, then phi in the low and the flags in the
// high half of a word, so that one 128-bit read brings a hit (five reads of 1 to 4 bytes with an
// address each before).
struct LdsHits {
  uint4* h;
  const uint8_t* tables;
  __device__ __forceinline__ Hit load(unsigned i) const
  {
    const uint4 v = h[i];
    return {__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), static_cast<int16_t>(v.w & 0xFFFFu),
            (v.w & (flag_used << 16)) != 0, (v.w & (flag_odd << 16)) != 0};
  }
  __device__ __forceinline__ int16_t phi(unsigned i) const { return static_cast<int16_t>(h[i].w & 0xFFFFu); }
  __device__ __forceinline__ bool used(unsigned i) const { return (h[i].w & (flag_used << 16)) != 0; }
  __device__ __forceinline__ void mark_used(unsigned i) const
  {
    (void) __hip_atomic_fetch_or(&h[i].w, uint32_t(flag_used) << 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
};

// Module parity of a hit from its LHCbID (SearchByTriplet.cu:498-499).
__device__ __forceinline__ uint8_t module_parity(uint32_t id) { return static_cast<uint8_t>(((id & 0x3fc0000u) >> 18) / 4 % 2); }

// Hits of one event read from the sorted cluster container in global memory.
struct GlobalHits {
  const float* xyz;
  const int16_t* ph;
  uint8_t* used_flags; // dev_hit_used
  const uint32_t* ids;
  const uint8_t* tables;
  __device__ __forceinline__ Hit load(unsigned i) const
  {
    return {xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2], ph[i], used_flags[i] != 0, module_parity(ids[i]) != 0};
  }
  __device__ __forceinline__ int16_t phi(unsigned i) const { return ph[i]; }
  __device__ __forceinline__ bool used(unsigned i) const { return used_flags[i] != 0; }
  __device__ __forceinline__ void mark_used(unsigned i) const { used_flags[i] = 1; }
};

// Hits of one event: phi and used flags in LDS, coordinates in global memory (events too large
// for the full LDS layout). Lanes that mark the same hit concurrently all store the same byte, so
// the read-modify-write cannot lose a bit.
struct MixedHits {
  const float* xyz;
  const int16_t* ph;
  uint8_t* flags;
  const uint8_t* tables;
  __device__ __forceinline__ Hit load(unsigned i) const
  {
    const uint8_t f = flags[i];
    return {xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2], ph[i], (f & flag_used) != 0, (f & flag_odd) != 0};
  }
  __device__ __forceinline__ int16_t phi(unsigned i) const { return ph[i]; }
  __device__ __forceinline__ bool used(unsigned i) const { return (flags[i] & flag_used) != 0; }
  __device__ __forceinline__ void mark_used(unsigned i) const { flags[i] |= flag_used; }
};

// Work counters of one thread (seeding evaluations, forwarding evaluations, extrapolations,
// search probes); only kept by the counting instantiation of the kernel.
struct WorkCount {
  uint32_t seed_eval = 0, fwd_eval = 0, extrap = 0, steps = 0;
  // Wall-clock ticks spent by the workgroup in each Phase, kept by thread 0 (which takes part
  // in every phase, so its marks follow the slowest wave only at barriers).
  unsigned long long phase[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  unsigned long long last = 0;
};

// forwarding; h1 compaction; seeding step 1 split into the h0 search (h1 and phi reads, then
// the search in the previous module pair) and the choice of the h0 candidates; a place for a wait
// that there is no more (always zero); the scoring of the pairs; the append; the rest.
enum Phase {
  phase_forwarding,
  phase_compaction,
  phase_seed1_search,
  phase_seed1_pendulum,
  phase_seed1_wait,
  phase_seed2,
  phase_seed3,
  phase_other,
  n_phases
};

template<bool count>
__device__ __forceinline__ void phase_mark(WorkCount& wc, Phase p)
{
  if constexpr (count) {
    if (threadIdx.x == 0) {
      const unsigned long long now = wall_clock64();
      wc.phase[p] += now - wc.last;
      wc.last = now;
    }
  }
}

// First position i of the sorted phis of hits [start, start + size) with phi >= value (the
// leftmost binary search of BinarySearch.cuh, same result on every input). Eight-way: each round
// probes seven split points at once (independent reads) and keeps the eighth of the range that
// holds the answer, so n hits take about log8(n) dependent round trips instead of log2(n).
// `steps` counts the probes.
template<bool count, typename H>
__device__ __forceinline__ unsigned counted_search(const H& hits, unsigned start, unsigned size, int16_t value, WorkCount& wc)
{
  unsigned lo = 0, hi = size; // answer in [lo, hi]; phi[< lo] < value <= phi[>= hi]
  while (lo < hi) {
    const unsigned span = hi - lo;
    unsigned p[7];
    bool below[7];
    int16_t v[7];
#pragma unroll
    for (unsigned j = 0; j < 7; ++j) {
      p[j] = lo + ((j + 1) * span) / 8; // lo <= p[j] < hi, non-decreasing in j
      v[j] = hits.phi(start + p[j]);
    }
    // All seven reads are issued before the first compare waits for one (the scheduler would
    // otherwise interleave read, wait and compare, one LDS round trip per probe).
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (unsigned j = 0; j < 7; ++j) below[j] = v[j] < value; // true for a prefix of j (sorted)
    if constexpr (count) wc.steps += 7;
    unsigned nlo = lo, nhi = hi;
#pragma unroll
    for (unsigned j = 0; j < 7; ++j)
      if (below[j]) nlo = p[j] + 1;
#pragma unroll
    for (int j = 6; j >= 0; --j)
      if (!below[j]) nhi = p[j];
    lo = nlo;
    hi = nhi;
  }
  return lo;
}

// The search in a module pair whose phis are out of order, where the answer depends on the way: the
// 8-way search for the bounds of the value's bucket of 1024, then that bucket's elements, counted
// directly for up to four (module pairs of more than 255 hits: the 8-way search over all hits).
template<bool count, typename H>
__device__ __forceinline__ unsigned irregular_search(const H& hits, const ModulePairData& mp, int16_t value, WorkCount& wc)
{
  unsigned lo = 0, hi = mp.hit_num;
  if (mp.hit_num <= 255u) {
    const int first = value & ~1023;
    lo = counted_search<count>(hits, mp.hit_start, mp.hit_num, static_cast<int16_t>(first), wc);
    if (first + 1024 <= 32767) hi = counted_search<count>(hits, mp.hit_start, mp.hit_num, static_cast<int16_t>(first + 1024), wc);
    if (hi <= lo) return lo;
    if (hi - lo <= 4) {
      unsigned c = lo;
      for (unsigned k = lo; k < hi; ++k) c += hits.phi(mp.hit_start + k) < value ? 1u : 0u;
      return c;
    }
  }
  return lo + counted_search<count>(hits, mp.hit_start + lo, hi - lo, value, wc);
}

// The same lower bound in a module pair through its bucket table: positions before the value's
// bucket hold smaller phis and positions after it larger ones, so the answer is the bucket's
// start plus the bucket's elements below the value (read directly for up to four, by
// the 8-way search for more). Module pairs without a table take the 8-way search.
template<bool count, typename H>
__device__ __forceinline__ unsigned mp_search(const H& hits, const ModulePairData& mp, int16_t value, WorkCount& wc)
{
  if (mp.table == irregular_phis) return irregular_search<count>(hits, mp, value, wc);
  if (mp.table == no_phi_table) return counted_search<count>(hits, mp.hit_start, mp.hit_num, value, wc);
  const uint8_t* t = hits.tables + mp.table + phi_bucket(value);
  const unsigned lo = t[0], hi = t[1];
  if (hi - lo > 4) return lo + counted_search<count>(hits, mp.hit_start + lo, hi - lo, value, wc);
  int16_t v[4];
#pragma unroll
  for (unsigned k = 0; k < 4; ++k) v[k] = hits.phi(mp.hit_start + (lo + k < hi ? lo + k : 0u));
  unsigned c = lo;
#pragma unroll
  for (unsigned k = 0; k < 4; ++k) c += lo + k < hi && v[k] < value ? 1u : 0u;
  return c;
}

// The phi bucket tables of all module pairs that have one, four module pairs per wave at a time:
// a histogram of the hits' buckets in LDS (`hist`, phi_buckets 16-bit counts per module pair),
// turned into positions by a wave scan, two buckets a lane. hist_waves: the waves that hist has
// room for. Module pairs whose phis are out of order are marked here.
constexpr unsigned hist_words = phi_buckets / 2;
constexpr unsigned hist_bytes = 4 * hist_words * sizeof(uint32_t);
// LDS of the ring's window, which first holds the tables' histograms.
__host__ __device__ constexpr unsigned window_bytes(unsigned window)
{
  return window * sizeof(uint2) > hist_bytes ? window * sizeof(uint2) : hist_bytes;
}
template<typename H>
__device__ __forceinline__ void
build_phi_tables(const H& hits, ModulePairData* mp, uint8_t* tables, uint32_t* hist, unsigned hist_waves, const Team& team)
{
  static_assert(hist_words == wave_size, "two buckets per lane");
  const unsigned builders = min(team.waves, hist_waves);
  if (team.wave >= builders) return;
  const unsigned l = lane_id();
  uint32_t* h = hist + 4 * hist_words * team.wave;
  const auto count = [&](unsigned u, int16_t phi) {
    const unsigned b = phi_bucket(phi);
    atomicAdd(&h[u * hist_words + b / 2], b & 1u ? 0x10000u : 1u);
  };
  for (unsigned m0 = 4 * team.wave; m0 < n_module_pairs; m0 += 4 * builders) {
    unsigned start[4], n[4];
    int16_t p[4], q[4];
    bool table[4];
#pragma unroll
    for (unsigned u = 0; u < 4; ++u) {
      const unsigned m = min(m0 + u, n_module_pairs - 1);
      start[u] = mp[m].hit_start;
      n[u] = m0 + u < n_module_pairs ? mp[m].hit_num : 0u;
      table[u] = mp[m].table != no_phi_table;
      h[u * hist_words + l] = 0;
    }
#pragma unroll
    for (unsigned u = 0; u < 4; ++u) {
      p[u] = l < n[u] ? hits.phi(start[u] + l) : int16_t(0);
      q[u] = l > 0 && l < n[u] ? hits.phi(start[u] + l - 1) : p[u]; // the hit before
    }
    Team::wave_fence();
#pragma unroll
    for (unsigned u = 0; u < 4; ++u) {
      if (table[u] && l < n[u]) count(u, p[u]);
      bool ordered = q[u] <= p[u];
      for (unsigned i = l + wave_size; i < n[u]; i += wave_size) {
        const int16_t phi = hits.phi(start[u] + i);
        ordered = ordered && hits.phi(start[u] + i - 1) <= phi;
        if (table[u]) count(u, phi);
      }
      if (__ballot(!ordered) && l == 0) mp[m0 + u].table = irregular_phis;
    }
    Team::wave_fence();
#pragma unroll
    for (unsigned u = 0; u < 4; ++u) {
      const uint32_t c = h[u * hist_words + l];
      const uint32_t both = (c & 0xFFFFu) + (c >> 16);
      const uint32_t before = wave_inclusive_scan(both) - both;
      if (table[u] && m0 + u < n_module_pairs) {
        uint16_t* t = reinterpret_cast<uint16_t*>(tables + (m0 + u) * phi_table_stride);
        t[l] = static_cast<uint16_t>(before | (before + (c & 0xFFFFu)) << 8);
        if (l == 0) t[phi_buckets / 2] = static_cast<uint16_t>(n[u]);
      }
    }
    Team::wave_fence();
  }
}

struct SearchShared {
  uint32_t extended;                 // hits added to tracks of four or more hits, all waves
  ModulePairData mp[n_module_pairs]; // hit range (event-relative) and module z of every module pair
  uint2 scan[2][16];                 // team_flag_scan scratch, used alternately
};

// The event's counters, identical in every lane of the workgroup (updated from block-wide
// scan totals), so no lane has to publish them through LDS.
struct Counters {
  uint32_t ttf = 0;        // atomics::tracks_to_follow
  uint32_t three = 0;      // atomics::number_of_three_hit_tracks
  uint32_t local_hits = 0; // atomics::local_number_of_hits
  uint32_t n_tracks = 0;   // dev_number_of_velo_tracks[event]
  uint32_t status = 0;
  uint32_t extended = 0;   // this wave's part of SearchShared::extended
  unsigned scan_buffer = 0;
};

template<unsigned n>
__device__ __forceinline__ Scan3 scan(const Team& team, SearchShared& sh, Counters& c, bool f0, bool f1 = false, bool f2 = false)
{
  const Scan3 s = team_flag_scan<n>(team, f0, f1, f2, sh.scan[c.scan_buffer]);
  c.scan_buffer ^= 1u;
  return s;
}

// A module pair's descriptor in scalar registers (the index is the same in every lane).
__device__ __forceinline__ ModulePairData module_pair_data(const SearchShared& sh, unsigned i)
{
  const ModulePairData m = sh.mp[i];
  ModulePairData r;
  r.hit_start = __builtin_amdgcn_readfirstlane(m.hit_start);
  r.hit_num = __builtin_amdgcn_readfirstlane(m.hit_num);
  r.z[0] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(m.z[0])));
  r.z[1] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(m.z[1])));
  r.table = __builtin_amdgcn_readfirstlane(m.table);
  return r;
}

// Seeding scratch in dynamic LDS, blockDim entries of each: the unused hits of the current module
// pair (one compaction chunk), the h0 candidate of every (h1, h0) pair, and in scored mode the
// chosen seed of every h1 (h0 | h2 << 16, or no_seed).
static_assert(initial_seeding_h0_candidates == 8 && seeding_h0_candidates == 4, "track_seeding splits lanes by K = 4 or 8");
constexpr uint32_t no_seed = 0xFFFFFFFFu;
constexpr unsigned seed_scratch_bytes_per_lane = 4 + 2 + 2;
struct SeedScratch {
  uint32_t* seed;
  uint16_t* h0;
  uint16_t* h1_chunk;
  uint16_t* unused;   // unused hits of the previous module pair (relative indices, ascending)
  uint16_t* before;   // per position of the previous module pair: the unused hits before it
  unsigned list_cap;  // entries of `unused` and `before`
};

struct ScorerLds;

struct EventOutputs {
  TrackHits* tracks;
  TrackletHits* three_hit_tracks;
  TrackletHits* tracklets;
  uint32_t* ttf;        // the ring of tracks to follow in HBM (max_tracks_to_follow entries)
  uint2* window_entries; // its last `window` positions in LDS (position p at p & window_mask)
  uint16_t* h1_indices;
  unsigned track_capacity;
  unsigned event_number;
  SeedLog seed_log;
  const ScorerLds* scorer;
  float scorer_threshold;
  unsigned window;      // LDS window positions (a power of two dividing max_tracks_to_follow)
  unsigned window_mask; // window - 1
};

// A line to be continued into a module pair: its start, slopes and phi at the module pair.
struct Line {
  float x0, y0, z0, tx, ty;
  int16_t phi;
};
__device__ __forceinline__ float scatter_at(const Line& l, const Hit& h)
{
  const float dz = h.z - l.z0;
  const float predx = l.x0 + l.tx * dz;
  const float predy = l.y0 + l.ty * dz;
  const float dx = predx - h.x;
  const float dy = predy - h.y;
  return dx * dx + dy * dy;
}

// The closest hit as the reference walks to it: from the leftmost hit at or above
// phi - phi_tolerance, wrapping around, until one lies further than phi_tolerance from phi
// (SearchByTriplet.cu:384-433, 520-560); unused_only: used hits are passed over (seeding).
template<bool count, bool unused_only, typename H>
__device__ __forceinline__ bool closest_hit_walk(
  WorkCount& wc, const H& hits, const ModulePairData& mp, const Line& l, int16_t phi_tolerance, float& best, uint32_t& best_index)
{
  bool any = false;
  unsigned p = mp_search<count>(hits, mp, static_cast<int16_t>(l.phi - phi_tolerance), wc);
  for (unsigned j = 0; j < mp.hit_num; ++j, ++p) {
    if (p >= mp.hit_num) p -= mp.hit_num;
    const Hit h = hits.load(mp.hit_start + p);
    const int16_t phi_diff = h.phi - l.phi;
    const int16_t abs_phi_diff = phi_diff < 0 ? -phi_diff : phi_diff;
    if (abs_phi_diff > phi_tolerance) break;
    if (unused_only && h.used) continue;
    if constexpr (count) ++(unused_only ? wc.seed_eval : wc.fwd_eval);
    const float scatter = scatter_at(l, h);
    if (scatter < best) {
      best = scatter;
      best_index = mp.hit_start + p;
      any = true;
    }
  }
  return any;
}

// Tolerances up to this one (an eighth of a turn) make every walk one run of the sorted hits.
constexpr int16_t max_run_tolerance = 8192;

// The hit of a module pair closest to a line: the first strict minimum of the scatter below
// `best`, in the order of closest_hit_walk and with the same result. Returns whether there is one.
// The hits within the tolerance are one run of the module pair's circle of hits, and the phi
// buckets of its two ends bound it from both sides with two table reads, so no search for its
// start and no hit read to find its end: the run and the few hits of the end buckets outside
// it are read four at a time and evaluated without branches, which lets their arithmetic overlap
// (one dependent operation takes 8 cycles here, an independent one 5; an LDS read 64). Nearly
// always one pass of four serves the whole wave. Where the walk differs from the run: its
// |difference| of 16 bits takes a hit exactly opposite for one within any tolerance, so it goes on
// through such hits where they are the next ones after the run (which may be empty); those lanes,
// tolerances beyond max_run_tolerance and module pairs out of order take the walk itself.
template<bool count, bool unused_only, typename H>
__device__ __forceinline__ bool closest_hit(
  WorkCount& wc, const H& hits, const ModulePairData& mp, const Line& l, int16_t phi_tolerance, float& best, uint32_t& best_index)
{
  const unsigned n = mp.hit_num;
  if (n == 0) return false;
  if (phi_tolerance < 0 || phi_tolerance > max_run_tolerance || mp.table == irregular_phis)
    return closest_hit_walk<count, unused_only>(wc, hits, mp, l, phi_tolerance, best, best_index);
  const int16_t from = static_cast<int16_t>(l.phi - phi_tolerance), to = static_cast<int16_t>(l.phi + phi_tolerance);
  unsigned lo, hi;
  if (mp.table == no_phi_table) {
    lo = counted_search<count>(hits, mp.hit_start, n, from, wc);
    hi = to == 32767 ? n : counted_search<count>(hits, mp.hit_start, n, static_cast<int16_t>(to + 1), wc);
  }
  else {
    const uint8_t* t = hits.tables + mp.table;
    lo = t[phi_bucket(from)];
    hi = t[phi_bucket(to) + 1];
  }
  const unsigned length = to < from ? n - lo + hi : hi - lo;
  const unsigned width = 2u * static_cast<unsigned>(phi_tolerance);
  // Position lo + j of the circle; positions beyond the run only stay in range.
  const auto position = [&](unsigned j) { return mp.hit_start + min(min(lo + j, lo + j - n), n - 1); };
  const int16_t after = hits.phi(position(length)); // the end buckets hold no opposite hit
  const float limit = best;
  uint32_t visits = 0;
  bool any = false;
  for (unsigned j0 = 0; j0 < length; j0 += 4) {
    unsigned index[4];
    Hit h[4];
#pragma unroll
    for (unsigned k = 0; k < 4; ++k) index[k] = position(j0 + k);
#pragma unroll
    for (unsigned k = 0; k < 4; ++k) h[k] = hits.load(index[k]);
    __builtin_amdgcn_sched_barrier(0); // all four reads are in flight before the first is waited for
#pragma unroll
    for (unsigned k = 0; k < 4; ++k) {
      const float scatter = scatter_at(l, h[k]);
      const bool in_run = j0 + k < length && static_cast<uint16_t>(h[k].phi - from) <= width;
      const bool visited = in_run && !(unused_only && h[k].used);
      if constexpr (count) visits += visited;
      const bool closer = visited && scatter < best;
      best = closer ? scatter : best;
      best_index = closer ? index[k] : best_index;
      any = any || closer;
    }
  }
  if (static_cast<uint16_t>(after - l.phi) == 0x8000u) {
    best = limit;
    return closest_hit_walk<count, unused_only>(wc, hits, mp, l, phi_tolerance, best, best_index);
  }
  if constexpr (count) (unused_only ? wc.seed_eval : wc.fwd_eval) += visits;
  return any;
}

// SearchByTriplet.cu:272-292: the phi at dz along the line from h0.
template<bool count>
__device__ __forceinline__ int16_t extrapolated_phi(WorkCount& wc, float h0x, float h0y, float tx, float ty, float dz)
{
  const float predx = tx * dz;
  const float predy = ty * dz;
  const float xp = h0x + predx;
  const float yp = h0y + predy;
  if constexpr (count) ++wc.extrap;
  return hit_phi_16(xp, yp);
}

// The learned scorer's weights in LDS (scored mode): W1 (K padded to 16) and W2 as bf16, the
// biases and w3 (bf16-rounded) as FP32.
// The scorer's weights in LDS, transposed for the products below: w1t[j][k] = bf16(W1[k][j])
// (k < 16, zero from 10), w2t[j2][j1] = bf16(W2[j1][j2]); biases and bf16(w3) in FP32.
struct ScorerLds {
  uint16_t w1t[32 * 16];
  uint16_t w2t[32 * 32];
  float b1[32], b2[32], w3[32];
  float b3;
};
constexpr unsigned scorer_lds_bytes = (sizeof(ScorerLds) + 15) & ~15u;

__device__ void load_scorer(const float* p, ScorerLds& w)
{
  using namespace mlp;
  for (unsigned t = threadIdx.x; t < 32 * 32; t += blockDim.x) {
    const unsigned j = t / 32, k = t % 32;
    w.w2t[t] = to_bf16(p[param_w2 + k * 32 + j]);
    if (t < 32 * 16) {
      const unsigned jj = t / 16, kk = t % 16;
      w.w1t[t] = kk < n_inputs ? to_bf16(p[param_w1 + kk * 32 + jj]) : 0;
    }
  }
  for (unsigned t = threadIdx.x; t < 32; t += blockDim.x) {
    w.b1[t] = p[param_b1 + t];
    w.b2[t] = p[param_b2 + t];
    w.w3[t] = from_bf16(to_bf16(p[param_w3 + t]));
  }
  if (threadIdx.x == 0) w.b3 = p[param_b3];
}

__device__ __forceinline__ mlp::bf16x4 bf16x4_from(uint2 v)
{
  mlp::bf16x4 r;
  r[0] = static_cast<short>(v.x & 0xFFFFu);
  r[1] = static_cast<short>(v.x >> 16);
  r[2] = static_cast<short>(v.y & 0xFFFFu);
  r[3] = static_cast<short>(v.y >> 16);
  return r;
}

// Logit of the seed of lane l (features fp[0..9]) for the lanes set in `live` (a ballot, so
// wave-uniform), with the products of k_mlp_score computed transposed: Z1^T = W1b^T xb^T and
// Z2^T = W2b^T A1b^T on v_mfma_f32_32x32x8_bf16. Seeds 32 rb + c form row block rb (computed
// only when one of its seeds is live), with seed c in column c. In that layout the hidden layer
// leaves the first product exactly where the second takes its operand (element 4 s + i of
// lane l is hidden unit 8 s + 4 (l / 32) + i of seed l % 32), and the output layer is a sum
// over the lane's 16 hidden units plus one exchange with lane l ^ 32 (the other 16), so the
// wave needs no LDS beyond the weights. The output sum runs in another order than
// k_mlp_score's. The whole wave must be active.
__device__ __forceinline__ float scorer_logit(const float* fp, uint64_t live, const ScorerLds& w)
{
  using namespace mlp;
  const unsigned l = lane_id(), h = l / 32, c = l % 32;
  // Features of the seed in lane l ^ 32: lanes l < 32 send features 4..7 (the operand of the
  // upper half in row block 0), lanes l >= 32 send 0..3, 8 and 9 (that of the lower half in row
  // block 1).
  float other[6];
#pragma unroll
  for (unsigned i = 0; i < 4; ++i) other[i] = __shfl_xor(h ? fp[i] : fp[4 + i], 32, wave_size);
  other[4] = __shfl_xor(fp[8], 32, wave_size);
  other[5] = __shfl_xor(fp[9], 32, wave_size);
  float logit = 0.f;
#pragma unroll
  for (unsigned rb = 0; rb < 2; ++rb) {
    if (!static_cast<uint32_t>(live >> (32 * rb))) continue;
    const bool own = h == rb; // this lane's seed is column c of the row block
    // B operand of the first product: features 4 h + i (k-step 0) and 8 + 4 h + i (k-step 1).
    bf16x4 x0, x1;
#pragma unroll
    for (unsigned i = 0; i < 4; ++i) {
      const float f0 = own ? fp[4 * h + i] : other[i];
      x0[i] = static_cast<short>(to_bf16(f0));
      const float f1 = h ? 0.f : (i < 2 ? (own ? fp[8 + i] : other[4 + i]) : 0.f);
      x1[i] = static_cast<short>(to_bf16(f1));
    }
    f32x16 acc = zero16();
    acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(
      bf16x4_from(*reinterpret_cast<const uint2*>(w.w1t + 16 * c + 4 * h)), x0, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(
      bf16x4_from(*reinterpret_cast<const uint2*>(w.w1t + 16 * c + 8 + 4 * h)), x1, acc, 0, 0, 0);
    f32x16 acc2 = zero16();
#pragma unroll
    for (unsigned st = 0; st < 4; ++st) {
      const float4 b1 = *reinterpret_cast<const float4*>(w.b1 + 8 * st + 4 * h);
      const float z[4] = {acc[4 * st] + b1.x, acc[4 * st + 1] + b1.y, acc[4 * st + 2] + b1.z,
                          acc[4 * st + 3] + b1.w};
      bf16x4 a1;
#pragma unroll
      for (unsigned i = 0; i < 4; ++i) a1[i] = static_cast<short>(to_bf16(z[i] > 0.f ? z[i] : 0.f));
      acc2 = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(
        bf16x4_from(*reinterpret_cast<const uint2*>(w.w2t + 32 * c + 8 * st + 4 * h)), a1, acc2, 0, 0, 0);
    }
    float part = 0.f;
#pragma unroll
    for (unsigned st = 0; st < 4; ++st) {
      const float4 b2 = *reinterpret_cast<const float4*>(w.b2 + 8 * st + 4 * h);
      const float4 w3 = *reinterpret_cast<const float4*>(w.w3 + 8 * st + 4 * h);
      const float z[4] = {acc2[4 * st] + b2.x, acc2[4 * st + 1] + b2.y, acc2[4 * st + 2] + b2.z,
                          acc2[4 * st + 3] + b2.w};
      const float ww[4] = {w3.x, w3.y, w3.z, w3.w};
#pragma unroll
      for (unsigned i = 0; i < 4; ++i) part += (z[i] > 0.f ? z[i] : 0.f) * ww[i];
    }
    const float sum = part + __shfl_xor(part, 32, wave_size);
    if (own) logit = sum + w.b3;
  }
  return logit;
}

// Scorer features of a seed (h0, h1, h2) whose h1 lies in module pair `module_pair` (no
// reference counterpart): h2's residual to the (h0, h1) line and h1's residual to the (h0, h2)
// line in x and y, the phi steps h0 -> h1 and h1 -> h2, the (h0, h1) slopes, the scatter and the
// module pair, each scaled to order one.
template<typename H>
__device__ __forceinline__ void
seed_features(const H& hits, unsigned h0, unsigned h1, unsigned h2, unsigned module_pair, float* f)
{
  const Hit a = hits.load(h0), b = hits.load(h1), c = hits.load(h2);
  const float x0 = a.x, y0 = a.y, z0 = a.z;
  const float x1 = b.x, y1 = b.y, z1 = b.z;
  const float x2 = c.x, y2 = c.y, z2 = c.z;
  const float td = 1.0f / (z1 - z0);
  const float tx = (x1 - x0) * td;
  const float ty = (y1 - y0) * td;
  const float dz2 = z2 - z0;
  const float dx2 = (x0 + tx * dz2) - x2;
  const float dy2 = (y0 + ty * dz2) - y2;
  const float td02 = 1.0f / (z2 - z0);
  const float dz1 = z1 - z0;
  const float dx1 = (x0 + ((x2 - x0) * td02) * dz1) - x1;
  const float dy1 = (y0 + ((y2 - y0) * td02) * dz1) - y1;
  const int16_t dphi01 = static_cast<int16_t>(b.phi - a.phi);
  const int16_t dphi12 = static_cast<int16_t>(c.phi - b.phi);
  f[0] = dx2 * 4.0f;
  f[1] = dy2 * 4.0f;
  f[2] = dx1 * 4.0f;
  f[3] = dy1 * 4.0f;
  f[4] = static_cast<float>(dphi01) * (1.0f / 512.0f);
  f[5] = static_cast<float>(dphi12) * (1.0f / 512.0f);
  f[6] = tx * 4.0f;
  f[7] = ty * 4.0f;
  f[8] = (dx2 * dx2 + dy2 * dy2) * 12.5f;
  f[9] = static_cast<float>(module_pair) * (1.0f / 32.0f);
}

// For the wave's seeding lanes: values of the other lanes of a group of K = 4 or 8, and the least
// key of the group, by DPP moves (quad permutations, and the mirror of half a row for K = 8).
template<int ctrl>
__device__ __forceinline__ uint32_t dpp(uint32_t v)
{
  return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), ctrl, 0xF, 0xF, true));
}
constexpr int dpp_xor1 = 0xB1, dpp_xor2 = 0x4E, dpp_xor3 = 0x1B, dpp_half_mirror = 0x141;

// How many of a group's 2 K keys (two per lane) lie below `mine`, of which a and b are this
// lane's own pair.
__device__ __forceinline__ uint32_t below4(uint32_t a, uint32_t b, uint32_t mine)
{
  uint32_t c = 0;
  c += dpp<dpp_xor1>(a) < mine ? 1u : 0u;
  c += dpp<dpp_xor2>(a) < mine ? 1u : 0u;
  c += dpp<dpp_xor3>(a) < mine ? 1u : 0u;
  c += dpp<dpp_xor1>(b) < mine ? 1u : 0u;
  c += dpp<dpp_xor2>(b) < mine ? 1u : 0u;
  c += dpp<dpp_xor3>(b) < mine ? 1u : 0u;
  return c;
}

template<int ctrl>
__device__ __forceinline__ void least(uint32_t& hi, uint32_t& lo)
{
  const uint32_t oh = dpp<ctrl>(hi), ol = dpp<ctrl>(lo);
  const bool less = oh < hi || (oh == hi && ol < lo);
  hi = less ? oh : hi;
  lo = less ? ol : lo;
}

// The seeds of the lanes with `found`, appended to the tracklets and the tracks to follow in lane order.
__device__ __forceinline__ void append_seeds(
  const Team& team, SearchShared& sh, Counters& cn, const EventOutputs& o, bool found, unsigned h0, unsigned h1, unsigned h2)
{
  const Scan3 s = scan<1>(team, sh, cn, found);
  if (found) {
    const unsigned tn = (cn.ttf + s.r[0]) % max_tracks_to_follow;
    TrackletHits tl;
    tl.hits[0] = static_cast<uint16_t>(h0);
    tl.hits[1] = static_cast<uint16_t>(h1);
    tl.hits[2] = static_cast<uint16_t>(h2);
    o.tracklets[tn] = tl;
    o.ttf[tn] = bit_seed | tn;
    o.window_entries[tn & o.window_mask] = window_seed(bit_seed | tn, h0, h1 | (h2 << 16));
  }
  cn.ttf += s.t[0];
}

// One record of the seed log; features and logit as the scorer had them, or computed here.
template<typename H>
__device__ __forceinline__ void log_seed(
  const H& hits, const EventOutputs& o, unsigned module_pair, unsigned h0, unsigned h1, unsigned h2, const float* features,
  const float* logit)
{
  const unsigned slot = atomicAdd(o.seed_log.counter, 1u);
  if (slot >= o.seed_log.capacity) return;
  uint32_t* rec = o.seed_log.records + 5 * (size_t) slot;
  rec[0] = o.event_number;
  rec[1] = module_pair;
  rec[2] = h0;
  rec[3] = h1;
  rec[4] = h2;
  float f[n_seed_features];
  if (!features) seed_features(hits, h0, h1, h2, module_pair, f);
  float* fo = o.seed_log.features + n_seed_features * (size_t) slot;
#pragma unroll
  for (unsigned k = 0; k < n_seed_features; ++k) fo[k] = features ? features[k] : f[k];
  if (logit && o.seed_log.logits) o.seed_log.logits[slot] = *logit;
}

// SearchByTriplet.cu:298-446, ordered, with the (h1, h0) pairs spread over lanes.
//
// The reference walks, per h1, its h0 candidates in pendulum order and, per h0, the h2 window
// in phi order, keeping the first strictly smaller scatter. Here rounds of C = lanes / K unused h1
// hits (K = h0 candidates considered) give every (h1, h0) pair a lane: the K lanes of an h1 choose
// its h0 candidates together, each scores its own over the h2 window (first strict minimum), and
// they keep the first strict minimum over the candidates in pendulum order: the same pair the
// sequential double loop selects. The round's seeds are appended in h1 order. Nothing between the
// choice of the candidates and the append crosses a wave, so a round has one barrier (in the
// append's scan) where it had three, and the choice takes two keys per lane where one lane ranked
// and sorted eight or sixteen.
//
// Choice of the h0 candidates, the first K unused hits of the previous module pair in the pendulum
// order (SearchByTriplet.cu:348-370), from the ascending list `unused` (u entries) of the module
// pair's unused hits (relative indices) instead of a walk over every position: the pendulum
// visits position start + off, off = 0, +1, -1, +2, -2, ..., each wrapped once into [0, n), so
// position x gets rank 2d - 1 if d = (x - start) mod n lies in [1, n/2] (right of start), else
// 2 ((start - x) mod n) (left, start itself included); ranks are a permutation of 0..n-1, and the
// walk keeps the unused positions of the K smallest ranks, in rank order. Those are among the K
// nearest unused entries on either side of start in the circular list, so of the 2 K entries
// around its lower bound (all u if u <= 2 K) every lane takes two, and an entry with c < K
// smaller ranks is candidate number c.
template<bool count, int seed_mode, typename H>
__device__ __forceinline__ void track_seeding(
  WorkCount& wc,
  const H& hits,
  const SeedScratch& ss,
  SearchShared& sh,
  Counters& cn,
  const EventOutputs& o,
  const Team& team,
  const ModulePairData prev,
  const ModulePairData cur,
  const ModulePairData next,
  unsigned module_pair,
  float max_scatter,
  int16_t phi_tolerance,
  unsigned K)
{
  const unsigned log2K = K == 8 ? 3u : 2u; // K is 4 or 8
  const unsigned C = team.lanes >> log2K;
  const float dz_next = next.z[0] - prev.z[0];
  const unsigned tid = threadIdx.x;

  // The list of unused hits of the previous module pair (its writes are ordered
  // before the rounds by the barrier before them).
  // The first team.lanes hits of both lists are compacted by one scan (seeding marks no hit used,
  // so both read the flags the last forwarding left).
  const bool use_list = prev.hit_num <= ss.list_cap;
  const bool free0 = use_list && tid < prev.hit_num && !hits.used(prev.hit_start + tid);
  const bool act0 = tid < cur.hit_num && !hits.used(cur.hit_start + tid);
  const Scan3 first = scan<2>(team, sh, cn, free0, act0);
  if (free0) ss.unused[first.r[0]] = static_cast<uint16_t>(tid);
  if (use_list && tid < prev.hit_num) ss.before[tid] = static_cast<uint16_t>(first.r[0]);
  unsigned n_unused = first.t[0];
  if (use_list) {
    for (unsigned c0 = team.lanes; c0 < prev.hit_num; c0 += team.lanes) {
      const unsigned r = c0 + tid;
      const bool free_hit = r < prev.hit_num && !hits.used(prev.hit_start + r);
      const Scan3 sc = scan<1>(team, sh, cn, free_hit);
      if (free_hit) ss.unused[n_unused + sc.r[0]] = static_cast<uint16_t>(r);
      if (r < prev.hit_num) ss.before[r] = static_cast<uint16_t>(n_unused + sc.r[0]);
      n_unused += sc.t[0];
    }
  }

  // Unused hits of the current module pair, compacted in index order one chunk of team.lanes
  // hits at a time (dev_rel_indices in global memory, the chunk's list in LDS); the seeds of a
  // chunk are made before the next chunk, which keeps the h1 order of the reference.
  uint32_t base = 0;
  for (unsigned c0 = 0; c0 < cur.hit_num; c0 += team.lanes) {
    const unsigned r = c0 + tid;
    bool act = act0;
    unsigned rank = first.r[1], n_h1 = first.t[1];
    if (c0 != 0) {
      act = r < cur.hit_num && !hits.used(cur.hit_start + r);
      const Scan3 sc = scan<1>(team, sh, cn, act);
      rank = sc.r[0];
      n_h1 = sc.t[0];
    }
    if (act) {
      o.h1_indices[base + rank] = cur.hit_start + r;
      ss.h1_chunk[rank] = cur.hit_start + r;
    }
    base += n_h1;
    if (n_h1 == 0) continue;
    team.sync();
    phase_mark<count>(wc, phase_compaction);

    for (unsigned r0 = 0; r0 < n_h1; r0 += C) {
      Team::wave_fence(); // the last round's candidates have been read
      // 1. The K lanes of h1 number q choose its h0 candidates.
      const unsigned k = tid & (K - 1);
      const unsigned q = r0 + (tid >> log2K);
      const bool active = q < n_h1;
      const unsigned h1_index = ss.h1_chunk[active ? q : 0u];
      const Hit h1 = hits.load(h1_index);
      uint16_t* const choice = ss.h0 + (tid & ~(K - 1));
      unsigned n_h0;
      if (use_list) {
        n_h0 = min(n_unused, K);
        if (n_unused) {
          const unsigned n = prev.hit_num, u = n_unused;
          const unsigned start = mp_search<count>(hits, prev, h1.phi, wc);
          phase_mark<count>(wc, phase_seed1_search);
          const unsigned s0 = start >= n ? start - n : start;
          // The lower bound of s0 in the list: the number of unused positions below s0.
          const unsigned p = ss.before[s0];
          // key = rank << 16 | position (n <= 1024 on this path: rank < 2048, position < 1024).
          constexpr uint32_t none = 0xFFFFFFFFu;
          const bool all = u <= 2 * K;
          uint32_t key[2], x[2];
          bool has[2];
#pragma unroll
          for (unsigned e = 0; e < 2; ++e) {
            const unsigned j = 2 * k + e;
            const int around = static_cast<int>(p + j) - static_cast<int>(K);
            const unsigned ring = static_cast<unsigned>(
              around < 0 ? around + static_cast<int>(u) : (around >= static_cast<int>(u) ? around - static_cast<int>(u) : around));
            has[e] = !all || j < u;
            x[e] = ss.unused[all ? (j < u ? j : 0u) : ring];
          }
#pragma unroll
          for (unsigned e = 0; e < 2; ++e) {
            const unsigned d = x[e] >= s0 ? x[e] - s0 : x[e] + n - s0;
            const unsigned rk = d == 0 ? 0u : (d <= n / 2 ? 2 * d - 1 : 2 * (n - d));
            key[e] = has[e] ? (rk << 16 | x[e]) : none;
          }
          uint32_t below[2] = {below4(key[0], key[1], key[0]) + (key[1] < key[0] ? 1u : 0u),
                               below4(key[0], key[1], key[1]) + (key[0] < key[1] ? 1u : 0u)};
          if (K == 8) {
            const uint32_t m0 = dpp<dpp_half_mirror>(key[0]), m1 = dpp<dpp_half_mirror>(key[1]);
#pragma unroll
            for (unsigned e = 0; e < 2; ++e)
              below[e] += below4(m0, m1, key[e]) + (m0 < key[e] ? 1u : 0u) + (m1 < key[e] ? 1u : 0u);
          }
#pragma unroll
          for (unsigned e = 0; e < 2; ++e)
            if (active && has[e] && below[e] < K) choice[below[e]] = static_cast<uint16_t>(prev.hit_start + x[e]);
        }
      }
      else {
        // Module pairs beyond the list's capacity: the pendulum walk itself, start, +1, -1,
        // +2, -2, ... (each wrapped once into the module pair), by the h1's first lane.
        unsigned n_found = 0;
        if (active && k == 0) {
          const int n = static_cast<int>(prev.hit_num);
          int phi_index = static_cast<int>(mp_search<count>(hits, prev, h1.phi, wc));
          for (unsigned i = 0; i < prev.hit_num && n_found < K; ++i) {
            phi_index += (i & 1u) ? static_cast<int>(i) : -static_cast<int>(i);
            const int in_bounds = phi_index < 0 ? phi_index + n : (phi_index >= n ? phi_index - n : phi_index);
            const unsigned h0_index = prev.hit_start + static_cast<unsigned>(in_bounds);
            if (!hits.used(h0_index)) choice[n_found++] = static_cast<uint16_t>(h0_index);
          }
        }
        n_h0 = __shfl(n_found, lane_id() & ~(K - 1), wave_size);
      }
      Team::wave_fence();
      phase_mark<count>(wc, phase_seed1_pendulum);

      // 2. Lane k of h1 scores the pair (h1, h0 number k) over the h2 window (first strict
      // minimum), and the K lanes keep the least (scatter, k): the first strict minimum over
      // the h0 candidates in pendulum order. A scatter below max_scatter is a non-negative float,
      // ordered as its bit pattern.
      float best = max_scatter;
      uint32_t best_h2 = 0;
      if (active && k < n_h0) {
        const Hit h0 = hits.load(choice[k]);
        const float td = 1.0f / (h1.z - h0.z);
        const float txn = h1.x - h0.x;
        const float tyn = h1.y - h0.y;
        const float tx = txn * td;
        const float ty = tyn * td;
        const Line line {h0.x, h0.y, h0.z, tx, ty, extrapolated_phi<count>(wc, h0.x, h0.y, tx, ty, dz_next)};
        closest_hit<count, true>(wc, hits, next, line, phi_tolerance, best, best_h2);
      }
      uint32_t key_hi = __float_as_uint(best), key_lo = (k << 16) | best_h2;
      least<dpp_xor1>(key_hi, key_lo);
      least<dpp_xor2>(key_hi, key_lo);
      if (K == 8) least<dpp_half_mirror>(key_hi, key_lo); // quads agree: any lane of the other one
      const bool found = active && k == 0 && __uint_as_float(key_hi) < max_scatter;
      const unsigned best_h0 = choice[found ? key_lo >> 16 : 0u];
      phase_mark<count>(wc, phase_seed2);
      if constexpr (seed_mode == seed_mode_scored) {
        // Decided below, a group at a time.
        if (active && k == 0) ss.seed[q] = found ? best_h0 | key_lo << 16 : no_seed;
      }
      else {
        const uint16_t h2_index = static_cast<uint16_t>(key_lo & 0xFFFFu);
        if constexpr (seed_mode == seed_mode_log) {
          if (found) log_seed(hits, o, module_pair, best_h0, h1_index, h2_index, nullptr, nullptr);
        }
        // 3. The round's seeds in h1 order.
        append_seeds(team, sh, cn, o, found, best_h0, h1_index, h2_index);
      }
      phase_mark<count>(wc, phase_seed3);
    }
    if constexpr (seed_mode == seed_mode_scored) {
      // Seeds are decided in groups of C consecutive h1 hits (a wave, or half of one when
      // C = 32), lane t: the chunk's h1 number t. A seed is kept when its logit reaches the
      // threshold; a group whose seeds would all go keeps them (plain search as fallback).
      team.sync();
      uint32_t seed = no_seed;
      unsigned h1_index = 0;
      if (tid < n_h1) {
        seed = ss.seed[tid];
        h1_index = ss.h1_chunk[tid];
      }
      bool found = seed != no_seed;
      const unsigned best_h0 = seed & 0xFFFFu, h2_index = seed >> 16;
      float fp[n_seed_features];
#pragma unroll
      for (unsigned kk = 0; kk < n_seed_features; ++kk) fp[kk] = 0.f;
      if (found) seed_features(hits, best_h0, h1_index, h2_index, module_pair, fp);
      const uint64_t live = __ballot(found);
      const float logit = live ? scorer_logit(fp, live, *o.scorer) : 0.f;
      const bool keep = found && logit >= o.scorer_threshold;
      if (found && o.seed_log.counter) log_seed(hits, o, module_pair, best_h0, h1_index, h2_index, fp, &logit);
      const uint64_t group = C >= wave_size ? ~0ull : (((1ull << C) - 1) << (lane_id() / C * C));
      if (__ballot(keep) & group) found = keep;
      append_seeds(team, sh, cn, o, found, best_h0, h1_index, h2_index);
      phase_mark<count>(wc, phase_seed3);
    }
  }
  cn.local_hits = base;
}

// SearchByTriplet.cu:451-609, ordered.
template<bool count, typename H>
__device__ __forceinline__ void track_forwarding(
  WorkCount& wc,
  const H& hits,
  SearchShared& sh,
  Counters& cn,
  const EventOutputs& o,
  const Team& team,
  const ModulePairData next,
  unsigned prev_ttf,
  unsigned diff_ttf,
  bool window,
  int16_t phi_tolerance,
  float max_scatter,
  unsigned max_skipped_modules)
{
  for (unsigned c = 0; c < diff_ttf; c += team.lanes) {
    const unsigned e = c + threadIdx.x;
    bool promote = false, reinsert = false, three = false;
    bool is_seed = false;
    unsigned skipped = 0; // the entry's bit_skipped field, in place
    unsigned number_of_hits = 0;
    bool found = false;
    uint32_t best_h2 = 0;
    unsigned first_hit = 0;
    unsigned track_number = 0;
    bool valid = false;
    unsigned h0_num = 0, h1_num = 0;
    if (e < diff_ttf) {
      const unsigned q = (prev_ttf + e) % max_tracks_to_follow;
      if (window) {
        // The entry and its track's last hits from LDS (written with the entry).
        const uint2 w = o.window_entries[q & o.window_mask];
        is_seed = (w.x & bit_seed) != 0;
        skipped = w.x & bit_skipped;
        h0_num = w.y & 0xFFFFu;
        h1_num = w.y >> 16;
        first_hit = (w.x >> seed_first_pos) & 0xFFFFu;
        number_of_hits = is_seed ? 3u : (w.x >> track_hits_pos) & 31u;
        track_number = w.x & (is_seed ? max_tracks_to_follow - 1 : window_track_number);
        // Guards that only matter once the slots of an event have overflowed (status raised).
        valid = is_seed || (track_number < o.track_capacity && number_of_hits >= 3 && number_of_hits < max_track_size);
      }
      else {
        uint32_t full = o.ttf[q];
        track_number = full & bit_track_number;
        is_seed = (full & bit_seed) != 0;
        const uint16_t* t_hits = nullptr;
        if (is_seed) {
          valid = track_number < max_tracks_to_follow;
          if (valid) t_hits = o.tracklets[track_number].hits;
          number_of_hits = 3;
        }
        else if (track_number < o.track_capacity) {
          // Guards that only matter once the slots of an event have overflowed (status raised).
          t_hits = o.tracks[track_number].hits;
          number_of_hits = o.tracks[track_number].hitsNum;
          valid = number_of_hits >= 3 && number_of_hits < max_track_size;
        }
        if (valid) {
          h0_num = t_hits[number_of_hits - 2];
          h1_num = t_hits[number_of_hits - 1];
          first_hit = t_hits[0];
        }
        // These reads are waited for here. Left pending, they would make the code after the
        // branch wait for all memory traffic, which on the usual path (the window) is the wave's
        // stores: a round trip to memory several times per module pair.
        asm volatile("" : "+v"(full), "+v"(h0_num), "+v"(h1_num), "+v"(first_hit), "+v"(number_of_hits));
        skipped = full & bit_skipped;
      }
    }
    if (valid) {
      const Hit h0 = hits.load(h0_num), h1 = hits.load(h1_num);
      const float td = 1.0f / (h1.z - h0.z);
      const float txn = h1.x - h0.x;
      const float tyn = h1.y - h0.y;
      const float tx = txn * td;
      const float ty = tyn * td;
      float best_fit = max_scatter;
      const Line line {h0.x, h0.y, h0.z, tx, ty,
                       extrapolated_phi<count>(wc, h0.x, h0.y, tx, ty, (h0.odd ? next.z[1] : next.z[0]) - h0.z)};
      found = closest_hit<count, false>(wc, hits, next, line, phi_tolerance, best_fit, best_h2);
      if (found) {
        promote = number_of_hits == 3;
        reinsert = number_of_hits + 1 < max_track_size;
      }
      else if ((skipped >> skipped_pos) < max_skipped_modules) {
        reinsert = true;
      }
      else if (number_of_hits == 3) {
        three = true;
      }
    }
    const Scan3 s = scan<3>(team, sh, cn, promote, reinsert, three);
    cn.extended += __popcll(__ballot(found && !promote));
    if (valid) {
      if (found) {
        hits.mark_used(best_h2);
        if (promote) {
          hits.mark_used(first_hit);
          hits.mark_used(h0_num);
          hits.mark_used(h1_num);
          track_number = cn.n_tracks + s.r[0];
          if (track_number < o.track_capacity) {
            TrackHits& t = o.tracks[track_number];
            t.hits[0] = static_cast<uint16_t>(first_hit);
            t.hits[1] = static_cast<uint16_t>(h0_num);
            t.hits[2] = static_cast<uint16_t>(h1_num);
            t.hits[3] = static_cast<uint16_t>(best_h2);
            t.hitsNum = 4;
          }
        }
        else {
          TrackHits& t = o.tracks[track_number];
          t.hits[number_of_hits] = static_cast<uint16_t>(best_h2);
          t.hitsNum = number_of_hits + 1;
        }
      }
      if (reinsert) {
        // Found: the track with the new hit. Not found: the same entry, one module more skipped.
        // A promoted track beyond the slots of its event is skipped when read back.
        const unsigned p = (cn.ttf + s.r[1]) % max_tracks_to_follow;
        const unsigned last2 = found ? h1_num | (best_h2 << 16) : h0_num | (h1_num << 16);
        // The field holds up to seven skipped modules; a limit beyond that is none (counting on would
        // make a track's entry a seed's).
        const uint32_t skips = found ? 0u : min(skipped + (1u << skipped_pos), bit_skipped);
        const bool seed = is_seed && !found;
        const uint32_t full = skips | (seed ? bit_seed : 0u) | track_number;
        o.ttf[p] = full;
        o.window_entries[p & o.window_mask] =
          seed ? window_seed(full, first_hit, last2) : window_track(skips, track_number, number_of_hits + (found ? 1u : 0u), last2);
      }
      if (three) {
        const unsigned p = cn.three + s.r[2];
        if (p < o.track_capacity) {
          TrackletHits t;
          t.hits[0] = static_cast<uint16_t>(first_hit);
          t.hits[1] = static_cast<uint16_t>(h0_num);
          t.hits[2] = static_cast<uint16_t>(h1_num);
          o.three_hit_tracks[p] = t;
        }
      }
    }
    // Chunks need no barrier between them: a chunk writes ring slots at and beyond the
    // counter, reads only the slots before it (distinct unless the ring overflows, which is
    // reported), and the used flags it sets are read by seeding after the caller's barrier.
    cn.n_tracks += s.t[0];
    cn.ttf += s.t[1];
    cn.three += s.t[2];
    if (cn.n_tracks > o.track_capacity) cn.status |= status_track_slots_overflow;
    if (cn.three > o.track_capacity) cn.status |= status_three_hit_slots_overflow;
  }
}

template<bool count, int seed_mode, typename H>
__device__ __forceinline__ void search_event(
  WorkCount& wc,
  const H& hits,
  const SeedScratch& ss,
  SearchShared& sh,
  Counters& cn,
  const EventOutputs& o,
  const Team& team,
  float phi_tolerance_f,
  float max_scatter,
  unsigned max_skipped_modules)
{
  // Module pairs are visited from the last one upstream: seeding on (first, first - 1,
  // first - 2), forwarding into first - 2 (SearchByTriplet.cu:160-236).
  phase_mark<count>(wc, phase_other);
  const int16_t phi_tolerance = f32_to_i16(phi_tolerance_f * convert_factor_i16);
  unsigned first_module_pair = n_module_pairs - 1;
  unsigned last_ttf = 0;
  ModulePairData prev = module_pair_data(sh, first_module_pair), cur = module_pair_data(sh, first_module_pair - 1),
                 next = module_pair_data(sh, first_module_pair - 2);
  for (;;) {
    // One inlined copy of track_seeding for both numbers of h0 candidates keeps the code small.
    track_seeding<count, seed_mode>(
      wc, hits, ss, sh, cn, o, team, prev, cur, next, first_module_pair - 1, max_scatter, phi_tolerance,
      first_module_pair == n_module_pairs - 1 ? initial_seeding_h0_candidates : seeding_h0_candidates);
    --first_module_pair;
    if (first_module_pair <= 1) break;
    prev = cur;
    cur = next;
    next = module_pair_data(sh, first_module_pair - 2);
    const unsigned prev_ttf = last_ttf;
    last_ttf = cn.ttf;
    const unsigned diff_ttf = last_ttf - prev_ttf;
    if (diff_ttf >= max_tracks_to_follow) cn.status |= status_ttf_ring_overflow;
    // The positions read here, [prev_ttf, last_ttf), and every position written from their
    // writing to their reading (this forwarding reinserts at most diff_ttf entries) span at most
    // 2 diff_ttf positions: within the LDS window they are all distinct. Beyond it the ring is
    // read back from HBM, after a fence that makes this workgroup's ring writes visible to it.
    const bool window = 2 * diff_ttf <= o.window;
    if (!window) __threadfence_block();
    // Orders the ring slots and tracklets written by the last seeding round before they are
    // read (seeding rounds end right after their writes, without a barrier).
    team.sync();
    track_forwarding<count>(
      wc, hits, sh, cn, o, team, next, prev_ttf, diff_ttf, window, phi_tolerance, max_scatter, max_skipped_modules);
    team.sync();
    phase_mark<count>(wc, phase_forwarding);
  }
  team.sync();
  const unsigned prev_ttf = last_ttf;
  last_ttf = cn.ttf;
  const unsigned diff_ttf = last_ttf - prev_ttf;
  if (diff_ttf >= max_tracks_to_follow) cn.status |= status_ttf_ring_overflow;
  // Both the entries (where they have left the window) and the tracklets are read back from HBM.
  const bool window = diff_ttf <= o.window; // nothing is written while these are read
  __threadfence_block();
  team.sync();
  for (unsigned c = 0; c < diff_ttf; c += team.lanes) {
    const unsigned e = c + threadIdx.x;
    bool seed = false;
    uint32_t full = 0;
    if (e < diff_ttf) {
      const unsigned q = (prev_ttf + e) % max_tracks_to_follow;
      full = window ? o.window_entries[q & o.window_mask].x : o.ttf[q];
      seed = (full & bit_seed) != 0;
    }
    const Scan3 s = scan<1>(team, sh, cn, seed);
    if (seed) {
      const unsigned p = cn.three + s.r[0];
      if (p < o.track_capacity) o.three_hit_tracks[p] = o.tracklets[full & (max_tracks_to_follow - 1)];
    }
    cn.three += s.t[0];
    if (cn.three > o.track_capacity) cn.status |= status_three_hit_slots_overflow;
  }
}

struct SearchArgs {
  const uint32_t* event_list;
  const uint32_t* number_of_events;
  const char* sorted_container;
  const uint32_t* offsets_estimated_input_size;
  const uint32_t* module_cluster_num;
  const Geometry* geometry;
  TrackHits* tracks;
  TrackletHits* tracklets;
  uint32_t* tracks_to_follow;
  TrackletHits* three_hit_tracks;
  uint8_t* hit_used;
  uint32_t* atomics_velo;
  uint16_t* rel_indices;
  uint32_t* number_of_velo_tracks;
  uint32_t* status;
  float phi_tolerance;
  float max_scatter;
  unsigned max_skipped_modules;
  unsigned lds_hits;
  unsigned hits_per_wave; // waves of a workgroup that work on an event: one more for every so many hits; 0: all
  unsigned long long* work_stats;
  unsigned long long* event_clock;
  unsigned n_list;
  uint32_t* work_counter;
  SeedLog seed_log;
  const float* scorer_params;
  float scorer_threshold;
  unsigned window;
  unsigned list_cap;
  // Optional: the three-hit filter at the end of each event, with its outputs and the event's track hits.
  TrackletHits* three_hit_tracks_output;
  uint32_t* number_of_three_hit_tracks_output;
  uint32_t* event_track_hits;
  float max_chi2;
};

// ThreeHitTracksFilter.cu:48-107
__device__ __forceinline__ float means_square_fit_chi2(const Hit& a, const Hit& b, const Hit& c)
{
  float s0, sx, sz, sxz, sz2, u0, uy, uz, uyz, uz2;
  s0 = sx = sz = sxz = sz2 = 0.0f;
  u0 = uy = uz = uyz = uz2 = 0.0f;
  const float xs[3] = {a.x, b.x, c.x}, ys[3] = {a.y, b.y, c.y}, zs[3] = {a.z, b.z, c.z};
#pragma unroll
  for (unsigned h = 0; h < 3; ++h) {
    const float x = xs[h], y = ys[h], z = zs[h];
    const float wx = param_w;
    const float wx_t_x = wx * x;
    const float wx_t_z = wx * z;
    s0 += wx;
    sx += wx_t_x;
    sz += wx_t_z;
    sxz += wx_t_x * z;
    sz2 += wx_t_z * z;
    const float wy = param_w;
    const float wy_t_y = wy * y;
    const float wy_t_z = wy * z;
    u0 += wy;
    uy += wy_t_y;
    uz += wy_t_z;
    uyz += wy_t_y * z;
    uz2 += wy_t_z * z;
  }
  const float dens = 1.0f / (sz2 * s0 - sz * sz);
  const float state_tx = (sxz * s0 - sx * sz) * dens;
  const float state_x = (sx * sz2 - sxz * sz) * dens;
  const float denu = 1.0f / (uz2 * u0 - uz * uz);
  const float state_ty = (uyz * u0 - uy * uz) * denu;
  const float state_y = (uy * uz2 - uyz * uz) * denu;
  float chi2 = 0.0f;
#pragma unroll
  for (unsigned h = 0; h < 3; ++h) {
    const float z = zs[h];
    const float x = state_x + state_tx * z;
    const float y = state_y + state_ty * z;
    const float dx = x - xs[h];
    const float dy = y - ys[h];
    chi2 += dx * dx * param_w + dy * dy * param_w;
  }
  return chi2 * 0.5f;
}

// The three-hit filter (ThreeHitTracksFilter.cu:109-169, ordered output) on the event's own
// three-hit tracks, with the hits and their flags where the search has them, and the number of
// hits of the event's tracks (four for each track, one for each extension, three for each kept
// three-hit track): what the filter, the track-hit count and two scans over the tracks took a
// launch each for. Where the ring of tracks to follow has overflowed, an entry can be read twice and
// its track extended by two lanes at once, so the stored tracks are counted themselves: the hits
// are placed by what each track holds.
template<typename H>
__device__ __forceinline__ void finish_event(
  const H& hits, const Team& team, SearchShared& sh, Counters& cn, const EventOutputs& o, const SearchArgs& a, unsigned toff)
{
  if (!a.three_hit_tracks_output) return;
  const bool overflow = cn.status & status_ttf_ring_overflow;
  const unsigned n_tracks = min(cn.n_tracks, o.track_capacity);
  if (lane_id() == 0 && cn.extended && !overflow) atomicAdd(&sh.extended, cn.extended);
  __threadfence_block(); // other lanes wrote the tracks
  team.sync();
  if (overflow) {
    for (unsigned i = threadIdx.x; i < n_tracks; i += team.lanes) atomicAdd(&sh.extended, o.tracks[i].hitsNum - 4u);
    team.sync();
  }
  const unsigned n_in = min(cn.three, o.track_capacity);
  TrackletHits* out = a.three_hit_tracks_output + toff;
  unsigned kept = 0;
  for (unsigned c = 0; c < n_in; c += team.lanes) {
    const unsigned i = c + threadIdx.x;
    bool keep = false;
    TrackletHits t;
    if (i < n_in) {
      t = o.three_hit_tracks[i];
      const Hit h0 = hits.load(t.hits[0]), h1 = hits.load(t.hits[1]), h2 = hits.load(t.hits[2]);
      keep = !(h0.used || h1.used || h2.used) && means_square_fit_chi2(h0, h1, h2) < a.max_chi2;
    }
    const Scan3 s = scan<1>(team, sh, cn, keep);
    if (keep) out[kept + s.r[0]] = t;
    kept += s.t[0];
  }
  if (threadIdx.x == 0) {
    a.number_of_three_hit_tracks_output[o.event_number] = kept;
    a.event_track_hits[o.event_number] = 4 * n_tracks + sh.extended + 3 * kept;
  }
}

// One workgroup per event, or (persistent, launched with a work counter) a resident grid whose
// workgroups take the next event slot from the counter until the slots run out; the persistent
// grid is an instantiation of its own, so the one-event kernel keeps no loop state live. Dynamic
// LDS: the seeding scratch (seed_scratch_bytes_per_lane per lane), the LDS window of the ring of
// tracks to follow (the ring itself, 2048 x u32, is written through to HBM), the list of
// unused hits of the previous module pair and, per position, the number of unused hits before
// it (list_cap x u16 each), the module pairs' phi bucket tables, then `lds_hits` hits of 16 bytes.
// Events with up to 16/3 x lds_hits hits keep phi and the
// flags in LDS and read coordinates from global memory; larger events run on global memory.
// Bound by the latency of an event's chain of 25 dependent seeding and forwarding steps and, with
// many events in flight, by VALU issue.
// The `count` instantiation also accumulates the work counters into work_stats[4] (one
// atomic per wave). With event_clock, each workgroup stores at event_clock[10 * event_number]
// its event's start and end time (wall clock ticks) and, in the counting instantiation, the
// ticks spent in each Phase.
// waves_per_simd: what the registers leave room for. The scored search takes 155 and runs three; with
// four (128 registers, 26 values spilled) an event takes 5 % longer, which pays where more events
// wait than three a CU.
template<bool count, int seed_mode, bool persistent, unsigned waves_per_simd = seed_mode == seed_mode_scored ? 3 : 1>
__global__ void __launch_bounds__(seed_mode == seed_mode_scored ? 256 : 1024, waves_per_simd)
  k_search_by_triplet(const SearchArgs a)
{
  extern __shared__ __align__(16) char dyn_all[];
  __shared__ SearchShared sh;
  __shared__ unsigned s_slot;
  WorkCount wc;
  SeedScratch ss;
  ss.seed = reinterpret_cast<uint32_t*>(dyn_all);
  ss.h0 = reinterpret_cast<uint16_t*>(ss.seed + blockDim.x);
  ss.h1_chunk = ss.h0 + blockDim.x;
  uint2* window_entries = reinterpret_cast<uint2*>(ss.h1_chunk + blockDim.x);
  ss.unused = reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(window_entries) + window_bytes(a.window));
  ss.before = ss.unused + a.list_cap;
  ss.list_cap = a.list_cap;
  uint8_t* phi_tables = reinterpret_cast<uint8_t*>(ss.before + a.list_cap);
  char* dyn = reinterpret_cast<char*>(phi_tables + phi_tables_bytes);
  ScorerLds* scorer = nullptr;
  if constexpr (seed_mode == seed_mode_scored) {
    scorer = reinterpret_cast<ScorerLds*>(dyn + (size_t) a.lds_hits * search_bytes_per_hit);
    load_scorer(a.scorer_params, *scorer);
    __syncthreads();
  }
  const unsigned total = a.offsets_estimated_input_size[n_module_pairs * a.number_of_events[0]];
  // One event: slot `slot` of the event list (the whole workgroup, uniform).
  const auto process_event = [&](unsigned slot) {
    const unsigned long long t_start = a.event_clock ? wall_clock64() : 0ull;
    wc.last = t_start;
    const unsigned event_number = a.event_list ? a.event_list[slot] : slot;
    const unsigned n_events = a.number_of_events[0];
    const uint32_t* mhs = a.offsets_estimated_input_size + event_number * n_module_pairs;
    const uint32_t* mhn = a.module_cluster_num + event_number * n_module_pairs;
    const unsigned hit_offset = mhs[0];
    const unsigned n_hits = mhs[n_module_pairs] - hit_offset;
    Team team;
    team.wave = __builtin_amdgcn_readfirstlane(threadIdx.x / wave_size);
    team.waves = blockDim.x / wave_size;
    if constexpr (!persistent && seed_mode != seed_mode_scored) {
      if (a.hits_per_wave) team.waves = min(team.waves, n_hits / a.hits_per_wave + 1);
      if (team.wave >= team.waves) return;
    }
    team.lanes = team.waves * wave_size;
    const Clusters cc {const_cast<char*>(a.sorted_container), total};

    const unsigned toff = track_offset(a.offsets_estimated_input_size, event_number);
    const unsigned container = track_container_size(total, n_events);
    const unsigned next_off =
      event_number + 1 < n_events ? track_offset(a.offsets_estimated_input_size, event_number + 1) : container;
    EventOutputs o;
    o.tracks = a.tracks + toff;
    o.three_hit_tracks = a.three_hit_tracks + toff;
    o.tracklets = a.tracklets + (size_t) event_number * max_tracks_to_follow;
    o.ttf = a.tracks_to_follow + (size_t) event_number * max_tracks_to_follow;
    o.window_entries = window_entries;
    o.h1_indices = a.rel_indices + hit_offset;
    o.event_number = event_number;
    o.seed_log = a.seed_log;
    o.scorer = scorer;
    o.scorer_threshold = a.scorer_threshold;
    o.window = a.window;
    o.window_mask = a.window - 1;
    // Slots of this event; the reference lets a busy event run into its neighbour's slots, here
    // nothing is written past the container and the overflow is reported.
    o.track_capacity = min(next_off > toff ? next_off - toff : 0u, container - min(toff, container));

    Counters cn;
    if (threadIdx.x == 0) sh.extended = 0;
    cn.status = n_hits > 65536u ? status_hit_index_overflow : 0u;
    if (threadIdx.x < n_module_pairs) {
      const unsigned m = threadIdx.x;
      sh.mp[m].hit_start = mhs[m] - hit_offset;
      sh.mp[m].hit_num = mhn[m];
      sh.mp[m].z[0] = a.geometry->module_zs[2 * m];
      sh.mp[m].z[1] = a.geometry->module_zs[2 * m + 1];
      sh.mp[m].table = mhn[m] <= 255u ? m * phi_table_stride : no_phi_table;
    }
    const uint32_t* gids = cc.ids() + hit_offset;
    const int16_t* gph = cc.phis() + hit_offset;
    const float* gxyz = cc.xyz() + 3 * (size_t) hit_offset;
    uint8_t* gused = a.hit_used + hit_offset;
    // The ring window holds nothing yet: it is the tables' histograms.
    uint32_t* const hist = reinterpret_cast<uint32_t*>(window_entries);
    const unsigned hist_waves = window_bytes(a.window) / hist_bytes;
    if (n_hits <= a.lds_hits) {
      uint4* hit = reinterpret_cast<uint4*>(dyn);
      // Two hits per lane and round, every load issued before the first store waits (the
      // scheduler would otherwise wait out one memory round trip per field).
      for (unsigned i0 = threadIdx.x; i0 < n_hits; i0 += 2 * team.lanes) {
        const unsigned i1 = i0 + team.lanes < n_hits ? i0 + team.lanes : i0;
        const float x0 = gxyz[3 * i0], y0 = gxyz[3 * i0 + 1], z0 = gxyz[3 * i0 + 2];
        const float x1 = gxyz[3 * i1], y1 = gxyz[3 * i1 + 1], z1 = gxyz[3 * i1 + 2];
        const int16_t p0 = gph[i0], p1 = gph[i1];
        const uint32_t id0 = gids[i0], id1 = gids[i1];
        __builtin_amdgcn_sched_barrier(0);
        const auto word = [](int16_t p, uint32_t id) {
          return static_cast<uint16_t>(p) | (module_parity(id) ? uint32_t(flag_odd) << 16 : 0u);
        };
        hit[i0] = make_uint4(__float_as_uint(x0), __float_as_uint(y0), __float_as_uint(z0), word(p0, id0));
        hit[i1] = make_uint4(__float_as_uint(x1), __float_as_uint(y1), __float_as_uint(z1), word(p1, id1));
      }
      team.sync();
      const LdsHits hits {hit, phi_tables};
      build_phi_tables(hits, sh.mp, phi_tables, hist, hist_waves, team);
      team.sync();
      search_event<count, seed_mode>(wc, hits, ss, sh, cn, o, team, a.phi_tolerance, a.max_scatter, a.max_skipped_modules);
      team.sync();
      for (unsigned i = threadIdx.x; i < n_hits; i += team.lanes) gused[i] = hits.used(i) ? 1 : 0;
      finish_event(hits, team, sh, cn, o, a, toff);
    }
    else if (mixed_bytes_per_hit * n_hits <= search_bytes_per_hit * a.lds_hits) {
      int16_t* ph = reinterpret_cast<int16_t*>(dyn);
      uint8_t* flags = reinterpret_cast<uint8_t*>(ph + n_hits);
      for (unsigned i0 = threadIdx.x; i0 < n_hits; i0 += 2 * team.lanes) {
        const unsigned i1 = i0 + team.lanes < n_hits ? i0 + team.lanes : i0;
        const int16_t p0 = gph[i0], p1 = gph[i1];
        const uint32_t id0 = gids[i0], id1 = gids[i1];
        __builtin_amdgcn_sched_barrier(0);
        ph[i0] = p0;
        flags[i0] = module_parity(id0) ? flag_odd : 0;
        ph[i1] = p1;
        flags[i1] = module_parity(id1) ? flag_odd : 0;
      }
      cn.status |= status_lds_fallback;
      team.sync();
      const MixedHits hits {gxyz, ph, flags, phi_tables};
      build_phi_tables(hits, sh.mp, phi_tables, hist, hist_waves, team);
      team.sync();
      search_event<count, seed_mode>(wc, hits, ss, sh, cn, o, team, a.phi_tolerance, a.max_scatter, a.max_skipped_modules);
      team.sync();
      for (unsigned i = threadIdx.x; i < n_hits; i += team.lanes) gused[i] = flags[i] & flag_used;
      finish_event(hits, team, sh, cn, o, a, toff);
    }
    else {
      for (unsigned i = threadIdx.x; i < n_hits; i += team.lanes) gused[i] = 0;
      cn.status |= status_lds_fallback;
      __threadfence_block();
      team.sync();
      const GlobalHits hits {gxyz, gph, gused, gids, phi_tables};
      build_phi_tables(hits, sh.mp, phi_tables, hist, hist_waves, team);
      team.sync();
      // The hits leave their LDS to the lists: such events are the ones whose module pairs are long.
      SeedScratch long_lists = ss;
      if (4 * a.lds_hits > a.list_cap) {
        long_lists.list_cap = min(4 * a.lds_hits, unused_list_cap);
        long_lists.unused = reinterpret_cast<uint16_t*>(dyn);
        long_lists.before = long_lists.unused + long_lists.list_cap;
      }
      search_event<count, seed_mode>(
        wc, hits, long_lists, sh, cn, o, team, a.phi_tolerance, a.max_scatter, a.max_skipped_modules);
      __threadfence_block(); // the used flags are read back from global memory
      team.sync();
      finish_event(hits, team, sh, cn, o, a, toff);
    }
    if constexpr (count) {
      // Wave reduction, then one atomic per wave.
      unsigned long long v[4] = {wc.seed_eval, wc.fwd_eval, wc.extrap, wc.steps};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
#pragma unroll
        for (unsigned d = 32; d > 0; d >>= 1) v[k] += __shfl_xor(v[k], d, wave_size);
        if (lane_id() == 0 && v[k]) atomicAdd(a.work_stats + k, v[k]);
      }
      wc.seed_eval = wc.fwd_eval = wc.extrap = wc.steps = 0;
    }
    if (threadIdx.x == 0) {
      uint32_t* at = a.atomics_velo + event_number * num_atomics;
      at[atomic_three_hit] = cn.three;
      at[atomic_ttf] = cn.ttf;
      at[atomic_local_hits] = cn.local_hits;
      a.number_of_velo_tracks[event_number] = min(cn.n_tracks, o.track_capacity);
      if (cn.status && a.status) atomicOr(a.status, cn.status);
      if (a.event_clock) {
        unsigned long long* ec = a.event_clock + event_clock_words * event_number;
        const unsigned long long t_end = wall_clock64();
        ec[0] = t_start;
        ec[1] = t_end;
        if constexpr (count) {
          phase_mark<count>(wc, phase_other);
#pragma unroll
          for (int k = 0; k < n_phases; ++k) {
            ec[2 + k] = wc.phase[k];
            wc.phase[k] = 0;
          }
        }
      }
    }
    if constexpr (persistent) __syncthreads(); // the next event reuses the LDS
  };
  if constexpr (persistent) {
    for (;;) {
      if (threadIdx.x == 0) s_slot = atomicAdd(a.work_counter, 1u);
      __syncthreads();
      const unsigned slot = s_slot;
      __syncthreads();
      if (slot >= a.n_list) break;
      process_event(slot);
    }
  }
  else {
    if (blockIdx.x < a.n_list) process_event(blockIdx.x);
  }
}

// ThreeHitTracksFilter.cu:109-169, ordered output.
__global__ void k_three_hit_filter(
  const uint32_t* event_list,
  const uint32_t* number_of_events,
  const char* sorted_container,
  const uint32_t* offsets_estimated_input_size,
  const TrackletHits* input_all,
  const uint32_t* atomics_all,
  const uint8_t* hit_used_all,
  TrackletHits* output_all,
  uint32_t* number_of_output,
  float max_chi2)
{
  __shared__ uint32_t scan[16];
  const unsigned event_number = event_list ? event_list[blockIdx.x] : blockIdx.x;
  const unsigned n_events = number_of_events[0];
  const unsigned total = offsets_estimated_input_size[n_module_pairs * n_events];
  const unsigned hit_offset = offsets_estimated_input_size[event_number * n_module_pairs];
  const Clusters cc {const_cast<char*>(sorted_container), total};
  const unsigned toff = track_offset(offsets_estimated_input_size, event_number);
  const TrackletHits* in = input_all + toff;
  const unsigned container = track_container_size(total, n_events);
  const unsigned next_off =
    event_number + 1 < n_events ? track_offset(offsets_estimated_input_size, event_number + 1) : container;
  const unsigned capacity = min(next_off > toff ? next_off - toff : 0u, container - min(toff, container));
  // The count can only exceed the event's slots once they overflowed (a status bit is set then).
  const unsigned n_in = min(atomics_all[event_number * num_atomics + atomic_three_hit], capacity);
  TrackletHits* out = output_all + toff;
  unsigned base = 0;
  for (unsigned c = 0; c < n_in; c += blockDim.x) {
    const unsigned i = c + threadIdx.x;
    bool keep = false;
    TrackletHits t;
    if (i < n_in) {
      t = in[i];
      const GlobalHits hits {cc.xyz() + 3 * (size_t) hit_offset, cc.phis() + hit_offset,
                             const_cast<uint8_t*>(hit_used_all) + hit_offset, cc.ids() + hit_offset, nullptr};
      const Hit h0 = hits.load(t.hits[0]), h1 = hits.load(t.hits[1]), h2 = hits.load(t.hits[2]);
      keep = !(h0.used || h1.used || h2.used) && means_square_fit_chi2(h0, h1, h2) < max_chi2;
    }
    uint32_t kept;
    const uint32_t r = block_flag_scan(keep, scan, &kept);
    if (keep) out[base + r] = t;
    base += kept;
  }
  if (threadIdx.x == 0) number_of_output[event_number] = base;
}

constexpr size_t lds_per_cu = 160 * 1024;

// Launch geometry: the seeding scratch, the ring window, the unused-hit list, then the hits.
static constexpr size_t launch_lds(unsigned block, unsigned lds_hits, unsigned window, unsigned list_cap)
{
  return seed_scratch_bytes_per_lane * (size_t) block + window_bytes(window) + 2 * 2 * (size_t) list_cap +
         phi_tables_bytes + (size_t) lds_hits * search_bytes_per_hit;
}
size_t search_dynamic_lds(unsigned block, unsigned lds_hits, unsigned window, unsigned list_cap)
{
  return launch_lds(block, lds_hits, window, list_cap);
}
// The workgroups of a launch that the LDS of a CU holds.
static constexpr unsigned workgroups_a_cu(unsigned block, unsigned lds_hits, unsigned window, unsigned list_cap)
{
  return static_cast<unsigned>(lds_per_cu / (launch_lds(block, lds_hits, window, list_cap) + sizeof(SearchShared) + 16));
}
static_assert(workgroups_a_cu(64, search_default_lds_hits, max_ring_window_knob, unused_list_cap) == 4, "default hits");
static_assert(workgroups_a_cu(256, search_default_lds_hits, ring_window, unused_list_cap) == 3, "default hits");

// Shape of a launch whose workgroup size is left to it: lanes, hits in LDS, ring window,
// unused-hit list, and the hits of an event per working wave.
struct SearchShape {
  unsigned block, lds_hits, window, list_cap, hits_per_wave;
};
constexpr unsigned very_crowded_hits = 5600; // 36 collisions
// Few events: every event has its LDS to itself (two workgroups fit a CU), and the launch lasts as
// long as its largest event: four waves for events from 2100 hits on, all hits in LDS (200 events
// of up to 1700 hits: 123 us against 142 us with 1500 hits in LDS and coordinates from memory), lists
// for module pairs of 1024 hits (200 events at nu = 45: 682 us; 942 with lists of 512). Up to
// 1024 very crowded ones take it too (600 events at nu = 60: 1065 us; 1373 with the next shape).
// Crowded ones: what four workgroups a CU leave, with phi and flags of 8800 hits in it and the long
// lists (1000 events at nu = 30: 592 us, 884 with the next shape; 2000 at nu = 45: 1426, 1982; 5000 at
// nu = 30: 1942, 2870 with the last).
// Up to 1024: all of them have to be in flight at once, so the LDS is what four
// workgroups a CU leave (1000 pile-up events: 174 us; with 2240 hits and three a CU 243 us; with
// 128-lane workgroups 310 us, with 512 lanes 213 us when the pass took 210 us). Up to 4096: five
// workgroups a CU, which their registers allow (whole passes with five and four: 1100 one-vertex events
// 282 and 346 us, 3000 pile-up events 655 and 683 us, 2000 stress events 835 and 844 us). Beyond, the
// workgroups stream through the chip and the most resident waves win: little LDS and two waves per event,
// up to 6144 events as workgroups of four waves whose last two end at once unless the event is
// large, since one large event of two waves outlasts these slices (5000 one-vertex events: 457 us, 411
// with two; with 1 % of them at nu = 60: 909, 1468). 20 000 events: 1.45 ms; 1.73 ms with 256
// lanes, 2.46 ms with 1500 hits in LDS, 4.32 ms with 256 lanes and 1760 hits before.
static SearchShape search_shape(unsigned n_events, unsigned mean_hits)
{
  if (n_events <= (mean_hits > very_crowded_hits ? 1024u : 512u)) return {256, 3072, 1024, 1024, 700};
  if (mean_hits > crowded_hits) return {256, 1650, 512, 1024, 700};
  if (n_events <= 1024) return {256, 1500, 1024, 512, 700};
  if (n_events <= 4096) return {256, 1180, 512, 512, 700};
  if (n_events <= 6144) return {256, 384, 512, 512, 1100};
  return {128, 384, 512, 512, 0};
}
static_assert(workgroups_a_cu(256, 3072, 1024, 1024) == 2 && workgroups_a_cu(256, 1650, 512, 1024) == 4 &&
              workgroups_a_cu(256, 1500, 1024, 512) == 4 && workgroups_a_cu(256, 1180, 512, 512) == 5, "the shapes' residency");

// The same for the scored search, whose workgroups have 256 lanes (their size is part of the pruning
// rule): 12 waves of it fit a CU by its registers, so up to 768 events are in flight at once and have
// the LDS of three workgroups (300 one-vertex events, whole pass: 232 us; 257 with 1760 hits and a
// window and a list of 1024; 200 events at nu = 45, search: 968 us; 1064 with a list of 512), as have up to 1024
// crowded ones (777 events at nu = 30: 608 us; 834 with the next shape). More of them take the
// instantiation of 16 waves a CU and the LDS that four workgroups leave (777 events: 298 us, 371 with
// three; 1000 pile-up events: 375, 440).
constexpr unsigned scored_waves_at_three = 3 * 4 * 256; // waves per SIMD, SIMDs, CUs
static SearchShape scored_shape(unsigned n_events, unsigned mean_hits)
{
  if (n_events * (256 / wave_size) <= scored_waves_at_three || (n_events <= 1024 && mean_hits > crowded_hits))
    return {256, 1920, 1024, 1024, 0};
  return {256, 1500, 512, 512, 0};
}

hipError_t launch_search_by_triplet(const SearchLaunch& a, hipStream_t s)
{
  if (!a.n_list) return hipSuccess;
  // Scored mode: seeds are decided in groups of block / K unused h1 hits of each chunk of block
  // positions (the pruning rule with seed_block = block), and a group's seeds must lie in one
  // wave for the in-wave scorer and decision: workgroups of 64, 128 or 256 lanes. The scorer's
  // weights take LDS from the hits (same residency).
  const bool scored = a.scorer_params != nullptr;
  const bool shaped = !a.block_dim && !a.work_counter;
  const SearchShape shape = !shaped ? SearchShape {256, search_default_lds_hits, ring_window, unused_list_cap, 0}
                            : scored ? scored_shape(a.n_list, a.mean_hits) : search_shape(a.n_list, a.mean_hits);
  const unsigned block = a.block_dim ? a.block_dim : shape.block;
  const unsigned hits_per_wave = shape.hits_per_wave;
  // Dynamic LDS stays within the device's per-workgroup limit (less the static part).
  const int max_lds = device_max_lds_per_block();
  if (!max_lds) return hipErrorInvalidDevice;
  if (scored && block != 64 && block != 128 && block != 256) return hipErrorInvalidConfiguration;
  // The LDS window of the ring: a power of two from 64 to 512 (it divides the ring); the list
  // of unused hits: a multiple of 16 up to 1024 (relative positions fit 16 bits either way).
  unsigned window = a.ring_window ? a.ring_window : shape.window;
  const unsigned list_cap = a.list_cap ? a.list_cap : shape.list_cap;
  if (window < 64 || a.ring_window > max_ring_window_knob || (window & (window - 1)) || list_cap % 16 || list_cap > unused_list_cap)
    return hipErrorInvalidValue;
  const size_t extra = scored ? scorer_lds_bytes + 16 : 0;
  const unsigned default_hits =
    scored && !shaped ? search_default_lds_hits - static_cast<unsigned>((extra + search_bytes_per_hit - 1) / search_bytes_per_hit)
           : shape.lds_hits;
  const unsigned wanted_hits = a.lds_hits ? a.lds_hits : default_hits;
  // Where the caller sets the workgroup or its hits, the long window must not cost a CU a workgroup
  // (256 lanes and 4096 hits, 1000 pile-up events: 437 us with one workgroup a CU, 245 with two).
  if (!a.ring_window && (!shaped || a.lds_hits)) {
    const auto per_cu = [&](unsigned w) { return lds_per_cu / (search_dynamic_lds(block, wanted_hits, w, list_cap) + extra + 1024); };
    if (per_cu(max_ring_window_knob) > per_cu(window)) window = max_ring_window_knob;
  }
  const size_t fixed = search_dynamic_lds(block, 0, window, list_cap) + extra + 1024;
  if ((size_t) max_lds <= fixed) return hipErrorInvalidConfiguration;
  const unsigned max_hits = static_cast<unsigned>(((size_t) max_lds - fixed) / search_bytes_per_hit);
  const unsigned lds_hits = min(wanted_hits, max_hits);
  const size_t dyn = search_dynamic_lds(block, lds_hits, window, list_cap) + extra;
  // Persistent mode: as many workgroups as stay resident (they take events from the counter).
  unsigned grid = a.n_list;
  if (a.work_counter) {
    const void* kernel = a.work_stats ? reinterpret_cast<const void*>(&k_search_by_triplet<true, seed_mode_plain, true>)
                         : a.scorer_params
                           ? reinterpret_cast<const void*>(&k_search_by_triplet<false, seed_mode_scored, true>)
                         : a.seed_log.counter
                           ? reinterpret_cast<const void*>(&k_search_by_triplet<false, seed_mode_log, true>)
                           : reinterpret_cast<const void*>(&k_search_by_triplet<false, seed_mode_plain, true>);
    const unsigned resident = device_resident_blocks(kernel, block, dyn);
    if (resident) grid = min(grid, resident);
  }
  SearchArgs k;
  k.event_list = a.event_list;
  k.number_of_events = a.number_of_events;
  k.sorted_container = a.sorted_container;
  k.offsets_estimated_input_size = a.offsets_estimated_input_size;
  k.module_cluster_num = a.module_cluster_num;
  k.geometry = reinterpret_cast<const Geometry*>(a.geometry);
  k.tracks = reinterpret_cast<TrackHits*>(a.tracks);
  k.tracklets = reinterpret_cast<TrackletHits*>(a.tracklets);
  k.tracks_to_follow = a.tracks_to_follow;
  k.three_hit_tracks = reinterpret_cast<TrackletHits*>(a.three_hit_tracks);
  k.hit_used = a.hit_used;
  k.atomics_velo = a.atomics_velo;
  k.rel_indices = a.rel_indices;
  k.number_of_velo_tracks = a.number_of_velo_tracks;
  k.status = a.status;
  k.phi_tolerance = a.phi_tolerance;
  k.max_scatter = a.max_scatter;
  k.max_skipped_modules = a.max_skipped_modules;
  k.lds_hits = lds_hits;
  k.hits_per_wave = hits_per_wave;
  k.work_stats = a.work_stats;
  k.event_clock = a.event_clock;
  k.n_list = a.n_list;
  k.work_counter = a.work_counter;
  k.seed_log = a.seed_log;
  k.scorer_params = a.scorer_params;
  k.scorer_threshold = a.scorer_threshold;
  k.window = window;
  k.list_cap = list_cap;
  k.three_hit_tracks_output = reinterpret_cast<TrackletHits*>(a.three_hit_tracks_output);
  k.number_of_three_hit_tracks_output = a.number_of_three_hit_tracks_output;
  k.event_track_hits = a.event_track_hits;
  k.max_chi2 = a.max_chi2;
#define VELO_LAUNCH_SEARCH_P(C, L, P) hipLaunchKernelGGL((k_search_by_triplet<C, L, P>), dim3(grid), dim3(block), dyn, s, k)
#define VELO_LAUNCH_SEARCH(C, L)                                                                                    \
  do {                                                                                                              \
    if (a.work_counter) VELO_LAUNCH_SEARCH_P(C, L, true);                                                           \
    else VELO_LAUNCH_SEARCH_P(C, L, false);                                                                         \
  } while (0)
  // Four waves a SIMD where the LDS lets them in and three leave events waiting.
  const unsigned waves = block / wave_size;
  const bool four = scored && !a.work_counter && a.n_list > scored_waves_at_three / waves &&
                    lds_per_cu / (dyn + 1024) * waves >= 16;
  if (a.work_stats) VELO_LAUNCH_SEARCH(true, seed_mode_plain);
  else if (four) hipLaunchKernelGGL((k_search_by_triplet<false, seed_mode_scored, false, 4>), dim3(grid), dim3(block), dyn, s, k);
  else if (a.scorer_params) VELO_LAUNCH_SEARCH(false, seed_mode_scored);
  else if (a.seed_log.counter) VELO_LAUNCH_SEARCH(false, seed_mode_log);
  else VELO_LAUNCH_SEARCH(false, seed_mode_plain);
#undef VELO_LAUNCH_SEARCH
#undef VELO_LAUNCH_SEARCH_P
  return hipGetLastError();
}

// The first n_big events of the list (the largest, when the list is ordered by descending hit
// count) in workgroups of big_block lanes with big_lds_hits hits of LDS on `side`, the others
// with the launch's own knobs on `s`. `side` waits for the work on `s` before it (fork) and `s`
// waits for `side` after both launches (join), so later work on `s` sees every event's outputs.
hipError_t launch_search_split(
  const SearchLaunch& a,
  unsigned n_big,
  unsigned big_block,
  unsigned big_lds_hits,
  hipStream_t s,
  hipStream_t side,
  hipEvent_t fork,
  hipEvent_t join)
{
  if (!a.event_list || !side || !fork || !join || n_big == 0 || n_big >= a.n_list || a.work_counter)
    return launch_search_by_triplet(a, s);
  hipError_t e = hipEventRecord(fork, s);
  if (e != hipSuccess) return e;
  e = hipStreamWaitEvent(side, fork, 0);
  if (e != hipSuccess) return e;
  SearchLaunch big = a;
  big.n_list = n_big;
  big.block_dim = big_block;
  big.lds_hits = big_lds_hits;
  // Launched first, so its large workgroups are placed before the many small ones.
  e = launch_search_by_triplet(big, side);
  SearchLaunch rest = a;
  rest.event_list = a.event_list + n_big;
  rest.n_list = a.n_list - n_big;
  const hipError_t e2 = launch_search_by_triplet(rest, s);
  // The join is recorded whatever happened above, so `side` never stays outside the run.
  const hipError_t e3 = hipEventRecord(join, side);
  const hipError_t e4 = e3 == hipSuccess ? hipStreamWaitEvent(s, join, 0) : e3;
  return e != hipSuccess ? e : (e2 != hipSuccess ? e2 : e4);
}

hipError_t launch_three_hit_tracks_filter(const ThreeHitFilterLaunch& a, hipStream_t s)
{
  if (!a.n_list) return hipSuccess;
  hipLaunchKernelGGL(
    k_three_hit_filter, dim3(a.n_list), dim3(256), 0, s, a.event_list, a.number_of_events, a.sorted_container,
    a.offsets_estimated_input_size, reinterpret_cast<const TrackletHits*>(a.three_hit_tracks_input), a.atomics_velo,
    a.hit_used, reinterpret_cast<TrackletHits*>(a.three_hit_tracks_output), a.number_of_three_hit_tracks_output,
    a.max_chi2);
  return hipGetLastError();
}

} // namespace velo

// Retina-cluster decoding for gfx950: the clusters come made by the front-end FPGAs, one 32-bit
// word each (bank type 73), and are decoded, keyed by (phi, id) and written sorted per module
// pair (device/velo/retinacluster_decoding/src/DecodeRetinaClusters.cu,
// CalculateNumberOfRetinaClustersPerSensor.cu).
//
//   k_retina_sensor_sizes   one wave per event: the cluster words of every sensor (v2/v3) or
//                           sensor pair (v4) slot, and (first event of the list) the bank of
//                           each slot
//   k_retina_decode         one wave per (event, module pair): decodes the module pair's words,
//                           ranks them by their 64-bit key in LDS (64 buckets of phi) and writes
//                           every cluster at its rank: the reference's sorting-key, permutation and
//                           sorted-decode kernels in one pass
//
// Where several words share a key (zero padding words, or identical clusters) they share a rank
// and the slot keeps the last of them in word order, which is what the reference's CPU target
// leaves there.
#include "velo_common.cuh"
#include "velo_kernels.h"

namespace velo {

namespace retina {
constexpr unsigned bank_type = 73; // LHCb::RawBank::VPRetinaCluster (mdf/lhcb/Event/RawBank.h:134)
constexpr unsigned waves_per_block = 2; // a finished wave keeps its LDS until its workgroup ends
constexpr unsigned key_cap = 512;  // keys of a module pair held in the wave's LDS slice
constexpr unsigned max_slots_per_mp = 8;

// What one wave holds in LDS: 6 KB.
struct Slice {
  int64_t key[key_cap];
  uint32_t newest[wave_size]; // of each phi bucket's words
  uint32_t before[wave_size]; // words of the buckets before each
  uint16_t next[key_cap];     // each word's successor in its bucket
  const uint32_t* word[max_slots_per_mp]; // the slots' banks
  uint32_t n_words[max_slots_per_mp], source[max_slots_per_mp];
};
constexpr uint32_t none = 0xFFFFu; // ends a bucket's list
static_assert(key_cap < none, "list ends");

// The bucket of a key: its top six bits, in key order.
__device__ __forceinline__ unsigned bucket_of(int64_t key) { return static_cast<unsigned>(key >> 58) + 32u; }

template<int version>
constexpr unsigned slots()
{
  return (version == 2 || version == 3) ? n_sensors : n_sensors / 2;
}

__device__ __forceinline__ void wave_sync_lds()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct Decoded {
  bool valid;
  uint32_t id;
  float x, y, z;
  int16_t phi;
  int64_t key;
};

// DecodeRetinaClusters.cu:101-149 (key) and :263-306 (cluster): centroid column and row with
// their fractions (v2: eighths, v3/v4: quarters, the row's bits kept in fy), the LHCbID with
// the fraction flags, the global position and phi; the key is (phi as u16) << 48 | id, or the
// largest key for a zero word.
template<int version>
__device__ __forceinline__ Decoded decode(const Geometry& g, uint32_t source, uint32_t word)
{
  Decoded d;
  unsigned sensor;
  if constexpr (version == 2 || version == 3) sensor = source;
  else sensor = (((source & 0x1FFu) << 1) | ((word >> 22) & 0x1u));
  d.valid = sensor < n_sensors;
  if (!d.valid) sensor = 0;
  const float* ltg = g.ltg + 12 * sensor;
  uint32_t cx, cy, or_fx, or_fy;
  float fx, fy;
  if constexpr (version == 2) {
    cx = (word >> 14) & 0x3FFu;
    fx = ((word >> 11) & 0x7u) / 8.f;
    cy = (word >> 3) & 0xFFu;
    fy = (word & 0x7FFu) / 8.f;
    or_fx = 0;
    or_fy = 0;
  }
  else {
    cx = (word >> 12) & 0x3FFu;
    fx = ((word >> 10) & 0x3u) / 4.f;
    cy = (word >> 2) & 0xFFu;
    fy = (word & 0x3FFu) / 4.f;
    or_fx = ((word >> 11) & 0x1u) | ((word >> 10) & 0x1u);
    or_fy = ((word >> 1) & 0x1u) | (word & 0x1u);
  }
  if (cx >= n_sensor_columns) {
    d.valid = false;
    cx = 0;
  }
  d.id = lhcb_id_of(sensor, cx >> 8, cx & 0xFFu, cy) | (or_fx << 27) | (or_fy << 26);
  const float local_x = g.local_x[cx] + fx * g.x_pitch[cx];
  const float local_y = (0.5f + fy) * pixel_size;
  d.x = ltg[0] * local_x + ltg[1] * local_y + ltg[9];
  d.y = ltg[3] * local_x + ltg[4] * local_y + ltg[10];
  d.z = ltg[6] * local_x + ltg[7] * local_y + ltg[11];
  d.phi = hit_phi_16(d.x, d.y);
  d.key = word == 0 ? 0x7FFFFFFFFFFFFFFFll
                    : static_cast<int64_t>(static_cast<uint64_t>(static_cast<uint16_t>(d.phi)) << 48) | d.id;
  return d;
}
} // namespace retina

using namespace retina;

// CalculateNumberOfRetinaClustersPerSensor.cu:12-53. The last bank of a slot in bank order
// wins, as on the CPU target; slots without a retina bank get 0.
template<int version>
__global__ void __launch_bounds__(wave_size) k_retina_sensor_sizes(
  const char* raw,
  const uint32_t* offsets,
  const uint32_t* sizes,
  const uint32_t* types,
  unsigned mep,
  const uint32_t* event_list,
  unsigned event_start,
  uint32_t* each_sensor_pair_size,
  uint32_t* retina_bank_index,
  uint32_t* event_totals,
  uint32_t* number_of_events,
  uint32_t* status)
{
  constexpr unsigned S = slots<version>();
  __shared__ int s_retina[S];
  __shared__ int s_any[S];
  const unsigned l = lane_id();
  const unsigned event_number = event_list ? event_list[blockIdx.x] : blockIdx.x;
  const RawEvent ev(raw, offsets, sizes, types, mep, event_number + event_start);
  for (unsigned i = l; i < S; i += wave_size) {
    s_retina[i] = -1;
    s_any[i] = -1;
  }
  wave_sync_lds();
  for (unsigned i = l; i < ev.n_banks; i += wave_size) {
    const RawBank b = raw_bank<version>(ev, i);
    const unsigned slot = (version == 2 || version == 3) ? b.sourceID : (b.sourceID & 0x1FFu);
    if (b.type == bank_type && slot < S) atomicMax(&s_retina[slot], static_cast<int>(i));
    const unsigned pair = b.sourceID & 0x1FFu;
    if (blockIdx.x == 0 && pair < S) atomicMax(&s_any[pair], static_cast<int>(i));
  }
  wave_sync_lds();
  uint32_t* out = each_sensor_pair_size + static_cast<size_t>(event_number) * S;
  uint32_t words = 0;
  for (unsigned i = l; i < S; i += wave_size) {
    const int bi = s_retina[i];
    const uint32_t n = bi >= 0 ? bank_n_sp<version>(raw_bank<version>(ev, static_cast<unsigned>(bi))) : 0u;
    out[i] = n;
    words += n;
    if (blockIdx.x == 0 && (s_any[i] >= 0 || event_totals)) retina_bank_index[i] = static_cast<uint32_t>(s_any[i]);
  }
  if (event_totals) {
    const uint32_t total = wave_inclusive_scan(words);
    if (l == wave_size - 1) event_totals[event_number] = total;
    if (blockIdx.x == 0 && l == 0) {
      number_of_events[0] = gridDim.x;
      status[0] = 0;
    }
  }
}

// DecodeRetinaClusters.cu:11-395 for one (event, module pair) per wave. Bound by the chain of dependent
// reads (slot, bank, header, word, geometry), so the slots' banks are looked up once, by a lane each,
// and the first 128 words stay decoded for the second pass; the rank of a word comes from the words
// of its phi bucket, where it was a comparison with every word; beyond key_cap words it is summed over
// tiles of them. 1000 pile-up events: 33 us (90); 200 events at nu = 60: 88 us (620, and 1340 where a
// word was compared with every word in memory).
template<int version>
__global__ void __launch_bounds__(waves_per_block* wave_size) k_retina_decode(
  const char* raw,
  const uint32_t* offsets,
  const uint32_t* sizes,
  const uint32_t* types,
  unsigned mep,
  const uint32_t* event_list,
  unsigned n_list,
  unsigned event_start,
  const Geometry* geometry,
  const uint32_t* offsets_each_sensor_pair_size,
  const uint32_t* retina_bank_index,
  const uint32_t* number_of_events,
  uint32_t* module_cluster_num,
  uint32_t* offsets_module_pair_cluster,
  char* cluster_container,
  uint32_t* hit_permutations,
  int64_t* hit_sorting_key,
  unsigned populate_items)
{
  constexpr unsigned S = slots<version>();
  constexpr unsigned step = S / n_module_pairs;
  __shared__ Slice s_slice[waves_per_block];
  static_assert(step <= max_slots_per_mp, "slots of a module pair");
  const unsigned wave = threadIdx.x / wave_size, l = lane_id();
  const unsigned item = blockIdx.x * waves_per_block + wave;
  // populate_module_pair_offsets_and_sizes (:11-36), element by element over every event's
  // module pairs (listed or not); the grid covers max(populate_items, listed items).
  if (l == 0 && item < populate_items) {
    offsets_module_pair_cluster[item + 1] = offsets_each_sensor_pair_size[static_cast<size_t>(item + 1) * step];
    if (item == 0) offsets_module_pair_cluster[0] = 0;
  }
  if (item >= n_list * n_module_pairs) return;
  const unsigned b = item / n_module_pairs, mp = item % n_module_pairs;
  const unsigned event_number = event_list ? event_list[b] : b;
  const uint32_t* sp_off = offsets_each_sensor_pair_size + static_cast<size_t>(event_number) * S;
  const uint32_t lo = sp_off[mp * step], hi = sp_off[(mp + 1) * step];
  const unsigned n = hi - lo;
  const unsigned total = offsets_each_sensor_pair_size[static_cast<size_t>(*number_of_events) * S];
  const Geometry& g = *geometry;
  const RawEvent ev(raw, offsets, sizes, types, mep, event_number + event_start);
  const bool in_lds = n <= key_cap;
  Slice& L = s_slice[wave];
  L.newest[l] = none;
  L.before[l] = 0;

  // The bank of each slot as the first event of the list placed it. A slot whose bank is missing in
  // this event or of another type has no valid word: such a word has no key in the reference (left
  // unset there); it ranks last here and is not written.
  const unsigned first_word = sp_off[mp * step + min(l, step)] - lo; // lane t: words before slot t
  if (l < step) {
    const uint32_t bi = retina_bank_index[mp * step + l];
    L.n_words[l] = 0;
    if (bi < ev.n_banks) {
      const RawBank bank = raw_bank<version>(ev, bi);
      L.word[l] = bank.word;
      L.source[l] = bank.sourceID;
      if (bank.type == bank_type) L.n_words[l] = bank_n_sp<version>(bank);
    }
  }
  wave_sync_lds();

  // Decode word k of the module pair (its slots' words, in slot and word order; words past the end
  // of a bank shorter than in the first event are invalid). The whole wave takes part.
  auto decode_at = [&](unsigned k) {
    unsigned t = 0, before = 0;
#pragma unroll
    for (unsigned j = 1; j < step; ++j) {
      const unsigned start = __builtin_amdgcn_readlane(first_word, j);
      if (start <= k) {
        t = j;
        before = start;
      }
    }
    Decoded d {};
    if (k < n && k - before < L.n_words[t]) d = decode<version>(g, L.source[t], L.word[t][k - before]);
    return d;
  };
  // Word k of the slice's tile, in the list of its bucket.
  auto enter = [&](unsigned k, int64_t key) {
    const unsigned bucket = bucket_of(key);
    L.key[k] = key;
    atomicAdd(&L.before[bucket], 1u);
    L.next[k] = static_cast<uint16_t>(atomicExch(&L.newest[bucket], k));
  };
  // From the number of words in each bucket to those in the buckets before it.
  auto count_before = [&]() {
    wave_sync_lds();
    const uint32_t count = L.before[l], before = wave_inclusive_scan(count) - count;
    wave_sync_lds();
    L.before[l] = before;
    wave_sync_lds();
  };
  // The tile's words below a key; last: none of them beyond position i has the key.
  auto below = [&](int64_t key, int i, bool& last) {
    const unsigned bucket = bucket_of(key);
    uint32_t position = L.before[bucket];
    last = true;
    for (unsigned j = L.newest[bucket]; j != none;) {
      const int64_t o = L.key[j];
      const unsigned next = L.next[j];
      position += key > o;
      last = last && !(static_cast<int>(j) > i && o == key);
      j = next;
    }
    return position;
  };
  uint32_t nonzero = 0;
  Decoded kept[2] {}; // the lane's first two words, for the ranking pass
  auto first_pass = [&](unsigned k) {
    const Decoded d = decode_at(k);
    if (k >= n) return d;
    const int64_t key = d.valid ? d.key : 0x7FFFFFFFFFFFFFFFll;
    hit_sorting_key[lo + k] = key;
    if (in_lds) enter(k, key);
    if (d.valid) nonzero += d.key != 0x7FFFFFFFFFFFFFFFll;
    else hit_permutations[lo + k] = 0;
    return d;
  };
  kept[0] = first_pass(l);
  if (n > wave_size) kept[1] = first_pass(l + wave_size);
  for (unsigned base = 2 * wave_size; base < n; base += wave_size) first_pass(base + l);
#pragma unroll
  for (unsigned d = 32; d > 0; d >>= 1) nonzero += __shfl_xor(nonzero, d, wave_size);
  if (l == 0) module_cluster_num[event_number * n_module_pairs + mp] = nonzero;
  if (in_lds) {
    count_before();
  }
  else {
    // More words: the tiles' positions of a word are added up in its entry of the permutation, in the
    // bits above bit 0, which the word's tile or a later one sets where the word isn't the last of its key.
    __threadfence_block();
    __builtin_amdgcn_wave_barrier();
    for (unsigned t0 = 0; t0 < n; t0 += key_cap) {
      if (t0) {
        wave_sync_lds(); // the tile before has been read
        L.newest[l] = none;
        L.before[l] = 0;
        wave_sync_lds();
      }
      for (unsigned k = l; k < min(key_cap, n - t0); k += wave_size) enter(k, hit_sorting_key[lo + t0 + k]);
      count_before();
      for (unsigned i = l; i < n; i += wave_size) {
        const uint32_t sum = t0 ? hit_permutations[lo + i] : 0u;
        bool last;
        const uint32_t more = below(hit_sorting_key[lo + i], static_cast<int>(i) - static_cast<int>(t0), last);
        hit_permutations[lo + i] = (sum + 2 * more) | (last ? 0u : 1u);
      }
    }
  }

  // Rank by key; the last word of a key's run writes the slot.
  const Clusters out {cluster_container, total};
  auto second_pass = [&](unsigned i, const Decoded& d) {
    if (i >= n) return;
    if (!d.valid) {
      if (!in_lds) hit_permutations[lo + i] = 0;
      return;
    }
    uint32_t position;
    bool last;
    if (in_lds) {
      position = below(d.key, static_cast<int>(i), last);
    }
    else {
      position = hit_permutations[lo + i] >> 1;
      last = !(hit_permutations[lo + i] & 1u);
    }
    const unsigned slot = lo + position;
    hit_permutations[lo + i] = slot;
    if (last) {
      out.ids()[slot] = d.id;
      out.xyz()[3 * (size_t) slot] = d.x;
      out.xyz()[3 * (size_t) slot + 1] = d.y;
      out.xyz()[3 * (size_t) slot + 2] = d.z;
      out.phis()[slot] = d.phi;
    }
  };
  second_pass(l, kept[0]);
  if (n > wave_size) second_pass(l + wave_size, kept[1]);
  for (unsigned base = 2 * wave_size; base < n; base += wave_size) second_pass(base + l, decode_at(base + l));
}

hipError_t launch_retina_sensor_sizes(const RetinaSizesLaunch& a, hipStream_t s)
{
  if (!a.n_list) return hipSuccess;
#define VELO_LAUNCH_RSS(V)                                                                                          \
  hipLaunchKernelGGL(                                                                                               \
    k_retina_sensor_sizes<V>, dim3(a.n_list), dim3(wave_size), 0, s, a.raw, a.offsets, a.sizes, a.types, unsigned(a.mep),            \
    a.event_list, a.event_start, a.each_sensor_pair_size, a.retina_bank_index, a.event_totals, a.number_of_events,   \
    a.status)
  switch (a.version) {
  case 2: VELO_LAUNCH_RSS(2); break;
  case 3: VELO_LAUNCH_RSS(3); break;
  default: VELO_LAUNCH_RSS(4); break;
  }
#undef VELO_LAUNCH_RSS
  return hipGetLastError();
}

hipError_t launch_retina_decode(const RetinaDecodeLaunch& a, hipStream_t s)
{
  const unsigned items = max(a.n_list * n_module_pairs, a.populate_items);
  if (!items) return hipSuccess;
  const unsigned grid = (items + waves_per_block - 1) / waves_per_block;
#define VELO_LAUNCH_RD(V)                                                                                           \
  hipLaunchKernelGGL(                                                                                               \
    k_retina_decode<V>, dim3(grid), dim3(waves_per_block * wave_size), 0, s, a.raw, a.offsets, a.sizes, a.types, unsigned(a.mep),    \
    a.event_list, a.n_list, a.event_start, reinterpret_cast<const Geometry*>(a.geometry),                         \
    a.offsets_each_sensor_pair_size, a.retina_bank_index, a.number_of_events, a.module_cluster_num,              \
    a.offsets_module_pair_cluster, a.cluster_container, a.hit_permutations, a.hit_sorting_key, a.populate_items)
  switch (a.version) {
  case 2: VELO_LAUNCH_RD(2); break;
  case 3: VELO_LAUNCH_RD(3); break;
  default: VELO_LAUNCH_RD(4); break;
  }
#undef VELO_LAUNCH_RD
  return hipGetLastError();
}

unsigned retina_sensor_slots(int version) { return (version == 2 || version == 3) ? n_sensors : n_sensors / 2; }

} // namespace velo

// Static hashmap: build and bulk query.
// Replaces pycuco::CUCOHashmap (include/cuco_hashmap.cuh:49-93 in the
// ShmTensor tree): same contract (immutable id -> value map, -1 for absent),
// own bucketed layout and wavefront-cooperative probing (see hashmap_dev.h).
#include <math.h>
#include <stdlib.h>

#include <mutex>

#include "common.h"
#include "hashmap.h"
#include "hashmap_dev.h"
#include "launchers.h"

namespace shmt {

// Densest physical fill of the table. A lookup costs one dependent HBM round
// trip per bucket on its probe chain; with 8 slots per 128-byte line about 5 %
// of the lines are full at 50 % fill against 31 % at 80 %, so denser requests
// are built at 50 % (capacity() still reports ceil(n / load_factor)).
constexpr double kMaxPhysicalLoad = 0.5;

static int64_t slots_needed(int64_t n, double lf) {
  if (lf > kMaxPhysicalLoad) lf = kMaxPhysicalLoad;
  int64_t cap = shmt_hashmap_capacity(n, lf);
  // always leave an empty slot so that a probe for an absent key terminates
  if (cap < n + 1) cap = n + 1;
  return cap;
}

static int format_for(int key_bytes, int val_bytes) {
  return (key_bytes == 4 && val_bytes == 4) ? kSlot8 : kSlot16;
}

static int64_t buckets_for(int64_t n, double lf, int fmt) {
  int64_t slots_per_bucket = kBucketBytes / fmt;
  int64_t slots = slots_needed(n, lf);
  return (slots + slots_per_bucket - 1) / slots_per_bucket;
}

// Bits that the value has in a packed word when keys span `key_span` ids: the key field is wide enough that
// it is never all ones (the empty slot).
static int packed_value_bits(int64_t key_span) {
  int key_bits = 1;
  while ((1ull << key_bits) - 1 < static_cast<uint64_t>(key_span)) ++key_bits;
  return 64 - key_bits;
}
constexpr int64_t kPackMaxSpan = 1ll << 62;  // 63 bits of key leave one of value
constexpr int64_t kPackMinKeys = (4 << 20) / (2 * kSlot16);

// ---- kernels ---------------------------------------------------------------

// Group insert of one (key, value) into the wide table. All 8 lanes of the
// probe group call with the same arguments.
__device__ __forceinline__ void group_insert16(uint64_t *table, uint32_t nbuckets,
                                               int64_t key, int64_t val) {
  const int sub = lane_id() & (kProbeGroup - 1);
  const int gbase = lane_id() & ~(kProbeGroup - 1);
  uint32_t b = reduce_range(hash_id(key), nbuckets);
  uint32_t probes = 0;
  while (probes < nbuckets) {
    uint64_t *slot = table + (static_cast<size_t>(b) * kProbeGroup + sub) * 2;
    // Fresh (L2-coherent) read of the slot key: another workgroup may have
    // claimed it since this CU last cached the line.
    int64_t k = static_cast<int64_t>(
        __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    if (group_ballot<kProbeGroup>(k == key)) return;  // duplicate key: first one wins
    uint64_t em = group_ballot<kProbeGroup>(k == -1);
    if (!em) {
      b = (b + 1 == nbuckets) ? 0 : b + 1;
      ++probes;
      continue;
    }
    const int target = __builtin_ctzll(em);
    int64_t old = 0;
    if (sub == target) {
      unsigned long long prev = atomicCAS(reinterpret_cast<unsigned long long *>(slot),
                                          ~0ull, static_cast<unsigned long long>(key));
      old = static_cast<int64_t>(prev);
      if (old == -1) slot[1] = static_cast<uint64_t>(val);
    }
    old = shfl64(old, gbase + target);
    if (old == -1 || old == key) return;
    // lost the race for that slot to a different key: look at the bucket again
  }
}

// Narrow table: each lane owns two words of the bucket and claims one with a
// single 64-bit compare-and-swap. `word` holds a key other than -1.
__device__ __forceinline__ void group_insert8(uint64_t *table, const MapView &m, uint64_t word) {
  const int sub = lane_id() & (kProbeGroup - 1);
  const int gbase = lane_id() & ~(kProbeGroup - 1);
  const uint64_t field = 1ull << m.val_bits;
  const uint32_t nbuckets = m.nbuckets;
  uint32_t b = map_bucket(m, slot8_key(m, word));
  uint32_t probes = 0;
  while (probes < nbuckets) {
    uint64_t *slot = table + (static_cast<size_t>(b) * kProbeGroup + sub) * 2;
    uint64_t w0 = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint64_t w1 = __hip_atomic_load(slot + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool e0 = (w0 == ~0ull), e1 = (w1 == ~0ull);
    const bool match = (!e0 && (w0 ^ word) < field) || (!e1 && (w1 ^ word) < field);
    if (group_ballot<kProbeGroup>(match)) return;
    uint64_t em = group_ballot<kProbeGroup>(e0 || e1);
    if (!em) {
      b = (b + 1 == nbuckets) ? 0 : b + 1;
      ++probes;
      continue;
    }
    const int target = __builtin_ctzll(em);
    int64_t old = 0;
    if (sub == target) {
      unsigned long long prev = atomicCAS(
          reinterpret_cast<unsigned long long *>(slot + (e0 ? 0 : 1)), ~0ull,
          static_cast<unsigned long long>(word));
      old = static_cast<int64_t>(prev);
    }
    old = shfl64(old, gbase + target);
    if (old == -1 || (static_cast<uint64_t>(old) ^ word) < field) return;
  }
}

// One wave takes 64 consecutive (key, value) pairs with coalesced loads; in
// step j the probe group g inserts pair g*8+j, so 8 inserts proceed per wave
// at a time and every bucket read is a full-line transaction.
template <int FMT>
__global__ __launch_bounds__(256) void hashmap_insert_kernel(
    uint64_t *table, MapView m, const void *keys, const void *vals,
    int64_t n, int key_bytes, int val_bytes) {
  const int lane = lane_id();
  const int gbase = lane & ~(kProbeGroup - 1);
  const int64_t waves_per_block = blockDim.x / kWave;
  int64_t wave = static_cast<int64_t>(blockIdx.x) * waves_per_block + threadIdx.x / kWave;
  const int64_t nwaves = static_cast<int64_t>(gridDim.x) * waves_per_block;
  for (int64_t base = wave * kWave; base < n; base += nwaves * kWave) {
    int64_t i = base + lane;
    int64_t mykey = -1, myval = -1;
    if (i < n) {
      mykey = map_key(m, load_int(keys, i, key_bytes));
      myval = load_int(vals, i, val_bytes);
    }
#pragma unroll 1
    for (int j = 0; j < kProbeGroup; ++j) {
      int64_t k = shfl64(mykey, gbase + j);
      int64_t v = shfl64(myval, gbase + j);
      if (base + gbase + j < n) {
        if (FMT == kSlot16)
          group_insert16(table, m.nbuckets, k, v);
        else if (k != -1)  // (-1 is the empty key)
          group_insert8(table, m, slot8_word(m, k, v));
      }
    }
  }
}

// ---- narrow table built partition by partition ---------------------------------
// A compare-and-swap per key on a table in memory runs at the rate of random
// device-scope atomics (about 20 G per second on this part) after a pass that
// cleared the table. Here the words are first dealt to partitions, runs of
// kPartBuckets consecutive buckets, and a workgroup then fills the buckets of
// its partition in LDS and writes them out whole: no clearing pass, and memory
// sees only coalesced accesses.
//   deal   a workgroup takes ITEMS x 1024 pairs, counts them per partition in
//          LDS, reserves room in every partition with one atomic each, orders
//          the words by partition in LDS and writes the runs.
//   fill   one workgroup per partition.
//   rest   words that found no room in the reserve of their partition (many
//          pairs of one key) or in the last buckets of the partition: inserted
//          one by one, as the general build does for all. Hardly ever any when
//          keys differ; of keys given many times, deal drops most repeats itself.
// Repeats, 4,194,304 pairs, whole constructor in place / by partitions: half on one key 870 / 111 us, 64 keys 201 / 96,
// 4,194 keys 111 / 127, 41,943 keys 118 / 121; 1,048,576 pairs of 10,486 keys 60 / 82, where hardly anything is inserted.
// 4,194,304 pairs of 16 bytes: clear 23 + insert 212 us before (16-byte slots; 13 + 191 with packed words), deal 33 +
// fill 37 + rest 5 us now. Deal reads 67 MB and writes 34, fill reads 34 and writes 67: 3 TB/s and 2.7 TB/s, with
// one and two workgroups per compute unit whose phases (load, count, order, write) hardly overlap.
// A bucket is filled in any slot order and a key goes to the first bucket of
// its probe sequence that has room, so lookups and `rest` see an ordinary table.
constexpr int kPartLog2Buckets = 9;
constexpr int kPartBuckets = 1 << kPartLog2Buckets;  // 64 KB of LDS: two workgroups per compute unit
constexpr int kPartMax = 2048;                       // partitions a dealing workgroup counts in LDS
constexpr int kPartBlock = 1024;
constexpr uint32_t kPartLookBack = 16;    // words in which a repeat of a key is looked for
constexpr int kPartRestBlocks = 1024;     // (none to do: 4 us, as with 64)

// Presence filter of a table of `nb` buckets (see filter_bits). What a lookup costs is the line it reads from beyond the
// L2s, which deliver some 52 G lines a second whether all of a line is asked for or 16 bytes of it; a request that is
// not a key needs none if a filter that the L2s hold says so. One word per bucket: 8 keys on average at half load, of which
// 1 absent request in 6 gets past; tables of more than 2^19 buckets share words, as 2 MiB is what an L2 of 4 MiB
// keeps beside the lines that stream through it (stand-alone probe, half of 16.8 M requests let through to a table
// of 64 MiB: no filter 320 us, 1 MiB 227, 2 MiB 239, 4 MiB 300).
constexpr int64_t kFilterMaxWords = 1 << 19;
// From 2^20 pairs on, where the table is four times the size of an L2. Below, many a line comes from the L2s all the same: 4.2 M
// requests to 600,000 keys, none / half / 70 per cent / all of them keys, 58 / 57 / 56 / 54 us without, 51 / 54 / 59 / 57 with a
// filter; to 1,048,576 keys 70 / 70 / 68 / 68 and 52 / 58 / 71 / 70.
constexpr int64_t kFilterMinKeys = 1 << 20;

static int filter_shift(int64_t nb) {
  int shift = 0;
  while ((nb >> shift) > kFilterMaxWords) ++shift;
  return shift;
}
__host__ __device__ __forceinline__ uint32_t filter_words(uint32_t nb, int shift) { return (nb + (1u << shift) - 1) >> shift; }

struct PartArgs {
  MapView map;
  uint64_t *table;
  const void *keys, *vals;
  int64_t n;
  int key_bytes, val_bytes;
  uint32_t parts;
  uint32_t room;        // words reserved per partition
  uint64_t *words;      // parts * room
  uint64_t *rest;       // n
  uint32_t *rest_count;
  uint32_t *filled;     // per partition: words dealt to it (may exceed room)
  uint32_t *filter;     // presence filter to be written, or null
  int filter_shift;
};

__device__ __forceinline__ uint32_t part_of(const MapView &m, uint64_t word) {
  return map_bucket(m, slot8_key(m, word)) >> kPartLog2Buckets;
}

template <int ITEMS>
__global__ __launch_bounds__(kPartBlock) void part_deal_kernel(PartArgs a) {
  __shared__ uint64_t staged[ITEMS * kPartBlock];
  __shared__ uint32_t start[kPartMax];  // words per partition, then where they start in `staged`
  __shared__ uint32_t base[kPartMax];   // where they go in the partition, minus start
  __shared__ uint32_t lds[kPartBlock / kWave];
  __shared__ uint32_t late_count, late_base;
  if (threadIdx.x == 0) late_count = 0;
  for (uint32_t p = threadIdx.x; p < kPartMax; p += kPartBlock) start[p] = 0;
  __syncthreads();
  const int64_t first = static_cast<int64_t>(blockIdx.x) * (ITEMS * kPartBlock);
  int64_t idx[ITEMS], key[ITEMS], val[ITEMS];
  bool ok[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    idx[j] = first + j * kPartBlock + threadIdx.x;
    ok[j] = idx[j] < a.n;
    key[j] = -1;
    val[j] = 0;
  }
  load_ints<ITEMS>(a.keys, idx, ok, a.key_bytes, key);
  load_ints<ITEMS>(a.vals, idx, ok, a.val_bytes, val);
  uint64_t word[ITEMS];
  uint32_t place[ITEMS];  // partition << 16 | rank among this workgroup's words of the partition
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const int64_t k = ok[j] ? map_key(a.map, key[j]) : -1;
    ok[j] = k != -1;  // (-1 is the empty key)
    word[j] = slot8_word(a.map, k, val[j]);
    place[j] = 0;
    if (ok[j]) {
      const uint32_t p = map_bucket(a.map, k) >> kPartLog2Buckets;
      place[j] = (p << 16) | atomicAdd(&start[p], 1u);  // (rank < ITEMS * 1024 <= 2^14)
    }
  }
  __syncthreads();
  // room in the partitions, and exclusive prefix of the counts: two neighbouring partitions per thread
  const uint32_t p0 = 2 * threadIdx.x;
  const uint32_t c0 = start[p0], c1 = start[p0 + 1];
  const uint32_t g0 = c0 ? atomicAdd(&a.filled[p0], c0) : 0;
  const uint32_t g1 = c1 ? atomicAdd(&a.filled[p0 + 1], c1) : 0;
  uint32_t total;
  const uint32_t before = block_exclusive_scan<uint32_t, kPartBlock>(c0 + c1, lds, &total);
  start[p0] = before;
  start[p0 + 1] = before + c0;
  base[p0] = g0 - before;
  base[p0 + 1] = g1 - (before + c0);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < ITEMS; ++j)
    if (ok[j]) staged[start[place[j] >> 16] + (place[j] & 0xFFFFu)] = word[j];
  __syncthreads();
  // Words without room. A partition that overflows holds few keys many times: a word whose key stands shortly before
  // it is dropped. One reservation per workgroup (a counter that every wave asks takes 250 us of a 4 M-pair deal).
  const uint64_t field = 1ull << a.map.val_bits;
  uint32_t late[ITEMS];  // place among the workgroup's words without room, ~0: none
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const uint32_t e = j * kPartBlock + threadIdx.x;
    late[j] = ~0u;
    if (e >= total) continue;
    const uint64_t w = staged[e];
    const uint32_t p = part_of(a.map, w);
    const uint32_t to = base[p] + e;
    if (to < a.room) {
      a.words[static_cast<size_t>(p) * a.room + to] = w;
    } else {
      const uint32_t from = e - start[p] > kPartLookBack ? e - kPartLookBack : start[p];
      bool again = false;
      for (uint32_t b = e; b > from && !again; --b) again = (staged[b - 1] ^ w) < field;
      if (!again) late[j] = atomicAdd(&late_count, 1u);
    }
  }
  __syncthreads();
  if (late_count == 0) return;
  if (threadIdx.x == 0) late_base = atomicAdd(a.rest_count, late_count);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < ITEMS; ++j)
    if (late[j] != ~0u) a.rest[late_base + late[j]] = staged[j * kPartBlock + threadIdx.x];
}

__global__ __launch_bounds__(kPartBlock) void part_fill_kernel(PartArgs a) {
  __shared__ alignas(16) unsigned long long slots[kPartBuckets * 16];
  __shared__ uint32_t present[kPartBuckets];  // this partition's words of the presence filter
  uint4 *const slots4 = reinterpret_cast<uint4 *>(slots);
  const uint32_t p = blockIdx.x;
  const uint32_t bucket0 = p << kPartLog2Buckets;
  const uint32_t nb = a.map.nbuckets - bucket0 < kPartBuckets ? a.map.nbuckets - bucket0 : kPartBuckets;
  const uint64_t field = 1ull << a.map.val_bits;
  constexpr int kHeld = 5;  // words a thread has in flight: all of a partition at half load (4,096 and a reserve)
  const uint32_t cnt = a.filled[p] < a.room ? a.filled[p] : a.room;
  const uint64_t *const words = a.words + static_cast<size_t>(p) * a.room;
  uint64_t held[kHeld];
  auto load = [&](uint32_t e0) {
#pragma unroll
    for (int j = 0; j < kHeld; ++j) {
      const uint32_t e = e0 + j * kPartBlock + threadIdx.x;
      held[j] = e < cnt ? words[e] : ~0ull;
    }
  };
  load(0);  // on their way while the slots are cleared
  for (uint32_t i = threadIdx.x; i < kPartBuckets * kProbeGroup; i += kPartBlock)
    slots4[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
  if (threadIdx.x < kPartBuckets) present[threadIdx.x] = 0;
  __syncthreads();
  for (uint32_t e0 = 0; e0 < cnt; e0 += kHeld * kPartBlock) {
    if (e0 > 0) load(e0);
#pragma unroll
    for (int j = 0; j < kHeld; ++j) {
      if (held[j] == ~0ull) continue;
      const uint32_t h = hash_id(slot8_key(a.map, held[j]));
      const uint32_t home = reduce_range(h, a.map.nbuckets) - bucket0;
      if (a.filter) atomicOr(&present[home >> a.filter_shift], filter_bits(h));
      bool placed = false;
      for (uint32_t b = home; b < nb && !placed; ++b) {
        // any order of the slots will do: threads that meet in a bucket start at different ones
        for (uint32_t step = 0; step < 16 && !placed; ++step) {
          unsigned long long *const slot = &slots[b * 16 + ((h + step) & 15)];
          unsigned long long seen = *slot;
          if (seen == ~0ull) {
            seen = atomicCAS(slot, ~0ull, static_cast<unsigned long long>(held[j]));
            placed = seen == ~0ull;
          }
          placed = placed || (seen ^ held[j]) < field;  // a pair of the same key is there: the first one wins
        }
      }
      if (!placed) a.rest[atomicAdd(a.rest_count, 1u)] = held[j];
    }
  }
  __syncthreads();
  uint4 *const out = reinterpret_cast<uint4 *>(a.table) + static_cast<size_t>(bucket0) * kProbeGroup;
  for (uint32_t i = threadIdx.x; i < nb * kProbeGroup; i += kPartBlock) out[i] = slots4[i];
  if (a.filter && threadIdx.x < filter_words(nb, a.filter_shift))
    a.filter[(bucket0 >> a.filter_shift) + threadIdx.x] = present[threadIdx.x];
}

// One word per probe group at a time: as a rule there are a few dozen, and a wave that took 64 of them would
// insert eight one after the other (11 us; 5 this way).
__global__ __launch_bounds__(256) void part_rest_kernel(PartArgs a) {
  const uint32_t n = *a.rest_count;
  const uint32_t groups = gridDim.x * (256 / kProbeGroup);
  for (uint32_t e = (blockIdx.x * 256 + threadIdx.x) / kProbeGroup; e < n; e += groups) {
    const uint64_t word = a.rest[e];
    if (a.filter && (lane_id() & (kProbeGroup - 1)) == 0) {  // (words that found no room in `deal` never got to `fill`)
      const uint32_t h = hash_id(slot8_key(a.map, word));
      atomicOr(&a.filter[reduce_range(h, a.map.nbuckets) >> a.filter_shift], filter_bits(h));
    }
    group_insert8(a.table, a.map, word);
  }
}

// ---- what do the keys look like? ---------------------------------------------
// One sweep over (keys, values): extrema of both, and whether value - key is
// the same for every pair. The host reads the result and picks the layout.
struct KeyStats {
  long long kmin, kmax, vmin, vmax;
  unsigned long long not_affine;  // != 0: value - key differs between pairs
  unsigned long long distinct;    // range candidates only: number of different keys
  unsigned long long not_ranked;  // != 0: keys do not ascend strictly, or value i is not value 0 + i
};

constexpr int kStatThreads = 1024;
constexpr int kStatBlocks = 256;           // workgroups of a sweep, one per compute unit, each leaving one partial result
constexpr int64_t kStatMarksOff = 256;     // scratch: one mark byte per id from here on (callers know it as more than a byte per id)

__device__ __forceinline__ int64_t wave_min64(int64_t v) {
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int64_t o = shfl64(v, lane_id() ^ d);
    v = o < v ? o : v;
  }
  return v;
}
__device__ __forceinline__ int64_t wave_max64(int64_t v) {
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int64_t o = shfl64(v, lane_id() ^ d);
    v = o > v ? o : v;
  }
  return v;
}

__device__ __host__ __forceinline__ void add_stats(KeyStats *to, const KeyStats &o) {
  to->kmin = o.kmin < to->kmin ? o.kmin : to->kmin;
  to->kmax = o.kmax > to->kmax ? o.kmax : to->kmax;
  to->vmin = o.vmin < to->vmin ? o.vmin : to->vmin;
  to->vmax = o.vmax > to->vmax ? o.vmax : to->vmax;
  to->not_affine |= o.not_affine;
  to->not_ranked |= o.not_ranked;
  to->distinct += o.distinct;
}

// Combines the calling workgroup's per-thread values into one KeyStats, valid
// in thread 0 (no atomics: thousands of them on a handful of addresses would
// cost more than the sweep).
__device__ __forceinline__ KeyStats block_combine(KeyStats mine) {
  __shared__ KeyStats per_wave[kStatThreads / kWave];
  mine.kmin = wave_min64(mine.kmin);
  mine.kmax = wave_max64(mine.kmax);
  mine.vmin = wave_min64(mine.vmin);
  mine.vmax = wave_max64(mine.vmax);
  mine.not_affine = __builtin_amdgcn_ballot_w64(mine.not_affine != 0) != 0;
  mine.not_ranked = __builtin_amdgcn_ballot_w64(mine.not_ranked != 0) != 0;
  mine.distinct = wave_last(wave_inclusive_scan(static_cast<uint64_t>(mine.distinct)));
  if (lane_id() == 0) per_wave[threadIdx.x / kWave] = mine;
  __syncthreads();
  KeyStats all = per_wave[0];
  if (threadIdx.x == 0) {
    for (unsigned w = 1; w < blockDim.x / kWave; ++w) add_stats(&all, per_wave[w]);
  }
  return all;
}

__device__ __forceinline__ KeyStats neutral_stats() {
  return KeyStats{INT64_MAX, INT64_MIN, INT64_MAX, INT64_MIN, 0, 0, 0};
}

// The sweep over all pairs. Bound by HBM: four pairs per thread are in flight, and the key before a pair's own comes from the
// lane next door: 4,194,304 pairs of 16 bytes 15.9 us, 4.2 TB/s (with one pair, and that key loaded again, 19.8).
constexpr int kStatItems = 4;
__global__ __launch_bounds__(kStatThreads) void key_stats_kernel(const void *keys, const void *vals, int64_t n,
                                                                 int key_bytes, int val_bytes, KeyStats *partials) {
  const int64_t v0 = load_int(vals, 0, val_bytes);
  const int64_t delta0 = v0 - load_int(keys, 0, key_bytes);
  KeyStats mine = neutral_stats();
  constexpr int64_t kSpan = kStatThreads * kStatItems;
  for (int64_t base = blockIdx.x * kSpan; base < n; base += gridDim.x * kSpan) {
    int64_t idx[kStatItems], before_idx[kStatItems], key[kStatItems], val[kStatItems], before[kStatItems];
    bool ok[kStatItems], first[kStatItems];
#pragma unroll
    for (int j = 0; j < kStatItems; ++j) {
      idx[j] = base + j * kStatThreads + threadIdx.x;
      before_idx[j] = idx[j] - 1;
      ok[j] = idx[j] < n;
      first[j] = ok[j] && lane_id() == 0 && idx[j] > 0;
      key[j] = val[j] = before[j] = 0;
    }
    load_ints<kStatItems>(keys, idx, ok, key_bytes, key);
    load_ints<kStatItems>(vals, idx, ok, val_bytes, val);
    load_ints<kStatItems>(keys, before_idx, first, key_bytes, before);
#pragma unroll
    for (int j = 0; j < kStatItems; ++j) {
      const int64_t next_door = shfl64(key[j], lane_id() - 1);
      if (!ok[j]) continue;
      const int64_t k = key[j], v = val[j], b = lane_id() == 0 ? before[j] : next_door;
      mine.kmin = k < mine.kmin ? k : mine.kmin;
      mine.kmax = k > mine.kmax ? k : mine.kmax;
      mine.vmin = v < mine.vmin ? v : mine.vmin;
      mine.vmax = v > mine.vmax ? v : mine.vmax;
      mine.not_affine |= (v - k != delta0);
      mine.not_ranked |= (v != v0 + idx[j]) || (idx[j] > 0 && b >= k);
    }
  }
  const KeyStats all = block_combine(mine);
  if (threadIdx.x == 0) partials[blockIdx.x] = all;
}

// The partial results of a sweep go straight to pinned host memory, one set per process, allocated on first use (a
// launch that merged them on the device took 4 us); map builds that run at the same time take turns at it.
static std::mutex g_stat_mutex;
static KeyStats *g_stat_slots = nullptr;      // pinned host memory, kStatBlocks
static KeyStats *g_stat_slots_dev = nullptr;  // its device alias

// Launch a sweep of nb <= kStatBlocks workgroups (`launch` is given where their results go) and wait for what it finds.
template <typename Launch>
static int read_stats(int nb, KeyStats *out, hipStream_t s, Launch launch) {
  std::lock_guard<std::mutex> lock(g_stat_mutex);
  if (g_stat_slots == nullptr) {
    void *p = nullptr, *d = nullptr;
    SHMT_HIP(hipHostMalloc(&p, kStatBlocks * sizeof(KeyStats), hipHostMallocMapped));
    SHMT_HIP(hipHostGetDevicePointer(&d, p, 0));
    g_stat_slots = static_cast<KeyStats *>(p);
    g_stat_slots_dev = static_cast<KeyStats *>(d);
  }
  launch(g_stat_slots_dev);
  SHMT_LAUNCH_CHECK();
  SHMT_HIP(hipStreamSynchronize(s));
  *out = g_stat_slots[0];
  for (int b = 1; b < nb; ++b) add_stats(out, g_stat_slots[b]);
  return SHMT_OK;
}

// Range candidates (as many pairs as ids between the extrema): every key marks
// its byte (plain stores: racing writers all write the same value), then the
// marked bytes are counted; fewer marks than pairs means a key repeats, and
// then some id of the range is missing.
__global__ __launch_bounds__(256) void key_mark_kernel(const void *keys, int64_t n, int key_bytes,
                                                       int64_t lo, uint8_t *seen) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
    const uint64_t off = static_cast<uint64_t>(load_int(keys, i, key_bytes) - lo);
    if (off < static_cast<uint64_t>(n)) seen[off] = 1;  // always true for a genuine candidate
  }
}

__global__ __launch_bounds__(256) void key_count_marks_kernel(const uint32_t *seen_words, int64_t nwords,
                                                              KeyStats *partials) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  KeyStats mine = neutral_stats();
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < nwords; i += stride)
    mine.distinct += __builtin_popcount(seen_words[i]);  // a marked byte is 0x01
  const KeyStats all = block_combine(mine);
  if (threadIdx.x == 0) partials[blockIdx.x] = all;
}

__global__ __launch_bounds__(256) void fill_zero_kernel(uint32_t *p, int64_t n) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = 0;
}

// Direct form: value[key - lo] for every pair (the table was filled with -1).
__global__ __launch_bounds__(256) void direct_build_kernel(int32_t *table, int64_t lo, int64_t span,
                                                           const void *keys, const void *vals, int64_t n,
                                                           int key_bytes, int val_bytes) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
    const uint64_t off = static_cast<uint64_t>(load_int(keys, i, key_bytes) - lo);
    if (off < static_cast<uint64_t>(span)) table[off] = static_cast<int32_t>(load_int(vals, i, val_bytes));
  }
}

// Rank form: one thread per 16-byte block = 96 consecutive ids. The keys
// ascend, so the thread finds the first key of its block by bisection (that
// index is the number of keys below the block) and walks the keys from there
// while they stay inside the block. Every block is written whole, the empty
// ones too: no clearing pass and no atomics.
__global__ __launch_bounds__(256) void rank_build_kernel(uint4 *table, int64_t nblocks, int64_t lo,
                                                         const void *keys, int64_t n, int key_bytes) {
  const int64_t b = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (b >= nblocks) return;
  const int64_t first_id = lo + b * kRankIdsPerBlock;
  int64_t below = 0, above = n;  // keys[below - 1] < first_id <= keys[above]
  while (below < above) {
    const int64_t mid = below + (above - below) / 2;
    if (load_int(keys, mid, key_bytes) < first_id)
      below = mid + 1;
    else
      above = mid;
  }
  uint32_t bits[3] = {0, 0, 0};
  for (int64_t j = below; j < n; ++j) {
    const uint64_t r = static_cast<uint64_t>(load_int(keys, j, key_bytes) - first_id);
    if (r >= static_cast<uint64_t>(kRankIdsPerBlock)) break;
    const uint32_t bit = 1u << (r & 31);
    bits[0] |= r < 32 ? bit : 0u;
    bits[1] |= (r >= 32 && r < 64) ? bit : 0u;
    bits[2] |= r >= 64 ? bit : 0u;
  }
  table[b] = make_uint4(static_cast<uint32_t>(below), bits[0], bits[1], bits[2]);
}

// Bulk query: a wave owns 64 consecutive requests; the first buckets of all
// 64 are in flight before one is examined, the requests of the next step as
// well, and results land in the lane that loaded the request, so request reads
// and result writes are both fully coalesced. Bound by random 128-byte lines, one per
// request and a few per cent of second buckets, of which this kernel gets some 50 G a second
// from beyond the L2s: 16,777,216 requests to a packed table (64 MiB) of 4,194,304 40-bit
// keys, half of them members, take 335 us, with the same requests again and again as well as
// with changing ones; 8,388,608 requests in 16-byte slots (128 MiB) 187 us. (Requests outside the key
// range of a packed table read no line of their own: half of them there, 204 us.) Each bucket load waiting for
// the one before, and all lanes of a group hashing all of its keys: 366 us. Eight waves per SIMD
// are asked for: the fragments alone are 32 registers.
// FILTER: the filter is asked first where that pays. It costs an access to the L2s per request and saves a line per
// request that it turns away. All waves of a launch have to do the same, for beside waves that read a line for every
// request the filter loses its place in the L2s: 16,777,216 requests to 4,194,304 keys (2 MiB of filter), 65 per cent of them keys,
// take 331 us without it, 311 with it, and 359 where every wave judged by its last 64 requests. So every wave asks the filter for the
// same 64 requests of the call while the lines of its own first ones are under way, and from then on uses it if kFilterAway of those were
// turned away. (Always asked, the filter meets the time without it at 13 of 64 turned away for 4 M keys and 8 M, at 5 for 2 M; the
// fewer steps a wave has, the more it takes.) Difference to lookups without filter at none / half / 60 / 70 / 80 per cent / all keys:
//   16.8 M requests to 4,194,304 keys at half load  -37 / -19 / -10 /   0 / +0.5 / +0.5 %  (337 / 333 / 331 / 331 / 330 / 328 us without)
//   to 8,000,000 keys (16 keys a word)              -32 /  -9 /   0 /  +1 / 0 / +0.5 %
//   to 1,048,576 keys                               -26 / -14 / -13 / +1.5 / +1 / +2 %
//   4.2 M requests to 4,194,304 keys                -34 / -10 /  +1 /  +3 / +1 / +1 %      (88 / 87 / 86 / 86 / 86 / 85 us without)
// Where waves have hardly a step after the first the sample costs more than it can give: half keys of 1.6 M requests +2 %, 2.6 M -3 %.
constexpr int kFilterAway = 18;
constexpr int64_t kFilterMinRequests = 1 << 21;

template <int FMT, bool FILTER>
__global__ __launch_bounds__(256, 8) void hashmap_query_kernel(
    MapView m, const void *req, int req_bytes, void *out, int out_bytes, int64_t n, const uint32_t *filter, int filter_shift) {
  const int lane = lane_id();
  const int64_t waves_per_block = blockDim.x / kWave;
  int64_t wave = static_cast<int64_t>(blockIdx.x) * waves_per_block + threadIdx.x / kWave;
  const int64_t nwaves = static_cast<int64_t>(gridDim.x) * waves_per_block;
  int64_t i = wave * kWave + lane;
  int64_t next = i < n ? load_int(req, i, req_bytes) : -1;  // the requests stay one step ahead of the probes
  bool ask = false, sample_inside = false;
  uint32_t sample_bits = 0, sample_word = 0;
  if (FILTER) {
    // (anywhere in each 64th of the requests: they may alternate)
    const int64_t share = n / kWave;
    const int64_t at = lane * share + reduce_range(hash_id(lane), static_cast<uint32_t>(share < UINT32_MAX ? share : UINT32_MAX));
    const int64_t key = map_key(m, load_int(req, at, req_bytes));
    const uint32_t h = hash_id(key);
    sample_inside = key != -1;  // (requests outside the key range read no line either way, and do not speak for the filter)
    sample_bits = filter_bits(h);
    sample_word = filter[reduce_range(h, m.nbuckets) >> filter_shift];
  }
  const int64_t first = i;
  for (; i - lane < n; i += nwaves * kWave) {
    const int64_t mykey = i < n ? map_key(m, next) : -1;  // tail lanes look up the sentinel, which resolves to -1
    const int64_t ahead = i + nwaves * kWave;
    if (ahead < n) next = load_int(req, ahead, req_bytes);
    uint64_t wanted = FILTER ? __builtin_amdgcn_ballot_w64(mykey != -1) : ~0ull;
    if (FILTER && ask) {
      const uint32_t h = hash_id(mykey), bits = filter_bits(h);
      wanted = __builtin_amdgcn_ballot_w64(mykey != -1 &&
                                           (filter[reduce_range(h, m.nbuckets) >> filter_shift] & bits) == bits);
    }
    const int64_t myres = wave_find<FMT, FILTER>(m, mykey, wanted);
    if (FILTER && i == first) {
      const uint64_t inside = __builtin_amdgcn_ballot_w64(sample_inside);
      const uint64_t away = inside & __builtin_amdgcn_ballot_w64((sample_word & sample_bits) != sample_bits);
      ask = __builtin_popcountll(away) * kWave >= __builtin_popcountll(inside) * kFilterAway;
    }
    if (i < n) store_int(out, i, out_bytes, myres);
  }
}

}  // namespace shmt

using namespace shmt;

extern "C" {

static int64_t filter_bytes(int64_t n, int64_t nbuckets);

int64_t shmt_hashmap_capacity(int64_t n, double load_factor) {
  if (n < 0 || !(load_factor > 0.0)) return -1;
  return static_cast<int64_t>(ceil(static_cast<double>(n) / load_factor));
}

int64_t shmt_hashmap_table_bytes(int64_t n, double load_factor, int key_bytes, int val_bytes) {
  if (n < 0 || !(load_factor > 0.0) || !(load_factor <= 1.0) || !width_ok(key_bytes) ||
      !width_ok(val_bytes)) {
    set_error("shmt_hashmap_table_bytes: bad arguments (n=%lld, load_factor=%g, key_bytes=%d, val_bytes=%d)",
              static_cast<long long>(n), load_factor, key_bytes, val_bytes);
    return -1;
  }
  return buckets_for(n, load_factor, format_for(key_bytes, val_bytes)) * kBucketBytes;
}

int64_t shmt_hashmap_plan_scratch_bytes(int64_t n) {
  if (n < 0) return -1;
  return kStatMarksOff + ((n + 3) / 4) * 4;
}

int shmt_hashmap_plan(const void *keys, const void *vals, int64_t n, int key_bytes, int val_bytes,
                      double load_factor, void *scratch, int64_t scratch_bytes,
                      shmt_hashmap_layout *layout, void *stream) {
  SHMT_REQUIRE(layout != nullptr, "shmt_hashmap_plan: layout is null");
  SHMT_REQUIRE(n >= 0, "shmt_hashmap_plan: n must be >= 0");
  SHMT_REQUIRE(width_ok(key_bytes) && width_ok(val_bytes),
               "shmt_hashmap_plan: ID can only be int32 or int64 (key_bytes=%d, val_bytes=%d)", key_bytes,
               val_bytes);
  SHMT_REQUIRE(load_factor > 0.0 && load_factor <= 1.0, "shmt_hashmap_plan: load_factor must be in (0, 1], got %g",
               load_factor);
  const int dtype_fmt = format_for(key_bytes, val_bytes);
  layout->kind = SHMT_MAP_BUCKETS;
  layout->slot_bytes = dtype_fmt;
  layout->lo = layout->span = layout->delta = 0;
  layout->table_bytes = buckets_for(n, load_factor, dtype_fmt) * kBucketBytes;
  if (n == 0) return SHMT_OK;
  SHMT_REQUIRE(keys != nullptr && vals != nullptr, "shmt_hashmap_plan: keys/vals are null");
  if (scratch == nullptr || scratch_bytes < shmt_hashmap_plan_scratch_bytes(n)) {
    set_error("shmt_hashmap_plan: scratch too small (%lld < %lld bytes)", static_cast<long long>(scratch_bytes),
              static_cast<long long>(shmt_hashmap_plan_scratch_bytes(n)));
    return SHMT_ENOMEM;
  }
  SHMT_REQUIRE((reinterpret_cast<uintptr_t>(scratch) & 15) == 0, "shmt_hashmap_plan: scratch must be 16-byte aligned");
  hipStream_t s = as_stream(stream);
  uint32_t *marks = reinterpret_cast<uint32_t *>(static_cast<char *>(scratch) + kStatMarksOff);  // one byte per id
  const unsigned nb = grid_for(n, kStatThreads * kStatItems, kStatBlocks);
  KeyStats st;
  int rc = read_stats(static_cast<int>(nb), &st, s, [&](KeyStats *partials) {
    hipLaunchKernelGGL(key_stats_kernel, dim3(nb), dim3(kStatThreads), 0, s, keys, vals, n, key_bytes, val_bytes, partials);
  });
  if (rc) return rc;

  const bool keys32 = st.kmin >= INT32_MIN && st.kmax <= INT32_MAX;
  const bool vals32 = st.vmin >= INT32_MIN && st.vmax <= INT32_MAX;
  // narrow slots whenever every key and value fits 32 bits, whatever the dtypes say
  int fmt = (keys32 && vals32) ? kSlot8 : kSlot16;
  const int64_t flat_limit = 2 * buckets_for(n, load_factor, fmt) * kBucketBytes;  // of a rank or direct table
  // ... and, packed, when a key's distance from the smallest one and the span of the values share 64 bits.
  // Only for tables that outgrow an L2 (4 MiB) in 16-byte slots: below that a lookup costs the same either way.
  if (fmt == kSlot16 && st.kmin >= 0 && st.kmax - st.kmin < kPackMaxSpan && n > kPackMinKeys) {
    const int64_t key_span = st.kmax - st.kmin + 1;
    const int val_bits = packed_value_bits(key_span);
    if (static_cast<uint64_t>(st.vmax) - static_cast<uint64_t>(st.vmin) < (1ull << val_bits)) {
      fmt = kSlot8;
      layout->lo = st.kmin;
      layout->span = key_span;
      layout->delta = static_cast<int64_t>(static_cast<uint64_t>(st.vmin) + (1ull << (val_bits - 1)));
    }
  }
  layout->slot_bytes = fmt;
  layout->table_bytes = buckets_for(n, load_factor, fmt) * kBucketBytes;
  if (fmt == kSlot8) layout->table_bytes += filter_bytes(n, layout->table_bytes / kBucketBytes);
  // flat forms need non-negative ids (-1 is the empty key) and a span that can be indexed
  if (st.kmin < 0 || st.kmax - st.kmin >= (1ll << 40)) return SHMT_OK;
  const int64_t span = st.kmax - st.kmin + 1;
  if (span == n && !st.not_affine) {
    // as many pairs as ids in the range and one offset for all: a range map unless a key repeats
    const int64_t words = (n + 3) / 4;
    hipLaunchKernelGGL(fill_zero_kernel, dim3(grid_for(words, 256 * 4)), dim3(256), 0, s, marks, words);
    hipLaunchKernelGGL(key_mark_kernel, dim3(grid_for(n, 256 * 8, 256 * 8)), dim3(256), 0, s, keys, n, key_bytes,
                       static_cast<int64_t>(st.kmin), reinterpret_cast<uint8_t *>(marks));
    const unsigned nbc = grid_for(words, 256 * 8, kStatBlocks);
    SHMT_LAUNCH_CHECK();
    KeyStats counted;
    rc = read_stats(static_cast<int>(nbc), &counted, s, [&](KeyStats *partials) {
      hipLaunchKernelGGL(key_count_marks_kernel, dim3(nbc), dim3(256), 0, s, marks, words, partials);
    });
    if (rc) return rc;
    if (counted.distinct == static_cast<unsigned long long>(n)) {
      layout->kind = SHMT_MAP_RANGE;
      layout->slot_bytes = 0;
      layout->lo = st.kmin;
      layout->span = span;
      layout->delta = st.vmin - st.kmin;  // value - key is one constant, so the minima pair up
      layout->table_bytes = kBucketBytes;  // nothing is stored; callers still pass a valid pointer
      return SHMT_OK;
    }
  }
  // pairs in ascending key order with consecutive values: bitmap with running counts, 16 bytes per 96 ids,
  // while that stays within twice the bucket table's size (ids up to 190 times as many as keys)
  const int64_t rank_bytes = ((span + kRankIdsPerBlock - 1) / kRankIdsPerBlock * 16 + kBucketBytes - 1) /
                             kBucketBytes * kBucketBytes;
  if (!st.not_ranked && n < (1ll << 32) && rank_bytes <= flat_limit) {
    layout->kind = SHMT_MAP_RANK;
    layout->slot_bytes = 16;
    layout->lo = st.kmin;
    layout->span = span;
    layout->delta = st.vmin;  // the first pair holds the smallest key and the smallest value
    layout->table_bytes = rank_bytes;
    return SHMT_OK;
  }
  // direct table while it stays within twice the bucket table's size (ids up to 8 times as many as
  // keys when both fit 32 bits): one load per lookup instead of a cooperative probe sequence
  if (vals32 && span * 4 <= flat_limit) {
    layout->kind = SHMT_MAP_DIRECT;
    layout->slot_bytes = 4;
    layout->lo = st.kmin;
    layout->span = span;
    layout->delta = 0;
    layout->table_bytes = (span * 4 + kBucketBytes - 1) / kBucketBytes * kBucketBytes;
  }
  return SHMT_OK;
}

// `layout` only matters for packed slots, `scratch` (optional) for the build by partitions.
static int build_buckets(shmt_hashmap_t **out, int fmt, const void *keys, const void *vals, int64_t n,
                         int key_bytes, int val_bytes, double load_factor, void *table_mem,
                         int64_t table_bytes, void *stream, const shmt_hashmap_layout *layout = nullptr,
                         void *scratch = nullptr, int64_t scratch_bytes = 0);

// Scratch of the build by partitions; parts == 0: the table is built in place.
struct PartPlan {
  uint32_t parts, room;
  int64_t words_off, rest_off, bytes;
};

// Whole constructor, keys of 30 / 40 bits, in place against by partitions: 2^17 pairs 64 / 62 us against 65 / 67,
// 2^18 68 / 69 against 61 / 59, 2^20 102 / 109 against 78 / 81, 2^22 247 / 279 against 123 / 123 (the
// 40-bit keys in place took 16-byte slots).
constexpr int64_t kPartMinKeys = 1 << 18;

static PartPlan part_plan(int fmt, int64_t n, int64_t nbuckets) {
  PartPlan p{0, 0, 0, 0, 0};
  const int64_t parts = (nbuckets + kPartBuckets - 1) / kPartBuckets;
  if (fmt != kSlot8 || n < kPartMinKeys || parts > kPartMax || n >= (1ll << 31)) return p;
  const double mean = static_cast<double>(n) * kPartBuckets / static_cast<double>(nbuckets);
  p.parts = static_cast<uint32_t>(parts);
  p.room = (static_cast<uint32_t>(mean + 6.0 * sqrt(mean)) + 79u) & ~15u;  // distinct keys spread evenly: six deviations
  p.words_off = ((static_cast<int64_t>(kPartMax) + 1) * 4 + 255) & ~255ll;
  p.rest_off = p.words_off + static_cast<int64_t>(p.parts) * p.room * 8;
  p.bytes = p.rest_off + n * 8;
  return p;
}

// Bytes of the presence filter behind the buckets, of tables that are built by partitions.
static int64_t filter_bytes(int64_t n, int64_t nbuckets) {
  if (n < kFilterMinKeys || part_plan(kSlot8, n, nbuckets).parts == 0) return 0;
  return (static_cast<int64_t>(filter_words(static_cast<uint32_t>(nbuckets), filter_shift(nbuckets))) * 4 + kBucketBytes - 1) /
         kBucketBytes * kBucketBytes;
}

int64_t shmt_hashmap_build_scratch_bytes(const shmt_hashmap_layout *layout, int64_t n, double load_factor) {
  if (layout == nullptr || n < 0 || !(load_factor > 0.0) || !(load_factor <= 1.0)) return -1;
  if (layout->kind != SHMT_MAP_BUCKETS || layout->slot_bytes != kSlot8) return 0;
  return part_plan(kSlot8, n, buckets_for(n, load_factor, kSlot8)).bytes;
}

int shmt_hashmap_create_planned(shmt_hashmap_t **out, const shmt_hashmap_layout *layout, const void *keys,
                                const void *vals, int64_t n, int key_bytes, int val_bytes,
                                double load_factor, void *table_mem, int64_t table_bytes, void *stream) {
  return shmt_hashmap_create_planned_scratch(out, layout, keys, vals, n, key_bytes, val_bytes, load_factor,
                                             table_mem, table_bytes, nullptr, 0, stream);
}

int shmt_hashmap_create_planned_scratch(shmt_hashmap_t **out, const shmt_hashmap_layout *layout, const void *keys,
                                        const void *vals, int64_t n, int key_bytes, int val_bytes,
                                        double load_factor, void *table_mem, int64_t table_bytes, void *scratch,
                                        int64_t scratch_bytes, void *stream) {
  SHMT_REQUIRE(out != nullptr && layout != nullptr, "shmt_hashmap_create_planned: null argument");
  *out = nullptr;
  SHMT_REQUIRE(n >= 0, "shmt_hashmap_create_planned: n must be >= 0");
  SHMT_REQUIRE(width_ok(key_bytes) && width_ok(val_bytes),
               "shmt_hashmap_create_planned: ID can only be int32 or int64 (key_bytes=%d, val_bytes=%d)",
               key_bytes, val_bytes);
  SHMT_REQUIRE(load_factor > 0.0 && load_factor <= 1.0,
               "shmt_hashmap_create_planned: load_factor must be in (0, 1], got %g", load_factor);
  if (layout->kind == SHMT_MAP_BUCKETS) {
    SHMT_REQUIRE(layout->slot_bytes == kSlot16 || layout->slot_bytes == kSlot8,
                 "shmt_hashmap_create_planned: bad slot size %d", layout->slot_bytes);
    // (16-byte slots have no use for an id range)
    SHMT_REQUIRE(layout->slot_bytes == kSlot16 || (layout->span >= 0 && layout->span <= kPackMaxSpan),
                 "shmt_hashmap_create_planned: bad id range of packed slots");
    return build_buckets(out, layout->slot_bytes, keys, vals, n, key_bytes, val_bytes, load_factor, table_mem,
                         table_bytes, stream, layout->slot_bytes == kSlot8 ? layout : nullptr, scratch, scratch_bytes);
  }
  SHMT_REQUIRE(layout->kind == SHMT_MAP_DIRECT || layout->kind == SHMT_MAP_RANGE || layout->kind == SHMT_MAP_RANK,
               "shmt_hashmap_create_planned: unknown layout kind %d", layout->kind);
  SHMT_REQUIRE(n > 0 && keys != nullptr && vals != nullptr && layout->lo >= 0 && layout->span > 0,
               "shmt_hashmap_create_planned: a flat layout needs keys and a non-negative id range");
  SHMT_REQUIRE(layout->kind != SHMT_MAP_RANK || n < (1ll << 32),
               "shmt_hashmap_create_planned: a rank layout holds fewer than 2^32 keys (32-bit running counts)");
  hipStream_t s = as_stream(stream);
  if (layout->kind == SHMT_MAP_DIRECT) {
    if (table_mem == nullptr || table_bytes < layout->table_bytes || layout->table_bytes < layout->span * 4) {
      set_error("shmt_hashmap_create_planned: table_mem too small (%lld < %lld bytes)",
                static_cast<long long>(table_bytes), static_cast<long long>(layout->table_bytes));
      return SHMT_ENOMEM;
    }
    SHMT_REQUIRE((reinterpret_cast<uintptr_t>(table_mem) & 127) == 0,
                 "shmt_hashmap_create_planned: table_mem must be 128-byte aligned");
    int rc = launch_fill_ones(table_mem, layout->table_bytes / 16, s);
    if (rc) return rc;
    hipLaunchKernelGGL(direct_build_kernel, dim3(grid_for(n, 256 * 4)), dim3(256), 0, s,
                       static_cast<int32_t *>(table_mem), layout->lo, layout->span, keys, vals, n, key_bytes,
                       val_bytes);
    SHMT_LAUNCH_CHECK();
  }
  if (layout->kind == SHMT_MAP_RANK) {
    const int64_t nblocks = (layout->span + kRankIdsPerBlock - 1) / kRankIdsPerBlock;
    if (table_mem == nullptr || table_bytes < layout->table_bytes || layout->table_bytes < nblocks * 16) {
      set_error("shmt_hashmap_create_planned: table_mem too small (%lld < %lld bytes)",
                static_cast<long long>(table_bytes), static_cast<long long>(layout->table_bytes));
      return SHMT_ENOMEM;
    }
    SHMT_REQUIRE((reinterpret_cast<uintptr_t>(table_mem) & 127) == 0,
                 "shmt_hashmap_create_planned: table_mem must be 128-byte aligned");
    hipLaunchKernelGGL(rank_build_kernel, dim3(grid_for(nblocks, 256)), dim3(256), 0, s,
                       static_cast<uint4 *>(table_mem), nblocks, layout->lo, keys, n, key_bytes);
    SHMT_LAUNCH_CHECK();
  }
  shmt_hashmap *h = static_cast<shmt_hashmap *>(calloc(1, sizeof(shmt_hashmap)));
  if (h == nullptr) {
    set_error("shmt_hashmap_create_planned: out of host memory");
    return SHMT_ENOMEM;
  }
  h->view = empty_map_view();
  h->view.buckets = static_cast<const uint4 *>(table_mem);
  h->view.key32 = (key_bytes == 4);
  h->view.kind = layout->kind == SHMT_MAP_DIRECT ? kKindDirect
                 : layout->kind == SHMT_MAP_RANK ? kKindRank : kKindRange;
  h->view.lo = layout->lo;
  h->view.span = layout->span;
  h->view.delta = layout->delta;
  h->kind = h->view.kind;
  h->fmt = kSlot8;  // kernels that branch on the kind at run time are launched in this form
  h->key_bytes = key_bytes;
  h->val_bytes = val_bytes;
  h->n = n;
  h->table_bytes = layout->kind == SHMT_MAP_RANGE ? 0 : layout->table_bytes;
  *out = h;
  return SHMT_OK;
}

int shmt_hashmap_create(shmt_hashmap_t **out, const void *keys, const void *vals, int64_t n,
                        int key_bytes, int val_bytes, double load_factor, void *table_mem,
                        int64_t table_bytes, void *stream) {
  SHMT_REQUIRE(width_ok(key_bytes) && width_ok(val_bytes),
               "shmt_hashmap_create: ID can only be int32 or int64 (key_bytes=%d, val_bytes=%d)",
               key_bytes, val_bytes);
  return build_buckets(out, format_for(key_bytes, val_bytes), keys, vals, n, key_bytes, val_bytes, load_factor,
                       table_mem, table_bytes, stream);
}

// Bucket table in slot format `fmt` (kSlot8 requires that every key and value fits 32 bits, or a layout with the
// id range of packed slots).
static int build_buckets(shmt_hashmap_t **out, const int fmt, const void *keys, const void *vals, int64_t n,
                         int key_bytes, int val_bytes, double load_factor, void *table_mem,
                         int64_t table_bytes, void *stream, const shmt_hashmap_layout *layout, void *scratch,
                         int64_t scratch_bytes) {
  SHMT_REQUIRE(out != nullptr, "shmt_hashmap_create: out is null");
  *out = nullptr;
  SHMT_REQUIRE(n >= 0, "shmt_hashmap_create: n must be >= 0");
  SHMT_REQUIRE(width_ok(key_bytes) && width_ok(val_bytes),
               "shmt_hashmap_create: ID can only be int32 or int64 (key_bytes=%d, val_bytes=%d)",
               key_bytes, val_bytes);
  SHMT_REQUIRE(load_factor > 0.0 && load_factor <= 1.0,
               "shmt_hashmap_create: load_factor must be in (0, 1], got %g", load_factor);
  SHMT_REQUIRE(n == 0 || (keys != nullptr && vals != nullptr),
               "shmt_hashmap_create: keys/vals are null");
  const int64_t nb = buckets_for(n, load_factor, fmt);
  SHMT_REQUIRE(nb < (1ll << 31), "shmt_hashmap_create: table too large (%lld buckets)",
               static_cast<long long>(nb));
  if (table_mem == nullptr || table_bytes < nb * kBucketBytes) {
    set_error("shmt_hashmap_create: table_mem too small (%lld < %lld bytes)",
              static_cast<long long>(table_bytes), static_cast<long long>(nb * kBucketBytes));
    return SHMT_ENOMEM;
  }
  SHMT_REQUIRE((reinterpret_cast<uintptr_t>(table_mem) & 127) == 0,
               "shmt_hashmap_create: table_mem must be 128-byte aligned");

  MapView view = empty_map_view();
  view.buckets = static_cast<const uint4 *>(table_mem);
  view.nbuckets = static_cast<uint32_t>(nb);
  view.key32 = (key_bytes == 4);
  view.fits32 = (fmt == kSlot8 && key_bytes == 8);
  if (layout != nullptr && layout->span > 0) {
    view.fits32 = 2;
    view.val_bits = packed_value_bits(layout->span);
    view.lo = layout->lo;
    view.span = layout->span;
    view.delta = layout->delta;
  }

  hipStream_t s = as_stream(stream);
  const PartPlan parts = part_plan(fmt, n, nb);
  uint32_t *filter = nullptr;  // in the memory that the plan asked for behind the buckets
  if (parts.parts > 0 && scratch != nullptr && scratch_bytes >= parts.bytes) {
    SHMT_REQUIRE((reinterpret_cast<uintptr_t>(scratch) & 15) == 0, "shmt_hashmap_create: scratch must be 16-byte aligned");
    char *const mem = static_cast<char *>(scratch);
    PartArgs a;
    a.map = view;
    a.table = static_cast<uint64_t *>(table_mem);
    a.keys = keys;
    a.vals = vals;
    a.n = n;
    a.key_bytes = key_bytes;
    a.val_bytes = val_bytes;
    a.parts = parts.parts;
    a.room = parts.room;
    a.filled = reinterpret_cast<uint32_t *>(mem);
    a.rest_count = a.filled + kPartMax;
    a.words = reinterpret_cast<uint64_t *>(mem + parts.words_off);
    a.rest = reinterpret_cast<uint64_t *>(mem + parts.rest_off);
    const int64_t with_filter = nb * kBucketBytes + filter_bytes(n, nb);
    if (with_filter > nb * kBucketBytes && layout != nullptr && layout->table_bytes >= with_filter && table_bytes >= with_filter)
      filter = reinterpret_cast<uint32_t *>(static_cast<char *>(table_mem) + nb * kBucketBytes);
    a.filter = filter;
    a.filter_shift = filter_shift(nb);
    hipLaunchKernelGGL(fill_zero_kernel, dim3(1), dim3(256), 0, s, a.filled, static_cast<int64_t>(kPartMax) + 1);
    // tiles of 16,384 pairs write longer runs, but there are to be enough of them: 4,194,304 pairs, whole constructor, 104 us
    // against 110 with tiles of 8,192 (deal 32 and 40), 2^21 75 both, 2^20 62 against 58
    const auto deal = n >= (1ll << 21) ? part_deal_kernel<16> : n >= (1ll << 20) ? part_deal_kernel<8> : part_deal_kernel<4>;
    const int64_t tile = (n >= (1ll << 21) ? 16 : n >= (1ll << 20) ? 8 : 4) * kPartBlock;
    hipLaunchKernelGGL(deal, dim3(static_cast<unsigned>((n + tile - 1) / tile)), dim3(kPartBlock), 0, s, a);
    hipLaunchKernelGGL(part_fill_kernel, dim3(parts.parts), dim3(kPartBlock), 0, s, a);
    hipLaunchKernelGGL(part_rest_kernel, dim3(kPartRestBlocks), dim3(256), 0, s, a);
    SHMT_LAUNCH_CHECK();
  } else {
    int rc = launch_fill_ones(table_mem, nb * (kBucketBytes / 16), s);
    if (rc) return rc;
    if (n > 0) {
      unsigned grid = grid_for(n, 256);
      if (fmt == kSlot16)
        hipLaunchKernelGGL(hashmap_insert_kernel<kSlot16>, dim3(grid), dim3(256), 0, s,
                           static_cast<uint64_t *>(table_mem), view, keys, vals, n, key_bytes, val_bytes);
      else
        hipLaunchKernelGGL(hashmap_insert_kernel<kSlot8>, dim3(grid), dim3(256), 0, s,
                           static_cast<uint64_t *>(table_mem), view, keys, vals, n, key_bytes, val_bytes);
      SHMT_LAUNCH_CHECK();
    }
  }

  shmt_hashmap *h = static_cast<shmt_hashmap *>(calloc(1, sizeof(shmt_hashmap)));
  if (h == nullptr) {
    set_error("shmt_hashmap_create: out of host memory");
    return SHMT_ENOMEM;
  }
  h->view = view;
  h->kind = kKindBuckets;
  h->fmt = fmt;
  h->key_bytes = key_bytes;
  h->val_bytes = val_bytes;
  h->n = n;
  h->table_bytes = nb * kBucketBytes;
  h->filter = filter;
  h->filter_shift = filter_shift(nb);
  *out = h;
  return SHMT_OK;
}

int shmt_hashmap_query(const shmt_hashmap_t *map, const void *requests, int req_bytes,
                       int64_t n, void *out, void *stream) {
  SHMT_REQUIRE(map != nullptr, "shmt_hashmap_query: map is null");
  SHMT_REQUIRE(n >= 0, "shmt_hashmap_query: n must be >= 0");
  SHMT_REQUIRE(width_ok(req_bytes), "shmt_hashmap_query: ID can only be int32 or int64");
  if (n == 0) return SHMT_OK;
  SHMT_REQUIRE(requests != nullptr && out != nullptr, "shmt_hashmap_query: null buffer");
  const bool filtered = map->filter != nullptr && n >= kFilterMinRequests;
  const unsigned grid = grid_for(n, 256);
  hipStream_t s = as_stream(stream);
  const auto kernel = map->fmt == kSlot16 ? hashmap_query_kernel<kSlot16, false>
                      : filtered          ? hashmap_query_kernel<kSlot8, true>
                                          : hashmap_query_kernel<kSlot8, false>;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, s, map->view, requests, req_bytes, out, map->val_bytes, n,
                     map->filter, map->filter_shift);
  SHMT_LAUNCH_CHECK();
  return SHMT_OK;
}

int shmt_hashmap_kind(const shmt_hashmap_t *map) { return map ? map->kind : -1; }
int64_t shmt_hashmap_used_bytes(const shmt_hashmap_t *map) { return map ? map->table_bytes : 0; }
int shmt_hashmap_key_bytes(const shmt_hashmap_t *map) { return map ? map->key_bytes : 0; }
int shmt_hashmap_val_bytes(const shmt_hashmap_t *map) { return map ? map->val_bytes : 0; }
int64_t shmt_hashmap_size(const shmt_hashmap_t *map) { return map ? map->n : 0; }
void shmt_hashmap_destroy(shmt_hashmap_t *map) { free(map); }

}  // extern "C"

// Device-side view of the static hashmap and the cooperative probe used by
// every kernel that consults it (bulk query, fetch/set, sampling plan).
//
// Layout in HBM: the table is an array of 128-byte buckets, one HBM/L2 line
// each. A probe group of 8 adjacent lanes reads one whole bucket with a
// single coalesced 16-byte-per-lane load and decides hit / miss / continue
// with a ballot, so one memory transaction inspects every slot of the line.
//   wide   (kSlot16): 8 slots {int64 key, int64 value}; used whenever the key
//                     or the value is 8 bytes wide (4-byte members are
//                     sign-extended on insert).
//   narrow (kSlot8) : 16 slots of one 64-bit word {key | value}, the key in the
//                     high bits; each lane sees two. Two ways to fill it:
//                     32 + 32 bits when every key and value fits 32 bits; or,
//                     packed, the key's distance from the smallest key above
//                     the value's distance from the middle of the values,
//                     when both together need at most 64 bits (a cache's slot
//                     numbers leave 40 bits and more to the keys). A table
//                     half the size is cleared, written and probed for.
// Empty slots hold all bits set; no key of either narrow form is stored so. Keys probe buckets
// linearly from hash(key) and are always placed in the first bucket of their
// probe sequence that still has a free slot, so a lookup stops at the first
// bucket that contains either the key or an empty slot.
//
// Three flat forms exist beside the bucket table, chosen when the map is built
// from what its keys look like (node ids are dense small integers, caches of
// re-numbered graphs hold an id range, and a cache built in id order numbers
// its rows by rank):
//   direct (kKindDirect): keys lie in [lo, lo + span) with span a small
//                     multiple of their number; the table is int32
//                     value[key - lo], -1 where no key was given. One 4-byte
//                     load per lookup, no probe sequence.
//   range  (kKindRange) : the keys are exactly the ids lo .. lo + span - 1 and
//                     every value is key + delta; lookups are arithmetic and
//                     touch no memory at all.
//   rank   (kKindRank)  : the pairs came in ascending key order with values
//                     v0, v0 + 1, v0 + 2, ...: the value is the key's rank
//                     among the keys (+ delta = v0). The table is a bitmap
//                     with running counts, 16-byte blocks {uint32 keys below
//                     this block, 96 presence bits}: one 16-byte load per
//                     lookup from a table of span / 6 bytes, which stays in
//                     the caches where a 4-byte-per-id table does not.
#pragma once
#include "wave.h"

#include <type_traits>

namespace shmt {

enum SlotFormat : int { kSlot16 = 16, kSlot8 = 8 };

constexpr int kProbeGroup = 8;      // lanes that cooperate on one key
constexpr int kBucketBytes = 128;

enum MapKind : int { kKindBuckets = 0, kKindDirect = 1, kKindRange = 2, kKindRank = 3 };

constexpr int kRankIdsPerBlock = 96;  // presence bits of one 16-byte rank block

struct MapView {
  const uint4 *buckets;   // bucket table: nbuckets * 8 uint4; direct form: int32 values[span];
                          // rank form: one uint4 block per 96 ids
  uint32_t nbuckets;
  int key32;              // 1: keys are int32 -> requests are narrowed before the lookup
  int kind;               // MapKind
  int fits32;             // narrow slots, 1: 64-bit keys that all fit 32 bits: a request that does not is
                          //    absent; 2: packed, looked up by key - lo
  int val_bits;           // narrow slots: low bits of a word that hold the value
  int64_t lo;             // flat forms, packed slots: smallest key
  int64_t span;           // flat forms, packed slots: keys lie in [lo, lo + span)
  int64_t delta;          // range form: value = key + delta; rank form: value = rank + delta; narrow slots:
                          //    value = stored signed field + delta
};

inline MapView empty_map_view() { return MapView{nullptr, 1, 0, kKindBuckets, 0, 32, 0, 0, 0}; }

// Normalise a request to the key domain of the map (what requests.to(key
// dtype) does in the reference): int32-keyed maps see the low 32 bits,
// sign-extended. A request that cannot be a key of a narrow-stored map
// becomes the empty sentinel, which every lookup resolves to -1.
__device__ __forceinline__ int64_t map_key(const MapView &m, int64_t req) {
  if (m.key32) req = static_cast<int64_t>(static_cast<int32_t>(req));
  if (m.fits32 == 2) {
    const uint64_t off = static_cast<uint64_t>(req) - static_cast<uint64_t>(m.lo);  // req < lo wraps around
    return off < static_cast<uint64_t>(m.span) ? static_cast<int64_t>(off) : -1;
  }
  if (m.fits32 && req != static_cast<int64_t>(static_cast<int32_t>(req))) return -1;
  return req;
}

// Narrow slots: the word of a normalised key (not -1) and its value, the key
// of a word, and the value in a word's low bits.
__device__ __forceinline__ uint64_t slot8_word(const MapView &m, int64_t key, int64_t val) {
  return (static_cast<uint64_t>(key) << m.val_bits) |
         ((static_cast<uint64_t>(val) - static_cast<uint64_t>(m.delta)) & ((1ull << m.val_bits) - 1));
}
__device__ __forceinline__ int64_t slot8_key(const MapView &m, uint64_t word) {
  if (m.fits32 == 2) return static_cast<int64_t>(word >> m.val_bits);
  return static_cast<int64_t>(word) >> 32;
}
__device__ __forceinline__ int64_t slot8_value(const MapView &m, uint64_t word) {
  const int s = 64 - m.val_bits;
  return static_cast<int64_t>(static_cast<uint64_t>(static_cast<int64_t>(word << s) >> s) + static_cast<uint64_t>(m.delta));
}

// Table entries that will not be looked at again soon (the probe of a row
// fetch) are read with the non-temporal cache policy, so that they do not push
// table rows out of the caches. They go through buffer loads, whose cache
// policy is an operand of the instruction: the same hint as metadata on an
// ordinary load is dropped whenever the optimiser merges the load with its
// plain twin on the other side of a branch. Buffer loads address with 32-bit
// byte offsets, so a table must stay below 4 GiB to be read this way
// (streamable()); larger ones are read with plain loads.
typedef uint32_t probe_u32x4 __attribute__((ext_vector_type(4)));
constexpr int kCachePolicyNonTemporal = 2;  // gfx94x / gfx950: bit 1 of the cache-policy operand

__device__ __forceinline__ __amdgpu_buffer_rsrc_t table_resource(const void *table) {
  // raw buffer over [table, table + 4 GiB): no stride, no swizzle; word 3 as gfx90a .. gfx950 want it for
  // untyped 32-bit data
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(table), 0, -1, 0x00020000);
}

// ... and it must be larger than the L2s together (64 MiB taken as the line): a table that the caches can
// hold is worth keeping there. (A bulk query over a 128 MiB table, which the memory-side cache holds when
// nothing else streams through it, measured 0.38 ms with plain loads and 0.48 ms streaming; the tables of a
// row fetch share that cache with the rows that stream through it, and there streaming wins from 160 MB up.)
__device__ __forceinline__ bool streamable(const MapView &m) {
  if (m.kind == kKindBuckets) return m.nbuckets >= (1u << 19) && m.nbuckets < (1u << 25);  // 128-byte buckets
  if (m.kind == kKindDirect) return m.span >= (1ll << 24) && m.span < (1ll << 30);          // 4-byte entries
  return false;
}

__device__ __forceinline__ uint4 load_bucket_streaming(const MapView &m, uint32_t bucket, int sub) {
  const uint32_t offset = (bucket * kProbeGroup + static_cast<uint32_t>(sub)) * 16u;
  const probe_u32x4 v =
      __builtin_amdgcn_raw_buffer_load_b128(table_resource(m.buckets), offset, 0, kCachePolicyNonTemporal);
  return make_uint4(v.x, v.y, v.z, v.w);
}

// Lookup in a flat map (kind != kKindBuckets); every lane for itself, in two
// steps so that a caller can put other work between the load and its use:
// flat_issue starts the one load a rank or direct map needs, flat_finish turns
// what came back into the value. STREAM: the entry of a direct table is read
// with a non-temporal load (see half_wave_issue for when a row fetch asks for
// that).
struct FlatPending {
  uint4 block;     // rank form: the 16-byte block of the key
  int32_t direct;  // direct form: the table entry
  bool inside;     // the key lies in [lo, lo + span)
};

template <bool STREAM = false>
__device__ __forceinline__ FlatPending flat_issue(const MapView &m, int64_t key) {
  FlatPending p;
  p.block = make_uint4(0, 0, 0, 0);
  p.direct = -1;
  const uint64_t off = static_cast<uint64_t>(key) - static_cast<uint64_t>(m.lo);  // key < lo wraps around
  p.inside = off < static_cast<uint64_t>(m.span);
  if (!p.inside || m.kind == kKindRange) return p;
  if (m.kind == kKindRank) {
    p.block = m.buckets[off / kRankIdsPerBlock];  // x: keys below this block; y, z, w: presence of ids 0-31, 32-63, 64-95
  } else {
    const int32_t *direct = reinterpret_cast<const int32_t *>(m.buckets);
    p.direct = STREAM ? static_cast<int32_t>(__builtin_amdgcn_raw_buffer_load_b32(
                            table_resource(m.buckets), static_cast<uint32_t>(off) * 4u, 0, kCachePolicyNonTemporal))
                      : direct[off];
  }
  return p;
}

__device__ __forceinline__ int64_t flat_finish(const MapView &m, int64_t key, const FlatPending &p) {
  if (!p.inside) return -1;
  if (m.kind == kKindRange) return key + m.delta;
  if (m.kind == kKindRank) {
    const uint64_t off = static_cast<uint64_t>(key) - static_cast<uint64_t>(m.lo);
    const uint32_t r = static_cast<uint32_t>(off % kRankIdsPerBlock);
    const uint4 b = p.block;
    const uint32_t word = r < 32 ? b.y : (r < 64 ? b.z : b.w);
    const uint32_t bit = r & 31;
    if (((word >> bit) & 1u) == 0) return -1;
    uint32_t below = __builtin_popcount(word & ((1u << bit) - 1u));
    if (r >= 32) below += __builtin_popcount(b.y);
    if (r >= 64) below += __builtin_popcount(b.z);
    return static_cast<int64_t>(b.x + below) + m.delta;
  }
  return static_cast<int64_t>(p.direct);
}

template <bool STREAM = false>
__device__ __forceinline__ int64_t flat_find(const MapView &m, int64_t key) {
  return flat_finish(m, key, flat_issue<STREAM>(m, key));
}

__device__ __forceinline__ uint32_t map_bucket(const MapView &m, int64_t key) {
  return reduce_range(hash_id(key), m.nbuckets);
}

// What a probe looks for and what it brings back, both 64 bits. Wanted: the
// key (wide slots), or the key in its place in a word (narrow slots). Found:
// the value, or the whole word; all ones when the key is absent (the sentinel
// too: its bits only equal those of empty slots). raw_value() turns what was
// found into the value, once per key and not once per probing lane.
template <int FMT>
__device__ __forceinline__ uint64_t probe_want(const MapView &m, int64_t key) {
  return FMT == kSlot16 ? static_cast<uint64_t>(key) : static_cast<uint64_t>(key) << m.val_bits;
}
template <int FMT>
__device__ __forceinline__ int64_t raw_value(const MapView &m, uint64_t raw) {
  return FMT == kSlot16 || raw == ~0ull ? static_cast<int64_t>(raw) : slot8_value(m, raw);
}

// Bitwise AND over the eight lanes of a probe group (lane exchanges 1, 2 and
// mirror-of-8 by DPP); every lane gets the result.
__device__ __forceinline__ uint32_t group_and(uint32_t v) {
  v &= static_cast<uint32_t>(__builtin_amdgcn_update_dpp(-1, static_cast<int>(v), 0xB1, 0xf, 0xf, false));   // quad_perm 1 0 3 2
  v &= static_cast<uint32_t>(__builtin_amdgcn_update_dpp(-1, static_cast<int>(v), 0x4E, 0xf, 0xf, false));   // quad_perm 2 3 0 1
  v &= static_cast<uint32_t>(__builtin_amdgcn_update_dpp(-1, static_cast<int>(v), 0x141, 0xf, 0xf, false));  // row_half_mirror
  return v;
}

// Lane J of every aligned group of eight, handed to the whole group.
template <int J>
__device__ __forceinline__ uint32_t group_bcast(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_ds_swizzle(static_cast<int>(v), (J << 5) | 0x18));  // lane & 24 | J
}
template <int J>
__device__ __forceinline__ uint64_t group_bcast64(uint64_t v) {
  const uint32_t lo = group_bcast<J>(static_cast<uint32_t>(v)), hi = group_bcast<J>(static_cast<uint32_t>(v >> 32));
  return (static_cast<uint64_t>(hi) << 32) | lo;
}

constexpr uint64_t kGroupBits = 0x0101010101010101ull;  // bit 8g: probe group g

// Examine the loaded fragments of one bucket per group (all lanes active).
// Returns, uniformly, bit 8g for every group g that is NOT done with its key:
// its bucket is full of other keys. The mask is scalar work, and what was
// found reaches every lane through three AND steps: against finding the
// matching lane with a ballot per group and asking it for the value, this
// takes a third of the vector instructions.
template <int FMT, typename Frag>
__device__ __forceinline__ uint64_t probe_buckets(const MapView &m, const Frag frag, uint64_t want, uint64_t *raw) {
  bool hit, empty;
  uint64_t mine;
  if (FMT == kSlot16) {
    const uint64_t k = (static_cast<uint64_t>(frag.y) << 32) | frag.x;
    mine = (static_cast<uint64_t>(frag.w) << 32) | frag.z;
    hit = (k == want);
    empty = (k == ~0ull);
  } else {
    const uint64_t w0 = (static_cast<uint64_t>(frag.y) << 32) | frag.x;
    const uint64_t w1 = (static_cast<uint64_t>(frag.w) << 32) | frag.z;
    const uint64_t field = 1ull << m.val_bits;
    const bool m0 = (w0 ^ want) < field, m1 = (w1 ^ want) < field;
    hit = m0 || m1;
    mine = m0 ? w0 : w1;  // (an empty slot that "matches" the sentinel is all ones: absent)
    empty = w0 == ~0ull || w1 == ~0ull;
  }
  const uint32_t lo = group_and(hit ? static_cast<uint32_t>(mine) : ~0u);
  const uint32_t hi = group_and(hit ? static_cast<uint32_t>(mine >> 32) : ~0u);
  *raw = (static_cast<uint64_t>(hi) << 32) | lo;
  uint64_t done = __builtin_amdgcn_ballot_w64(hit || empty);
  done |= done >> 4;
  done |= done >> 2;
  done |= done >> 1;
  return ~done & kGroupBits;
}

// Keeps a loaded fragment in registers: left to itself the compiler reads the
// half that a select picks from a second time.
__device__ __forceinline__ void keep_loaded(uint4 *frag) {
  asm volatile("" : "+v"(frag->x), "+v"(frag->y), "+v"(frag->z), "+v"(frag->w));
}
// (as one operand, see WaveProbe)
__device__ __forceinline__ void keep_loaded(probe_u32x4 *frag) { asm volatile("" : "+v"(*frag)); }

// Presence filter of a large narrow table: one word per 1 << shift home buckets, two bits of it set for every key. A
// key whose bits are not both set is absent. The bucket number uses the top bits of the hash, these use the low ones.
__device__ __forceinline__ uint32_t filter_bits(uint32_t hash) { return (1u << (hash & 31u)) | (1u << ((hash >> 5) & 31u)); }

// Whole-wave find: every lane brings its own (already normalised) key; the
// wave's eight probe groups resolve the 64 keys, eight keys per group. The
// first buckets of all 64 keys are loaded before any is examined, so the
// number of dependent HBM round trips is the longest probe chain among the 64
// keys, not the sum. Every lane hashes its own key; the group only shares the
// bucket number. Every lane gets the value for its own key (or -1). All 64
// lanes must be active; lanes with nothing to look up pass -1 (the empty
// sentinel, which resolves to -1 in one round). Flat maps are answered by
// every lane for itself.
// SKIP: see wave_probe_load. The fragments are one operand each there, of which the compiler makes no copies with a wait
// behind every load; the other form is compiled without such copies either way, and 3 % faster as it is
// (16.8 M requests to a table of 4 MiB 147 us, 152 with one operand each).
template <int FMT, bool SKIP = false>
struct WaveProbe {
  typename std::conditional<SKIP, probe_u32x4, uint4>::type frag[kProbeGroup];
  uint64_t want, res;
  uint64_t open;  // bit l: the key of lane l is not resolved (uniform)
  uint32_t home;
};

// SKIP: keys that are not in `wanted` (bit l: the key of lane l) are known to be absent and read no line. Their lanes ask
// for an address behind the table, which a buffer load answers with zeros without a request: loads under a lane mask
// would each end in a wait (the table must be below 4 GiB, see table_resource).
constexpr uint32_t kNoBucket = ~0u;

template <int FMT, int J, bool SKIP = false>
__device__ __forceinline__ void wave_probe_load(const MapView &m, WaveProbe<FMT, SKIP> *p, __amdgpu_buffer_rsrc_t table) {
  if constexpr (J < kProbeGroup) {
    const uint32_t sub = lane_id() & (kProbeGroup - 1);
    const uint32_t home = group_bcast<J>(p->home);
    if constexpr (SKIP) {
      p->frag[J] = __builtin_amdgcn_raw_buffer_load_b128(
          table, home == kNoBucket ? kNoBucket : (home * kProbeGroup + sub) * 16u, 0, 0);
    } else {
      p->frag[J] = m.buckets[static_cast<size_t>(home) * kProbeGroup + sub];
    }
    wave_probe_load<FMT, J + 1, SKIP>(m, p, table);
  }
}

template <int FMT, int J, bool SKIP>
__device__ __forceinline__ void wave_probe_examine(const MapView &m, WaveProbe<FMT, SKIP> *p) {
  if constexpr (J < kProbeGroup) {
    uint64_t raw;
    p->open |= probe_buckets<FMT>(m, p->frag[J], group_bcast64<J>(p->want), &raw) << J;
    if ((lane_id() & (kProbeGroup - 1)) == J) p->res = raw;
    wave_probe_examine<FMT, J + 1, SKIP>(m, p);
  }
}

// One more bucket for the keys that are not resolved (their first one was full of other keys). Only the groups
// that have such a key read a line: it is the lines that lookups are bound by.
template <int FMT, bool SKIP>
__device__ __forceinline__ void wave_probe_walk(const MapView &m, WaveProbe<FMT, SKIP> *p, uint32_t round) {
  const int sub = lane_id() & (kProbeGroup - 1), gbase = lane_id() & ~(kProbeGroup - 1);
#pragma unroll 1
  for (int j = 0; j < kProbeGroup; ++j) {
    if (((p->open >> j) & kGroupBits) == 0) continue;
    uint32_t b = static_cast<uint32_t>(__shfl(static_cast<int>(p->home), gbase + j, kWave)) + round;
    if (b >= m.nbuckets) b -= m.nbuckets;
    const uint64_t want = static_cast<uint64_t>(shfl64(static_cast<int64_t>(p->want), gbase + j));
    uint4 frag = make_uint4(0, 0, 0, 0);
    if ((p->open >> (gbase + j)) & 1ull) {
      frag = m.buckets[static_cast<size_t>(b) * kProbeGroup + sub];
      keep_loaded(&frag);
    }
    uint64_t raw;
    const uint64_t still = probe_buckets<FMT>(m, frag, want, &raw) << j;
    if (sub == j && ((p->open >> lane_id()) & 1ull)) p->res = raw;
    p->open &= still | ~(kGroupBits << j);
  }
}

template <int FMT, bool SKIP = false>
__device__ __forceinline__ int64_t wave_find(const MapView &m, int64_t mykey, uint64_t wanted = ~0ull) {
  if (!SKIP && m.kind != kKindBuckets) return flat_find(m, mykey);  // uniform across the launch
  WaveProbe<FMT, SKIP> p;
  p.want = probe_want<FMT>(m, mykey);
  p.home = map_bucket(m, mykey);
  p.open = 0;
  // (used where SKIP: ends with the table, words as in table_resource)
  const __amdgpu_buffer_rsrc_t table = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint4 *>(m.buckets), 0, static_cast<int>(m.nbuckets * static_cast<uint32_t>(kBucketBytes)), 0x00020000);
  if (SKIP && !__builtin_amdgcn_inverse_ballot_w64(wanted)) p.home = kNoBucket;
  wave_probe_load<FMT, 0, SKIP>(m, &p, table);
#pragma unroll
  for (int j = 0; j < kProbeGroup; ++j) keep_loaded(&p.frag[j]);
  wave_probe_examine<FMT, 0, SKIP>(m, &p);
  if constexpr (SKIP) {
    p.open &= wanted;
    if (!__builtin_amdgcn_inverse_ballot_w64(wanted)) p.res = ~0ull;
  }
  for (uint32_t round = 1; p.open != 0 && round < m.nbuckets; ++round) wave_probe_walk<FMT, SKIP>(m, &p, round);
  return raw_value<FMT>(m, p.res);
}

// True (in every lane) when some key of lanes 0 .. 31 also appears in another
// of those lanes at lane distance 1, 2, 4, 8 or 16: under skewed access a
// handful of hot keys take most of the requests and show up twice within 32
// rows nearly every time, under uniform access over a large key set next to
// never. A hint for the cache policy of the lookup, nothing more. All lanes
// must be active; lanes that bring no key pass `has_key` false.
__device__ __forceinline__ bool tile_repeats(int64_t mykey, bool has_key) {
  bool again = false;
#pragma unroll
  for (int d = 1; d < 32; d *= 2) again |= mykey == shfl64(mykey, lane_id() ^ d);
  return __builtin_amdgcn_ballot_w64(again && has_key && lane_id() < 32) != 0;
}

// Find for a wave whose lanes 0 .. 31 bring one (already normalised) key each
// (a fetch tile of 32 rows); lanes 32 .. 63 bring nothing. The keys are dealt
// four to a probe group (group g takes the keys of lanes 4g .. 4g + 3), so all
// eight groups work, the first bucket of every key is in flight at once (32
// lines), and a lookup that ends in its first bucket costs ONE dependent round
// trip; wave_find would leave the upper four groups looking up the empty
// sentinel while the lower four walk through eight keys each in two passes.
// STREAM: read the buckets with non-temporal loads. A
// table far larger than the caches is read once per row and its lines only
// push table rows out: measured on 1,048,576 uniform all-hit rows of 256 B
// through a 640 MB table, 125 us with plain probe loads and 112 us with
// non-temporal ones. Under skewed access the buckets of hot keys are what the
// caches should keep, and there non-temporal probes cost 10 % (Zipf(1.1)
// batch: 112 us plain, 123 us non-temporal). The caller therefore asks for
// streaming only for tiles that show no sign of skew (tile_repeats).
// Every lane below 32 gets the value for its own key (or -1). All 64 lanes
// must be active. Flat maps are answered by every lane for itself.
constexpr int kHalfWaveKeys = 4;  // keys per probe group of a 32-key lookup

// The lookup in two steps, so that a caller can put other work (moving the
// rows of the tile before) between the loads and their use: half_wave_issue
// deals the keys to the groups and starts the load of every key's first
// bucket; half_wave_finish examines what came back and walks on, bucket by
// bucket, for the few keys whose first bucket was full of other keys.
struct HalfWaveProbe {
  uint4 frag[kHalfWaveKeys];  // (the keys are dealt again by half_wave_finish: cheaper than keeping them in registers)
};

template <int FMT, bool STREAM>
__device__ __forceinline__ void half_wave_issue(const MapView &m, int64_t mykey, HalfWaveProbe *p) {
  const int sub = lane_id() & (kProbeGroup - 1);
  const int grp = lane_id() / kProbeGroup;
  const uint32_t home = map_bucket(m, mykey);
#pragma unroll
  for (int j = 0; j < kHalfWaveKeys; ++j) {
    const uint32_t b = static_cast<uint32_t>(__shfl(static_cast<int>(home), grp * kHalfWaveKeys + j, kWave));
    p->frag[j] = STREAM ? load_bucket_streaming(m, b, sub) : m.buckets[static_cast<size_t>(b) * kProbeGroup + sub];
  }
}

template <int FMT>
__device__ __forceinline__ int64_t half_wave_finish(const MapView &m, int64_t mykey, const HalfWaveProbe &p) {
  const int lane = lane_id();
  const int sub = lane & (kProbeGroup - 1);
  const int grp = lane / kProbeGroup;
  uint64_t res = ~0ull;  // lane 8g + j ends up with what was found for the key of lane 4g + j
  uint64_t open = 0;     // bit 8g + j: that key is not resolved (uniform)
#pragma unroll
  for (int j = 0; j < kHalfWaveKeys; ++j) {
    const uint64_t want = probe_want<FMT>(m, shfl64(mykey, grp * kHalfWaveKeys + j));
    uint64_t raw;
    open |= probe_buckets<FMT>(m, p.frag[j], want, &raw) << j;
    if (sub == j) res = raw;
  }
  for (uint32_t round = 1; open != 0 && round < m.nbuckets; ++round) {  // some bucket was full of other keys: walk on
#pragma unroll 1
    for (int j = 0; j < kHalfWaveKeys; ++j) {
      if (((open >> j) & kGroupBits) == 0) continue;
      const int64_t key = shfl64(mykey, grp * kHalfWaveKeys + j);
      uint4 frag = make_uint4(0, 0, 0, 0);  // (a group whose key is resolved reads no line)
      if ((open >> (grp * kProbeGroup + j)) & 1ull) {
        uint32_t b = map_bucket(m, key) + round;
        if (b >= m.nbuckets) b -= m.nbuckets;
        frag = m.buckets[static_cast<size_t>(b) * kProbeGroup + sub];
      }
      uint64_t raw;
      const uint64_t still = probe_buckets<FMT>(m, frag, probe_want<FMT>(m, key), &raw) << j;
      if (sub == j && ((open >> lane) & 1ull)) res = raw;
      open &= still | ~(kGroupBits << j);
    }
  }
  const uint64_t mine = static_cast<uint64_t>(
      shfl64(static_cast<int64_t>(res), (lane / kHalfWaveKeys) * kProbeGroup + (lane & (kHalfWaveKeys - 1))));
  return raw_value<FMT>(m, mine);
}

}  // namespace shmt

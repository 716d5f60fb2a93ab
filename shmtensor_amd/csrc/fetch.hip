// Feature row gather (fetch) and scatter (set) through the HBM cache.
// Replaces the twelve kernels of src/cache_feature_fetch.cu:15-224 and
// src/cache_feature_set.cu:6-207 in the ShmTensor tree with one templated
// kernel.
//
// A wave owns tiles of up to 32 consecutive rows.
// Phase 1 (lane per row): coalesced load of the ids, then the cache slot of
// every row at once: the wave's eight probe groups look the ids up
// cooperatively (one 128-byte bucket line per probe, the first bucket of all
// 32 keys in flight together), or every lane reads its slot from a flat map
// (direct table: one 4-byte load; rank bitmap: one 16-byte load; id range:
// arithmetic), or the mask is loaded. Each lane ends up holding the source
// (fetch) or destination (set) address of its row. A wave with several tiles
// keeps phase 1 of the next tiles in flight while it moves rows.
// Phase 2: the row addresses are broadcast with lane shuffles and the rows are
// moved with the widest vector access the row size and base pointers allow (16
// bytes per lane when aligned). Rows of 8, 16, 32 or 64 vectors (or nearly) take
// a sub-wave group of as many lanes each; the vectors of other short rows
// are dealt to the lanes one after the other, whatever row they belong to, so
// that no lane is left over at the end of a row; long rows (wide_from) are moved
// one by one by the whole wave, with four vectors per lane in flight. The
// dependent chain id -> bucket -> row is paid once per tile
// instead of once per row.
//
// A fetch can also go out as two launches (shmt_fetch_cached_part /
// shmt_fetch_missed_part): the rows that hit now, the rows that miss (marked
// in a bitmap) by a small grid that a caller may put on another stream.
//
// Measured on MI355X (1,048,576 rows of 256 B): the kernel is register-lean
// on purpose. Eight resident waves per SIMD with one row in flight
// per lane group beat four waves with eight rows in flight by 25-50 % on
// mixed hit/miss batches, because a wave that waits on a host-link read
// (loads return in issue order) then holds back little other work; setting
// missed rows apart in LDS for dedicated waves was measured slower than this
// and is not done.
#include "common.h"
#include "hashmap.h"
#include "hashmap_dev.h"

namespace shmt {

enum RouteMode : int { kDirect = 0, kMap16 = 1, kMap8 = 2, kMask = 3, kMapFlat = 4 };

struct RowArgs {
  char *miss;          // table addressed by id (pinned host alias or device)
  char *cache;         // table addressed by slot (HBM)
  char *dense;         // fetch: output rows; set: update rows
  const void *indices;
  const void *mask;
  MapView map;
  int64_t Q;
  const int64_t *count;  // when set: only the first min(Q, *count) rows are moved (device memory)
  int64_t *count_seen;   // when set: receives *count as soon as the kernel starts (pinned host memory)
  int64_t row_bytes;
  int idx_bytes;
  int mask_bytes;
  int log2_lanes;      // lanes per row in phase 2 = 1 << log2_lanes, in [8, 64]
  int log2_tile;       // rows per wave tile = 1 << log2_tile, at most 32
  uint32_t nvec;        // vectors per row (kDealt)
  uint32_t nvec_magic;  // floor((2^32 - 1) / nvec): the high half of i * magic is i / nvec, or one less
  uint32_t group_step;  // kDealt: vectors that a wave moves at a time with a lane group per row; 0: always dealt out
  int stream_dense;     // kWide: `dense` is accessed past the caches
  int link_rows;        // kWide, fetch of 16-byte vectors: missed rows keep one vector per lane in flight
  uint32_t *miss_bits;  // DEFER: bit (i & 31) of word i / 32 is set when row i missed the cache
};

// Native vector types (the non-temporal builtins do not take HIP's struct vectors).
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Table rows are addressed through integers that travelled across lanes, so
// the compiler cannot tell that they point to global memory; saying so turns
// generic (flat) accesses into global ones.
template <typename VT>
__device__ __forceinline__ VT gload(const char *p) {
  return *reinterpret_cast<const VT __attribute__((address_space(1))) *>(reinterpret_cast<uintptr_t>(p));
}
template <typename VT>
__device__ __forceinline__ void gstore(char *p, VT v) {
  *reinterpret_cast<VT __attribute__((address_space(1))) *>(reinterpret_cast<uintptr_t>(p)) = v;
}

constexpr int kRowsBlock = 256;    // threads per workgroup
constexpr int kRowsWavesPerSimd = 8;  // register budget: 512 / 8 = 64 VGPRs
// Rows a lane group moves concurrently (single-vector rows). Measured on 1,048,576 all-hit rows of
// 256 B: 1 row in flight per group 92 us, 2 rows 96 us, 4 rows 94 us (eight resident waves per SIMD
// already keep the memory system busy; shorter load/store bursts per wave mix reads and writes better).
constexpr int kRowsInFlight = 1;
// Vectors a lane moves concurrently when they are dealt out one by one, and the waves per SIMD the register
// budget is set for. 262,144 rows, all hits, buffers not in the caches, one / two in flight (with lane groups
// before): fetch of 33 floats 22.0 / 23.9 (27.9) us, 300 floats 123 / 137 (144), 300 halves 71 / 91 (107); set
// of 33 floats 25.4 / 30.6 (35.8), 50 floats 27.5 / 30.6 (29.1), but 100 floats 45.8 / 43.9 (48.5) and 300 floats
// 178 / 171 (171): a set of 16-byte vectors takes two, which need the registers of six waves. Four gain nothing.
constexpr int vecs_in_flight(bool set, int vector_bytes) { return set && vector_bytes == 16 ? 2 : 1; }
// How the rows of a tile are moved: a lane group per row with one vector per lane, vectors dealt out one by one,
// or one row after the other by the whole wave.
enum RowRoute : int { kOneVec, kDealt, kWide };
constexpr int rows_waves_per_simd(bool set, bool through, int route, int vector_bytes) {
  if (route == kWide) return vector_bytes == 16 || through ? 6 : kRowsWavesPerSimd;
  return route == kOneVec || vecs_in_flight(set, vector_bytes) == 1 ? kRowsWavesPerSimd : 6;
}

// One row of more than 64 vectors, moved by the whole wave: a lane has kWideInFlight vectors in flight, also
// where the row ends among them. A row of 16-byte vectors that comes over the host link has one: the link is full
// without more, and more cost it reads (16,384 rows of 512 floats 590 us with one, 615 with four, 1,024 floats
// 1174 / 1230; 1,000 rows 78 / 97). Narrower vectors are faster with four (4,097 bytes 1740 / 1495, 1,001 halves
// 806 / 648, 301 floats 403 / 394), and so are calls of few rows (below).
constexpr int kWideInFlight = 4;
constexpr bool may_stream(bool set, int vector_bytes) { return vector_bytes >= (set ? 4 : 16); }
// (1- and 2-byte vectors are held in registers of their own: packed into one, each load would wait for the last)
template <typename VT> struct Held { using type = VT; };
template <> struct Held<uint8_t> { using type = uint32_t; };
template <> struct Held<uint16_t> { using type = uint32_t; };
template <typename VT, bool SET, bool STREAM, int kInFlight = kWideInFlight>
__device__ __forceinline__ void move_wide_row(char *dense, char *table, char *second, int64_t row_bytes) {
  constexpr int64_t step = kWave * static_cast<int64_t>(sizeof(VT));
  for (int64_t off = lane_id() * static_cast<int64_t>(sizeof(VT)); off < row_bytes; off += kInFlight * step) {
    typename Held<VT>::type v[kInFlight];
#pragma unroll
    for (int u = 0; u < kInFlight; ++u) {
      if (off + u * step >= row_bytes) continue;
      if (SET && STREAM)
        v[u] = __builtin_nontemporal_load(reinterpret_cast<const VT *>(dense + off + u * step));
      else
        v[u] = gload<VT>((SET ? dense : table) + off + u * step);
    }
#pragma unroll
    for (int u = 0; u < kInFlight; ++u) {
      if (off + u * step >= row_bytes) continue;
      const VT x = static_cast<VT>(v[u]);
      if (SET) {
        gstore<VT>(table + off + u * step, x);
        if (second) gstore<VT>(second + off + u * step, x);
      } else if (STREAM) {
        __builtin_nontemporal_store(x, reinterpret_cast<VT *>(dense + off + u * step));
      } else {
        gstore<VT>(dense + off + u * step, x);
      }
    }
  }
}
// Rows per wave tile, at most. 32 measured 2 % faster than 64 on all-hit rows (90 against 92 us) and the
// same on mixed hit / miss batches; 16 gains nothing more and costs the bucket-table probe 15 %.
constexpr int kMaxLog2Tile = 5;
constexpr int64_t kL2Bytes = 32ll << 20;      // the L2s together
constexpr int64_t kCacheBytes = 256ll << 20;  // the memory-side cache
constexpr int64_t kLargeOutput = 160ll << 20;  // an output that it does not hold beside the rows read

// THROUGH (set only, with a map or mask): rows that hit the cache are written
// to the id-addressed table as well, so that table never goes stale.
// DEFER (fetch only, with a map or mask; tiles of exactly 32 rows): rows that
// miss the cache are not moved; every tile leaves one word of a bitmap that
// marks them for rows_missed_kernel (no counter, no atomics, nothing to clear).
template <typename VT, int MODE, bool SET, int ROUTE, bool THROUGH = false, bool DEFER = false>
__global__ __launch_bounds__(kRowsBlock, rows_waves_per_simd(SET, THROUGH, ROUTE, sizeof(VT))) void rows_kernel(RowArgs a) {
  static_assert(!THROUGH || (SET && MODE != kDirect), "write-through is a cached set");
  static_assert(!DEFER || (!SET && MODE != kDirect), "only a cached fetch sets its misses aside");
  const int lane = lane_id();
  const int L = 1 << a.log2_lanes;
  const int gl = lane & (L - 1);
  const int grp = lane >> a.log2_lanes;
  const int rows_per_step = kWave >> a.log2_lanes;
  const int tile = 1 << a.log2_tile;
  const int64_t waves_per_block = blockDim.x / kWave;
  const int64_t wave = static_cast<int64_t>(blockIdx.x) * waves_per_block + threadIdx.x / kWave;
  const int64_t nwaves = static_cast<int64_t>(gridDim.x) * waves_per_block;
  const int64_t R = a.row_bytes;
  const int64_t my_off = static_cast<int64_t>(gl) * sizeof(VT);
  int64_t Q = a.Q;
  if (a.count) {
    const int64_t counted = *a.count;
    if (counted < Q) Q = counted;
    if (a.count_seen && blockIdx.x == 0 && threadIdx.x == 0) {
      publish_size(a.count_seen, counted);
    }
  }

  // ---- phase 1, pipelined over the wave's tiles ----
  // Where a row lives takes two dependent loads (its id, then the map entry) before the row itself can be
  // touched. A wave with several tiles to do keeps those loads ahead of the rows: while the rows of tile t
  // move, the map loads of tile t + 1 and the ids of tile t + 2 are in flight, and what is looked at next has
  // long arrived. Measured on the hits of a 1,048,576-row Zipf batch (256-byte rows, hot rows in the caches,
  // 1.28 GB bucket table): 84 us with the three steps one after the other per tile, 72 us with the ids kept
  // ahead; all-hit uniform rows through the rank bitmap 107.6 -> 105 us.
  const int64_t stride = nwaves * tile;
  const int64_t base0 = wave * tile;
  if (base0 >= Q) return;  // (whole waves only: no barrier follows)
  struct Ids {  // step A: the ids of a tile (and its mask entries), one row per lane
    int64_t idx, masked;
    bool live;
  };
  auto load_ids = [&](int64_t base) {
    Ids t;
    const int64_t i = base + lane;
    t.live = lane < tile && i < Q;
    t.idx = t.live ? load_int(a.indices, i, a.idx_bytes) : 0;
    t.masked = -1;
    if (MODE == kMask && t.live) t.masked = load_int(a.mask, i, a.mask_bytes);
    return t;
  };
  struct Lookup {  // step B: the map loads of a tile, in flight
    int64_t idx, key, masked;
    bool live;
    HalfWaveProbe probe;
    FlatPending flat;
  };
  // Map entries are read with the streaming policy (see half_wave_issue) until a tile of this wave shows a
  // repeated id: from then on the wave takes the access for skewed and lets the caches keep what it reads.
  bool stream = streamable(a.map);
  auto start_lookup = [&](const Ids &t, Lookup *l) {
    l->idx = t.idx;
    l->masked = t.masked;
    l->live = t.live;
    l->key = -1;
    if (MODE == kMap16 || MODE == kMap8) {
      constexpr int FMT = MODE == kMap16 ? kSlot16 : kSlot8;
      l->key = t.live ? map_key(a.map, t.idx) : -1;
      if (stream && tile_repeats(l->key, t.live)) stream = false;
      if (stream)
        half_wave_issue<FMT, true>(a.map, l->key, &l->probe);
      else
        half_wave_issue<FMT, false>(a.map, l->key, &l->probe);
    } else if (MODE == kMapFlat) {
      // direct, rank or range form of the map: one load, or arithmetic only
      l->key = t.live ? map_key(a.map, t.idx) : -1;
      if (stream && tile_repeats(l->key, t.live)) stream = false;
      if (stream)
        l->flat = flat_issue<true>(a.map, l->key);
      else
        l->flat = flat_issue<false>(a.map, l->key);
    }
  };
  auto finish_lookup = [&](const Lookup &l) -> int64_t {  // step C: the slot of this lane's row, or -1
    if (MODE == kMask) return l.masked;
    if (MODE == kMap16) return half_wave_finish<kSlot16>(a.map, l.key, l.probe);
    if (MODE == kMap8) return half_wave_finish<kSlot8>(a.map, l.key, l.probe);
    if (MODE == kMapFlat) return l.live ? flat_finish(a.map, l.key, l.flat) : -1;
    return -1;
  };
  // (Bucket maps keep only the ids ahead: four bucket fragments per lane held across the row moves cost more
  // registers than eight resident waves per SIMD leave, and the spills cost more than the overlap gains.)
  constexpr bool kLookupAhead = MODE != kMap16 && MODE != kMap8;
  Ids ids_next = load_ids(base0), ids_after = load_ids(base0 + stride);
  Lookup ahead;
  start_lookup(ids_next, &ahead);
  int64_t slot = finish_lookup(ahead);
  int64_t idx = ahead.idx;
  bool live = ahead.live;
  if (kLookupAhead) {
    if (base0 + stride < Q) start_lookup(ids_after, &ahead);
    ids_after = load_ids(base0 + 2 * stride);
  }

  for (int64_t base = base0; base < Q; base += stride) {
    if (DEFER) {
      const uint64_t missed = __builtin_amdgcn_ballot_w64(live && slot < 0);
      if (lane == 0) a.miss_bits[base >> 5] = static_cast<uint32_t>(missed);
    }
    const int64_t my_table_row =
        DEFER && slot < 0 ? 0 : reinterpret_cast<int64_t>(slot >= 0 ? a.cache + slot * R : a.miss + idx * R);
    // write-through: second destination of a row that hit (0: none)
    const int64_t my_second_row =
        THROUGH && slot >= 0 ? reinterpret_cast<int64_t>(a.miss + idx * R) : 0;
    const int nrows = static_cast<int>(Q - base < tile ? Q - base : tile);

    // ---- phase 2: move the rows ----
    if (ROUTE == kOneVec) {
      // row_bytes <= L * sizeof(VT): one vector per lane per row
      const bool in = my_off < R;
      for (int r0 = 0; r0 < nrows; r0 += kRowsInFlight * rows_per_step) {
        VT v[kRowsInFlight];
        char *trow[kRowsInFlight];
        char *second[kRowsInFlight];
        // shuffles run with every lane active: a lane can only read the row
        // address held by a lane that takes part in the same instruction
#pragma unroll
        for (int u = 0; u < kRowsInFlight; ++u) {
          trow[u] = reinterpret_cast<char *>(
              shfl64(my_table_row, (r0 + u * rows_per_step + grp) & (kWave - 1)));
          second[u] = THROUGH ? reinterpret_cast<char *>(shfl64(
                                    my_second_row, (r0 + u * rows_per_step + grp) & (kWave - 1)))
                              : nullptr;
        }
#pragma unroll
        for (int u = 0; u < kRowsInFlight; ++u) {
          const int row = r0 + u * rows_per_step + grp;
          if (row < nrows && in && (!DEFER || trow[u])) {
            if (SET)
              v[u] = __builtin_nontemporal_load(
                  reinterpret_cast<const VT *>(a.dense + (base + row) * R + my_off));
            else
              v[u] = gload<VT>(trow[u] + my_off);
          }
        }
#pragma unroll
        for (int u = 0; u < kRowsInFlight; ++u) {
          const int row = r0 + u * rows_per_step + grp;
          if (row < nrows && in && (!DEFER || trow[u])) {
            if (SET) {
              gstore<VT>(trow[u] + my_off, v[u]);
              if (THROUGH && second[u]) gstore<VT>(second[u] + my_off, v[u]);
            } else
              __builtin_nontemporal_store(
                  v[u], reinterpret_cast<VT *>(a.dense + (base + row) * R + my_off));
          }
        }
      }
    } else if (ROUTE == kWide) {
      for (int row = 0; row < nrows; ++row) {
        char *const trow = reinterpret_cast<char *>(lane64(my_table_row, row));
        char *const second = THROUGH ? reinterpret_cast<char *>(lane64(my_second_row, row)) : nullptr;
        if (DEFER && !trow) continue;
        char *const drow = a.dense + (base + row) * R;
        if (!SET && !DEFER && sizeof(VT) == 16 && a.link_rows && (MODE == kDirect || lane64(slot, row) < 0))
          move_wide_row<VT, SET, false, 1>(drow, trow, second, R);
        else if (may_stream(SET, sizeof(VT)) && a.stream_dense)
          move_wide_row<VT, SET, may_stream(SET, sizeof(VT))>(drow, trow, second, R);
        else
          move_wide_row<VT, SET, false>(drow, trow, second, R);
      }
    } else {
      constexpr int kVecsInFlight = vecs_in_flight(SET, sizeof(VT));
      const uint32_t total = static_cast<uint32_t>(nrows) * a.nvec;
      char *const dense = a.dense + base * R;  // the tile's rows lie one behind the other
      // Rows that come over the host link get a lane group each after all: a row that is split between two steps, or
      // whose vectors are shifted against the groups of four lanes that read a line together, costs link reads (16,384
      // rows, 5 % hits, 50 floats: 95 us in lane groups, 101 dealt out; 20 floats: 66 / 67.5), unless a lane group would
      // be half empty (33 floats: 78 / 81, with 90 % hits 15.0 / 13.7). From one row in 16 on the link is what the
      // tile waits for.
      uint32_t per_step = kVecsInFlight * kWave, my_vec = lane;
      if (!SET && !DEFER && a.group_step &&
          16 * __builtin_popcountll(__builtin_amdgcn_ballot_w64(live && slot < 0)) >= nrows) {
        per_step = a.group_step;
        my_vec = static_cast<uint32_t>(gl) < a.nvec ? static_cast<uint32_t>(grp) * a.nvec + gl : 1u << 31;  // (an idle lane)
      }
      for (uint32_t v0 = 0; v0 < total; v0 += per_step) {
        VT v[kVecsInFlight];
        char *at[kVecsInFlight];
        char *second[kVecsInFlight];
        bool on[kVecsInFlight];
#pragma unroll
        for (int u = 0; u < kVecsInFlight; ++u) {  // (every lane takes part in the shuffles)
          const uint32_t i = v0 + u * kWave + my_vec;
          uint32_t row = __umulhi(i, a.nvec_magic);
          uint32_t vec = i - row * a.nvec;
          if (vec >= a.nvec) {
            ++row;
            vec -= a.nvec;
          }
          const uint32_t off = vec * static_cast<uint32_t>(sizeof(VT));
          char *const trow = reinterpret_cast<char *>(shfl64(my_table_row, row & (kWave - 1)));
          on[u] = i < total && (!DEFER || trow);
          at[u] = trow + off;
          second[u] = nullptr;
          if (THROUGH) {
            char *const srow = reinterpret_cast<char *>(shfl64(my_second_row, row & (kWave - 1)));
            second[u] = srow ? srow + off : nullptr;
          }
        }
#pragma unroll
        for (int u = 0; u < kVecsInFlight; ++u) {
          if (!on[u]) continue;
          if (SET)
            v[u] = __builtin_nontemporal_load(reinterpret_cast<const VT *>(dense) + (v0 + u * kWave + my_vec));
          else
            v[u] = gload<VT>(at[u]);
        }
#pragma unroll
        for (int u = 0; u < kVecsInFlight; ++u) {
          if (!on[u]) continue;
          if (SET) {
            gstore<VT>(at[u], v[u]);
            if (THROUGH && second[u]) gstore<VT>(second[u], v[u]);
          } else {
            __builtin_nontemporal_store(v[u], reinterpret_cast<VT *>(dense) + (v0 + u * kWave + my_vec));
          }
        }
      }
    }
    // ---- the next tile's lookup ends here; the one after starts; the ids of the one after that are asked for ----
    if (base + stride < Q) {
      if (!kLookupAhead) start_lookup(ids_after, &ahead);
      slot = finish_lookup(ahead);
      idx = ahead.idx;
      live = ahead.live;
      if (kLookupAhead) {
        if (base + 2 * stride < Q) start_lookup(ids_after, &ahead);
        ids_after = load_ids(base + 3 * stride);
      } else {
        ids_after = load_ids(base + 2 * stride);
      }
    }
  }
}

// Second half of a fetch whose misses were set aside (rows_kernel with DEFER):
// moves the rows marked in the bitmap from the id-addressed table. These are
// host-link reads when the table lives in pinned host memory. The link is
// saturated by the reads of a few dozen waves, and every read beyond that only
// lengthens the queue that all other link traffic of the GPU (the cold
// adjacency of the next mini-batch's sampling) and, measured, even its HBM
// traffic waits in; so the grid is small by design and the rest of the GPU
// stays free for what other streams have queued.
// A wave takes kMissedChunk bitmap words (32 rows each) per pass: one lane per
// word, a wave scan of the popcounts, the set bits expanded into a position
// list in LDS; then lane groups move kMissedRows rows at a time, all their
// loads issued before the first store.
struct MissedArgs {
  const char *table;
  char *dense;
  const void *indices;
  const uint32_t *bits;
  const int64_t *count;  // optional: only the first min(rows, *count) rows exist
  int64_t rows;
  int64_t row_bytes;
  int idx_bytes;
  int log2_lanes;
};

constexpr int kMissedRows = 2;     // rows a lane group has in flight
constexpr int kMissedChunk = 32;   // bitmap words per wave pass: 1,024 rows
constexpr int kMissedBlocks = 48;  // default grid

__global__ __launch_bounds__(kRowsBlock) void rows_missed_kernel(MissedArgs a) {
  using VT = u32x4;
  __shared__ uint32_t positions[kRowsBlock / kWave][kMissedChunk * 32];
  const int lane = lane_id();
  const int L = 1 << a.log2_lanes;
  const int gl = lane & (L - 1);
  const int grp = lane >> a.log2_lanes;
  const int rows_per_step = kWave >> a.log2_lanes;
  const int per_pass = kMissedRows * rows_per_step;  // <= 16: lane groups hold 8 lanes at least
  const int wave_in_block = threadIdx.x / kWave;
  const int64_t waves_per_block = blockDim.x / kWave;
  const int64_t wave = static_cast<int64_t>(blockIdx.x) * waves_per_block + wave_in_block;
  const int64_t nwaves = static_cast<int64_t>(gridDim.x) * waves_per_block;
  const int64_t R = a.row_bytes;
  const int64_t step = static_cast<int64_t>(L) * sizeof(VT);
  const int64_t my_off = static_cast<int64_t>(gl) * sizeof(VT);
  int64_t Q = a.rows;
  if (a.count) {
    const int64_t counted = *a.count;
    if (counted < Q) Q = counted < 0 ? 0 : counted;
  }
  const int64_t nwords = (Q + 31) >> 5;
  uint32_t *const mine = positions[wave_in_block];
  // Words are dealt to the waves one by one (word w0 + lane * nwaves to lane `lane` of wave w0), not in
  // runs: misses cluster (the first rows of a mini-batch's input nodes are its seeds, mostly cold), and a
  // wave that owned a run of 1,024 such rows would still be moving them long after the others were done.
  for (int64_t w0 = wave; w0 < nwords; w0 += nwaves * kMissedChunk) {
    const int64_t my_word = w0 + lane * nwaves;
    uint32_t word = 0;
    if (lane < kMissedChunk && my_word < nwords) word = a.bits[my_word];
    const uint32_t cnt = __builtin_popcount(word);
    const uint32_t inc = wave_inclusive_scan(cnt);
    const int total = static_cast<int>(wave_last(inc));
    uint32_t at = inc - cnt;
    while (word) {
      mine[at++] = static_cast<uint32_t>(my_word << 5) + static_cast<uint32_t>(__builtin_ctz(word));
      word &= word - 1;
    }
    // the list is written and read by this wave only: order its LDS accesses, no workgroup barrier
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int e0 = 0; e0 < total; e0 += per_pass) {
      int64_t my_src = 0, my_dst = 0;
      if (lane < per_pass && e0 + lane < total) {
        const int64_t pos = mine[e0 + lane];
        const int64_t idx = load_int(a.indices, pos, a.idx_bytes);
        my_src = reinterpret_cast<int64_t>(a.table + idx * R);
        my_dst = reinterpret_cast<int64_t>(a.dense + pos * R);
      }
      const char *src[kMissedRows];
      char *dst[kMissedRows];
#pragma unroll
      for (int u = 0; u < kMissedRows; ++u) {
        src[u] = reinterpret_cast<const char *>(shfl64(my_src, u * rows_per_step + grp));
        dst[u] = reinterpret_cast<char *>(shfl64(my_dst, u * rows_per_step + grp));
      }
      for (int64_t off = my_off; off < R; off += step) {
        VT v[kMissedRows];
#pragma unroll
        for (int u = 0; u < kMissedRows; ++u)
          if (src[u]) v[u] = gload<VT>(src[u] + off);
#pragma unroll
        for (int u = 0; u < kMissedRows; ++u)
          if (src[u]) __builtin_nontemporal_store(v[u], reinterpret_cast<VT *>(dst[u] + off));
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

template <int ROUTE>
static void launch_defer(int mode, unsigned grid, hipStream_t s, const RowArgs &a) {
  switch (mode) {
    case kMap16:
      hipLaunchKernelGGL((rows_kernel<u32x4, kMap16, false, ROUTE, false, true>), dim3(grid), dim3(kRowsBlock), 0, s, a);
      break;
    case kMap8:
      hipLaunchKernelGGL((rows_kernel<u32x4, kMap8, false, ROUTE, false, true>), dim3(grid), dim3(kRowsBlock), 0, s, a);
      break;
    case kMapFlat:
      hipLaunchKernelGGL((rows_kernel<u32x4, kMapFlat, false, ROUTE, false, true>), dim3(grid), dim3(kRowsBlock), 0, s, a);
      break;
    default:
      hipLaunchKernelGGL((rows_kernel<u32x4, kMask, false, ROUTE, false, true>), dim3(grid), dim3(kRowsBlock), 0, s, a);
      break;
  }
}

static int pick_vector_bytes(int64_t row_bytes, const void *p0, const void *p1, const void *p2) {
  uintptr_t bits = static_cast<uintptr_t>(row_bytes);
  bits |= reinterpret_cast<uintptr_t>(p0) | reinterpret_cast<uintptr_t>(p1) |
          reinterpret_cast<uintptr_t>(p2);
  int v = 16;
  while (v > 1 && (bits & (v - 1))) v >>= 1;
  return v;
}

template <typename VT, int ROUTE>
static void launch_through(int mode, unsigned grid, hipStream_t s, const RowArgs &a) {
  switch (mode) {
    case kMap16:
      hipLaunchKernelGGL((rows_kernel<VT, kMap16, true, ROUTE, true>), dim3(grid), dim3(kRowsBlock), 0, s, a);
      break;
    case kMap8:
      hipLaunchKernelGGL((rows_kernel<VT, kMap8, true, ROUTE, true>), dim3(grid), dim3(kRowsBlock), 0, s, a);
      break;
    case kMapFlat:
      hipLaunchKernelGGL((rows_kernel<VT, kMapFlat, true, ROUTE, true>), dim3(grid), dim3(kRowsBlock), 0, s, a);
      break;
    default:
      hipLaunchKernelGGL((rows_kernel<VT, kMask, true, ROUTE, true>), dim3(grid), dim3(kRowsBlock), 0, s, a);
      break;
  }
}

template <typename VT, bool SET, int ROUTE>
static void launch_mode(int mode, unsigned grid, hipStream_t s, const RowArgs &a) {
  switch (mode) {
    case kDirect:
      hipLaunchKernelGGL((rows_kernel<VT, kDirect, SET, ROUTE>), dim3(grid), dim3(kRowsBlock), 0, s, a);
      break;
    case kMap16:
      hipLaunchKernelGGL((rows_kernel<VT, kMap16, SET, ROUTE>), dim3(grid), dim3(kRowsBlock), 0, s, a);
      break;
    case kMap8:
      hipLaunchKernelGGL((rows_kernel<VT, kMap8, SET, ROUTE>), dim3(grid), dim3(kRowsBlock), 0, s, a);
      break;
    case kMapFlat:
      hipLaunchKernelGGL((rows_kernel<VT, kMapFlat, SET, ROUTE>), dim3(grid), dim3(kRowsBlock), 0, s, a);
      break;
    default:
      hipLaunchKernelGGL((rows_kernel<VT, kMask, SET, ROUTE>), dim3(grid), dim3(kRowsBlock), 0, s, a);
      break;
  }
}

template <typename VT, bool SET>
static void launch_vec(int route, bool through, int mode, unsigned grid, hipStream_t s,
                       const RowArgs &a) {
  if (SET && through && mode != kDirect) {
    if (route == kOneVec)
      launch_through<VT, kOneVec>(mode, grid, s, a);
    else if (route == kDealt)
      launch_through<VT, kDealt>(mode, grid, s, a);
    else
      launch_through<VT, kWide>(mode, grid, s, a);
    return;
  }
  if (route == kOneVec)
    launch_mode<VT, SET, kOneVec>(mode, grid, s, a);
  else if (route == kDealt)
    launch_mode<VT, SET, kDealt>(mode, grid, s, a);
  else
    launch_mode<VT, SET, kWide>(mode, grid, s, a);
}

// Rows of more vectors than this go one by one (kWide), shorter ones that fill no lane group are dealt out. All hits,
// us for 100 MB of output or update in all (for 400 MB), dealt out / one by one:
//   fetch  16-byte vectors  65: 50 / 42 (156 / 190), 75: 54 / 41 (171 / 190), 88: 58 / 41 (187 / 164), 128: 46 / 36 (163 / 166)
//          8-byte           65: 55 / 46 (186 / 194), 75: 59 / 45 (185 / 192; 314 MB 140 / 158), 89: 63 / 43 (187 / 190), 145: 74 / 42 (201 / 191)
//          4-byte           65: 30 / 38 (251 / 234), 89: 53 / 43 (243 / 200), 257: 122 / 55 (329 / 231)
//          2-byte           65: 25 / 25 (231 / 249; 160 MB 110 / 149), 89: 32 / 25 (348 / 273), 257: 140 / 65 (538 / 255)
//          1-byte           97: 27 / 24 (186 / 221), 113: 31 / 24 (257 / 237), 257: 91 / 57 (607 / 355)
//   set    16-byte          65: 54 / 57 (240 / 234), 75: 51 / 51 (233 / 227), 128: 41 / 44 (195 / 180)
//          8-byte           75: 53 / 57 (234 / 249), 97: 56 / 57 (254 / 244; 160 MB 90 / 98), 145: 69 / 53 (243 / 232)
//          4-byte           97: 55 / 60 (236 / 261), 127: 67 / 68 (252 / 266), 145: 72 / 58 (249 / 251), 257: 112 / 81 (330 / 288)
//          2-byte           75: 41 / 41 (291 / 291), 89: 47 / 42 (335 / 307), 257: 114 / 90 (398 / 334)
//          1-byte           65: 41 / 25 (292 / 244), 257: 131 / 66 (793 / 381)
// (With at most two loads in flight per lane, as dealt out, rows of 5 to 15 KB took up to 2.7 times as long.)
static int64_t wide_from(bool set, int vector_bytes, int64_t dense_bytes) {
  switch (vector_bytes) {
    case 16: return !set && dense_bytes > kLargeOutput ? 87 : 64;
    case 8: return set ? 112 : dense_bytes > kLargeOutput ? 87 : 64;
    case 4: return set ? 128 : 80;
    case 2: return 80;
    default: return set ? 64 : 112;
  }
}

// Whether `dense` is accessed past the caches (kWide). A fetch does so when the memory-side cache cannot hold its
// output (rows of 128 16-byte vectors, 400 MB: 178 us plain, 164 streaming; 100 MB: 36 / 38). A set does so with an
// update that would push the rows it writes out of that cache (100 MB: 49 plain, 44 streaming), but not with one
// small enough to lie in the L2s (512 vectors, 16 MB: 7.0 / 8.5), nor, when it is larger than the cache, with rows
// that do not end on a line (100 vectors, 400 MB: 193 / 213).
static bool stream_dense(bool set, int vector_bytes, int64_t row_bytes, int64_t dense_bytes) {
  if (!may_stream(set, vector_bytes)) return false;
  if (!set) return dense_bytes > kLargeOutput;
  return dense_bytes > kL2Bytes && (dense_bytes <= kCacheBytes || row_bytes % 128 == 0);
}

static bool in_host_memory(const void *p) {
  hipPointerAttribute_t attr;
  if (hipPointerGetAttributes(&attr, p) == hipSuccess) return attr.type == hipMemoryTypeHost;
  (void)hipGetLastError();
  return false;
}

template <bool SET>
static int move_rows(const char *who, void *miss, void *cache, const void *indices, int idx_bytes,
                     const shmt_hashmap_t *map, const void *mask, int mask_bytes, void *dense,
                     int64_t Q, int64_t row_bytes, void *stream, bool through = false,
                     const int64_t *count = nullptr, int64_t *count_seen = nullptr,
                     uint32_t *miss_bits = nullptr) {
  SHMT_REQUIRE(Q >= 0, "%s: Q must be >= 0", who);
  SHMT_REQUIRE(row_bytes > 0, "%s: row_bytes must be > 0", who);
  SHMT_REQUIRE(width_ok(idx_bytes), "%s: ID can only be int32 or int64 (idx_bytes=%d)", who, idx_bytes);
  SHMT_REQUIRE(!(map && mask), "%s: pass a hashmap or a mask, not both", who);
  if (Q == 0) return SHMT_OK;
  SHMT_REQUIRE(indices != nullptr && dense != nullptr, "%s: null indices/rows buffer", who);
  SHMT_REQUIRE(miss != nullptr, "%s: the id-addressed table is null", who);
  int mode = kDirect;
  if (map) {
    mode = map->kind != kKindBuckets ? kMapFlat : (map->fmt == kSlot16 ? kMap16 : kMap8);
    // an empty map never yields a slot, so an empty (null) cache table is fine with it
    SHMT_REQUIRE(cache != nullptr || map->n == 0, "%s: cache table is null", who);
  } else if (mask) {
    mode = kMask;
    SHMT_REQUIRE(width_ok(mask_bytes), "%s: mask can only be int32 or int64", who);
    SHMT_REQUIRE(cache != nullptr, "%s: cache table is null", who);
  }

  RowArgs a;
  a.miss = static_cast<char *>(miss);
  a.cache = static_cast<char *>(cache);
  a.dense = static_cast<char *>(dense);
  a.indices = indices;
  a.mask = mask;
  if (map) a.map = map->view; else a.map = empty_map_view();
  a.Q = Q;
  a.count = count;
  a.count_seen = count_seen;
  a.row_bytes = row_bytes;
  a.idx_bytes = idx_bytes;
  a.mask_bytes = mask_bytes;
  a.miss_bits = miss_bits;

  const int vb = pick_vector_bytes(row_bytes, miss, cache, dense);
  const int64_t nvec = row_bytes / vb;
  int log2_lanes = 3;
  while (log2_lanes < 6 && (1ll << log2_lanes) < nvec) ++log2_lanes;
  a.log2_lanes = log2_lanes;
  // Tile of 64 rows per wave when there are rows enough to occupy the chip
  // (256 CUs x 8 waves); fewer rows per wave otherwise, down to one phase-2 step.
  // A lane group per row where the row fills it. A fetch of 16-byte vectors also where it fills three quarters of
  // 8, 16 or 32 lanes: 262,144 rows of 100 floats 44.4 us, 45.7 with the vectors dealt out, 112 floats 45.0 / 45.7;
  // but with 64 lanes 200 floats 92.0 / 81.4, 208 floats 82.6 / 81.0, 240 floats 97.2 / 95.5.
  const int64_t lanes = 1ll << log2_lanes;
  const bool one_vec = nvec == lanes || (!SET && vb == 16 && lanes < kWave && nvec < lanes && 4 * nvec >= 3 * lanes);
  const int64_t dense_bytes = Q * row_bytes;
  // (misses of a fetch: rows over the host link)
  const bool link = !SET && !one_vec && in_host_memory(miss);
  const int64_t dealt_most = link && mode == kDirect ? kWave : wide_from(SET, vb, dense_bytes);
  const int route = one_vec ? kOneVec : nvec > dealt_most ? kWide : kDealt;
  a.stream_dense = stream_dense(SET, vb, row_bytes, dense_bytes);
  // (256 waves fill the link: 256 rows of 2,048 floats 40.3 us with one vector in flight, 43.3 with four; 64 rows of
  // 8,192 floats 45.9 / 40.2. Few missed rows among hits keep waves waiting that have long ones: 4,096 rows, 90 %
  // hits, of 8,192 floats 257 / 239, of 1,024 floats, 16,384 rows, 130 / 127, but with 20 % hits 946 / 988)
  a.link_rows = link && Q >= 256 && (mode == kDirect || nvec <= 1024);
  a.nvec = route == kDealt ? static_cast<uint32_t>(nvec) : 0u;
  a.nvec_magic = route == kDealt ? 0xFFFFFFFFu / a.nvec : 0u;
  const bool by_group = route == kDealt && link && nvec <= lanes && (mode == kDirect || 16 * nvec >= 9 * lanes);
  a.group_step = by_group ? (kWave >> log2_lanes) * a.nvec : 0u;
  int log2_tile = kMaxLog2Tile;
  int log2_least = one_vec ? 6 - log2_lanes : 0;  // fewest rows per tile: a wave's worth of vectors, or eight
  while (!one_vec && log2_least < 3 && (nvec << log2_least) < kWave) ++log2_least;
  while (log2_tile > log2_least && (Q >> log2_tile) < 2048) --log2_tile;
  if (miss_bits) log2_tile = 5;  // one bitmap word per tile
  a.log2_tile = log2_tile;
  // As many workgroups as the device holds at once (256 units x 8 waves per SIMD): beyond that a wave takes
  // several tiles and keeps the lookups of the next ones in flight while it moves rows.
  const unsigned grid = grid_for(Q, static_cast<int64_t>(kRowsBlock / kWave) << log2_tile,
                                 256 * rows_waves_per_simd(SET, through, route, vb));
  hipStream_t s = as_stream(stream);
  if (miss_bits) {
    SHMT_REQUIRE(!SET && mode != kDirect, "%s: only a fetch through a hashmap or mask sets its misses aside", who);
    SHMT_REQUIRE(vb == 16, "%s: rows and tables must allow 16-byte accesses (row_bytes %lld)", who,
                 static_cast<long long>(row_bytes));
    SHMT_REQUIRE(Q < (1ll << 32), "%s: at most 2^32 - 1 rows", who);
    if (route == kOneVec)
      launch_defer<kOneVec>(mode, grid, s, a);
    else if (route == kDealt)
      launch_defer<kDealt>(mode, grid, s, a);
    else
      launch_defer<kWide>(mode, grid, s, a);
    SHMT_LAUNCH_CHECK();
    return SHMT_OK;
  }
  switch (vb) {
    case 16: launch_vec<u32x4, SET>(route, through, mode, grid, s, a); break;
    case 8: launch_vec<u32x2, SET>(route, through, mode, grid, s, a); break;
    case 4: launch_vec<uint32_t, SET>(route, through, mode, grid, s, a); break;
    case 2: launch_vec<uint16_t, SET>(route, through, mode, grid, s, a); break;
    default: launch_vec<uint8_t, SET>(route, through, mode, grid, s, a); break;
  }
  SHMT_LAUNCH_CHECK();
  return SHMT_OK;
}

}  // namespace shmt

extern "C" {

int shmt_fetch(const void *miss_data, const void *cache_data, const void *indices, int idx_bytes,
               const shmt_hashmap_t *map, const void *mask, int mask_bytes, void *out, int64_t Q,
               int64_t row_bytes, void *stream) {
  return shmt::move_rows<false>("shmt_fetch", const_cast<void *>(miss_data),
                                const_cast<void *>(cache_data), indices, idx_bytes, map, mask,
                                mask_bytes, out, Q, row_bytes, stream);
}

int shmt_fetch_counted(const void *miss_data, const void *cache_data, const void *indices,
                       int idx_bytes, const shmt_hashmap_t *map, const void *mask, int mask_bytes,
                       void *out, int64_t max_rows, const int64_t *count, int64_t *count_seen,
                       int64_t row_bytes, void *stream) {
  SHMT_REQUIRE(count != nullptr, "shmt_fetch_counted: count is null");
  return shmt::move_rows<false>("shmt_fetch_counted", const_cast<void *>(miss_data),
                                const_cast<void *>(cache_data), indices, idx_bytes, map, mask,
                                mask_bytes, out, max_rows, row_bytes, stream, false, count, count_seen);
}

int shmt_fetch_cached_part(const void *miss_data, const void *cache_data, const void *indices, int idx_bytes,
                           const shmt_hashmap_t *map, const void *mask, int mask_bytes, void *out,
                           int64_t max_rows, const int64_t *count, int64_t row_bytes, uint32_t *miss_bits,
                           void *stream) {
  SHMT_REQUIRE(miss_bits != nullptr || max_rows == 0, "shmt_fetch_cached_part: miss_bits is null");
  SHMT_REQUIRE(map != nullptr || mask != nullptr, "shmt_fetch_cached_part: needs a hashmap or a mask");
  return shmt::move_rows<false>("shmt_fetch_cached_part", const_cast<void *>(miss_data),
                                const_cast<void *>(cache_data), indices, idx_bytes, map, mask, mask_bytes, out,
                                max_rows, row_bytes, stream, false, count, nullptr, miss_bits);
}

int shmt_fetch_missed_part(const void *miss_data, const void *indices, int idx_bytes, const uint32_t *miss_bits,
                           void *out, int64_t max_rows, const int64_t *count, int64_t row_bytes, int max_blocks,
                           void *stream) {
  using namespace shmt;
  SHMT_REQUIRE(width_ok(idx_bytes), "shmt_fetch_missed_part: ID can only be int32 or int64 (idx_bytes=%d)", idx_bytes);
  SHMT_REQUIRE(max_rows >= 0 && max_rows < (1ll << 32), "shmt_fetch_missed_part: max_rows must be in [0, 2^32)");
  SHMT_REQUIRE(max_blocks >= 0, "shmt_fetch_missed_part: max_blocks must be >= 0");
  if (max_rows == 0) return SHMT_OK;
  SHMT_REQUIRE(miss_data && indices && miss_bits && out, "shmt_fetch_missed_part: null buffer");
  SHMT_REQUIRE(row_bytes > 0 && pick_vector_bytes(row_bytes, miss_data, out, nullptr) == 16,
               "shmt_fetch_missed_part: rows and tables must allow 16-byte accesses (row_bytes %lld)",
               static_cast<long long>(row_bytes));
  MissedArgs a;
  a.table = static_cast<const char *>(miss_data);
  a.dense = static_cast<char *>(out);
  a.indices = indices;
  a.bits = miss_bits;
  a.count = count;
  a.rows = max_rows;
  a.row_bytes = row_bytes;
  a.idx_bytes = idx_bytes;
  int log2_lanes = 3;
  while (log2_lanes < 6 && (1ll << log2_lanes) < row_bytes / 16) ++log2_lanes;
  a.log2_lanes = log2_lanes;
  const int64_t chunks = ((max_rows + 31) / 32 + kMissedChunk - 1) / kMissedChunk;
  const unsigned grid = grid_for(chunks, kRowsBlock / kWave, max_blocks > 0 ? max_blocks : kMissedBlocks);
  hipLaunchKernelGGL(rows_missed_kernel, dim3(grid), dim3(kRowsBlock), 0, as_stream(stream), a);
  SHMT_LAUNCH_CHECK();
  return SHMT_OK;
}

int shmt_set(void *miss_data, void *cache_data, const void *indices, int idx_bytes,
             const shmt_hashmap_t *map, const void *mask, int mask_bytes, const void *update,
             int64_t Q, int64_t row_bytes, void *stream) {
  return shmt::move_rows<true>("shmt_set", miss_data, cache_data, indices, idx_bytes, map, mask,
                               mask_bytes, const_cast<void *>(update), Q, row_bytes, stream);
}

int shmt_set_through(void *miss_data, void *cache_data, const void *indices, int idx_bytes,
                     const shmt_hashmap_t *map, const void *mask, int mask_bytes, const void *update,
                     int64_t Q, int64_t row_bytes, void *stream) {
  return shmt::move_rows<true>("shmt_set_through", miss_data, cache_data, indices, idx_bytes, map, mask,
                               mask_bytes, const_cast<void *>(update), Q, row_bytes, stream, true);
}

}  // extern "C"

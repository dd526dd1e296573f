// layers.hip -- one layer of node-wise sampling (column slice + sample + unique +
// relabel) in three launches, for layers small enough that launches and the
// host's waits cost more than the work.
//
// The layer's keys are laid out with a fixed number of places per column, so that
// nothing has to be counted before it can be sampled: batch b, whose columns are
// [s_lo, s_lo + ns), owns (fanout + 1) ns positions from (fanout + 1) s_lo on -- its
// seeds first, then fanout places per column, of which a short column leaves some
// empty.  Order of positions = order of the keys of the layer (seeds of a batch,
// then its edges), so first occurrences, ranks and labels come out as they do from
// the packed layout.
//   pick    a column on fanout + 1 neighbouring lanes (its seed and its picks).
//           Keys are first made distinct inside the work-group in LDS -- a hub that
//           every column picks would otherwise be thousands of atomics on one
//           word -- and then go into one table in global memory, smallest position
//           first.  Every position keeps the slot its key landed in.
//   flag    every position reads the first position of its key from that slot; per
//           64 positions a word of which are first occurrences and one of which
//           are edges; counts per tile of 1024 positions
//   label   every work-group adds up the tiles' counts for itself (at most 1024),
//           then writes frontier, labels and offsets of its tile, and empties its
//           share of the table for the layer after the next.  Work-group 0 reports the
//           offsets of all batches to the host.
// A layer whose columns are the frontier of one that is queued ahead of it does not wait
// for that one's labels: its pick finds column c by the tiles' counts, in the list of new keys
// that flag left of each tile, and runs beside the label pass in one launch, with a table of its
// own.  L layers are 2 L + 1 dependent launches.
// GraphSAGE [25,10], 1024 seeds: six launches 44.5 us, label 6.0 and pick 9.2 of them; five
// 39.5, the two together 10.8 (51.5 and 47.1 us a pass).
// The number of columns is read from the device (the last entry of the previous
// layer's frontier offsets), launches are sized by its bound, and nothing is waited
// for between layers.
// GraphSAGE [25,10], 1024 seeds, 100 K nodes: 16 launches and four waits, 128 us,
// before; seven launches and one wait, 50 us, now.  The launches are chains of dependent
// loads, a round trip to memory each, so every load is sent off as soon as its address is
// known: ahead of the number of columns (a place below the bound is read whatever it
// holds), of the sum over the tiles, of the work-group's own dedup, and of the stores that
// empty the table (the six launches: 48.7 us without that, 41.8 with it; the nine of
// [15,10,5] in 8 batches 110.7 and 99.8).
#include "common.h"
#include "hashtable.h"

namespace gs {

constexpr int kPickThreads = 512;
constexpr int kLayerMaxBatches = 511;  // whose offsets a pick beside the labels finds for itself
static_assert(kLayerMaxBatches < kPickThreads, "a thread a batch");
constexpr int kPickSlots = 1024;  // LDS table of a work-group's keys, at most half full
constexpr int kPickShift = 22;    // 32 - log2(kPickSlots)
constexpr int kLayerTile = 1024;  // positions per work-group of flag and label
constexpr int kLayerWords = kLayerTile / kWave;
constexpr int kLayerWordsPerWave = kLayerWords / (kBlock / kWave);
constexpr int kLayerMaxTiles = 1024;
constexpr uint32_t kNoSlot = 0xFFFFFFFFu;
static_assert(kPickThreads * 2 <= kPickSlots, "the LDS table is at most half full");

// 64 positions: which are first occurrences / edges, and how many of either their
// tile has before them.
struct alignas(16) LayerWord {
  uint64_t first, edge;
  uint32_t first_before, edge_before;
  uint64_t unused;
};

struct LayerWs {
  uint64_t* table[2];  // [slots] key << 32 | first position, empty when a layer begins with it
  uint32_t* slot;      // [positions] slot of the position's key, kNoSlot: no key here
  uint32_t* first;     // [positions] first position of the key
  uint32_t* key;       // [positions] a tile's new keys in order, from its first position on
  LayerWord* words;    // [tiles * kLayerWords]
  uint2* tile_cnt;     // [tiles] first occurrences, edges
  int64_t* picked;     // [columns * fanout] rows of a weighted layer
  int32_t* wide;       // [1] raised by a seed that is no id of the matrix
  int64_t slots, tiles;
  size_t total;
};

static int64_t layer_table_slots(int64_t positions) {
  int64_t slots = 4096;
  while (slots < 2 * positions) slots <<= 1;
  return slots;
}

static LayerWs carve_layer(void* ws, int64_t positions, int weighted) {
  Carver c(ws);
  LayerWs w;
  const int64_t n = positions > 0 ? positions : 1;
  w.slots = layer_table_slots(n);
  w.tiles = ceil_div(n, kLayerTile);
  // (first, so that their places do not depend on the rest; weighted layers, which never run
  // beside another's labels, have the first alone)
  w.table[0] = c.take<uint64_t>((size_t)w.slots);
  w.table[1] = weighted ? nullptr : c.take<uint64_t>((size_t)w.slots);
  w.wide = c.take<int32_t>(1);
  w.slot = c.take<uint32_t>((size_t)n);
  w.first = c.take<uint32_t>((size_t)n);
  w.key = c.take<uint32_t>((size_t)n);
  w.words = c.take<LayerWord>((size_t)w.tiles * kLayerWords);
  w.tile_cnt = c.take<uint2>((size_t)w.tiles);
  w.picked = c.take<int64_t>(weighted ? (size_t)n : 1);
  w.total = c.total();
  return w;
}

// The layer's columns: ids, how many (on the device), and their batches.
struct LayerColumns {
  const int64_t* ids;
  const int64_t* ptr;  // [B + 1] offsets of the batches, null: one batch of `count`
  int64_t B, count;    // count: bound of the number of columns when ptr is given
  __device__ __forceinline__ int64_t num() const { return ptr ? ptr[B] : count; }
  // A place among those of the bound, for a load that does not wait for the number of
  // columns (what lies past that number is not looked at).
  __device__ __forceinline__ int64_t place(int64_t p, int64_t width) const {
    return p < count * width ? p : 0;
  }
  __device__ __forceinline__ int64_t lo(int64_t b) const { return ptr ? ptr[b] : 0; }
  __device__ __forceinline__ int64_t hi(int64_t b) const { return ptr ? ptr[b + 1] : count; }
  // batch of a column, at or after batch b0
  __device__ __forceinline__ int64_t batch_of(int64_t c, int64_t b0) const {
    if (!ptr) return 0;
    int64_t b = b0;
    while (b + 1 < B && ptr[b + 1] <= c) ++b;
    return b;
  }
};

// The batches' offsets, one a lane, where a wavefront has lanes for all of them: asked for
// once, beside a kernel's first loads, and compared with from then on, where a search takes a
// trip to the cache a step, and the ends of a batch two more.  All lanes call these together.
// kMany: of kernels for more batches than one; those for one have no code for any of it
// (two layers of 1024 seeds 39.2 us of kernels with it and 37.7 without, 47.9 and 46.2 a call).
template <bool kMany>
struct HeldBatches {
  int64_t at;  // ptr[lane], INT64_MAX past the last
  int B;
  bool held;
  __device__ __forceinline__ explicit HeldBatches(const LayerColumns& cols)
      : at(0), B((int)cols.B), held(kMany && cols.ptr && cols.B < kWave) {
    if (held) {
      at = cols.ptr[lane_id() <= B ? lane_id() : B];
      if (lane_id() > B) at = INT64_MAX;
    }
  }
  __device__ __forceinline__ int64_t ptr(int b) const { return __shfl((long long)at, b, kWave); }
  __device__ __forceinline__ int64_t num(const LayerColumns& cols) const {
    return held ? wave_uniform_first(ptr(B)) : cols.num();
  }
  // batch of column x / width, x the same in every lane and below the last batch's end
  __device__ __forceinline__ int of_uniform(int64_t x, int width) const {
    return __popcll(__ballot(lane_id() < B && at * width <= x)) - 1;
  }
  // batch of column x / width, which lies in one of lo to hi
  __device__ __forceinline__ int of(int64_t x, int width, int lo, int hi) const {
    int b = lo;
    for (int k = lo + 1; k <= hi; ++k)
      if (ptr(k) * width <= x) b = k;
    return b;
  }
};

// The slot of a key in the global table after (key, position) went in; `cur` is what its
// first slot was seen to hold.
__device__ __forceinline__ uint32_t layer_insert(uint64_t* table, uint32_t mask, uint32_t key,
                                                 uint32_t position, uint64_t cur) {
  const uint64_t mine = ((uint64_t)key << 32) | position;
  uint32_t slot = hash32(key) & mask;
  for (uint32_t probes = 0; probes <= mask; ++probes) {  // at most half full: ends early
    if (cur == kEmptySlot) {
      cur = atomicCAS((unsigned long long*)(table + slot), (unsigned long long)kEmptySlot,
                      (unsigned long long)mine);
      if (cur == kEmptySlot) return slot;
    }
    if ((uint32_t)(cur >> 32) == key) {
      // a stale read can only cost an atomic: positions of a slot only decrease
      if (cur > mine) atomicMin((unsigned long long*)(table + slot), (unsigned long long)mine);
      return slot;
    }
    slot = (slot + 1) & mask;
    cur = table[slot];
  }
  return 0;
}

// A column that a lane works for: its id, its batch's first column and how many that has.
struct PickColumn {
  int64_t id, b, s_lo, ns;
};

// What a lane of a pick knows before its column is.
struct PickLane {
  int64_t first_col, c;  // of the work-group; this lane's
  int group, lane, width;
  bool in_group;
  __device__ __forceinline__ PickLane(unsigned block, int fanout, int cols_per_wave) {
    const int wave_lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    first_col = (int64_t)block * (kPickThreads / kWave * cols_per_wave);
    width = fanout + 1;
    group = wave_lane / width;
    lane = wave_lane - group * width;  // 0: the seed, j + 1: pick j
    c = first_col + wave * cols_per_wave + group;
    in_group = group < cols_per_wave;
  }
};

struct PickShared {
  uint32_t tags[kPickSlots], mins[kPickSlots], global_slot[kPickSlots];
  __device__ __forceinline__ void clear() {
    for (int i = threadIdx.x; i < kPickSlots; i += kPickThreads) {
      tags[i] = kNoSlot;
      mins[i] = 0xFFFFFFFFu;
    }
  }
};

// The rest of a pick, behind sh.clear(): `column(&start, &deg)` gives the lane's column and where
// it lies, and is called by live lanes only.
// picked: rows drawn by another kernel, fanout places per column; null: uniform.
template <typename IdT, typename Column>
__device__ __forceinline__ void pick_columns(const PickLane& l, bool live, Column column,
                                             const IdT* __restrict__ indices, int fanout,
                                             int replace, PhiloxKey key, uint32_t stride,
                                             const int64_t* __restrict__ picked, uint64_t* table,
                                             uint32_t mask, uint32_t* __restrict__ slot_of,
                                             int32_t* wide, PickShared& sh) {
  uint32_t my_key = kNoSlot, position = 0;
  if (live) {
    int64_t start, deg;
    const PickColumn col = column(&start, &deg);
    const int64_t fb = col.s_lo * l.width, c = l.c;
    int64_t row = -1;
    if (l.lane == 0) {
      row = col.id;
      if ((uint64_t)col.id >= (uint64_t)stride) {  // no id of this matrix: the caller takes another path
        *wide = 1;
        row = 0;
      }
      position = (uint32_t)(fb + (c - col.s_lo));
    } else {
      position = (uint32_t)(fb + col.ns + (c - col.s_lo) * fanout + (l.lane - 1));
      const int64_t j = l.lane - 1;
      if (picked) {
        const int64_t have = replace ? (deg > 0 ? fanout : 0) : (deg < fanout ? deg : fanout);
        if (j < have) row = picked[c * fanout + j];
      } else if (replace) {
        if (deg > 0)
          row = (int64_t)indices[start + (int64_t)philox_bounded(key, (uint64_t)c, (uint64_t)j,
                                                                 (uint64_t)deg)];
      } else if (deg <= fanout) {
        if (j < deg) row = (int64_t)indices[start + j];
      } else {
        row = (int64_t)indices[start + floyd_slot((int)j, l.group * l.width + 1, fanout, deg, key,
                                                  (uint64_t)c)];
      }
    }
    if (row >= 0) my_key = (uint32_t)col.b * stride + (uint32_t)row;
  }
  // (looked at now, so that the answer is there when the work-group knows whose key it is)
  const uint64_t seen = my_key != kNoSlot ? table[hash32(my_key) & mask] : 0ull;
  __syncthreads();
  uint32_t at = 0;
  if (my_key != kNoSlot) {
    at = (my_key * 0x85EBCA6Bu) >> kPickShift;
    for (;;) {
      uint32_t cur = sh.tags[at];
      if (cur == kNoSlot) cur = atomicCAS(&sh.tags[at], kNoSlot, my_key);
      if (cur == kNoSlot || cur == my_key) break;
      at = (at + 1) & (kPickSlots - 1);
    }
    if (sh.mins[at] > position) atomicMin(&sh.mins[at], position);
  }
  __syncthreads();
  if (my_key != kNoSlot && sh.mins[at] == position)
    sh.global_slot[at] = layer_insert(table, mask, my_key, position, seen);
  __syncthreads();
  if (live) slot_of[position] = my_key != kNoSlot ? sh.global_slot[at] : kNoSlot;
}

template <typename IdT, bool kMany>
__global__ __launch_bounds__(kPickThreads) void layer_pick_kernel(
    const int64_t* __restrict__ indptr, int64_t num_cols, const IdT* __restrict__ indices,
    LayerColumns cols, int fanout, int cols_per_wave, int replace, PhiloxKey key, uint32_t stride,
    const int64_t* __restrict__ picked, uint64_t* table, uint32_t mask,
    uint32_t* __restrict__ slot_of, int32_t* wide) {
  __shared__ PickShared sh;
  const PickLane l(blockIdx.x, fanout, cols_per_wave);
  // one round trip for the number of columns and the id, of a place that may be no column's
  const int64_t id = cols.ids[cols.place(l.c, 1)];
  const HeldBatches<kMany> batches(cols);
  const int64_t n = batches.num(cols);
  if (l.first_col >= n) return;  // uniform per work-group
  sh.clear();
  int64_t held_b = 0, held_lo = 0, held_hi = 0;
  if (batches.held) {
    const int64_t last_col = l.first_col + kPickThreads / kWave * cols_per_wave - 1;
    const int b = batches.of(l.c, 1, batches.of_uniform(l.first_col, 1),
                             batches.of_uniform(last_col < n ? last_col : n - 1, 1));
    held_b = b;
    held_lo = batches.ptr(b);
    held_hi = batches.ptr(b + 1);
  }
  pick_columns(
      l, l.in_group && l.c < n,
      [&](int64_t* start, int64_t* deg) {
        *deg = column_degree(indptr, num_cols, id, start);
        if (batches.held) return PickColumn{id, held_b, held_lo, held_hi - held_lo};
        const int64_t b0 =
            kMany && cols.ptr ? segment_of(cols.ptr, cols.B, wave_uniform_first(l.first_col)) : 0;
        const int64_t b = kMany ? cols.batch_of(l.c, b0) : 0;
        return PickColumn{id, b, cols.lo(b), cols.hi(b) - cols.lo(b)};
      },
      indices, fanout, replace, key, stride, picked, table, mask, slot_of, wide, sh);
}

// What the work-groups of a tile know about the batches in it.
struct TileBatches {
  int64_t b_lo, b_hi;  // batches of the tile's first and last position
  __device__ __forceinline__ int64_t of(const LayerColumns& cols, int width, int64_t p) const {
    int64_t b = b_lo;
    while (b < b_hi && cols.ptr[b + 1] * width <= p) ++b;
    return b;
  }
};
template <bool kMany>
__device__ __forceinline__ TileBatches tile_batches(const LayerColumns& cols, const HeldBatches<kMany>& held,
                                                    int width, int64_t p0, int64_t p_last) {
  if (!kMany || !cols.ptr) return TileBatches{0, 0};
  if (held.held) return TileBatches{held.of_uniform(p0, width), held.of_uniform(p_last, width)};
  return TileBatches{segment_of(cols.ptr, cols.B, wave_uniform_first(p0 / width)),
                     segment_of(cols.ptr, cols.B, wave_uniform_first(p_last / width))};
}

template <bool kMany>
__global__ __launch_bounds__(kBlock) void layer_flag_kernel(
    LayerColumns cols, int fanout, const uint64_t* __restrict__ table,
    const uint32_t* __restrict__ slot_of, uint32_t* __restrict__ first,
    uint32_t* __restrict__ keys, LayerWord* __restrict__ words, uint2* __restrict__ tile_cnt) {
  __shared__ uint32_t wave_first[kBlock / kWave], wave_edge[kBlock / kWave];
  const int width = fanout + 1;
  const int64_t p0 = (int64_t)blockIdx.x * kLayerTile;
  const int wave = threadIdx.x / kWave, lane = lane_id();
  const int64_t wave_p0 = p0 + (int64_t)wave * kLayerWordsPerWave * kWave;
  uint32_t s[kLayerWordsPerWave], rank[kLayerWordsPerWave];
  uint64_t e[kLayerWordsPerWave];
#pragma unroll
  for (int j = 0; j < kLayerWordsPerWave; ++j)
    s[j] = slot_of[cols.place(wave_p0 + j * kWave + lane, width)];
  const HeldBatches<kMany> held(cols);
  const int64_t N = held.num(cols) * width;
  if (p0 >= N) return;
#pragma unroll
  for (int j = 0; j < kLayerWordsPerWave; ++j) {
    if (wave_p0 + j * kWave + lane >= N) s[j] = kNoSlot;
    e[j] = s[j] != kNoSlot ? table[s[j]] : 0ull;
  }
  const TileBatches batches =
      tile_batches(cols, held, width, p0, p0 + kLayerTile - 1 < N ? p0 + kLayerTile - 1 : N - 1);
  LayerWord mine{0ull, 0ull, 0u, 0u, 0ull};
  uint32_t firsts = 0, edges = 0;
#pragma unroll
  for (int j = 0; j < kLayerWordsPerWave; ++j) {
    const int64_t p = wave_p0 + j * kWave + lane;
    bool is_first = false, is_edge = false;
    int64_t s_lo = 0, s_hi = 0;
    if (held.held) {
      const int b = held.of(p, width, (int)batches.b_lo, (int)batches.b_hi);
      s_lo = held.ptr(b);
      s_hi = held.ptr(b + 1);
    }
    if (s[j] != kNoSlot) {
      const uint32_t f = (uint32_t)e[j];
      first[p] = f;
      is_first = f == (uint32_t)p;
      if (!held.held) {
        const int64_t b = batches.of(cols, width, p);
        s_lo = cols.lo(b);
        s_hi = cols.hi(b);
      }
      is_edge = p - s_lo * width >= s_hi - s_lo;
    }
    const uint64_t fw = __ballot(is_first), ew = __ballot(is_edge);
    if (lane == j) mine = LayerWord{fw, ew, firsts, edges, 0ull};
    rank[j] = is_first ? firsts + (uint32_t)__popcll(fw & ((1ull << lane) - 1ull)) : kNoSlot;
    firsts += (uint32_t)__popcll(fw);
    edges += (uint32_t)__popcll(ew);
  }
  if (lane == 0) {
    wave_first[wave] = firsts;
    wave_edge[wave] = edges;
  }
  __syncthreads();
  uint32_t fb = 0, eb = 0, fa = 0, ea = 0;
#pragma unroll
  for (int w = 0; w < kBlock / kWave; ++w) {
    if (w < wave) {
      fb += wave_first[w];
      eb += wave_edge[w];
    }
    fa += wave_first[w];
    ea += wave_edge[w];
  }
#pragma unroll
  for (int j = 0; j < kLayerWordsPerWave; ++j)
    if (rank[j] != kNoSlot) keys[p0 + fb + rank[j]] = (uint32_t)(e[j] >> 32);
  if (lane < kLayerWordsPerWave) {
    mine.first_before += fb;
    mine.edge_before += eb;
    words[(int64_t)blockIdx.x * kLayerWords + wave * kLayerWordsPerWave + lane] = mine;
  }
  if (threadIdx.x == 0) tile_cnt[blockIdx.x] = make_uint2(fa, ea);
}

struct LayerOut {
  int64_t *frontier, *frontier_ptr, *row, *col, *edge_ptr, *block_indptr;  // block_indptr may be null
  // for the host: frontier_ptr[B + 1], edge_ptr[B + 1], seeds distinct[B], wide seeds[1]
  int64_t* mirror;
};

// What a layer's flag pass left, and what its label pass empties.
struct LayerLabels {
  LayerColumns cols;
  int fanout;
  uint32_t stride;
  const uint32_t *first, *keys;
  const LayerWord* words;
  const uint2* tile_cnt;
  uint64_t* table;
  int64_t table_slots;
  const int32_t* wide;
  LayerOut out;
};
struct LabelShared {
  uint2 before[kLayerMaxTiles];  // first occurrences and edges before a tile
  uint64_t smem[kPickThreads / kWave + 1];
};

// Work-group `block` of `blocks`.  kThreads: of the launch (alone 11.6 us with 256 and 12.8
// with 512 on 150 K positions).
template <int kThreads, bool kMany>
__device__ __forceinline__ void label_tile(const LayerLabels& layer, unsigned block,
                                           unsigned blocks, LabelShared& sh) {
  const LayerColumns& cols = layer.cols;
  const int fanout = layer.fanout;
  const uint32_t stride = layer.stride;
  const uint32_t *__restrict__ first = layer.first, *__restrict__ keys = layer.keys;
  const LayerWord* __restrict__ words = layer.words;
  const uint2* __restrict__ tile_cnt = layer.tile_cnt;
  uint64_t* __restrict__ table = layer.table;
  const LayerOut& out = layer.out;
  uint2* before = sh.before;
  // The table is done with: its share emptied by every work-group of the launch, last of
  // all (loads behind stores are waited for with them).
  auto empty_table = [&] {
    for (int64_t i = (int64_t)block * kThreads + threadIdx.x; i < layer.table_slots;
         i += (int64_t)blocks * kThreads)
      table[i] = kEmptySlot;
  };
  const int width = fanout + 1;
  // What a position needs does not wait for the counts: its word, a key, and the word of
  // its key's first position travel while the tiles are added up, and so do the words of
  // the tile's first batch.
  constexpr int kItems = kLayerTile / kThreads;
  const int64_t p0 = (int64_t)block * kLayerTile;
  LayerWord word[kItems];
  uint32_t key[kItems], first_of[kItems];
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const int64_t q = cols.place(p0 + i * kThreads + threadIdx.x, width);
    word[i] = words[q / kWave];
    key[i] = keys[q];
    first_of[i] = first[q];
  }
  constexpr int kPer = kLayerMaxTiles / kThreads;
  uint2 cnt[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j)
    cnt[j] = tile_cnt[(int64_t)threadIdx.x * kPer + j < blocks ? threadIdx.x * kPer + j : 0];
  const HeldBatches<kMany> held(cols);
  const int64_t n = held.num(cols), N = n * width;
  const int64_t tiles = (N + kLayerTile - 1) / kLayerTile;
  if (block != 0 && (int64_t)block >= tiles) return empty_table();
  const TileBatches batches =
      tile_batches(cols, held, width, p0, p0 + kLayerTile - 1 < N ? p0 + kLayerTile - 1 : N - 1);
  LayerWord first_word[kItems];
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const int64_t p = p0 + i * kThreads + threadIdx.x;
    // (no key was sent to this position: nothing was written there)
    const bool edge = p < N && ((word[i].edge >> (int)(p % kWave)) & 1ull);
    if (!edge) first_of[i] = 0;
    first_word[i] = words[first_of[i] / kWave];
  }
  int64_t b = batches.b_lo, b_of[kItems];
  int64_t s_lo, ns;
  if (held.held) {
    s_lo = wave_uniform_first(held.ptr((int)b));
    ns = wave_uniform_first(held.ptr((int)b + 1)) - s_lo;
  } else {
    s_lo = cols.lo(b);
    ns = cols.hi(b) - s_lo;
  }
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const int64_t p = p0 + i * kThreads + threadIdx.x;
    if (held.held) b_of[i] = held.of(p, width, (int)batches.b_lo, (int)batches.b_hi);
    else b_of[i] = p < N ? batches.of(cols, width, p) : b;
  }
  int64_t fb = s_lo * width;
  LayerWord word_b = words[cols.place(fb, width) / kWave];
  LayerWord word_q = words[cols.place(fb + (ns > 0 ? ns - 1 : 0), width) / kWave];
  uint64_t sum = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    if ((int64_t)threadIdx.x * kPer + j >= tiles) cnt[j] = make_uint2(0u, 0u);
    sum += ((uint64_t)cnt[j].y << 32) | cnt[j].x;
  }
  uint64_t total;
  uint64_t run = block_exclusive_sum<uint64_t, kThreads>(sum, sh.smem, &total);
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    before[threadIdx.x * kPer + j] = make_uint2((uint32_t)run, (uint32_t)(run >> 32));
    run += ((uint64_t)cnt[j].y << 32) | cnt[j].x;
  }
  __syncthreads();
  const uint32_t all_first = (uint32_t)total, all_edges = (uint32_t)(total >> 32);
  auto ranks_in = [&](const LayerWord& w, int64_t p, uint32_t* f, uint32_t* e) {
    if (p >= N) {  // counts before position p <= N
      *f = all_first;
      *e = all_edges;
      return;
    }
    const uint2 t = before[p / kLayerTile];
    const uint64_t below = (1ull << (int)(p % kWave)) - 1ull;
    *f = t.x + w.first_before + (uint32_t)__popcll(w.first & below);
    *e = t.y + w.edge_before + (uint32_t)__popcll(w.edge & below);
  };
  auto ranks = [&](int64_t p, uint32_t* f, uint32_t* e) {
    ranks_in(words[p < N ? p / kWave : 0], p, f, e);
  };
  auto rank_in = [&](const LayerWord& w, uint32_t p) {
    return before[p / kLayerTile].x + w.first_before +
           (uint32_t)__popcll(w.first & ((1ull << (int)(p % kWave)) - 1ull));
  };
  auto rank_first = [&](uint32_t p) { return rank_in(words[p / kWave], p); };
  // w: the word of the batch's last seed
  auto seeds_distinct = [&](const LayerWord& w, int64_t fb, int64_t ns, uint32_t f0) {
    if (ns == 0) return true;
    const int64_t q = fb + ns - 1;
    return ((w.first >> (int)(q % kWave)) & 1ull) &&
           rank_in(w, (uint32_t)q) - f0 == (uint32_t)(ns - 1);
  };
  if (block == 0) {
    for (int64_t b = threadIdx.x; b <= cols.B; b += kThreads) {
      const int64_t s_lo = b < cols.B ? cols.lo(b) : n;
      uint32_t f, e;
      ranks(s_lo * width, &f, &e);
      out.frontier_ptr[b] = f;
      out.edge_ptr[b] = e;
      store_for_host(out.mirror + b, f);
      store_for_host(out.mirror + (cols.B + 1) + b, e);
      if (b < cols.B) {
        const int64_t s_hi = cols.hi(b), last = s_lo * width + (s_hi > s_lo ? s_hi - s_lo - 1 : 0);
        if (out.block_indptr) {
          uint32_t f1, e1;
          ranks(s_hi * width, &f1, &e1);
          out.block_indptr[s_hi + b] = e1 - e;  // the last offset of the block
        }
        store_for_host(out.mirror + 2 * (cols.B + 1) + b,
                       seeds_distinct(words[cols.place(last, width) / kWave], s_lo * width,
                                      s_hi - s_lo, f)
                           ? 1
                           : 0);
      } else {
        store_for_host(out.mirror + 3 * cols.B + 2, *layer.wide);
      }
    }
  }
  if (p0 >= N) return empty_table();
  uint32_t f0, e0;
  ranks_in(word_b, fb, &f0, &e0);
  bool distinct = seeds_distinct(word_q, fb, ns, f0);
  const uint2 t = before[block];
  // the frontier's share of the tile: its new keys, in order
  const uint32_t tile_firsts = ((int64_t)block + 1 < tiles ? before[block + 1].x : all_first) - t.x;
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const uint32_t r = i * kThreads + threadIdx.x;
    if (r < tile_firsts) out.frontier[t.x + r] = (int64_t)(key[i] % stride);
  }
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const int64_t p = p0 + i * kThreads + threadIdx.x;
    if (p >= N) break;
    if (b_of[i] != b) {
      b = b_of[i];
      s_lo = cols.lo(b);
      ns = cols.hi(b) - s_lo;
      fb = s_lo * width;
      ranks(fb, &f0, &e0);
      distinct = seeds_distinct(words[cols.place(fb + (ns > 0 ? ns - 1 : 0), width) / kWave], fb, ns, f0);
    }
    const LayerWord& w = word[i];
    const int bit = (int)(p % kWave);
    const uint64_t below = (1ull << bit) - 1ull;
    const uint32_t local = (uint32_t)(p - fb);
    if (local < (uint32_t)ns) continue;
    const uint32_t slot = local - (uint32_t)ns;
    const uint32_t c = slot / (uint32_t)fanout;  // the column, counted in its batch
    const uint32_t e = t.y + w.edge_before + (uint32_t)__popcll(w.edge & below);
    if (out.block_indptr && slot - c * (uint32_t)fanout == 0)
      out.block_indptr[s_lo + c + b] = e - e0;
    if ((w.edge >> bit) & 1ull) {
      out.row[e] = rank_in(first_word[i], first_of[i]) - f0;
      out.col[e] = distinct ? c : rank_first(first[fb + c]) - f0;
    }
  }
  empty_table();
}

template <bool kMany>
__global__ __launch_bounds__(kBlock) void layer_label_kernel(LayerLabels layer) {
  __shared__ LabelShared sh;
  label_tile<kBlock, kMany>(layer, blockIdx.x, gridDim.x, sh);
}

// Labels of a layer and picks of the one whose columns are its frontier: the first
// `pick_blocks` work-groups pick.
template <typename IdT, bool kMany>
__global__ __launch_bounds__(kPickThreads) void layer_label_pick_kernel(
    LayerLabels before, unsigned pick_blocks, const int64_t* __restrict__ indptr, int64_t num_cols,
    const IdT* __restrict__ indices, int fanout, int cols_per_wave, int replace, PhiloxKey key,
    uint64_t* table, uint32_t mask, uint32_t* __restrict__ slot_of, int32_t* wide) {
  if (blockIdx.x >= pick_blocks) {
    __shared__ LabelShared label;
    label_tile<kPickThreads, kMany>(before, blockIdx.x - pick_blocks, gridDim.x - pick_blocks, label);
    return;
  }
  __shared__ PickShared sh;
  __shared__ uint32_t tile_first[kLayerMaxTiles + 1];  // columns before a tile's
  __shared__ uint32_t batch_first[kLayerMaxBatches + 1];
  __shared__ uint32_t smem[kPickThreads / kWave + 1];
  const int t = threadIdx.x;
  const PickLane l(blockIdx.x, fanout, cols_per_wave);
  const LayerColumns& prev = before.cols;
  const int prev_width = before.fanout + 1;
  constexpr int kPer = kLayerMaxTiles / kPickThreads;
  const int64_t most_tiles = (prev.count * prev_width + kLayerTile - 1) / kLayerTile;
  uint32_t cnt[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j)
    cnt[j] = before.tile_cnt[t * kPer + j < most_tiles ? t * kPer + j : 0].x;
  const int64_t prev_n = prev.num(), N = prev_n * prev_width;
  const int64_t tiles = (N + kLayerTile - 1) / kLayerTile;
  // where a batch's keys begin, and the word of that position
  const int64_t p = t < prev.B ? prev.lo(t) * prev_width : N;
  const LayerWord word = before.words[p < N ? p / kWave : 0];
  sh.clear();
  uint32_t sum = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    if (t * kPer + j >= tiles) cnt[j] = 0;
    sum += cnt[j];
  }
  uint32_t n;
  uint32_t run = block_exclusive_sum<uint32_t, kPickThreads>(sum, smem, &n);
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    tile_first[t * kPer + j] = run;
    run += cnt[j];
  }
  if (t == 0) tile_first[kLayerMaxTiles] = n;
  if (l.first_col >= (int64_t)n) return;  // uniform per work-group
  __syncthreads();
  if (t <= prev.B)
    batch_first[t] = p >= N ? n
                            : tile_first[p / kLayerTile] + word.first_before +
                                  (uint32_t)__popcll(word.first & ((1ull << (int)(p % kWave)) - 1ull));
  __syncthreads();
  pick_columns(
      l, l.in_group && l.c < (int64_t)n,
      [&](int64_t* start, int64_t* deg) {
        const uint32_t c = (uint32_t)l.c;
        int lo = 0, hi = (int)tiles;  // tile_first[lo] <= c < tile_first[hi], whose tiles are done
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (tile_first[mid] <= c) lo = mid;
          else hi = mid;
        }
        const uint32_t found = before.keys[(int64_t)lo * kLayerTile + (c - tile_first[lo])];
        const uint32_t b = kMany ? found / before.stride : 0u;
        const int64_t id = (int64_t)(found - b * before.stride);
        *deg = column_degree(indptr, num_cols, id, start);
        return PickColumn{id, b, batch_first[b], batch_first[b + 1] - batch_first[b]};
      },
      indices, fanout, replace, key, before.stride, (const int64_t*)nullptr, table, mask, slot_of,
      wide, sh);
}

__global__ __launch_bounds__(kBlock) void layer_clear_kernel(uint64_t* table0, uint64_t* table1,
                                                             int64_t slots, int32_t* wide) {
  int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i == 0) *wide = 0;
  for (; i < slots; i += (int64_t)gridDim.x * kBlock) {
    table0[i] = kEmptySlot;
    if (table1) table1[i] = kEmptySlot;
  }
}

// weighted.hip: draws of a weighted layer into fanout places per column, the number
// of columns read from the device.
int launch_weighted_places(const int64_t* indptr, int64_t num_cols, const int64_t* indices,
                           const int64_t* cdf, const int64_t* column_ids, const int64_t* num_dev,
                           int64_t bound, int64_t fanout, int replace, PhiloxKey key,
                           int64_t* out_rows, hipStream_t s);

}  // namespace gs

extern "C" {

int64_t gs_layer_max_positions(void) { return (int64_t)gs::kLayerMaxTiles * gs::kLayerTile; }

size_t gs_layer_workspace_bytes(int64_t max_positions, int weighted) {
  if (max_positions < 0 || max_positions > gs_layer_max_positions()) return 0;
  return gs::carve_layer(nullptr, max_positions, weighted).total;
}

int gs_layer_begin(int64_t max_positions, int weighted, void* workspace, size_t workspace_bytes,
                   gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(max_positions >= 0 && max_positions <= gs_layer_max_positions(),
             "layer_begin: %lld positions", (long long)max_positions);
  const LayerWs w = carve_layer(workspace, max_positions, weighted);
  if (workspace == nullptr || workspace_bytes < w.total) {
    set_error("layer workspace too small: %zu < %zu", workspace_bytes, w.total);
    return GS_ERR_WORKSPACE;
  }
  int64_t blocks = ceil_div(w.slots, kBlock * 4);
  if (blocks > 2048) blocks = 2048;
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("layer_clear", s,
            layer_clear_kernel<<<dim3((unsigned)blocks), dim3(kBlock), 0, s>>>(
                w.table[0], w.table[1], w.slots, w.wide));
  return GS_OK;
}

int gs_sample_layer(const int64_t* indptr, int64_t num_cols, const int64_t* indices,
                    const int32_t* indices32, const int64_t* cdf, int64_t id_stride,
                    const int64_t* columns, int64_t num_columns, const int64_t* col_ptr,
                    int64_t num_batches, int64_t fanout, int replace, uint64_t seed,
                    uint64_t call_id, int64_t* out_frontier, int64_t* out_frontier_ptr,
                    int64_t* out_row, int64_t* out_col, int64_t* out_edge_ptr,
                    int64_t* out_block_indptr, int64_t* mirror,
                    int64_t max_positions, void* workspace, size_t workspace_bytes,
                    gs_stream_t stream) {
  const gs_layer layer{indptr, num_cols, indices, indices32, cdf, id_stride, columns, num_columns,
                       col_ptr, num_batches, fanout, replace, seed, call_id, out_frontier,
                       out_frontier_ptr, out_row, out_col, out_edge_ptr, out_block_indptr, mirror,
                       max_positions, workspace, workspace_bytes, 0};
  const int rc = gs_sample_layer_next(nullptr, &layer, stream);
  return rc != GS_OK ? rc : gs_sample_layer_next(&layer, nullptr, stream);
}

static int check_layer(const gs_layer& l) {
  using namespace gs;
  GS_REQUIRE(l.num_cols >= 0 && l.num_columns >= 1, "sample_layer: no columns");
  GS_REQUIRE(l.num_batches >= 1 && (l.col_ptr || l.num_batches == 1),
             "sample_layer: %lld batches need col_ptr", (long long)l.num_batches);
  GS_REQUIRE(l.fanout >= 1 && l.fanout < kWave, "sample_layer: fanout %lld", (long long)l.fanout);
  GS_REQUIRE(l.id_stride >= 1 && l.id_stride >= l.num_cols &&
                 l.num_batches <= (int64_t)0xFFFFFFFEll / l.id_stride,
             "sample_layer: %lld batches of ids below %lld", (long long)l.num_batches,
             (long long)l.id_stride);
  GS_REQUIRE(l.num_columns * (l.fanout + 1) <= l.max_positions &&
                 l.max_positions <= gs_layer_max_positions(),
             "sample_layer: %lld positions", (long long)(l.num_columns * (l.fanout + 1)));
  GS_REQUIRE(l.indptr && l.columns && l.out_frontier && l.out_frontier_ptr && l.out_row &&
                 l.out_col && l.out_edge_ptr && l.mirror,
             "sample_layer: null pointer");
  GS_REQUIRE(l.table == 0 || (l.table == 1 && !l.cdf), "sample_layer: table %d", l.table);
  const LayerWs w = carve_layer(l.workspace, l.max_positions, l.cdf != nullptr);
  if (l.workspace == nullptr || l.workspace_bytes < w.total) {
    set_error("layer workspace too small: %zu < %zu", l.workspace_bytes, w.total);
    return GS_ERR_WORKSPACE;
  }
  return GS_OK;
}

int gs_sample_layer_next(const gs_layer* before, const gs_layer* layer, gs_stream_t stream) {
  using namespace gs;
  int rc = before ? check_layer(*before) : GS_OK;
  if (rc == GS_OK && layer) rc = check_layer(*layer);
  if (rc != GS_OK) return rc;
  hipStream_t s = as_stream(stream);
  LayerLabels labels{};
  unsigned label_grid = 0;
  if (before) {
    const gs_layer& l = *before;
    const LayerWs w = carve_layer(l.workspace, l.max_positions, l.cdf != nullptr);
    const int64_t positions = l.num_columns * (l.fanout + 1);
    labels = LayerLabels{LayerColumns{l.columns, l.col_ptr, l.num_batches, l.num_columns},
                         (int)l.fanout, (uint32_t)l.id_stride, w.first, w.key, w.words, w.tile_cnt,
                         w.table[l.table], layer_table_slots(positions), w.wide,
                         LayerOut{l.out_frontier, l.out_frontier_ptr, l.out_row, l.out_col,
                                  l.out_edge_ptr, l.out_block_indptr, l.mirror}};
    label_grid = (unsigned)ceil_div(positions, kLayerTile);
  }
  // (beside the labels of the layer before, whose frontier its columns are)
  const bool beside = before && layer && !layer->cdf && layer->table != before->table &&
                      layer->workspace == before->workspace &&
                      layer->max_positions == before->max_positions && !before->cdf &&
                      layer->columns == before->out_frontier &&
                      layer->col_ptr == before->out_frontier_ptr &&
                      layer->num_batches == before->num_batches &&
                      layer->id_stride == before->id_stride &&
                      layer->num_batches <= kLayerMaxBatches;
  if (before && !beside)
    GS_LAUNCH("layer_label", s,
              if (before->num_batches > 1)
                layer_label_kernel<true><<<dim3(label_grid), dim3(kBlock), 0, s>>>(labels);
              else layer_label_kernel<false><<<dim3(label_grid), dim3(kBlock), 0, s>>>(labels));
  if (!layer) return GS_OK;
  const gs_layer& l = *layer;
  const LayerWs w = carve_layer(l.workspace, l.max_positions, l.cdf != nullptr);
  const int64_t positions = l.num_columns * (l.fanout + 1);
  const int64_t slots = layer_table_slots(positions);  // of the table, what this layer uses
  const PhiloxKey key = make_key(l.seed, l.call_id);
  const LayerColumns cols{l.columns, l.col_ptr, l.num_batches, l.num_columns};
  const int cols_per_wave = kWave / ((int)l.fanout + 1);
  const unsigned pick_grid =
      (unsigned)ceil_div(l.num_columns, (kPickThreads / kWave) * cols_per_wave);
  uint64_t* table = w.table[l.table];
  if (l.cdf) {
    rc = launch_weighted_places(l.indptr, l.num_cols, l.indices, l.cdf, l.columns,
                                l.col_ptr ? l.col_ptr + l.num_batches : nullptr, l.num_columns,
                                l.fanout, l.replace, key, w.picked, s);
    if (rc != GS_OK) return rc;
  }
#define GS_PICK(T, MANY, IDS)                                                                       \
  do {                                                                                        \
    if (beside)                                                                               \
      GS_LAUNCH("layer_label_pick", s,                                                        \
                (layer_label_pick_kernel<T, MANY>)<<<dim3(pick_grid + label_grid), dim3(kPickThreads), 0, \
                                             s>>>(                                            \
                    labels, pick_grid, l.indptr, l.num_cols, IDS, (int)l.fanout, cols_per_wave, \
                    l.replace, key, table, (uint32_t)(slots - 1), w.slot, w.wide));           \
    else                                                                                      \
      GS_LAUNCH("layer_pick", s,                                                              \
                (layer_pick_kernel<T, MANY>)<<<dim3(pick_grid), dim3(kPickThreads), 0, s>>>(  \
                    l.indptr, l.num_cols, IDS, cols, (int)l.fanout, cols_per_wave, l.replace, \
                    key, (uint32_t)l.id_stride, l.cdf ? w.picked : nullptr, table,            \
                    (uint32_t)(slots - 1), w.slot, w.wide));                                  \
  } while (0)
#define GS_PICK_AND_FLAG(MANY)                                                                \
  do {                                                                                        \
    if (l.indices32) GS_PICK(int32_t, MANY, l.indices32);                                     \
    else GS_PICK(int64_t, MANY, l.indices);                                                   \
    GS_LAUNCH("layer_flag", s,                                                                \
              layer_flag_kernel<MANY><<<dim3((unsigned)ceil_div(positions, kLayerTile)),      \
                                        dim3(kBlock), 0, s>>>(cols, (int)l.fanout, table,     \
                                                              w.slot, w.first, w.key, w.words, \
                                                              w.tile_cnt));                   \
  } while (0)
  if (l.num_batches > 1) GS_PICK_AND_FLAG(true);
  else GS_PICK_AND_FLAG(false);
#undef GS_PICK_AND_FLAG
#undef GS_PICK
  return GS_OK;
}

}  // extern "C"

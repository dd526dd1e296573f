// membership.hip -- slicing across the compressed axis: keep the edges whose
// minor id (row id of a CSC, or any id array of a COO) belongs to a picked set
// and relabel that id to its position in the set.
//
//   count: hash the picked ids (smallest position wins for repeated ids); a
//          wave tests a chunk of 256 consecutive edges as four coalesced rows, sends
//          away by a filter in LDS what is not picked, looks the rest up, and leaves
//          the new ids (positions in the picked set) of the chunk's kept edges in
//          edge order, their places in the chunk, and their number; scan of the
//          chunk counts; out_indptr[c] = kept edges before indptr[c].
//   fill : a lane per kept edge, in output order; the new id and the place come
//          from the chunk's staged run, so the fill pass reads neither the ids
//          nor the table again.
//
// A table slot is  low 32 bits of the id << 32 | position in the picked set.
// While every picked id is below 2^32 - 1 those bits are the id, and an edge
// whose id is larger cannot match.  When a picked id is larger (an id of a very
// large graph, an id encoded as id + batch * num_rows) the insert pass raises a
// flag, and every match of the 32-bit halves is then confirmed against the
// picked id itself.
#include <algorithm>
#include <type_traits>
#include <vector>

#include "common.h"
#include "hashtable.h"
#include "listlabels.h"
#include "scan.h"

namespace gs {

constexpr int kMemberWords = kBlock / kWave;  // rows of 64 edges per chunk of kBlock edges
// Chunks one wave takes at a time.  A long run shares the look-up of its columns
// among more edges; on a short edge list it leaves the machine idle while few waves
// walk through their chains of dependent loads: one chunk while even that makes no
// more than 1024 work-groups (four of them fit a compute unit), two beyond that
// (kMemberWavesPerSimd says why no more).  Fixed runs of eight took, on slices of 5 to 38 thousand
// edges, 24-49 us to flag and 33-46 us to fill (5 to 19 work-groups).
constexpr int kMemberLongRun = 2;
constexpr int64_t kMemberShortChunks = 4096;
// The fill pass alone goes to four beyond 64 Mi edges (29 M edges: 59 us with two, 69
// with four; a row slice of 602 M: 3.34 ms with two, 3.10 with four).
constexpr int kMemberHugeRun = 4;
constexpr int64_t kMemberHugeChunks = int64_t(1) << 18;
constexpr int kMemberThreads = 1024;  // 16 waves share one table
// Two of the large work-groups share a compute unit, which takes at most 64 registers
// a lane.  Runs of eight chunks with a look-up for every row took 90 to 128 registers,
// one work-group was resident, and a launch of 590 or 890 work-groups left its second
// round half empty: 136 us on 29 M edges of 512 columns and 110 on 19 M.  Two chunks a
// run, as many work-groups as are resident: 90 and 66 (and four chunks a run 64 and 45
// where two now take 64 and 43).
constexpr int kMemberWavesPerSimd = 8;
constexpr int kMemberLdsSlots = 4096;  // of a table in LDS (32 KB)
// Picked sets of up to so many ids have theirs in LDS: half of its slots.  Count passes that
// tell no first edges, us, at the bound and one id past it, with the launches that make a table
// in L2: 28 M edges 51 and 59, 8 M 49 and 42, 1 M 26 and 21.  On the shorter lists the table in
// L2 is ahead from about 1500 ids on, but first edges, and with them slices that are only
// handed on, need the one in LDS.
constexpr int kMemberLdsIds = kMemberLdsSlots / 2;
constexpr int64_t kMemberSmallEdges = int64_t(1) << 23;  // below: work-groups of kBlock threads
// Work-groups of a launch that stages its table in LDS, at most: what is resident on 256
// compute units is 512 large ones or 768 small ones.
constexpr int64_t kMemberMostGroups = 1024;

// A table too large for LDS is looked up in L2, one request per probe, and the
// flag pass then runs at the rate of those requests.  Most edges are not kept
// (a slice picks a small part of the rows), so a filter that does fit LDS sends
// them away first: a word of 32 bits per id group, three bits per picked id
// (a blocked Bloom filter; of absent ids one in twenty-four passes with 65 536 ids, 4.6 a
// word, and one in five at the bound).  Only ids that pass go on to the table.
constexpr int kFilterWords = 14336;            // 56 KB of LDS, two work-groups a compute unit
constexpr int kFilterBits = 3;
// (16 M edges of 2.33 M rows, us: 131 072 picked ids 144 with the filter, one more 240 without)
constexpr int64_t kFilterMaxIds = 131072;

// Ids that may be picked, by a word of 32 bits per id group in LDS: an id whose bits
// are not all set is not picked.  One multiplication serves the word and the bits.
template <int kWords, int kBits>
struct IdFilter {
  __device__ __forceinline__ static uint32_t hash(uint32_t key) { return key * 0x9E3779B1u; }
  __device__ __forceinline__ static uint32_t word(uint32_t h) {
    return (kWords & (kWords - 1)) == 0 ? h >> (32 - __builtin_ctz(kWords))
                                        : __umulhi(h, (uint32_t)kWords);
  }
  // (shifts go by the low five bits of their count)
  __device__ __forceinline__ static uint32_t bits(uint32_t h) {
    uint32_t b = 0;
#pragma unroll
    for (int i = 0; i < kBits; ++i) b |= 0x80000000u >> ((h >> (13 - 5 * i)) & 31u);
    return b;
  }
  // negative or not, by the word of the hash
  __device__ __forceinline__ static int32_t passes(uint32_t w, uint32_t h) {
    uint32_t all = ~0u;
#pragma unroll
    for (int i = 0; i < kBits; ++i) all &= w << ((h >> (13 - 5 * i)) & 31u);
    return (int32_t)all;
  }
};
using L2Filter = IdFilter<kFilterWords, kFilterBits>;

// The same for a few ids, one bit each, by a product of 24 bits (one of 32 takes the time of four
// other instructions).  The word comes from the product's top bits and the bit from those below,
// and the key's upper half is folded onto its lower first: ids in steps (the nodes of one part
// of a partition, of one type) differ in bits of which neither the key's own low ones nor its low
// 24 need hold any.  Of 233 K ids in steps of 1, 8, 32 and 4096 that are not picked 0.6, 0.8, 0.7
// and 0.7 % pass with 512 picked ones in 2048 words and 2.5, 2.7, 2.7 and 2.6 % with 2048; with
// the key's low five bits for the bit 0.6, 5.8, 22 and 23 % did and 2.4, 22, 62 and 65 %, and 31 M
// edges of 1500 picked ids in steps of 256 took the flag pass 69 us where 41 now.
template <int kWords>
struct FewIdFilter {
  static_assert((kWords & (kWords - 1)) == 0, "the top bits of a product are a word");
  __host__ __device__ __forceinline__ static uint32_t hash(uint32_t key) {
    return ((key ^ (key >> 12)) & 0xFFFFFFu) * 0x9E3779u;
  }
  __host__ __device__ __forceinline__ static uint32_t word(uint32_t h) {
    return h >> (32 - __builtin_ctz(kWords));
  }
  __host__ __device__ __forceinline__ static uint32_t bits(uint32_t h) {
    return 0x80000000u >> ((h >> 16) & 31u);
  }
  __host__ __device__ __forceinline__ static int32_t passes(uint32_t w, uint32_t h) {
    return (int32_t)(w << ((h >> 16) & 31u));
  }
};
// Words for the work-groups of so many threads.
constexpr int few_filter_words(int threads) { return threads == kMemberThreads ? 2048 : 1024; }

// Up to this many chunks the offsets of chunks and columns take one launch
// (member_offsets_kernel), in which a work-group adds up the counts of all chunks before
// its own: two bytes each, 256 KB at this bound (4.2 us on 4 M edges, 6.4 on 17 M and 8.7
// at the bound, where three launches that read every count once take 15.2).
constexpr int64_t kOffsetsMaxChunks = int64_t(1) << 17;

constexpr int kMostLabelBatches = 32;  // whose labels are made beside the offsets
constexpr int kRecordWords = 4;  // of a RunRecord, 64 bits each
struct MemberWs {
  uint64_t* table;     // [member_table_slots(num_picked)], a table in L2
  uint32_t* staged;    // [chunks * kBlock]: per chunk, the new ids of its kept edges, in order
  uint8_t* staged_pos;  // [chunks * kBlock]: and their places in the chunk
  int64_t* chunk_off;  // [chunks + 1]
  uint16_t* chunk_kept;  // [chunks] kept edges of a chunk, for lists of up to kOffsetsMaxChunks
  struct RunRecord* records;  // [chunks / kMemberLongRun] of a long slice that is read in place
  int* wide;           // [1] set when a picked id does not fit the upper half of a slot
  uint32_t* filter;    // [kFilterWords] which ids may be in the table (member_filtered)
  uint32_t* firsts;    // [first_groups * num_picked] per work-group of the flag pass, the first edge it kept by each id
  int64_t first_groups;
  uint32_t* first_parts;  // [kMostLabelBatches] behind `wide`: how many parts of the first edges are told (ListLabels)
  void* scan_ws;
  size_t scan_ws_bytes;
  int64_t chunks;
  size_t total;
};

// Whether every work-group builds the table in LDS for itself, and whether a filter lies in
// front of a table in L2.
static bool member_in_lds(int64_t num_picked) { return num_picked <= kMemberLdsIds; }
static bool member_filtered(int64_t num_picked) {
  return !member_in_lds(num_picked) && num_picked <= kFilterMaxIds;
}

// Slots of the table in L2: four per picked id (fewer probes for the ids that are
// not there, which are most: 1.4 instead of 2.5 on average) while that stays a small
// part of a die's L2, else two.
constexpr int64_t kMemberRoomyIds = 65536;   // 4 slots * 8 B * 65536 = 2 MB
static uint64_t member_table_slots(int64_t num_picked) {
  if (member_in_lds(num_picked)) return 0;
  return (uint64_t)((num_picked <= kMemberRoomyIds ? 4 : 2) * num_picked + 2);
}

// Whether the flag pass leaves a RunRecord of every run.  (Their columns are 32 bits wide.)
static bool member_columns_fit(const SliceView& view) { return view.n <= (int64_t)UINT32_MAX; }
static bool member_told(int64_t nnz, const SliceView& view) {
  return view.sub_indptr != nullptr && nnz >= kMemberSmallEdges && member_columns_fit(view);
}

// firsts: with room for first edges, behind the rest, which lies where it does without.
static MemberWs carve_member(void* ws, int64_t nnz, int64_t num_picked, bool firsts = false) {
  Carver c(ws);
  MemberWs w;
  w.chunks = ceil_div(nnz > 0 ? nnz : 1, kBlock);
  w.table = c.take<uint64_t>((size_t)member_table_slots(num_picked));
  w.staged = c.take<uint32_t>((size_t)w.chunks * kBlock);
  w.staged_pos = c.take<uint8_t>((size_t)w.chunks * kBlock);
  w.chunk_off = c.take<int64_t>((size_t)w.chunks + 1);
  w.chunk_kept =
      c.take<uint16_t>(w.chunks <= kOffsetsMaxChunks ? (size_t)ceil_div(w.chunks, 8) * 8 : 0);
  w.records = (RunRecord*)c.take<uint64_t>(
      nnz >= kMemberSmallEdges ? (size_t)ceil_div(w.chunks, kMemberLongRun) * kRecordWords : 0);
  w.wide = c.take<int>(1 + kMostLabelBatches);
  w.first_parts = w.wide ? (uint32_t*)(w.wide + 1) : nullptr;
  w.filter = c.take<uint32_t>(member_filtered(num_picked) ? (size_t)kFilterWords : 0);
  w.scan_ws_bytes = scan_workspace_bytes(w.chunks + 1);
  w.scan_ws = c.take<char>(w.scan_ws_bytes);
  w.first_groups =
      firsts && member_in_lds(num_picked) ? std::min(w.chunks, kMemberMostGroups) : 0;
  w.firsts = c.take<uint32_t>((size_t)(w.first_groups * num_picked));
  w.total = c.total();
  return w;
}

// The look-ups run once per edge, so they are kept to 32-bit arithmetic: an
// admissible id fits 32 bits, the home slot is one multiply and one
// multiply-high, and a probe compares the upper half of a packed slot.
constexpr uint32_t kNoKey = 0xFFFFFFFFu;  // upper half of the empty slot; no admissible id

__device__ __forceinline__ uint32_t member_home(uint32_t key, uint32_t cap) {
  return __umulhi(key * 0x9E3779B1u, cap);
}

// 32-bit form of an id when every picked id fits 32 bits: kNoKey for one that
// no picked id can equal
__device__ __forceinline__ uint32_t member_key(uint64_t id) {
  return id <= kMaxPackedKey ? (uint32_t)id : kNoKey;
}
// 32-bit tag of any id: its low half, kept clear of kNoKey
__device__ __forceinline__ uint32_t member_tag(uint64_t id) {
  const uint32_t t = (uint32_t)id;
  return t == kNoKey ? kNoKey - 1 : t;
}

// *wide must be 0 before the launch.  Two picked ids with the same tag are the
// same id unless one of them is wide, so matches are always confirmed here (the
// picked set is small next to the edges).
__device__ __forceinline__ void member_insert_one(const int64_t* __restrict__ picked, int64_t i,
                                                  uint64_t* table, uint32_t cap,
                                                  int* __restrict__ wide, uint32_t* filter) {
  const uint64_t id = (uint64_t)picked[i];
  if (id > kMaxPackedKey) *wide = 1;  // every writer stores the same value
  const uint32_t key = member_tag(id);
  if (filter) {
    const uint32_t h = L2Filter::hash(key);
    atomicOr(filter + L2Filter::word(h), L2Filter::bits(h));
  }
  const uint64_t mine = ((uint64_t)key << 32) | (uint64_t)i;
  uint32_t slot = member_home(key, cap);
  for (uint32_t probes = 0; probes < cap; ++probes) {  // the table has free slots: ends early
    uint64_t cur = __hip_atomic_load(table + slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (cur == kEmptySlot) {
      cur = atomicCAS((unsigned long long*)(table + slot), (unsigned long long)kEmptySlot,
                      (unsigned long long)mine);
      if (cur == kEmptySlot) return;
    }
    // a slot only ever holds positions of one id; a repeated id keeps its smallest
    if ((uint32_t)(cur >> 32) == key && (uint64_t)picked[(uint32_t)cur] == id) {
      atomicMin((unsigned long long*)(table + slot), (unsigned long long)mine);
      return;
    }
    if (++slot == cap) slot = 0;
  }
}

__global__ __launch_bounds__(kBlock) void member_insert_kernel(
    const int64_t* __restrict__ picked, int64_t n, uint64_t* table, uint32_t cap,
    int* __restrict__ wide, uint32_t* filter) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  member_insert_one(picked, i, table, cap, wide, filter);
}

// Empties the table and lowers the wide-id flag.
__global__ __launch_bounds__(kBlock) void member_clear_kernel(uint64_t* table, int64_t n,
                                                              int* __restrict__ wide,
                                                              uint32_t* filter) {
  int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i == 0) *wide = 0;
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  if (filter)
    for (int64_t j = i; j < kFilterWords; j += stride) filter[j] = 0u;
  for (; i < n; i += stride) table[i] = kEmptySlot;
}

struct MemberTable {
  const uint64_t* slots;
  uint32_t cap;

  __device__ __forceinline__ uint32_t key_at(uint32_t slot) const {
    return (uint32_t)(slots[slot] >> 32);
  }
  __device__ __forceinline__ uint32_t value_at(uint32_t slot) const {
    return (uint32_t)slots[slot];
  }

  // N look-ups in step: the probes of a round are issued together, so a lane
  // waits for the longest of its N probe runs instead of their sum.  slot[j]
  // is where key[j] sits, cap when it is absent (or kNoKey); value[j] is its position.
  template <int N>
  __device__ __forceinline__ void find_many(const uint32_t (&key)[N], uint32_t (&slot)[N],
                                            uint32_t (&value)[N]) const {
    uint32_t open = 0;  // bit j: key j is still probing
#pragma unroll
    for (int j = 0; j < N; ++j) {
      slot[j] = cap;
      value[j] = 0;
      if (key[j] != kNoKey) {
        slot[j] = member_home(key[j], cap);
        open |= 1u << j;
      }
    }
    for (uint32_t probes = 0; open != 0 && probes < cap; ++probes) {
      uint64_t cur[N];
#pragma unroll
      for (int j = 0; j < N; ++j) cur[j] = (open >> j) & 1u ? slots[slot[j]] : 0ull;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        if (!((open >> j) & 1u)) continue;
        if ((uint32_t)(cur[j] >> 32) == key[j]) {
          open &= ~(1u << j);
          value[j] = (uint32_t)cur[j];
        } else if ((uint32_t)(cur[j] >> 32) == kNoKey) {
          open &= ~(1u << j);
          slot[j] = cap;
        } else if (++slot[j] == cap) {
          slot[j] = 0;
        }
      }
    }
#pragma unroll
    for (int j = 0; j < N; ++j)
      if ((open >> j) & 1u) slot[j] = cap;  // probe budget spent: cannot happen with free slots
  }

  // One look-up whose tag matches are confirmed against the picked ids (the
  // path of picked sets with ids of 2^32 - 1 and above).
  __device__ __forceinline__ uint32_t find_confirmed(uint64_t id,
                                                     const int64_t* __restrict__ picked) const {
    const uint32_t tag = member_tag(id);
    uint32_t slot = member_home(tag, cap);
    for (uint32_t probes = 0; probes < cap; ++probes) {
      const uint32_t cur = key_at(slot);
      if (cur == kNoKey) return cap;
      if (cur == tag && (uint64_t)picked[value_at(slot)] == id) return slot;
      if (++slot == cap) slot = 0;
    }
    return cap;
  }
};

// A small table (the picked set of a layer-wise sampler is a few hundred ids) is
// built in LDS by every work-group for itself, from the ids (a launch that built it in
// memory for all took 5 to 6 us in front of the flag pass), as buckets of four keys: 64 lanes
// probing 64 different slots cost the vector cache a tag look-up each, the LDS
// a few cycles in all.  A look-up reads
// one bucket (16 bytes, one instruction) and compares four keys, and goes on to
// the next bucket only from a full one.  With at most two keys per bucket on
// average nearly every look-up ends at its first bucket, where a linear table
// makes a wave repeat its probe loop until the longest of its probe runs
// has ended.
constexpr int kMemberBuckets = kMemberLdsSlots / 4;
struct BucketTable {
  const uint4* keys;       // [kMemberBuckets] filled from .x on; kNoKey = free
  const uint32_t* values;  // [kMemberLdsSlots] position in the picked set, by slot

  __device__ __forceinline__ static uint32_t home(uint32_t key) {
    return __umulhi(key * 0x9E3779B1u, (uint32_t)kMemberBuckets);
  }

  // Where a bucket holds a key, 4 where it does not.
  __device__ __forceinline__ static uint32_t place_in(const uint4& k, uint32_t key) {
    return k.x == key ? 0u : k.y == key ? 1u : k.z == key ? 2u : k.w == key ? 3u : 4u;
  }
  // Whether a full bucket holds an id whose key may stand for several: its position is then
  // no larger than i.
  __device__ __forceinline__ static bool merge_confirmed(uint32_t b, uint32_t key, uint64_t id,
                                                         uint32_t i,
                                                         const int64_t* __restrict__ picked,
                                                         const uint32_t* lds_keys,
                                                         uint32_t* lds_values) {
    for (uint32_t slot = b * 4; slot < b * 4 + 4; ++slot) {
      const uint32_t held = __hip_atomic_load(lds_keys + slot, __ATOMIC_ACQUIRE,
                                              __HIP_MEMORY_SCOPE_WORKGROUP);
      if (held != key || (uint64_t)picked[lds_values[slot]] != id) continue;
      atomicMin(lds_values + slot, i);
      return true;
    }
    return false;
  }

  // A repeated id takes slots until its bucket is full and then meets itself there: with a
  // slot for every copy the n-th walked n / 4 full buckets, in every work-group (2047 copies of
  // one id, row slices of 300 K and 8 M edges: 1013 and 1440 us, now 45 and 61, where as many
  // ids apart take 21 and 40).  Ids that the filter has not met need not look.
  // fill: a counter per bucket, only used here; seen(key) is called for every id, after a
  // barrier, and tells whether it may have been called for the key before.  Returns whether an
  // id does not fit 32 bits (and a key is then no more than a part of its id), the same for
  // every thread.
  template <int kThreads, typename Seen>
  __device__ __forceinline__ bool stage(const int64_t* __restrict__ picked, uint32_t num_picked,
                                        uint32_t* lds_keys, uint32_t* lds_values, uint32_t* fill,
                                        Seen seen) {
    keys = reinterpret_cast<const uint4*>(lds_keys);
    values = lds_values;
    constexpr int kShare = kMemberLdsIds / kThreads;
    uint64_t id[kShare];
    bool wide = false;
#pragma unroll
    for (int j = 0; j < kShare; ++j) {
      const uint32_t i = j * kThreads + threadIdx.x;
      id[j] = i < num_picked ? (uint64_t)picked[i] : 0;
    }
    for (uint32_t i = threadIdx.x; i < (uint32_t)kMemberLdsSlots; i += kThreads)
      lds_keys[i] = kNoKey;
    for (uint32_t i = threadIdx.x; i < (uint32_t)kMemberBuckets; i += kThreads) fill[i] = 0;
#pragma unroll
    for (int j = 0; j < kShare; ++j) wide |= id[j] > kMaxPackedKey;
    wide = __syncthreads_or(wide) != 0;
    uint32_t slot[kShare];
#pragma unroll
    for (int j = 0; j < kShare; ++j) {
      const uint32_t i = j * kThreads + threadIdx.x;
      if (i >= num_picked) continue;
      const uint32_t key = member_tag(id[j]);
      const bool again = seen(key);
      slot[j] = kMemberLdsSlots;  // (none of its own)
      uint32_t b = home(key);
      for (int tries = 0; tries < kMemberBuckets; ++tries) {  // fewer keys than slots: ends early
        const uint32_t at = atomicAdd(&fill[b], 1u);
        if (at < 4u) {
          slot[j] = b * 4 + at;
          lds_values[slot[j]] = i;
          if (wide) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");  // for whoever sees the key
          lds_keys[slot[j]] = key;
          break;
        }
        if (again && (wide ? merge_confirmed(b, key, id[j], i, picked, lds_keys, lds_values)
                           : place_in(keys[b], key) < 4u))
          break;
        b = (b + 1) & (kMemberBuckets - 1);
      }
    }
    __syncthreads();
    if (wide) return true;
    // a look-up ends at the first of a repeated id's slots, whose position is the smallest
#pragma unroll
    for (int j = 0; j < kShare; ++j) {
      const uint32_t i = j * kThreads + threadIdx.x;
      if ((uint32_t)(j * kThreads) >= num_picked) break;
      const uint32_t first = find(i < num_picked ? member_tag(id[j]) : kNoKey);
      if (i < num_picked && first != slot[j]) atomicMin(&lds_values[first], i);
    }
    __syncthreads();
    return false;
  }

  // Where a key sits, kMemberLdsSlots when it is absent (or kNoKey).  Every lane of the
  // wavefront calls this.  The first bucket is read whole, in one instruction and without a
  // branch: compares that end early were four reads one behind the other.
  __device__ __forceinline__ uint32_t find(uint32_t key) const {
    uint32_t b = home(key);
    uint4 k = keys[b];
    asm volatile("" : "+v"(k.x), "+v"(k.y), "+v"(k.z), "+v"(k.w));
    uint32_t hit = place_in(k, key);
    uint32_t slot = hit < 4u && key != kNoKey ? b * 4 + hit : (uint32_t)kMemberLdsSlots;
    bool on = hit == 4u && k.w != kNoKey && key != kNoKey;  // (a bucket with room would hold the key)
    for (int rounds = 1; rounds < kMemberBuckets && __any(on); ++rounds) {
      if (!on) continue;
      b = (b + 1) & (kMemberBuckets - 1);
      k = keys[b];
      hit = place_in(k, key);
      if (hit < 4u) slot = b * 4 + hit;
      on = hit == 4u && k.w != kNoKey;
    }
    return slot;
  }

  // The smallest position of an id among ids that may not fit 32 bits, kNoKey when it is
  // absent: every match of the keys is confirmed against the picked id.
  __device__ __forceinline__ uint32_t find_confirmed(uint64_t id,
                                                     const int64_t* __restrict__ picked) const {
    const uint32_t tag = member_tag(id);
    uint32_t b = home(tag), best = kNoKey;
    for (int rounds = 0; rounds < kMemberBuckets; ++rounds) {
      const uint32_t* k = reinterpret_cast<const uint32_t*>(keys + b);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (k[e] != tag) continue;
        const uint32_t at = values[b * 4 + e];
        if (at < best && (uint64_t)picked[at] == id) best = at;
      }
      if (k[3] == kNoKey) break;
      b = (b + 1) & (kMemberBuckets - 1);
    }
    return best;
  }
};

// The key of an id in a column whose ids are `offset` more than they say; for 32-bit ids
// 0 <= offset < 2^31, so that a sum below zero, kNoKey here, is found by clamping the id.
__device__ __forceinline__ uint32_t offset_key(int32_t id, int64_t offset) {
  const int32_t least = -1 - (int32_t)offset;
  return (uint32_t)(id > least ? id : least) + (uint32_t)offset;
}
__device__ __forceinline__ uint32_t offset_key(int64_t id, int64_t offset) {
  return member_key((uint64_t)(id + offset));
}

// How many lanes below this one are in the set, and `base`.
__device__ __forceinline__ uint32_t lanes_below(uint64_t set, uint32_t base) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(set >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)set, base));
}
// An index of a slice's pointer in LDS: every entry of it up to kEntries, and some of them
// beyond that.
template <int kThreads>
struct PointerIndex {
  static constexpr int kShare = kMemberWords, kEntries = kThreads * kShare;
  uint32_t entries, step;  // none: 0
  uint32_t own[kShare];    // entries j * kThreads + threadIdx.x
  __device__ __forceinline__ void request(const int64_t* __restrict__ ptr, int64_t n, int64_t nnz) {
    const bool fits = n > 0 && nnz <= (int64_t)UINT32_MAX && n <= (int64_t)UINT32_MAX / 2;
    step = fits ? (uint32_t)((n + kEntries - 1) / kEntries) : 0u;
    entries = fits ? (uint32_t)((n + step - 1) / step) : 0u;
#pragma unroll
    for (int j = 0; j < kShare; ++j) {
      const uint32_t i = j * kThreads + threadIdx.x;
      own[j] = i < entries ? (uint32_t)ptr[(int64_t)i * step] : 0u;
    }
  }
  __device__ __forceinline__ void place(uint32_t* lds) const {
#pragma unroll
    for (int j = 0; j < kShare; ++j) {
      const uint32_t i = j * kThreads + threadIdx.x;
      if (i < entries) lds[i] = own[j];
    }
  }
};
// Where a run of edges lies in the columns of a slice that is read in place.  The flag pass of a
// long slice looks them up and leaves them for the passes over what it kept.
struct __align__(16) RunRecord {
  int64_t shift[2];   // of the first two columns
  uint32_t lo, more;  // the first edge's column; how many further on the last one's is
  uint32_t split;     // edges before the second column
  uint32_t unused;
  // The same record for every lane of the wavefront.
  __device__ __forceinline__ SliceView::Run run(const SliceView& view, int64_t first) const {
    auto of = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
    SegmentSpan span;
    span.lo = of(lo);
    span.hi = span.lo + of(more);
    if (span.hi - span.lo > 1) return view.run(first, span);
    SliceView::Run r{};
    r.first = first;
    r.span = span;
    r.split = span.hi != span.lo ? first + of(split) : INT64_MAX;
    r.shift[0] = wave_uniform_first(shift[0]);
    r.shift[1] = wave_uniform_first(shift[1]);
    if (view.key_offset) {
      r.offset[0] = view.key_offset[span.lo];
      r.offset[1] = view.key_offset[span.hi];
    }
    return r;
  }
};
static_assert(sizeof(RunRecord) == kRecordWords * sizeof(uint64_t), "the workspace holds them");
// Those of a work-group's runs of kRunEdges edges, by their numbers.
template <int kRuns, int kRunEdges>
struct RunColumns {
  int64_t shift[2][kRuns];  // of the first two columns
  uint32_t lo[kRuns], more[kRuns];  // the first edge's column; how many further on the last one's is
  uint32_t split[kRuns];    // edges before the second column
  // A thread looks up one run.
  template <typename Index>
  __device__ __forceinline__ void find(const SliceView& view, int64_t nnz, int64_t run, int number,
                                       const uint32_t* lds, const Index& index,
                                       RunRecord* __restrict__ records) {
    const int64_t first = run * kRunEdges;
    const int64_t last = (first + kRunEdges < nnz ? first + kRunEdges : nnz) - 1;
    // the last columns that begin at or before the two edges
    int64_t c[2] = {0, 0}, end[2] = {view.n, view.n};
    if (lds && index.entries > 0) {
      uint32_t at[2] = {0, 0};
      for (uint32_t step = 1u << (31 - __builtin_clz(index.entries)); step > 0; step >>= 1) {
        uint32_t probe[2];
#pragma unroll
        for (int k = 0; k < 2; ++k)
          probe[k] = at[k] + step < index.entries ? lds[at[k] + step] : UINT32_MAX;
        at[0] = at[0] + step < index.entries && (int64_t)probe[0] <= first ? at[0] + step : at[0];
        at[1] = at[1] + step < index.entries && (int64_t)probe[1] <= last ? at[1] + step : at[1];
      }
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        c[k] = (int64_t)at[k] * index.step;
        if (c[k] + index.step < view.n) end[k] = c[k] + index.step;
      }
    }
    while (end[0] - c[0] > 1 || end[1] - c[1] > 1) {
      int64_t mid[2], begins[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        mid[k] = (c[k] + end[k]) >> 1;  // (c[k] itself where it is found)
        begins[k] = view.sub_indptr[mid[k]];
      }
      if (begins[0] <= first) c[0] = mid[0];
      else end[0] = mid[0];
      if (begins[1] <= last) c[1] = mid[1];
      else end[1] = mid[1];
    }
    int64_t start[2], id[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      start[k] = view.sub_indptr[c[k]];
      id[k] = view.cols[c[k]];
    }
    // (an id outside the matrix is an empty column: neither edge lies in one)
    const RunRecord r{{view.indptr[id[0]] - start[0], view.indptr[id[1]] - start[1]},
                      (uint32_t)c[0], (uint32_t)(c[1] - c[0]), (uint32_t)(start[1] - first), 0u};
    shift[0][number] = r.shift[0];
    shift[1][number] = r.shift[1];
    lo[number] = r.lo;
    more[number] = r.more;
    split[number] = r.split;
    records[run] = r;
  }
  __device__ __forceinline__ SliceView::Run run(const SliceView& view, int64_t first, int number) const {
    return RunRecord{{shift[0][number], shift[1][number]}, lo[number], more[number], split[number], 0u}
        .run(view, first);
  }
};

// What the ids of a run are tested with: the table in LDS and a filter of all its ids
// in front of it, or the table in L2 and the filter that the insert pass left.
// kRunEdges: of the runs whose columns are looked up for a work-group; none: 0.
template <bool kInLds, int kThreads, int kRunEdges>
struct MemberShared {
  static constexpr int kWords = !kInLds ? kFilterWords : few_filter_words(kThreads);
  static constexpr int kRuns = kThreads / (kInLds ? 4 : 8);  // looked up at a time
  using Filter = std::conditional_t<kInLds, FewIdFilter<kInLds ? kWords : 1>, L2Filter>;
  // (the queues lie within the reach of an instruction's offset)
  uint32_t queue_key[kThreads * kMemberWords];   // a chunk's worth per wave
  uint8_t queue_place[kThreads * kMemberWords];
  __align__(16) uint32_t keys[kInLds ? kMemberLdsSlots : 4];
  uint32_t values[kInLds ? kMemberLdsSlots : 4];
  uint32_t first[kInLds ? kMemberLdsIds : 4];  // first edge kept by each picked id
  __align__(16) uint32_t filter[kWords];
  RunColumns<(kRunEdges > 0 ? kRuns : 1), kRunEdges> columns;
  uint32_t next_run;  // of the work-group's, for the next wavefront that is done with its own
};
// Work-groups that a compute unit holds, with 160 KB of LDS and 2048 threads: two of 1024
// threads, of kBlock threads three with the table in LDS and two with the filter.
template <bool kInLds, int kThreads>
constexpr int kMemberResident =
    std::min(160 * 1024 / (int)sizeof(MemberShared<kInLds, kThreads, 1>), 2048 / kThreads);
static_assert(kMemberResident<true, kMemberThreads> == 2 && kMemberResident<false, kMemberThreads> == 2 &&
                  kMemberResident<true, kBlock> == 3,
              "what the figures were measured with");

// Whether a row of 64 edges holds picked ids is told by the filter, a word of LDS and
// eight instructions an edge; the edges that pass are packed into the wave's queue, and
// only they, 64 at a time, go through a look-up and are written out.  Most edges of a
// slice are not kept, and the pass is bound by the instructions it issues, which keep the
// vector units busy for two thirds of it: with a look-up for every row 91 us on 31 M edges of
// which a quarter is kept and 66 on 20 M with one kept in twenty-five, with the queue 67 and 36,
// with the columns of runs told beforehand, runs that the wavefronts take one by one and the
// words of the filter read together 51 and 34 (reading the ids and writing what is kept take 33
// and 17 at the rate of a copy; the table, the filter and the columns 6).  Ids of the next run
// asked for ahead, for registers that then spill, were slower: 58 and 38.  Behind the filter,
// table in L2: 83 -> 52 on 18.5 M edges, and where columns are short, 8.4 M edges of 19 K
// columns, 43 -> 38 (a run of two columns waited for its loads one by one).
// kThreads: work-group size.  A large one shares a staged table among more
// edges; a small one spreads a short edge list over all compute units.
// kRun: chunks per wave and run, whose ids are in flight together.
// IdT: int64_t, or int32_t when the ids are read from a matrix's narrow copy.
// kView: the edges are those of a column slice read in place.
template <bool kInLds, int kThreads, int kRun, typename IdT, bool kView>
__global__ __launch_bounds__(kThreads, kThreads == kMemberThreads ? kMemberWavesPerSimd : 1)
void member_flag_kernel(
    const IdT* __restrict__ ids, int64_t nnz,
    const uint64_t* __restrict__ global_table, uint32_t cap,
    const int64_t* __restrict__ picked, uint32_t num_picked, const int* __restrict__ wide_flag,
    int64_t* __restrict__ chunk_count, uint16_t* __restrict__ chunk_kept,
    uint32_t* __restrict__ staged, uint8_t* __restrict__ staged_pos,
    const uint32_t* __restrict__ filter, uint32_t* __restrict__ firsts,
    uint32_t* __restrict__ first_parts, RunRecord* __restrict__ records, SliceView view) {
  constexpr int kRunEdges = kRun * kBlock;
  // (small ones have about a run a wavefront, which looks it up for itself: 4 us less on 0.3 M edges)
  constexpr bool kTold = kView && kThreads == kMemberThreads;  // the columns of runs, by RunColumns
  using Shared = MemberShared<kInLds, kThreads, kTold ? kRunEdges : 0>;
  using Filter = typename Shared::Filter;
  __shared__ Shared sh;
  const bool filtered = kInLds || filter != nullptr;
  if (kInLds && firsts && blockIdx.x == 0 && threadIdx.x < kMostLabelBatches) first_parts[threadIdx.x] = 0u;
  const MemberTable table{global_table, cap};
  BucketTable buckets;
  bool wide;  // the same for every thread of the launch
  PointerIndex<kThreads> index;
  if (kTold) index.request(view.sub_indptr, view.n, nnz);
  if (kInLds) {
    static_assert(sizeof(sh.queue_key) >= kMemberBuckets * sizeof(uint32_t), "counters lie there");
    for (int i = threadIdx.x; i < Shared::kWords; i += kThreads) sh.filter[i] = 0u;
    if (firsts)
      for (uint32_t i = threadIdx.x; i < num_picked; i += kThreads) sh.first[i] = UINT32_MAX;
    wide = buckets.template stage<kThreads>(
        picked, num_picked, sh.keys, sh.values, sh.queue_key, [&](uint32_t key) {
          const uint32_t h = Filter::hash(key), bit = Filter::bits(h);
          return (~atomicOr(&sh.filter[Filter::word(h)], bit) & bit) == 0u;
        });
  } else {
    wide = *wide_flag != 0;
  }
  if (!kInLds && filtered) {
    constexpr int kVecs = Shared::kWords / 4, kShare = (kVecs + kThreads - 1) / kThreads;
    uint4 words[kShare];  // (all in flight, as above)
#pragma unroll
    for (int j = 0; j < kShare; ++j) {
      const int i = j * kThreads + threadIdx.x;
      words[j] = reinterpret_cast<const uint4*>(filter)[i < kVecs ? i : kVecs - 1];
    }
#pragma unroll
    for (int j = 0; j < kShare; ++j) {
      const int i = j * kThreads + threadIdx.x;
      if (i < kVecs) reinterpret_cast<uint4*>(sh.filter)[i] = words[j];
    }
    __syncthreads();
  }
  const int64_t num_chunks = ceil_div_dev(nnz, kBlock);
  const int lane = lane_id();
  const int wave = threadIdx.x / kWave;
  const uint32_t queue0 = wave_uniform_first(wave * kBlock);  // where this wave's queue starts
  // A work-group takes runs of kRun chunks, the work-groups of the launch striding over them
  // (a launch with fewer work-groups than would have a run a wavefront stages its tables once
  // for many; neighbouring runs are the short columns' in one and long ones' in another: 126 us
  // where strides took 69).  Its wavefronts take them from it one by one: with as many for each
  // the last ended at 55 us where half were done at 40 (31 M edges), and at 37 for 25 (19 M).
  const int64_t num_runs = ceil_div_dev(num_chunks, kRun);

  // What is kept of the chunks at hand, the same in every lane; the first of two counts alone.
  int kept = 0, kept_first = 0;
  // writes the lanes' edges that were found behind the others; `second`: of the chunk behind
  // the first of two, which all lanes of that follow
  auto keep = [&](int64_t chunk, bool found, bool second, uint32_t value, uint32_t place) {
    const uint64_t peers = __ballot(found);
    kept_first += __popcll(peers & ~__ballot(second));
    if (found) {
      const uint32_t at = lanes_below(peers, kept) + (second ? kBlock - kept_first : 0);
      (staged + chunk * kBlock)[at] = value;
      (staged_pos + chunk * kBlock)[at] = (uint8_t)place;
      if (kInLds && firsts) {
        const uint32_t e = (uint32_t)(chunk * kBlock) + place + (second ? kBlock : 0);
        if (sh.first[value] > e) atomicMin(&sh.first[value], e);
      }
    }
    kept += __popcll(peers);
  };
  auto finish_chunk = [&](int64_t chunk, int count) {
    if (chunk_kept) {
      chunk_kept[chunk] = (uint16_t)count;
    } else {
      chunk_count[chunk] = count;
      if (chunk == num_chunks - 1) chunk_count[num_chunks] = 0;
    }
  };
  // The edges of a chunk that the filter lets through are queued and looked up, 64 at a time;
  // those of two chunks together where the queue holds them: of one chunk few pass, or a few
  // more than one look-up takes.
  uint32_t end = queue0, second0 = ~0u;  // of the queue; where the second chunk's begin in it
  auto enqueue = [&](bool may, uint32_t key, int row) {
    const uint64_t peers = __ballot(may);
    if (may) {
      const uint32_t at = lanes_below(peers, end);
      sh.queue_key[at] = key;
      sh.queue_place[at] = (uint8_t)(row * kWave + lane);
    }
    end += __popcll(peers);
  };
  auto look_up = [&](int64_t chunk) {
    wave_lds_fence();
    if (kInLds) {
      for (uint32_t q0 = queue0; q0 < end; q0 += kWave) {
        const uint32_t q = q0 + lane < end ? q0 + lane : end - 1;
        const uint32_t slot = buckets.find(q0 + lane < end ? sh.queue_key[q] : kNoKey);
        keep(chunk, slot < kMemberLdsSlots, q >= second0,
             sh.values[slot & (kMemberLdsSlots - 1)], sh.queue_place[q]);
      }
    } else {
      // a table in L2 answers after a round trip: two edges a lane go through their
      // probe rounds together
      constexpr int kN = 2;
#pragma unroll 1
      for (uint32_t q0 = queue0; q0 < end; q0 += kN * kWave) {
        uint32_t k[kN], slot[kN], place[kN], value[kN];
#pragma unroll
        for (int i = 0; i < kN; ++i) {
          const uint32_t at = q0 + i * kWave + lane, q = at < end ? at : end - 1;
          k[i] = at < end ? sh.queue_key[q] : kNoKey;
          place[i] = sh.queue_place[q];
        }
        table.find_many(k, slot, value);
#pragma unroll
        for (int i = 0; i < kN; ++i)
          keep(chunk, slot[i] < cap, q0 + i * kWave + lane >= second0, value[i], place[i]);
      }
    }
    wave_lds_fence();  // the next queue overwrites this one
    if (lane == 0) {
      finish_chunk(chunk, kept_first);
      if (second0 != ~0u) finish_chunk(chunk + 1, kept - kept_first);
    }
    kept = kept_first = 0;
    end = queue0;
    second0 = ~0u;
  };
  // Negative where the filter lets a key through.  (The words are read together: a queue's writes
  // behind each would be waited for by the next.)
  auto test = [&](const auto& key, auto& may) {
    constexpr int kKeys = sizeof(key) / sizeof(uint32_t);
    const uint32_t(&k)[kKeys] = reinterpret_cast<const uint32_t(&)[kKeys]>(key);
    int32_t(&m)[kKeys] = reinterpret_cast<int32_t(&)[kKeys]>(may);
#pragma unroll
    for (int j = 0; j < kKeys; ++j)
      m[j] = filtered ? (int32_t)sh.filter[Filter::word(Filter::hash(k[j]))] : INT32_MIN;
    if (!filtered) return;
#pragma unroll
    for (int j = 0; j < kKeys; ++j) m[j] = Filter::passes((uint32_t)m[j], Filter::hash(k[j]));
  };
  auto flag_chunk = [&](int64_t chunk, const uint32_t (&key)[kMemberWords]) {
    int32_t may[kMemberWords];
    test(key, may);
#pragma unroll
    for (int j = 0; j < kMemberWords; ++j) enqueue(may[j] < 0, key[j], j);
    look_up(chunk);
  };
  auto flag_two_chunks = [&](int64_t chunk, const uint32_t (&key)[2][kMemberWords]) {
    int32_t may[2][kMemberWords];
    test(key, may);
#pragma unroll
    for (int j = 0; j < kMemberWords; ++j) enqueue(may[0][j] < 0, key[0][j], j);
    uint32_t after = end;
#pragma unroll
    for (int j = 0; j < kMemberWords; ++j) after += __popcll(__ballot(may[1][j] < 0));
    const bool together = after - queue0 <= kBlock;
    if (together) second0 = end;
    else look_up(chunk);
#pragma unroll
    for (int j = 0; j < kMemberWords; ++j) enqueue(may[1][j] < 0, key[1][j], j);
    look_up(together ? chunk : chunk + 1);
  };

  // A run over several columns, or of a call with wide ids.
  auto slow_run = [&](int64_t run, const SliceView::Run& vrun) {
    // id of the lane's edge of a row, or of the last edge for a lane past the end: on a
    // run of several columns the look-up shuffles, so all lanes go through it together
    auto id_of = [&](int64_t row, bool* in) -> uint64_t {
      *in = row + lane < nnz;
      if (row >= nnz) row = nnz - 1;
      const int64_t e = *in ? row + lane : nnz - 1;
      if (!kView) return (uint64_t)(int64_t)ids[e];
      if (vrun.near()) return (uint64_t)((int64_t)ids[vrun.place(e)] + vrun.id_offset(e));
      int64_t c, offset;
      const int64_t p = view.row_position(vrun, row, e, &c, &offset);
      return (uint64_t)((int64_t)ids[p] + offset);
    };
    // (one chunk's look-ups at a time: all of them unrolled would set the kernel's
    // registers, and with them how many work-groups a compute unit holds)
#pragma unroll 1
    for (int64_t chunk = run * kRun; chunk < num_chunks && chunk < (run + 1) * kRun; ++chunk) {
      if (!wide) {
        uint32_t key[kMemberWords];
#pragma unroll
        for (int j = 0; j < kMemberWords; ++j) {
          bool in;
          const uint64_t id = id_of(chunk * kBlock + j * kWave, &in);
          key[j] = in ? member_key(id) : kNoKey;
        }
        flag_chunk(chunk, key);
      } else {
#pragma unroll 1
        for (int j = 0; j < kMemberWords; ++j) {
          bool in;
          const uint64_t id = id_of(chunk * kBlock + j * kWave, &in);
          const uint32_t h = Filter::hash(member_tag(id));
          const bool may = in && (!filtered || Filter::passes(sh.filter[Filter::word(h)], h) < 0);
          uint32_t value = kNoKey;
          if (may && kInLds) {
            value = buckets.find_confirmed(id, picked);
          } else if (may) {
            const uint32_t slot = table.find_confirmed(id, picked);
            if (slot < cap) value = table.value_at(slot);
          }
          keep(chunk, value != kNoKey, false, value, j * kWave + lane);
        }
        if (lane == 0) finish_chunk(chunk, kept);
        kept = kept_first = 0;
      }
    }
  };

  // Of a slice that is read in place the columns of kRuns runs are told at once, a thread a
  // run: six loads one behind the other for each run as it came, which eight wavefronts a SIMD
  // hid in part (31 M edges: 66 us, 57 with the look-ups ahead).
  const int64_t own_runs =
      num_runs > blockIdx.x ? (num_runs - 1 - blockIdx.x) / gridDim.x + 1 : 0;
  int64_t run0 = 0;  // of those looked up
  auto prepare_runs = [&](const uint32_t* lds) {
    if (threadIdx.x == 0) sh.next_run = 0;
    if (kTold && threadIdx.x < Shared::kRuns && run0 + threadIdx.x < own_runs)
      sh.columns.find(view, nnz, blockIdx.x + (run0 + threadIdx.x) * gridDim.x, threadIdx.x, lds, index,
                      records);
    __syncthreads();
  };
  if (kTold) {
    index.place(sh.queue_key);
    __syncthreads();
  }
  prepare_runs(sh.queue_key);
  for (;;) {
    // (the compiler must not join what lane 0 alone does here and at the end of a run: it has
    // made a loop of the other lanes, in which the number is always 0)
    __builtin_amdgcn_wave_barrier();
    uint32_t number = 0;
    if (lane == 0) number = atomicAdd(&sh.next_run, 1u);
    __builtin_amdgcn_wave_barrier();
    number = __builtin_amdgcn_readfirstlane(number);
    if (kTold && number >= (uint32_t)Shared::kRuns) {  // every wavefront comes here, or none
      if (run0 + Shared::kRuns >= own_runs) break;
      __syncthreads();
      run0 += Shared::kRuns;
      prepare_runs(nullptr);
      continue;
    }
    if (run0 + number >= own_runs) break;
    const int64_t run = blockIdx.x + (run0 + number) * gridDim.x;
    const int64_t chunk0 = run * kRun, e_first = run * kRunEdges;
    const bool whole = e_first + kRunEdges <= nnz;
    // With a view the edges are those of a column slice that was never written, and an
    // edge's id is read from the parent's array.
    SliceView::Run vrun{};
    vrun.split = INT64_MAX;  // no view: every edge at distance 0, offset 0
    if constexpr (kTold) vrun = sh.columns.run(view, e_first, (int)number);
    else if (kView) vrun = view.run(e_first, (whole ? e_first + kRunEdges : nnz) - 1);
    if (wide || (kView && !vrun.near())) {
      slow_run(run, vrun);
      continue;
    }
    // The ids of the run are requested together, before anything is
    // stored: a store between a load and its use makes the wait for the load
    // (loads and stores count down one in-order counter) a wait for everything.
    uint32_t keys[kRun][kMemberWords];
    const int64_t shift = wave_uniform_first(vrun.shift[0]);
    const int64_t offset = wave_uniform_first(vrun.offset[0]);
    if (whole && vrun.span.lo == vrun.span.hi &&
        (sizeof(IdT) == 8 || (offset >= 0 && offset <= INT32_MAX))) {
      // all in one column: the lanes' places follow from the wave's
      const IdT* from = ids + (e_first + shift);
      IdT id[kRun][kMemberWords];
#pragma unroll
      for (int c = 0; c < kRun; ++c)
#pragma unroll
        for (int j = 0; j < kMemberWords; ++j) id[c][j] = from[c * kBlock + j * kWave + lane];
#pragma unroll
      for (int c = 0; c < kRun; ++c)
#pragma unroll
        for (int j = 0; j < kMemberWords; ++j) keys[c][j] = offset_key(id[c][j], offset);
    } else {
#pragma unroll
      for (int c = 0; c < kRun; ++c)
#pragma unroll
        for (int j = 0; j < kMemberWords; ++j) {
          // (a lane past the end reads the last edge: a branch would wait for the load in it)
          const int64_t at = (chunk0 + c) * kBlock + j * kWave + lane, e = at < nnz ? at : nnz - 1;
          const uint32_t key = member_key(
              kView ? (uint64_t)((int64_t)ids[vrun.place(e)] + vrun.id_offset(e)) : (uint64_t)(int64_t)ids[e]);
          keys[c][j] = at < nnz ? key : kNoKey;
        }
    }
    static_assert(kRun <= 2, "two chunks meet in the queue");
    if constexpr (kRun == 2) {
      if (chunk0 + 1 < num_chunks) {
        flag_two_chunks(chunk0, keys);
        continue;
      }
    }
    flag_chunk(chunk0, keys[0]);
  }
  if (kInLds && firsts) {
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < num_picked; i += kThreads)
      firsts[(int64_t)blockIdx.x * num_picked + i] = sh.first[i];
  }
}

// Which edge is the first of each picked id is what a relabel of the slice goes by.  A pass over
// the kept edges' rows told it (58 MB and 19 us on 7.2 M of 28.8 M edges, behind a launch of 5
// that cleared its output); here the flag pass keeps the least in LDS, a compare an edge it
// keeps, and the work-groups' lists of them are read beside the offsets: LADIES 691 -> 662 us.
// The first edge kept by each of kWave picked ids, of those that the flag pass's work-groups
// have found: the place of an edge among all, which orders the ids as the kept edges do.
__device__ __forceinline__ void member_first(int64_t part, const uint32_t* __restrict__ firsts,
                                             int64_t groups, int64_t num_picked,
                                             int64_t* __restrict__ out_first) {
  constexpr int kWaves = 1024 / kWave, kAhead = 8;
  __shared__ uint32_t least[kWaves][kWave];
  const int wave = threadIdx.x / kWave, lane = lane_id();
  const int64_t i = part * kWave + lane, at = i < num_picked ? i : num_picked - 1;
  uint32_t m = UINT32_MAX;
  for (int64_t g0 = wave; g0 < groups; g0 += kAhead * kWaves) {
    uint32_t v[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const int64_t g = g0 + j * kWaves;
      v[j] = firsts[(g < groups ? g : g0) * num_picked + at];
    }
#pragma unroll
    for (int j = 0; j < kAhead; ++j) m = v[j] < m ? v[j] : m;
  }
  least[wave][lane] = m;
  __syncthreads();
  if (wave > 0 || i >= num_picked) return;
#pragma unroll
  for (int w = 1; w < kWaves; ++w) m = least[w][lane] < m ? least[w][lane] : m;
  // (seen by other dies as soon as it is stored: a fence for the whole device would have them
  // write their L2 back, 5 us)
  __hip_atomic_store(out_first + i, m == UINT32_MAX ? INT64_MAX : (int64_t)m, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__global__ __launch_bounds__(1024) void member_first_kernel(
    const uint32_t* __restrict__ firsts, int64_t groups, int64_t num_picked,
    int64_t* __restrict__ out_first) {
  member_first(blockIdx.x, firsts, groups, num_picked, out_first);
}

// How many of the kept edges of e's chunk, whose places are in order, lie before e.  Two
// rounds of sixteen places each.
__device__ __forceinline__ int member_below(int64_t e, int kept,
                                            const uint8_t* __restrict__ staged_pos) {
  const int64_t chunk = e / kBlock;
  const int in_chunk = (int)(e - chunk * kBlock);
  if (in_chunk == 0 || kept == 0) return 0;
  const uint8_t* places = staged_pos + chunk * kBlock;
  constexpr int kFan = 16;
  static_assert(kFan * kFan >= kBlock, "two rounds reach every place");
  int below = 0;
#pragma unroll
  for (int i = 1; i < kFan; ++i) {  // whole blocks of kFan places
    const int at = i * kFan - 1;
    below += at < kept && places[at < kept ? at : 0] < in_chunk ? kFan : 0;
  }
  int more = 0;
#pragma unroll
  for (int i = 0; i < kFan; ++i) {
    const int at = below + i;
    more += at < kept && places[at < kept ? at : 0] < in_chunk ? 1 : 0;
  }
  return below + more;
}

// Offsets of the chunks and of the columns of a list of up to kOffsetsMaxChunks chunks in
// one launch.  A work-group takes kOffsetsTile chunks and the columns that begin in them;
// what the chunks before it keep it adds up for itself, while two of its wavefronts look
// for its columns.  Bound by that chain of loads.  Tile sums, their scan and the columns
// in three launches took 15 us behind the flag pass on 8 to 29 M edges, this takes 9 to 10
// (tiles of 2048 chunks 11, and 16 where 19 K columns are short and meet in few tiles).
constexpr int kOffsetsThreads = 1024;
static_assert(kOffsetsThreads == 1024 && kOffsetsThreads == kLabelThreads,
              "member_first() and list_labels_of() run in these work-groups too");
constexpr int kOffsetsTile = 512;
// Labels of the picked rows and of the columns (list_labels_of).  They wait for the first edges
// alone: the work-group that tells the last part of those goes on with them while others are at
// the offsets (31 M edges and 512 picks, 20 M and 400: 21 us in two launches, now 16; 37 K and
// 10 K edges 20 and 18, now 15 and 12; of 8 batches of 384 keys 20 us, of which the labels 11 in a
// launch of their own, now 17).
struct ListLabels {
  const int64_t* seeds;  // null: none are wanted
  const int64_t* list_ids;
  int num_seeds;
  uint32_t* parts_told;  // [kMostLabelBatches], 0 before the launch
  int64_t *frontier, *count_mirror, *list_label, *seed_label;
  // of batches (null: there is one), as gs_batch_list_labels says; `frontier` is that of the bounds
  const int64_t *seeds_ptr, *list_ptr;
  int64_t id_stride;
  int num_batches;
  int64_t* counts;
};

// The labels of the batches whose first edges the work-group of this part is the last to tell.
// Lane b looks at batch b, whose rows lie in a part or in several (without rows: in one).
__device__ __forceinline__ void member_batch_labels(unsigned part, unsigned parts, int64_t num_picked,
                                                    const int64_t* __restrict__ first,
                                                    const ListLabels& labels) {
  static_assert(kMostLabelBatches <= kWave, "a lane a batch");
  __shared__ uint32_t told[kMostLabelBatches];
  const int lane = lane_id(), b = lane < labels.num_batches ? lane : 0;
  const int64_t s0 = labels.seeds_ptr[b], s1 = labels.seeds_ptr[b + 1];
  const int64_t l0 = labels.list_ptr[b], l1 = labels.list_ptr[b + 1];
  const bool fits = s0 >= 0 && s1 >= s0 && s1 <= labels.num_seeds && l0 >= 0 && l1 >= l0 &&
                    l1 <= num_picked && (s1 - s0) + (l1 - l0) <= kLabelMaxKeys;
  unsigned p0 = fits ? (unsigned)(l0 / kWave) : 0u;
  if (p0 >= parts) p0 = parts - 1;
  const unsigned p1 = fits && l1 > l0 ? (unsigned)((l1 - 1) / kWave) : p0;
  const bool mine = lane < labels.num_batches && p0 <= part && part <= p1;
  if (threadIdx.x < kWave) {  // (which has stored this part)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (mine)
      told[b] = __hip_atomic_fetch_add(labels.parts_told + b, 1u, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  const uint64_t fitting = __ballot(fits);
  uint64_t left = __ballot(mine && told[b] == p1 - p0);
  for (; left; left &= left - 1) {
    const int i = __builtin_ctzll(left);
    int total = -1;
    if ((fitting >> i) & 1) {
      const int64_t seed0 = labels.seeds_ptr[i], id0 = labels.list_ptr[i];
      total = list_labels_of<true>(labels.seeds + seed0, (int)(labels.seeds_ptr[i + 1] - seed0),
                                   labels.list_ids + id0, labels.id_stride, first + id0,
                                   (int)(labels.list_ptr[i + 1] - id0),
                                   labels.frontier + seed0 + id0, labels.list_label + id0,
                                   labels.seed_label + seed0);
    }
    if (threadIdx.x == 0) labels.counts[i] = total;
    __syncthreads();
  }
}

enum { kNoLabels, kOneList, kBatchLists };
template <int kLabels>
__global__ __launch_bounds__(kOffsetsThreads) void member_offsets_kernel(
    const int64_t* __restrict__ indptr, int64_t num_major,
    const uint8_t* __restrict__ staged_pos, const uint16_t* __restrict__ chunk_kept,
    int64_t nnz, int64_t* __restrict__ chunk_off, int64_t* __restrict__ out_indptr,
    int64_t* __restrict__ out_total, unsigned tiles, const uint32_t* __restrict__ firsts,
    int64_t first_groups, int64_t num_picked, int64_t* __restrict__ out_first,
    double* __restrict__ col_zeros, ListLabels labels) {
  // (the first work-groups tell the first edges where out_first is asked for: those that go on
  // with the labels are under way when the others begin)
  const unsigned parts = gridDim.x - tiles;
  if (blockIdx.x < parts) {
    member_first(blockIdx.x, firsts, first_groups, num_picked, out_first);
    if constexpr (kLabels == kBatchLists) {
      member_batch_labels(blockIdx.x, parts, num_picked, out_first, labels);
    } else if constexpr (kLabels == kOneList) {
      __shared__ uint32_t told;
      if (threadIdx.x < kWave) {  // (which has stored this part)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (threadIdx.x == 0)
          told = __hip_atomic_fetch_add(labels.parts_told, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __syncthreads();
      if (told + 1 != parts) return;
      const int total = list_labels_of<true>(labels.seeds, labels.num_seeds, labels.list_ids, 0, out_first,
                                       (int)num_picked, labels.frontier, labels.list_label,
                                       labels.seed_label);
      if (threadIdx.x == 0) store_for_host(labels.count_mirror, total);
    }
    return;
  }
  const unsigned tile = blockIdx.x - parts;
  __shared__ uint32_t smem[kOffsetsThreads / kWave + 1];
  __shared__ uint32_t before[kOffsetsTile + 1];  // kept edges of the tile before each chunk
  __shared__ int64_t col_range[2];
  const int64_t num_chunks = ceil_div_dev(nnz, kBlock);
  const int64_t chunk0 = (int64_t)tile * kOffsetsTile;
  const bool last_tile = tile + 1 == tiles;
  const int t = threadIdx.x, wave = t / kWave;
  const bool owns = t < kOffsetsTile && chunk0 + t < num_chunks;
  const uint32_t own = owns ? chunk_kept[chunk0 + t] : 0u;
  constexpr int kSearchers = 2;  // wavefronts that look for the tile's columns meanwhile
  uint32_t mine = 0;
  if (wave < kSearchers) {
    if (indptr) {
      const int64_t e = wave_uniform_first((chunk0 + (wave ? kOffsetsTile : 0)) * kBlock);
      int64_t c;
      if (wave ? last_tile : tile == 0) c = wave ? num_major + 1 : 0;
      else c = indptr[0] >= e ? 0 : wave_segment_of(indptr, num_major + 1, e - 1) + 1;
      if (lane_id() == 0) col_range[wave] = c;
    }
  } else {
    // the chunks before the tile, eight a load
    const uint4* vecs = reinterpret_cast<const uint4*>(chunk_kept);
    const int64_t num_vecs = chunk0 / 8;
    constexpr int kAhead = 8, kAdders = kOffsetsThreads - kSearchers * kWave;
    for (int64_t v0 = t - kSearchers * kWave; v0 < num_vecs; v0 += kAhead * kAdders) {
      uint4 v[kAhead];
#pragma unroll
      for (int j = 0; j < kAhead; ++j) {
        const int64_t at = v0 + j * kAdders;
        v[j] = vecs[at < num_vecs ? at : 0];
      }
#pragma unroll
      for (int j = 0; j < kAhead; ++j) {
        // (a chunk keeps at most 256: sums of four fit the halves)
        const uint32_t s = v[j].x + v[j].y + v[j].z + v[j].w;
        if (v0 + j * kAdders < num_vecs) mine += (s & 0xFFFFu) + (s >> 16);
      }
    }
  }
  uint32_t base, in_tile;
  (void)block_exclusive_sum<uint32_t, kOffsetsThreads>(mine, smem, &base);
  const uint32_t run = block_exclusive_sum<uint32_t, kOffsetsThreads>(own, smem, &in_tile);
  if (t < kOffsetsTile) before[t] = run;
  if (t == 0) before[kOffsetsTile] = in_tile;
  if (owns) chunk_off[chunk0 + t] = (int64_t)base + run;
  const int64_t total = (int64_t)base + in_tile;  // of the last tile: of all
  if (last_tile && t == 0) {
    chunk_off[num_chunks] = total;
    if (out_total) store_for_host(out_total, total);
  }
  if (indptr == nullptr) return;
  __syncthreads();
  for (int64_t c = col_range[0] + t; c < col_range[1]; c += kOffsetsThreads) {
    const int64_t e = indptr[c];
    int64_t r = total;
    if (e < nnz) {
      const int64_t i = e / kBlock - chunk0;
      r = base + before[i] + member_below(e, (int)(before[i + 1] - before[i]), staged_pos);
    }
    out_indptr[c] = r;
    if (col_zeros && c < num_major) col_zeros[c] = 0.0;
  }
}

// The columns alone, behind a scan of the chunks' counts.
__global__ __launch_bounds__(kBlock) void member_indptr_kernel(
    const int64_t* __restrict__ indptr, int64_t num_major,
    const uint8_t* __restrict__ staged_pos, const int64_t* __restrict__ chunk_off,
    double* __restrict__ col_zeros, int64_t nnz, int64_t* __restrict__ out_indptr, int64_t* __restrict__ out_total) {
  const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const int64_t num_chunks = ceil_div_dev(nnz, kBlock);
  if (c == 0 && out_total) store_for_host(out_total, nnz > 0 ? chunk_off[num_chunks] : 0);
  if (indptr == nullptr || c > num_major) return;
  if (col_zeros && c < num_major) col_zeros[c] = 0.0;
  const int64_t e = indptr[c];
  int64_t r = 0;
  if (nnz > 0) {
    const int64_t chunk = e < nnz ? e / kBlock : num_chunks;
    r = chunk_off[chunk];
    if (e < nnz) r += member_below(e, (int)(chunk_off[chunk + 1] - r), staged_pos);
  }
  out_indptr[c] = r;
}

// The kept edges of kRun consecutive chunks, which a wavefront writes: they are one piece of the
// output, and a lane takes one of them whichever chunk it is of.  Of two chunks with one edge in
// four kept two or three rows of 64 are written where a row for every 64 places of either took
// four, each behind a branch of its own in which the one before was waited for (7.1 M of 31 M
// edges with values 86 us so and 73 now, 0.8 M of 20 M without 20 and 18; 95 and 23 with a look-up
// of the columns by every wavefront in front of it).
template <int kRun>
struct KeptEdges {
  int64_t first, out0;  // edge of the slice; place of the first kept one
  int kept;
  int before[kRun];     // kept edges of the chunks before each
  const uint32_t* staged;
  const uint8_t* places;
  __device__ __forceinline__ KeptEdges(int64_t first_chunk, int64_t num_chunks,
                                       const int64_t* __restrict__ chunk_off,
                                       const uint32_t* __restrict__ all_staged,
                                       const uint8_t* __restrict__ all_places) {
    const int lane = lane_id();
    const int64_t lane_chunk = first_chunk + (lane < kRun ? lane : kRun);
    const int64_t off = chunk_off[lane_chunk < num_chunks ? lane_chunk : num_chunks];
    first = first_chunk * kBlock;
    out0 = wave_uniform_first(off);
#pragma unroll
    for (int c = 0; c < kRun; ++c) before[c] = (int)(wave_uniform_first(__shfl((long long)off, c, kWave)) - out0);
    kept = (int)(wave_uniform_first(__shfl((long long)off, kRun, kWave)) - out0);
    staged = all_staged + first;
    places = all_places + first;
  }
  // Picked id's place and edge of the slice for kept edge i, or the last one.
  __device__ __forceinline__ void get(int i, uint32_t* minor, int* edge) const {
    const int k = i < kept ? i : kept - 1;
    int at = k, chunk = 0;
#pragma unroll
    for (int c = 1; c < kRun; ++c)
      if (k >= before[c]) {
        at = k + c * kBlock - before[c];
        chunk = c * kBlock;
      }
    *minor = staged[at];
    *edge = chunk + (int)places[at];
  }
  // write(N as an integral_constant, i0): kept edges i0 to i0 + 64 N - 1, as far as there are.
  template <typename Write>
  __device__ __forceinline__ void in_rows(Write write) const {
    int i0 = 0;
    for (; kept - i0 > 2 * kWave; i0 += 4 * kWave) write(std::integral_constant<int, 4>(), i0);
    if (kept - i0 > kWave) write(std::integral_constant<int, 2>(), i0);
    else if (kept - i0 > 0) write(std::integral_constant<int, 1>(), i0);
  }
};

// A wave writes the kept edges of kRun consecutive chunks: the columns of the wave's first and
// last edge take a search each where the flag pass has not left them (one column covers the
// whole span unless columns are short).  The work goes with the kept edges, not with all of
// them: a lane per edge that looked its flag up took 88 us on 19 M edges of which
// one in twenty-five is kept, and 84 on 29 M with one in four; this took 32 and 59.
// kEdgeMajor: the id on the other axis comes from edge_major (an edge list)
// instead of the compressed pointer.
// kView: the edges are those of a column slice read in place (without it none of
// the view's look-ups is compiled in).
template <bool kEdgeMajor, bool kView, int kRun>
__global__ __launch_bounds__(kBlock) void member_fill_kernel(
    int64_t nnz, const int64_t* __restrict__ chunk_off, const uint32_t* __restrict__ staged,
    const uint8_t* __restrict__ staged_pos, const int64_t* __restrict__ indptr, int64_t num_major,
    const int64_t* __restrict__ edge_major, int64_t* __restrict__ out_major,
    int64_t* __restrict__ out_minor, int64_t* __restrict__ out_select,
    const RunRecord* __restrict__ records, SliceView view) {
  const int64_t num_chunks = ceil_div_dev(nnz, kBlock);
  const int64_t wave =
      wave_uniform_first((int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave);
  const int64_t first_chunk = wave * kRun;
  if (first_chunk >= num_chunks) return;
  const bool told = kRun == kMemberLongRun && records != nullptr;
  const RunRecord record = told ? records[wave] : RunRecord{};
  const KeptEdges<kRun> edges(first_chunk, num_chunks, chunk_off, staged, staged_pos);
  if (edges.kept == 0) return;
  const int64_t e_end = edges.first + kRun * kBlock < nnz ? edges.first + kRun * kBlock : nnz;
  SegmentSpan span{0, 0};
  SliceView::Run vrun{};
  if (kView) {  // indptr is the view's column pointer: one look-up serves both
    vrun = told ? record.run(view, edges.first) : view.run(edges.first, e_end - 1);
  } else if (out_major && !kEdgeMajor) {
    span = segment_span(indptr, num_major, edges.first, e_end - 1);
  }
  edges.in_rows([&](auto rows, int i0) {
    constexpr int kRows = decltype(rows)::value;
    uint32_t minor[kRows];
    int64_t e[kRows], parent_pos[kRows], major[kRows];
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      int at;
      edges.get(i0 + j * kWave + lane_id(), &minor[j], &at);
      e[j] = edges.first + at;
    }
    // with a view: the edge's place in the parent and its column in the slice
    // (on a scattered run the look-up shuffles: all lanes take it, the ones past
    // the last kept edge with that edge)
    if (kView && !vrun.near()) {
#pragma unroll
      for (int j = 0; j < kRows; ++j) {
        int64_t offset;
        parent_pos[j] = view.position(vrun, e[j], &major[j], &offset);
      }
    } else {
#pragma unroll
      for (int j = 0; j < kRows; ++j) {
        parent_pos[j] = kView ? vrun.place(e[j]) : e[j];
        major[j] = kView ? vrun.column(e[j]) : 0;
      }
    }
    if (!kView && out_major)
#pragma unroll
      for (int j = 0; j < kRows; ++j)
        major[j] = kEdgeMajor ? edge_major[e[j]] : span.segment_at(indptr, e[j]);
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      const int i = i0 + j * kWave + lane_id();
      if (i >= edges.kept) continue;
      out_minor[edges.out0 + i] = (int64_t)minor[j];
      out_select[edges.out0 + i] = parent_pos[j];
      if (out_major) out_major[edges.out0 + i] = major[j];
    }
  });
}

// The same for a slice whose edges are only wanted with the labels of their ends, and with
// the values they have in the parent, divided by a value of their row: the ids, places and
// columns that the passes for these would read are not written.  7.3 M kept edges of 28 M: the
// labels alone 41 us (152 MB, 3.7 TB/s), where member_fill took 64 and a pass for the labels
// 34; with values 91, of which the gather of one value in four is 45 (a line in any case),
// where the two and a pass for the values took 155.  With the sums over columns made here as
// well, one atomic for a wave in one column, the whole slice took 347 us; with a pass over
// the values behind it 241.
struct LabelledEdges {
  const int64_t* row_label;  // by place among the picked rows; labels are below 2^32
  const int64_t* col_label;  // by column of the slice
  int64_t* row;
  int64_t* col;
  const float* values;  // of the parent's edges; null: none are wanted
  int64_t num_values;
  const float* row_divisor;  // by place among the picked rows, or null
  float* out;
};

template <bool kValues, int kRun>
__global__ __launch_bounds__(kBlock) void member_label_kernel(
    int64_t nnz, const int64_t* __restrict__ chunk_off, const uint32_t* __restrict__ staged,
    const uint8_t* __restrict__ staged_pos, LabelledEdges labels,
    const RunRecord* __restrict__ records, SliceView view) {
  const int64_t num_chunks = ceil_div_dev(nnz, kBlock);
  const int64_t wave =
      wave_uniform_first((int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave);
  const int64_t first_chunk = wave * kRun;
  if (first_chunk >= num_chunks) return;
  const bool told = kRun == kMemberLongRun && records != nullptr;
  const RunRecord record = told ? records[wave] : RunRecord{};
  const KeptEdges<kRun> edges(first_chunk, num_chunks, chunk_off, staged, staged_pos);
  if (edges.kept == 0) return;
  const int64_t e_end = edges.first + kRun * kBlock < nnz ? edges.first + kRun * kBlock : nnz;
  const SliceView::Run run = told ? record.run(view, edges.first) : view.run(edges.first, e_end - 1);
  edges.in_rows([&](auto rows, int i0) {
    constexpr int kRows = decltype(rows)::value;
    uint32_t minor[kRows];
    int at[kRows];
#pragma unroll
    for (int j = 0; j < kRows; ++j) edges.get(i0 + j * kWave + lane_id(), &minor[j], &at[j]);
    int64_t place[kRows], column[kRows];
    if (run.near()) {
#pragma unroll
      for (int j = 0; j < kRows; ++j) {
        place[j] = run.place(edges.first + at[j]);
        column[j] = run.column(edges.first + at[j]);
      }
    } else {  // (the look-up shuffles: all lanes take it)
#pragma unroll
      for (int j = 0; j < kRows; ++j) {
        int64_t offset;
        place[j] = view.position(run, edges.first + at[j], &column[j], &offset);
      }
    }
    // (all loads before the first store, which they might alias for all the compiler knows)
    float v[kRows], by[kRows];
    uint32_t row[kRows], col[kRows];
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      row[j] = (uint32_t)labels.row_label[minor[j]];
      col[j] = (uint32_t)labels.col_label[column[j]];
      v[j] = 0.f;
    }
    if (kValues && labels.num_values > 0) {
#pragma unroll
      for (int j = 0; j < kRows; ++j)  // (edge data may be shorter than the matrix has edges)
        v[j] = labels.values[(uint64_t)place[j] < (uint64_t)labels.num_values ? place[j] : 0];
#pragma unroll
      for (int j = 0; j < kRows; ++j)
        if ((uint64_t)place[j] >= (uint64_t)labels.num_values) v[j] = 0.f;
    }
    if (kValues && labels.row_divisor) {
#pragma unroll
      for (int j = 0; j < kRows; ++j) by[j] = labels.row_divisor[minor[j]];
#pragma unroll
      for (int j = 0; j < kRows; ++j) v[j] /= by[j];
    }
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      const int i = i0 + j * kWave + lane_id();
      if (i >= edges.kept) continue;
      const int64_t pos = edges.out0 + i;
      // (past L2 where the list is long: the passes over the values behind this one find more
      // there, LADIES 577 -> 569 us; what a short list leaves may be read from it)
      if (kRun > 1) {
        __builtin_nontemporal_store((int64_t)row[j], labels.row + pos);
        __builtin_nontemporal_store((int64_t)col[j], labels.col + pos);
      } else {
        labels.row[pos] = (int64_t)row[j];
        labels.col[pos] = (int64_t)col[j];
      }
      if (kValues) labels.out[pos] = v[j];
    }
  });
}

}  // namespace gs

extern "C" {

size_t gs_minor_slice_workspace_bytes(int64_t nnz, int64_t num_picked) {
  if (nnz < 0 || num_picked < 0) return 0;
  return gs::carve_member(nullptr, nnz, num_picked).total;
}

size_t gs_col_row_slice_first_workspace_bytes(int64_t slice_nnz, int64_t num_rows_picked) {
  if (slice_nnz < 0 || num_rows_picked < 0) return 0;
  return gs::carve_member(nullptr, slice_nnz, num_rows_picked, true).total;
}

static int minor_slice_count_impl(const int64_t* ids, const int32_t* ids32, int64_t nnz,
                                  const int64_t* picked,
                                  int64_t num_picked, const int64_t* indptr,
                                  int64_t num_major, int64_t* out_indptr,
                                  int64_t* out_total, void* workspace,
                                  size_t workspace_bytes, gs_stream_t stream,
                                  gs::SliceView view, int64_t* out_first = nullptr,
                                  double* col_zeros = nullptr,
                                  gs::ListLabels labels = gs::ListLabels{}) {
  using namespace gs;
  GS_REQUIRE(nnz >= 0 && num_picked >= 0 && num_major >= 0,
             "minor_slice_count: negative size");
  GS_REQUIRE(!out_first || (num_picked >= 1 && member_in_lds(num_picked) && nnz >= 1 &&
                            nnz < (int64_t)UINT32_MAX),
             "minor_slice_count: no first edges of %lld ids among %lld edges",
             (long long)num_picked, (long long)nnz);
  GS_REQUIRE((nnz == 0 || ids || ids32) && (num_picked == 0 || picked),
             "minor_slice_count: null pointer");
  GS_REQUIRE((indptr == nullptr) == (out_indptr == nullptr),
             "minor_slice_count: indptr and out_indptr go together");
  GS_REQUIRE(out_indptr || out_total, "minor_slice_count: nothing to write");
  // positions among the picked ids are 32-bit values and the table (two slots
  // per id) is addressed with 32-bit arithmetic
  GS_REQUIRE(num_picked < (int64_t(1) << 30),
             "minor_slice_count: at most 2^30 - 1 picked ids, got %lld", (long long)num_picked);
  MemberWs w = carve_member(workspace, nnz, num_picked, out_first != nullptr);
  if (workspace == nullptr || workspace_bytes < w.total) {
    set_error("minor_slice workspace too small: %zu < %zu", workspace_bytes, w.total);
    return GS_ERR_WORKSPACE;
  }
  hipStream_t s = as_stream(stream);
  const uint32_t cap = (uint32_t)member_table_slots(num_picked);
  const bool in_lds = member_in_lds(num_picked);
  uint32_t* filter = member_filtered(num_picked) ? w.filter : nullptr;
  if (!in_lds) {
    GS_LAUNCH("member_clear", s,
              member_clear_kernel<<<dim3((unsigned)ceil_div((int64_t)cap, kBlock * 4)),
                                    dim3(kBlock), 0, s>>>(w.table, (int64_t)cap, w.wide, filter));
    GS_LAUNCH("member_insert", s,
              member_insert_kernel<<<dim3((unsigned)ceil_div(num_picked, kBlock)),
                                     dim3(kBlock), 0, s>>>(picked, num_picked,
                                                           w.table, cap, w.wide, filter));
  }
  uint16_t* kept = w.chunks <= kOffsetsMaxChunks ? w.chunk_kept : nullptr;
  if (nnz > 0) {
    const bool small = nnz < kMemberSmallEdges || !member_columns_fit(view);
    const int threads = small ? kBlock : kMemberThreads;
    const int run = w.chunks <= kMemberShortChunks ? 1 : kMemberLongRun;
    // a large list, or work-groups that stage a table or a filter: as many of them as are
    // resident, each staging once and striding over its runs (row slices of 1 M and 8 M edges,
    // us, with a small work-group for every 2048 edges and with these: 300 picks 21 and 18, 42
    // and 28; 2047 picks 34 and 26, 79 and 39; 5000 picks 34 and 33, 65 and 60)
    const int per_cu =
        in_lds ? (small ? kMemberResident<true, kBlock> : kMemberResident<true, kMemberThreads>)
               : (small ? kMemberResident<false, kBlock> : kMemberResident<false, kMemberThreads>);
    const int64_t resident = (int64_t)per_cu * num_compute_units();
    int64_t blocks = ceil_div(w.chunks, (threads / kWave) * run);
    if ((in_lds || filter || !small) && blocks > resident) blocks = resident;
    if (in_lds && blocks > kMemberMostGroups) blocks = kMemberMostGroups;
    uint32_t* firsts = out_first ? w.firsts : nullptr;
    const dim3 grid((unsigned)blocks);
#define GS_MEMBER_FLAG_AS(LDS, THREADS, RUN, IDT, IDS, VIEW)                                  \
  GS_LAUNCH("member_flag", s,                                                                 \
            (member_flag_kernel<LDS, THREADS, RUN, IDT, VIEW>)<<<grid, dim3(THREADS), 0, s>>>( \
                IDS, nnz, w.table, cap, picked, (uint32_t)num_picked, w.wide, w.chunk_off, kept,   \
                w.staged, w.staged_pos, filter, firsts, w.first_parts, w.records, view))
#define GS_MEMBER_FLAG_IDS(LDS, THREADS, RUN)                                                 \
  do {                                                                                        \
    const bool in_place = view.sub_indptr != nullptr;                                         \
    if (ids32 && in_place) GS_MEMBER_FLAG_AS(LDS, THREADS, RUN, int32_t, ids32, true);        \
    else if (ids32) GS_MEMBER_FLAG_AS(LDS, THREADS, RUN, int32_t, ids32, false);              \
    else if (in_place) GS_MEMBER_FLAG_AS(LDS, THREADS, RUN, int64_t, ids, true);              \
    else GS_MEMBER_FLAG_AS(LDS, THREADS, RUN, int64_t, ids, false);                           \
  } while (0)
#define GS_MEMBER_FLAG(LDS)                                                                   \
  do {                                                                                        \
    if (!small) GS_MEMBER_FLAG_IDS(LDS, kMemberThreads, kMemberLongRun);                      \
    else if (run == 1) GS_MEMBER_FLAG_IDS(LDS, kBlock, 1);                                    \
    else GS_MEMBER_FLAG_IDS(LDS, kBlock, kMemberLongRun);                                     \
  } while (0)
    if (in_lds) GS_MEMBER_FLAG(true);
    else GS_MEMBER_FLAG(false);
#undef GS_MEMBER_FLAG
#undef GS_MEMBER_FLAG_IDS
#undef GS_MEMBER_FLAG_AS
    const unsigned first_parts = out_first ? (unsigned)ceil_div(num_picked, kWave) : 0u;
    if (kept) {
      const unsigned tiles = (unsigned)ceil_div(w.chunks, kOffsetsTile);
      labels.parts_told = w.first_parts;
#define GS_MEMBER_OFFSETS(LABELS)                                                             \
  GS_LAUNCH("member_offsets", s,                                                              \
            (member_offsets_kernel<LABELS>)<<<dim3(tiles + first_parts),                      \
                                              dim3(kOffsetsThreads), 0, s>>>(                 \
                indptr, num_major, w.staged_pos, kept, nnz, w.chunk_off, out_indptr,          \
                out_total, tiles, firsts, blocks, num_picked, out_first, col_zeros, labels))
      if (labels.list_ptr) GS_MEMBER_OFFSETS(kBatchLists);
      else if (labels.seeds) GS_MEMBER_OFFSETS(kOneList);
      else GS_MEMBER_OFFSETS(kNoLabels);
#undef GS_MEMBER_OFFSETS
      return GS_OK;
    }
    if (out_first)
      GS_LAUNCH("member_first", s,
                member_first_kernel<<<dim3(first_parts), dim3(1024), 0, s>>>(firsts, blocks,
                                                                             num_picked, out_first));
    if (labels.seeds && !labels.list_ptr) {
      const int rc = gs_list_labels(labels.seeds, labels.num_seeds, labels.list_ids, out_first, num_picked,
                                    labels.frontier, nullptr, labels.count_mirror, labels.list_label,
                                    labels.seed_label, stream);
      if (rc != GS_OK) return rc;
    }
    int rc = exclusive_scan_i64(w.chunk_off, w.chunk_off, w.chunks + 1, w.scan_ws,
                                w.scan_ws_bytes, s);
    if (rc != GS_OK) return rc;
  }
  const int64_t n = indptr ? num_major + 1 : 1;
  GS_LAUNCH("member_indptr", s,
            member_indptr_kernel<<<dim3((unsigned)ceil_div(n, kBlock)),
                                   dim3(kBlock), 0, s>>>(indptr, num_major, w.staged_pos,
                                                         w.chunk_off, col_zeros, nnz,
                                                         out_indptr, out_total));
  return GS_OK;
}

static int minor_slice_fill_impl(const int64_t* ids, int64_t nnz, int64_t num_picked,
                                 const int64_t* indptr, int64_t num_major,
                                 const int64_t* edge_major, int64_t* out_major,
                                 int64_t* out_minor, int64_t* out_select,
                                 void* workspace, size_t workspace_bytes,
                                 gs_stream_t stream, gs::SliceView view) {
  using namespace gs;
  GS_REQUIRE(nnz >= 0 && num_picked >= 0 && num_major >= 0,
             "minor_slice_fill: negative size");
  if (nnz == 0) return GS_OK;
  GS_REQUIRE(ids, "minor_slice_fill: null ids");
  GS_REQUIRE(out_major == nullptr || edge_major != nullptr || indptr != nullptr,
             "minor_slice_fill: out_major needs edge_major or indptr");
  MemberWs w = carve_member(workspace, nnz, num_picked);
  if (workspace == nullptr || workspace_bytes < w.total) {
    set_error("minor_slice workspace too small: %zu < %zu", workspace_bytes, w.total);
    return GS_ERR_WORKSPACE;
  }
  hipStream_t s = as_stream(stream);
  const int run = w.chunks <= kMemberShortChunks ? 1
                  : w.chunks <= kMemberHugeChunks ? kMemberLongRun : kMemberHugeRun;
  const dim3 grid((unsigned)ceil_div(w.chunks, (kBlock / kWave) * run));
#define GS_MEMBER_FILL_RUN(MAJOR, VIEW, RUN)                                           \
  GS_LAUNCH("member_fill", s,                                                          \
            (member_fill_kernel<MAJOR, VIEW, RUN>)<<<grid, dim3(kBlock), 0, s>>>(      \
                nnz, w.chunk_off, w.staged, w.staged_pos, indptr, num_major, edge_major, \
                out_major, out_minor, out_select, member_told(nnz, view) ? w.records : nullptr, view))
#define GS_MEMBER_FILL(MAJOR, VIEW)                                                    \
  do {                                                                                 \
    if (run == 1) GS_MEMBER_FILL_RUN(MAJOR, VIEW, 1);                                  \
    else if (run == kMemberLongRun) GS_MEMBER_FILL_RUN(MAJOR, VIEW, kMemberLongRun);   \
    else GS_MEMBER_FILL_RUN(MAJOR, VIEW, kMemberHugeRun);                              \
  } while (0)
  if (view.sub_indptr != nullptr) {
    GS_REQUIRE(!edge_major, "minor_slice_fill: a slice read in place has no edge list");
    GS_MEMBER_FILL(false, true);
  } else if (edge_major) {
    GS_MEMBER_FILL(true, false);
  } else {
    GS_MEMBER_FILL(false, false);
  }
#undef GS_MEMBER_FILL
#undef GS_MEMBER_FILL_RUN
  return GS_OK;
}

int gs_minor_slice_count(const int64_t* ids, int64_t nnz, const int64_t* picked,
                         int64_t num_picked, const int64_t* indptr,
                         int64_t num_major, int64_t* out_indptr,
                         int64_t* out_total, void* workspace,
                         size_t workspace_bytes, gs_stream_t stream) {
  return minor_slice_count_impl(ids, nullptr, nnz, picked, num_picked, indptr, num_major,
                                out_indptr, out_total, workspace, workspace_bytes, stream,
                                gs::no_view());
}

int gs_minor_slice_fill(const int64_t* ids, int64_t nnz, int64_t num_picked,
                        const int64_t* indptr, int64_t num_major,
                        const int64_t* edge_major, int64_t* out_major,
                        int64_t* out_minor, int64_t* out_select,
                        void* workspace, size_t workspace_bytes,
                        gs_stream_t stream) {
  return minor_slice_fill_impl(ids, nnz, num_picked, indptr, num_major, edge_major, out_major,
                               out_minor, out_select, workspace, workspace_bytes, stream,
                               gs::no_view());
}

static int check_slice_view(const int64_t* indptr, const int64_t* indices, const int64_t* cols,
                            int64_t num_cols_picked, const int64_t* sub_indptr,
                            int64_t slice_nnz, const char* who) {
  using namespace gs;
  GS_REQUIRE(num_cols_picked >= 0 && slice_nnz >= 0, "%s: negative size", who);
  GS_REQUIRE(sub_indptr, "%s: null sub_indptr", who);
  GS_REQUIRE(slice_nnz == 0 || (indptr && indices && cols && num_cols_picked > 0),
             "%s: null pointer", who);
  return GS_OK;
}

int gs_col_row_slice_count(const int64_t* indptr, const int64_t* indices,
                           const int32_t* indices32, const int64_t* cols,
                           const int64_t* key_offset, int64_t num_cols_picked,
                           const int64_t* sub_indptr, int64_t slice_nnz,
                           const int64_t* rows, int64_t num_rows_picked,
                           int64_t* out_indptr, int64_t* out_total, void* workspace,
                           size_t workspace_bytes, gs_stream_t stream) {
  return gs_col_row_slice_count_first(indptr, indices, indices32, cols, key_offset,
                                      num_cols_picked, sub_indptr, slice_nnz, rows,
                                      num_rows_picked, out_indptr, out_total, nullptr, nullptr,
                                      workspace, workspace_bytes, stream);
}

int64_t gs_probe_few_id_filter(const int32_t* picked, int64_t num_picked, const int32_t* ids,
                               int64_t num_ids, int small) {
  auto passing = [&](auto filter) {
    using Filter = decltype(filter);
    std::vector<uint32_t> words(gs::few_filter_words(small ? gs::kBlock : gs::kMemberThreads), 0u);
    for (int64_t i = 0; i < num_picked; ++i) {
      const uint32_t h = Filter::hash((uint32_t)picked[i]);
      words[Filter::word(h)] |= Filter::bits(h);
    }
    int64_t n = 0;
    for (int64_t i = 0; i < num_ids; ++i) {
      const uint32_t h = Filter::hash((uint32_t)ids[i]);
      n += Filter::passes(words[Filter::word(h)], h) < 0;
    }
    return n;
  };
  if (num_picked < 0 || num_ids < 0 || (num_picked > 0 && !picked) || (num_ids > 0 && !ids)) return -1;
  return small ? passing(gs::FewIdFilter<gs::few_filter_words(gs::kBlock)>{})
               : passing(gs::FewIdFilter<gs::few_filter_words(gs::kMemberThreads)>{});
}

int gs_col_row_slice_tells_first(int64_t slice_nnz, int64_t num_rows_picked) {
  return num_rows_picked >= 1 && gs::member_in_lds(num_rows_picked) && slice_nnz >= 1 &&
         slice_nnz < (int64_t)UINT32_MAX;
}

int gs_col_row_slice_count_first(const int64_t* indptr, const int64_t* indices,
                                 const int32_t* indices32, const int64_t* cols,
                                 const int64_t* key_offset, int64_t num_cols_picked,
                                 const int64_t* sub_indptr, int64_t slice_nnz,
                                 const int64_t* rows, int64_t num_rows_picked,
                                 int64_t* out_indptr, int64_t* out_total, int64_t* out_first,
                                 double* col_zeros, void* workspace, size_t workspace_bytes,
                                 gs_stream_t stream) {
  int rc = check_slice_view(indptr, indices, cols, num_cols_picked, sub_indptr, slice_nnz,
                            "col_row_slice_count");
  if (rc != GS_OK) return rc;
  const gs::SliceView view{sub_indptr, cols, indptr, key_offset, num_cols_picked};
  return minor_slice_count_impl(indices, indices32, slice_nnz, rows, num_rows_picked, sub_indptr,
                                num_cols_picked, out_indptr, out_total, workspace,
                                workspace_bytes, stream, view, out_first, col_zeros);
}

int gs_col_row_slice_count_labels(const int64_t* indptr, const int64_t* indices,
                                  const int32_t* indices32, const int64_t* cols,
                                  int64_t num_cols_picked, const int64_t* sub_indptr,
                                  int64_t slice_nnz, const int64_t* rows, int64_t num_rows_picked,
                                  int64_t* out_indptr, int64_t* out_total, int64_t* out_first,
                                  double* col_zeros, int64_t* out_frontier,
                                  int64_t* out_count_mirror, int64_t* out_row_label,
                                  int64_t* out_col_label, void* workspace, size_t workspace_bytes,
                                  gs_stream_t stream) {
  int rc = check_slice_view(indptr, indices, cols, num_cols_picked, sub_indptr, slice_nnz,
                            "col_row_slice_count");
  if (rc != GS_OK) return rc;
  GS_REQUIRE(gs_col_row_slice_tells_first(slice_nnz, num_rows_picked) && out_first && rows && cols &&
                 num_rows_picked + num_cols_picked <= GS_LIST_LABELS_MAX_KEYS,
             "col_row_slice_count_labels: no labels of %lld rows and %lld columns",
             (long long)num_rows_picked, (long long)num_cols_picked);
  GS_REQUIRE(out_frontier && out_count_mirror && out_row_label && out_col_label,
             "col_row_slice_count_labels: null pointer");
  const gs::SliceView view{sub_indptr, cols, indptr, nullptr, num_cols_picked};
  const gs::ListLabels labels{cols, rows, (int)num_cols_picked, nullptr, out_frontier,
                              out_count_mirror, out_row_label, out_col_label};
  return minor_slice_count_impl(indices, indices32, slice_nnz, rows, num_rows_picked, sub_indptr,
                                num_cols_picked, out_indptr, out_total, workspace,
                                workspace_bytes, stream, view, out_first, col_zeros, labels);
}

int gs_col_row_slice_count_batch_labels(
    const int64_t* indptr, const int64_t* indices, const int32_t* indices32, const int64_t* cols,
    const int64_t* key_offset, int64_t num_cols_picked, const int64_t* sub_indptr,
    int64_t slice_nnz, const int64_t* rows, int64_t num_rows_picked, int64_t* out_indptr,
    int64_t* out_total, int64_t* out_first, double* col_zeros, const int64_t* cols_ptr,
    const int64_t* list_ids, const int64_t* list_ptr, int64_t id_stride, int64_t num_batches,
    int64_t* out_frontier, int64_t* unique_ptr, int64_t* unique_ptr_mirror, int64_t* out_row_label,
    int64_t* out_col_label, int64_t* scratch, void* workspace, size_t workspace_bytes,
    gs_stream_t stream) {
  using namespace gs;
  int rc = check_slice_view(indptr, indices, cols, num_cols_picked, sub_indptr, slice_nnz,
                            "col_row_slice_count");
  if (rc != GS_OK) return rc;
  GS_REQUIRE(gs_col_row_slice_tells_first(slice_nnz, num_rows_picked) && out_first && rows && cols &&
                 num_batches >= 1,
             "col_row_slice_count_batch_labels: no labels of %lld rows of %lld batches",
             (long long)num_rows_picked, (long long)num_batches);
  GS_REQUIRE(cols_ptr && list_ids && list_ptr && out_frontier && unique_ptr && unique_ptr_mirror &&
                 out_row_label && out_col_label && scratch,
             "col_row_slice_count_batch_labels: null pointer");
  const SliceView view{sub_indptr, cols, indptr, key_offset, num_cols_picked};
  int64_t* const counts = scratch + num_cols_picked + num_rows_picked;
  // (few batches: a work-group may have to label several that share its part)
  const bool beside = num_batches <= kMostLabelBatches && num_batches * kWave <= num_rows_picked &&
                      num_cols_picked <= INT32_MAX &&
                      ceil_div(slice_nnz, kBlock) <= kOffsetsMaxChunks;
  ListLabels labels{};
  if (beside)
    labels = ListLabels{cols, list_ids, (int)num_cols_picked, nullptr, scratch, nullptr,
                        out_row_label, out_col_label, cols_ptr, list_ptr, id_stride,
                        (int)num_batches, counts};
  rc = minor_slice_count_impl(indices, indices32, slice_nnz, rows, num_rows_picked, sub_indptr,
                              num_cols_picked, out_indptr, out_total, workspace, workspace_bytes,
                              stream, view, out_first, col_zeros, labels);
  if (rc != GS_OK) return rc;
  if (!beside)
    return gs_batch_list_labels(cols, cols_ptr, num_cols_picked, list_ids, list_ptr,
                                num_rows_picked, id_stride, num_batches, nullptr, nullptr, nullptr,
                                0, out_first, out_frontier, unique_ptr, unique_ptr_mirror,
                                out_row_label, out_col_label, nullptr, nullptr, scratch, stream);
  return batch_list_frontier(cols_ptr, list_ptr, counts, num_batches, scratch, out_frontier,
                             unique_ptr, unique_ptr_mirror, as_stream(stream));
}

int gs_col_row_slice_fill(const int64_t* indptr, const int64_t* indices, const int64_t* cols,
                          int64_t num_cols_picked, const int64_t* sub_indptr,
                          int64_t slice_nnz, int64_t num_rows_picked, int64_t* out_major,
                          int64_t* out_minor, int64_t* out_select, void* workspace,
                          size_t workspace_bytes, gs_stream_t stream) {
  int rc = check_slice_view(indptr, indices, cols, num_cols_picked, sub_indptr, slice_nnz,
                            "col_row_slice_fill");
  if (rc != GS_OK) return rc;
  const gs::SliceView view{sub_indptr, cols, indptr, nullptr, num_cols_picked};
  return minor_slice_fill_impl(indices, slice_nnz, num_rows_picked, sub_indptr,
                               num_cols_picked, nullptr, out_major, out_minor, out_select,
                               workspace, workspace_bytes, stream, view);
}

int gs_col_row_slice_labels(const int64_t* indptr, const int64_t* cols, int64_t num_cols_picked,
                            const int64_t* sub_indptr, int64_t slice_nnz, int64_t num_rows_picked,
                            const int64_t* row_label, const int64_t* col_label, int64_t* out_row,
                            int64_t* out_col, const float* values, int64_t num_values,
                            const float* row_divisor, float* out_values, void* workspace,
                            size_t workspace_bytes, gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(num_cols_picked >= 0 && slice_nnz >= 0 && num_rows_picked >= 0 && num_values >= 0,
             "col_row_slice_labels: negative size");
  if (slice_nnz == 0) return GS_OK;
  GS_REQUIRE(indptr && cols && sub_indptr && row_label && col_label && out_row && out_col &&
                 num_cols_picked > 0 && num_rows_picked > 0,
             "col_row_slice_labels: null pointer");
  GS_REQUIRE(!values == !out_values && (values || !row_divisor),
             "col_row_slice_labels: values and their output go together");
  MemberWs w = carve_member(workspace, slice_nnz, num_rows_picked);
  if (workspace == nullptr || workspace_bytes < w.total) {
    set_error("minor_slice workspace too small: %zu < %zu", workspace_bytes, w.total);
    return GS_ERR_WORKSPACE;
  }
  hipStream_t s = as_stream(stream);
  const SliceView view{sub_indptr, cols, indptr, nullptr, num_cols_picked};
  const LabelledEdges edges{row_label, col_label, out_row, out_col, values,
                            num_values, row_divisor, out_values};
  const int run = w.chunks <= kMemberShortChunks ? 1 : kMemberLongRun;
  const dim3 grid((unsigned)ceil_div(w.chunks, (kBlock / kWave) * run));
#define GS_MEMBER_LABEL(VALUES, RUN)                                             \
  GS_LAUNCH("member_label", s,                                                   \
            (member_label_kernel<VALUES, RUN>)<<<grid, dim3(kBlock), 0, s>>>(    \
                slice_nnz, w.chunk_off, w.staged, w.staged_pos, edges,           \
                member_told(slice_nnz, view) ? w.records : nullptr, view))
  if (values && run == 1) GS_MEMBER_LABEL(true, 1);
  else if (values) GS_MEMBER_LABEL(true, kMemberLongRun);
  else if (run == 1) GS_MEMBER_LABEL(false, 1);
  else GS_MEMBER_LABEL(false, kMemberLongRun);
#undef GS_MEMBER_LABEL
  return GS_OK;
}

}  // extern "C"

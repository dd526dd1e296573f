// listlabels.h -- frontier and labels of a short list of ids, by one work-group in LDS.
#ifndef GSAMPLER_CSRC_LISTLABELS_H_
#define GSAMPLER_CSRC_LISTLABELS_H_

#include "common.h"

namespace gs {

constexpr int kLabelThreads = 1024;
constexpr int kLabelWaves = kLabelThreads / kWave;
constexpr int kLabelMaxKeys = GS_LIST_LABELS_MAX_KEYS;
constexpr int kLabelSlots = 2 * kLabelMaxKeys;  // open addressing, at most half full
constexpr int kLabelIdBits = 12;                // list positions in the low bits of an order value
constexpr uint32_t kLabelEmpty = 0xFFFFFFFFu;
static_assert(kLabelMaxKeys <= (1 << kLabelIdBits), "a list position must fit the order value");
static_assert(kLabelMaxKeys == 2 * kLabelThreads, "two seeds and two listed ids per thread");

__device__ __forceinline__ uint32_t label_slot(int64_t key, uint32_t slots) {
  return (uint32_t)(((uint64_t)key * 0x9E3779B97F4A7C15ull) >> 40) & (slots - 1);
}

// Returns the number of keys in the frontier.  id_stride > 0: the key of a listed
// id is its remainder (ids encoded as id + batch * stride).
// The order of the keys is that of numbers: a seed's position, or behind all seeds a listed
// id's first edge.  A table keeps the least number of every key; the listed ids that own
// theirs are put in order by runs of 64, a wavefront's by counting, and an id's rank is the
// sum of its places in all runs, which are searched together.  One work-group, bound by the
// latency of its steps: four barriers where a bitonic sort in front of the table took twenty,
// and 512 seeds with 512 ids 13 to 15 us, 12 now; 1024 with 400 13 to 14 and 9 to 11.
// kFresh: first_pos was told by other work-groups of the launch.
template <bool kFresh = false>
__device__ __forceinline__ int list_labels_of(
    const int64_t* __restrict__ seeds, int num_seeds, const int64_t* __restrict__ list_ids,
    int64_t id_stride, const int64_t* __restrict__ first_pos, int num_ids,
    int64_t* __restrict__ out_frontier, int64_t* __restrict__ out_list_label,
    int64_t* __restrict__ out_seed_label) {
  __shared__ int64_t keys[kLabelMaxKeys];    // of the seeds, then of the listed ids
  __shared__ uint64_t least[kLabelSlots];    // by slot, the least number of its key
  __shared__ uint32_t table[kLabelSlots];    // slot -> a position of the key that owns it; later its label
  __shared__ uint64_t runs[kLabelMaxKeys];   // numbers of owners among the listed ids, runs of 64 in order
  __shared__ int32_t owners[2][kLabelWaves];  // among the seeds, by 64 of them
  __shared__ int32_t listed_owners[2 * kLabelWaves];
  const int t = threadIdx.x, lane = lane_id(), wave = t / kWave;
  const int u = t ^ (kLabelThreads - kWave);  // the seeds' wavefronts and the ids' meet in the middle
  const int n = num_seeds + num_ids;
  const uint32_t slots = n <= kLabelSlots / 4 ? kLabelSlots / 2 : kLabelSlots;

  int64_t key[4];  // of seeds t and t + 1024, of listed ids u and u + 1024
  uint64_t when[4];
  bool used[4];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int s = j * kLabelThreads + t, l = j * kLabelThreads + u;
    used[j] = s < num_seeds;
    key[j] = used[j] ? seeds[s] : 0;
    when[j] = (uint64_t)s;
    const int64_t* const from = first_pos + (l < num_ids ? l : 0);
    const int64_t first =
        l >= num_ids ? INT64_MAX
        : kFresh     ? __hip_atomic_load(from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                     : *from;
    key[2 + j] = l < num_ids ? list_ids[l] : 0;
    used[2 + j] = first != INT64_MAX;  // by any edge
    when[2 + j] = (((uint64_t)first + 1) << kLabelIdBits) | (uint64_t)l;
  }
  for (uint32_t i = t; i < slots; i += kLabelThreads) {
    table[i] = kLabelEmpty;
    least[i] = ~0ull;
  }
  if (id_stride > 0) {
#pragma unroll
    for (int j = 2; j < 4; ++j)
      key[j] = ((uint64_t)(key[j] | id_stride) >> 32) == 0
                   ? (int64_t)((uint32_t)key[j] % (uint32_t)id_stride)
                   : key[j] % id_stride;
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int s = j * kLabelThreads + t, l = j * kLabelThreads + u;
    if (s < num_seeds) keys[s] = key[j];
    if (l < num_ids) keys[num_seeds + l] = key[2 + j];
  }
  __syncthreads();

  // 1. a slot for every key that is used, and its least number
  uint32_t slot[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    slot[j] = label_slot(key[j], slots);
    if (!used[j]) continue;
    const uint32_t own = (uint32_t)(j < 2 ? j * kLabelThreads + t
                                          : num_seeds + (j - 2) * kLabelThreads + u);
    while (true) {
      uint32_t cur = table[slot[j]];
      if (cur == kLabelEmpty) {
        cur = atomicCAS(&table[slot[j]], kLabelEmpty, own);
        if (cur == kLabelEmpty) break;  // the slot is this key's now
      }
      if (keys[cur] == key[j]) break;
      slot[j] = (slot[j] + 1) & (slots - 1);
    }
    atomicMin((unsigned long long*)&least[slot[j]], (unsigned long long)when[j]);
  }
  __syncthreads();

  // 2. first occurrences: how many of the seeds lie before one, and the listed ids' in runs
  bool owns[4];
  uint64_t peers[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    owns[j] = used[j] && least[slot[j]] == when[j];
    peers[j] = __ballot(owns[j]);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if (lane == 0) {
      owners[j][wave] = __popcll(peers[j]);
      listed_owners[j * kLabelWaves + u / kWave] = __popcll(peers[2 + j]);
    }
    int place = 0;
    for (uint64_t left = peers[2 + j]; left; left &= left - 1) {
      const int l = __builtin_ctzll(left);
      const uint64_t other =
          ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(when[2 + j] >> 32), l) << 32) |
          (uint32_t)__builtin_amdgcn_readlane((int)when[2 + j], l);
      place += other < when[2 + j];
    }
    if (owns[2 + j]) runs[j * kLabelThreads + (u & ~(kWave - 1)) + place] = when[2 + j];
  }
  __syncthreads();

  // 3. ranks
  int seed_owners = 0, total = 0, before[2] = {0, 0};
#pragma unroll
  for (int w = 0; w < 2 * kLabelWaves; ++w) {
    const int c = owners[w / kLabelWaves][w % kLabelWaves];
    if (w < wave) before[0] += c;
    if (w < kLabelWaves + wave) before[1] += c;
    seed_owners += c;
    total += c + listed_owners[w];
  }
  const int num_runs = (num_ids + kWave - 1) / kWave;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (!owns[j]) continue;
    int rank;
    if (j < 2) {
      rank = before[j] + __popcll(peers[j] & ((1ull << lane) - 1ull));
    } else {
      rank = seed_owners;
      constexpr int kTogether = 8;
      for (int r0 = 0; r0 < num_runs; r0 += kTogether) {
        int lo[kTogether], many[kTogether];  // numbers of run r0 + i known to be smaller
#pragma unroll
        for (int i = 0; i < kTogether; ++i) {
          many[i] = r0 + i < num_runs ? listed_owners[r0 + i] : 0;
          lo[i] = 0;
        }
#pragma unroll
        for (int step = kWave; step >= 1; step >>= 1) {
          uint64_t probe[kTogether];
#pragma unroll
          for (int i = 0; i < kTogether; ++i) {
            const int at = lo[i] + step - 1;
            probe[i] = runs[(r0 + i < num_runs ? r0 + i : r0) * kWave + (at < kWave ? at : kWave - 1)];
          }
#pragma unroll
          for (int i = 0; i < kTogether; ++i)
            if (lo[i] + step <= many[i] && probe[i] < when[j]) lo[i] += step;
        }
#pragma unroll
        for (int i = 0; i < kTogether; ++i) rank += lo[i];
      }
    }
    out_frontier[rank] = key[j];
    table[slot[j]] = (uint32_t)rank;
  }
  __syncthreads();

  // 4. labels
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int s = j * kLabelThreads + t, l = j * kLabelThreads + u;
    if (s < num_seeds) out_seed_label[s] = table[slot[j]];
    if (l < num_ids) out_list_label[l] = used[2 + j] ? table[slot[2 + j]] : 0;  // (0: no edge uses it)
  }
  return total;
}

// The frontiers of batches, each at the place of its bound, moved together; the batch pointer, its
// last entry -1 where a batch's count is, for the host too.
int batch_list_frontier(const int64_t* seeds_ptr, const int64_t* list_ptr, const int64_t* counts,
                        int64_t num_batches, const int64_t* bound_frontier, int64_t* out_frontier,
                        int64_t* unique_ptr, int64_t* mirror, hipStream_t s);

}  // namespace gs

#endif  // GSAMPLER_CSRC_LISTLABELS_H_

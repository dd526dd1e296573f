// compact.hip -- column slices of a super-batch whose rows are numbered anew:
// batch b's rows that some edge of its columns uses get consecutive numbers in
// the order of their ids, batch after batch (encoded slicing,
// src/cuda/batch/slicing.cu:25-27 of the reference, followed there by a sorted
// unique with inverse).
//
// An edge's key is  row id + batch * num_rows,  a value of a dense range, so
// nothing is sorted or hashed:
//   clear   one flag byte per key of the range
//   mark    the edges of the slice, read in place from the parent: the flag of
//           every key that occurs is set.  A flag is looked at before it is
//           written (most keys occur many times: 23 M edges onto 0.5 M keys), and
//           all writers store the same byte, so there are no atomics
//   words   the flags of 64 keys become one rank word (their bits + set flags of
//           the group before it), 4096 keys are a group with a count
//   offsets group counts -> group offsets; where every batch's rows begin
//   rows    set flags write their row id to the list of rows
//   fill    the slice itself: the new number of an edge's row is the rank of its
//           key, one gather in a table of range / 4 bytes that a die's L2 holds
// Measured on 8 batches, 233 K rows: the sorted unique took 1100 us for 23 M edges (ten
// passes of a 64-bit radix sort and the passes around it); here the numbering takes 121
// us for 18.5 M, 102 of them in the mark pass, and the fill, which writes the slice, 142.
#include "common.h"
#include "sums.h"

namespace gs {

constexpr int kCompactGroup = 4096;  // keys per group
constexpr int kCompactWords = kCompactGroup / kWave;
struct alignas(16) CompactWord {
  uint64_t bits;
  uint32_t before;
  uint32_t unused;
};

struct CompactWs {
  uint8_t* flags;      // [groups * kCompactGroup]
  CompactWord* words;  // [groups * kCompactWords]
  int64_t* group_cnt;  // [groups]
  int64_t* group_off;  // [groups + 1]
  int64_t groups;
  size_t total;
};

static CompactWs carve_compact(void* ws, int64_t range) {
  Carver c(ws);
  CompactWs w;
  w.groups = ceil_div(range > 0 ? range : 1, kCompactGroup);
  w.flags = c.take<uint8_t>((size_t)w.groups * kCompactGroup);
  w.words = c.take<CompactWord>((size_t)w.groups * kCompactWords);
  w.group_cnt = c.take<int64_t>((size_t)w.groups);
  w.group_off = c.take<int64_t>((size_t)w.groups + 1);
  w.total = c.total();
  return w;
}

// A wavefront of the passes over a slice takes `rounds` rounds of kItems rows of
// 64 edges.  Four rounds of eight share the look-up of the columns among 2048
// edges; a short slice is spread thinner, or a handful of work-groups walks
// through its chains of dependent loads (18 thousand edges in 10 work-groups:
// mark 60 us, fill 46 us).  Two rows a wavefront up to 2^19 edges (1024
// work-groups, as many as are resident), one round of eight up to 2^22.
struct CompactSplit {
  int items, rounds;
  int64_t run() const { return (int64_t)items * rounds * kWave; }
};
static CompactSplit compact_split(int64_t nnz) {
  if (nnz <= int64_t(1) << 19) return {2, 1};
  if (nnz <= int64_t(1) << 22) return {8, 1};
  return {8, 4};
}

__global__ __launch_bounds__(kBlock) void compact_clear_kernel(uint4* flags, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  for (; i < n; i += stride) flags[i] = make_uint4(0u, 0u, 0u, 0u);
}

// key_offset of a column: stride times the batch it belongs to.
__global__ __launch_bounds__(kBlock) void compact_offsets_of_columns_kernel(
    const int64_t* __restrict__ batch_ptr, int64_t num_batches, int64_t stride, int64_t n,
    int64_t* __restrict__ out) {
  const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (c < n) out[c] = segment_of(batch_ptr, num_batches, c) * stride;
}

// The keys of kItems rows of 64 edges from e0 on (edges past the end
// repeat the last one: the look-ups below shuffle, so all lanes stay together).
template <typename IdT, int kItems>
__device__ __forceinline__ void slice_keys(const SliceView& view, const SliceView::Run& r,
                                           const IdT* __restrict__ ids, int64_t nnz, int64_t e0,
                                           int64_t (&key)[kItems],
                                           int64_t (&place)[kItems],
                                           int64_t (&column)[kItems]) {
  const int lane = lane_id();
  if (r.near()) {
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      int64_t e = e0 + j * kWave + lane;
      if (e >= nnz) e = nnz - 1;
      place[j] = r.place(e);
      column[j] = r.column(e);
      key[j] = (int64_t)ids[place[j]] + r.id_offset(e);
    }
    return;
  }
  int64_t offset[kItems];
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const int64_t row = e0 + j * kWave < nnz ? e0 + j * kWave : nnz - 1;
    const int64_t e = row + lane < nnz ? row + lane : nnz - 1;
    place[j] = view.row_position(r, row, e, &column[j], &offset[j]);
  }
#pragma unroll
  for (int j = 0; j < kItems; ++j) key[j] = (int64_t)ids[place[j]] + offset[j];
}

template <typename IdT, int kItems>
__global__ __launch_bounds__(kBlock) void compact_mark_kernel(const IdT* __restrict__ ids,
                                                              int64_t nnz, SliceView view,
                                                              int rounds, uint8_t* flags) {
  const int64_t run_edges = (int64_t)kItems * rounds * kWave;
  const int64_t run = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
  const int64_t first = run * run_edges;
  if (first >= nnz) return;  // whole wavefronts leave together
  const int64_t stop = first + run_edges < nnz ? first + run_edges : nnz;
  const SliceView::Run r = view.run(first, stop - 1);
  for (int64_t e0 = first; e0 < stop; e0 += kItems * kWave) {
    int64_t key[kItems], place[kItems], column[kItems];
    slice_keys(view, r, ids, nnz, e0, key, place, column);
    uint8_t have[kItems];
#pragma unroll
    for (int j = 0; j < kItems; ++j) have[j] = flags[key[j]];
#pragma unroll
    for (int j = 0; j < kItems; ++j)
      if (!have[j]) flags[key[j]] = 1;
  }
}

// ------------------------------------------------ sums of a slice that is not written
// A layer-wise sampler asks an encoded slice for the sums of its squared edge values on
// its rows, picks rows by them and keeps those rows' edges.  Nothing of that needs the
// slice, nor the new numbers of its edges' rows: the sums are made by key (row id +
// batch * num_rows), from ids and values read in place, onto entries that begin at -0.
// Squares are not negative, so an entry is -0 afterwards exactly if no edge has its key:
// the sums are the flags of `mark`, and numbering the rows is a pass over the keys.
// 8 batches, 233 K rows, 18.5 M edges, us: mark 103, fill 137, values 62 and sums onto
// 418 K rows 142, as against sums onto 1.86 M keys 146 and 18 for clearing and numbering
// them; the flag pass of the row slice that follows takes 83 in place of 78.  A step of
// two layers with picks of 256: 1349 -> 1109.
struct EncodedSumsWs {
  CompactWs rows;
  float* sums;  // [groups * kCompactGroup]
  void* sum_ws;
  size_t sum_ws_bytes, total;
};

static EncodedSumsWs carve_encoded_sums(void* ws, int64_t nnz, int64_t range) {
  Carver c(ws);
  EncodedSumsWs w;
  w.rows.groups = ceil_div(range > 0 ? range : 1, kCompactGroup);
  w.rows.flags = nullptr;
  w.rows.words = c.take<CompactWord>((size_t)w.rows.groups * kCompactWords);
  w.rows.group_cnt = c.take<int64_t>((size_t)w.rows.groups);
  w.rows.group_off = c.take<int64_t>((size_t)w.rows.groups + 1);
  w.sums = c.take<float>((size_t)w.rows.groups * kCompactGroup);
  w.sum_ws_bytes = sliced_square_sum_bytes(nnz, w.rows.groups * kCompactGroup);
  w.sum_ws = c.take<uint8_t>(w.sum_ws_bytes);
  w.total = c.total();
  return w;
}

constexpr uint32_t kMinusZero = 0x80000000u;

__device__ __forceinline__ bool compact_flag(uint8_t flag) { return flag != 0; }
__device__ __forceinline__ bool compact_flag(float sum) { return __float_as_uint(sum) != kMinusZero; }

// One work-group per group; a wavefront takes consecutive words, lane l the
// flags l, l + 64, ...: the ballots are the words.
template <typename FlagT>
__global__ __launch_bounds__(kBlock) void compact_words_kernel(const FlagT* __restrict__ flags,
                                                               CompactWord* __restrict__ words,
                                                               int64_t* __restrict__ group_cnt) {
  constexpr int kPer = kCompactWords / (kBlock / kWave);
  __shared__ uint32_t wave_total[kBlock / kWave];
  const int64_t group = blockIdx.x;
  const int wave = threadIdx.x / kWave, lane = lane_id();
  const int64_t word0 = group * kCompactWords + wave * kPer;
  FlagT f[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) f[j] = flags[(word0 + j) * kWave + lane];
  uint64_t my_bits = 0;
  uint32_t my_before = 0, total = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const uint64_t bits = __ballot(compact_flag(f[j]));
    if (lane == j) {
      my_bits = bits;
      my_before = total;
    }
    total += (uint32_t)__popcll(bits);
  }
  if (lane == 0) wave_total[wave] = total;
  __syncthreads();
  uint32_t base = 0, all = 0;
#pragma unroll
  for (int w = 0; w < kBlock / kWave; ++w) {
    if (w < wave) base += wave_total[w];
    all += wave_total[w];
  }
  if (lane < kPer) words[word0 + lane] = CompactWord{my_bits, base + my_before, 0u};
  if (threadIdx.x == 0) group_cnt[group] = (int64_t)all;
}

__device__ __forceinline__ int64_t compact_rank(int64_t key, const CompactWord* __restrict__ words,
                                                const int64_t* __restrict__ group_off) {
  const CompactWord w = words[key / kWave];
  return group_off[key / kCompactGroup] + w.before +
         __popcll(w.bits & ((1ull << (int)(key % kWave)) - 1ull));
}

// One work-group: group counts -> group offsets, then the first row of every
// batch (batch b's keys begin at b * stride), also for the host.
constexpr int kCompactScanThreads = 1024;
__global__ __launch_bounds__(kCompactScanThreads) void compact_offsets_kernel(
    const int64_t* __restrict__ group_cnt, int64_t groups, int64_t* group_off,
    const CompactWord* __restrict__ words, int64_t num_batches, int64_t stride,
    int64_t* __restrict__ row_ptr, int64_t* row_ptr_mirror) {
  __shared__ int64_t smem[kCompactScanThreads / kWave + 1];
  constexpr int kPer = 8;
  int64_t carry = 0;
  for (int64_t base = 0; base < groups; base += kCompactScanThreads * kPer) {
    const int64_t i0 = base + (int64_t)threadIdx.x * kPer;
    int64_t v[kPer], sum = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      v[j] = i0 + j < groups ? group_cnt[i0 + j] : 0;
      sum += v[j];
    }
    int64_t total;
    int64_t run = carry + block_exclusive_sum<int64_t, kCompactScanThreads>(sum, smem, &total);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      if (i0 + j < groups) group_off[i0 + j] = run;
      run += v[j];
    }
    carry += total;
  }
  if (threadIdx.x == 0) group_off[groups] = carry;
  __syncthreads();
  for (int64_t b = threadIdx.x; b <= num_batches; b += kCompactScanThreads) {
    int64_t r = carry;
    if (b < num_batches) {
      const int64_t key = b * stride;
      const CompactWord w = words[key / kWave];
      // written above by other threads of this work-group
      r = __hip_atomic_load(group_off + key / kCompactGroup, __ATOMIC_RELAXED,
                            __HIP_MEMORY_SCOPE_AGENT) +
          w.before + __popcll(w.bits & ((1ull << (int)(key % kWave)) - 1ull));
    }
    row_ptr[b] = r;
    if (row_ptr_mirror) store_for_host(row_ptr_mirror + b, r);
  }
}

// Row ids of the keys that occur, in order, and their sums.  A wavefront takes kPer words.
__global__ __launch_bounds__(kBlock) void compact_rows_kernel(
    const CompactWord* __restrict__ words, const int64_t* __restrict__ group_off, int64_t stride,
    const float* __restrict__ sums, int64_t* __restrict__ out_rows, float* __restrict__ out_sums) {
  constexpr int kPer = kCompactWords / (kBlock / kWave);
  const int64_t group = blockIdx.x;
  const int wave = threadIdx.x / kWave, lane = lane_id();
  const int64_t word0 = group * kCompactWords + wave * kPer;
  CompactWord mine{0ull, 0u, 0u};
  if (lane < kPer) mine = words[word0 + lane];
  const int64_t first = group_off[group];
  // a group lies inside one batch or across few: the row of its first key by one division
  const int64_t key0 = word0 * kWave;
  const int64_t row0 = key0 % stride;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const uint64_t bits = __shfl((unsigned long long)mine.bits, j, kWave);
    const uint32_t before = __shfl(mine.before, j, kWave);
    if ((bits >> lane) & 1ull) {
      int64_t row = row0 + j * kWave + lane;
      while (row >= stride) row -= stride;
      const int64_t at = first + before + __popcll(bits & ((1ull << lane) - 1ull));
      out_rows[at] = row;
      if (sums) out_sums[at] = sums[(word0 + j) * kWave + lane];
    }
  }
}

template <typename IdT, int kItems>
__global__ __launch_bounds__(kBlock) void compact_fill_kernel(
    const IdT* __restrict__ ids, int64_t nnz, SliceView view, int rounds, const CompactWord* __restrict__ words,
    const int64_t* __restrict__ group_off, int64_t* __restrict__ out_col,
    int64_t* __restrict__ out_row, int64_t* __restrict__ out_select) {
  const int64_t run_edges = (int64_t)kItems * rounds * kWave;
  const int64_t run = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
  const int64_t first = run * run_edges;
  if (first >= nnz) return;
  const int64_t stop = first + run_edges < nnz ? first + run_edges : nnz;
  const SliceView::Run r = view.run(first, stop - 1);
  const int lane = lane_id();
  for (int64_t e0 = first; e0 < stop; e0 += kItems * kWave) {
    int64_t key[kItems], place[kItems], column[kItems], rank[kItems];
    slice_keys(view, r, ids, nnz, e0, key, place, column);
#pragma unroll
    for (int j = 0; j < kItems; ++j) rank[j] = compact_rank(key[j], words, group_off);
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const int64_t e = e0 + j * kWave + lane;
      if (e >= nnz) continue;
      out_row[e] = rank[j];
      out_select[e] = place[j];
      if (out_col) out_col[e] = column[j];
    }
  }
}

static int check_compact(int64_t num_cols_picked, int64_t nnz, int64_t num_batches, int64_t stride,
                         const char* who) {
  GS_REQUIRE(num_cols_picked >= 0 && nnz >= 0, "%s: negative size", who);
  GS_REQUIRE(num_batches >= 1 && stride >= 0, "%s: %lld batches of %lld rows", who,
             (long long)num_batches, (long long)stride);
  GS_REQUIRE(stride == 0 || num_batches <= (int64_t(1) << 40) / stride,
             "%s: %lld batches of %lld rows are too many keys", who, (long long)num_batches,
             (long long)stride);
  return GS_OK;
}

}  // namespace gs

extern "C" {

size_t gs_slice_compact_workspace_bytes(int64_t num_batches, int64_t stride) {
  if (num_batches < 1 || stride < 0 || (stride > 0 && num_batches > (int64_t(1) << 40) / stride))
    return 0;
  return gs::carve_compact(nullptr, num_batches * stride).total;
}

int gs_slice_compact_count(const int64_t* indptr, const int64_t* indices, const int32_t* indices32,
                           const int64_t* cols, int64_t num_cols_picked,
                           const int64_t* sub_indptr, int64_t nnz, const int64_t* batch_ptr,
                           int64_t num_batches, int64_t stride, int64_t* out_key_offset,
                           int64_t* row_ptr, int64_t* row_ptr_mirror, void* workspace,
                           size_t workspace_bytes, gs_stream_t stream) {
  using namespace gs;
  int rc = check_compact(num_cols_picked, nnz, num_batches, stride, "slice_compact_count");
  if (rc != GS_OK) return rc;
  GS_REQUIRE(row_ptr && batch_ptr && (num_cols_picked == 0 || out_key_offset),
             "slice_compact_count: null pointer");
  GS_REQUIRE(nnz == 0 || (indptr && (indices || indices32) && cols && sub_indptr && num_cols_picked > 0),
             "slice_compact_count: null pointer");
  CompactWs w = carve_compact(workspace, num_batches * stride);
  if (workspace == nullptr || workspace_bytes < w.total) {
    set_error("slice_compact workspace too small: %zu < %zu", workspace_bytes, w.total);
    return GS_ERR_WORKSPACE;
  }
  hipStream_t s = as_stream(stream);
  if (num_cols_picked > 0)
    GS_LAUNCH("compact_columns", s,
              compact_offsets_of_columns_kernel<<<dim3((unsigned)ceil_div(num_cols_picked, kBlock)),
                                                  dim3(kBlock), 0, s>>>(
                  batch_ptr, num_batches, stride, num_cols_picked, out_key_offset));
  const int64_t vecs = w.groups * (kCompactGroup / 16);
  int64_t blocks = ceil_div(vecs, kBlock * 4);
  if (blocks > 8192) blocks = 8192;
  GS_LAUNCH("compact_clear", s,
            compact_clear_kernel<<<dim3((unsigned)blocks), dim3(kBlock), 0, s>>>((uint4*)w.flags,
                                                                                 vecs));
  const SliceView view{sub_indptr, cols, indptr, out_key_offset, num_cols_picked};
  if (nnz > 0) {
    const CompactSplit split = compact_split(nnz);
    const dim3 grid((unsigned)ceil_div(ceil_div(nnz, split.run()), kBlock / kWave));
#define GS_COMPACT_MARK(IDT, IDS, ITEMS)                                                       \
  GS_LAUNCH("compact_mark", s,                                                                 \
            (compact_mark_kernel<IDT, ITEMS>)<<<grid, dim3(kBlock), 0, s>>>(IDS, nnz, view,    \
                                                                            split.rounds, w.flags))
    if (indices32 && split.items == 2) GS_COMPACT_MARK(int32_t, indices32, 2);
    else if (indices32) GS_COMPACT_MARK(int32_t, indices32, 8);
    else if (split.items == 2) GS_COMPACT_MARK(int64_t, indices, 2);
    else GS_COMPACT_MARK(int64_t, indices, 8);
#undef GS_COMPACT_MARK
  }
  GS_LAUNCH("compact_words", s,
            compact_words_kernel<uint8_t><<<dim3((unsigned)w.groups), dim3(kBlock), 0, s>>>(
                w.flags, w.words, w.group_cnt));
  GS_LAUNCH("compact_offsets", s,
            compact_offsets_kernel<<<dim3(1), dim3(kCompactScanThreads), 0, s>>>(
                w.group_cnt, w.groups, w.group_off, w.words, num_batches, stride, row_ptr,
                row_ptr_mirror));
  return GS_OK;
}

int gs_slice_compact_fill(const int64_t* indptr, const int64_t* indices, const int32_t* indices32,
                          const int64_t* cols, int64_t num_cols_picked, const int64_t* sub_indptr,
                          int64_t nnz, const int64_t* key_offset, int64_t num_batches,
                          int64_t stride, int64_t* out_rows, int64_t* out_coo_col,
                          int64_t* out_indices, int64_t* out_select, void* workspace,
                          size_t workspace_bytes, gs_stream_t stream) {
  using namespace gs;
  int rc = check_compact(num_cols_picked, nnz, num_batches, stride, "slice_compact_fill");
  if (rc != GS_OK) return rc;
  if (nnz == 0) return GS_OK;
  GS_REQUIRE(indptr && (indices || indices32) && cols && sub_indptr && key_offset && out_rows &&
                 num_cols_picked > 0 && stride > 0,
             "slice_compact_fill: null pointer");
  GS_REQUIRE((out_indices == nullptr) == (out_select == nullptr) && (out_indices || !out_coo_col),
             "slice_compact_fill: out_indices and out_select go together");
  CompactWs w = carve_compact(workspace, num_batches * stride);
  if (workspace == nullptr || workspace_bytes < w.total) {
    set_error("slice_compact workspace too small: %zu < %zu", workspace_bytes, w.total);
    return GS_ERR_WORKSPACE;
  }
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("compact_rows", s,
            compact_rows_kernel<<<dim3((unsigned)w.groups), dim3(kBlock), 0, s>>>(
                w.words, w.group_off, stride, nullptr, out_rows, nullptr));
  if (out_indices == nullptr) return GS_OK;
  const SliceView view{sub_indptr, cols, indptr, key_offset, num_cols_picked};
  const CompactSplit split = compact_split(nnz);
  const dim3 grid((unsigned)ceil_div(ceil_div(nnz, split.run()), kBlock / kWave));
#define GS_COMPACT_FILL(IDT, IDS, ITEMS)                                                       \
  GS_LAUNCH("compact_fill", s,                                                                 \
            (compact_fill_kernel<IDT, ITEMS>)<<<grid, dim3(kBlock), 0, s>>>(                   \
                IDS, nnz, view, split.rounds, w.words, w.group_off, out_coo_col, out_indices,  \
                out_select))
  if (indices32 && split.items == 2) GS_COMPACT_FILL(int32_t, indices32, 2);
  else if (indices32) GS_COMPACT_FILL(int32_t, indices32, 8);
  else if (split.items == 2) GS_COMPACT_FILL(int64_t, indices, 2);
  else GS_COMPACT_FILL(int64_t, indices, 8);
#undef GS_COMPACT_FILL
  return GS_OK;
}

size_t gs_encoded_square_sums_workspace_bytes(int64_t nnz, int64_t num_batches, int64_t stride) {
  if (nnz < 0 || num_batches < 1 || stride < 0 ||
      (stride > 0 && num_batches > ((int64_t(1) << 31) - 1) / stride))
    return 0;
  return gs::carve_encoded_sums(nullptr, nnz, num_batches * stride).total;
}

// (Four bytes a key are cleared, read back twice and added to; without ranges of rows an
// atomic per tile and key is the cost, which a written slice's fewer rows need not pay.)
int gs_encoded_square_sums_pay(int64_t nnz, int64_t num_batches, int64_t stride) {
  if (nnz < 1 || num_batches < 1 || stride < 1 ||
      num_batches > ((int64_t(1) << 31) - 1) / stride)
    return 0;
  const int64_t keys = num_batches * stride;
  if (nnz >= (int64_t(1) << 20))
    return gs::sums_by_range(nnz, gs::ceil_div(keys, gs::kCompactGroup) * gs::kCompactGroup) ? 1 : 0;
  return keys <= (int64_t(1) << 22) || keys / 16 <= nnz ? 1 : 0;
}

int gs_encoded_square_sums(const int64_t* indptr, const int64_t* indices, const int32_t* indices32,
                           const int64_t* cols, int64_t num_cols_picked,
                           const int64_t* sub_indptr, int64_t nnz, const int64_t* key_offset,
                           int64_t num_batches, int64_t stride, const int64_t* edge_map,
                           const float* efeat, int64_t* row_ptr, int64_t* row_ptr_mirror,
                           void* workspace, size_t workspace_bytes, gs_stream_t stream) {
  using namespace gs;
  int rc = check_compact(num_cols_picked, nnz, num_batches, stride, "encoded_square_sums");
  if (rc != GS_OK) return rc;
  GS_REQUIRE(stride == 0 || num_batches <= ((int64_t(1) << 31) - 1) / stride,
             "encoded_square_sums: too many keys");
  GS_REQUIRE(row_ptr, "encoded_square_sums: null pointer");
  GS_REQUIRE(nnz == 0 || (indptr && indices && cols && sub_indptr && key_offset && efeat &&
                          num_cols_picked > 0),
             "encoded_square_sums: null pointer");
  const int64_t range = num_batches * stride;
  EncodedSumsWs w = carve_encoded_sums(workspace, nnz, range);
  if (workspace == nullptr || workspace_bytes < w.total) {
    set_error("encoded_square_sums workspace too small: %zu < %zu", workspace_bytes, w.total);
    return GS_ERR_WORKSPACE;
  }
  hipStream_t s = as_stream(stream);
  // (all groups whole, so that those of the last one past the keys count as none too)
  const SliceView view{sub_indptr, cols, indptr, key_offset, num_cols_picked};
  rc = sliced_square_sum(view, indices, indices32, nnz, edge_map, efeat, w.sums,
                         w.rows.groups * kCompactGroup, w.sum_ws, w.sum_ws_bytes, s,
                         SumsOnto{true, -0.f});
  if (rc != GS_OK) return rc;
  GS_LAUNCH("compact_words", s,
            compact_words_kernel<float><<<dim3((unsigned)w.rows.groups), dim3(kBlock), 0, s>>>(
                w.sums, w.rows.words, w.rows.group_cnt));
  GS_LAUNCH("compact_offsets", s,
            compact_offsets_kernel<<<dim3(1), dim3(kCompactScanThreads), 0, s>>>(
                w.rows.group_cnt, w.rows.groups, w.rows.group_off, w.rows.words, num_batches,
                stride, row_ptr, row_ptr_mirror));
  return GS_OK;
}

int gs_encoded_square_sums_rows(int64_t nnz, int64_t num_batches, int64_t stride,
                                int64_t* out_rows, float* out_sums, void* workspace,
                                size_t workspace_bytes, gs_stream_t stream) {
  using namespace gs;
  int rc = check_compact(0, nnz, num_batches, stride, "encoded_square_sums_rows");
  if (rc != GS_OK) return rc;
  if (nnz == 0 || stride == 0) return GS_OK;
  GS_REQUIRE(out_rows && out_sums, "encoded_square_sums_rows: null pointer");
  EncodedSumsWs w = carve_encoded_sums(workspace, nnz, num_batches * stride);
  if (workspace == nullptr || workspace_bytes < w.total) {
    set_error("encoded_square_sums workspace too small: %zu < %zu", workspace_bytes, w.total);
    return GS_ERR_WORKSPACE;
  }
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("compact_rows", s,
            compact_rows_kernel<<<dim3((unsigned)w.rows.groups), dim3(kBlock), 0, s>>>(
                w.rows.words, w.rows.group_off, stride, w.sums, out_rows, out_sums));
  return GS_OK;
}

}  // extern "C"

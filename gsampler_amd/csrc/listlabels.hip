// listlabels.hip -- frontier and labels of a matrix whose rows are positions
// in a short list of ids (what a row slice by a few hundred picked ids leaves
// behind): one work-group, everything in LDS.
//
// Every edge of local row l carries the same key list_ids[l], so the listed
// ids, ordered by the first edge that uses each, give the same first-occurrence
// frontier as the edges themselves would (seeds first); the labels of the
// edges are then two gathers by local row and by column.
#include "common.h"
#include "listlabels.h"

namespace gs {

__global__ __launch_bounds__(kLabelThreads) void list_labels_kernel(
    const int64_t* __restrict__ seeds, int num_seeds, const int64_t* __restrict__ list_ids,
    const int64_t* __restrict__ first_pos, int num_ids, int64_t* __restrict__ out_frontier,
    int64_t* __restrict__ out_count, int64_t* out_count_mirror,
    int64_t* __restrict__ out_list_label, int64_t* __restrict__ out_seed_label) {
  const int total = list_labels_of(seeds, num_seeds, list_ids, 0, first_pos, num_ids, out_frontier,
                                   out_list_label, out_seed_label);
  if (threadIdx.x == 0) {
    if (out_count) *out_count = total;
    if (out_count_mirror) store_for_host(out_count_mirror, total);
  }
}

// The same for every mini-batch of a super-batch whose rows are positions in a
// list with a segment per batch (what a row slice of an encoded batch matrix
// leaves behind).  The general path partitions and hashes every edge; here each
// batch has a few hundred keys and millions of edges between them, all of them in
// a few buckets of that partition.  One work-group a batch, its frontier to the
// place of its bound; then the frontiers move together, and one pass over the
// edges gathers their labels and checks that each edge's row lies in its batch's
// segment, which nothing else guarantees: if one does not, or a batch has too many
// keys, the size that reaches the host is -1 and the general path is taken.
// Measured on 8 batches, 3.9 M edges, 256 listed ids and 384 seeds each: partition,
// hash, rank and label passes with the gather and decode in front of them 400 us,
// this path 45 us behind the first-position pass (11 us).
__global__ __launch_bounds__(kLabelThreads) void batch_list_labels_kernel(
    const int64_t* __restrict__ seeds, const int64_t* __restrict__ seeds_ptr,
    const int64_t* __restrict__ list_ids, const int64_t* __restrict__ list_ptr, int64_t num_ids,
    int64_t id_stride, const int64_t* __restrict__ first_pos,
    int64_t* __restrict__ bound_frontier, int64_t* __restrict__ counts,
    int64_t* __restrict__ out_list_label, int64_t* __restrict__ out_seed_label) {
  const int64_t b = blockIdx.x;
  const int64_t s0 = seeds_ptr[b], s1 = seeds_ptr[b + 1];
  const int64_t l0 = list_ptr[b], l1 = list_ptr[b + 1];
  if (l0 < 0 || l1 < l0 || l1 > num_ids || (s1 - s0) + (l1 - l0) > kLabelMaxKeys) {
    if (threadIdx.x == 0) counts[b] = -1;  // the whole work-group leaves
    return;
  }
  const int total = list_labels_of(seeds + s0, (int)(s1 - s0), list_ids + l0, id_stride,
                                   first_pos + l0, (int)(l1 - l0), bound_frontier + s0 + l0,
                                   out_list_label + l0, out_seed_label + s0);
  if (threadIdx.x == 0) counts[b] = total;
}

// A work-group per batch: its frontier to its place behind those of the batches
// before it.  The first one also clears or raises the flag of a refused batch.  mirror: no pass
// over edges can refuse any more, and the batch pointer is the host's too (in a launch of its own,
// which is for those that can, 3 us and the gap in front of it).
__global__ __launch_bounds__(kBlock) void batch_list_frontier_kernel(
    const int64_t* __restrict__ seeds_ptr, const int64_t* __restrict__ list_ptr,
    const int64_t* __restrict__ counts, int64_t num_batches,
    const int64_t* __restrict__ bound_frontier, int64_t* __restrict__ out_frontier,
    int64_t* __restrict__ unique_ptr, int* __restrict__ refused, int64_t* mirror) {
  __shared__ int64_t smem[kBlock / kWave + 1];
  __shared__ int any_refused;
  const int64_t b = blockIdx.x;
  if (threadIdx.x == 0) any_refused = 0;
  __syncthreads();
  int64_t mine = 0, base;
  for (int64_t i = threadIdx.x; i < num_batches; i += kBlock) {
    const int64_t n = counts[i];
    if (n < 0) any_refused = 1;  // every writer stores the same value
    if (i < b && n > 0) mine += n;
  }
  block_exclusive_sum<int64_t, kBlock>(mine, smem, &base);
  const int64_t n = counts[b] > 0 ? counts[b] : 0;
  if (threadIdx.x == 0) {
    unique_ptr[b] = base;
    if (mirror) store_for_host(mirror + b, base);
    if (b == num_batches - 1) {
      const int64_t total = mirror && any_refused ? -1 : base + n;
      unique_ptr[num_batches] = total;
      if (mirror) store_for_host(mirror + num_batches, total);
    }
    if (b == 0 && refused) *refused = any_refused;
  }
  if (n == 0) return;
  const int64_t* from = bound_frontier + seeds_ptr[b] + list_ptr[b];
  for (int64_t i = threadIdx.x; i < n; i += kBlock) out_frontier[base + i] = from[i];
}

constexpr int kEdgeLabelItems = 8;
constexpr int kEdgeLabelTile = kBlock * kEdgeLabelItems;
__global__ __launch_bounds__(kBlock) void batch_list_edges_kernel(
    const int64_t* __restrict__ row, const int64_t* __restrict__ col, int64_t nnz,
    const int64_t* __restrict__ edge_ptr, const int64_t* __restrict__ list_ptr,
    int64_t num_batches, int64_t num_ids, int64_t num_seeds,
    const int64_t* __restrict__ list_label, const int64_t* __restrict__ seed_label,
    int64_t* __restrict__ out_row, int64_t* __restrict__ out_col, int* __restrict__ refused) {
  const int64_t e0 = (int64_t)blockIdx.x * kEdgeLabelTile;
  const int64_t last = e0 + kEdgeLabelTile <= nnz ? e0 + kEdgeLabelTile - 1 : nnz - 1;
  const SegmentSpan span = segment_span(edge_ptr, num_batches, e0, last);
  const int64_t lo = list_ptr[span.lo], hi = list_ptr[span.lo + 1];
  int64_t r[kEdgeLabelItems], c[kEdgeLabelItems];
#pragma unroll
  for (int j = 0; j < kEdgeLabelItems; ++j) {
    const int64_t e = e0 + j * kBlock + threadIdx.x;
    r[j] = e < nnz ? row[e] : 0;
    c[j] = e < nnz ? col[e] : 0;
  }
  bool outside = false;
#pragma unroll
  for (int j = 0; j < kEdgeLabelItems; ++j) {
    const int64_t e = e0 + j * kBlock + threadIdx.x;
    if (e >= nnz) continue;
    if (span.lo == span.hi) {
      outside |= r[j] < lo || r[j] >= hi;
    } else {
      const int64_t b = span.segment_at(edge_ptr, e);
      outside |= r[j] < list_ptr[b] || r[j] >= list_ptr[b + 1];
    }
    // (rows and columns may be the caller's: none is read past the lists)
    const bool row_in = (uint64_t)r[j] < (uint64_t)num_ids, col_in = (uint64_t)c[j] < (uint64_t)num_seeds;
    outside |= !row_in || !col_in;
    out_row[e] = list_label[row_in ? r[j] : 0];
    out_col[e] = seed_label[col_in ? c[j] : 0];
  }
  if (__any(outside) && lane_id() == 0) *refused = 1;
}

// The same for one batch.  kByIndptr: the edges are grouped by column, whose number then
// comes from the pointer in place of a read per edge: two gathers over 7.2 M edges took
// 47 us, this takes 33 (173 MB, 36 at the rate of a copy from memory: the rows are still
// in the last-level cache).
template <bool kByIndptr>
__global__ __launch_bounds__(kBlock) void list_edges_kernel(
    const int64_t* __restrict__ row, const int64_t* __restrict__ col,
    const int64_t* __restrict__ indptr, int64_t num_cols, int64_t nnz, int64_t num_ids,
    const int64_t* __restrict__ list_label, const int64_t* __restrict__ seed_label,
    int64_t* __restrict__ out_row, int64_t* __restrict__ out_col) {
  // a wavefront takes neighbouring edges, so that most have one column or two between them
  constexpr int kWaveEdges = kEdgeLabelItems * kWave;
  const int64_t e0 = (int64_t)blockIdx.x * kEdgeLabelTile + threadIdx.x / kWave * kWaveEdges;
  if (e0 >= nnz) return;  // whole wavefronts
  const int64_t last = e0 + kWaveEdges <= nnz ? e0 + kWaveEdges - 1 : nnz - 1;
  int64_t r[kEdgeLabelItems], c[kEdgeLabelItems];
#pragma unroll
  for (int j = 0; j < kEdgeLabelItems; ++j) {
    const int64_t at = e0 + j * kWave + lane_id(), e = at < last ? at : last;
    r[j] = row[e];
    if (!kByIndptr) c[j] = col[e];
  }
  if (kByIndptr) {
    const SegmentSpan span = segment_span(indptr, num_cols, e0, last);
    if (span.hi - span.lo <= 1) {
      const int64_t split = indptr[span.hi];  // (of one column: not after e0)
#pragma unroll
      for (int j = 0; j < kEdgeLabelItems; ++j)
        c[j] = e0 + j * kWave + lane_id() < split ? span.lo : span.hi;
    } else {
#pragma unroll
      for (int j = 0; j < kEdgeLabelItems; ++j) {
        const int64_t at = e0 + j * kWave + lane_id();
        c[j] = span.segment_at(indptr, at < last ? at : last);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < kEdgeLabelItems; ++j) {
    r[j] = list_label[(uint64_t)r[j] < (uint64_t)num_ids ? r[j] : 0];
    c[j] = seed_label[(uint64_t)c[j] < (uint64_t)num_cols ? c[j] : 0];
  }
#pragma unroll
  for (int j = 0; j < kEdgeLabelItems; ++j) {
    const int64_t e = e0 + j * kWave + lane_id();
    if (e > last) break;
    out_row[e] = r[j];
    out_col[e] = c[j];
  }
}

// The batch pointer of the frontier for the host: its last entry -1 if refused, on the device
// too (the host copy may be made again from there).
__global__ __launch_bounds__(kBlock) void batch_list_publish_kernel(
    int64_t* __restrict__ unique_ptr, int64_t num_batches, const int* __restrict__ refused,
    int64_t* mirror) {
  for (int64_t b = threadIdx.x; b <= num_batches; b += kBlock) {
    const bool none = b == num_batches && *refused;
    if (none) unique_ptr[b] = -1;
    store_for_host(mirror + b, none ? -1 : unique_ptr[b]);
  }
}

int batch_list_frontier(const int64_t* seeds_ptr, const int64_t* list_ptr, const int64_t* counts,
                        int64_t num_batches, const int64_t* bound_frontier, int64_t* out_frontier,
                        int64_t* unique_ptr, int64_t* mirror, hipStream_t s) {
  GS_LAUNCH("list_frontier", s,
            batch_list_frontier_kernel<<<dim3((unsigned)num_batches), dim3(kBlock), 0, s>>>(
                seeds_ptr, list_ptr, counts, num_batches, bound_frontier, out_frontier, unique_ptr,
                nullptr, mirror));
  return GS_OK;
}

}  // namespace gs

extern "C" int gs_list_labels(const int64_t* seeds, int64_t num_seeds, const int64_t* list_ids,
                              const int64_t* first_pos, int64_t num_ids,
                              int64_t* out_frontier, int64_t* out_count,
                              int64_t* out_count_mirror, int64_t* out_list_label,
                              int64_t* out_seed_label, gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(num_seeds >= 0 && num_ids >= 0, "list_labels: negative size");
  GS_REQUIRE(num_seeds + num_ids <= kLabelMaxKeys,
             "list_labels: %lld seeds + %lld listed ids exceed %d keys; use gs_unique_count / "
             "gs_unique_relabel",
             (long long)num_seeds, (long long)num_ids, kLabelMaxKeys);
  GS_REQUIRE(num_seeds == 0 || (seeds && out_seed_label), "list_labels: null seeds");
  GS_REQUIRE(num_ids == 0 || (list_ids && first_pos && out_list_label),
             "list_labels: null list");
  GS_REQUIRE(num_seeds + num_ids == 0 || out_frontier, "list_labels: null out_frontier");
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("list_labels", s,
            list_labels_kernel<<<dim3(1), dim3(kLabelThreads), 0, s>>>(
                seeds, (int)num_seeds, list_ids, first_pos, (int)num_ids, out_frontier,
                out_count, out_count_mirror, out_list_label, out_seed_label));
  return GS_OK;
}

extern "C" int gs_list_edge_labels(const int64_t* row, const int64_t* col, const int64_t* indptr,
                                   int64_t num_cols, int64_t nnz, const int64_t* list_label,
                                   int64_t num_ids, const int64_t* seed_label, int64_t* out_row,
                                   int64_t* out_col, gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(num_cols >= 0 && nnz >= 0 && num_ids >= 0, "list_edge_labels: negative size");
  if (nnz == 0) return GS_OK;
  GS_REQUIRE(row && (col || indptr) && list_label && seed_label && out_row && out_col &&
                 num_cols > 0 && num_ids > 0,
             "list_edge_labels: null pointer");
  hipStream_t s = as_stream(stream);
  const dim3 grid((unsigned)ceil_div(nnz, kEdgeLabelTile));
  if (indptr)
    GS_LAUNCH("list_edges", s,
              list_edges_kernel<true><<<grid, dim3(kBlock), 0, s>>>(
                  row, nullptr, indptr, num_cols, nnz, num_ids, list_label, seed_label, out_row,
                  out_col));
  else
    GS_LAUNCH("list_edges", s,
              list_edges_kernel<false><<<grid, dim3(kBlock), 0, s>>>(
                  row, col, nullptr, num_cols, nnz, num_ids, list_label, seed_label, out_row,
                  out_col));
  return GS_OK;
}

extern "C" int gs_batch_list_labels(
    const int64_t* seeds, const int64_t* seeds_ptr, int64_t num_seeds, const int64_t* list_ids,
    const int64_t* list_ptr, int64_t num_ids, int64_t id_stride, int64_t num_batches,
    const int64_t* row, const int64_t* col, const int64_t* edge_ptr, int64_t nnz,
    const int64_t* first_pos, int64_t* out_frontier, int64_t* unique_ptr,
    int64_t* unique_ptr_mirror, int64_t* out_list_label, int64_t* out_seed_label,
    int64_t* out_row, int64_t* out_col, int64_t* scratch, gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(num_seeds >= 0 && num_ids >= 0 && nnz >= 0, "batch_list_labels: negative size");
  GS_REQUIRE(num_batches >= 1 && num_batches <= INT32_MAX, "batch_list_labels: %lld batches",
             (long long)num_batches);
  GS_REQUIRE(seeds_ptr && list_ptr && unique_ptr && unique_ptr_mirror && scratch,
             "batch_list_labels: null pointer");
  GS_REQUIRE(num_seeds == 0 || (seeds && out_seed_label), "batch_list_labels: null seeds");
  GS_REQUIRE(num_ids == 0 || (list_ids && first_pos && out_list_label),
             "batch_list_labels: null list");
  GS_REQUIRE(num_seeds + num_ids == 0 || out_frontier, "batch_list_labels: null out_frontier");
  GS_REQUIRE(nnz == 0 || (row && col && edge_ptr && out_row && out_col && num_seeds > 0 &&
                          num_ids > 0),
             "batch_list_labels: null edges");
  hipStream_t s = as_stream(stream);
  int64_t* bound = scratch;
  int64_t* counts = bound + num_seeds + num_ids;
  int* refused = (int*)(counts + num_batches);
  const dim3 batches((unsigned)num_batches);
  GS_LAUNCH("list_labels", s,
            batch_list_labels_kernel<<<batches, dim3(kLabelThreads), 0, s>>>(
                seeds, seeds_ptr, list_ids, list_ptr, num_ids, id_stride, first_pos, bound, counts,
                out_list_label, out_seed_label));
  if (nnz == 0)
    return batch_list_frontier(seeds_ptr, list_ptr, counts, num_batches, bound, out_frontier,
                               unique_ptr, unique_ptr_mirror, s);
  GS_LAUNCH("list_frontier", s,
            batch_list_frontier_kernel<<<batches, dim3(kBlock), 0, s>>>(
                seeds_ptr, list_ptr, counts, num_batches, bound, out_frontier, unique_ptr,
                refused, nullptr));
  GS_LAUNCH("list_edges", s,
              batch_list_edges_kernel<<<dim3((unsigned)ceil_div(nnz, kEdgeLabelTile)),
                                        dim3(kBlock), 0, s>>>(
                  row, col, nnz, edge_ptr, list_ptr, num_batches, num_ids, num_seeds,
                  out_list_label, out_seed_label, out_row, out_col, refused));
  GS_LAUNCH("list_publish", s,
            batch_list_publish_kernel<<<dim3(1), dim3(kBlock), 0, s>>>(unique_ptr, num_batches,
                                                                       refused, unique_ptr_mirror));
  return GS_OK;
}

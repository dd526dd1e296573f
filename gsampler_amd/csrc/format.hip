// format.hip -- CSC <-> COO conversion kernels.
#include "common.h"

namespace gs {

// Column id of every edge: the segment of indptr that holds the edge position,
// looked up per tile of consecutive edges.
constexpr int kCooItems = 8;
constexpr int kCooTile = kBlock * kCooItems;

__global__ __launch_bounds__(kBlock) void csc2coo_kernel(
    const int64_t* __restrict__ indptr, int64_t num_cols, int64_t nnz,
    int64_t* __restrict__ out_col) {
  const int64_t e0 = (int64_t)blockIdx.x * kCooTile;
  if (e0 >= nnz) return;
  const int64_t e_last = e0 + kCooTile - 1 < nnz ? e0 + kCooTile - 1 : nnz - 1;
  const SegmentSpan span = segment_span(indptr, num_cols, e0, e_last);
#pragma unroll
  for (int j = 0; j < kCooItems; ++j) {
    const int64_t e = e0 + j * kBlock + threadIdx.x;
    if (e >= nnz) break;
    out_col[e] = span.segment_at(indptr, e);
  }
}

// indptr[c] = number of entries of the sorted column array that are < c.
__global__ __launch_bounds__(kBlock) void sorted_to_indptr_kernel(
    const int64_t* __restrict__ sorted, int64_t nnz, int64_t num_cols,
    int64_t* __restrict__ indptr) {
  const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (c > num_cols) return;
  int64_t lo = 0, hi = nnz;  // first position with sorted[pos] >= c
  while (lo < hi) {
    int64_t mid = (lo + hi) >> 1;
    if (sorted[mid] < c)
      lo = mid + 1;
    else
      hi = mid;
  }
  indptr[c] = lo;
}

}  // namespace gs

namespace gs {

// first[r] = smallest e with ids[e] == r (INT64_MAX for an id that does not
// occur), for ids in a small dense range [0, num_ids).  Atomics from all dies
// on a few hundred addresses would queue up at the memory side, so a
// work-group first takes the minimum over its tile of edges in LDS and then
// sends one atomic per id it met -- and only if the value in memory is not
// already smaller, which it is for every tile but the first few.
//
// A work-group is one trip to memory for its edges, one chain of LDS operations and
// one trip for the ids it met: what bounds it is that chain, not the bytes (tiles of 8192
// edges and 256 threads, four such trips one after the other and 64-bit words in LDS, took
// 40 us on 7.2 M edges and 15 on 3.1 M; now 21 and 8).
constexpr int kFirstLdsIds = GS_FIRST_POSITION_FEW_IDS;
constexpr int kFirstThreads = 1024;
constexpr int kFirstItems = 16;
constexpr int kFirstTile = kFirstThreads * kFirstItems;

__global__ __launch_bounds__(kFirstThreads) void first_position_lds_kernel(
    const int64_t* __restrict__ ids, int64_t n, int64_t num_ids, long long* first) {
  __shared__ uint32_t tile_min[kFirstLdsIds];  // edges counted from the tile's first
  const int64_t e0 = (int64_t)blockIdx.x * kFirstTile;
  const uint32_t len = (uint32_t)(e0 + kFirstTile < n ? kFirstTile : n - e0);
  int64_t r[kFirstItems];
#pragma unroll
  for (int j = 0; j < kFirstItems; ++j) {
    const uint32_t i = j * kFirstThreads + threadIdx.x;
    r[j] = ids[e0 + (i < len ? i : len - 1)];
  }
  for (int i = threadIdx.x; i < num_ids; i += kFirstThreads) tile_min[i] = UINT32_MAX;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kFirstItems; ++j) {
    const uint32_t i = j * kFirstThreads + threadIdx.x;
    if (i < len && (uint64_t)r[j] < (uint64_t)num_ids && tile_min[r[j]] > i)
      atomicMin(&tile_min[r[j]], i);
  }
  __syncthreads();
  constexpr int kShare = kFirstLdsIds / kFirstThreads;
  long long held[kShare];
#pragma unroll
  for (int j = 0; j < kShare; ++j) {
    const int i = j * kFirstThreads + threadIdx.x;
    held[j] = i < num_ids ? __hip_atomic_load(first + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                          : -1;
  }
#pragma unroll
  for (int j = 0; j < kShare; ++j) {
    const int i = j * kFirstThreads + threadIdx.x;
    if (i >= num_ids || tile_min[i] == UINT32_MAX) continue;
    const long long m = e0 + tile_min[i];
    if (held[j] > m) atomicMin(first + i, m);
  }
}

// The same for a range of ids too large for LDS: one atomic per edge unless a
// smaller position is already there.
__global__ __launch_bounds__(kBlock) void first_position_kernel(
    const int64_t* __restrict__ ids, int64_t n, int64_t num_ids, long long* first) {
  const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (e >= n) return;
  const int64_t r = ids[e];
  if (r < 0 || r >= num_ids) return;
  if (__hip_atomic_load(first + r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) > e)
    atomicMin(first + r, (long long)e);
}

__global__ __launch_bounds__(kBlock) void fill_i64_kernel(int64_t* p, int64_t n, int64_t v) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = v;
}

}  // namespace gs

extern "C" {

int gs_csc2coo(const int64_t* indptr, int64_t num_cols, int64_t nnz,
               int64_t* out_col, gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(num_cols >= 0 && nnz >= 0, "csc2coo: negative size");
  if (nnz == 0) return GS_OK;
  GS_REQUIRE(indptr && out_col, "csc2coo: null pointer");
  GS_REQUIRE(num_cols > 0, "csc2coo: %lld edges but no columns", (long long)nnz);
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("csc2coo", s,
            csc2coo_kernel<<<dim3((unsigned)ceil_div(nnz, kCooTile)), dim3(kBlock),
                             0, s>>>(indptr, num_cols, nnz, out_col));
  return GS_OK;
}

int gs_sorted_to_indptr(const int64_t* sorted_ids, int64_t nnz, int64_t num_cols,
                        int64_t* out_indptr, gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(num_cols >= 0 && nnz >= 0, "sorted_to_indptr: negative size");
  GS_REQUIRE(out_indptr && (nnz == 0 || sorted_ids),
             "sorted_to_indptr: null pointer");
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("sorted_to_indptr", s,
            sorted_to_indptr_kernel<<<dim3((unsigned)ceil_div(num_cols + 1, kBlock)),
                                      dim3(kBlock), 0, s>>>(sorted_ids, nnz,
                                                            num_cols, out_indptr));
  return GS_OK;
}

int gs_first_position(const int64_t* ids, int64_t n, int64_t num_ids,
                      int64_t* out_first, gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(n >= 0 && num_ids >= 0, "first_position: negative size");
  if (num_ids == 0) return GS_OK;
  GS_REQUIRE(out_first && (n == 0 || ids), "first_position: null pointer");
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("first_position_init", s,
            fill_i64_kernel<<<dim3((unsigned)ceil_div(num_ids, kBlock)), dim3(kBlock), 0,
                              s>>>(out_first, num_ids, INT64_MAX));
  if (n > 0 && num_ids <= kFirstLdsIds)
    GS_LAUNCH("first_position", s,
              first_position_lds_kernel<<<dim3((unsigned)ceil_div(n, kFirstTile)),
                                          dim3(kFirstThreads), 0, s>>>(ids, n, num_ids,
                                                                (long long*)out_first));
  else if (n > 0)
    GS_LAUNCH("first_position", s,
              first_position_kernel<<<dim3((unsigned)ceil_div(n, kBlock)), dim3(kBlock), 0,
                                      s>>>(ids, n, num_ids, (long long*)out_first));
  return GS_OK;
}

}  // extern "C"

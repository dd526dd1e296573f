// batch.hip -- small super-batch bookkeeping kernels.
#include "common.h"

namespace gs {

__global__ __launch_bounds__(kBlock) void decode_batch_ids_kernel(
    const int64_t* __restrict__ encoded, int64_t n, int64_t stride,
    int64_t* __restrict__ orig, int64_t* __restrict__ batch) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const int64_t v = encoded[i];
  const int64_t b = v / stride;
  if (batch) batch[i] = b;
  if (orig) orig[i] = v - b * stride;
}

// out[i] = ids[i] + batch of item i * stride (without ids: the offset alone).  A few
// thousand items, whose batch pointer stays in the scalar cache: one launch where the
// batch of every item, the product and the sum were three (a ShaDow slice: five in all,
// 26 us with the gaps between them).
__global__ __launch_bounds__(kBlock) void encode_batch_ids_kernel(
    const int64_t* __restrict__ ids, const int64_t* __restrict__ batch_ptr, int64_t num_batches,
    int64_t n, int64_t stride, int64_t* __restrict__ out) {
  const int64_t first = (int64_t)blockIdx.x * kBlock, i = first + threadIdx.x;
  const int64_t last = first + kBlock < n ? first + kBlock - 1 : n - 1;
  const SegmentSpan span = segment_span(batch_ptr, num_batches, first, last);
  if (i >= n) return;
  out[i] = (ids ? ids[i] : 0) + span.segment_at(batch_ptr, i) * stride;
}

// The same for ids picked from a list: id = ids[index[i]] (without index: ids[i]), which goes
// out as it is, moved by its batch, and the move alone, whatever of the three is wanted: one
// launch where a gather and up to two of the above were.  A place outside the list reads no id
// and raises `refused`.  An id that is no row is moved past the rows of all batches, where
// nothing meets it: moved by its batch it would be another batch's row.
__global__ __launch_bounds__(kBlock) void pick_batch_ids_kernel(
    const int64_t* __restrict__ ids, int64_t num_ids, const int64_t* __restrict__ index,
    const int64_t* __restrict__ batch_ptr, int64_t num_batches, int64_t n, int64_t stride,
    int64_t* __restrict__ out_id, int64_t* __restrict__ out_moved,
    int64_t* __restrict__ out_offset, int64_t* refused) {
  const int64_t first = (int64_t)blockIdx.x * kBlock, i = first + threadIdx.x;
  const int64_t last = first + kBlock < n ? first + kBlock - 1 : n - 1;
  const int64_t at = i < n ? (index ? index[i] : i) : 0;
  const bool listed = (uint64_t)at < (uint64_t)num_ids;
  const int64_t id = listed ? ids[at] : 0;
  const SegmentSpan span = segment_span(batch_ptr, num_batches, first, last);
  if (i >= n) return;
  if (!listed && refused) store_for_host(refused, 1);
  const int64_t offset = span.segment_at(batch_ptr, i) * stride;
  if (out_id) out_id[i] = id;
  if (out_moved)
    out_moved[i] = (uint64_t)id < (uint64_t)stride ? id + offset : num_batches * stride;
  if (out_offset) out_offset[i] = offset;
}

// out[e] = the id behind local row rows[e], its remainder by stride where that is not 0 (ids
// encoded as id + batch * stride): a gather, the quotients, and the batch pointer that came
// with those and that nobody read were three launches.  A row outside the list reads its
// first id and raises `refused`.
__global__ __launch_bounds__(kBlock) void local_ids_kernel(
    const int64_t* __restrict__ table, int64_t num_ids, const int64_t* __restrict__ rows,
    int64_t n, int64_t stride, int64_t* __restrict__ out, int64_t* refused) {
  constexpr int kItems = 4;
  const int64_t e0 = (int64_t)blockIdx.x * (kBlock * kItems) + threadIdx.x;
  int64_t v[kItems];
  bool outside = false;
#pragma unroll
  for (int j = 0; j < kItems; ++j) v[j] = rows[e0 + j * kBlock < n ? e0 + j * kBlock : n - 1];
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const bool listed = (uint64_t)v[j] < (uint64_t)num_ids;
    outside |= !listed;
    v[j] = table[listed ? v[j] : 0];
  }
  if (outside && refused) store_for_host(refused, 1);
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    if (stride > 0 && (uint64_t)v[j] >= (uint64_t)stride) v[j] %= stride;
    if (e0 + j * kBlock < n) out[e0 + j * kBlock] = v[j];
  }
}

// Batch b's piece is indptr[offset[b] .. offset[b+1]] (inclusive) rebased to 0,
// written at out[offset[b] - offset[0] + b ...]: the pieces tile the output.  A
// work-group takes kSplitTile consecutive output elements; the pieces start at
// offset[b] - offset[0] + b, which increases strictly with b, so the batches of
// the tile's first and last element are looked up once per work-group (the
// position is the same in every lane: scalar loads) and an element searches
// only between them -- not at all when one piece covers the tile.
// No more pieces than a wavefront has lanes, as most calls have: a lane holds where its piece
// begins and what it begins with, and the piece of an element is told by comparing with those,
// so that two trips to memory lie in front of the stores, not one per step of a search.  64
// batches of 65 K, 592 K and 3.5 M columns in all, us: 7.7, 10.0 and 18.1 with the search, now
// 4.6, 4.6 and 12.9.
constexpr int kSplitItems = 4;
constexpr int kSplitTile = kBlock * kSplitItems;

__device__ __forceinline__ int64_t piece_of(const int64_t* __restrict__ offset, int64_t first,
                                            int64_t lo, int64_t hi, int64_t p) {
  while (hi - lo > 1) {  // the piece lies in [lo, hi)
    const int64_t mid = (lo + hi) >> 1;
    if (offset[mid] - first + mid <= p)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

__device__ __forceinline__ void split_tile(
    int64_t tile, const int64_t* __restrict__ indptr, const int64_t* __restrict__ offset,
    int64_t num_batches, int64_t out_len, int64_t* __restrict__ out) {
  const int64_t p0 = tile * kSplitTile;
  if (p0 >= out_len) return;
  const int64_t p_last = p0 + kSplitTile - 1 < out_len ? p0 + kSplitTile - 1 : out_len - 1;
  if (num_batches <= kWave) {
    const int lane = lane_id();
    const int64_t begin = offset[lane < num_batches ? lane : num_batches - 1];
    const int64_t first = wave_uniform_first(begin);
    const int64_t start = lane < num_batches ? begin - first + lane : INT64_MAX;
    const int b_lo = __popcll(__ballot(start <= p0)) - 1;
    const int b_hi = __popcll(__ballot(start <= p_last)) - 1;
    const int64_t base = indptr[begin];
    int piece[kSplitItems];
    int64_t v[kSplitItems];
#pragma unroll
    for (int i = 0; i < kSplitItems; ++i) {
      int64_t p = p0 + i * kBlock + threadIdx.x;
      if (p > p_last) p = p_last;
      int b = b_lo;
      for (int k = b_lo + 1; k <= b_hi; ++k)
        if (p >= (int64_t)__shfl((long long)start, k, kWave)) b = k;
      piece[i] = b;
      v[i] = indptr[p + first - b];
    }
#pragma unroll
    for (int i = 0; i < kSplitItems; ++i) {
      const int64_t p = p0 + i * kBlock + threadIdx.x;
      const int64_t from = (int64_t)__shfl((long long)base, piece[i], kWave);
      if (p <= p_last) out[p] = v[i] - from;
    }
    return;
  }
  const int64_t first = offset[0];
  const int64_t b_lo = piece_of(offset, first, 0, num_batches, p0);
  const int64_t b_hi = piece_of(offset, first, b_lo, num_batches, p_last);
  int64_t begin = offset[b_lo], base = indptr[begin];
#pragma unroll
  for (int i = 0; i < kSplitItems; ++i) {
    const int64_t p = p0 + i * kBlock + threadIdx.x;
    if (p > p_last) break;
    int64_t b = b_lo;
    if (b_lo != b_hi) {
      b = piece_of(offset, first, b_lo, b_hi + 1, p);
      begin = offset[b];
      base = indptr[begin];
    }
    out[p] = indptr[begin + (p - (begin - first + b))] - base;
  }
}

__global__ __launch_bounds__(kBlock) void split_indptr_kernel(
    const int64_t* __restrict__ indptr, const int64_t* __restrict__ offset,
    int64_t num_batches, int64_t out_len, int64_t* __restrict__ out) {
  split_tile(blockIdx.x, indptr, offset, num_batches, out_len, out);
}

// distinct[b] = 1 when the seeds of batch b are pairwise different.  The
// frontier of a batch lists its keys in first-occurrence order, seeds first, so
// the seeds are distinct exactly when the last seed sits at place ns - 1.
__device__ __forceinline__ int64_t seeds_distinct(
    int64_t b, const int64_t* __restrict__ frontier, const int64_t* __restrict__ frontier_ptr,
    const int64_t* __restrict__ seeds, const int64_t* __restrict__ seeds_ptr) {
  const int64_t s_lo = seeds_ptr[b], ns = seeds_ptr[b + 1] - s_lo;
  const int64_t f_lo = frontier_ptr[b], nu = frontier_ptr[b + 1] - f_lo;
  return ns <= 0 || (nu >= ns && frontier[f_lo + ns - 1] == seeds[s_lo + ns - 1]);
}
__global__ __launch_bounds__(kBlock) void seeds_distinct_kernel(
    const int64_t* __restrict__ frontier, const int64_t* __restrict__ frontier_ptr,
    const int64_t* __restrict__ seeds, const int64_t* __restrict__ seeds_ptr,
    int64_t num_batches, int64_t* __restrict__ distinct) {
  const int64_t b = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (b < num_batches) distinct[b] = seeds_distinct(b, frontier, frontier_ptr, seeds, seeds_ptr);
}

// Both for the hand-over of a layer's blocks, the flags straight to the host as well: one
// launch of 6 us where the pointers, the flags and the flags' copy were three, 11 us and the
// gaps.
__global__ __launch_bounds__(kBlock) void block_offsets_kernel(
    const int64_t* __restrict__ indptr, const int64_t* __restrict__ seeds_ptr,
    int64_t num_batches, int64_t out_len, int64_t* __restrict__ out, unsigned tiles,
    const int64_t* __restrict__ frontier, const int64_t* __restrict__ frontier_ptr,
    const int64_t* __restrict__ seeds, int64_t* __restrict__ distinct, int64_t* distinct_mirror) {
  if (blockIdx.x < tiles) {
    split_tile(blockIdx.x, indptr, seeds_ptr, num_batches, out_len, out);
    return;
  }
  const int64_t b = (int64_t)(blockIdx.x - tiles) * kBlock + threadIdx.x;
  if (b >= num_batches) return;
  const int64_t flag = seeds_distinct(b, frontier, frontier_ptr, seeds, seeds_ptr);
  distinct[b] = flag;
  if (distinct_mirror) store_for_host(distinct_mirror + b, flag);
}

}  // namespace gs

extern "C" {

int gs_batch_seeds_distinct(const int64_t* frontier, const int64_t* frontier_ptr,
                            const int64_t* seeds, const int64_t* seeds_ptr,
                            int64_t num_batches, int64_t* out_distinct,
                            gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(num_batches >= 0, "batch_seeds_distinct: negative size");
  if (num_batches == 0) return GS_OK;
  GS_REQUIRE(frontier_ptr && seeds_ptr && out_distinct, "batch_seeds_distinct: null pointer");
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("seeds_distinct", s,
            seeds_distinct_kernel<<<dim3((unsigned)ceil_div(num_batches, kBlock)), dim3(kBlock),
                                    0, s>>>(frontier, frontier_ptr, seeds, seeds_ptr,
                                            num_batches, out_distinct));
  return GS_OK;
}

int gs_batch_block_offsets(const int64_t* indptr, const int64_t* seeds_ptr, int64_t num_batches,
                           int64_t out_len, int64_t* out, const int64_t* frontier,
                           const int64_t* frontier_ptr, const int64_t* seeds, int64_t* distinct,
                           int64_t* distinct_mirror, gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(num_batches >= 0 && out_len >= 0, "batch_block_offsets: negative size");
  if (num_batches == 0) return GS_OK;
  GS_REQUIRE(indptr && seeds_ptr && (out || out_len == 0) && frontier_ptr && distinct,
             "batch_block_offsets: null pointer");
  hipStream_t s = as_stream(stream);
  const unsigned tiles = (unsigned)ceil_div(out_len, kSplitTile);
  GS_LAUNCH("block_offsets", s,
            block_offsets_kernel<<<dim3(tiles + (unsigned)ceil_div(num_batches, kBlock)),
                                   dim3(kBlock), 0, s>>>(indptr, seeds_ptr, num_batches, out_len,
                                                         out, tiles, frontier, frontier_ptr, seeds,
                                                         distinct, distinct_mirror));
  return GS_OK;
}

int gs_decode_batch_ids(const int64_t* encoded, int64_t n, int64_t stride,
                        int64_t* out_orig, int64_t* out_batch,
                        gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(n >= 0, "decode_batch_ids: negative size");
  GS_REQUIRE(stride > 0, "decode_batch_ids: stride must be positive, got %lld",
             (long long)stride);
  if (n == 0) return GS_OK;
  GS_REQUIRE(encoded, "decode_batch_ids: null pointer");
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("decode_batch_ids", s,
            decode_batch_ids_kernel<<<dim3((unsigned)ceil_div(n, kBlock)),
                                      dim3(kBlock), 0, s>>>(encoded, n, stride,
                                                            out_orig, out_batch));
  return GS_OK;
}

int gs_encode_batch_ids(const int64_t* ids, const int64_t* batch_ptr, int64_t num_batches,
                        int64_t n, int64_t stride, int64_t* out, gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(n >= 0 && num_batches >= 0, "encode_batch_ids: negative size");
  if (n == 0) return GS_OK;
  GS_REQUIRE(num_batches > 0 && batch_ptr && out, "encode_batch_ids: null pointer");
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("encode_batch_ids", s,
            encode_batch_ids_kernel<<<dim3((unsigned)ceil_div(n, kBlock)), dim3(kBlock), 0, s>>>(
                ids, batch_ptr, num_batches, n, stride, out));
  return GS_OK;
}

int gs_pick_batch_ids(const int64_t* ids, int64_t num_ids, const int64_t* index,
                      const int64_t* batch_ptr, int64_t num_batches, int64_t n, int64_t stride,
                      int64_t* out_id, int64_t* out_moved, int64_t* out_offset,
                      int64_t* refused, gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(n >= 0 && num_ids >= 0 && num_batches >= 0, "pick_batch_ids: negative size");
  if (n == 0) return GS_OK;
  GS_REQUIRE(num_batches > 0 && batch_ptr && (ids || num_ids == 0), "pick_batch_ids: null pointer");
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("pick_batch_ids", s,
            pick_batch_ids_kernel<<<dim3((unsigned)ceil_div(n, kBlock)), dim3(kBlock), 0, s>>>(
                ids, num_ids, index, batch_ptr, num_batches, n, stride, out_id, out_moved,
                out_offset, refused));
  return GS_OK;
}

int gs_local_ids(const int64_t* table, int64_t num_ids, const int64_t* rows, int64_t n,
                 int64_t stride, int64_t* out, int64_t* refused, gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(n >= 0 && num_ids >= 0 && stride >= 0, "local_ids: negative size");
  if (n == 0) return GS_OK;
  GS_REQUIRE(num_ids > 0 && table && rows && out, "local_ids: null pointer");
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("local_ids", s,
            local_ids_kernel<<<dim3((unsigned)ceil_div(n, kBlock * 4)), dim3(kBlock), 0, s>>>(
                table, num_ids, rows, n, stride, out, refused));
  return GS_OK;
}

int gs_split_indptr(const int64_t* indptr, const int64_t* offset,
                    int64_t num_batches, int64_t out_len, int64_t* out,
                    gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(num_batches >= 0 && out_len >= 0, "split_indptr: negative size");
  if (num_batches == 0 || out_len == 0) return GS_OK;
  GS_REQUIRE(indptr && offset && out, "split_indptr: null pointer");
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("split_indptr", s,
            split_indptr_kernel<<<dim3((unsigned)ceil_div(out_len, kSplitTile)),
                                  dim3(kBlock), 0, s>>>(indptr, offset,
                                                        num_batches, out_len, out));
  return GS_OK;
}

}  // extern "C"

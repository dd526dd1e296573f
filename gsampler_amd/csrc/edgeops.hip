// edgeops.hip -- edge-wise compute operators of layer-wise samplers:
// generalized SDDMM (a value per edge from its endpoints), generalized SpMM
// (reduce edge values onto rows or columns) and their fusions (sum of squares,
// sum of e / u, two u-op-v products in one sweep).
//
// Endpoint convention (same as the reference, src/cuda/sddmm.cu:37-38,134-135):
// on COO  src = row[e], dst = col[e]; on a compressed matrix src = indices[e]
// and dst = the segment of indptr that holds e.  Targets: 0 = src ("u"),
// 1 = edge, 2 = dst ("v").  All kernels are memory bound; features are scalar
// in every sampler that uses them, so the fast paths are the feature-length-1
// ones and the general-length paths favour simplicity.
#include <type_traits>

#include "common.h"
#include "scan.h"
#include "sums.h"

namespace gs {

enum { kOpAdd = 0, kOpSub, kOpMul, kOpDiv, kOpCopyLhs, kOpCopyRhs, kOpDot };
enum { kReduceSum = 0, kReduceMax, kReduceMin };

template <typename T>
__device__ __forceinline__ T apply_op(int op, const T* l, const T* r,
                                      int64_t reduce_size) {
  switch (op) {
    case kOpAdd: return l[0] + r[0];
    case kOpSub: return l[0] - r[0];
    case kOpMul: return l[0] * r[0];
    case kOpDiv: return l[0] / r[0];
    case kOpCopyLhs: return l[0];
    case kOpCopyRhs: return r[0];
    default: {
      T acc = 0;
      for (int64_t k = 0; k < reduce_size; ++k) acc += l[k] * r[k];
      return acc;
    }
  }
}

__device__ __forceinline__ int64_t pick(int target, int64_t src, int64_t eid,
                                        int64_t dst) {
  return target == 0 ? src : (target == 1 ? eid : dst);
}

struct EdgeView {
  int compressed;      // 1: (indptr, indices), 0: (row, col)
  const int64_t* a;    // row | indptr
  const int64_t* b;    // col | indices
  int64_t num_major;   // segments of indptr
  const int64_t* edge_map;
  // Segments that the edges [e_first, e_last] of one work-group touch
  // (compressed form only): looked up once per wavefront.
  __device__ __forceinline__ SegmentSpan span(int64_t e_first, int64_t e_last) const {
    if (!compressed) return SegmentSpan{0, 0};
    return segment_span(a, num_major, e_first, e_last);
  }
  __device__ __forceinline__ void endpoints(const SegmentSpan& sp, int64_t e, int64_t* src,
                                            int64_t* dst, int64_t* eid) const {
    if (compressed) {
      *src = b[e];
      *dst = sp.segment_at(a, e);
    } else {
      *src = a[e];
      *dst = b[e];
    }
    *eid = edge_map ? edge_map[e] : e;
  }
};

// Element idx of an [nnz, out_len] output -> its edge and its place in the feature.
// A 64-bit division takes some forty instructions, more than the rest of an element:
// none for scalars, a 32-bit one while the whole output has fewer than 2^32 elements.
__device__ __forceinline__ void split_index(int64_t idx, int64_t total, int64_t out_len, int64_t* e,
                                            int64_t* f) {
  if (out_len == 1) {
    *e = idx;
    *f = 0;
  } else if (total < (int64_t(1) << 32)) {
    const uint32_t q = (uint32_t)idx / (uint32_t)out_len;
    *e = q;
    *f = (uint32_t)idx - q * (uint32_t)out_len;
  } else {
    *e = idx / out_len;
    *f = idx - *e * out_len;
  }
}

// A work-group handles kBlock * ITEMS consecutive elements of an
// [nnz, out_len] output.  On a compressed form ITEMS = kEdgeItems, so that the
// look-up of the segments its edges touch is paid once per 2048 elements; an
// edge list needs no look-up and runs with one element per thread.
constexpr int kEdgeItems = 8;

template <int ITEMS>
__device__ __forceinline__ SegmentSpan block_edge_span(const EdgeView& g, int64_t nnz,
                                                       int64_t out_len) {
  const int64_t idx0 = (int64_t)blockIdx.x * (kBlock * ITEMS);
  int64_t idx_last = idx0 + kBlock * ITEMS - 1;
  if (idx_last > nnz * out_len - 1) idx_last = nnz * out_len - 1;
  return g.span(idx0 / out_len, idx_last / out_len);
}

// ------------------------------------------------------------------ SDDMM
template <typename T, int ITEMS>
__global__ __launch_bounds__(kBlock) void sddmm_kernel(
    EdgeView g, int64_t nnz, int op, const T* __restrict__ lhs,
    const T* __restrict__ rhs, T* __restrict__ out, int lhs_target,
    int rhs_target, int64_t lhs_len, int64_t rhs_len, int64_t out_len,
    int64_t reduce_size, const int64_t* __restrict__ lhs_off,
    const int64_t* __restrict__ rhs_off) {
  const int64_t idx0 = (int64_t)blockIdx.x * (kBlock * ITEMS);
  if (idx0 >= nnz * out_len) return;
  const SegmentSpan sp = block_edge_span<ITEMS>(g, nnz, out_len);
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const int64_t idx = idx0 + j * kBlock + threadIdx.x;
    if (idx >= nnz * out_len) break;
    int64_t e, f;
    split_index(idx, nnz * out_len, out_len, &e, &f);
    int64_t src, dst, eid;
    g.endpoints(sp, e, &src, &dst, &eid);
    const int64_t lf = lhs_off ? lhs_off[f] : f, rf = rhs_off ? rhs_off[f] : f;
    const T* l = op == kOpCopyRhs
                     ? nullptr
                     : lhs + pick(lhs_target, src, eid, dst) * lhs_len + lf * reduce_size;
    const T* r = op == kOpCopyLhs
                     ? nullptr
                     : rhs + pick(rhs_target, src, eid, dst) * rhs_len + rf * reduce_size;
    out[eid * out_len + f] = apply_op<T>(op, l, r, reduce_size);
  }
}

// One value an edge on an edge list (the divisions of a layer-wise sampler): lhs_ids
// and rhs_ids are the id array an operand is read through, null for a value of the
// edge's own.  Four edges a lane, whose loads are in flight together, and only the
// ids that an operand needs: 7.3 M edges 41 us one edge a lane with both ids,
// 28 so (602 M edges: 2.85 and 1.63 ms).
constexpr int kScalarItems = 4;
template <typename T>
__global__ __launch_bounds__(kBlock) void sddmm_scalar_kernel(
    int64_t nnz, int op, const int64_t* __restrict__ edge_map,
    const int64_t* __restrict__ lhs_ids, const int64_t* __restrict__ rhs_ids,
    const T* __restrict__ lhs, const T* __restrict__ rhs, T* __restrict__ out) {
  const int64_t e0 = (int64_t)blockIdx.x * (kBlock * kScalarItems) + threadIdx.x;
  int64_t e[kScalarItems], eid[kScalarItems], li[kScalarItems], ri[kScalarItems];
#pragma unroll
  for (int j = 0; j < kScalarItems; ++j) {
    const int64_t at = e0 + j * kBlock;
    e[j] = eid[j] = at < nnz ? at : nnz - 1;
  }
  if (edge_map)
#pragma unroll
    for (int j = 0; j < kScalarItems; ++j) eid[j] = edge_map[e[j]];
#pragma unroll
  for (int j = 0; j < kScalarItems; ++j) li[j] = ri[j] = eid[j];
  if (lhs_ids)
#pragma unroll
    for (int j = 0; j < kScalarItems; ++j) li[j] = lhs_ids[e[j]];
  if (rhs_ids)
#pragma unroll
    for (int j = 0; j < kScalarItems; ++j) ri[j] = rhs_ids[e[j]];
  T l[kScalarItems] = {}, r[kScalarItems] = {};
  if (op != kOpCopyRhs)
#pragma unroll
    for (int j = 0; j < kScalarItems; ++j) l[j] = lhs[li[j]];
  if (op != kOpCopyLhs)
#pragma unroll
    for (int j = 0; j < kScalarItems; ++j) r[j] = rhs[ri[j]];
#pragma unroll
  for (int j = 0; j < kScalarItems; ++j)
    if (e0 + j * kBlock < nnz) out[eid[j]] = apply_op<T>(op, &l[j], &r[j], 1);
}

// ------------------------------------------------------------- edge scores
// What an attention sampler does with every edge -- products of two endpoints' features
// summed over the feature, quotients, a weighted sum of those, its positive part, a
// small constant -- in one pass: nothing between the endpoints' rows and the score is
// written.  368 K edges, two products over 16 features of 100 K rows and a quotient:
// 2 x 46 us for the products and their sums, 4 for the quotient and 279 for stacking
// the three, the matrix-vector product, which is given a work-group an edge, and the
// rest; 18 us here, bound by the gathers of the 64-byte rows from L2.
//
// Additions go in the order torch's own kernels take, so that a sampler draws the same
// samples with and without this pass: a feature of length len is folded at the largest
// power of two P <= len (x[t] + x[t + P]) and then added up in pairs of neighbours, the
// terms in pairs half their number apart.
struct ScoreArgs {
  gs_score_term term[GS_SCORE_MAX_TERMS];
  int num_terms, len, positive_part;
  float shift;
  const float* weights;
};

template <int P, bool kWide>
__device__ __forceinline__ float products_sum(const float* __restrict__ l,
                                              const float* __restrict__ r, int len) {
#pragma clang fp contract(off)
  constexpr int kMost = 2 * P;  // (P <= len < 2 P)
  float x[kMost];
  if (kWide) {  // rows of whole, aligned 16 bytes
#pragma unroll
    for (int q = 0; q < kMost / 4; ++q) {
      float4 a = make_float4(0, 0, 0, 0), b = a;
      if (4 * q < len) {
        a = ((const float4*)l)[q];
        b = ((const float4*)r)[q];
      }
      x[4 * q] = a.x * b.x;
      x[4 * q + 1] = a.y * b.y;
      x[4 * q + 2] = a.z * b.z;
      x[4 * q + 3] = a.w * b.w;
    }
  } else {
#pragma unroll
    for (int t = 0; t < kMost; ++t) x[t] = t < len ? l[t] * r[t] : 0.f;
  }
#pragma unroll
  for (int t = 0; t < P; ++t) x[t] += t + P < len ? x[t + P] : 0.f;
#pragma unroll
  for (int d = 1; d < P; d <<= 1)
#pragma unroll
    for (int t = 0; t + d < P; t += 2 * d) x[t] += x[t + d];
  return x[0];
}

template <int P, bool kWide, int ITEMS>
__global__ __launch_bounds__(kBlock) void edge_score_kernel(EdgeView g, int64_t nnz,
                                                            ScoreArgs args,
                                                            float* __restrict__ out) {
#pragma clang fp contract(off)
  const int64_t e0 = (int64_t)blockIdx.x * (kBlock * ITEMS);
  if (e0 >= nnz) return;
  const SegmentSpan sp = block_edge_span<ITEMS>(g, nnz, 1);
  for (int j = 0; j < ITEMS; ++j) {
    const int64_t e = e0 + j * kBlock + threadIdx.x;
    if (e >= nnz) break;
    int64_t src, dst, eid;
    g.endpoints(sp, e, &src, &dst, &eid);
    float v[GS_SCORE_MAX_TERMS];
#pragma unroll
    for (int k = 0; k < GS_SCORE_MAX_TERMS; ++k) {
      v[k] = 0.f;
      if (k >= args.num_terms) continue;
      const gs_score_term& t = args.term[k];
      const int64_t li = pick(t.lhs_target, src, eid, dst), ri = pick(t.rhs_target, src, eid, dst);
      if (t.kind == GS_SCORE_VALUE) v[k] = t.lhs[eid];
      else if (t.kind == GS_SCORE_QUOTIENT) v[k] = t.lhs[li] / t.rhs[ri];
      else v[k] = products_sum<P, kWide>(t.lhs + li * args.len, t.rhs + ri * args.len, args.len);
      if (args.weights) v[k] *= args.weights[k];
    }
    float s = args.num_terms > 2 ? (v[0] + v[2]) + (v[1] + v[3]) : v[0] + v[1];
    if (args.positive_part) s = s < 0.f ? 0.f : s;  // (NaN stays)
    out[eid] = s + args.shift;
  }
}

// Two SDDMMs (u op v) that share one edge sweep.
template <typename T, int ITEMS>
__global__ __launch_bounds__(kBlock) void fused_u_op_v_kernel(
    EdgeView g, int64_t nnz, int op, const T* __restrict__ lhs1,
    const T* __restrict__ rhs1, T* __restrict__ out1,
    const T* __restrict__ lhs2, const T* __restrict__ rhs2,
    T* __restrict__ out2, int64_t lhs_len, int64_t rhs_len, int64_t out_len,
    int64_t reduce_size, const int64_t* __restrict__ lhs_off,
    const int64_t* __restrict__ rhs_off) {
  const int64_t idx0 = (int64_t)blockIdx.x * (kBlock * ITEMS);
  if (idx0 >= nnz * out_len) return;
  const SegmentSpan sp = block_edge_span<ITEMS>(g, nnz, out_len);
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const int64_t idx = idx0 + j * kBlock + threadIdx.x;
    if (idx >= nnz * out_len) break;
    const int64_t e = idx / out_len, f = idx - e * out_len;
    int64_t src, dst, eid;
    g.endpoints(sp, e, &src, &dst, &eid);
    const int64_t lf = (lhs_off ? lhs_off[f] : f) * reduce_size;
    const int64_t rf = (rhs_off ? rhs_off[f] : f) * reduce_size;
    out1[eid * out_len + f] = apply_op<T>(op, lhs1 + src * lhs_len + lf,
                                          rhs1 + dst * rhs_len + rf, reduce_size);
    out2[eid * out_len + f] = apply_op<T>(op, lhs2 + src * lhs_len + lf,
                                          rhs2 + dst * rhs_len + rf, reduce_size);
  }
}

// ------------------------------------------------------------------- SpMM
// Value an edge contributes: kind 0 = op(u, e), 1 = e * e, 2 = e / u.
template <typename T>
__device__ __forceinline__ T edge_value(int kind, int op, const T* u, const T* e) {
  if (kind == 1) return e[0] * e[0];
  if (kind == 2) return e[0] / u[0];
  return apply_op<T>(op, u, e, 1);
}

__device__ __forceinline__ void atomic_reduce(float* addr, float v, int reduce) {
  if (reduce == kReduceSum) {
    unsafeAtomicAdd(addr, v);
    return;
  }
  unsigned int* p = (unsigned int*)addr;
  unsigned int old = *p;
  for (;;) {
    float cur = __uint_as_float(old);
    bool better = reduce == kReduceMax ? v > cur : v < cur;
    if (!better) return;
    unsigned int prev = atomicCAS(p, old, __float_as_uint(v));
    if (prev == old) return;
    old = prev;
  }
}

// Coordinate form: one thread per (edge, feature), atomics onto the output.
__global__ __launch_bounds__(kBlock) void spmm_coo_kernel(
    const int64_t* __restrict__ row, const int64_t* __restrict__ col,
    const int64_t* __restrict__ edge_map, int64_t nnz, int kind, int op,
    int reduce, const float* __restrict__ ufeat, const float* __restrict__ efeat,
    float* out, int u_target, int64_t ufeat_len, int64_t efeat_len,
    int64_t out_len, const int64_t* __restrict__ u_off,
    const int64_t* __restrict__ e_off) {
  const int64_t idx = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (idx >= nnz * out_len) return;
  const int64_t e = idx / out_len, f = idx - e * out_len;
  const int64_t src = u_target == 0 ? row[e] : col[e];
  const int64_t dst = u_target == 0 ? col[e] : row[e];
  const int64_t eid = edge_map ? edge_map[e] : e;
  const float* u = ufeat ? ufeat + src * ufeat_len + (u_off ? u_off[f] : f) : nullptr;
  const float* ev = efeat ? efeat + eid * efeat_len + (e_off ? e_off[f] : f) : nullptr;
  atomic_reduce(out + dst * out_len + f, edge_value<float>(kind, op, u, ev), reduce);
}

// Second pass of arg-max / arg-min in coordinate form: the edge whose value
// equals the reduced output records its source and edge id.
__global__ __launch_bounds__(kBlock) void spmm_coo_arg_kernel(
    const int64_t* __restrict__ row, const int64_t* __restrict__ col,
    const int64_t* __restrict__ edge_map, int64_t nnz, int op,
    const float* __restrict__ ufeat, const float* __restrict__ efeat,
    const float* __restrict__ out, int64_t* arg_u, int64_t* arg_e, int u_target,
    int64_t ufeat_len, int64_t efeat_len, int64_t out_len,
    const int64_t* __restrict__ u_off, const int64_t* __restrict__ e_off) {
  const int64_t idx = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (idx >= nnz * out_len) return;
  const int64_t e = idx / out_len, f = idx - e * out_len;
  const int64_t src = u_target == 0 ? row[e] : col[e];
  const int64_t dst = u_target == 0 ? col[e] : row[e];
  const int64_t eid = edge_map ? edge_map[e] : e;
  const float* u = ufeat ? ufeat + src * ufeat_len + (u_off ? u_off[f] : f) : nullptr;
  const float* ev = efeat ? efeat + eid * efeat_len + (e_off ? e_off[f] : f) : nullptr;
  if (edge_value<float>(0, op, u, ev) == out[dst * out_len + f]) {
    if (arg_u) arg_u[dst * out_len + f] = src;
    if (arg_e) arg_e[dst * out_len + f] = eid;
  }
}

// Compressed form, scalar features: a group of G lanes per segment strides over
// its edges and reduces with shuffles -- no atomics, hubs spread over a wave.
template <int G>
__global__ __launch_bounds__(kBlock) void spmm_csc_scalar_kernel(
    const int64_t* __restrict__ indptr, const int64_t* __restrict__ indices,
    const int64_t* __restrict__ edge_map, int64_t num_major, int kind, int op,
    int reduce, const float* __restrict__ ufeat, const float* __restrict__ efeat,
    float* __restrict__ out, int64_t* __restrict__ arg_u,
    int64_t* __restrict__ arg_e) {
  const int lane = threadIdx.x & (G - 1);
  const int64_t c = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / G;
  if (c >= num_major) return;
  const int64_t lo = indptr[c], hi = indptr[c + 1];
  // reduction starts from 0: outputs are zero-initialised accumulators
  float acc = 0.f;
  int64_t best_u = 0, best_e = 0;
  for (int64_t i = lo + lane; i < hi; i += G) {
    const int64_t eid = edge_map ? edge_map[i] : i;
    const int64_t cid = indices[i];
    const float v = edge_value<float>(kind, op, ufeat ? ufeat + cid : nullptr,
                                      efeat ? efeat + eid : nullptr);
    if (reduce == kReduceSum) {
      acc += v;
    } else if (reduce == kReduceMax ? v > acc : v < acc) {
      acc = v;
      best_u = cid;
      best_e = eid;
    }
  }
#pragma unroll
  for (int d = G / 2; d > 0; d >>= 1) {
    const float o = __shfl_down(acc, d, G);
    const int64_t ou = __shfl_down(best_u, d, G);
    const int64_t oe = __shfl_down(best_e, d, G);
    if (reduce == kReduceSum) {
      acc += o;
    } else if (reduce == kReduceMax ? o > acc : o < acc) {
      acc = o;
      best_u = ou;
      best_e = oe;
    }
  }
  if (lane == 0) {
    out[c] += acc;
    if (reduce != kReduceSum) {
      if (arg_u) arg_u[c] = best_u;
      if (arg_e) arg_e[c] = best_e;
    }
  }
}

// Compressed form, general feature length: one thread per (segment, feature).
__global__ __launch_bounds__(kBlock) void spmm_csc_kernel(
    const int64_t* __restrict__ indptr, const int64_t* __restrict__ indices,
    const int64_t* __restrict__ edge_map, int64_t num_major, int kind, int op,
    int reduce, const float* __restrict__ ufeat, const float* __restrict__ efeat,
    float* __restrict__ out, int64_t* __restrict__ arg_u,
    int64_t* __restrict__ arg_e, int64_t ufeat_len, int64_t efeat_len,
    int64_t out_len, const int64_t* __restrict__ u_off,
    const int64_t* __restrict__ e_off) {
  const int64_t idx = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (idx >= num_major * out_len) return;
  const int64_t c = idx / out_len, f = idx - c * out_len;
  const int64_t uf = u_off ? u_off[f] : f, ef = e_off ? e_off[f] : f;
  float acc = 0.f;
  int64_t best_u = 0, best_e = 0;
  for (int64_t i = indptr[c]; i < indptr[c + 1]; ++i) {
    const int64_t eid = edge_map ? edge_map[i] : i;
    const int64_t cid = indices[i];
    const float v =
        edge_value<float>(kind, op, ufeat ? ufeat + cid * ufeat_len + uf : nullptr,
                          efeat ? efeat + eid * efeat_len + ef : nullptr);
    if (reduce == kReduceSum) {
      acc += v;
    } else if (reduce == kReduceMax ? v > acc : v < acc) {
      acc = v;
      best_u = cid;
      best_e = eid;
    }
  }
  out[idx] += acc;
  if (reduce != kReduceSum) {
    if (arg_u) arg_u[idx] = best_u;
    if (arg_e) arg_e[idx] = best_e;
  }
}

// ------------------------------------------------- load-balanced scalar sums
// The sums of layer-wise samplers run over slices of power-law graphs: one
// column (or row) can hold a large share of all edges.  Both kernels below are
// edge-parallel, combine inside LDS what a tile of edges adds to the same
// output, and send one atomic per (tile, output) to memory.
constexpr int kSumItems = 8;
constexpr int kSumTile = kBlock * kSumItems;
constexpr int kSumSegs = 2048;   // segments one tile can accumulate in LDS
constexpr int kCooSlots = 4096;  // combining table of the coordinate kernel
constexpr int kDies = 8;         // accelerator dies of an MI355X, one L2 each
constexpr int64_t kPrivateMinEdges = 1 << 20;

// out[i] += sum of the per-die copies; the copies were zero-filled before.
__global__ __launch_bounds__(kBlock) void spmm_fold_kernel(
    const float* __restrict__ copies, int64_t n, float* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  float acc = 0.f;
#pragma unroll
  for (int d = 0; d < kDies; ++d) acc += copies[d * n + i];
  if (acc != 0.f) out[i] += acc;
}

__global__ __launch_bounds__(kBlock) void spmm_zero_kernel(float* p, int64_t n, float value) {
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBlock)
    p[i] = value;
}

// Per-die copies pay off when there are many edges per output row.
static size_t private_bytes(int format, int64_t nnz, int64_t num_out) {
  if (format != GS_FMT_COO || nnz < kPrivateMinEdges || num_out <= 0 ||
      num_out > nnz / 4)
    return 0;
  return (size_t)kDies * (size_t)num_out * sizeof(float);
}

// Sum of v over the wavefront if every lane is active and targets the same
// output (then *uniform is set and lane 0 should add the result).
__device__ __forceinline__ float wave_sum_if_uniform(float v, int64_t target,
                                                     bool active, bool* uniform) {
  const int64_t t0 = wave_uniform_first(target);
  *uniform = __all(active && target == t0);
  if (!*uniform) return v;
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) v += __shfl_down(v, d, kWave);
  return v;
}

// Compressed form: tile of consecutive edges; the segments it touches are
// consecutive, so LDS accumulators are indexed directly.  On large inputs a
// work-group takes kCscRounds tiles in a row: the look-up of the columns it
// covers (two dependent chains of loads over indptr) is then paid once per
// 8192 edges.
constexpr int kCscRounds = 4;

__global__ __launch_bounds__(kBlock) void spmm_csc_sum_kernel(
    const int64_t* __restrict__ indptr, const int64_t* __restrict__ indices,
    const int64_t* __restrict__ edge_map, int64_t num_major, int64_t nnz,
    int kind, int op, const float* __restrict__ ufeat,
    const float* __restrict__ efeat, float* out, int rounds) {
  __shared__ float acc[kSumSegs];
  __shared__ int64_t bounds[kSumSegs + 1];
  const int64_t tile_len = (int64_t)kSumTile * rounds;
  const int64_t tile0 = (int64_t)blockIdx.x * tile_len;
  const int64_t tile_end = tile0 + tile_len < nnz ? tile0 + tile_len : nnz;
  // A lane takes quads of neighbouring edges: item i of a round is edge
  //   base + (i / 4) * 4 * kBlock + 4 * lane + i % 4,
  // so that values which come straight from the edge array arrive as 16-byte loads.
  static_assert(kSumItems % 4 == 0, "a lane takes whole quads");
  auto edge_of = [](int64_t base, int i) {
    return base + (int64_t)(i >> 2) * (4 * kBlock) + 4 * (int)threadIdx.x + (i & 3);
  };
  const bool plain = edge_map == nullptr && ufeat == nullptr && efeat != nullptr;
  auto load_round = [&](int64_t base, float (&val)[kSumItems]) {
#pragma unroll
    for (int q = 0; q < kSumItems / 4; ++q) {
      const int64_t e = edge_of(base, 4 * q);
      if (plain && e + 3 < tile_end) {
        struct Quad {
          float v[4];
        } held;
        __builtin_memcpy(&held, efeat + e, sizeof(Quad));
#pragma unroll
        for (int j = 0; j < 4; ++j)
          val[4 * q + j] = edge_value<float>(kind, op, nullptr, &held.v[j]);
        continue;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        val[4 * q + j] = 0.f;
        if (e + j < tile_end) {
          const int64_t eid = edge_map ? edge_map[e + j] : e + j;
          val[4 * q + j] = edge_value<float>(kind, op, ufeat ? ufeat + indices[e + j] : nullptr,
                                             efeat ? efeat + eid : nullptr);
        }
      }
    }
  };
  // the first round's values before anything else: their loads are in flight
  // while the columns are looked up
  float val[kSumItems];
  load_round(tile0, val);
  // a long column covers the whole tile, and then the second look-up is a single
  // comparison
  const SegmentSpan columns = segment_span(indptr, num_major, tile0, tile_end - 1);
  const int64_t c0 = columns.lo, c1 = columns.hi;
  if (c0 == c1) {
    // the whole tile lies inside one column: no accumulators to clear, one add
    float mine = 0.f;
    for (int r = 0; r < rounds; ++r) {
      if (r > 0) load_round(tile0 + (int64_t)r * kSumTile, val);  // (0 past the tile's end)
      float round_sum = 0.f;
#pragma unroll
      for (int i = 0; i < kSumItems; ++i) round_sum += val[i];
      mine += round_sum;
    }
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) mine += __shfl_down(mine, d, kWave);
    if (lane_id() == 0) acc[threadIdx.x / kWave] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
      float sum = acc[0];
#pragma unroll
      for (int w = 1; w < kBlock / kWave; ++w) sum += acc[w];
      unsafeAtomicAdd(out + c0, sum);
    }
    return;
  }
  const int64_t nseg = c1 - c0 + 1;
  const bool in_lds = nseg <= kSumSegs;
  if (in_lds) {
    for (int64_t j = threadIdx.x; j <= nseg; j += kBlock) {
      bounds[j] = indptr[c0 + j];
      if (j < nseg) acc[j] = 0.f;
    }
    __syncthreads();
  }
  for (int r = 0; r < rounds; ++r) {
    const int64_t base = tile0 + (int64_t)r * kSumTile;
    if (base >= tile_end) break;
    if (r > 0) load_round(base, val);
    // a round that lies inside one column (any column of 2048 edges or more
    // has such rounds): the lanes add their values up first, and the
    // wavefront sends one sum
    const int64_t round_last = base + kSumTile - 1 < tile_end - 1 ? base + kSumTile - 1
                                                                : tile_end - 1;
    const int64_t s_first = in_lds ? segment_of(bounds, nseg, wave_uniform_first(base))
                                   : segment_of(indptr + c0, nseg, wave_uniform_first(base));
    const int64_t s_next = in_lds ? bounds[s_first + 1] : indptr[c0 + s_first + 1];
    if (s_next > round_last) {
      float mine = 0.f;
#pragma unroll
      for (int i = 0; i < kSumItems; ++i) mine += val[i];   // inactive slots hold 0
#pragma unroll
      for (int d = kWave / 2; d > 0; d >>= 1) mine += __shfl_down(mine, d, kWave);
      if (lane_id() == 0) {
        if (in_lds) atomicAdd(&acc[s_first], mine);
        else unsafeAtomicAdd(out + c0 + s_first, mine);
      }
      continue;
    }
#pragma unroll
    for (int i = 0; i < kSumItems; ++i) {
      const int64_t e = edge_of(base, i);
      const bool active = e < tile_end;
      int64_t seg = 0;
      if (active)
        seg = in_lds ? segment_of(bounds, nseg, e) : segment_of(indptr + c0, nseg, e);
      bool uniform;
      const float total = wave_sum_if_uniform(val[i], seg, active, &uniform);
      if (uniform) {
        if (lane_id() == 0) {
          if (in_lds) atomicAdd(&acc[seg], total);
          else unsafeAtomicAdd(out + c0 + seg, total);
        }
      } else if (active) {
        if (in_lds) atomicAdd(&acc[seg], val[i]);
        else unsafeAtomicAdd(out + c0 + seg, val[i]);
      }
    }
  }
  if (!in_lds) return;
  __syncthreads();
  for (int64_t j = threadIdx.x; j < nseg; j += kBlock)
    if (acc[j] != 0.f) unsafeAtomicAdd(out + c0 + j, acc[j]);
}

// ------------------------------------------------------- columns normalised
// The end of a LADIES layer, out[e] = q[e] / (sum of q over e's column) with q[e] =
// values[select[e]] / row_divisor[row[e]], in two passes over the edges: the first writes
// q and adds it up, the second divides.  7.3 M edges in 1024 columns: gather, division,
// sums and division took 40 + 28 + 41 + 23 us, each a launch of its own.
// Sums are of 64 bits, rounded once.
__global__ __launch_bounds__(kBlock) void normalise_clear_kernel(double* sums, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) sums[i] = 0.0;
}

// The columns of a run of edges [first, end) that a wavefront has, each for a team of lanes:
// sixteen where they are few, one where they are many, the wavefront for a long one.
// part(team as an integral_constant, column, where it begins in the run, how many of its edges
// are there); none of a team leaves it before the others.
template <typename Part>
__device__ __forceinline__ void columns_of_run(const int64_t* __restrict__ indptr, SegmentSpan span,
                                               int64_t first, int64_t end, Part part) {
  constexpr int kFew = 16, kTeam = 16;
  const int lane = lane_id();
  const bool few = span.hi - span.lo < kFew;
  const int longest = few ? 16 * kTeam : kWave;  // of the columns that are not the wavefront's
  for (int64_t c0 = span.lo; c0 <= span.hi; c0 += kWave) {
    const int64_t c = c0 + lane <= span.hi ? c0 + lane : span.hi;
    const int64_t s = indptr[c] > first ? indptr[c] : first;
    const int64_t t = indptr[c + 1] < end ? indptr[c + 1] : end;
    const int begin = (int)(s - first), n = c0 + lane <= span.hi && t > s ? (int)(t - s) : 0;
    if (few) {
      for (int c1 = 0; c1 <= span.hi - span.lo; c1 += kWave / kTeam) {
        const int from = __shfl(begin, c1 + lane / kTeam, kWave);
        const int many = __shfl(n, c1 + lane / kTeam, kWave);
        if (many <= longest)
          part(std::integral_constant<int, kTeam>(), c0 + c1 + lane / kTeam, from, many);
      }
    } else if (n <= longest) {
      part(std::integral_constant<int, 1>(), c, begin, n);
    }
    for (uint64_t left = __ballot(n > longest); left; left &= left - 1) {
      const int l = __builtin_ctzll(left);
      part(std::integral_constant<int, kWave>(), c0 + l, __shfl(begin, l, kWave), __shfl(n, l, kWave));
    }
  }
}

// The same edge by edge, for a run most of whose columns are empty: part(column, place in the
// run, whether there is such an edge), by all lanes, for 64 neighbouring edges at a time.  The
// columns of 256 edges are searched for together, a step for twice as many columns, where going
// through the columns takes a step for 64 more of them (with eight rows of 64 in place of four
// the registers leave fewer wavefronts resident).  Sums and division, us, by columns and so:
// 5000 edges of 10 K columns 34 and 36, of 16 K 48 and 32, of 100 K 213 and 42, of 1 M 1634 and
// 69; 1 M edges of 4 M columns 75 and 66.
constexpr int64_t kSparseColumns = 2;  // an edge, from where on
__device__ __forceinline__ bool is_sparse(SegmentSpan span, int64_t edges) {
  return span.hi - span.lo >= kSparseColumns * edges;
}
template <typename Part>
__device__ __forceinline__ void edges_of_run(const int64_t* __restrict__ indptr, SegmentSpan span,
                                             int64_t first, int64_t end, Part part) {
  constexpr int kRows = 4;
  const int n = (int)(end - first);
  const int64_t most = span.hi - span.lo;
  const int64_t* const begins = indptr + span.lo;
  for (int i0 = 0; i0 < n; i0 += kRows * kWave) {
    int64_t e[kRows], c[kRows];  // c: the last column known to begin at or before the edge
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      const int at = i0 + j * kWave + lane_id();
      e[j] = first + (at < n ? at : n - 1);
      c[j] = 0;
    }
    for (int64_t step = int64_t(1) << (63 - __builtin_clzll((uint64_t)most)); step > 0; step >>= 1) {
      int64_t begin[kRows];
#pragma unroll
      for (int j = 0; j < kRows; ++j) begin[j] = begins[c[j] + step <= most ? c[j] + step : most];
#pragma unroll
      for (int j = 0; j < kRows; ++j)
        if (c[j] + step <= most && begin[j] <= e[j]) c[j] += step;
    }
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      const int at = i0 + j * kWave + lane_id();
      part(span.lo + c[j], at, at < n);
    }
  }
}

// A wavefront adds up a run of kItems * 64 edges.  The look-up of its columns (two or three
// loads, one behind the other) is on its way with the values; where columns meet the run goes
// to LDS and is read back column by column, the short ones a lane each.  What bounds it is the
// adds to one sum, 30 ns each: a column of a power law's hub has a sixth of all edges, and with
// an add for every 2048 edges of it 7.1 M edges of 512 columns (28 MB) took 32 us.  So the
// wavefronts of a work-group that are inside one column add once: 13 us.  37 K edges of as many
// columns: 9.8 and 5.8 us, 10.7 with every column the whole wavefront's.
// kItems: eight, which is 4.2 million edges in the work-groups that are resident together (four
// a compute unit), or 32 beyond that.  Values that are gathered or divided on the way always go
// by eight (the indexes of 32 would be 128 registers).
constexpr int kRunItems = 8, kLongRunItems = 32;
constexpr int64_t kLongRuns = int64_t(1) << 22;
constexpr int kRunThreads = 512;
template <bool kSelect, bool kDivide, int kItems>
__global__ __launch_bounds__(kRunThreads) void normalise_sum_kernel(
    const int64_t* __restrict__ indptr, int64_t num_cols, const int64_t* __restrict__ rows,
    int64_t nnz, const float* __restrict__ values, int64_t num_values,
    const int64_t* __restrict__ select, const float* __restrict__ row_divisor,
    double* __restrict__ sums, float* __restrict__ out) {
  constexpr int kWaves = kRunThreads / kWave;
  __shared__ float held[kWaves][kItems * kWave];
  __shared__ double wave_sum[kWaves];
  __shared__ int64_t wave_column[kWaves];  // -1: there is no such sum
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  float* const run = held[wave];
  if (lane == 0) wave_column[wave] = -1;
  const int64_t first =
      wave_uniform_first(((int64_t)blockIdx.x * kWaves + wave) * (kItems * kWave));
  if (first < nnz) {
    const int64_t end = first + kItems * kWave < nnz ? first + kItems * kWave : nnz;
    float v[kItems];
    if (kSelect || kDivide) {
      int64_t at[kItems], row[kItems];
#pragma unroll
      for (int i = 0; i < kItems; ++i) {
        const int64_t e0 = first + i * kWave + lane, e = e0 < end ? e0 : end - 1;
        at[i] = kSelect ? select[e] : e;
        row[i] = kDivide ? rows[e] : 0;
      }
#pragma unroll
      for (int i = 0; i < kItems; ++i)
        v[i] = values[!kSelect || (uint64_t)at[i] < (uint64_t)num_values ? at[i] : 0];
      if (kSelect) {  // (edge data may be shorter than the edges that `select` names)
#pragma unroll
        for (int i = 0; i < kItems; ++i)
          if ((uint64_t)at[i] >= (uint64_t)num_values) v[i] = 0.f;
      }
      if (kDivide) {
#pragma unroll
        for (int i = 0; i < kItems; ++i) v[i] /= row_divisor[row[i]];
      }
    } else if (end - first == kItems * kWave) {
      const float* const from = values + first;
#pragma unroll
      for (int i = 0; i < kItems; ++i) v[i] = from[i * kWave + lane];
    } else {
#pragma unroll
      for (int i = 0; i < kItems; ++i) {
        const int64_t e = first + i * kWave + lane;
        v[i] = values[e < end ? e : end - 1];
      }
    }
    const SegmentSpan span = segment_span(indptr, num_cols, first, end - 1);
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      const int64_t e = first + i * kWave + lane;
      if (e < end) {
        if (kSelect || kDivide) out[e] = v[i];
      } else {
        v[i] = 0.f;
      }
    }
    if (span.lo == span.hi) {
      double mine = 0.0;
#pragma unroll
      for (int i = 0; i < kItems; ++i) mine += (double)v[i];
#pragma unroll
      for (int d = kWave / 2; d > 0; d >>= 1) mine += __shfl_down(mine, d, kWave);
      if (lane == 0) {
        wave_sum[wave] = mine;
        wave_column[wave] = span.lo;
      }
    } else {
#pragma unroll
      for (int i = 0; i < kItems; ++i) run[i * kWave + lane] = v[i];
      wave_lds_fence();
      if (is_sparse(span, end - first))
        edges_of_run(indptr, span, first, end, [&](int64_t c, int at, bool live) {
          // (each column's edges in these 64 are neighbours: their sum at the first of them)
          double mine = live ? (double)run[at] : 0.0;
          for (int d = 1; d < kWave; d <<= 1) {
            const double other = __shfl_down(mine, d, kWave);
            if ((int64_t)__shfl_down((long long)c, d, kWave) == c && lane + d < kWave) mine += other;
          }
          const bool begins = (int64_t)__shfl_up((long long)c, 1, kWave) != c || lane == 0;
          if (live && begins) unsafeAtomicAdd(sums + c, mine);
        });
      else columns_of_run(indptr, span, first, end, [&](auto team, int64_t c, int begin, int n) {
        constexpr int kTeam = decltype(team)::value;
        double mine = 0.0;
        for (int i = lane % kTeam; i < n; i += kTeam) mine += (double)run[begin + i];
#pragma unroll
        for (int d = kTeam / 2; d > 0; d >>= 1) mine += __shfl_down(mine, d, kTeam);
        if (lane % kTeam == 0 && n > 0) unsafeAtomicAdd(sums + c, mine);
      });
    }
  }
  __syncthreads();
  if (threadIdx.x >= kWaves) return;
  const int64_t c = wave_column[threadIdx.x];
  if (c < 0 || (threadIdx.x > 0 && wave_column[threadIdx.x - 1] == c)) return;
  double sum = wave_sum[threadIdx.x];
  for (int w = threadIdx.x + 1; w < kWaves && wave_column[w] == c; ++w) sum += wave_sum[w];
  unsafeAtomicAdd(sums + c, sum);
}

// group: so many tiles in a row were one work-group's of the sums, whose die has their values
// (7.1 M edges: 17.2 us with the dies' tiles in turn, 15.4 so).  A wavefront for itself, as above,
// and where columns meet their sums go to the places of their edges in LDS (work-groups that
// of 2048 edges that searched a column for each took 15.4 and 7.8 us on 7.1 M and 37 K edges of
// 512 columns, 22.8 on two layers of 8 batches; this 12.9, 5.0 and 14.6).
__global__ __launch_bounds__(kRunThreads) void normalise_divide_kernel(
    const int64_t* __restrict__ indptr, int64_t num_cols, int64_t nnz,
    const double* __restrict__ sums, const float* values, float* out, unsigned group) {
  constexpr int kWaves = kRunThreads / kWave;
  __shared__ float divisors[kWaves][kRunItems * kWave];
  const unsigned nth = blockIdx.x / kDies;  // of its die
  const int64_t tile = (int64_t)(nth / group * kDies + blockIdx.x % kDies) * group + nth % group;
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int64_t first = wave_uniform_first((tile * kWaves + wave) * (kRunItems * kWave));
  if (first >= nnz) return;
  const int64_t end = first + kRunItems * kWave < nnz ? first + kRunItems * kWave : nnz;
  float v[kRunItems], by[kRunItems];
#pragma unroll
  for (int i = 0; i < kRunItems; ++i) {
    const int64_t e = first + i * kWave + lane;
    v[i] = values[e < end ? e : end - 1];
  }
  const SegmentSpan span = segment_span(indptr, num_cols, first, end - 1);
  if (span.lo == span.hi) {
    const float s = (float)sums[span.lo];
#pragma unroll
    for (int i = 0; i < kRunItems; ++i) by[i] = s;
  } else {
    float* const run = divisors[wave];
    if (is_sparse(span, end - first))
      edges_of_run(indptr, span, first, end, [&](int64_t c, int at, bool live) {
        if (live) run[at] = (float)sums[c];
      });
    else columns_of_run(indptr, span, first, end, [&](auto team, int64_t c, int begin, int n) {
      constexpr int kTeam = decltype(team)::value;
      const float s = n > 0 ? (float)sums[c] : 0.f;
      for (int i = lane % kTeam; i < n; i += kTeam) run[begin + i] = s;
    });
    wave_lds_fence();
#pragma unroll
    for (int i = 0; i < kRunItems; ++i) by[i] = run[i * kWave + lane];
  }
#pragma unroll
  for (int i = 0; i < kRunItems; ++i) {
    const int64_t e = first + i * kWave + lane;
    if (e < end) out[e] = v[i] / by[i];
  }
}

// Coordinate form: outputs arrive in any order, so the tile combines them in
// a small LDS hash table; an edge that finds no slot within a few probes adds
// to memory directly.  What bounds it is the atomics, one per tile and row present:
// tiles of 512 edges, for four times the work-groups on a short list, took 74 us on
// 150 thousand edges of which a hub row draws many, where tiles of 2048 take 42.
__global__ __launch_bounds__(kBlock) void spmm_coo_sum_kernel(
    const int64_t* __restrict__ row, const int64_t* __restrict__ col,
    const int64_t* __restrict__ edge_map, int64_t nnz, int kind, int op,
    const float* __restrict__ ufeat, const float* __restrict__ efeat, float* out,
    int u_target, int64_t copy_stride, SliceView view) {
  __shared__ long long keys[kCooSlots];
  __shared__ float vals[kCooSlots];
  for (int j = threadIdx.x; j < kCooSlots; j += kBlock) {
    keys[j] = -1;
    vals[j] = 0.f;
  }
  __syncthreads();
  // consecutive work-groups run on consecutive dies: with copy_stride > 0 every
  // die adds to a copy of its own
  out += (int64_t)(blockIdx.x % kDies) * copy_stride;
  const int64_t tile0 = (int64_t)blockIdx.x * kSumTile;
  const int64_t* dst_ids = u_target == 0 ? col : row;
  const int64_t* src_ids = u_target == 0 ? row : col;
  // all loads of the tile first, so that they are in flight together
  // (with a view: the edges of a column slice that was never written, dst_ids
  // and efeat being the parent's arrays)
  SliceView::Run vrun{};
  vrun.split = INT64_MAX;  // no view: every edge at distance 0
  if (view.on() && tile0 < nnz)
    vrun = view.run(tile0, (tile0 + kSumTile < nnz ? tile0 + kSumTile : nnz) - 1);
  int64_t dst[kSumItems];
  float val[kSumItems];
#pragma unroll
  for (int i = 0; i < kSumItems; ++i) {
    const int64_t e = tile0 + i * kBlock + threadIdx.x;
    dst[i] = -1;
    val[i] = 0.f;
    if (e < nnz && vrun.near()) {
      const int64_t p = vrun.place(e);
      dst[i] = dst_ids[p] + vrun.id_offset(e);
      const int64_t eid = edge_map ? edge_map[p] : p;
      val[i] = edge_value<float>(kind, op, ufeat ? ufeat + src_ids[p] : nullptr,
                                 efeat ? efeat + eid : nullptr);
    }
  }
  if (!vrun.near()) {
#pragma unroll
    for (int i = 0; i < kSumItems; ++i) {
      const int64_t e = tile0 + i * kBlock + threadIdx.x;
      int64_t col, offset;  // (looked up by all lanes together, a lane past the end included)
      const int64_t row = wave_uniform_first(e) < nnz ? wave_uniform_first(e) : nnz - 1;
      const int64_t p = view.row_position(vrun, row, e < nnz ? e : nnz - 1, &col, &offset);
      if (e < nnz) {
        dst[i] = dst_ids[p] + offset;
        val[i] = edge_value<float>(kind, op, ufeat ? ufeat + src_ids[p] : nullptr,
                                   efeat ? efeat + (edge_map ? edge_map[p] : p) : nullptr);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < kSumItems; ++i) {
    if (dst[i] < 0) continue;
    uint32_t slot =
        (uint32_t)(((uint64_t)dst[i] * 0x9E3779B97F4A7C15ull) >> 40) & (kCooSlots - 1);
    bool placed = false;
    for (int probe = 0; probe < 8 && !placed; ++probe) {
      long long k = keys[slot];
      if (k == -1) k = (long long)atomicCAS((unsigned long long*)&keys[slot],
                                            ~0ull, (unsigned long long)dst[i]);
      if (k == -1 || k == (long long)dst[i]) {
        atomicAdd(&vals[slot], val[i]);
        placed = true;
      }
      slot = (slot + 1) & (kCooSlots - 1);
    }
    if (!placed) unsafeAtomicAdd(out + dst[i], val[i]);
  }
  __syncthreads();
  for (int j = threadIdx.x; j < kCooSlots; j += kBlock)
    if (keys[j] != -1) unsafeAtomicAdd(out + keys[j], vals[j]);
}

static int coo_sum_launch(const int64_t* row, const int64_t* col, const int64_t* edge_map,
                          int64_t nnz, int kind, int op, const float* ufeat, const float* efeat,
                          float* out, int u_target, SliceView view, hipStream_t s) {
  GS_LAUNCH("spmm_coo_sum", s,
            spmm_coo_sum_kernel<<<dim3((unsigned)ceil_div(nnz, (int64_t)kSumTile)), dim3(kBlock), 0,
                                  s>>>(row, col, edge_map, nnz, kind, op, ufeat, efeat, out,
                                       u_target, (int64_t)0, view));
  return GS_OK;
}

// ------------------------------------------- coordinate sums by row ranges
// Atomic adds to device memory are executed next to the memory, at a rate far
// below what the edges stream at, and a tile of a large slice rarely adds
// twice to the same row.  Large coordinate-form sums therefore go through a
// partition by row range: (1) a work-group sorts a tile of 8192 edges by range in
// LDS and writes (row within range, value) to the tile's own place, 6 bytes an
// edge, with the start and length of every range's run in a table of (range, tile)
// cells, (2) a work-group per range cuts the tiles into units of about 32 Ki of
// its entries, (3) a work-group sums a unit in LDS and stores kRangeRows partial
// sums, (4) the partial sums of a range are folded into the output.  The edges are
// read once, nothing is counted beforehand, and no pass uses an atomic on device
// memory.  The floor is 8 + 6 bytes an edge through pass 1 and
// 6 + the rate of fp64 adds in LDS through pass 3.  On a slice of 29 M edges and
// 233 K rows a counting pass, a scan, and a scatter of 8-byte pairs to places
// chosen by the scan took 353 us, with the sums; this takes 190 (part 106, sums 64, fold 10).
constexpr int kRangeShift = 13;
constexpr int kRangeRows = 1 << kRangeShift;  // 64 KB of LDS accumulators
constexpr int kMaxRanges = 1024;
constexpr int kPartThreads = 512;
constexpr int kPartItems = 16;
constexpr int kPartTile = kPartThreads * kPartItems;
constexpr int kPartWaveRun = kPartItems * kWave;  // consecutive edges of a wavefront
// Counters of the sort: a range has up to 32 of them, chosen by lane, because most
// lanes of a wave meet at the range that holds the hubs' rows and adds to one LDS
// word are taken one after another.
constexpr int kPartCounters = kMaxRanges;
constexpr int kPartMaxCopyBits = 5;
constexpr int kUnitEntries = 32768;  // entries one work-group sums, to within a tile
// The accumulators of a range take 64 KB of LDS, so two work-groups share a
// compute unit: 1024 threads each keep all its wavefront slots busy.
constexpr int kAccThreads = 1024;
constexpr int kUnitsThreads = 1024;
static_assert(kPartTile < (1 << 16) && kRangeRows <= (1 << 16), "16-bit rows, starts and lengths");
static_assert(kPartTile < kUnitEntries, "every unit begins at a tile of its own");

struct RowUnit {
  int32_t range, tile0, tile1, unused;
};
struct RangeUnits {
  int32_t base, count;
};

struct RowRangePlan {
  int64_t ranges = 0, tiles = 0, tile_stride = 0, max_units = 0;
  int copy_bits = 0;
  size_t off_cells = 0, off_rows = 0, off_values = 0, off_units = 0, off_range_units = 0,
         off_total = 0, off_partial = 0, total = 0;
};

// Worth it when the slice is large and rows repeat; empty plan otherwise.
static RowRangePlan row_range_plan(int format, int64_t nnz, int64_t num_out) {
  RowRangePlan p;
  if (format != GS_FMT_COO || nnz < kPrivateMinEdges ||
      nnz >= ((int64_t)1 << 31) || num_out <= 0 || num_out > nnz / 4 ||
      ceil_div(num_out, kRangeRows) > kMaxRanges)
    return p;
  p.ranges = ceil_div(num_out, kRangeRows);
  while (p.copy_bits < kPartMaxCopyBits && (p.ranges << (p.copy_bits + 1)) <= kPartCounters)
    ++p.copy_bits;
  p.tiles = ceil_div(nnz, (int64_t)kPartTile);
  p.tile_stride = (p.tiles + 7) / 8 * 8;
  p.max_units = nnz / kUnitEntries + p.ranges;
  auto take = [&p](size_t bytes) {
    const size_t at = p.total;
    p.total += (bytes + 255) / 256 * 256;
    return at;
  };
  p.off_cells = take((size_t)(p.ranges * p.tile_stride) * sizeof(uint32_t));
  p.off_rows = take((size_t)(p.tiles * kPartTile) * sizeof(uint16_t));
  p.off_values = take((size_t)(p.tiles * kPartTile) * sizeof(float));
  p.off_units = take((size_t)p.max_units * sizeof(RowUnit));
  p.off_range_units = take((size_t)p.ranges * sizeof(RangeUnits));
  p.off_total = take(sizeof(int));
  p.off_partial = take((size_t)p.max_units * kRangeRows * sizeof(float));
  return p;
}

// cells[range * tile_stride + tile] = first entry of the run inside the tile, and its
// length in the upper half.
__device__ __forceinline__ uint32_t run_cell(uint32_t start, uint32_t length) {
  return start | (length << 16);
}

// With a view the edges are those of a column slice that was never written:
// dst_ids and efeat are then the parent's arrays (see SliceView).  A wavefront
// takes consecutive edges, so it looks up the few columns of its own run only.
// kKeys: the view moves its columns' ids (keys below 2^31).
template <typename IdT, bool kKeys>
__global__ __launch_bounds__(kPartThreads, 6) void rowsum_part_kernel(
    const IdT* __restrict__ dst_ids, const int64_t* __restrict__ src_ids,
    const int64_t* __restrict__ edge_map, int64_t nnz, int64_t num_out, int kind,
    int op, const float* __restrict__ ufeat, const float* __restrict__ efeat,
    int ranges, int copy_bits, int64_t tile_stride, uint32_t* __restrict__ cells,
    uint16_t* __restrict__ rows, float* __restrict__ values, int* __restrict__ unit_total,
    SliceView view) {
  __shared__ uint32_t count[kPartCounters + 1];
  __shared__ uint32_t wave_total[kPartThreads / kWave];
  __shared__ __align__(16) uint16_t lds_row[kPartTile];
  __shared__ __align__(16) float lds_val[kPartTile];
  const int t = threadIdx.x, lane = lane_id();
  const int counters = ranges << copy_bits;
  if (blockIdx.x == 0 && t == 0) *unit_total = 0;  // counted up by the next kernel
  for (int j = t; j < kPartCounters + 1; j += kPartThreads) count[j] = 0;

  // 1. all loads of the run, so that they are in flight together
  const int64_t first = (int64_t)blockIdx.x * kPartTile + (int64_t)(t / kWave) * kPartWaveRun;
  int row[kPartItems];
  float val[kPartItems];
#pragma unroll
  for (int i = 0; i < kPartItems; ++i) {
    row[i] = -1;
    val[i] = 0.f;
  }
  if (first < nnz) {  // whole wavefronts
    SliceView::Run vrun{};
    vrun.split = INT64_MAX;  // no view: every edge at distance 0
    if (view.on())
      vrun = view.run(first, (first + kPartWaveRun < nnz ? first + kPartWaveRun : nnz) - 1);
    const bool shifted = vrun.near();  // the same in every lane
    auto take = [&](int i, int64_t p, int64_t offset) {
      const int64_t dst = (int64_t)dst_ids[p] + (kKeys ? offset : 0);
      const int64_t eid = edge_map ? edge_map[p] : p;
      val[i] = edge_value<float>(kind, op, ufeat ? ufeat + src_ids[p] : nullptr,
                                 efeat ? efeat + eid : nullptr);
      row[i] = dst >= 0 && dst < num_out ? (int)dst : -1;
    };
    if (shifted && edge_map == nullptr && ufeat == nullptr && efeat != nullptr) {
      // no branch between the loads, or each would be waited for inside its own
      IdT id[kPartItems];
#pragma unroll
      for (int i = 0; i < kPartItems; ++i) {
        const int64_t e = first + i * kWave + lane;
        const int64_t p = vrun.place(e < nnz ? e : nnz - 1);
        id[i] = dst_ids[p];
        val[i] = efeat[p];
      }
#pragma unroll
      for (int i = 0; i < kPartItems; ++i) {
        const int64_t e = first + i * kWave + lane;
        const int64_t dst = (int64_t)id[i] +
                            (kKeys ? (e < vrun.split ? (int)vrun.offset[0] : (int)vrun.offset[1]) : 0);
        row[i] = first + i * kWave + lane < nnz && dst >= 0 && dst < num_out ? (int)dst : -1;
        val[i] = edge_value<float>(kind, op, nullptr, &val[i]);
      }
    } else if (shifted) {
#pragma unroll
      for (int i = 0; i < kPartItems; ++i) {
        const int64_t e = first + i * kWave + lane;
        if (e < nnz) take(i, vrun.place(e), vrun.id_offset(e));
      }
    } else {
#pragma unroll
      for (int i = 0; i < kPartItems; ++i) {
        const int64_t e = first + i * kWave + lane;
        int64_t col, offset;  // (looked up by all lanes together, a lane past the end included)
        const int64_t row = first + i * kWave < nnz ? first + i * kWave : nnz - 1;
        const int64_t p = view.row_position(vrun, row, e < nnz ? e : nnz - 1, &col, &offset);
        if (e < nnz) take(i, p, offset);
      }
    }
  }
  __syncthreads();

  // 2. an edge's place among those of its counter
  const int copy = lane & ((1 << copy_bits) - 1);
  uint32_t place[kPartItems];
#pragma unroll
  for (int i = 0; i < kPartItems; ++i)
    place[i] = row[i] >= 0
                   ? atomicAdd(&count[((row[i] >> kRangeShift) << copy_bits) + copy], 1u)
                   : 0u;
  __syncthreads();

  // 3. counts -> first places (two counters per thread; the last word becomes the total)
  static_assert(kPartCounters == 2 * kPartThreads, "two counters per thread");
  const uint32_t c0 = count[2 * t], c1 = count[2 * t + 1];
  uint32_t incl = c0 + c1;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t o = __shfl_up(incl, d, kWave);
    if (lane >= d) incl += o;
  }
  if (lane == kWave - 1) wave_total[t / kWave] = incl;
  __syncthreads();
  uint32_t before = incl - (c0 + c1);
  for (int w = 0; w < t / kWave; ++w) before += wave_total[w];
  count[2 * t] = before;
  count[2 * t + 1] = before + c0;
  if (t == kPartThreads - 1) count[kPartCounters] = before + c0 + c1;
  __syncthreads();

  // 4. sorted in LDS, the runs' cells, and the tile written in order
#pragma unroll
  for (int i = 0; i < kPartItems; ++i) {
    if (row[i] < 0) continue;
    const uint32_t at = count[((row[i] >> kRangeShift) << copy_bits) + copy] + place[i];
    lds_row[at] = (uint16_t)(row[i] & (kRangeRows - 1));
    lds_val[at] = val[i];
  }
  for (int r = t; r < ranges; r += kPartThreads) {
    const uint32_t start = count[r << copy_bits];
    cells[(int64_t)r * tile_stride + blockIdx.x] =
        run_cell(start, count[(r + 1) << copy_bits] - start);
  }
  const uint32_t total = count[counters];
  __syncthreads();
  // places past the total hold what LDS held before; no cell covers them
  uint4* to_rows = reinterpret_cast<uint4*>(rows + (int64_t)blockIdx.x * kPartTile);
  float4* to_values = reinterpret_cast<float4*>(values + (int64_t)blockIdx.x * kPartTile);
  const uint4* from_rows = reinterpret_cast<const uint4*>(lds_row);
  const float4* from_values = reinterpret_cast<const float4*>(lds_val);
#pragma unroll
  for (int i = 0; i < kPartItems / 8; ++i)
    if ((uint32_t)(i * kPartThreads + t) * 8u < total)
      to_rows[i * kPartThreads + t] = from_rows[i * kPartThreads + t];
#pragma unroll
  for (int i = 0; i < kPartItems / 4; ++i)
    if ((uint32_t)(i * kPartThreads + t) * 4u < total)
      to_values[i * kPartThreads + t] = from_values[i * kPartThreads + t];
}

// A work-group per range: unit k of the range is the tiles whose last entry is
// between k and k + 1 times kUnitEntries entries into the range.  No unit is left
// out, since a tile holds fewer entries than a unit; tiles in front of the range's
// first entry and behind its last belong to none.
__global__ __launch_bounds__(kUnitsThreads) void rowsum_units_kernel(
    const uint32_t* __restrict__ cells, int64_t tiles, int64_t tile_stride, int* unit_total,
    RangeUnits* __restrict__ range_units, RowUnit* __restrict__ units) {
  constexpr int kPer = 8;
  __shared__ int64_t smem[kUnitsThreads / kWave + 1];
  __shared__ int base_of_range;
  const int r = blockIdx.x, t = threadIdx.x;
  const uint32_t* mine = cells + (int64_t)r * tile_stride;
  auto load = [&](int64_t i0, uint32_t (&c)[kPer]) {
#pragma unroll
    for (int j = 0; j < kPer; ++j) c[j] = i0 + j < tiles ? mine[i0 + j] >> 16 : 0u;
  };
  // entries of the range
  int64_t carry = 0;
  for (int64_t b = 0; b < tiles; b += kUnitsThreads * kPer) {
    uint32_t c[kPer];
    load(b + (int64_t)t * kPer, c);
    int64_t sum = 0, total;
#pragma unroll
    for (int j = 0; j < kPer; ++j) sum += c[j];
    block_exclusive_sum<int64_t, kUnitsThreads>(sum, smem, &total);
    carry += total;
    __syncthreads();
  }
  if (t == 0) {
    const int n = carry > 0 ? (int)((carry - 1) / kUnitEntries) + 1 : 0;
    base_of_range = n > 0 ? atomicAdd(unit_total, n) : 0;
    range_units[r] = RangeUnits{base_of_range, n};
  }
  __syncthreads();
  if (carry == 0) return;
  const int base = base_of_range;
  int64_t run0 = 0;
  for (int64_t b = 0; b < tiles; b += kUnitsThreads * kPer) {
    uint32_t c[kPer];
    const int64_t i0 = b + (int64_t)t * kPer;
    load(i0, c);
    int64_t sum = 0, total;
#pragma unroll
    for (int j = 0; j < kPer; ++j) sum += c[j];
    int64_t run = run0 + block_exclusive_sum<int64_t, kUnitsThreads>(sum, smem, &total);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      if (c[j] == 0) continue;
      const int64_t k = (run + c[j] - 1) / kUnitEntries;
      if (run == 0 || (run - 1) / kUnitEntries != k) {
        units[base + k].range = r;
        units[base + k].tile0 = (int32_t)(i0 + j);
        if (k > 0) units[base + k - 1].tile1 = (int32_t)(i0 + j);
      }
      run += c[j];
      if (run == carry) units[base + k].tile1 = (int32_t)(i0 + j + 1);
    }
    run0 += total;
    __syncthreads();
  }
}

// The runs of a unit are cut into chunks of one entry a lane, listed in LDS; a
// wavefront takes eight chunks at a time.  (A range without hubs has about a
// hundred entries a tile: chunks of 256 left half of the lanes idle.)
constexpr int kAccChunk = kWave;
constexpr int kAccAhead = 8;
constexpr int kAccTiles = kAccThreads;  // tiles listed at a time
constexpr int kAccMaxChunks = (kUnitEntries + kPartTile) / kAccChunk + kAccTiles;

__global__ __launch_bounds__(kAccThreads, 8) void rowsum_accumulate_kernel(
    const uint16_t* __restrict__ rows, const float* __restrict__ values,
    const uint32_t* __restrict__ cells, int64_t tile_stride, const RowUnit* __restrict__ units,
    const int* __restrict__ unit_total, float* __restrict__ partial) {
  // (they begin at -0, which only additions move: a row of no entry stays -0, a row
  // whose entries are zeros becomes +0)
  // Accumulators in double: this part adds doubles in LDS at twice the rate of
  // floats (602 M entries: 1.55 against 3.05 ms), and a slice's sums then carry
  // no rounding of their own before they are rounded to float once.
  __shared__ double acc[kRangeRows];
  __shared__ uint2 chunks[kAccMaxChunks];  // tile; start inside it and length
  __shared__ uint32_t smem[kAccThreads / kWave + 1];
  const int t = threadIdx.x, lane = lane_id(), wave = t / kWave;
  const int64_t u = blockIdx.x;
  if (u >= *unit_total) return;
  const RowUnit unit = units[u];
  for (int j = t; j < kRangeRows; j += kAccThreads) acc[j] = -0.0;
  for (int tile0 = unit.tile0; tile0 < unit.tile1; tile0 += kAccTiles) {
    const int tile = tile0 + t;
    uint32_t start = 0, length = 0;
    if (tile < unit.tile1) {
      const uint32_t cell = cells[(int64_t)unit.range * tile_stride + tile];
      start = cell & 0xFFFFu;
      length = cell >> 16;
    }
    const uint32_t n = (length + kAccChunk - 1) / kAccChunk;
    uint32_t num_chunks;
    uint32_t at = block_exclusive_sum<uint32_t, kAccThreads>(n, smem, &num_chunks);
    for (uint32_t k = 0; k < n; ++k) {
      const uint32_t left = length - k * kAccChunk;
      chunks[at + k] = make_uint2((uint32_t)tile, (start + k * kAccChunk) |
                                                      ((left < kAccChunk ? left : kAccChunk) << 16));
    }
    __syncthreads();
    for (uint32_t c0 = (uint32_t)wave * kAccAhead; c0 < num_chunks;
         c0 += kAccAhead * (kAccThreads / kWave)) {
      int row[kAccAhead];
      float val[kAccAhead];
      bool live[kAccAhead];
#pragma unroll
      for (int i = 0; i < kAccAhead; ++i) {
        const uint32_t c = c0 + i;
        const uint2 d = chunks[c < num_chunks ? c : num_chunks - 1];
        const int len = (int)(d.y >> 16);  // at least one
        const int64_t at = (int64_t)d.x * kPartTile + (d.y & 0xFFFFu) + (lane < len ? lane : len - 1);
        live[i] = c < num_chunks && lane < len;
        row[i] = (int)rows[at];
        val[i] = values[at];
      }
#pragma unroll
      for (int i = 0; i < kAccAhead; ++i) {
        // one row for the whole wavefront (a sum over sorted targets): adds to one
        // word would be taken one after another
        const int row0 = __builtin_amdgcn_readfirstlane(row[i]);
        if (__all(live[i] && row[i] == row0)) {
          double sum = (double)val[i];
#pragma unroll
          for (int d = kWave / 2; d > 0; d >>= 1) sum += __shfl_down(sum, d, kWave);
          if (lane == 0) atomicAdd(&acc[row0], sum);
        } else if (live[i]) {
          atomicAdd(&acc[row[i]], (double)val[i]);
        }
      }
    }
    __syncthreads();
  }
  float* mine = partial + u * kRangeRows;
  for (int j = t; j < kRangeRows; j += kAccThreads) mine[j] = (float)acc[j];
}

// out[row] += the row's partial sums over all units of its range.  Ranges
// differ a lot in how many units they have (the rows of hubs sit in one range
// and draw half of the edges), so a work-group takes 128 rows, four a lane, and its
// eight groups of 32 lanes a share of the units each: a range of 500 units is 63
// loads deep.  The shares are added in double and the row is rounded once.  (A
// work-group per share whose shares met in eight float atomics a row took 11.7 us on
// 233 K rows with 32 units a range and 22 on 1.67 M rows with four; this takes
// 9.9 and 13.)
constexpr int kFoldLanes = 32;
constexpr int kFoldRows = 4 * kFoldLanes;
constexpr int kFoldShares = kBlock / kFoldLanes;
static_assert(kRangeRows % kFoldRows == 0, "the rows of a work-group share a range");

// range_units: null when every range has `parts` units, one range after the other.
// onto.fresh: `out` need not have been cleared (a launch of 2 to 4 us and the way to it).
__global__ __launch_bounds__(kBlock) void rowsum_fold_kernel(
    const float* __restrict__ partial, const RangeUnits* __restrict__ range_units, int parts,
    int64_t num_out, float* __restrict__ out, SumsOnto onto) {
  __shared__ double share_sum[kFoldShares][kFoldRows];
  const int share = threadIdx.x / kFoldLanes, lane_row = threadIdx.x % kFoldLanes * 4;
  const int64_t row0 = (int64_t)blockIdx.x * kFoldRows;
  const int range = (int)(row0 >> kRangeShift);
  const RangeUnits ru = range_units ? range_units[range] : RangeUnits{range * parts, parts};
  const int64_t u1 = (int64_t)ru.base + ru.count;
  // (a unit has the sums of all rows of its range, also of those past num_out)
  const float* p = partial + (row0 & (kRangeRows - 1)) + lane_row;
  auto sums_of = [&](int64_t u) { return *reinterpret_cast<const float4*>(p + u * kRangeRows); };
  double acc[4] = {-0.0, -0.0, -0.0, -0.0};
  auto add = [&](const float4& v) {
    acc[0] += (double)v.x;
    acc[1] += (double)v.y;
    acc[2] += (double)v.z;
    acc[3] += (double)v.w;
  };
  int64_t u = (int64_t)ru.base + share;
  for (; u + 7 * kFoldShares < u1; u += 8 * kFoldShares) {  // eight loads in flight
    float4 v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = sums_of(u + k * kFoldShares);
#pragma unroll
    for (int k = 0; k < 8; ++k) add(v[k]);
  }
  for (; u < u1; u += kFoldShares) add(sums_of(u));
#pragma unroll
  for (int k = 0; k < 4; ++k) share_sum[share][lane_row + k] = acc[k];
  __syncthreads();
  const int64_t i = row0 + threadIdx.x;
  if (threadIdx.x >= kFoldRows || i >= num_out) return;
  double sum = -0.0;
#pragma unroll
  for (int s = 0; s < kFoldShares; ++s) sum += share_sum[s][threadIdx.x];
  const bool any = __double_as_longlong(sum) != INT64_MIN;  // (the bits of -0)
  if (onto.fresh) out[i] = any ? onto.base + (float)sum : onto.base;
  else if (any) out[i] += (float)sum;
}

// dst_ids32: the same ids as dst_ids in 32 bits (a matrix's narrow copy), read
// instead when given.
static int row_range_sum(const RowRangePlan& p, const int64_t* dst_ids, const int32_t* dst_ids32,
                         const int64_t* src_ids, const int64_t* edge_map,
                         int64_t nnz, int64_t num_out, int kind, int op,
                         const float* ufeat, const float* efeat, float* out,
                         void* workspace, hipStream_t s, SliceView view = no_view(),
                         SumsOnto onto = {}) {
  char* ws = (char*)workspace;
  uint32_t* cells = (uint32_t*)(ws + p.off_cells);
  uint16_t* rows = (uint16_t*)(ws + p.off_rows);
  float* values = (float*)(ws + p.off_values);
  RowUnit* units = (RowUnit*)(ws + p.off_units);
  RangeUnits* range_units = (RangeUnits*)(ws + p.off_range_units);
  int* unit_total = (int*)(ws + p.off_total);
  float* partial = (float*)(ws + p.off_partial);
  const int ranges = (int)p.ranges;
  const dim3 tiles_grid((unsigned)p.tiles);
#define GS_ROWSUM_PART(IDT, IDS, KEYS)                                                        \
  GS_LAUNCH("rowsum_part", s,                                                                 \
            (rowsum_part_kernel<IDT, KEYS>)<<<tiles_grid, dim3(kPartThreads), 0, s>>>(        \
                IDS, src_ids, edge_map, nnz, num_out, kind, op, ufeat, efeat, ranges,         \
                p.copy_bits, p.tile_stride, cells, rows, values, unit_total, view))
  if (view.sub_indptr != nullptr && view.key_offset != nullptr) {
    if (dst_ids32) GS_ROWSUM_PART(int32_t, dst_ids32, true);
    else GS_ROWSUM_PART(int64_t, dst_ids, true);
  } else {
    if (dst_ids32) GS_ROWSUM_PART(int32_t, dst_ids32, false);
    else GS_ROWSUM_PART(int64_t, dst_ids, false);
  }
#undef GS_ROWSUM_PART
  GS_LAUNCH("rowsum_units", s,
            rowsum_units_kernel<<<dim3((unsigned)ranges), dim3(kUnitsThreads), 0, s>>>(
                cells, p.tiles, p.tile_stride, unit_total, range_units, units));
  GS_LAUNCH("rowsum_accumulate", s,
            rowsum_accumulate_kernel<<<dim3((unsigned)p.max_units), dim3(kAccThreads), 0, s>>>(
                rows, values, cells, p.tile_stride, units, unit_total, partial));
  GS_LAUNCH("rowsum_fold", s,
            rowsum_fold_kernel<<<dim3((unsigned)ceil_div(num_out, kFoldRows)), dim3(kBlock), 0,
                                 s>>>(partial, range_units, 0, num_out, out, onto));
  return GS_OK;
}

// ---------------------------------------- short slices: every range reads every edge
// Below the edges that are worth a partition, atomics on device memory are dear for
// another reason: the rows of hubs are in every tile, and adds to one word are
// executed one after another.  There the ids are few enough for a work-group per range of
// rows and part of the edges to read the ids of its whole part (from L2) and add the
// values of its own rows in LDS; the parts are folded as above.
// 170 K edges of 233 K rows of a power-law graph: 46 us with an atomic a tile and row, now
// 19 and 4 for the fold; 900 K edges 159 and 75; 8 K edges 18 and 12.  With 10 K rows 43
// and 15, 177 and 18.  A range more is a pass more over the ids: at 500 K rows (62 ranges)
// both take the same, at 1 M 57 against 101 on 300 K edges, hence the bound on the ranges.
constexpr int kScanThreads = 1024;
constexpr int kScanWaves = kScanThreads / kWave;
constexpr int kScanRows = 4;    // rows of 64 edges in flight
constexpr int kScanRun = 1024;  // edges whose columns are looked up together
// Two work-groups a compute unit (one: 42 and 105 us on 300 K and 900 K edges where two
// take 35 and 75).
constexpr int kScanGroups = 512;
constexpr int kScanMaxRanges = 32;
constexpr int64_t kScanMinEdges = 2048;

struct RowScanPlan {
  int64_t ranges = 0, parts = 0, wave_edges = 0;
  size_t total = 0;
};
static RowScanPlan row_scan_plan(int64_t nnz, int64_t num_out) {
  RowScanPlan p;
  const int64_t ranges = ceil_div(num_out > 0 ? num_out : 1, kRangeRows);
  if (nnz < kScanMinEdges || nnz >= kPrivateMinEdges || num_out <= 0 || ranges > kScanMaxRanges)
    return p;
  int64_t parts = kScanGroups / ranges;
  // whole rows of a wavefront, as many for each
  const int64_t wave_edges = ceil_div(ceil_div(nnz, parts * kScanWaves), kWave) * kWave;
  parts = ceil_div(nnz, wave_edges * kScanWaves);
  p.ranges = ranges;
  p.parts = parts;
  p.wave_edges = wave_edges;
  p.total = (size_t)(ranges * parts) * kRangeRows * sizeof(float);
  return p;
}

template <typename IdT>
__global__ __launch_bounds__(kScanThreads, 8) void rowsum_scan_kernel(
    const IdT* __restrict__ dst_ids, const int64_t* __restrict__ edge_map, int64_t nnz,
    int64_t num_out, const float* __restrict__ efeat, int ranges, int parts, int64_t wave_edges,
    float* __restrict__ partial, SliceView view) {
  __shared__ double acc[kRangeRows];
  const int t = threadIdx.x, lane = lane_id();
  const int range = blockIdx.x % ranges, part = blockIdx.x / ranges;
  const int64_t row0 = (int64_t)range << kRangeShift;
  const uint32_t rows = (uint32_t)(num_out - row0 < kRangeRows ? num_out - row0 : kRangeRows);
  for (int j = t; j < kRangeRows; j += kScanThreads) acc[j] = -0.0;
  __syncthreads();
  const int64_t first =
      wave_uniform_first(((int64_t)part * kScanWaves + t / kWave) * wave_edges);
  const int64_t stop = first + wave_edges < nnz ? first + wave_edges : nnz;
  for (int64_t run = first; run < stop; run += kScanRun) {
    const int64_t run_stop = run + kScanRun < stop ? run + kScanRun : stop;
    const SliceView::Run r = view.run(run, run_stop - 1);
#pragma unroll 1
    for (int64_t e0 = run; e0 < run_stop; e0 += kScanRows * kWave) {
      int64_t place[kScanRows], key[kScanRows];
#pragma unroll
      for (int i = 0; i < kScanRows; ++i) {
        // (a lane, or a row, past the end reads the last edge)
        const int64_t at = e0 + i * kWave < run_stop ? e0 + i * kWave : run_stop - 1;
        const int64_t e = at + lane < run_stop ? at + lane : run_stop - 1;
        if (r.near()) {
          place[i] = r.place(e);
          key[i] = r.id_offset(e);
        } else {
          int64_t col;
          place[i] = view.row_position(r, at, e, &col, &key[i]);
        }
      }
#pragma unroll
      for (int i = 0; i < kScanRows; ++i) key[i] += (int64_t)dst_ids[place[i]] - row0;
      float val[kScanRows];
#pragma unroll
      for (int i = 0; i < kScanRows; ++i) {
        const bool mine = e0 + i * kWave + lane < run_stop && (uint64_t)key[i] < (uint64_t)rows;
        if (!mine) key[i] = -1;
        val[i] = mine ? efeat[edge_map ? edge_map[place[i]] : place[i]] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < kScanRows; ++i) {
        const double sq = (double)(val[i] * val[i]);
        // one row for the whole wavefront: adds to one word would be taken one after another
        const int key0 = __builtin_amdgcn_readfirstlane((int)key[i]);
        if (key0 >= 0 && __all((int)key[i] == key0)) {
          double sum = sq;
#pragma unroll
          for (int d = kWave / 2; d > 0; d >>= 1) sum += __shfl_down(sum, d, kWave);
          if (lane == 0) atomicAdd(&acc[key0], sum);
        } else if (key[i] >= 0) {
          atomicAdd(&acc[key[i]], sq);
        }
      }
    }
  }
  __syncthreads();
  float* mine = partial + ((int64_t)range * parts + part) * kRangeRows;
  for (int j = t; j < kRangeRows; j += kScanThreads) mine[j] = (float)acc[j];
}

bool sums_by_range(int64_t nnz, int64_t num_out) {
  return row_range_plan(GS_FMT_COO, nnz, num_out).total > 0;
}

size_t sliced_square_sum_bytes(int64_t nnz, int64_t num_out) {
  const size_t scan = row_scan_plan(nnz, num_out).total;
  return scan > 0 ? scan : row_range_plan(GS_FMT_COO, nnz, num_out).total;
}

int sliced_square_sum(SliceView view, const int64_t* indices, const int32_t* indices32,
                      int64_t nnz, const int64_t* edge_map, const float* efeat, float* out,
                      int64_t num_out, void* workspace, size_t workspace_bytes, hipStream_t s,
                      SumsOnto onto) {
  const RowRangePlan plan = row_range_plan(GS_FMT_COO, nnz, num_out);
  if (plan.total > 0 && workspace != nullptr && workspace_bytes >= plan.total)
    return row_range_sum(plan, indices, indices32, nullptr, edge_map, nnz, num_out, 1,
                         kOpCopyRhs, nullptr, efeat, out, workspace, s, view, onto);
  const RowScanPlan scan = row_scan_plan(nnz, num_out);
  if (scan.total > 0 && workspace != nullptr && workspace_bytes >= scan.total) {
    float* partial = (float*)workspace;
    const dim3 grid((unsigned)(scan.ranges * scan.parts));
#define GS_ROWSUM_SCAN(IDT, IDS)                                                              \
  GS_LAUNCH("rowsum_scan", s,                                                                 \
            rowsum_scan_kernel<IDT><<<grid, dim3(kScanThreads), 0, s>>>(                      \
                IDS, edge_map, nnz, num_out, efeat, (int)scan.ranges, (int)scan.parts,        \
                scan.wave_edges, partial, view))
    if (indices32) GS_ROWSUM_SCAN(int32_t, indices32);
    else GS_ROWSUM_SCAN(int64_t, indices);
#undef GS_ROWSUM_SCAN
    GS_LAUNCH("rowsum_fold", s,
              rowsum_fold_kernel<<<dim3((unsigned)ceil_div(num_out, kFoldRows)), dim3(kBlock), 0,
                                   s>>>(partial, nullptr, (int)scan.parts, num_out, out, onto));
    return GS_OK;
  }
  if (onto.fresh) {
    const int64_t blocks = ceil_div(num_out, (int64_t)kBlock * 4);
    GS_LAUNCH("spmm_zero", s,
              spmm_zero_kernel<<<dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(kBlock), 0,
                                 s>>>(out, num_out, onto.base));
  }
  if (nnz == 0) return GS_OK;
  // short slices: combined per tile in LDS, one atomic per (tile, row present);
  // ids outside [0, num_out) cannot occur for a slice of a checked matrix
  return coo_sum_launch(indices, indices, edge_map, nnz, 1, kOpCopyRhs, nullptr, efeat, out,
                        2, view, s);
}

static int check_view(int format, const int64_t* a, const int64_t* b,
                      int64_t num_major, int64_t nnz, const char* who) {
  GS_REQUIRE(format == GS_FMT_COO || format == GS_FMT_COMPRESSED,
             "%s: unknown format %d", who, format);
  GS_REQUIRE(nnz >= 0 && num_major >= 0, "%s: negative size", who);
  GS_REQUIRE(nnz == 0 || (a && b), "%s: null structure pointer", who);
  return GS_OK;
}

static int spmm_launch(int format, const int64_t* a, const int64_t* b,
                       int64_t num_major, int64_t nnz, const int64_t* edge_map,
                       int kind, int op, int reduce, const float* ufeat,
                       const float* efeat, float* out, int64_t* arg_u,
                       int64_t* arg_e, int u_target, int64_t ufeat_len,
                       int64_t efeat_len, int64_t out_len, const int64_t* u_off,
                       const int64_t* e_off, int64_t num_out, void* workspace,
                       size_t workspace_bytes, hipStream_t s) {
  if (nnz == 0 || out_len == 0) return GS_OK;
  const bool scalar = out_len == 1 && (ufeat == nullptr || ufeat_len == 1) &&
                      (efeat == nullptr || efeat_len == 1);
  if (scalar && reduce == kReduceSum) {
    const dim3 grid((unsigned)ceil_div(nnz, kSumTile));
    if (format == GS_FMT_COO) {
      const RowRangePlan plan = row_range_plan(format, nnz, num_out);
      if (plan.total > 0 && workspace != nullptr && workspace_bytes >= plan.total)
        return row_range_sum(plan, u_target == 0 ? b : a, nullptr, u_target == 0 ? a : b,
                             edge_map, nnz, num_out, kind, op, ufeat, efeat, out,
                             workspace, s);
      const size_t need = private_bytes(format, nnz, num_out);
      if (need > 0 && workspace != nullptr && workspace_bytes >= need) {
        float* copies = (float*)workspace;
        const int64_t total = (int64_t)kDies * num_out;
        int64_t zb = ceil_div(total, kBlock * 4);
        if (zb > 4096) zb = 4096;
        GS_LAUNCH("spmm_zero", s,
                  spmm_zero_kernel<<<dim3((unsigned)zb), dim3(kBlock), 0, s>>>(
                      copies, total, 0.f));
        GS_LAUNCH("spmm_coo_sum", s,
                  spmm_coo_sum_kernel<<<grid, dim3(kBlock), 0, s>>>(
                      a, b, edge_map, nnz, kind, op, ufeat, efeat, copies,
                      u_target, num_out, no_view()));
        GS_LAUNCH("spmm_fold", s,
                  spmm_fold_kernel<<<dim3((unsigned)ceil_div(num_out, kBlock)),
                                     dim3(kBlock), 0, s>>>(copies, num_out, out));
        return GS_OK;
      }
      return coo_sum_launch(a, b, edge_map, nnz, kind, op, ufeat, efeat, out, u_target,
                            no_view(), s);
    } else {
      // four tiles per work-group once there are work-groups to spare
      const int rounds = nnz >= ((int64_t)kSumTile * kCscRounds) * 8192 ? kCscRounds : 1;
      GS_LAUNCH("spmm_csc_sum", s,
                spmm_csc_sum_kernel<<<dim3((unsigned)ceil_div(nnz, (int64_t)kSumTile * rounds)),
                                      dim3(kBlock), 0, s>>>(
                    a, b, edge_map, num_major, nnz, kind, op, ufeat, efeat, out, rounds));
    }
    return GS_OK;
  }
  if (format == GS_FMT_COO) {
    const int64_t total = nnz * out_len;
    GS_LAUNCH("spmm_coo", s,
              spmm_coo_kernel<<<dim3((unsigned)ceil_div(total, kBlock)),
                                dim3(kBlock), 0, s>>>(
                  a, b, edge_map, nnz, kind, op, reduce, ufeat, efeat, out,
                  u_target, ufeat_len, efeat_len, out_len, u_off, e_off));
    if (reduce != kReduceSum && (arg_u || arg_e))
      GS_LAUNCH("spmm_coo_arg", s,
                spmm_coo_arg_kernel<<<dim3((unsigned)ceil_div(total, kBlock)),
                                      dim3(kBlock), 0, s>>>(
                    a, b, edge_map, nnz, op, ufeat, efeat, out, arg_u, arg_e,
                    u_target, ufeat_len, efeat_len, out_len, u_off, e_off));
    return GS_OK;
  }
  if (scalar) {
    const int64_t avg = nnz / (num_major > 0 ? num_major : 1);
#define GS_SPMM_SCALAR(G)                                                      \
  GS_LAUNCH("spmm_csc_scalar", s,                                              \
            spmm_csc_scalar_kernel<G><<<dim3((unsigned)ceil_div(num_major * G, kBlock)), \
                                        dim3(kBlock), 0, s>>>(                 \
                a, b, edge_map, num_major, kind, op, reduce, ufeat, efeat, out, \
                arg_u, arg_e))
    if (avg <= 8)
      GS_SPMM_SCALAR(4);
    else if (avg <= 64)
      GS_SPMM_SCALAR(16);
    else
      GS_SPMM_SCALAR(64);
#undef GS_SPMM_SCALAR
    return GS_OK;
  }
  GS_LAUNCH("spmm_csc", s,
            spmm_csc_kernel<<<dim3((unsigned)ceil_div(num_major * out_len, kBlock)),
                              dim3(kBlock), 0, s>>>(
                a, b, edge_map, num_major, kind, op, reduce, ufeat, efeat, out,
                arg_u, arg_e, ufeat_len, efeat_len, out_len, u_off, e_off));
  return GS_OK;
}

}  // namespace gs

extern "C" {

int gs_sddmm(int format, const int64_t* a, const int64_t* b, int64_t num_major,
             int64_t nnz, const int64_t* edge_map, int op, int dtype,
             const void* lhs, const void* rhs, void* out, int lhs_target,
             int rhs_target, int64_t lhs_len, int64_t rhs_len, int64_t out_len,
             int64_t reduce_size, const int64_t* lhs_off, const int64_t* rhs_off,
             gs_stream_t stream) {
  using namespace gs;
  int rc = check_view(format, a, b, num_major, nnz, "sddmm");
  if (rc != GS_OK) return rc;
  GS_REQUIRE(op >= kOpAdd && op <= kOpDot, "sddmm: unknown operator %d", op);
  GS_REQUIRE(dtype == GS_F32 || dtype == GS_F64, "sddmm: unknown dtype %d", dtype);
  GS_REQUIRE(lhs_target >= 0 && lhs_target <= 2 && rhs_target >= 0 && rhs_target <= 2,
             "sddmm: targets must be 0 (u), 1 (e) or 2 (v)");
  GS_REQUIRE(out_len >= 0 && reduce_size >= 1, "sddmm: bad feature sizes");
  if (nnz == 0 || out_len == 0) return GS_OK;
  GS_REQUIRE(out && (lhs || op == kOpCopyRhs) && (rhs || op == kOpCopyLhs),
             "sddmm: null operand");
  hipStream_t s = as_stream(stream);
  const EdgeView g{format == GS_FMT_COMPRESSED, a, b, num_major, edge_map};
#define GS_SDDMM_LAUNCH(T, ITEMS)                                                         \
  GS_LAUNCH("sddmm", s,                                                                   \
            (sddmm_kernel<T, ITEMS>)<<<dim3((unsigned)ceil_div(nnz * out_len, kBlock * ITEMS)), \
                                     dim3(kBlock), 0, s>>>(                               \
                g, nnz, op, (const T*)lhs, (const T*)rhs, (T*)out, lhs_target, rhs_target, \
                lhs_len, rhs_len, out_len, reduce_size, lhs_off, rhs_off))
  // (targets: 0 = row ids, 1 = the edge's own, 2 = column ids)
#define GS_SDDMM_SCALAR(T)                                                                    \
  GS_LAUNCH("sddmm", s,                                                                       \
            sddmm_scalar_kernel<T><<<dim3((unsigned)ceil_div(nnz, kBlock * kScalarItems)),    \
                                     dim3(kBlock), 0, s>>>(                                   \
                nnz, op, edge_map, lhs_target == 0 ? a : lhs_target == 2 ? b : nullptr,       \
                rhs_target == 0 ? a : rhs_target == 2 ? b : nullptr, (const T*)lhs,           \
                (const T*)rhs, (T*)out))
  if (!g.compressed && out_len == 1 && reduce_size == 1 && lhs_len == 1 && rhs_len == 1 &&
      !lhs_off && !rhs_off) {
    if (dtype == GS_F32) GS_SDDMM_SCALAR(float);
    else GS_SDDMM_SCALAR(double);
  } else if (g.compressed) {
    if (dtype == GS_F32) GS_SDDMM_LAUNCH(float, kEdgeItems);
    else GS_SDDMM_LAUNCH(double, kEdgeItems);
  } else {
    if (dtype == GS_F32) GS_SDDMM_LAUNCH(float, 1);
    else GS_SDDMM_LAUNCH(double, 1);
  }
#undef GS_SDDMM_LAUNCH
#undef GS_SDDMM_SCALAR
  return GS_OK;
}

int gs_edge_score(int format, const int64_t* a, const int64_t* b, int64_t num_major,
                  int64_t nnz, const int64_t* edge_map, const gs_score_term* terms,
                  int num_terms, int64_t feature_len, const float* weights, int positive_part,
                  float shift, float* out, gs_stream_t stream) {
  using namespace gs;
  int rc = check_view(format, a, b, num_major, nnz, "edge_score");
  if (rc != GS_OK) return rc;
  GS_REQUIRE(terms && num_terms >= 1 && num_terms <= GS_SCORE_MAX_TERMS,
             "edge_score: 1 to %d terms", GS_SCORE_MAX_TERMS);
  GS_REQUIRE(weights || num_terms == 1, "edge_score: several terms need weights");
  if (nnz == 0) return GS_OK;
  ScoreArgs args{};
  bool products = false, wide = true;
  for (int k = 0; k < num_terms; ++k) {
    const gs_score_term& t = terms[k];
    GS_REQUIRE(t.kind >= GS_SCORE_VALUE && t.kind <= GS_SCORE_PRODUCTS,
               "edge_score: unknown kind of term %d", t.kind);
    GS_REQUIRE(t.lhs && (t.rhs || t.kind == GS_SCORE_VALUE), "edge_score: null operand");
    GS_REQUIRE(t.kind == GS_SCORE_VALUE || (t.lhs_target >= 0 && t.lhs_target <= 2 &&
                                            t.rhs_target >= 0 && t.rhs_target <= 2),
               "edge_score: targets must be 0 (u), 1 (e) or 2 (v)");
    if (t.kind == GS_SCORE_PRODUCTS) {
      products = true;
      wide = wide && (((uintptr_t)t.lhs | (uintptr_t)t.rhs) & 15) == 0;
    }
    args.term[k] = t;
  }
  GS_REQUIRE(!products || (feature_len >= 1 && feature_len <= GS_SCORE_MAX_LEN),
             "edge_score: features of 1 to %d values", GS_SCORE_MAX_LEN);
  GS_REQUIRE(out, "edge_score: null output");
  args.num_terms = num_terms;
  args.len = products ? (int)feature_len : 1;
  args.positive_part = positive_part;
  args.shift = shift;
  args.weights = weights;
  wide = wide && args.len % 4 == 0;
  hipStream_t s = as_stream(stream);
  const EdgeView g{format == GS_FMT_COMPRESSED, a, b, num_major, edge_map};
#define GS_SCORE_LAUNCH(P, WIDE, ITEMS)                                                       \
  GS_LAUNCH("edge_score", s,                                                                  \
            (edge_score_kernel<P, WIDE, ITEMS>)<<<dim3((unsigned)ceil_div(nnz, kBlock * ITEMS)), \
                                                  dim3(kBlock), 0, s>>>(g, nnz, args, out))
#define GS_SCORE_BY_FORM(P, WIDE)                     \
  do {                                                \
    if (g.compressed) GS_SCORE_LAUNCH(P, WIDE, kEdgeItems); \
    else GS_SCORE_LAUNCH(P, WIDE, 1);                 \
  } while (0)
#define GS_SCORE_BY_WIDTH(P)            \
  do {                                  \
    if (wide) GS_SCORE_BY_FORM(P, true); \
    else GS_SCORE_BY_FORM(P, false);    \
  } while (0)
  if (args.len >= 32) GS_SCORE_BY_WIDTH(32);
  else if (args.len >= 16) GS_SCORE_BY_WIDTH(16);
  else if (args.len >= 8) GS_SCORE_BY_WIDTH(8);
  else if (args.len >= 4) GS_SCORE_BY_WIDTH(4);
  else if (args.len >= 2) GS_SCORE_BY_FORM(2, false);
  else GS_SCORE_BY_FORM(1, false);
#undef GS_SCORE_BY_WIDTH
#undef GS_SCORE_BY_FORM
#undef GS_SCORE_LAUNCH
  return GS_OK;
}

int gs_normalise_columns(const int64_t* indptr, int64_t num_cols, const int64_t* rows,
                         int64_t nnz, const float* values, int64_t num_values,
                         const int64_t* select, const float* row_divisor, double* sums, float* out,
                         gs_stream_t stream) {
  if (nnz > 0 && num_cols > 0 && sums)
    GS_LAUNCH("normalise_clear", gs::as_stream(stream),
              gs::normalise_clear_kernel<<<dim3((unsigned)gs::ceil_div(num_cols, gs::kBlock)),
                                           dim3(gs::kBlock), 0, gs::as_stream(stream)>>>(sums,
                                                                                        num_cols));
  return gs_normalise_columns_cleared(indptr, num_cols, rows, nnz, values, num_values, select,
                                      row_divisor, sums, out, stream);
}

int gs_normalise_columns_cleared(const int64_t* indptr, int64_t num_cols, const int64_t* rows,
                                 int64_t nnz, const float* values, int64_t num_values,
                                 const int64_t* select, const float* row_divisor, double* sums,
                                 float* out, gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(num_cols >= 0 && nnz >= 0, "normalise_columns: negative size");
  if (nnz == 0) return GS_OK;
  GS_REQUIRE(num_cols > 0 && indptr && values && sums && out && (rows || !row_divisor),
             "normalise_columns: null pointer");
  GS_REQUIRE(num_values >= 1 && (select || num_values >= nnz), "normalise_columns: %lld values",
             (long long)num_values);
  hipStream_t s = as_stream(stream);
  const bool moved = select || row_divisor, long_runs = !moved && nnz > kLongRuns;
  const unsigned run = kRunThreads * (long_runs ? kLongRunItems : kRunItems);
  const dim3 grid((unsigned)ceil_div(nnz, (int64_t)run));
#define GS_NORMALISE_SUM(SELECT, DIVIDE, ITEMS)                                               \
  GS_LAUNCH("normalise_sum", s,                                                               \
            (normalise_sum_kernel<SELECT, DIVIDE, ITEMS>)<<<grid, dim3(kRunThreads), 0, s>>>( \
                indptr, num_cols, rows, nnz, values, num_values, select, row_divisor, sums, out))
  if (select && row_divisor) GS_NORMALISE_SUM(true, true, kRunItems);
  else if (select) GS_NORMALISE_SUM(true, false, kRunItems);
  else if (row_divisor) GS_NORMALISE_SUM(false, true, kRunItems);
  else if (!long_runs) GS_NORMALISE_SUM(false, false, kRunItems);
  else GS_NORMALISE_SUM(false, false, kLongRunItems);
#undef GS_NORMALISE_SUM
  const unsigned group = run / (kRunThreads * kRunItems);
  GS_LAUNCH("normalise_divide", s,
            normalise_divide_kernel<<<dim3((unsigned)ceil_div(grid.x, kDies) * kDies * group),
                                      dim3(kRunThreads), 0, s>>>(
                indptr, num_cols, nnz, sums, moved ? out : values, out, group));
  return GS_OK;
}

int gs_fused_u_op_v(int format, const int64_t* a, const int64_t* b,
                    int64_t num_major, int64_t nnz, const int64_t* edge_map,
                    int op, int dtype,
                    const void* lhs1, const void* rhs1, void* out1,
                    const void* lhs2, const void* rhs2, void* out2,
                    int64_t lhs_len, int64_t rhs_len, int64_t out_len,
                    int64_t reduce_size, const int64_t* lhs_off,
                    const int64_t* rhs_off, gs_stream_t stream) {
  using namespace gs;
  int rc = check_view(format, a, b, num_major, nnz, "fused_u_op_v");
  if (rc != GS_OK) return rc;
  GS_REQUIRE((op >= kOpAdd && op <= kOpDiv) || op == kOpDot,
             "fused_u_op_v: operator %d needs both operands", op);
  GS_REQUIRE(dtype == GS_F32 || dtype == GS_F64, "fused_u_op_v: unknown dtype %d", dtype);
  if (nnz == 0 || out_len == 0) return GS_OK;
  GS_REQUIRE(lhs1 && rhs1 && out1 && lhs2 && rhs2 && out2, "fused_u_op_v: null operand");
  hipStream_t s = as_stream(stream);
  const EdgeView g{format == GS_FMT_COMPRESSED, a, b, num_major, edge_map};
#define GS_UOPV_LAUNCH(T, ITEMS)                                                          \
  GS_LAUNCH("fused_u_op_v", s,                                                            \
            (fused_u_op_v_kernel<T, ITEMS>)<<<dim3((unsigned)ceil_div(nnz * out_len,      \
                                                                      kBlock * ITEMS)),   \
                                            dim3(kBlock), 0, s>>>(                        \
                g, nnz, op, (const T*)lhs1, (const T*)rhs1, (T*)out1, (const T*)lhs2,     \
                (const T*)rhs2, (T*)out2, lhs_len, rhs_len, out_len, reduce_size, lhs_off, \
                rhs_off))
  if (g.compressed) {
    if (dtype == GS_F32) GS_UOPV_LAUNCH(float, kEdgeItems);
    else GS_UOPV_LAUNCH(double, kEdgeItems);
  } else {
    if (dtype == GS_F32) GS_UOPV_LAUNCH(float, 1);
    else GS_UOPV_LAUNCH(double, 1);
  }
#undef GS_UOPV_LAUNCH
  return GS_OK;
}

size_t gs_spmm_workspace_bytes(int format, int64_t nnz, int64_t num_out) {
  const gs::RowRangePlan plan = gs::row_range_plan(format, nnz, num_out);
  if (plan.total > 0) return plan.total;
  return gs::private_bytes(format, nnz, num_out);
}

int gs_spmm(int format, const int64_t* a, const int64_t* b, int64_t num_major,
            int64_t nnz, const int64_t* edge_map, int op, int reduce,
            const float* ufeat, const float* efeat, float* out, int64_t* arg_u,
            int64_t* arg_e, int u_target, int64_t ufeat_len, int64_t efeat_len,
            int64_t out_len, const int64_t* u_off, const int64_t* e_off,
            int64_t num_out, void* workspace, size_t workspace_bytes,
            gs_stream_t stream) {
  using namespace gs;
  int rc = check_view(format, a, b, num_major, nnz, "spmm");
  if (rc != GS_OK) return rc;
  GS_REQUIRE((op >= kOpAdd && op <= kOpCopyRhs), "spmm: unknown operator %d", op);
  GS_REQUIRE(reduce >= kReduceSum && reduce <= kReduceMin, "spmm: unknown reducer %d", reduce);
  GS_REQUIRE(u_target == 0 || u_target == 2, "spmm: u_target must be 0 or 2");
  if (nnz == 0 || out_len == 0) return GS_OK;
  GS_REQUIRE(out && (ufeat || op == kOpCopyRhs) && (efeat || op == kOpCopyLhs),
             "spmm: null operand");
  return spmm_launch(format, a, b, num_major, nnz, edge_map, 0, op, reduce,
                     op == kOpCopyRhs ? nullptr : ufeat,
                     op == kOpCopyLhs ? nullptr : efeat, out, arg_u, arg_e,
                     u_target, ufeat_len, efeat_len, out_len, u_off, e_off,
                     num_out, workspace, workspace_bytes, as_stream(stream));
}

int gs_e_square_sum(int format, const int64_t* a, const int64_t* b,
                    int64_t num_major, int64_t nnz, const int64_t* edge_map,
                    const float* efeat, float* out, int u_target,
                    int64_t feat_len, int64_t num_out, void* workspace,
                    size_t workspace_bytes, gs_stream_t stream) {
  using namespace gs;
  int rc = check_view(format, a, b, num_major, nnz, "e_square_sum");
  if (rc != GS_OK) return rc;
  GS_REQUIRE(u_target == 0 || u_target == 2, "e_square_sum: u_target must be 0 or 2");
  if (nnz == 0 || feat_len == 0) return GS_OK;
  GS_REQUIRE(efeat && out, "e_square_sum: null operand");
  return spmm_launch(format, a, b, num_major, nnz, edge_map, 1, kOpCopyRhs,
                     kReduceSum, nullptr, efeat, out, nullptr, nullptr, u_target,
                     0, feat_len, feat_len, nullptr, nullptr, num_out, workspace,
                     workspace_bytes, as_stream(stream));
}

size_t gs_sliced_e_square_sum_workspace_bytes(int64_t slice_nnz, int64_t num_out) {
  if (slice_nnz < 0 || num_out < 0) return 0;
  return gs::sliced_square_sum_bytes(slice_nnz, num_out);
}

int gs_sliced_e_square_sum(const int64_t* indptr, const int64_t* indices,
                           const int32_t* indices32, const int64_t* cols,
                           int64_t num_cols_picked, const int64_t* sub_indptr,
                           int64_t slice_nnz, const int64_t* edge_map, const float* efeat,
                           float* out,
                           int64_t num_out, void* workspace, size_t workspace_bytes,
                           gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(num_cols_picked >= 0 && slice_nnz >= 0 && num_out >= 0,
             "sliced_e_square_sum: negative size");
  if (slice_nnz == 0) return GS_OK;
  GS_REQUIRE(indptr && indices && cols && sub_indptr && efeat && out,
             "sliced_e_square_sum: null pointer");
  const SliceView view{sub_indptr, cols, indptr, nullptr, num_cols_picked};
  return sliced_square_sum(view, indices, indices32, slice_nnz, edge_map, efeat, out, num_out,
                           workspace, workspace_bytes, as_stream(stream));
}

int gs_sliced_e_square_sums(const int64_t* indptr, const int64_t* indices,
                            const int32_t* indices32, const int64_t* cols,
                            int64_t num_cols_picked, const int64_t* sub_indptr,
                            int64_t slice_nnz, const int64_t* edge_map, const float* efeat,
                            float* out, int64_t num_out, void* workspace, size_t workspace_bytes,
                            gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(num_cols_picked >= 0 && slice_nnz >= 0 && num_out >= 0,
             "sliced_e_square_sums: negative size");
  if (num_out == 0) return GS_OK;
  GS_REQUIRE(out && (slice_nnz == 0 || (indptr && indices && cols && sub_indptr && efeat)),
             "sliced_e_square_sums: null pointer");
  const SliceView view{sub_indptr, cols, indptr, nullptr, num_cols_picked};
  return sliced_square_sum(view, indices, indices32, slice_nnz, edge_map, efeat, out, num_out,
                           workspace, workspace_bytes, as_stream(stream), SumsOnto{true, 0.f});
}

int gs_e_div_u_sum(int format, const int64_t* a, const int64_t* b,
                   int64_t num_major, int64_t nnz, const int64_t* edge_map,
                   const float* ufeat, const float* efeat, float* out,
                   int u_target, int64_t feat_len, int64_t num_out,
                   void* workspace, size_t workspace_bytes, gs_stream_t stream) {
  using namespace gs;
  int rc = check_view(format, a, b, num_major, nnz, "e_div_u_sum");
  if (rc != GS_OK) return rc;
  GS_REQUIRE(u_target == 0 || u_target == 2, "e_div_u_sum: u_target must be 0 or 2");
  if (nnz == 0 || feat_len == 0) return GS_OK;
  GS_REQUIRE(ufeat && efeat && out, "e_div_u_sum: null operand");
  return spmm_launch(format, a, b, num_major, nnz, edge_map, 2, kOpDiv,
                     kReduceSum, ufeat, efeat, out, nullptr, nullptr, u_target,
                     feat_len, feat_len, feat_len, nullptr, nullptr, num_out,
                     workspace, workspace_bytes, as_stream(stream));
}

}  // extern "C"

// weighted.hip -- weighted sampling: per column (individual) and over a list
// (collective / layer-wise), with and without replacement.
//
// Without replacement: Efraimidis-Spirakis in exponential-clock form.  Item i
// gets key (-log2 u_i) / w_i, the K smallest keys win (same ranking as the K
// largest u^(1/w)).  The key uses correctly rounded double operations only, so
// the CPU check computes bit-identical keys; ties break to the smaller index.
// With replacement: integer CDF (weights quantised against the exact maximum,
// integer prefix sums are order-independent) and a binary search per pick.
#include "common.h"
#include "scan.h"

// The sampling keys must come out bit-identical to the CPU check: no implicit
// fusing of a multiply into a neighbouring add anywhere in this file.
#pragma clang fp contract(off)

#include <cstdlib>
#include <cstring>
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_segmented_radix_sort.hpp>

namespace gs {

// ------------------------------------------------------------ key arithmetic
// x / y for finite normal y > 0 from fused multiply-adds only: a bit-trick
// reciprocal estimate (12 % off at worst), six Newton steps, one residual
// correction.  Hardware division is avoided because its last bit need not
// agree between a GPU and a CPU; every operation here is a correctly rounded
// IEEE operation, so the result is reproducible anywhere (it lies within an
// ulp or two of the true quotient, which is all a sampling key needs).
__device__ __forceinline__ double det_div(double x, double y) {
  double r = __longlong_as_double(0x7FDE623822FC16E6ll - __double_as_longlong(y));
#pragma unroll
  for (int i = 0; i < 6; ++i) r = __fma_rn(r, __fma_rn(-y, r, 1.0), r);
  const double q = __dmul_rn(x, r);
  return __fma_rn(__fma_rn(-y, q, x), r, q);
}

__device__ __forceinline__ double neg_log2_unit(uint64_t r64) {
  const uint64_t v = (r64 >> 12) + 1;  // [1, 2^52]: exact as a double
  int e = 63 - __clzll((long long)v);
  double m = ldexp((double)(long long)v, -e);  // [1, 2)
  if (m > 0x1.6a09e667f3bcdp+0) {
    m = __dmul_rn(m, 0.5);
    e += 1;
  }
  const double s = det_div(__dsub_rn(m, 1.0), __dadd_rn(m, 1.0));
  const double s2 = __dmul_rn(s, s);
  double p = 0x1.1964ec6fc9491p-3;
  p = __fma_rn(p, s2, 0x1.3703c1f4d0ffep-3);
  p = __fma_rn(p, s2, 0x1.5b9ac9b743f0dp-3);
  p = __fma_rn(p, s2, 0x1.89f3b1694cffep-3);
  p = __fma_rn(p, s2, 0x1.c68f568d31761p-3);
  p = __fma_rn(p, s2, 0x1.0c9a84994022dp-2);
  p = __fma_rn(p, s2, 0x1.484b13d7c02a9p-2);
  p = __fma_rn(p, s2, 0x1.a61762a7adedap-2);
  p = __fma_rn(p, s2, 0x1.2776c50ef9bfep-1);
  p = __fma_rn(p, s2, 0x1.ec709dc3a03fep-1);
  p = __fma_rn(p, s2, 0x1.71547652b82fep+1);
  return __fma_rn(-s, p, (double)(52 - e));
}

__device__ __forceinline__ double weighted_key(PhiloxKey key, uint64_t pos,
                                               uint64_t draw, float w) {
  if (!(w > 0.0f)) return __longlong_as_double(0x7ff0000000000000ll);  // +inf
  const Words4 wd = philox(key, pos, draw);
  const uint64_t r = ((uint64_t)wd.y << 32) | wd.x;
  return det_div(neg_log2_unit(r), (double)w);
}

__global__ void weighted_key_probe_kernel(PhiloxKey key, uint64_t pos,
                                          uint64_t draw, float w, uint64_t r64,
                                          double* out) {
  out[0] = neg_log2_unit(r64);
  out[1] = weighted_key(key, pos, draw, w);
}

__device__ __forceinline__ bool key_less(double ka, int64_t ia, double kb,
                                         int64_t ib) {
  return ka < kb || (ka == kb && ia < ib);
}

// -------------------------------------------- per column, without replacement
// One wavefront per requested column.  Every lane keeps the K smallest keys of
// the edges it visits (lane l sees offsets l, l + 64, ...) as a sorted list in
// LDS, laid out [slot][thread] so that a wavefront touches consecutive banks.
// The 64 sorted lists are then merged by K rounds of a wavefront arg-min.
__global__ __launch_bounds__(kBlock) void sample_weighted_kernel(
    const int64_t* __restrict__ indptr, int64_t num_cols,
    const int64_t* __restrict__ indices, const float* __restrict__ probs,
    const int64_t* __restrict__ column_ids, int64_t num_items, int fanout,
    PhiloxKey key, const int64_t* __restrict__ sub_indptr,
    int64_t* __restrict__ out_coo_col, int64_t* __restrict__ out_indices,
    int64_t* __restrict__ out_select, ColumnLabels labels) {
  extern __shared__ __align__(8) unsigned char smem[];
  const int nthreads = blockDim.x;
  double* lkey = (double*)smem;                               // [fanout][nthreads]
  int* lidx = (int*)(smem + (size_t)fanout * nthreads * sizeof(double));
  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int64_t item = ((int64_t)blockIdx.x * nthreads + tid) / kWave;
  if (item >= num_items) return;
  const int64_t c = column_ids ? column_ids[item] : item;
  int64_t in_start;
  const int64_t deg = column_degree(indptr, num_cols, c, &in_start);
  if (deg == 0) return;
  const int64_t out_start = sub_indptr[item];
  const int K = fanout;

  if (deg <= K) {  // whole column, original order, zero weights included
    for (int64_t j = lane; j < deg; j += kWave) {
      const int64_t p = in_start + j;
      out_indices[out_start + j] = indices ? indices[p] : p;
      out_select[out_start + j] = p;
      if (out_coo_col) out_coo_col[out_start + j] = labels.of(item);
    }
    return;
  }

  int cnt = 0;
  for (int64_t j = lane; j < deg; j += kWave) {
    const double k = weighted_key(key, (uint64_t)item, (uint64_t)j, probs[in_start + j]);
    // offsets grow along a lane, so an equal key never displaces a kept one
    if (cnt == K && !(k < lkey[(K - 1) * nthreads + tid])) continue;
    int s = cnt < K ? cnt : K - 1;
    while (s > 0 && k < lkey[(s - 1) * nthreads + tid]) {
      lkey[s * nthreads + tid] = lkey[(s - 1) * nthreads + tid];
      lidx[s * nthreads + tid] = lidx[(s - 1) * nthreads + tid];
      --s;
    }
    lkey[s * nthreads + tid] = k;
    lidx[s * nthreads + tid] = (int)(j / kWave);  // j = lane + 64 * (stored value)
    if (cnt < K) ++cnt;
  }

  int head = 0;
  int64_t mine = -1;  // lane r keeps the winner of round r
  for (int r = 0; r < K; ++r) {
    double k = __longlong_as_double(0x7ff0000000000000ll);
    int64_t off = INT64_MAX;
    if (head < cnt) {
      k = lkey[head * nthreads + tid];
      off = (int64_t)lidx[head * nthreads + tid] * kWave + lane;
    }
    double bk = k;
    int64_t bo = off;
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) {
      const double ok = __shfl_xor(bk, d, kWave);
      const int64_t oo = __shfl_xor(bo, d, kWave);
      if (key_less(ok, oo, bk, bo)) {
        bk = ok;
        bo = oo;
      }
    }
    if (off == bo) ++head;  // offsets are unique, so exactly one lane advances
    if (lane == r) mine = bo;
  }
  if (lane < K) {
    const int64_t p = in_start + mine;
    out_indices[out_start + lane] = indices ? indices[p] : p;
    out_select[out_start + lane] = p;
    if (out_coo_col) out_coo_col[out_start + lane] = labels.of(item);
  }
}

// ----------------------------------------------- per column, with replacement
__device__ __forceinline__ uint64_t quantise(float w, double scale) {
  return w > 0.0f ? (uint64_t)__dmul_rn((double)w, scale) : 0ull;
}

// Exact max of the weights, integer CDF, one binary search per output slot.  A
// wavefront takes a column of up to kReplLong edges, the whole work-group one of
// its longer columns after the other; a lane takes eight neighbouring edges, so
// that their loads are in flight together and one scan serves 512 edges.  The CDF
// of a column of up to kReplHeld edges stays in LDS, and its weights in registers
// between the two passes; longer ones use the scratch slice of the column.  The
// sums are integers: the split does not change them.
// What bounds it is the chain of loads of the longest column.  A wavefront per
// column that read 64 edges at a time took 195 us on 794 columns with 368 Ki edges
// (a power law: the longest has some twenty thousand); this takes 30 us.
constexpr int kReplThreads = 512;
constexpr int kReplWaves = kReplThreads / kWave;
constexpr int kReplItems = 8;
constexpr int kReplHeld = kReplItems * kWave;
constexpr int kReplLong = 2048;

// The weights of edges [j0, j0 + kReplItems) of a column, 0 beyond its end.
__device__ __forceinline__ void repl_load(const float* __restrict__ w, int64_t j0, int64_t deg,
                                          float (&out)[kReplItems]) {
  struct Held {
    float v[kReplItems];
  };
  if (j0 + kReplItems <= deg) {
    Held h;
    __builtin_memcpy(&h, w + j0, sizeof(Held));
#pragma unroll
    for (int i = 0; i < kReplItems; ++i) out[i] = h.v[i];
    return;
  }
#pragma unroll
  for (int i = 0; i < kReplItems; ++i) out[i] = j0 + i < deg ? w[j0 + i] : 0.0f;
}

__device__ __forceinline__ float repl_max(const float (&w)[kReplItems], float m) {
#pragma unroll
  for (int i = 0; i < kReplItems; ++i)
    if (w[i] > m) m = w[i];
  return m;
}

__device__ __forceinline__ float wave_max(float m) {
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) {
    const float o = __shfl_xor(m, d, kWave);
    if (o > m) m = o;
  }
  return m;
}

// Weights -> quantised inclusive sums over the lane's edges; the last is the lane's total.
__device__ __forceinline__ void repl_sums(const float (&w)[kReplItems], double scale,
                                          uint64_t (&q)[kReplItems]) {
  uint64_t run = 0;
#pragma unroll
  for (int i = 0; i < kReplItems; ++i) {
    run += quantise(w[i], scale);
    q[i] = run;
  }
}

__device__ __forceinline__ double repl_scale(float wmax) {
  return wmax > 0.0f ? det_div(2147483648.0, (double)wmax) : 0.0;
}

__device__ __forceinline__ void repl_store(uint64_t* cdf, int64_t j0, int64_t deg, uint64_t before,
                                           const uint64_t (&q)[kReplItems]) {
#pragma unroll
  for (int i = 0; i < kReplItems; ++i)
    if (j0 + i < deg) cdf[j0 + i] = before + q[i];
}

__global__ __launch_bounds__(kReplThreads) void sample_weighted_replace_kernel(
    const int64_t* __restrict__ indptr, int64_t num_cols,
    const int64_t* __restrict__ indices, const float* __restrict__ probs,
    const int64_t* __restrict__ column_ids, int64_t num_items, int64_t fanout,
    PhiloxKey key, const int64_t* __restrict__ sub_indptr,
    const int64_t* __restrict__ cdf_offsets, uint64_t* cdf_scratch,
    int64_t* __restrict__ out_coo_col, int64_t* __restrict__ out_indices,
    int64_t* __restrict__ out_select, ColumnLabels labels) {
  __shared__ uint64_t held[kReplWaves][kReplHeld];
  __shared__ int64_t col_deg[kReplWaves], col_start[kReplWaves], col_cdf[kReplWaves];
  __shared__ uint64_t col_total[kReplWaves];
  __shared__ float wave_wmax[kReplWaves];
  __shared__ uint64_t smem[kReplWaves + 1];
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int64_t item = (int64_t)blockIdx.x * kReplWaves + wave;
  int64_t deg = 0, in_start = 0, at = 0;
  if (item < num_items) {
    deg = column_degree(indptr, num_cols, column_ids ? column_ids[item] : item, &in_start);
    if (deg > 0) at = cdf_offsets ? cdf_offsets[item] : in_start;
  }
  if (lane == 0) {
    col_deg[wave] = deg;
    col_start[wave] = in_start;
    col_cdf[wave] = at;
  }
  if (deg > 0 && deg <= kReplHeld) {
    float w[kReplItems];
    uint64_t q[kReplItems];
    repl_load(probs + in_start, lane * kReplItems, deg, w);
    repl_sums(w, repl_scale(wave_max(repl_max(w, 0.0f))), q);
    const uint64_t incl = wave_inclusive_sum(q[kReplItems - 1]);
    repl_store(held[wave], lane * kReplItems, deg, incl - q[kReplItems - 1], q);
    if (lane == kWave - 1) col_total[wave] = incl;
  } else if (deg > 0 && deg <= kReplLong) {
    float wmax = 0.0f;
    for (int64_t base = 0; base < deg; base += kReplHeld) {
      float w[kReplItems];
      repl_load(probs + in_start, base + lane * kReplItems, deg, w);
      wmax = repl_max(w, wmax);
    }
    const double scale = repl_scale(wave_max(wmax));
    uint64_t carry = 0;
    for (int64_t base = 0; base < deg; base += kReplHeld) {
      float w[kReplItems];
      uint64_t q[kReplItems];
      repl_load(probs + in_start, base + lane * kReplItems, deg, w);
      repl_sums(w, scale, q);
      const uint64_t incl = wave_inclusive_sum(q[kReplItems - 1]);
      repl_store(cdf_scratch + at, base + lane * kReplItems, deg, carry + incl - q[kReplItems - 1],
                 q);
      carry += __shfl((unsigned long long)incl, kWave - 1, kWave);
    }
    if (lane == 0) col_total[wave] = carry;
  }
  __syncthreads();
  for (int c = 0; c < kReplWaves; ++c) {
    const int64_t n = col_deg[c];  // the same for every thread
    if (n <= kReplLong) continue;
    const float* from = probs + col_start[c];
    float wmax = 0.0f;
    for (int64_t base = 0; base < n; base += kReplThreads * kReplItems) {
      float w[kReplItems];
      repl_load(from, base + (int64_t)threadIdx.x * kReplItems, n, w);
      wmax = repl_max(w, wmax);
    }
    wmax = wave_max(wmax);
    if (lane == 0) wave_wmax[wave] = wmax;
    __syncthreads();
#pragma unroll
    for (int v = 0; v < kReplWaves; ++v)
      if (wave_wmax[v] > wmax) wmax = wave_wmax[v];
    const double scale = repl_scale(wmax);
    uint64_t carry = 0;
    for (int64_t base = 0; base < n; base += kReplThreads * kReplItems) {
      const int64_t j0 = base + (int64_t)threadIdx.x * kReplItems;
      float w[kReplItems];
      uint64_t q[kReplItems];
      repl_load(from, j0, n, w);
      repl_sums(w, scale, q);
      uint64_t sum;
      const uint64_t before =
          block_exclusive_sum<uint64_t, kReplThreads>(q[kReplItems - 1], smem, &sum);
      repl_store(cdf_scratch + col_cdf[c], j0, n, carry + before, q);
      carry += sum;
    }
    if (threadIdx.x == 0) col_total[c] = carry;
    __syncthreads();
  }
  // every CDF was written by this work-group, in front of a barrier
  if (deg == 0) return;
  const int64_t out_start = sub_indptr[item];
  const uint64_t total = col_total[wave];
  auto pick = [&](const uint64_t* cdf, int64_t j) {
    const uint64_t t = total > 0 ? philox_bounded(key, (uint64_t)item, (uint64_t)j, total) : 0ull;
    int64_t lo = 0, hi = deg;  // first position whose value exceeds t, or the last one
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (cdf[mid] > t)
        hi = mid;
      else
        lo = mid + 1;
    }
    const int64_t p = in_start + (lo < deg ? lo : deg - 1);
    out_indices[out_start + j] = indices ? indices[p] : p;
    out_select[out_start + j] = p;
    if (out_coo_col) out_coo_col[out_start + j] = labels.of(item);
  };
  if (deg <= kReplHeld)
    for (int64_t j = lane; j < fanout; j += kWave) pick(held[wave], j);
  else
    for (int64_t j = lane; j < fanout; j += kWave) pick(cdf_scratch + at, j);
}

// ------------------------------------------- persistent packed CDF of a matrix
// One 64-bit entry per edge, built once per (matrix, weights):
//   cdf[0]      = row_bits, the number of low bits of an entry that hold a row id
//                 (0: no row ids packed, the sampler reads them from `indices`)
//   cdf[e + 1]  = share(e) << row_bits | row id of edge e
// share(e) is the part of its column's mass that lies at or before edge e, in
// units of 2^-cb (cb = min(62, 64 - row_bits)): the weights of a column are
// quantised to 31 bits against the column's exact maximum (integers, so their
// prefix sums G do not depend on the order of additions), and
//   share(e) = floor(G(e) * 2^cb / T)   for G(e) < T = the column's total,
//   share(e) = 2^cb - 1                 from the last positive item on
// (0 everywhere in a column without positive weights).  Item j of a column
// owns [share(j - 1), share(j)); a draw is a search for the item whose interval
// holds a point, over 8-byte entries, and the row id of the item arrives with
// the entry that ends the search: a pick costs the lines of its search and
// nothing else.  (Row ids and prefix sums in arrays of their own cost a random
// 128-byte line per pick for the row id and two for the ends of the column's
// slice of a global prefix sum.)
// Both passes take tiles of consecutive edges and look the tile's first and
// last column up once per wavefront; an edge then searches only among
// the columns of its tile instead of all of them.
constexpr int kCdfItems = 8;
constexpr int kCdfTile = kBlock * kCdfItems;
constexpr int kCdfMaxRowBits = 32;

// Column maxima: the tile's maxima are first taken in LDS (integer atomics on
// the bit patterns: positive floats order like their bits), then every column
// the tile touches sends one atomic to memory.  With one atomic per edge the
// pass ran at the rate of the memory-side atomic units.
constexpr int kCdfSegs = 4096;

__global__ __launch_bounds__(kBlock) void cdf_colmax_kernel(
    const int64_t* __restrict__ indptr, int64_t num_cols,
    const float* __restrict__ probs, int64_t nnz, unsigned int* colmax_bits) {
  __shared__ unsigned int tile_max[kCdfSegs];
  const int64_t e0 = (int64_t)blockIdx.x * kCdfTile;
  if (e0 >= nnz) return;
  const int64_t e_last = e0 + kCdfTile - 1 < nnz ? e0 + kCdfTile - 1 : nnz - 1;
  float w[kCdfItems];
#pragma unroll
  for (int j = 0; j < kCdfItems; ++j) {
    const int64_t e = e0 + j * kBlock + threadIdx.x;
    w[j] = e <= e_last ? probs[e] : 0.0f;
  }
  const SegmentSpan span = segment_span(indptr, num_cols, e0, e_last);
  const int64_t nseg = span.hi - span.lo + 1;
  const bool in_lds = nseg <= kCdfSegs;
  if (in_lds) {
    for (int64_t j = threadIdx.x; j < nseg; j += kBlock) tile_max[j] = 0u;
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < kCdfItems; ++j) {
    const int64_t e = e0 + j * kBlock + threadIdx.x;
    if (e > e_last || !(w[j] > 0.0f)) continue;
    const int64_t c = span.segment_at(indptr, e);
    if (in_lds) atomicMax(&tile_max[c - span.lo], __float_as_uint(w[j]));
    else atomicMax(colmax_bits + c, __float_as_uint(w[j]));
  }
  if (!in_lds) return;
  __syncthreads();
  for (int64_t j = threadIdx.x; j < nseg; j += kBlock)
    if (tile_max[j] != 0u) atomicMax(colmax_bits + span.lo + j, tile_max[j]);
}

// prefix[e] = quantised weight of edge e (the device-wide scan that follows
// turns it into the sum of all quantised weights before e); prefix[nnz] = 0.
__global__ __launch_bounds__(kBlock) void cdf_quantise_kernel(
    const int64_t* __restrict__ indptr, int64_t num_cols,
    const float* __restrict__ probs, int64_t nnz,
    const unsigned int* __restrict__ colmax_bits, int64_t* __restrict__ prefix) {
  const int64_t e0 = (int64_t)blockIdx.x * kCdfTile;
  if (e0 > nnz) return;
  if (e0 == nnz) {  // prefix[nnz] = 0 closes the exclusive scan
    if (threadIdx.x == 0) prefix[nnz] = 0;
    return;
  }
  const int64_t e_last = e0 + kCdfTile - 1 < nnz ? e0 + kCdfTile - 1 : nnz - 1;
  const SegmentSpan span = segment_span(indptr, num_cols, e0, e_last);
#pragma unroll
  for (int j = 0; j < kCdfItems; ++j) {
    const int64_t e = e0 + j * kBlock + threadIdx.x;
    if (e > e_last) break;
    uint64_t q = 0;
    const float wmax = __uint_as_float(colmax_bits[span.segment_at(indptr, e)]);
    if (wmax > 0.0f) q = quantise(probs[e], det_div(2147483648.0, (double)wmax));
    prefix[e] = (int64_t)q;
  }
  if (e_last == nnz - 1 && threadIdx.x == 0) prefix[nnz] = 0;
}

__global__ __launch_bounds__(kBlock) void cdf_zero_kernel(unsigned int* p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// floor(a * 2^bits / t) for a < t < 2^63, by shift and subtract: exact integer
// arithmetic, so the CPU check (a 128-bit division) agrees to the bit.
__device__ __forceinline__ uint64_t scale_share(uint64_t a, uint64_t t, int bits) {
  uint64_t rem = a, q = 0;
  for (int i = 0; i < bits; ++i) {
    rem <<= 1;
    q <<= 1;
    if (rem >= t) {
      rem -= t;
      q |= 1ull;
    }
  }
  return q;
}

// prefix[] (global exclusive prefix sums of the quantised weights) -> entries.
__global__ __launch_bounds__(kBlock) void cdf_pack_kernel(
    const int64_t* __restrict__ indptr, int64_t num_cols,
    const int64_t* __restrict__ indices, int64_t nnz,
    const int64_t* __restrict__ prefix, int row_bits, uint64_t* __restrict__ cdf) {
  const int64_t e0 = (int64_t)blockIdx.x * kCdfTile;
  if (blockIdx.x == 0 && threadIdx.x == 0) cdf[0] = (uint64_t)row_bits;
  if (e0 >= nnz) return;
  const int64_t e_last = e0 + kCdfTile - 1 < nnz ? e0 + kCdfTile - 1 : nnz - 1;
  const SegmentSpan span = segment_span(indptr, num_cols, e0, e_last);
  const int cb = 64 - row_bits < 62 ? 64 - row_bits : 62;
  const uint64_t full = (1ull << cb) - 1ull;
  const uint64_t row_mask = row_bits ? (~0ull >> (64 - row_bits)) : 0ull;
#pragma unroll
  for (int j = 0; j < kCdfItems; ++j) {
    const int64_t e = e0 + j * kBlock + threadIdx.x;
    if (e > e_last) break;
    const int64_t c = span.segment_at(indptr, e);
    const uint64_t base = (uint64_t)prefix[indptr[c]];
    const uint64_t t = (uint64_t)prefix[indptr[c + 1]] - base;
    const uint64_t a = (uint64_t)prefix[e + 1] - base;
    const uint64_t share = a == t ? (t ? full : 0ull) : scale_share(a, t, cb);
    const uint64_t row = row_bits ? ((uint64_t)indices[e] & row_mask) : 0ull;
    cdf[e + 1] = (share << row_bits) | row;
  }
}

// Search of one draw over a column's entries col[1 .. deg] (col[j] is the entry of
// item j - 1, so its share is the point where item j starts): the item whose interval
// holds x is the last j in [0, deg) with start(j) <= x, for start(0) = 0 <= x <
// start(deg) = the column's mass.  Shares of weights are close to a straight line, so
// kInterpolations guesses interpolate; every later step is a plain bisection, which
// bounds the worst case for any weights.  Where a step looks never changes which item
// the search ends at.
//
// A step looks at a window of four entries by two 16-byte loads: the line is paid for
// by the first of them, and a draw ends after 2.0 dependent steps where one entry a
// step took 3.7 (the slowest of 64 lanes 4.3 and 8.2; columns of a power law, lognormal
// weights).  Windows lie at multiples of 32 bytes, so that they cross no line, but for
// those at a column's ends, which are moved inside it: every entry of a window is one of
// col[1 .. deg - 1], in order, so that one comparison an entry narrows both bounds.
//
// Positions are 32-bit from a base that the rare longer column is first bisected down
// to, entries are compared as they lie in memory (share above row id; `beyond` is the
// least entry that starts after x) and guesses are made from their upper words: a
// wavefront of fan-out 5 takes 2770 vector instructions where 64-bit positions, shares
// and guesses of double precision took 3960, 57 % of the issue slots.
constexpr int kInterpolations = 8;
constexpr int kWindow = 4;
typedef uint64_t EntryPair __attribute__((ext_vector_type(2), aligned(8)));
struct CdfSearch {
  int64_t base;       // item `lo` of the search is item base + lo of the column
  uint32_t lo, hi;    // the item lies in [lo, hi)
  uint64_t e_lo, e_hi;  // their entries (those of the column's bounds have no row id)
  __device__ __forceinline__ void narrow(uint32_t mid, uint64_t entry, uint64_t beyond) {
    if (entry < beyond) {
      lo = mid;
      e_lo = entry;
    } else {
      hi = mid;
      e_hi = entry;
    }
  }
};

// Leaves the item at s.base + s.lo, the entry it starts at in s.e_lo and the one it ends
// at, which carries its row id, in s.e_hi -- unless the search ended at the column's
// last item, whose entry it has not looked at (returns true).  `mass` is what the
// column's shares add up to.
__device__ __forceinline__ bool cdf_locate(CdfSearch& s, const uint64_t* __restrict__ col,
                                           int64_t deg, uint64_t mass, int row_bits,
                                           uint64_t x) {
  const uint64_t beyond = (x + 1) << row_bits;
  s.base = 0;
  s.e_lo = 0;
  s.e_hi = mass << row_bits;
  int64_t rest = deg;
  while (rest > 0x7FFFFFFFll) {
    const int64_t half = rest >> 1;
    const uint64_t entry = col[s.base + half];
    if (entry < beyond) {
      s.base += half;
      rest -= half;
      s.e_lo = entry;
    } else {
      rest = half;
      s.e_hi = entry;
    }
  }
  const uint64_t* at = col + s.base;
  s.lo = 0;
  s.hi = (uint32_t)rest;
  if (rest <= kWindow) {  // too short for a window
    while (s.hi - s.lo > 1) {
      const uint32_t mid = (s.lo + s.hi) >> 1;
      s.narrow(mid, at[mid], beyond);
    }
    return s.base + s.hi == deg;
  }
  // windows begin at 1 .. rest - kWindow; `shift` entries above a multiple of 32 bytes
  const uint32_t shift = (uint32_t)((uintptr_t)at >> 3) & (kWindow - 1);
  const uint32_t last = (uint32_t)rest - kWindow;
  int guesses = 0;
  while (s.hi - s.lo > 1) {
    uint32_t mid = (s.lo + s.hi) >> 1;
    if (guesses < kInterpolations) {
      ++guesses;
      const float part = (float)(uint32_t)((beyond - s.e_lo) >> 32) *
                         __builtin_amdgcn_rcpf((float)(uint32_t)((s.e_hi - s.e_lo) >> 32));
      // (0/0, of shares closer than the upper words tell apart, is a step of 1)
      const float range = (float)(s.hi - s.lo);
      const uint32_t step = (uint32_t)fminf(fmaxf(part * range, 1.0f), range);
      mid = s.lo + step < s.hi ? s.lo + step : s.hi - 1;
    }
    const uint32_t aligned = ((mid + shift) & ~(uint32_t)(kWindow - 1)) - shift;
    const uint32_t first = (uint32_t)min(max((int32_t)aligned, 1), (int32_t)last);
    const EntryPair p0 = *(const EntryPair*)(at + first);
    const EntryPair p1 = *(const EntryPair*)(at + first + 2);
    const bool b0 = p0.x < beyond, b1 = p0.y < beyond, b2 = p1.x < beyond, b3 = p1.y < beyond;
    const uint32_t count = (uint32_t)b0 + b1 + b2 + b3;
    if (b0) {
      s.lo = first + count - 1;
      s.e_lo = b3 ? p1.y : b2 ? p1.x : b1 ? p0.y : p0.x;
    }
    if (!b3) {
      s.hi = first + count;
      s.e_hi = !b0 ? p0.x : !b1 ? p0.y : !b2 ? p1.x : p1.y;
    }
  }
  return s.base + s.hi == deg;
}

constexpr int kMaxCdfFanout = 64;

// One lane per requested column.
// Without replacement: successive weighted sampling.  Draw j takes a uniform
// point r of the mass that is still there and maps it past the intervals of the
// items already taken (x = r + the lengths of all taken intervals that start at
// or before x, found by iterating from x = r), so no draw repeats an item and
// a column costs exactly fanout searches whatever its weights look like; when
// the positive mass runs out, zero-weight items follow in index order.
// An earlier version let a group of lanes search independent points of the
// whole mass at once and skipped repeats: columns whose degree or effective
// number of items is close to the fan-out then need several rounds, every round
// costs the whole wavefront a Philox block and a search per lane, and the
// bookkeeping of repeats alone was half of the kernel's time.
// With replacement: one independent point of the whole mass per output slot.
// Streams: pos = column position, draw = output slot.
// The taken intervals live in registers, in the order of their starts: every access
// runs over the slots with a predicate instead of indexing.
// The picks wait in LDS, packed as the wavefront's columns write them, and leave
// together at the end: neighbouring lanes then store neighbouring outputs, whole lines
// at a time (3.5 M columns with fanout 5: 4.5 M write requests of 64 bytes, 6.6 M when
// they were held in registers and stored by their own lanes, 33 M stored pick by pick).
// Work-groups are one wavefront where the picks of four would not leave room for others.
// What bounds it, 3.5 M columns of a 124 M-edge power-law graph, fanout 5: lines, 6.6 a
// column at 43 G/s of the part's 48; 540 us (698 with a search of one entry a step and
// the picks in registers).  592 K columns with fanout 10: 232 us (322), 65 K with fanout
// 15, one wavefront a SIMD and so its own chain of loads: 77 us (89).
// (Fan-outs up to 10 are capped at 128 registers, four wavefronts a SIMD: 250 us with
// three for fanout 10.  Three for fanout 5 leave more lines in L2 between the draws of a
// column, 5.7 a column, and take 607 us.  Non-temporal stores change nothing.)
template <int KMAX>
constexpr int kCdfThreads = KMAX <= 16 ? kBlock : kWave;

template <int KMAX, typename Row>
__global__ __launch_bounds__(kCdfThreads<KMAX>, KMAX <= 10 ? 4 : 1) void sample_weighted_cdf_kernel(
    const int64_t* __restrict__ indptr, int64_t num_cols,
    const int64_t* __restrict__ indices, const uint64_t* __restrict__ cdf,
    const int64_t* __restrict__ column_ids, int64_t num_items, int fanout,
    int replace, PhiloxKey key, const int64_t* __restrict__ sub_indptr,
    int64_t* __restrict__ out_coo_col, Row* __restrict__ out_indices,
    int64_t* __restrict__ out_select, ColumnLabels labels,
    const int64_t* __restrict__ col_span, const int64_t* __restrict__ num_dev) {
  constexpr int kThreads = kCdfThreads<KMAX>;
  __shared__ uint2 s_pick[kThreads * KMAX];  // offset in the column, row id
  __shared__ uint8_t s_owner[kThreads * KMAX];
  uint2* const wave_pick = s_pick + threadIdx.x / kWave * (kWave * KMAX);
  uint8_t* const wave_owner = s_owner + threadIdx.x / kWave * (kWave * KMAX);
  const int64_t item = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const bool live = item < (num_dev ? *num_dev : num_items);
  const int row_bits = (int)cdf[0];  // the same word for every lane: a scalar load
  const uint64_t row_mask = row_bits ? (~0ull >> (64 - row_bits)) : 0ull;
  int64_t col_label = item, in_start = 0, out_start = 0, deg = 0;
  if (live) {
    // (asked for here, so that its loads travel with the ones below)
    if (out_coo_col) col_label = labels.of_near(item, item - lane_id());
    deg = column_span(col_span, column_ids, indptr, num_cols, item, &in_start);
    // (without offsets every column has `fanout` places of its own)
    out_start = sub_indptr ? sub_indptr[item] : item * fanout;
  }
  const uint64_t* col = cdf + in_start;  // col[j], 1 <= j <= deg: entry of item j - 1
  // A column's shares add up to 2^cb - 1, or to 0 when it has no positive weight.
  // Which of the two is in the column's last entry, one more random line that a
  // column longer than the fan-out only reads when a search ends at its last item
  // (in a column without mass the first search does: every share is 0).
  const int cb = 64 - row_bits < 62 ? 64 - row_bits : 62;
  const uint64_t full = (1ull << cb) - 1ull;
  // What does not fit is written pick by pick: columns of 2^32 or more items (no graph
  // seen so far has one, nothing forbids it) and fanouts above KMAX, which only occur
  // with replacement.
  const bool hold = deg <= 0xFFFFFFFFll && fanout <= KMAX;
  const int64_t picks = deg == 0 ? 0 : replace || deg > fanout ? fanout : deg;
  const int held = hold ? (int)picks : 0;
  const int held_end = wave_inclusive_sum(held), held_at = held_end - held;
  auto pick_at = [&](int slot, int64_t off, uint64_t entry) {
    if (hold) {
      wave_pick[held_at + slot] = make_uint2((uint32_t)off, (uint32_t)(entry & row_mask));
      wave_owner[held_at + slot] = (uint8_t)lane_id();
      return;
    }
    const int64_t p = in_start + off;
    out_indices[out_start + slot] =
        (Row)(row_bits ? (int64_t)(entry & row_mask) : indices ? indices[p] : p);
    if (out_select) out_select[out_start + slot] = p;
    if (out_coo_col) out_coo_col[out_start + slot] = col_label;
  };
  CdfSearch s;
  if (deg == 0) {
  } else if (replace) {
    bool mass = true;
    for (int j = 0; j < fanout; ++j) {
      if (mass && cdf_locate(s, col, deg, full, row_bits,
                             philox_bounded(key, (uint64_t)item, (uint64_t)j, full))) {
        s.e_hi = col[deg];
        mass = (s.e_hi >> row_bits) != 0;
      }
      pick_at(j, mass ? s.base + s.lo : deg - 1, s.e_hi);  // no positive weight: the last item
    }
  } else if (deg <= fanout) {  // whole column, original order, zero weights included
    uint64_t entry[KMAX];
#pragma unroll
    for (int i = 0; i < KMAX; ++i) entry[i] = col[i < deg ? i + 1 : deg];
#pragma unroll
    for (int i = 0; i < KMAX; ++i)
      if (i < deg) pick_at(i, i, entry[i]);
  } else {
    // the intervals taken so far, in the order of their starts
    uint64_t start[KMAX], len[KMAX];
#pragma unroll
    for (int i = 0; i < KMAX; ++i) {
      start[i] = ~0ull;  // never at or before a point
      len[i] = 0;
    }
    uint64_t removed = 0;
    int taken = 0;
#pragma unroll 1
    for (int j = 0; j < fanout; ++j) {
      if (removed >= full) break;
      // a point of the mass that is left, moved past the intervals before it
      uint64_t x = philox_bounded(key, (uint64_t)item, (uint64_t)j, full - removed);
#pragma unroll
      for (int i = 0; i < KMAX; ++i)
        if (i < j) x += start[i] <= x ? len[i] : 0ull;
      if (cdf_locate(s, col, deg, full, row_bits, x)) {  // the last item's entry is unread
        s.e_hi = col[deg];
        if ((s.e_hi >> row_bits) == 0) break;  // a column without mass
      }
      uint64_t at = s.e_lo >> row_bits, length = (s.e_hi >> row_bits) - at;
      removed += length;
      pick_at(j, s.base + s.lo, s.e_hi);
      taken = j + 1;
#pragma unroll
      for (int i = 0; i < KMAX; ++i)
        if (i <= j) {
          const bool before = at < start[i];
          const uint64_t moved_start = start[i], moved_len = len[i];
          start[i] = before ? at : moved_start;
          len[i] = before ? length : moved_len;
          at = before ? moved_start : at;
          length = before ? moved_len : length;
        }
    }
    // fewer than fanout items have positive weight: zero-weight items in order
    if (taken < fanout) {
      uint64_t before = 0;
      for (int64_t off = 0; taken < fanout && off < deg; ++off) {
        const uint64_t entry = col[off + 1], here = entry >> row_bits;
        if (here == before) pick_at(taken++, off, entry);
        before = here;
      }
    }
  }
  // (the picks are shared among lanes of this wavefront only)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  __builtin_amdgcn_wave_barrier();
  const int total = __shfl(held_end, kWave - 1, kWave);
  const int64_t shift = out_start - held_at;
  for (int q0 = 0; q0 < total; q0 += kWave) {
    const int q = q0 + lane_id();
    const bool mine = q < total;
    const uint2 pick = mine ? wave_pick[q] : make_uint2(0, 0);
    const int owner = mine ? wave_owner[q] : 0;
    const int64_t to = __shfl(shift, owner, kWave) + q;
    const int64_t p = __shfl(in_start, owner, kWave) + pick.x;
    const int64_t label = __shfl(col_label, owner, kWave);
    if (!mine) continue;
    out_indices[to] = (Row)(row_bits ? (int64_t)pick.y : indices ? indices[p] : p);
    if (out_select) out_select[to] = p;
    if (out_coo_col) out_coo_col[to] = label;
  }
}

// The same picks where there are few columns: a column on sixteen neighbouring lanes.  A lane
// that owns its column goes through a chain of dependent loads for every draw, and where the
// device has no other wavefronts to run meanwhile, that chain is the time: 3 to 4.5 us a draw.
// Here the column's entries (of a longer one, kHeld of them at equal distances) are in LDS
// before the first draw, and a step of a search is one comparison by all lanes of a column and a
// count of those that hold.
//   draws      lane j's random number is draw j's
//   intervals  lane i holds the i-th of those taken, in the order of their starts: where it
//              starts in the mass that was left (`from`) and what it and those before it come
//              to (`sum`).  A point r of the mass that is left lies past as many of them as
//              have from <= r, and the new one is put in behind those
//   search     which of sixteen pieces of the held entries, which entry of that; in a column
//              of more than kHeld, sixteen entries a step from there on
constexpr int kTeam = 16;   // lanes of a column, and the most draws
constexpr int kHeld = 128;  // entries of a column in LDS
static_assert(kHeld % kTeam == 0 && kHeld / kTeam <= kTeam, "a lane for every entry of a piece");
// Columns per draw up to which a call goes this way.  A column costs a wavefront sixteen times
// the instructions, and of a long one up to kHeld lines are read however few the draws: with
// columns met by their degree (the frontiers of layers) in a graph of 2.45 M nodes and hubs of
// millions, us, a lane a column and this: fanout 5, 64 columns 17 and 11, 4096 20 and 19, 8192
// 20 and 24; fanout 10, 64 33 and 18, 8192 39 and 35, 16384 48 and 42, 32768 49 and 77; fanout
// 15, 64 63 and 23, 16384 84 and 55, 32768 83 and 99.  Columns met evenly gain up to four times as
// many.  (Windows of sixteen entries from a guess in place of the held ones of a long column:
// fanout 15, 64 columns 30, 32768 80.)
constexpr int64_t kTeamColumns = 1024;

template <typename Row>
__global__ __launch_bounds__(kBlock) void sample_weighted_team_kernel(
    const int64_t* __restrict__ indptr, int64_t num_cols,
    const int64_t* __restrict__ indices, const uint64_t* __restrict__ cdf,
    const int64_t* __restrict__ column_ids, int64_t num_items, int fanout, PhiloxKey key,
    const int64_t* __restrict__ sub_indptr, int64_t* __restrict__ out_coo_col,
    Row* __restrict__ out_indices, int64_t* __restrict__ out_select, ColumnLabels labels,
    const int64_t* __restrict__ col_span, const int64_t* __restrict__ num_dev) {
  constexpr int kPiece = kHeld / kTeam;
  __shared__ uint64_t s_held[kBlock / kTeam][kHeld];
  const int lane = lane_id(), t = lane % kTeam, team0 = lane - t;
  uint64_t* const held = s_held[threadIdx.x / kTeam];
  const int64_t item = (int64_t)blockIdx.x * (kBlock / kTeam) + threadIdx.x / kTeam;
  const int row_bits = (int)cdf[0];
  const uint64_t row_mask = row_bits ? (~0ull >> (64 - row_bits)) : 0ull;
  const int64_t id = column_ids ? column_ids[item < num_items ? item : num_items - 1] : item;
  if (item >= (num_dev ? *num_dev : num_items)) return;  // whole teams leave together
  int64_t col_label = item, in_start = 0;
  if (out_coo_col) col_label = labels.of_near(item, item - (threadIdx.x % kWave) / kTeam);
  const int64_t deg = col_span ? column_span(col_span, column_ids, indptr, num_cols, item, &in_start)
                               : column_degree(indptr, num_cols, id, &in_start);
  const int64_t out_start = sub_indptr ? sub_indptr[item] : item * fanout;
  const uint64_t* const col = cdf + in_start;  // col[j], 1 <= j <= deg: entry of item j - 1
  auto store = [&](int64_t slot, int64_t off, uint64_t entry) {
    const int64_t p = in_start + off;
    out_indices[out_start + slot] =
        (Row)(row_bits ? (int64_t)(entry & row_mask) : indices ? indices[p] : p);
    if (out_select) out_select[out_start + slot] = p;
    if (out_coo_col) out_coo_col[out_start + slot] = col_label;
  };
  if (deg <= fanout) {  // whole column, original order, zero weights included
    if (t < deg) store(t, t, col[t + 1]);
    return;
  }
  // lanes of this team for which it holds, counted
  auto count = [&](bool holds) {
    return (int)__popc((uint32_t)(__ballot(holds) >> team0) & ((1u << kTeam) - 1u));
  };
  // held[i]: the entry that ends stretch i of `step` entries
  const int64_t step = (deg + kHeld - 1) / kHeld;
  const int stretches = (int)((deg + step - 1) / step);
  uint64_t entry[kPiece];
#pragma unroll
  for (int i = 0; i < kPiece; ++i) {
    const int64_t end = (int64_t)(i * kTeam + t + 1) * step;
    entry[i] = col[end < deg ? end : deg];
  }
  const Words4 words = philox(key, (uint64_t)item, (uint64_t)t);
  const uint64_t random = ((uint64_t)words.y << 32) | words.x;
#pragma unroll
  for (int i = 0; i < kPiece; ++i) held[i * kTeam + t] = entry[i];
  // (by this wavefront's lanes only)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const uint64_t pivot = held[t * kPiece + kPiece - 1];
  const int cb = 64 - row_bits < 62 ? 64 - row_bits : 62;
  const uint64_t full = (1ull << cb) - 1ull;
  // (a column without mass has share 0 throughout)
  const bool mass = (held[stretches - 1] >> row_bits) != 0;
  uint64_t from = 0, sum = 0, removed = 0, my_entry = 0;
  int64_t my_off = 0;
  int taken = 0;
  while (mass && taken < fanout && removed < full) {
    const uint64_t r = __umul64hi(
        (uint64_t)__shfl((unsigned long long)random, team0 + taken, kWave), full - removed);
    const int before = count(t < taken && from <= r);
    const uint64_t skipped = before ? (uint64_t)__shfl((unsigned long long)sum, team0 + before - 1, kWave) : 0ull;
    // the first entry that starts after x ends the item that holds it
    const uint64_t beyond = (r + skipped + 1) << row_bits;
    const int piece = count(pivot < beyond);
    const uint64_t mine = held[(piece < kTeam ? piece : kTeam - 1) * kPiece + t % kPiece];
    const int at = piece * kPiece + count(t < kPiece && mine < beyond);
    int64_t off = at;
    uint64_t e_lo, e_hi;
    if (step == 1) {
      e_lo = at ? held[at - 1] : 0ull;
      e_hi = held[at];
    } else {
      int64_t lo = (int64_t)at * step;  // among entries lo + 1 to lo + len
      int64_t len = lo + step < deg ? step : deg - lo;
      while (len >= kTeam) {
        const int64_t part = (len + kTeam - 1) / kTeam;
        const int64_t end = (int64_t)(t + 1) * part < len ? (int64_t)(t + 1) * part : len;
        const int64_t passed = part * count(col[lo + end] < beyond);
        lo += passed;
        len = part < len - passed ? part : len - passed;
      }
      const uint64_t e = lo + t == 0 ? 0ull : col[lo + (t <= len ? t : len)];
      const int c = count(t >= 1 && t <= len && e < beyond);
      off = lo + c;
      e_lo = (uint64_t)__shfl((unsigned long long)e, team0 + c, kWave);
      e_hi = (uint64_t)__shfl((unsigned long long)e, team0 + c + 1, kWave);
    }
    const uint64_t start = e_lo >> row_bits, length = (e_hi >> row_bits) - start;
    const uint64_t from_up = (uint64_t)__shfl_up((unsigned long long)from, 1, kTeam);
    const uint64_t sum_up = (uint64_t)__shfl_up((unsigned long long)sum, 1, kTeam);
    if (t > before) {
      from = from_up - length;
      sum = sum_up + length;
    } else if (t == before) {
      from = start - skipped;
      sum = skipped + length;
    }
    if (t == taken) {
      my_off = off;
      my_entry = e_hi;
    }
    removed += length;
    ++taken;
  }
  if (t < taken) store(t, my_off, my_entry);
  // fewer than fanout items have positive weight: zero-weight items in order
  for (int64_t o = t; taken < fanout && o - t < deg; o += kTeam) {
    const uint64_t e = col[o < deg ? o + 1 : deg], prev = o == 0 ? 0ull : col[o < deg ? o : deg];
    const bool zero = o < deg && (e >> row_bits) == (prev >> row_bits);
    const uint32_t zeros = (uint32_t)(__ballot(zero) >> team0) & ((1u << kTeam) - 1u);
    const int slot = taken + (int)__popc(zeros & ((1u << t) - 1u));
    if (zero && slot < fanout) store(slot, o, e);
    taken += (int)__popc(zeros);
  }
}

template <int KMAX, typename Row>
static int launch_weighted_cdf(const int64_t* indptr, int64_t num_cols,
                               const int64_t* indices, const int64_t* cdf,
                               const int64_t* column_ids, int64_t num_items,
                               int fanout, int replace, PhiloxKey key,
                               const int64_t* sub_indptr, int64_t* out_coo_col,
                               Row* out_indices, int64_t* out_select,
                               ColumnLabels labels, const int64_t* col_span,
                               const int64_t* num_dev, hipStream_t s) {
  GS_LAUNCH("sample_weighted_cdf", s,
            (sample_weighted_cdf_kernel<KMAX, Row>)
                <<<dim3((unsigned)ceil_div(num_items, kCdfThreads<KMAX>)),
                   dim3(kCdfThreads<KMAX>), 0, s>>>(
                indptr, num_cols, indices, (const uint64_t*)cdf, column_ids, num_items,
                fanout, replace, key, sub_indptr, out_coo_col, out_indices, out_select, labels,
                col_span, num_dev));
  return GS_OK;
}

// (every slot of the register arrays costs instructions in every draw whether it is
// used or not: the common fan-outs get arrays of their own size)
template <typename Row>
static int launch_weighted_cdf_any(const int64_t* indptr, int64_t num_cols,
                                   const int64_t* indices, const int64_t* cdf,
                                   const int64_t* column_ids, int64_t num_items, int fanout,
                                   int replace, PhiloxKey key, const int64_t* sub_indptr,
                                   int64_t* out_coo_col, Row* out_indices,
                                   int64_t* out_select, ColumnLabels labels,
                                   const int64_t* col_span, const int64_t* num_dev,
                                   hipStream_t s) {
  if (!replace && fanout <= kTeam && num_items <= kTeamColumns * fanout) {
    GS_LAUNCH("sample_weighted_team", s,
              sample_weighted_team_kernel<Row>
                  <<<dim3((unsigned)ceil_div(num_items, kBlock / kTeam)), dim3(kBlock), 0, s>>>(
                      indptr, num_cols, indices, (const uint64_t*)cdf, column_ids, num_items, fanout,
                      key, sub_indptr, out_coo_col, out_indices, out_select, labels, col_span,
                      num_dev));
    return GS_OK;
  }
#define GS_CDF_ARGS                                                              \
  indptr, num_cols, indices, cdf, column_ids, num_items, fanout, replace, key, sub_indptr, \
      out_coo_col, out_indices, out_select, labels, col_span, num_dev, s
  if (fanout <= 4) return launch_weighted_cdf<4, Row>(GS_CDF_ARGS);
  if (fanout == 5) return launch_weighted_cdf<5, Row>(GS_CDF_ARGS);
  if (fanout <= 8) return launch_weighted_cdf<8, Row>(GS_CDF_ARGS);
  if (fanout <= 10) return launch_weighted_cdf<10, Row>(GS_CDF_ARGS);
  if (fanout <= 12) return launch_weighted_cdf<12, Row>(GS_CDF_ARGS);
  if (fanout <= 15) return launch_weighted_cdf<15, Row>(GS_CDF_ARGS);
  if (fanout <= 16) return launch_weighted_cdf<16, Row>(GS_CDF_ARGS);
  if (fanout <= 24) return launch_weighted_cdf<24, Row>(GS_CDF_ARGS);
  if (fanout <= 32) return launch_weighted_cdf<32, Row>(GS_CDF_ARGS);
  return launch_weighted_cdf<64, Row>(GS_CDF_ARGS);
#undef GS_CDF_ARGS
}

int launch_weighted_places(const int64_t* indptr, int64_t num_cols, const int64_t* indices,
                           const int64_t* cdf, const int64_t* column_ids, const int64_t* num_dev,
                           int64_t bound, int64_t fanout, int replace, PhiloxKey key,
                           int64_t* out_rows, hipStream_t s) {
  return launch_weighted_cdf_any(indptr, num_cols, indices, cdf, column_ids, bound, (int)fanout,
                                 replace, key, nullptr, nullptr, out_rows, nullptr,
                                 ColumnLabels{nullptr, 0}, nullptr, num_dev, s);
}

// Weighted picks of columns through the CDF, row ids of either width.
template <typename Row>
static int sample_weighted_by_cdf(const int64_t* indptr, int64_t num_cols, const int64_t* indices,
                                  const int64_t* cdf, const int64_t* column_ids, int64_t num_items,
                                  int64_t fanout, int replace, uint64_t seed, uint64_t call_id,
                                  const int64_t* sub_indptr, const int64_t* col_span,
                                  int64_t* out_coo_col, Row* out_indices, int64_t* out_select,
                                  const int64_t* col_batch_ptr, int64_t num_col_batches,
                                  gs_stream_t stream) {
  GS_REQUIRE(num_items >= 0 && num_cols >= 0, "sample_weighted: negative size");
  GS_REQUIRE(col_batch_ptr == nullptr || num_col_batches >= 1,
             "sample_weighted: col_batch_ptr given but num_col_batches = %lld",
             (long long)num_col_batches);
  GS_REQUIRE(fanout >= 0, "sample_weighted: negative fanout %lld", (long long)fanout);
  if (num_items == 0 || fanout == 0) return GS_OK;
  GS_REQUIRE(indptr && cdf && sub_indptr && out_indices, "sample_weighted: null pointer");
  GS_REQUIRE(column_ids != nullptr || num_items <= num_cols,
             "sample_weighted: %lld items but the matrix has %lld columns",
             (long long)num_items, (long long)num_cols);
  GS_REQUIRE(replace || fanout <= kMaxCdfFanout,
             "sample_weighted: fanout %lld > %d is not supported without replacement",
             (long long)fanout, kMaxCdfFanout);
  GS_REQUIRE(fanout <= INT32_MAX, "sample_weighted: fanout too large");
  return launch_weighted_cdf_any(indptr, num_cols, indices, cdf, column_ids, num_items, (int)fanout,
                                 replace, make_key(seed, call_id), sub_indptr, out_coo_col,
                                 out_indices, out_select,
                                 ColumnLabels{col_batch_ptr, num_col_batches}, col_span, nullptr,
                                 as_stream(stream));
}

// ------------------------------------------------------------ list sampling
__global__ __launch_bounds__(kBlock) void list_keys_kernel(
    const float* __restrict__ probs, int64_t n, PhiloxKey key,
    uint64_t* __restrict__ keys, int64_t* __restrict__ iota) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  // non-negative doubles (and +inf) order like their bit patterns
  keys[i] = (uint64_t)__double_as_longlong(weighted_key(key, (uint64_t)i, 0, probs[i]));
  iota[i] = i;
}

// Per segment: number of picks (replace: K for a non-empty segment; else
// min(K, n_b)).  One extra thread writes the trailing 0 for the scan.
__global__ void list_counts_kernel(const int64_t* __restrict__ range, int64_t n,
                                   int64_t nseg, int64_t num_picks, int replace,
                                   int64_t* __restrict__ counts) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b > nseg) return;
  int64_t cnt = 0;
  if (b < nseg) {
    const int64_t nb = range ? range[b + 1] - range[b] : n;
    cnt = replace ? (nb > 0 ? num_picks : 0) : (nb < num_picks ? nb : num_picks);
  }
  counts[b] = cnt;
}

// The same for at most kBlock - 1 segments, with the running sum: one launch
// instead of counts + scan.  words: zeroed as well (the selection's histograms and
// counters; a launch of its own for them takes 4.7 us in a row of launches).
__global__ __launch_bounds__(kBlock) void list_offsets_kernel(
    const int64_t* __restrict__ range, int64_t n, int64_t nseg, int64_t num_picks, int replace,
    int64_t* __restrict__ out_range, uint32_t* __restrict__ words, int64_t num_words) {
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < num_words;
       i += (int64_t)gridDim.x * kBlock)
    words[i] = 0u;
  if (blockIdx.x != 0) return;
  __shared__ int64_t smem[kBlock / kWave + 1];
  const int64_t b = threadIdx.x;
  int64_t cnt = 0;
  if (b < nseg) {
    const int64_t nb = range ? range[b + 1] - range[b] : n;
    cnt = replace ? (nb > 0 ? num_picks : 0) : (nb < num_picks ? nb : num_picks);
  }
  int64_t total;
  const int64_t before = block_exclusive_sum(cnt, smem, &total);
  if (b <= nseg) out_range[b] = before;
}

// Copies the first out_range[b+1] - out_range[b] sorted values of every
// segment; a segment that is taken whole keeps its original order.
__global__ __launch_bounds__(kBlock) void list_take_kernel(
    const int64_t* __restrict__ sorted_vals, const int64_t* __restrict__ range,
    int64_t n, int64_t nseg, int64_t num_picks,
    const int64_t* __restrict__ out_range, int64_t total,
    int64_t* __restrict__ out_index, const float* __restrict__ probs,
    float* __restrict__ out_value) {
  const int64_t o = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (o >= total) return;
  const int64_t b = nseg == 1 ? 0 : segment_of(out_range, nseg, o);
  const int64_t lo = range ? range[b] : 0;
  const int64_t nb = (range ? range[b + 1] : n) - lo;
  const int64_t k = o - out_range[b];
  const int64_t i = nb <= num_picks ? lo + k : sorted_vals[lo + k];
  out_index[o] = i;
  if (out_value) out_value[o] = probs[i];
}

// Integer CDF of a list segment by segment is a device-wide problem; segments
// are handled one wavefront each (layer-wise samplers have few, long segments
// at most a few hundred thousand items long).
__global__ __launch_bounds__(kBlock) void list_replace_kernel(
    const float* __restrict__ probs, const int64_t* __restrict__ range,
    int64_t n, int64_t nseg, int64_t num_picks, PhiloxKey key,
    const int64_t* __restrict__ out_range, uint64_t* cdf_scratch,
    int64_t* __restrict__ out_index, float* __restrict__ out_value) {
  const int lane = lane_id();
  const int64_t b = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / kWave;
  if (b >= nseg) return;
  const int64_t lo = range ? range[b] : 0, hi = range ? range[b + 1] : n;
  const int64_t nb = hi - lo;
  if (nb == 0) return;
  uint64_t* cdf = cdf_scratch + lo;
  float wmax = 0.0f;
  for (int64_t j = lane; j < nb; j += kWave) {
    const float w = probs[lo + j];
    if (w > wmax) wmax = w;
  }
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) {
    const float o = __shfl_xor(wmax, d, kWave);
    if (o > wmax) wmax = o;
  }
  const double scale = wmax > 0.0f ? det_div(2147483648.0, (double)wmax) : 0.0;
  uint64_t carry = 0;
  for (int64_t base = 0; base < nb; base += kWave) {
    const int64_t j = base + lane;
    uint64_t q = (j < nb && wmax > 0.0f) ? quantise(probs[lo + j], scale) : 0ull;
    q = wave_inclusive_sum(q);
    if (j < nb) cdf[j] = carry + q;
    carry += __shfl(q, kWave - 1, kWave);
  }
  const uint64_t total = carry;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  const int64_t out_start = out_range[b];
  for (int64_t k = lane; k < num_picks; k += kWave) {
    const uint64_t t = total > 0 ? philox_bounded(key, (uint64_t)b, (uint64_t)k, total) : 0ull;
    int64_t l = 0, h = nb;
    while (l < h) {
      const int64_t mid = (l + h) >> 1;
      const uint64_t v = __hip_atomic_load(cdf + mid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (v > t)
        h = mid;
      else
        l = mid + 1;
    }
    const int64_t i = lo + (l < nb ? l : nb - 1);
    out_index[out_start + k] = i;
    if (out_value) out_value[out_start + k] = probs[i];
  }
}

// Zeroes n 32-bit words (a kernel rather than a memset so that callers may
// capture the launches in a HIP graph).
__global__ __launch_bounds__(kBlock) void table_fill_kernel32(uint32_t* __restrict__ words,
                                                              int64_t n) {
  int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  for (; i < n; i += stride) words[i] = 0u;
}

// ---------------------------------------------- the K smallest keys by selection
// Without replacement the pick is "the K smallest keys, in ascending order, ties
// to the smaller index".  Sorting all n keys for that costs sixteen launches of
// a radix sort, and making them all is most of what is left: a key is two divisions
// and a logarithm of correctly rounded double operations, some hundred instructions.
// For K up to kSelMaxPicks the kernels below select by a cheap 32-bit key first:
//   bounds   an approximate key of every item (kept), off by less than kSelMargin of
//            itself, histogram of its exponent and 1 or 3 bits of its fraction per
//            segment
//   emit     the bin that holds the K-th smallest approximate key follows from that
//            histogram (every work-group scans it for itself); K items lie below the
//            bin's end, so no key above that end and the margin is among the K
//            smallest.  The others are the candidates, whose keys are computed and
//            appended to the segment's list
//   finish   a segment's candidates are ordered by (key, index) in LDS and the first K
//            written out (sixteen work-groups per segment share the comparisons)
// The number of keys below x grows no faster than x, so the candidates are about K times
// the width of a bin, 1.5 or 1.125, unless keys repeat; a list too long for LDS is
// narrowed by a byte-wise radix selection over keys and indices first.  Items of weight
// zero all have the key +inf: where picks come to them, a work-group leaves its own out
// if enough of them lie before it (100 K items, 300 of them positive, 400 picks: 710 us
// without that).
// 2.45 M items, 400 picks, us: keys 25, two levels of histograms 10 and 11 and finish 7
// when all keys were made; now bounds 13, emit 8, finish 6.
constexpr int kSelBins = 2048;
// Long segments: neighbouring work-groups add to one of eight histograms, and half as many
// items a work-group, twice as many of them, fill the device better than the adds to the same
// words cost.  One segment of 1 M, 2.45 M and 10 M items, 400, 400 and 1000 picks, all of the
// selection: 35, 38 and 93 us with one histogram and sixteen items a thread, 28, 35 and 73;
// shorter segments only pay for clearing and reading eight (20 K items 20 and 22, eight
// segments of 233 K 41 and 41).  Bounds alone is then at the instructions of its draws, 12 of
// 16 us at 2.45 M.
constexpr int kSelCopies = 8;
constexpr int64_t kSelLongSegment = int64_t(1) << 19;
constexpr int kSelTile = 4096;  // shortest average segment the selection takes on
constexpr int64_t kSelMaxPicks = 2048;
constexpr int kFinishThreads = 1024;
constexpr int kFinishSlots = 4096;
constexpr int kFinishSplit = 16;  // work-groups that share the ordering of one segment's picks

__host__ __device__ inline bool list_can_select(int64_t n, int64_t nseg) {
  return n < (int64_t(1) << 31) && (nseg == 1 || n / nseg >= kSelTile);
}

// Approximate keys.  Weights outside [2^-100, 2^100] go by their exact key, so that no
// intermediate overflows or loses bits; a result below 2^-126 may be flushed to 0, which
// is why no bound lies below kSelLeast.
constexpr float kSelMargin = 0x1p-10f;  // (2^-20.4 is the most met in 3 10^8 draws)
constexpr float kSelLeast = 0x1p-120f;

// -log2 of neg_log2_unit's argument, in 32 bits.
__device__ __forceinline__ float neg_log2_unit_approx(uint64_t r64) {
  const uint64_t v = (r64 >> 12) + 1;  // u = v / 2^52
  if (v >> 51) {                       // u >= 1/2: from 1 - u, which keeps its bits
    const uint64_t c = (1ull << 52) - v;
    const float t = fmaf((float)(uint32_t)(c >> 32), 0x1p-20f, (float)(uint32_t)c * 0x1p-52f);
    if (t < 0x1p-4f) {
      const float series =
          fmaf(t, fmaf(t, fmaf(t, fmaf(t, 0.2f, 0.25f), 0.33333334f), 0.5f), 1.0f);
      return 1.4426950f * t * series;
    }
    return -__builtin_amdgcn_logf(1.0f - t);
  }
  const float u = fmaf((float)(uint32_t)(v >> 32), 0x1p-20f, (float)(uint32_t)v * 0x1p-52f);
  return -__builtin_amdgcn_logf(u);
}

__device__ __forceinline__ float weighted_key_approx(PhiloxKey key, uint64_t pos, float w) {
  if (!(w > 0.0f)) return __uint_as_float(0x7f800000u);  // +inf
  if (!(w >= 0x1p-100f && w <= 0x1p100f)) {
    const double k = weighted_key(key, pos, 0, w);
    // (what is no number from 0 to +inf is ordered behind them by its bits)
    return k >= 0.0 && !(__double_as_longlong(k) < 0) ? (float)k : __uint_as_float(0x7f800000u);
  }
  const Words4 wd = philox(key, pos, 0);
  return neg_log2_unit_approx(((uint64_t)wd.y << 32) | wd.x) * __builtin_amdgcn_rcpf(w);
}

__device__ __forceinline__ uint32_t sel_bin(float k, int shift) {
  return __float_as_uint(k) >> shift;
}
// Keys above this are not among as many smallest as lie in the bins up to `bin`.
__device__ __forceinline__ float sel_bound(uint32_t bin, int shift) {
  const float end = __uint_as_float(bin + 1 < 0x7f800000u >> shift ? (bin + 1) << shift : 0x7f800000u);
  return fmaxf(end, kSelLeast) * (1.0f + 4.0f * kSelMargin);
}

// The bin of a kSelBins-bin histogram that holds the want-th smallest item
// (1-based, want <= number of items), and the number of items in the bins
// below it.  Called by the whole work-group; the result is the same in every
// thread.
__device__ __forceinline__ void find_bin(const uint32_t* __restrict__ hist, int copies,
                                         int64_t copy_words, int bins, uint32_t want,
                                         uint32_t* smem, uint32_t* found, uint32_t* bin,
                                         uint32_t* below) {
  constexpr int kPer = kSelBins / kBlock;
  const int first = threadIdx.x * kPer;
  uint32_t c[kPer] = {}, sum = 0;
  if (first < bins) {
    for (int copy = 0; copy < copies; ++copy)
#pragma unroll
      for (int j = 0; j < kPer; ++j) c[j] += hist[copy * copy_words + first + j];
#pragma unroll
    for (int j = 0; j < kPer; ++j) sum += c[j];
  }
  uint32_t total;
  uint32_t run = block_exclusive_sum(sum, smem, &total);
  const uint32_t target = want - 1;
  if (target >= run && target < run + sum) {
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      if (target >= run && target < run + c[j]) {
        found[0] = threadIdx.x * kPer + j;
        found[1] = run;
      }
      run += c[j];
    }
  }
  __syncthreads();
  *bin = found[0];
  *below = found[1];
  __syncthreads();
}

struct SelSegment {
  int64_t lo, hi;
};
__device__ __forceinline__ SelSegment sel_segment(const int64_t* __restrict__ range, int64_t n,
                                                  int64_t seg) {
  return range ? SelSegment{range[seg], range[seg + 1]} : SelSegment{0, n};
}
// A segment's candidates lie in kSelLists lists: neighbouring tiles share one, which begins where
// their items do and so has room for all of them.  Work-groups that append wait for one another
// by the counter's line, some 10 ns each: with one list a segment, its counters side by side, emit
// took 9.6 us on 2.45 M items and 400 picks, 14.3 on eight segments of 233 K and 256, 6.4 on one of
// 233 K and 512; with eight, a line each, 8.3, 10.4 and 5.7.
constexpr int kSelLists = 8;
constexpr int kSelCountStride = 32;  // words, a line of the L2
struct SelLists {
  int64_t lo;
  int tile_shift;             // items of a tile
  uint32_t first_tile, tiles;  // of the segment; of a list
  __device__ __forceinline__ SelLists(SelSegment sg, int shift)
      : lo(sg.lo), tile_shift(shift), first_tile((uint32_t)(sg.lo >> shift)) {
    tiles = ((uint32_t)((sg.hi - 1) >> shift) - first_tile + kSelLists) / kSelLists;
  }
  __device__ __forceinline__ int of_tile(uint32_t t) const {
    int list = 0;
#pragma unroll
    for (int c = 1; c < kSelLists; ++c) list += t - first_tile >= c * tiles;
    return list;
  }
  __device__ __forceinline__ int64_t begin(int list) const {
    return list == 0 ? lo : (int64_t)(first_tile + list * tiles) << tile_shift;
  }
  static __device__ __forceinline__ int64_t counter(int64_t seg, int list) {
    return (seg * kSelLists + list) * kSelCountStride;
  }
};
__device__ __forceinline__ SegmentSpan sel_span(const int64_t* __restrict__ range, int64_t nseg,
                                                int64_t i0, int64_t i_last) {
  return range ? segment_span(range, nseg, i0, i_last) : SegmentSpan{0, 0};
}

template <int kSelItems>
__global__ __launch_bounds__(kBlock) void list_bounds_kernel(
    const float* __restrict__ probs, const int64_t* __restrict__ range, int64_t n,
    int64_t nseg, PhiloxKey key, int shift, float* __restrict__ keys, uint32_t* hists, int copies,
    uint32_t* __restrict__ tile_never) {
  __shared__ uint32_t lh[kSelBins];
  __shared__ uint32_t never;
  uint32_t* hist = hists + (int64_t)(blockIdx.x % copies) * nseg * kSelBins;
  const int64_t i0 = (int64_t)blockIdx.x * (kBlock * kSelItems);
  const int64_t i_last = i0 + (kBlock * kSelItems) - 1 < n ? i0 + (kBlock * kSelItems) - 1 : n - 1;
  const SegmentSpan span = sel_span(range, nseg, i0, i_last);
  // all loads first, or each would be waited for inside its own branch
  float w[kSelItems];
#pragma unroll
  for (int j = 0; j < kSelItems; ++j) {
    const int64_t i = i0 + j * kBlock + threadIdx.x;
    w[j] = probs[i <= i_last ? i : i_last];
  }
  const int bins = (int)(0x80000000u >> shift);
  for (int b = threadIdx.x; b < bins; b += kBlock) lh[b] = 0;
  if (threadIdx.x == 0) never = 0;
  __syncthreads();
  uint32_t mine = 0;
#pragma unroll
  for (int j = 0; j < kSelItems; ++j)
    mine += (uint32_t)__popcll(__ballot(!(w[j] > 0.0f) && i0 + j * kBlock + threadIdx.x <= i_last));
  if (mine && lane_id() == 0) atomicAdd(&never, mine);
#pragma unroll
  for (int j = 0; j < kSelItems; ++j) {
    const int64_t i = i0 + j * kBlock + threadIdx.x;
    if (i > i_last) break;
    // non-negative floats (and +inf) order like their bit patterns
    const float k = weighted_key_approx(key, (uint64_t)i, w[j]);
    keys[i] = k;
    const int64_t seg = span.segment_at(range, i);
    if (seg == span.lo)
      atomicAdd(&lh[sel_bin(k, shift)], 1u);
    else
      atomicAdd(&hist[seg * kSelBins + sel_bin(k, shift)], 1u);
  }
  __syncthreads();
  if (threadIdx.x == 0) tile_never[blockIdx.x] = never;
  for (int b = threadIdx.x; b < bins; b += kBlock)
    if (lh[b]) atomicAdd(&hist[span.lo * kSelBins + b], lh[b]);
}

template <int kSelItems>
__global__ __launch_bounds__(kBlock) void list_emit_kernel(
    const float* __restrict__ probs, const int64_t* __restrict__ range, int64_t n, int64_t nseg,
    int64_t num_picks, PhiloxKey key, int shift, const float* __restrict__ keys,
    const uint32_t* __restrict__ hist, int copies, const uint32_t* __restrict__ tile_never,
    uint32_t* counts, uint64_t* __restrict__ cand_key, int64_t* __restrict__ cand_idx) {
  __shared__ uint32_t smem[kBlock / kWave + 1];
  __shared__ uint32_t found[2];
  __shared__ uint32_t base;
  const int64_t i0 = (int64_t)blockIdx.x * (kBlock * kSelItems);
  const int64_t i_last = i0 + (kBlock * kSelItems) - 1 < n ? i0 + (kBlock * kSelItems) - 1 : n - 1;
  // (loaded before the histogram is looked at, so that both travel together)
  float k[kSelItems];
#pragma unroll
  for (int j = 0; j < kSelItems; ++j) {
    const int64_t i = i0 + j * kBlock + threadIdx.x;
    k[j] = keys[i <= i_last ? i : i_last];
  }
  const SegmentSpan span = sel_span(range, nseg, i0, i_last);
  for (int64_t seg = span.lo; seg <= span.hi; ++seg) {  // the same in every thread
    const SelSegment sg = sel_segment(range, n, seg);
    if (sg.hi - sg.lo <= num_picks) continue;  // taken whole
    uint32_t bin, below;
    find_bin(hist + seg * kSelBins, copies, nseg * kSelBins, (int)(0x80000000u >> shift),
             (uint32_t)num_picks, smem, found, &bin, &below);
    const float bound = sel_bound(bin, shift);
    uint32_t is_cand = 0;  // one bit per item of this thread
#pragma unroll
    for (int j = 0; j < kSelItems; ++j) {
      const int64_t i = i0 + j * kBlock + threadIdx.x;
      if (i >= sg.lo && i < sg.hi && i <= i_last && k[j] <= bound) is_cand |= 1u << j;
    }
    if (bin == 0x7f800000u >> shift) {
      // Fewer positive weights than picks: items of weight zero follow in the order of
      // their indices.  Those of this tile do not if the tiles of the segment before it
      // have enough of them.
      constexpr int64_t kTile = kBlock * kSelItems;
      uint32_t before = 0, all;
      for (int64_t t = ceil_div_dev(sg.lo, kTile) + threadIdx.x; t < (int64_t)blockIdx.x; t += kBlock)
        before += tile_never[t];
      (void)block_exclusive_sum(before, smem, &all);
      if (all >= (uint32_t)num_picks)
        for (uint32_t left = is_cand; left; left &= left - 1) {
          const int j = __ffs((int)left) - 1;
          if (!(probs[i0 + j * kBlock + threadIdx.x] > 0.0f)) is_cand &= ~(1u << j);
        }
    }
    uint32_t cands;
    uint32_t at = block_exclusive_sum((uint32_t)__popc(is_cand), smem, &cands);
    const SelLists lists(sg, __builtin_ctz(kBlock * kSelItems));
    const int list = lists.of_tile(blockIdx.x);
    if (threadIdx.x == 0) base = cands ? atomicAdd(&counts[SelLists::counter(seg, list)], cands) : 0u;
    __syncthreads();
    const int64_t room = lists.begin(list);
    at += base;
    while (is_cand) {
      const int j = __ffs((int)is_cand) - 1;
      is_cand &= is_cand - 1;
      const int64_t i = i0 + j * kBlock + threadIdx.x;
      if (room + at < sg.hi) {  // always
        // non-negative doubles (and +inf) order like their bit patterns
        cand_key[room + at] =
            (uint64_t)__double_as_longlong(weighted_key(key, (uint64_t)i, 0, probs[i]));
        cand_idx[room + at] = i;
      }
      ++at;
    }
    __syncthreads();
  }
}

// (key, index) as one number.
__device__ __forceinline__ unsigned __int128 sel_composite(uint64_t k, int64_t i) {
  return ((unsigned __int128)k << 32) | (unsigned __int128)(uint32_t)i;
}

__global__ __launch_bounds__(kFinishThreads) void list_finish_kernel(
    const int64_t* __restrict__ range, int64_t n, int64_t num_picks, int tile_shift,
    const uint32_t* __restrict__ counts, const uint64_t* __restrict__ cand_key,
    const int64_t* __restrict__ cand_idx, const int64_t* __restrict__ out_range,
    int64_t* __restrict__ out_index, const float* __restrict__ probs,
    float* __restrict__ out_value) {
  auto pick = [&](int64_t at, int64_t i) {
    out_index[at] = i;
    if (out_value) out_value[at] = probs[i];
  };
  __shared__ uint64_t sk[kFinishSlots];
  __shared__ int64_t si[kFinishSlots];
  __shared__ uint32_t hist[256];
  __shared__ uint32_t chosen[2];
  __shared__ uint32_t appended;
  const int64_t seg = blockIdx.x;
  const SelSegment sg = sel_segment(range, n, seg);
  const int64_t nb = sg.hi - sg.lo, out0 = out_range[seg];
  uint32_t many[kSelLists];
#pragma unroll
  for (int c = 0; c < kSelLists; ++c) many[c] = counts[SelLists::counter(seg, c)];
  if (nb <= num_picks) {  // taken whole, in the original order
    if (blockIdx.y == 0)
      for (int64_t k = threadIdx.x; k < nb; k += kFinishThreads) pick(out0 + k, sg.lo + k);
    return;
  }
  // (no list is longer than its segment; restated here because indices follow from it)
  const SelLists lists(sg, tile_shift);
  uint32_t M = 0, list_end[kSelLists];
#pragma unroll
  for (int c = 0; c < kSelLists; ++c) {
    const int64_t room = sg.hi - lists.begin(c);
    M += room <= 0 ? 0u : (int64_t)many[c] < room ? many[c] : (uint32_t)room;
    list_end[c] = M;
  }
  auto place = [&](uint32_t t) {
    int list = 0;
    uint32_t before = 0;
#pragma unroll
    for (int c = 0; c + 1 < kSelLists; ++c)
      if (t >= list_end[c]) {
        list = c + 1;
        before = list_end[c];
      }
    return lists.begin(list) + (t - before);
  };
  uint32_t total = M;
  if (total <= (uint32_t)kFinishSlots) {
    for (uint32_t t = threadIdx.x; t < M; t += kFinishThreads) {
      const int64_t at = place(t);
      sk[t] = cand_key[at];
      si[t] = cand_idx[at];
    }
  } else {
    // the `want` smallest of the M candidates: fix the composite of the last
    // of them byte by byte, most significant first
    uint32_t want = (uint32_t)num_picks;
    unsigned __int128 fixed = 0;
    for (int d = 0; d < 12; ++d) {
      const int shift = 8 * (11 - d);
      for (int b = threadIdx.x; b < 256; b += kFinishThreads) hist[b] = 0;
      __syncthreads();
      for (uint32_t t = threadIdx.x; t < M; t += kFinishThreads) {
        const int64_t at = place(t);
        const unsigned __int128 c = sel_composite(cand_key[at], cand_idx[at]);
        if ((c >> (shift + 8)) == (fixed >> (shift + 8)))
          atomicAdd(&hist[(uint32_t)(c >> shift) & 255u], 1u);
      }
      __syncthreads();
      if (threadIdx.x == 0) {
        uint32_t run = 0, b = 0;
        for (; b < 255 && run + hist[b] < want; ++b) run += hist[b];
        chosen[0] = b;
        chosen[1] = run;
      }
      __syncthreads();
      fixed |= (unsigned __int128)chosen[0] << shift;
      want -= chosen[1];
      __syncthreads();
    }
    if (threadIdx.x == 0) appended = 0;
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < M; t += kFinishThreads) {
      const int64_t from = place(t);
      const uint64_t k = cand_key[from];
      const int64_t i = cand_idx[from];
      if (sel_composite(k, i) <= fixed) {
        const uint32_t at = atomicAdd(&appended, 1u);
        if (at < (uint32_t)kFinishSlots) {
          sk[at] = k;
          si[at] = i;
        }
      }
    }
    total = (uint32_t)num_picks;
  }
  __syncthreads();
  // Order by (key, index): the rank of an item is the number of smaller ones.
  // The kFinishSplit work-groups of a segment all hold all items and each ranks
  // its share of them (shares go by index, so that they do not depend on the
  // order the lists were filled in): the comparisons (the square of the number
  // of items) are more than one compute unit should do alone.  A wavefront takes four of the
  // work-group's items and compares them with 64 others at a time, whose keys are loaded once
  // for the four (a thread for an item and an eighth of the others, which read them one after
  // the other, took 6.6 of 11 us with 630 items and 5.0 of 8 with 452; now 8.7 and 5.4 in all).
  __shared__ uint16_t my_items[kFinishSlots];
  if (threadIdx.x == 0) appended = 0;
  __syncthreads();
  for (uint32_t t = threadIdx.x; t < total; t += kFinishThreads)
    if ((uint32_t)si[t] % kFinishSplit == blockIdx.y) my_items[atomicAdd(&appended, 1u)] = (uint16_t)t;
  __syncthreads();
  const uint32_t mine = appended;
  constexpr uint32_t kItems = 4, kWaves = kFinishThreads / kWave;
  const uint32_t lane = (uint32_t)lane_id(), wave = threadIdx.x / kWave;
  // (as many a wavefront as give every one some)
  const uint32_t each = mine > kWaves * (kItems - 1) ? kItems : (mine + kWaves - 1) / kWaves;
  for (uint32_t m0 = wave * each; m0 < mine; m0 += kWaves * each) {
    uint64_t k[kItems];
    int64_t i[kItems];
    uint32_t rank[kItems];
#pragma unroll
    for (uint32_t j = 0; j < kItems; ++j) {
      const uint32_t t = my_items[m0 + j < mine ? m0 + j : m0];
      k[j] = sk[t];
      i[j] = si[t];
      rank[j] = 0;
    }
    for (uint32_t o = lane; o < total + lane; o += kWave) {  // the same rounds for every lane
      const uint32_t at = o < total ? o : total - 1;
      const uint64_t ko = sk[at];
      const int64_t io = si[at];
#pragma unroll
      for (uint32_t j = 0; j < kItems; ++j)
        if (j < each)
          rank[j] += (uint32_t)__popcll(__ballot(o < total && (ko < k[j] || (ko == k[j] && io < i[j]))));
    }
    // lane j writes item j
    uint32_t r = rank[0];
    int64_t index = i[0];
#pragma unroll
    for (uint32_t j = 1; j < kItems; ++j)
      if (lane == j) {
        r = rank[j];
        index = i[j];
      }
    if (lane < each && m0 + lane < mine && r < (uint32_t)num_picks) pick(out0 + r, index);
  }
}

struct ListWs {
  uint64_t *keys_in, *keys_out;  // also the CDF scratch when sampling with replacement
  int64_t *vals_in, *vals_out;
  void* sort_ws;
  size_t sort_ws_bytes;
  void* scan_ws;
  size_t scan_ws_bytes;
  // selection (list_can_select): histograms, then counters, in one block; the
  // approximate keys lie in keys_in
  uint32_t* sel_block;
  size_t sel_words;
  uint32_t *hist, *counts, *tile_never;
  int copies;  // of the histograms, [copies][segments][kSelBins]
  size_t total;
};

static size_t sort_temp_bytes(int64_t n, int64_t nseg) {
  size_t flat = 0, seg = 0;
  uint64_t* k = nullptr;
  int64_t* v = nullptr;
  (void)rocprim::radix_sort_pairs(nullptr, flat, k, k, v, v, (size_t)(n > 0 ? n : 1), 0, 64);
  const int64_t* off = nullptr;
  (void)rocprim::segmented_radix_sort_pairs(nullptr, seg, k, k, v, v, (size_t)(n > 0 ? n : 1),
                                            (unsigned)(nseg > 0 ? nseg : 1), off, off, 0, 64);
  return flat > seg ? flat : seg;
}

static ListWs carve_list(void* ws, int64_t n, int64_t nseg) {
  Carver c(ws);
  ListWs w;
  const size_t m = (size_t)(n > 0 ? n : 1);
  w.keys_in = c.take<uint64_t>(m);
  w.keys_out = c.take<uint64_t>(m);
  w.vals_in = c.take<int64_t>(m);
  w.vals_out = c.take<int64_t>(m);
  w.sort_ws_bytes = sort_temp_bytes(n, nseg);
  w.sort_ws = c.take<char>(w.sort_ws_bytes);
  w.scan_ws_bytes = scan_workspace_bytes(nseg + 1);
  w.scan_ws = c.take<char>(w.scan_ws_bytes);
  const size_t segs = list_can_select(n, nseg) ? (size_t)nseg : 0;
  w.copies = nseg > 0 && n / nseg >= kSelLongSegment ? kSelCopies : 1;
  w.sel_words = segs * ((size_t)w.copies * kSelBins + kSelLists * kSelCountStride);
  w.sel_block = c.take<uint32_t>(w.sel_words);
  w.hist = w.sel_block;
  w.counts = w.hist ? w.hist + segs * w.copies * kSelBins : nullptr;
  w.tile_never = c.take<uint32_t>(segs ? m / (kBlock * 4) + 1 : 0);
  w.total = c.total();
  return w;
}

}  // namespace gs

extern "C" {

int gs_weighted_key_probe(uint64_t seed, uint64_t call_id, uint64_t pos,
                          uint64_t draw, float w, uint64_t r64, double* out2,
                          gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(out2, "weighted_key_probe: null output");
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("weighted_key_probe", s,
            weighted_key_probe_kernel<<<dim3(1), dim3(1), 0, s>>>(
                make_key(seed, call_id), pos, draw, w, r64, out2));
  return GS_OK;
}

size_t gs_weight_cdf_workspace_bytes(int64_t num_cols, int64_t nnz) {
  if (num_cols < 0 || nnz < 0) return 0;
  return gs::align_up((size_t)(num_cols > 0 ? num_cols : 1) * sizeof(unsigned int), 256) +
         gs::align_up((size_t)(nnz + 1) * sizeof(int64_t), 256) +
         gs::scan_workspace_bytes(nnz + 1);
}

int gs_weight_cdf_build(const int64_t* indptr, int64_t num_cols, const int64_t* indices,
                        int64_t num_rows, const float* probs, int64_t nnz, int64_t* cdf,
                        void* workspace, size_t workspace_bytes, gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(num_cols >= 0 && nnz >= 0, "weight_cdf_build: negative size");
  GS_REQUIRE(cdf && (nnz == 0 || (indptr && probs)), "weight_cdf_build: null pointer");
  GS_REQUIRE(indices == nullptr || num_rows >= 0, "weight_cdf_build: negative num_rows");
  const size_t need = gs_weight_cdf_workspace_bytes(num_cols, nnz);
  if (workspace == nullptr || workspace_bytes < need) {
    set_error("weight_cdf_build workspace too small: %zu < %zu", workspace_bytes, need);
    return GS_ERR_WORKSPACE;
  }
  // bits that hold any row id below num_rows; ids too wide to share an entry
  // with a useful share stay in `indices`
  int row_bits = 0;
  if (indices != nullptr) {
    row_bits = 1;
    while (row_bits < 63 && (int64_t(1) << row_bits) < num_rows) ++row_bits;
    if (row_bits > kCdfMaxRowBits) row_bits = 0;
  }
  hipStream_t s = as_stream(stream);
  unsigned int* colmax = (unsigned int*)workspace;
  const size_t colmax_bytes =
      align_up((size_t)(num_cols > 0 ? num_cols : 1) * sizeof(unsigned int), 256);
  int64_t* prefix = (int64_t*)((char*)workspace + colmax_bytes);
  const size_t prefix_bytes = align_up((size_t)(nnz + 1) * sizeof(int64_t), 256);
  void* scan_ws = (char*)prefix + prefix_bytes;
  if (num_cols > 0)
    GS_LAUNCH("cdf_zero", s,
              cdf_zero_kernel<<<dim3((unsigned)ceil_div(num_cols, kBlock)), dim3(kBlock),
                                0, s>>>(colmax, num_cols));
  if (nnz > 0)
    GS_LAUNCH("cdf_colmax", s,
              cdf_colmax_kernel<<<dim3((unsigned)ceil_div(nnz, kCdfTile)), dim3(kBlock), 0,
                                  s>>>(indptr, num_cols, probs, nnz, colmax));
  GS_LAUNCH("cdf_quantise", s,
            cdf_quantise_kernel<<<dim3((unsigned)ceil_div(nnz + 1, kCdfTile)), dim3(kBlock),
                                  0, s>>>(indptr, num_cols, probs, nnz, colmax, prefix));
  const int rc = exclusive_scan_i64(prefix, prefix, nnz + 1, scan_ws,
                                    workspace_bytes - colmax_bytes - prefix_bytes, s);
  if (rc != GS_OK) return rc;
  GS_LAUNCH("cdf_pack", s,
            cdf_pack_kernel<<<dim3((unsigned)ceil_div(nnz > 0 ? nnz : 1, kCdfTile)),
                              dim3(kBlock), 0, s>>>(indptr, num_cols, indices, nnz, prefix,
                                                    row_bits, (uint64_t*)cdf));
  return GS_OK;
}

int gs_csc_col_sample_weighted_fill(
    const int64_t* indptr, int64_t num_cols, const int64_t* indices,
    const float* probs, const int64_t* cdf,
    const int64_t* column_ids, int64_t num_items,
    int64_t fanout, int replace, uint64_t seed, uint64_t call_id,
    const int64_t* sub_indptr, const int64_t* col_span, const int64_t* cdf_offsets,
    void* cdf_scratch,
    int64_t* out_coo_col, int64_t* out_indices, int64_t* out_select,
    const int64_t* col_batch_ptr, int64_t num_col_batches, gs_stream_t stream) {
  using namespace gs;
  if (cdf != nullptr)
    return sample_weighted_by_cdf<int64_t>(indptr, num_cols, indices, cdf, column_ids, num_items,
                                           fanout, replace, seed, call_id, sub_indptr, col_span,
                                           out_coo_col, out_indices, out_select, col_batch_ptr,
                                           num_col_batches, stream);
  GS_REQUIRE(num_items >= 0 && num_cols >= 0, "sample_weighted: negative size");
  GS_REQUIRE(col_batch_ptr == nullptr || num_col_batches >= 1,
             "sample_weighted: col_batch_ptr given but num_col_batches = %lld",
             (long long)num_col_batches);
  const ColumnLabels labels{col_batch_ptr, num_col_batches};
  GS_REQUIRE(fanout >= 0, "sample_weighted: negative fanout %lld", (long long)fanout);
  if (num_items == 0 || fanout == 0) return GS_OK;
  GS_REQUIRE(indptr && probs && sub_indptr && out_indices && out_select,
             "sample_weighted: null pointer");
  GS_REQUIRE(column_ids != nullptr || num_items <= num_cols,
             "sample_weighted: %lld items but the matrix has %lld columns",
             (long long)num_items, (long long)num_cols);
  const PhiloxKey key = make_key(seed, call_id);
  hipStream_t s = as_stream(stream);
  if (replace) {
    GS_REQUIRE(cdf_scratch, "sample_weighted: sampling with replacement needs the CDF scratch");
    GS_REQUIRE(column_ids == nullptr || cdf_offsets != nullptr,
               "sample_weighted: cdf_offsets are required with column_ids");
    GS_LAUNCH("sample_weighted_replace", s,
              sample_weighted_replace_kernel<<<dim3((unsigned)ceil_div(num_items, kReplWaves)),
                                               dim3(kReplThreads), 0, s>>>(
                  indptr, num_cols, indices, probs, column_ids, num_items, fanout,
                  key, sub_indptr, cdf_offsets, (uint64_t*)cdf_scratch, out_coo_col,
                  out_indices, out_select, labels));
    return GS_OK;
  }
  GS_REQUIRE(fanout <= 64,
             "sample_weighted: fanout %lld > 64 is not supported without replacement",
             (long long)fanout);
  const int threads = fanout <= 32 ? kBlock : kBlock / 2;
  const size_t lds = (size_t)fanout * threads * (sizeof(double) + sizeof(int));
  static bool raised = false;
  if (!raised) {
    GS_HIP(hipFuncSetAttribute((const void*)sample_weighted_kernel,
                               hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024));
    raised = true;
  }
  const int64_t blocks = ceil_div(num_items * kWave, threads);
  GS_LAUNCH("sample_weighted", s,
            sample_weighted_kernel<<<dim3((unsigned)blocks), dim3(threads), lds, s>>>(
                indptr, num_cols, indices, probs, column_ids, num_items,
                (int)fanout, key, sub_indptr, out_coo_col, out_indices,
                out_select, labels));
  return GS_OK;
}

int gs_csc_col_sample_weighted_fill_rows32(
    const int64_t* indptr, int64_t num_cols, const int64_t* indices, const int64_t* cdf,
    const int64_t* column_ids, int64_t num_items, int64_t fanout, int replace, uint64_t seed,
    uint64_t call_id, const int64_t* sub_indptr, const int64_t* col_span, int64_t* out_coo_col,
    int32_t* out_rows, const int64_t* col_batch_ptr, int64_t num_col_batches, gs_stream_t stream) {
  // (without row ids the kernels hand on positions of edges, which have no such bound)
  GS_REQUIRE(indices, "sample_weighted_rows32: null indices");
  return gs::sample_weighted_by_cdf<int32_t>(indptr, num_cols, indices, cdf, column_ids, num_items,
                                             fanout, replace, seed, call_id, sub_indptr, col_span,
                                             out_coo_col, out_rows, nullptr, col_batch_ptr,
                                             num_col_batches, stream);
}

size_t gs_list_sample_workspace_bytes(int64_t n, int64_t num_segments) {
  if (n < 0 || num_segments < 1) return 0;
  return gs::carve_list(nullptr, n, num_segments).total;
}

int gs_list_sample_weighted_count(const int64_t* range, int64_t n,
                                  int64_t num_segments, int64_t num_picks,
                                  int replace, int64_t* out_range,
                                  void* workspace, size_t workspace_bytes,
                                  gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(n >= 0 && num_segments >= 1 && num_picks >= 0,
             "list_sample_count: bad sizes");
  GS_REQUIRE(range != nullptr || num_segments == 1,
             "list_sample_count: %lld segments need a range array", (long long)num_segments);
  GS_REQUIRE(out_range, "list_sample_count: null out_range");
  ListWs w = carve_list(workspace, n, num_segments);
  if (workspace == nullptr || workspace_bytes < w.total) {
    set_error("list_sample workspace too small: %zu < %zu", workspace_bytes, w.total);
    return GS_ERR_WORKSPACE;
  }
  hipStream_t s = as_stream(stream);
  if (num_segments < kBlock) {
    GS_LAUNCH("list_counts", s,
              list_offsets_kernel<<<dim3(1), dim3(kBlock), 0, s>>>(
                  range, n, num_segments, num_picks, replace, out_range, nullptr, 0));
    return GS_OK;
  }
  GS_LAUNCH("list_counts", s,
            list_counts_kernel<<<dim3((unsigned)ceil_div(num_segments + 1, kBlock)),
                                 dim3(kBlock), 0, s>>>(range, n, num_segments,
                                                       num_picks, replace, out_range));
  return exclusive_scan_i64(out_range, out_range, num_segments + 1, w.scan_ws,
                            w.scan_ws_bytes, s);
}

// Whether the picks go by selection.
static bool list_selects(int64_t n, int64_t num_segments, int64_t num_picks, int replace) {
  return !replace && num_picks >= 1 && num_picks <= gs::kSelMaxPicks &&
         gs::list_can_select(n, num_segments);
}
static dim3 list_zero_grid(const gs::ListWs& w) {
  return dim3((unsigned)gs::ceil_div((int64_t)w.sel_words, gs::kBlock * 8));
}

// zeroed: the selection's histograms and counters are zero already.
static int list_fill(const float* probs, const int64_t* range, int64_t n, int64_t num_segments,
                     int64_t num_picks, int replace, uint64_t seed, uint64_t call_id,
                     const int64_t* out_range, int64_t total_picks, int64_t* out_index,
                     float* out_value, void* workspace, size_t workspace_bytes,
                     gs_stream_t stream, bool zeroed) {
  using namespace gs;
  GS_REQUIRE(n >= 0 && num_segments >= 1 && num_picks >= 0 && total_picks >= 0,
             "list_sample_fill: bad sizes");
  if (total_picks == 0 || n == 0) return GS_OK;
  GS_REQUIRE(probs && out_range && out_index, "list_sample_fill: null pointer");
  GS_REQUIRE(range != nullptr || num_segments == 1,
             "list_sample_fill: %lld segments need a range array", (long long)num_segments);
  ListWs w = carve_list(workspace, n, num_segments);
  if (workspace == nullptr || workspace_bytes < w.total) {
    set_error("list_sample workspace too small: %zu < %zu", workspace_bytes, w.total);
    return GS_ERR_WORKSPACE;
  }
  const PhiloxKey key = make_key(seed, call_id);
  hipStream_t s = as_stream(stream);
  if (replace) {
    GS_LAUNCH("list_replace", s,
              list_replace_kernel<<<dim3((unsigned)ceil_div(num_segments * kWave, kBlock)),
                                    dim3(kBlock), 0, s>>>(
                  probs, range, n, num_segments, num_picks, key, out_range,
                  w.keys_in, out_index, out_value));
    return GS_OK;
  }
  if (list_selects(n, num_segments, num_picks, replace)) {
    // few items per thread while that still fills the device, else sixteen (fewer
    // work-groups meet at the same histogram bins), eight where there are copies of those
    // or sixteen would leave less than four work-groups a compute unit (256 picks of 1.05 M
    // items, kernels of a call in us with sixteen and with eight: in 8 segments 54 and 47, in 64
    // 64 and 57; of 2.45 M 57 and 50, 66 and 60; of 4.19 M 69 and 63, 75 and 71; with 1024 picks
    // of 3.5 M in 8 segments, the worst of 64 to 1024 picks, 69 and 70)
    const int items = n < (int64_t(1) << 20) ? 4 : w.copies > 1 || n < (int64_t(1) << 22) ? 8 : 16;
    // bins half a power of two wide, an eighth where many picks make candidates dear
    // (they are compared with one another): 233 K items 24 and 27 us with 400 picks, 69
    // and 58 with 2048
    const int shift = num_picks <= 512 ? 22 : 20;
    const dim3 tiles((unsigned)ceil_div(n, kBlock * items));
    if (!zeroed)
      GS_LAUNCH("list_zero", s,
                table_fill_kernel32<<<list_zero_grid(w), dim3(kBlock), 0, s>>>(
                    w.sel_block, (int64_t)w.sel_words));
#define GS_SEL_LAUNCH(name, kernel, ...)                                              \
  GS_LAUNCH(name, s,                                                                  \
            if (items == 16) kernel<16><<<tiles, dim3(kBlock), 0, s>>>(__VA_ARGS__);     \
            else if (items == 8) kernel<8><<<tiles, dim3(kBlock), 0, s>>>(__VA_ARGS__);  \
            else kernel<4><<<tiles, dim3(kBlock), 0, s>>>(__VA_ARGS__))
    GS_SEL_LAUNCH("list_bounds", list_bounds_kernel, probs, range, n, num_segments, key, shift,
                  (float*)w.keys_in, w.hist, w.copies, w.tile_never);
    GS_SEL_LAUNCH("list_emit", list_emit_kernel, probs, range, n, num_segments, num_picks, key, shift,
                  (const float*)w.keys_in, w.hist, w.copies, w.tile_never, w.counts, w.keys_out, w.vals_out);
#undef GS_SEL_LAUNCH
    GS_LAUNCH("list_finish", s,
              list_finish_kernel<<<dim3((unsigned)num_segments, kFinishSplit), dim3(kFinishThreads), 0, s>>>(
                  range, n, num_picks, __builtin_ctz(kBlock * items), w.counts, w.keys_out, w.vals_out,
                  out_range, out_index, probs, out_value));
    return GS_OK;
  }
  GS_LAUNCH("list_keys", s,
            list_keys_kernel<<<dim3((unsigned)ceil_div(n, kBlock)), dim3(kBlock), 0, s>>>(
                probs, n, key, w.keys_in, w.vals_in));
  size_t temp = w.sort_ws_bytes;
  {
    ProfScope ps("list_sort", s);
    if (num_segments == 1) {
      GS_HIP(rocprim::radix_sort_pairs(w.sort_ws, temp, w.keys_in, w.keys_out,
                                       w.vals_in, w.vals_out, (size_t)n, 0, 64, s));
    } else {
      GS_HIP(rocprim::segmented_radix_sort_pairs(
          w.sort_ws, temp, w.keys_in, w.keys_out, w.vals_in, w.vals_out,
          (size_t)n, (unsigned)num_segments, range, range + 1, 0, 64, s));
    }
  }
  GS_LAUNCH("list_take", s,
            list_take_kernel<<<dim3((unsigned)ceil_div(total_picks, kBlock)),
                               dim3(kBlock), 0, s>>>(w.vals_out, range, n,
                                                     num_segments, num_picks,
                                                     out_range, total_picks,
                                                     out_index, probs, out_value));
  return GS_OK;
}

int gs_list_sample_weighted_fill(const float* probs, const int64_t* range,
                                 int64_t n, int64_t num_segments,
                                 int64_t num_picks, int replace, uint64_t seed,
                                 uint64_t call_id, const int64_t* out_range,
                                 int64_t total_picks, int64_t* out_index,
                                 void* workspace, size_t workspace_bytes,
                                 gs_stream_t stream) {
  return list_fill(probs, range, n, num_segments, num_picks, replace, seed, call_id, out_range,
                   total_picks, out_index, nullptr, workspace, workspace_bytes, stream, false);
}

int gs_list_sample_weighted(const float* probs, const int64_t* range, int64_t n,
                            int64_t num_segments, int64_t num_picks, int replace, uint64_t seed,
                            uint64_t call_id, int64_t* out_range, int64_t total_picks,
                            int64_t* out_index, void* workspace, size_t workspace_bytes,
                            gs_stream_t stream) {
  return gs_list_sample_weighted_values(probs, range, n, num_segments, num_picks, replace, seed,
                                        call_id, out_range, total_picks, out_index, nullptr,
                                        workspace, workspace_bytes, stream);
}

int gs_list_sample_weighted_values(const float* probs, const int64_t* range, int64_t n,
                                   int64_t num_segments, int64_t num_picks, int replace,
                                   uint64_t seed, uint64_t call_id, int64_t* out_range,
                                   int64_t total_picks, int64_t* out_index, float* out_value,
                                   void* workspace, size_t workspace_bytes, gs_stream_t stream) {
  using namespace gs;
  const bool begin = total_picks > 0 && n > 0 && num_segments >= 1 && num_segments < kBlock &&
                     (range != nullptr || num_segments == 1) && out_range &&
                     list_selects(n, num_segments, num_picks, replace);
  if (begin) {
    const ListWs w = carve_list(workspace, n, num_segments);
    if (workspace == nullptr || workspace_bytes < w.total) {
      set_error("list_sample workspace too small: %zu < %zu", workspace_bytes, w.total);
      return GS_ERR_WORKSPACE;
    }
    hipStream_t s = as_stream(stream);
    GS_LAUNCH("list_counts", s,
              list_offsets_kernel<<<list_zero_grid(w), dim3(kBlock), 0, s>>>(
                  range, n, num_segments, num_picks, replace, out_range, w.sel_block,
                  (int64_t)w.sel_words));
  } else {
    const int rc = gs_list_sample_weighted_count(range, n, num_segments, num_picks, replace,
                                                 out_range, workspace, workspace_bytes, stream);
    if (rc != GS_OK) return rc;
  }
  return list_fill(probs, range, n, num_segments, num_picks, replace, seed, call_id, out_range,
                   total_picks, out_index, out_value, workspace, workspace_bytes, stream, begin);
}

}  // extern "C"

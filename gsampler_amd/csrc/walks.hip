// walks.hip -- uniform random walk and node2vec over CSC in-neighbours.
// A lane per walk, up to sixteen per second-order walk; traces are stored
// step-major, out[step * N + walk], so that neighbouring lanes write neighbouring
// ids (the reference uses the same layout, src/cuda/fusion/random_walk.cu:34).
// Streams: pos = walk index;
// random walk draw = step; node2vec draw = step << 32 | attempt.
#include "common.h"

#pragma clang fp contract(off)

namespace gs {

// Work-groups of one wavefront while there are fewer walks than fill the machine.
constexpr int64_t kFewWalks = int64_t(1) << 16;

// Where the column behind an edge lies: what a step needs to know about the node it
// arrives at.  hops[e] belongs to row id indices[e]; with the table a step is one
// load in the chain (the hop of the edge it draws) where it is two without (the id,
// then that column's offsets), and the id itself is only written out.
struct alignas(8) Hop {
  uint32_t start, degree;
};

__global__ __launch_bounds__(kBlock) void hop_table_kernel(
    const int64_t* __restrict__ indptr, int64_t num_cols, const int64_t* __restrict__ indices,
    int64_t nnz, Hop* __restrict__ hops) {
  const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (e >= nnz) return;
  int64_t start;
  const int64_t deg = column_degree(indptr, num_cols, indices[e], &start);
  hops[e] = Hop{(uint32_t)start, (uint32_t)deg};
}

// The random words of a step depend on none of its loads and are drawn while one is
// on its way.  (Picks kept in registers and stored eight steps at a time, so that no
// load waits for a store in the in-order counter they share, cost more instructions
// than it saved waits: 5000 walks of 57 steps on 7.5 M edges 48.9 us, now 42.8, with
// the hop table 34.1 and 31.7; short walks were behind the plain loop.)
template <typename IdT, bool kHops>
__global__ __launch_bounds__(kBlock) void random_walk_kernel(
    const int64_t* __restrict__ indptr, const IdT* __restrict__ indices,
    const Hop* __restrict__ hops, int64_t num_cols, const int64_t* __restrict__ seeds,
    int64_t num_seeds, int64_t walk_length, PhiloxKey key, int64_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= num_seeds) return;
  int64_t curr = seeds[i];
  out[i] = curr;
  int64_t start = 0, deg = 0;
  if (kHops) deg = column_degree(indptr, num_cols, curr, &start);
  Words4 w = philox(key, (uint64_t)i, 1);
  for (int64_t step = 1; step <= walk_length; ++step) {
    int64_t pick = -1;
    const uint64_t r = ((uint64_t)w.y << 32) | w.x;
    if (!kHops) deg = column_degree(indptr, num_cols, curr, &start);
    if (deg > 0) {
      const int64_t e = start + (int64_t)__umul64hi(r, (uint64_t)deg);
      if (kHops) {
        const Hop next = hops[e];
        start = next.start;
        deg = next.degree;
      }
      pick = (int64_t)indices[e];
    }
    w = philox(key, (uint64_t)i, (uint64_t)(step + 1));
    curr = pick;
    out[step * num_seeds + i] = pick;
  }
}

// Is `target` among the sorted ids ptr[0, n)?  kWide: three probes a round, in
// flight together -- half the dependent round trips of a bisection for half as many
// loads again, which pays while the machine is not full.
template <bool kWide, typename IdT>
__device__ __forceinline__ bool sorted_contains(const IdT* ptr, int64_t n, int64_t target) {
  int64_t lo = 0, hi = n;  // ids before lo are smaller, ids from hi on are not
  if (kWide)
    while (hi - lo > 3) {
      const int64_t quarter = (hi - lo) >> 2;
      const int64_t m0 = lo + quarter, m1 = m0 + quarter, m2 = m1 + quarter;
      const int64_t v0 = (int64_t)ptr[m0], v1 = (int64_t)ptr[m1], v2 = (int64_t)ptr[m2];
      if (v0 == target || v1 == target || v2 == target) return true;
      if (v1 < target) {
        lo = (v2 < target ? m2 : m1) + 1;
        if (v2 >= target) hi = m2;
      } else {
        hi = v0 < target ? m1 : m0;
        if (v0 < target) lo = m0 + 1;
      }
    }
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    const int64_t v = (int64_t)ptr[mid];
    if (v == target) return true;
    if (v < target)
      lo = mid + 1;
    else
      hi = mid;
  }
  return false;
}

constexpr uint32_t kMaxAttempts = 1u << 16;

// Second-order walk by rejection sampling (src/cuda/fusion/node2vec.cu:90-135):
// every attempt draws an integer level y = floor(u * max(p, q)) and a uniform
// candidate; the candidate is accepted outright when y < min(p, q, 1), else when
// y < h with h = p for a return to the previous node, q for a neighbour of the
// previous node, 1 otherwise.
//
// G lanes walk one walk: lane g of a group looks at attempts g, g + G, ... of a
// step, and the lowest accepted attempt is the one that counts, so a step takes one
// round of loads where one lane takes as many as the slowest of 64 walks has
// attempts.  Worth it while the machine is not full: a candidate that a group looks
// at in vain costs a line.  (30 000 walks of 40 steps on 9 M edges: 173 us with one
// lane a walk, 76 with four at p = 2, q = 0.5; 1318 and 374 with eight at p = 0.25,
// q = 4, where a candidate in sixteen is accepted for sure.  1 M walks on 124 M
// edges are bound by lines: 3.3 ms with one lane, 3.9 with two.)
// (A loop in which every lane goes on to its own next step, instead of waiting for
// its wavefront at every step, was 28 % slower there: the lanes' stores of a step no
// longer meet in a line.)
template <typename IdT, int G, bool kHops>
__global__ __launch_bounds__(kBlock) void node2vec_kernel(
    const int64_t* __restrict__ indptr, const IdT* __restrict__ indices,
    const Hop* __restrict__ hops, int64_t num_cols, const int64_t* __restrict__ seeds, int64_t num_seeds,
    int64_t walk_length, double p, double q, PhiloxKey key,
    int64_t* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t i = t / G;
  const uint32_t g = (uint32_t)(t % G);
  if (i >= num_seeds) return;  // whole groups leave together
  const int group0 = lane_id() - (int)g;
  const double max_scale = p > q ? p : q;
  const double reject_from = max_scale > 1.0 ? max_scale : 1.0;
  double accept_below = p < q ? p : q;
  if (accept_below > 1.0) accept_below = 1.0;
  int64_t curr = seeds[i];
  int64_t last = -1;  // no previous node before the first step
  int64_t last_start = 0, last_deg = 0;
  if (g == 0) out[i] = curr;
  int64_t held = -1;  // the pick of step s waits in lane s % G of the group
  int64_t next_start, next_deg = column_degree(indptr, num_cols, curr, &next_start);
  for (int64_t step = 1; step <= walk_length; ++step) {
    int64_t pick = -1, start = next_start, deg = next_deg;
    if (!kHops && step > 1) deg = column_degree(indptr, num_cols, curr, &start);
    next_deg = 0;
    if (deg > 0) {
      if (deg == 1) {
        pick = (int64_t)indices[start];
        if (kHops) {
          const Hop n = hops[start];
          next_start = n.start;
          next_deg = n.degree;
        }
      } else {
        for (uint32_t attempt = g;; attempt += G) {
          const Words4 w = philox(key, (uint64_t)i, ((uint64_t)step << 32) | attempt);
          const double u = (double)((w.z >> 8) + 1u) * 0x1p-24;  // (0, 1]
          const int y = (int)floor(u * max_scale);
          const uint64_t r = ((uint64_t)w.y << 32) | w.x;
          const int64_t e = start + (int64_t)__umul64hi(r, (uint64_t)deg);
          Hop hop{0, 0};
          if (kHops) hop = hops[e];
          const int64_t cand = (int64_t)indices[e];
          bool taken = attempt + 1 >= kMaxAttempts || (double)y < accept_below;
          if (!taken && (double)y < reject_from) {
            double h = 1.0;
            if (cand == last) {
              h = p;
            } else if (((double)y < q) != ((double)y < 1.0) && last_deg > 0) {
              // the verdict differs between a neighbour of the previous node
              // (h = q) and any other node (h = 1) only for levels between q and
              // 1; everywhere else the adjacency search would change nothing
              if (sorted_contains<kHops>(indices + last_start, last_deg, cand)) h = q;
            }
            taken = (double)y < h;
          }
          pick = cand;
          if (G == 1) {
            next_start = hop.start;
            next_deg = hop.degree;
            if (taken) break;
          } else {
            const uint64_t hits = (__ballot(taken) >> group0) & ((1ull << G) - 1ull);
            if (hits) {
              const int winner = group0 + __ffsll((unsigned long long)hits) - 1;
              pick = __shfl(cand, winner, kWave);
              if (kHops) {
                next_start = (uint32_t)__shfl((int)hop.start, winner, kWave);
                next_deg = (uint32_t)__shfl((int)hop.degree, winner, kWave);
              }
              break;
            }
          }
        }
      }
    }
    last = curr;
    last_start = start;
    last_deg = deg;
    curr = pick;
    if (G == 1) {
      out[step * num_seeds + i] = pick;
    } else {
      if ((uint32_t)(step % G) == g) held = pick;
      if (step % G == G - 1 || step == walk_length) {
        const int64_t s = step - step % G + g;  // what this lane holds, if of this round
        if (s >= 1 && s <= step) out[s * num_seeds + i] = held;
      }
    }
  }
}

// What a second-order walk needs to know about a column whose ids are sorted, in 32
// bytes: where it lies (as pack_span writes it) and the ids at the first 6 of its
// sevenths.  An id is in the column only between two marks, so
//   * a candidate that would only be accepted as the return to the previous node is
//     drawn, compared with the place the marks leave that node and rejected without
//     being read, six times in seven;
//   * the search for a candidate among the previous node's neighbours begins with a
//     seventh of them, usually a line or two.
constexpr int kMarks = 6;
struct alignas(32) ColumnMarks {
  uint64_t span;
  uint32_t id[kMarks];
};

// Position of mark m, in [0, kMarks), of a column whose span was packed (deg < 2^24).
__device__ __forceinline__ uint32_t mark_at(uint32_t deg, int m) {
  return deg * (uint32_t)(m + 1) / (kMarks + 1);
}

__global__ __launch_bounds__(kBlock) void column_marks_kernel(
    const int64_t* __restrict__ indptr, int64_t num_cols, const int64_t* __restrict__ indices,
    ColumnMarks* __restrict__ marks) {
  const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (c >= num_cols) return;
  const int64_t start = indptr[c], deg = indptr[c + 1] - start;
  ColumnMarks out;
  out.span = (uint64_t)pack_span(start, deg);
#pragma unroll
  for (int m = 0; m < kMarks; ++m)
    out.id[m] = deg > 0 && out.span != kSpanLookUp ? (uint32_t)indices[start + mark_at((uint32_t)deg, m)] : 0u;
  marks[c] = out;
}

// Level of an attempt, an integer in [0, max_scale].
__device__ __forceinline__ double level_of(const Words4& w, double max_scale) {
  const double u = (double)((w.z >> 8) + 1u) * 0x1p-24;  // (0, 1]
  return (double)(int)floor(u * max_scale);
}

// Positions [*from, *to) of a column in which `target` may lie, by its marks; true if a
// mark is the target itself.
__device__ __forceinline__ bool between_marks(const uint32_t (&mark)[kMarks], uint32_t deg,
                                              uint32_t target, uint32_t* from, uint32_t* to) {
  int below = 0, upto = 0;
#pragma unroll
  for (int m = 0; m < kMarks; ++m) {
    below += mark[m] < target;
    upto += mark[m] <= target;
  }
  *from = below == 0 ? 0 : mark_at(deg, below - 1) + 1;
  *to = upto == kMarks ? deg : mark_at(deg, upto);
  return upto > below;
}

// The same walk with marks, a lane a walk, for calls that fill the machine.
// 1 M walks of 80 steps on 124 M edges, p = 2, q = 0.5: the kernel above reads two
// candidates a step, one of them in vain, 175 M lines in 3.31 ms; this one 130 M in
// 2.52, both at the part's line rate (52 G/s).  80 M of those are the chosen candidates,
// the rest marks and candidates read to be rejected: 2, 4 and 14 marks in place of 6 take
// 2.62, 2.59 and 2.49 ms (more bytes a column reject more and miss L2 more often).  Non-temporal reads of the candidates
// leave 4 % more of the marks in L2 and take 2.70 ms.
// Drawn by each lane for its own walk, attempts of arithmetic only were the bound
// (2.68 ms; 5.85 at p = 4, q = 0.25, where a candidate in four is accepted: 2.92 now).
// kSearch: q > 1, where levels in [1, q) need the candidate looked up among the previous
// node's neighbours and every attempt reads its candidate.
template <typename IdT, bool kSearch>
__global__ __launch_bounds__(kBlock) void node2vec_marks_kernel(
    const int64_t* __restrict__ indptr, const IdT* __restrict__ indices,
    const ColumnMarks* __restrict__ marks, int64_t num_cols, const int64_t* __restrict__ seeds,
    int64_t num_seeds, int64_t walk_length, double p, double q, PhiloxKey key,
    int64_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = lane_id();
  const bool live = i < num_seeds;  // (the other lanes draw for their wavefront's walks)
  const double max_scale = p > q ? p : q;
  const double reject_from = max_scale > 1.0 ? max_scale : 1.0;
  double accept_below = p < q ? p : q;
  if (accept_below > 1.0) accept_below = 1.0;
  int64_t curr = live ? seeds[i] : -1, last = -1;
  int64_t last_start = 0;
  uint32_t last_deg = 0;
  uint32_t last_mark[kMarks];
#pragma unroll
  for (int m = 0; m < kMarks; ++m) last_mark[m] = 0;
  bool last_marked = false;
  if (live) out[i] = curr;
  for (int64_t step = 1; step <= walk_length; ++step) {
    int64_t start = 0;
    uint32_t deg = 0, mark[kMarks];
#pragma unroll
    for (int m = 0; m < kMarks; ++m) mark[m] = 0;
    uint64_t span = 0;
    if (curr >= 0 && curr < num_cols) {
      const ColumnMarks c = marks[curr];
      span = c.span;
#pragma unroll
      for (int m = 0; m < kMarks; ++m) mark[m] = c.id[m];
    }
    // (the first words of a step depend on no load and are drawn while the marks travel)
    Words4 w = philox(key, (uint64_t)i, (uint64_t)step << 32);
    const bool marked = span != kSpanLookUp;
    if (marked) {
      start = (int64_t)(span & ((1ull << kSpanStartBits) - 1ull));
      deg = (uint32_t)(span >> kSpanStartBits);
    } else {
      deg = (uint32_t)column_degree(indptr, num_cols, curr, &start);
    }
    int64_t pick = -1;
    // where the previous node may lie in this column (there is none before the first step)
    uint32_t from = 0, to = last >= 0 ? deg : 0;
    if (marked && last >= 0 && deg > 0) between_marks(mark, deg, (uint32_t)last, &from, &to);
    if (kSearch) {
      if (deg == 1) {
        pick = (int64_t)indices[start];
      } else if (deg > 0) {
        for (uint32_t attempt = 0;; ++attempt) {
          double y;
          uint32_t at;
          bool sure, search;
          for (;; ++attempt) {
            if (attempt > 0) w = philox(key, (uint64_t)i, ((uint64_t)step << 32) | attempt);
            y = level_of(w, max_scale);
            at = (uint32_t)__umul64hi(((uint64_t)w.y << 32) | w.x, (uint64_t)deg);
            sure = attempt + 1 >= kMaxAttempts || y < accept_below;
            search = (y < q) != (y < 1.0) && last_deg > 0;
            if (sure || (y < reject_from && (search || (y < p && at >= from && at < to)))) break;
          }
          const int64_t cand = (int64_t)indices[start + at];
          pick = cand;
          if (sure) break;
          double h = 1.0;
          if (cand == last) {
            h = p;
          } else if (search) {
            uint32_t lo = 0, hi = last_deg;
            bool found = false;
            if (last_marked) found = between_marks(last_mark, last_deg, (uint32_t)cand, &lo, &hi);
            if (found || sorted_contains<false>(indices + last_start + lo, (int64_t)hi - lo, cand))
              h = q;
          }
          if (y < h) break;
        }
      }
    } else {
      // An attempt is sure, or accepted if its candidate is the previous node, or
      // rejected, whatever else its candidate is.  Attempts are drawn for as many walks
      // as are undecided by all lanes of the wavefront; of each walk the first one that
      // is not rejected counts.
      constexpr uint32_t kNone = ~0u;
      uint32_t chosen = kNone, check0 = kNone, check1 = kNone, next = 1;
      bool back = false;
      // what an attempt at position `at` is
      auto sure_at = [&](uint32_t attempt, double y) {
        return attempt + 1 >= kMaxAttempts || y < accept_below;
      };
      auto note = [&](bool sure, uint32_t at) {  // true: the walk is decided
        if (sure) chosen = at;
        else if (check0 == kNone) check0 = at;
        else if (check1 == kNone) check1 = at;
        else back = (int64_t)indices[start + at] == last;
        return sure || back;
      };
      bool pending = deg > 1;
      if (deg == 1) chosen = 0;
      if (pending) {
        const double y = level_of(w, max_scale);
        const uint32_t at = (uint32_t)__umul64hi(((uint64_t)w.y << 32) | w.x, (uint64_t)deg);
        const bool sure = sure_at(0, y);
        if (sure || (y < reject_from && y < p && at >= from && at < to)) pending = !note(sure, at);
      }
      for (;;) {
        const uint64_t open = __ballot(pending);
        if (open == 0) break;
        const int walks = __popcll(open);
        const int shift = walks == 1 ? 6 : __clz(walks - 1) - 26;  // lanes a walk: 2^shift
        const int rank = (int)__builtin_amdgcn_mbcnt_hi(
            (uint32_t)(open >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)open, 0));
        // lane k learns which walk is the k-th undecided one, and then its own group's
        const int order = __builtin_amdgcn_ds_permute((pending ? rank : kWave - 1) << 2,
                                                      pending ? lane : -1);
        const int mine = lane >> shift;
        const int owner = __shfl(order, mine, kWave) & (kWave - 1);
        const uint32_t attempt = (uint32_t)__shfl((int)next, owner, kWave) +
                                 (uint32_t)(lane & ((1 << shift) - 1));
        const uint32_t o_deg = (uint32_t)__shfl((int)deg, owner, kWave);
        const uint32_t o_from = (uint32_t)__shfl((int)from, owner, kWave);
        const uint32_t o_to = (uint32_t)__shfl((int)to, owner, kWave);
        w = philox(key, (uint64_t)(i - lane + owner), ((uint64_t)step << 32) | attempt);
        const double y = level_of(w, max_scale);
        const uint32_t at = (uint32_t)__umul64hi(((uint64_t)w.y << 32) | w.x, (uint64_t)o_deg);
        const bool sure = sure_at(attempt, y);
        const bool counts =
            mine < walks &&
            (sure || (y < reject_from && y < p && at >= o_from && at < o_to));
        const int group0 = (rank << shift) & (kWave - 1);
        const uint64_t group = shift == 6 ? ~0ull : (1ull << (1 << shift)) - 1ull;
        const uint64_t hits = (__ballot(counts) >> group0) & group;
        const uint64_t sures = __ballot(sure) >> group0;
        const int first = hits ? __ffsll((unsigned long long)hits) - 1 : 0;
        const uint32_t found = (uint32_t)__shfl((int)at, group0 + first, kWave);
        if (pending) {
          if (hits) {
            pending = !note((sures >> first) & 1ull, found);
            next += (uint32_t)first + 1;
          } else {
            next += 1u << shift;
          }
        }
      }
      if (deg > 0) {
        int64_t c0 = -1, c1 = -1;
        if (chosen != kNone) pick = (int64_t)indices[start + chosen];
        if (check0 != kNone) c0 = (int64_t)indices[start + check0];
        if (check1 != kNone) c1 = (int64_t)indices[start + check1];
        if (back || (c0 == last && check0 != kNone) || (c1 == last && check1 != kNone)) pick = last;
      }
    }
    last = curr;
    if (kSearch) {
      last_start = start;
      last_deg = deg;
      last_marked = marked;
#pragma unroll
      for (int m = 0; m < kMarks; ++m) last_mark[m] = mark[m];
    }
    curr = pick;
    if (live) out[step * num_seeds + i] = pick;
  }
}

// Whether candidates are mostly rejected: only those of level 0, one in max(p, q), are
// accepted whatever they are.
static bool rare_picks(double p, double q) { return p > 3.0 || q > 3.0; }

// Whether the first candidate stands, all but once in 2^24 (the only level is 0).
static bool sure_picks(double p, double q) { return p <= 1.0 && q <= 1.0; }

// Up to how many walks a call goes by the hop table.  Few walks are bound by the
// latency of their chains of loads, which the table shortens; more are bound by lines,
// of which it costs as many as it saves -- a second line a candidate for a group that
// looks at sixteen at once -- and the column pointer's are the better cached ones.
// Without / with the table, us, 9 M edges:
//   first order, 56 steps     1 K walks 47 / 32    16 K 49 / 38     24 K 51 / 51, 33 K 53 / 69
//     (measured with picks stored eight at a time)
//   second order, 40 steps
//     max(p, q) <= 1          one lane without the table is as fast (first candidates stand)
//     q < 1 (no search)       2 K walks 44 / 35 and 45 / 37         4 K 46 / 49, 8 K 51 / 95
//     q > 1, picks rare       8 K walks 286 / 243                   16 K 322 / 461
//     q > 1, others           32 K walks 351 / 296, 493 / 414
// (with q > 1 the searches take most of the time, and they go three probes at once
// where there is a table).
static int64_t hop_walks(bool second_order, double p, double q) {
  if (!second_order) return int64_t(1) << 14;
  if (sure_picks(p, q)) return 0;
  if (q <= 1.0) return int64_t(1) << 11;
  return rare_picks(p, q) ? int64_t(1) << 13 : int64_t(1) << 15;
}

// Up to how many lanes a call spreads its walks over, a group of lanes a walk (the best
// of 1, 2, 4, 8, 16 lanes at 1.5 K to 300 K walks of 20 steps): about 200 K where every
// second candidate is accepted, 400 K where fewer are or candidates are searched for
// (120 K walks on 9 M edges, one lane and two: p = 1, q = 4 872 and 520 us, p = 0.5,
// q = 2 481 and 309, p = 2, q = 0.5 107 and 98).
static int64_t walk_lanes(double p, double q) {
  return q > 1.0 || rare_picks(p, q) ? 400000 : 200000;
}

// From how many walks on a call goes by marks: those that go by one lane a walk and are
// bound by lines.  Without / with marks, us:
//   124 M edges    1 M walks, 80 steps    p = 2, q = 0.5  3308 / 2513    p = 4, q = 0.25  5494 / 2919
//                                         p = 0.25, q = 4  14 886 / 14 294
//   9 M edges      300 K walks, 40 steps  388 / 320, 678 / 468, 2078 / 1808
//                  60 K walks by groups   115 / 154, 168 / 264, 548 / 1296
static int64_t marks_walks(double p, double q) {
  return sure_picks(p, q) ? INT64_MAX : walk_lanes(p, q) / 2 + 1;
}

template <typename IdT>
static int node2vec_marks(const int64_t* indptr, const IdT* indices, const ColumnMarks* marks,
                          int64_t num_cols, const int64_t* seeds, int64_t num_seeds,
                          int64_t walk_length, double p, double q, uint64_t seed,
                          uint64_t call_id, int64_t* out_traces, gs_stream_t stream) {
  GS_REQUIRE(num_seeds >= 0 && walk_length >= 0 && num_cols >= 0,
             "node2vec: negative size");
  GS_REQUIRE(p > 0.0 && q > 0.0, "node2vec: p and q must be positive");
  if (num_seeds == 0) return GS_OK;
  GS_REQUIRE(indptr && seeds && out_traces, "node2vec: null pointer");
  hipStream_t s = as_stream(stream);
  const int threads = num_seeds < kFewWalks ? kWave : kBlock;
#define GS_NODE2VEC_MARKS(SEARCH)                                                                \
  GS_LAUNCH("node2vec", s,                                                                      \
            (node2vec_marks_kernel<IdT, SEARCH>)<<<dim3((unsigned)ceil_div(num_seeds, threads)), \
                                                   dim3(threads), 0, s>>>(                      \
                indptr, indices, marks, num_cols, seeds, num_seeds, walk_length, p, q,          \
                make_key(seed, call_id), out_traces))
  if (q > 1.0) GS_NODE2VEC_MARKS(true);
  else GS_NODE2VEC_MARKS(false);
#undef GS_NODE2VEC_MARKS
  return GS_OK;
}

template <typename IdT>
static int random_walk(const int64_t* indptr, const IdT* indices, const Hop* hops,
                       int64_t num_cols, const int64_t* seeds, int64_t num_seeds,
                       int64_t walk_length, uint64_t seed, uint64_t call_id, int64_t* out_traces,
                       gs_stream_t stream) {
  GS_REQUIRE(num_seeds >= 0 && walk_length >= 0 && num_cols >= 0,
             "random_walk: negative size");
  if (num_seeds == 0) return GS_OK;
  GS_REQUIRE(indptr && seeds && out_traces, "random_walk: null pointer");
  hipStream_t s = as_stream(stream);
  const int threads = num_seeds < kFewWalks ? kWave : kBlock;
#define GS_RANDOM_WALK(HOPS)                                                                     \
  GS_LAUNCH("random_walk", s,                                                                    \
            (random_walk_kernel<IdT, HOPS>)<<<dim3((unsigned)ceil_div(num_seeds, threads)),      \
                                              dim3(threads), 0, s>>>(                            \
                indptr, indices, hops, num_cols, seeds, num_seeds, walk_length,                  \
                make_key(seed, call_id), out_traces))
  if (hops && num_seeds <= hop_walks(false, 1.0, 1.0)) GS_RANDOM_WALK(true);
  else GS_RANDOM_WALK(false);
#undef GS_RANDOM_WALK
  return GS_OK;
}

template <typename IdT>
static int node2vec(const int64_t* indptr, const IdT* indices, const Hop* hops, int64_t num_cols,
                    const int64_t* seeds, int64_t num_seeds, int64_t walk_length, double p,
                    double q, uint64_t seed, uint64_t call_id, int64_t* out_traces,
                    gs_stream_t stream) {
  GS_REQUIRE(num_seeds >= 0 && walk_length >= 0 && num_cols >= 0,
             "node2vec: negative size");
  GS_REQUIRE(p > 0.0 && q > 0.0, "node2vec: p and q must be positive");
  if (num_seeds == 0) return GS_OK;
  GS_REQUIRE(indptr && seeds && out_traces, "node2vec: null pointer");
  hipStream_t s = as_stream(stream);
  // As many lanes a walk as keep the call's lanes below what fills the machine; one
  // where the first candidate stands (32 K walks of 20 steps on 9 M edges: 22 us, with
  // four lanes 35).
  const int64_t lanes = walk_lanes(p, q);
  int group = 16;
  while (group > 1 && num_seeds * group > lanes) group >>= 1;
  if (sure_picks(p, q)) group = 1;
  const int threads = num_seeds * group < kFewWalks ? kWave : kBlock;
#define GS_NODE2VEC(G, HOPS)                                                                    \
  GS_LAUNCH("node2vec", s,                                                                      \
            (node2vec_kernel<IdT, G, HOPS>)<<<dim3((unsigned)ceil_div(num_seeds * (G), threads)), \
                                              dim3(threads), 0, s>>>(                           \
                indptr, indices, hops, num_cols, seeds, num_seeds, walk_length, p, q,           \
                make_key(seed, call_id), out_traces))
  const bool use_hops = hops && num_seeds <= hop_walks(true, p, q);
  if (group == 16) {
    if (use_hops) GS_NODE2VEC(16, true);
    else GS_NODE2VEC(16, false);
  } else if (group == 8) {
    if (use_hops) GS_NODE2VEC(8, true);
    else GS_NODE2VEC(8, false);
  } else if (group == 4) {
    if (use_hops) GS_NODE2VEC(4, true);
    else GS_NODE2VEC(4, false);
  } else if (group == 2) {
    GS_NODE2VEC(2, false);
  } else {
    GS_NODE2VEC(1, false);
  }
#undef GS_NODE2VEC
  return GS_OK;
}

}  // namespace gs

extern "C" {

int gs_hop_table(const int64_t* indptr, int64_t num_cols, const int64_t* indices, int64_t nnz,
                 void* hops, gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(num_cols >= 0 && nnz >= 0 && nnz < (int64_t(1) << 32), "hop_table: bad size");
  if (nnz == 0) return GS_OK;
  GS_REQUIRE(indptr && indices && hops, "hop_table: null pointer");
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("hop_table", s,
            hop_table_kernel<<<dim3((unsigned)ceil_div(nnz, kBlock)), dim3(kBlock), 0, s>>>(
                indptr, num_cols, indices, nnz, (Hop*)hops));
  return GS_OK;
}

size_t gs_column_marks_bytes(int64_t num_cols) {
  return num_cols > 0 ? sizeof(gs::ColumnMarks) * (size_t)num_cols : 0;
}

int gs_column_marks(const int64_t* indptr, int64_t num_cols, const int64_t* indices, void* marks,
                    gs_stream_t stream) {
  using namespace gs;
  GS_REQUIRE(num_cols >= 0 && num_cols <= (int64_t(1) << 31), "column_marks: bad size");
  if (num_cols == 0) return GS_OK;
  GS_REQUIRE(indptr && indices && marks, "column_marks: null pointer");
  GS_REQUIRE(((uintptr_t)marks & (alignof(ColumnMarks) - 1)) == 0, "column_marks: misaligned");
  hipStream_t s = as_stream(stream);
  GS_LAUNCH("column_marks", s,
            column_marks_kernel<<<dim3((unsigned)ceil_div(num_cols, kBlock)), dim3(kBlock), 0, s>>>(
                indptr, num_cols, indices, (ColumnMarks*)marks));
  return GS_OK;
}

int64_t gs_marks_walks(double p, double q) { return gs::marks_walks(p, q); }

int gs_node2vec_marks(const int64_t* indptr, const int64_t* indices, const int32_t* indices32,
                      const void* marks, int64_t num_cols, const int64_t* seeds,
                      int64_t num_seeds, int64_t walk_length, double p, double q, uint64_t seed,
                      uint64_t call_id, int64_t* out_traces, gs_stream_t stream) {
  GS_REQUIRE(marks != nullptr && ((uintptr_t)marks & (alignof(gs::ColumnMarks) - 1)) == 0,
             "node2vec: null or misaligned marks");
  const gs::ColumnMarks* m = (const gs::ColumnMarks*)marks;
  if (indices32)
    return gs::node2vec_marks(indptr, indices32, m, num_cols, seeds, num_seeds, walk_length, p, q,
                              seed, call_id, out_traces, stream);
  return gs::node2vec_marks(indptr, indices, m, num_cols, seeds, num_seeds, walk_length, p, q,
                            seed, call_id, out_traces, stream);
}

int64_t gs_hop_walks(int second_order, double p, double q) {
  return gs::hop_walks(second_order != 0, p, q);
}

int gs_random_walk(const int64_t* indptr, const int64_t* indices, int64_t num_cols,
                   const int64_t* seeds, int64_t num_seeds, int64_t walk_length,
                   uint64_t seed, uint64_t call_id, int64_t* out_traces,
                   gs_stream_t stream) {
  return gs::random_walk(indptr, indices, nullptr, num_cols, seeds, num_seeds, walk_length, seed,
                         call_id, out_traces, stream);
}

int gs_random_walk_hops(const int64_t* indptr, const int64_t* indices, const void* hops,
                        int64_t num_cols, const int64_t* seeds, int64_t num_seeds,
                        int64_t walk_length, uint64_t seed, uint64_t call_id,
                        int64_t* out_traces, gs_stream_t stream) {
  return gs::random_walk(indptr, indices, (const gs::Hop*)hops, num_cols, seeds, num_seeds,
                         walk_length, seed, call_id, out_traces, stream);
}

int gs_node2vec(const int64_t* indptr, const int64_t* indices, int64_t num_cols,
                const int64_t* seeds, int64_t num_seeds, int64_t walk_length,
                double p, double q, uint64_t seed, uint64_t call_id,
                int64_t* out_traces, gs_stream_t stream) {
  return gs::node2vec(indptr, indices, nullptr, num_cols, seeds, num_seeds, walk_length, p, q,
                      seed, call_id, out_traces, stream);
}

int gs_node2vec_hops(const int64_t* indptr, const int64_t* indices, const int32_t* indices32,
                     const void* hops, int64_t num_cols, const int64_t* seeds, int64_t num_seeds,
                     int64_t walk_length, double p, double q, uint64_t seed, uint64_t call_id,
                     int64_t* out_traces, gs_stream_t stream) {
  const gs::Hop* h = (const gs::Hop*)hops;
  // (a lane that takes its first candidate is bound by the latency of its loads while
  // there are few of them, and a 64-bit id needs no widening: 16 K walks of 20 steps
  // 20.8 us, 23.6 with the narrow ids; from 64 K walks on those are ahead)
  if (indices32 && !(gs::sure_picks(p, q) && num_seeds < gs::kFewWalks))
    return gs::node2vec(indptr, indices32, h, num_cols, seeds, num_seeds, walk_length, p, q, seed,
                        call_id, out_traces, stream);
  return gs::node2vec(indptr, indices, h, num_cols, seeds, num_seeds, walk_length, p, q, seed,
                      call_id, out_traces, stream);
}

}  // extern "C"

// walks_misc.cc -- walks, per-column index sort, compaction and the batched
// column+row slice of gs_classes.Graph.
#include "abi_call.h"
#include "graph.h"

namespace gs {

// Kept for matrices of up to 2^24 edges (128 MB): there it stays in the last-level
// cache, and making it costs a fraction of a walk.  A matrix that is walked once
// never makes it, nor one whose calls have too many walks for it.
torch::Tensor Compressed::hop_table() const {
  constexpr int64_t kMaxEdges = int64_t(1) << 24;
  const int64_t nnz = indices.numel();
  if (nnz == 0 || nnz > kMaxEdges || !indices.is_cuda() || !indptr.is_cuda()) return {};
  std::lock_guard<std::mutex> lock(derived_.guard);
  Derived& d = current_derived();
  if (!narrow_ids_allowed().load()) {
    d.hops.drop();
    return {};
  }
  if (!d.hops.defined() && d.walks++ == 0) return {};
  if (capturing()) return {};
  if (!d.hops.defined()) {
    torch::Tensor t = new_ids(nnz, indices);
    GS_CALL(gs_hop_table(cptr(indptr), indptr.numel() - 1, cptr(indices), nnz, t.data_ptr(),
                         cur_stream()));
    d.hops.set(t);
  }
  return d.hops.on_current_stream();
}

// 32 bytes a column.  Making them reads up to four lines a column, of which they save
// one or two a step.
torch::Tensor Compressed::column_marks(int64_t steps) const {
  constexpr int64_t kMinEdges = int64_t(1) << 20;  // (below, ids stay in cache)
  constexpr int64_t kStepsPerColumn = 4;
  const int64_t cols = indptr.numel() - 1;
  if (indices.numel() < kMinEdges || num_minor < 0 || num_minor >= (int64_t(1) << 31) ||
      indices.numel() >= (int64_t(1) << 32) || cols >= (int64_t(1) << 31) || !indices.is_cuda() || !indptr.is_cuda())
    return {};
  std::lock_guard<std::mutex> lock(derived_.guard);
  Derived& d = current_derived();
  if (!narrow_ids_allowed().load()) {
    d.marks.drop();
    return {};
  }
  if (!d.marks.defined() && (d.steps += steps) < kStepsPerColumn * cols) return {};
  if (capturing()) return {};
  if (!d.marks.defined()) {
    torch::Tensor t = new_ids((int64_t)gs_column_marks_bytes(cols) / 8, indices);
    GS_CALL(gs_column_marks(cptr(indptr), cols, cptr(indices), t.data_ptr(), cur_stream()));
    d.marks.set(t);
  }
  return d.marks.on_current_stream();
}

// Traces are stored step-major ([walk_length + 1][num_seeds] in memory) and
// returned with shape [num_seeds, walk_length + 1] exactly as the reference
// does (src/cuda/fusion/random_walk.cu:34,67): callers obtain per-step rows
// with `.reshape(-1, num_seeds)`.
torch::Tensor Graph::RandomWalk(torch::Tensor seeds, int64_t walk_length) {
  TORCH_CHECK(csc_ != nullptr, "RandomWalk needs the CSC format");
  TORCH_CHECK(walk_length >= 0, "walk_length must be non-negative");
  seeds = ids(seeds, "seeds");
  const int64_t n = seeds.numel();
  torch::Tensor out = new_ids(n * (walk_length + 1), seeds);
  const RandomState& rs = random_state();
  const torch::Tensor hops = n <= gs_hop_walks(0, 1.0, 1.0) ? csc_->hop_table() : torch::Tensor();
  GS_CALL(gs_random_walk_hops(cptr(csc_->indptr), cptr(csc_->indices), cptr(hops), num_cols_,
                              cptr(seeds), n, walk_length, rs.seed, next_call_id(), mptr(out),
                              cur_stream()));
  return out.reshape({n, -1});
}

torch::Tensor Graph::Node2Vec(torch::Tensor seeds, int64_t walk_length, double p,
                              double q) {
  TORCH_CHECK(csc_ != nullptr, "Node2Vec needs the CSC format");
  TORCH_CHECK(walk_length >= 0, "walk_length must be non-negative");
  TORCH_CHECK(p > 0 && q > 0, "Node2Vec: p and q must be positive");
  // The connectivity test bisects the previous node's column: row ids must be
  // sorted inside every column.  Looked at once per matrix (one pass over the
  // edges); the reference walks on unsorted columns without noticing.
  if (!csc_sorted_) {
    const torch::Tensor& idx = csc_->indices;
    const int64_t nnz = idx.numel();
    if (nnz > 1) {
      torch::Tensor drop = idx.slice(0, 1).lt(idx.slice(0, 0, nnz - 1));
      torch::Tensor ends = csc_->indptr.slice(0, 1, num_cols_) - 1;  // last edge of a column
      ends = ends.masked_select(ends.ge(0).logical_and(ends.lt(nnz - 1)));
      drop.index_fill_(0, ends.to(drop.device()), false);
      TORCH_CHECK(!drop.any().item<bool>(),
                  "Node2Vec needs row ids sorted inside every column: call SortCSCIndices first");
    }
    csc_sorted_ = true;
  }
  seeds = ids(seeds, "seeds");
  const int64_t n = seeds.numel();
  torch::Tensor out = new_ids(n * (walk_length + 1), seeds);
  const RandomState& rs = random_state();
  // The copy costs 2.1 ps an edge (255 us on 124 M) and saves 0.7 to 8 ps a step, or
  // some 20 and more where q > 1 has candidates looked up among the neighbours before.
  const int64_t steps = n * walk_length;
  const torch::Tensor narrow = csc_->narrow_indices(q > 1.0 ? 16 * steps : steps);
  const torch::Tensor marks = n >= gs_marks_walks(p, q) ? csc_->column_marks(steps) : torch::Tensor();
  if (marks.defined()) {
    GS_CALL(gs_node2vec_marks(cptr(csc_->indptr), cptr(csc_->indices),
                              narrow.defined() ? narrow.data_ptr<int32_t>() : nullptr,
                              marks.data_ptr(), num_cols_, cptr(seeds), n, walk_length, p, q,
                              rs.seed, next_call_id(), mptr(out), cur_stream()));
    return out.reshape({n, -1});
  }
  const torch::Tensor hops = n <= gs_hop_walks(1, p, q) ? csc_->hop_table() : torch::Tensor();
  GS_CALL(gs_node2vec_hops(cptr(csc_->indptr), cptr(csc_->indices),
                           narrow.defined() ? narrow.data_ptr<int32_t>() : nullptr, cptr(hops),
                           num_cols_, cptr(seeds), n, walk_length, p, q, rs.seed, next_call_id(),
                           mptr(out), cur_stream()));
  return out.reshape({n, -1});
}

void Graph::SortCSCIndices() {
  TORCH_CHECK(csc_ != nullptr, "SortCSCIndices: the graph has no CSC format");
  TORCH_CHECK(!csc_->e_ids.has_value(), "SortCSCIndices: the CSC format carries e_ids");
  const int64_t nnz = csc_->indices.numel();
  torch::Tensor sorted = new_ids(nnz, csc_->indices);
  // row ids lie in [0, num_rows): the loaders check that
  torch::Tensor ws = new_workspace(gs_segment_sort_workspace_bytes(nnz, num_cols_, num_rows_),
                                   csc_->indices);
  GS_CALL(gs_segment_sort_i64(cptr(csc_->indptr), num_cols_, cptr(csc_->indices),
                              mptr(sorted), nnz, num_rows_, ws.data_ptr(), ws.numel(),
                              cur_stream()));
  csc_->indices = sorted;
  csc_->forget_derived();
  csc_sorted_ = true;
  coo_ = nullptr;  // derived formats followed the old edge order
  csr_ = nullptr;
}

// (sorted distinct ids, rank of every element among them): TensorCompact,
// src/cuda/compact.cu:11-34, which is torch's sorted unique with inverse.
static std::tuple<torch::Tensor, torch::Tensor> compact_ids(const torch::Tensor& x) {
  auto r = torch::_unique2(x, /*sorted=*/true, /*return_inverse=*/true,
                           /*return_counts=*/false);
  return {std::get<0>(r), std::get<1>(r)};
}

// Drops ids that no edge uses on `axis` (0 rows, 1 columns) and renumbers the
// rest densely; returns the kept original ids.  Formats whose compressed axis
// is the compacted one are dropped (they can be rebuilt from the COO).
GraphAndIndex Graph::Compact(int64_t axis) {
  TORCH_CHECK(axis == 0 || axis == 1, "Compact: axis must be 0 or 1");
  torch::Tensor kept, local;
  std::shared_ptr<Coordinate> coo;
  std::shared_ptr<Compressed> csc, csr;
  if (coo_) {
    const torch::Tensor& src = axis == 0 ? coo_->row : coo_->col;
    std::tie(kept, local) = compact_ids(src);
    coo = std::make_shared<Coordinate>(*coo_);
    (axis == 0 ? coo->row : coo->col) = local;
  }
  const std::shared_ptr<Compressed>& other = axis == 0 ? csc_ : csr_;
  if (other) {
    const torch::Tensor& coo_src = coo_ ? (axis == 0 ? coo_->row : coo_->col) : other->indices;
    torch::Tensor ids_local;
    if (coo_ && other->indices.is_same(coo_src)) {
      ids_local = local;
    } else {
      torch::Tensor k2;
      std::tie(k2, ids_local) = compact_ids(other->indices);
      if (!kept.defined()) kept = k2;
    }
    auto m = std::make_shared<Compressed>(*other);
    m->indices = ids_local;
    m->forget_derived();
    (axis == 0 ? csc : csr) = m;
  }
  TORCH_CHECK(kept.defined(), "Compact: the graph has no format with explicit ids on axis ",
              axis);
  auto g = c10::make_intrusive<Graph>(axis == 0 ? kept.numel() : num_rows_,
                                      axis == 0 ? num_cols_ : kept.numel());
  g->coo_ = coo;
  g->csc_ = csc;
  g->csr_ = csr;
  g->num_edges_ = num_edges_;
  return {g, kept};
}

}  // namespace gs

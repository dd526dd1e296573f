// fused_slices.cc -- operators that read a column slice A[:, cols] straight
// from the matrix it is a slice of, without writing it first: the row sums of
// squared edge values over the slice, and the row slice of the slice
// (A[rows, cols]).  gs.jit.compile rewrites  A[:, cols] -> sum(e^2, axis=1) /
// -> [rows, :]  into these when nothing else reads the slice, which is the
// shape of a layer-wise sampler (examples/ladies/ladies.py:7-21 of the
// reference); the reference fuses the second pair only, and only for
// super-batches (src/cuda/fusion/column_row_slicing.cu).
#include <ATen/autocast_mode.h>
#include <ATen/PythonTorchFunctionTLS.h>

#include "abi_call.h"
#include "graph.h"

namespace gs {

// Offsets and size of A[:, cols]: shared by the operators of this file when
// they are handed the same tensor of columns (one wait for the size, not two)
// on the same stream: another one would have to wait for what is queued on the
// first, and memory that is freed there may be written again while it reads.
// `wait`: for the size as well (the host copy of one that is not waited for keeps the offsets).
std::shared_ptr<Graph::SliceOffsets> Graph::slice_offsets_for(const torch::Tensor& cols, bool wait) {
  const Compressed& m = compressed(kCSC);
  wait |= cols.numel() > (1 << 16);
  std::shared_ptr<SliceOffsets> so;
  {
    std::lock_guard<std::mutex> lock(slice_offsets_guard_);
    if (slice_offsets_ && slice_offsets_->cols.is_same(cols) &&
        slice_offsets_->version == (int64_t)cols._version() &&
        slice_offsets_->indptr_version == (int64_t)m.indptr._version() &&
        slice_offsets_->epoch == cache_epoch() && slice_offsets_->stream == cur_stream())
      so = slice_offsets_;
  }
  if (!so) {
    so = std::make_shared<SliceOffsets>();
    so->cols = cols;
    so->version = cols._version();
    so->indptr_version = m.indptr._version();
    so->epoch = cache_epoch();
    so->stream = cur_stream();
    so->sub_indptr = wait ? slice_offsets(m, cols, &so->nnz) : slice_offsets_ahead(m, cols, &so->total);
    std::lock_guard<std::mutex> lock(slice_offsets_guard_);
    slice_offsets_ = so;
  }
  if (wait) {
    std::lock_guard<std::mutex> lock(so->guard);
    if (so->nnz < 0) so->nnz = OffsetMirror::values(so->total)[0];
  }
  return so;
}

// A sampler whose picks do not depend on the slice (FastGCN) asks for its offsets before it
// picks: their number is at hand when the slice is made, where the device stood still while
// it travelled to the host (FastGCN of 1024 seeds 228 -> 215 us a pass).
void Graph::PrepareSlice(torch::Tensor cols) {
  if (!csc_ || !csc_->indices.is_cuda() || !csc_->indptr.is_cuda() || !cols.is_cuda() ||
      cols.scalar_type() != torch::kInt64 || cols.dim() != 1 || !cols.is_contiguous() ||
      cols.numel() == 0)
    return;
  slice_offsets_for(cols, false);
}

// A slice of a matrix in device memory is read in place whatever its columns are like:
// a wavefront looks the columns of its run of edges up once, all lanes together
// (200 K columns of 2 to 300 edges, 1 K to 150 K of them picked: row sums of squares 43
// to 387 us in place, 60 to 931 by writing the slice first, row slices 75 to 402 and 103
// to 866; the row slice of 8.4 M edges in 9.4 K columns 98 and 161).  From pinned host
// memory the ids would cross the bus again for every pass: there only slices of long
// columns are, which take fewer bytes in place even so.
bool Graph::read_in_place(const Compressed& m, int64_t slice_nnz, int64_t num_cols_picked) {
  if (m.indices.is_cuda()) return true;
  return slice_nnz >= (int64_t(1) << 20) && slice_nnz >= 4096 * num_cols_picked;
}

// The int32 copy of the ids for passes over a slice: made at once for a large slice of
// long columns, else when such passes have read as many ids as the matrix has edges.
static torch::Tensor narrow_for_slice(const Compressed& m, int64_t slice_nnz, int64_t num_cols_picked) {
  const bool large = slice_nnz >= (int64_t(1) << 20) && slice_nnz >= 4096 * num_cols_picked;
  return m.narrow_indices(large ? -1 : slice_nnz);
}

const MajorResult& Graph::written_slice(SliceOffsets& so) {
  std::lock_guard<std::mutex> lock(so.guard);
  if (!so.written.indptr.defined()) so.written = major_slice(compressed(kCSC), so.cols, true, {}, 0);
  return so.written;
}

// out[row] += sum of efeat^2 over the edges of A[:, cols]; efeat is aligned with
// this matrix's edges (as edge data of the Python layer is).
void Graph::SlicedESquareSum(torch::Tensor cols, torch::Tensor efeat, torch::Tensor out) {
  cols = ids(cols, "cols");
  const Compressed& m = compressed(kCSC);
  TORCH_CHECK(efeat.defined() && out.defined(), "SlicedESquareSum: undefined operand");
  TORCH_CHECK(efeat.is_cuda() && out.is_cuda() && efeat.scalar_type() == torch::kFloat32 &&
                  out.scalar_type() == torch::kFloat32,
              "SlicedESquareSum needs float32 tensors on the GPU");
  efeat = efeat.contiguous();
  TORCH_CHECK(out.is_contiguous(), "SlicedESquareSum: out must be contiguous");
  TORCH_CHECK(efeat.numel() == m.indices.numel(), "SlicedESquareSum: ", efeat.numel(),
              " edge values for ", m.indices.numel(), " edges (scalar edge values only)");
  TORCH_CHECK(out.numel() == num_rows_, "SlicedESquareSum: out has ", out.numel(),
              " entries for ", num_rows_, " rows");
  const std::shared_ptr<SliceOffsets> shared = slice_offsets_for(cols);
  SliceOffsets& so = *shared;
  if (so.nnz == 0) return;
  if (!read_in_place(m, so.nnz, cols.numel())) {
    const MajorResult& r = written_slice(so);
    torch::Tensor w = efeat.index_select(0, edge_index(m.e_ids, r.select));
    torch::Tensor ws =
        new_workspace(gs_spmm_workspace_bytes(GS_FMT_COO, so.nnz, num_rows_), m.indptr);
    GS_CALL(gs_e_square_sum(GS_FMT_COO, cptr(r.minor_ids), cptr(r.major_ids), 0, so.nnz, nullptr,
                            w.data_ptr<float>(), out.data_ptr<float>(), 2, 1, num_rows_,
                            ws.data_ptr(), (size_t)ws.numel(), cur_stream()));
    return;
  }
  torch::Tensor ws = new_workspace(gs_sliced_e_square_sum_workspace_bytes(so.nnz, num_rows_),
                                   m.indptr);
  const torch::Tensor e_ids = m.e_ids.has_value() ? m.e_ids.value() : torch::Tensor();
  const torch::Tensor narrow = narrow_for_slice(m, so.nnz, cols.numel());
  GS_CALL(gs_sliced_e_square_sum(cptr(m.indptr), cptr(m.indices),
                                 narrow.defined() ? narrow.data_ptr<int32_t>() : nullptr,
                                 cptr(cols), cols.numel(),
                                 cptr(so.sub_indptr), so.nnz, cptr(e_ids),
                                 efeat.data_ptr<float>(), out.data_ptr<float>(), num_rows_,
                                 ws.data_ptr(), (size_t)ws.numel(), cur_stream()));
}

c10::optional<torch::Tensor> Graph::SlicedSquareSums(torch::Tensor cols, torch::Tensor efeat) {
  const Compressed& m = compressed(kCSC);
  if (!plain_values(efeat, true) || efeat.dim() != 1 || !efeat.is_contiguous() ||
      efeat.numel() != m.indices.numel() || !m.indices.is_cuda() ||
      at::impl::torch_function_mode_enabled() || at::autocast::is_autocast_enabled(at::kCUDA))
    return {};
  cols = ids(cols, "cols");
  const std::shared_ptr<SliceOffsets> so = slice_offsets_for(cols);
  torch::Tensor out = torch::empty({num_rows_}, efeat.options().requires_grad(false));
  torch::Tensor ws = new_workspace(gs_sliced_e_square_sum_workspace_bytes(so->nnz, num_rows_),
                                   m.indptr);
  const torch::Tensor e_ids = m.e_ids.has_value() ? m.e_ids.value() : torch::Tensor();
  const torch::Tensor narrow = narrow_for_slice(m, so->nnz, cols.numel());
  GS_CALL(gs_sliced_e_square_sums(cptr(m.indptr), cptr(m.indices),
                                  narrow.defined() ? narrow.data_ptr<int32_t>() : nullptr,
                                  cptr(cols), cols.numel(), cptr(so->sub_indptr), so->nnz,
                                  cptr(e_ids), efeat.data_ptr<float>(), out.data_ptr<float>(),
                                  num_rows_, ws.data_ptr(), (size_t)ws.numel(), cur_stream()));
  return out;
}

// Shared by the plain and the super-batched form.  key_offset (per picked
// column) and `picked` carry the batch in their values when there are batches.
static MajorResult col_row_slice(const Compressed& m, const torch::Tensor& cols,
                                 const torch::Tensor& sub_indptr, int64_t nnz,
                                 const torch::Tensor& key_offset, const torch::Tensor& picked,
                                 bool with_coo, torch::Tensor* firsts = nullptr,
                                 torch::Tensor* zeros = nullptr) {
  const int64_t n = cols.numel(), np = picked.numel();
  MajorResult r;
  r.indptr = new_ids(n + 1, m.indptr);
  // the number of kept edges goes straight to pinned host memory; the fill pass
  // is queued into buffers sized by the bound (every edge kept) and runs while
  // the number travels
  AsyncCount kept = AsyncCount::mirrored();
  const torch::Tensor narrow = narrow_for_slice(m, nnz, n);
  // (the relabel of a slice with far fewer rows than edges goes by its rows' first edges)
  // (and its edges' values are often divided by sums over their columns: cleared in passing)
  const bool tells = firsts && nnz >= 8 * np && gs_col_row_slice_tells_first(nnz, np);
  torch::Tensor ws = new_workspace(tells ? gs_col_row_slice_first_workspace_bytes(nnz, np)
                                         : gs_minor_slice_workspace_bytes(nnz, np), m.indptr);
  if (zeros) {
    const torch::Tensor buffer = new_ids((tells ? np : 0) + n, m.indptr);
    *zeros = piece_of(buffer, 0, n, false);
    if (tells) *firsts = piece_of(buffer, n, np, false);
  }
  GS_CALL(gs_col_row_slice_count_first(
      cptr(m.indptr), cptr(m.indices), narrow.defined() ? narrow.data_ptr<int32_t>() : nullptr,
      cptr(cols), cptr(key_offset), n, cptr(sub_indptr), nnz, cptr(picked), np, mptr(r.indptr),
      kept.mirror(), tells ? mptr(*firsts) : nullptr, zeros ? (double*)mptr(*zeros) : nullptr,
      ws.data_ptr(), ws.numel(), cur_stream()));
  kept.arm();
  const int64_t size = nnz <= kBoundLimit ? nnz : kept.get();
  r.minor_ids = new_ids(size, m.indptr);
  r.select = new_ids(size, m.indptr);
  if (with_coo) r.major_ids = new_ids(size, m.indptr);
  GS_CALL(gs_col_row_slice_fill(cptr(m.indptr), cptr(m.indices), cptr(cols), n,
                                cptr(sub_indptr), nnz, np,
                                with_coo ? mptr(r.major_ids) : nullptr, mptr(r.minor_ids),
                                mptr(r.select), ws.data_ptr(), ws.numel(), cur_stream()));
  const int64_t k = kept.get();
  r.minor_ids = trim_to(r.minor_ids, k);
  r.select = trim_to(r.select, k);
  if (with_coo) r.major_ids = trim_to(r.major_ids, k);
  return r;
}

// A[rows, cols]: rows become positions in `rows`, columns positions in `cols`;
// the edge index addresses this matrix's edges.
GraphAndIndex Graph::ColRowSlicing(torch::Tensor cols, torch::Tensor rows, int64_t on_format,
                                   int64_t output_format) {
  TORCH_CHECK(on_format == kCSC, "ColRowSlicing runs on the CSC format, got ", on_format);
  TORCH_CHECK(output_format != 0 && (output_format & kCSR) == 0,
              "ColRowSlicing produces CSC and COO, got output_format ", output_format);
  cols = ids(cols, "cols");
  rows = ids(rows, "rows");
  const Compressed& m = compressed(kCSC);
  const std::shared_ptr<SliceOffsets> shared = slice_offsets_for(cols);
  SliceOffsets& so = *shared;
  MajorResult r;
  torch::Tensor firsts, zeros;
  if (read_in_place(m, so.nnz, cols.numel())) {
    r = col_row_slice(m, cols, so.sub_indptr, so.nnz, torch::Tensor(), rows,
                      output_format & kCOO, &firsts, &zeros);
  } else {
    const MajorResult& sliced = written_slice(so);
    Compressed tmp(sliced.indptr, sliced.minor_ids);
    r = minor_slice(tmp, rows, output_format & kCOO);
    r.select = sliced.select.index_select(0, r.select);
  }
  GraphPtr g = derive(kCSC, output_format, r, rows.numel(), cols.numel());
  g->keep_row_firsts(firsts, r.minor_ids);
  g->keep_column_zeros(zeros);
  return {g, edge_index(m.e_ids, r.select)};
}

// Plain float32 values on the GPU, one a place, which nothing else has to see.
static bool plain_row_of_values(const torch::Tensor& t) {
  return plain_values(t, false) && t.dim() == 1 && t.is_contiguous() && t.size(0) > 0;
}

// Whether the edge values that such a slice is to hand on, divided by those of its rows, can
// be left by the pass that labels its edges (as NormaliseColumns says).
static bool values_in_passing(const Compressed& m, const c10::optional<torch::Tensor>& values,
                              const c10::optional<torch::Tensor>& row_divisor, int64_t num_rows) {
  if (!values.has_value()) return !row_divisor.has_value();
  return !m.e_ids.has_value() && plain_row_of_values(*values) &&
         (!row_divisor.has_value() ||
          (plain_row_of_values(*row_divisor) && row_divisor->size(0) >= num_rows)) &&
         !at::impl::torch_function_mode_enabled() && !at::autocast::is_autocast_enabled(at::kCUDA);
}

// What the kept edges of a row slice are handed on as.  Passes of compiled samplers, us, with
// the slice written first and handed on, when that came: LADIES of 512 seeds 631, 571; of 8
// batches of 128 seeds 693, 643; FastGCN of 1024 seeds 284, 228; subgraphs of 8.4 M edges between
// 19 K nodes 240, 218.
struct HandedOn {
  torch::Tensor row, col, values;
  // Behind the count pass; the arrays are sized by the slice's edges until trimmed.
  void queue(const Compressed& m, const torch::Tensor& cols, const torch::Tensor& sub_indptr,
             int64_t nnz, int64_t num_picked, const int64_t* row_label, const int64_t* col_label,
             const c10::optional<torch::Tensor>& of, const c10::optional<torch::Tensor>& divisor,
             torch::Tensor& ws) {
    row = new_ids(nnz, m.indptr), col = new_ids(nnz, m.indptr);
    if (of.has_value()) values = torch::empty({nnz}, of->options().requires_grad(false));
    GS_CALL(gs_col_row_slice_labels(
        cptr(m.indptr), cptr(cols), cols.numel(), cptr(sub_indptr), nnz, num_picked, row_label,
        col_label, mptr(row), mptr(col), of.has_value() ? of->data_ptr<float>() : nullptr,
        of.has_value() ? of->size(0) : 0, divisor.has_value() ? divisor->data_ptr<float>() : nullptr,
        of.has_value() ? values.data_ptr<float>() : nullptr, ws.data_ptr(), ws.numel(),
        cur_stream()));
  }
  // Of `kept` edges: the values by their sums over columns, which are cleared.
  void finish(int64_t kept, const torch::Tensor& indptr, double* sums) {
    if (values.defined() && kept > 0)
      GS_CALL(gs_normalise_columns_cleared(cptr(indptr), indptr.numel() - 1, nullptr, kept,
                                           values.data_ptr<float>(), kept, nullptr, nullptr, sums,
                                           values.data_ptr<float>(), cur_stream()));
    row = trim_to(row, kept), col = trim_to(col, kept);
    if (values.defined()) values = trim_to(values, kept);
  }
  c10::optional<torch::Tensor> normalised() const {
    return values.defined() ? c10::optional<torch::Tensor>(values) : c10::nullopt;
  }
};

// Worth it when the slice's edges outnumber its rows and columns by far, as
// `use_list_labels` says of those that are kept; here the number of these is not waited for.
c10::optional<std::tuple<torch::Tensor, torch::Tensor, torch::Tensor, c10::optional<torch::Tensor>>>
Graph::RelabelledRows(torch::Tensor cols, torch::Tensor rows, c10::optional<torch::Tensor> values,
                      c10::optional<torch::Tensor> row_divisor) {
  const Compressed& m = compressed(kCSC);
  const int64_t R = rows.numel(), S = cols.numel();
  if (!m.indices.is_cuda() || !m.indptr.is_cuda() || R == 0 || S == 0 ||
      R + S > GS_LIST_LABELS_MAX_KEYS || !values_in_passing(m, values, row_divisor, R))
    return {};
  cols = ids(cols, "cols");
  rows = ids(rows, "rows");
  const std::shared_ptr<SliceOffsets> so = slice_offsets_for(cols);
  const int64_t nnz = so->nnz;
  if (nnz < 8 * (R + S) || nnz > kBoundLimit || !gs_col_row_slice_tells_first(nnz, R)) return {};
  const torch::Tensor narrow = narrow_for_slice(m, nnz, S);
  torch::Tensor ws = new_workspace(gs_col_row_slice_first_workspace_bytes(nnz, R), m.indptr);
  torch::Tensor indptr = new_ids(S + 1, m.indptr);
  // first edges and labels of the rows, labels of the columns and their sums
  torch::Tensor small = new_ids(2 * R + 2 * S, m.indptr);
  int64_t* const first = mptr(small);
  int64_t* const row_label = first + R;
  int64_t* const col_label = row_label + R;
  double* const sums = (double*)(col_label + S);
  torch::Tensor frontier = new_ids(R + S, m.indptr);
  AsyncCount kept = AsyncCount::mirrored(), nodes = AsyncCount::mirrored();
  GS_CALL(gs_col_row_slice_count_labels(
      cptr(m.indptr), cptr(m.indices), narrow.defined() ? narrow.data_ptr<int32_t>() : nullptr,
      cptr(cols), S, cptr(so->sub_indptr), nnz, cptr(rows), R, mptr(indptr), kept.mirror(), first,
      sums, mptr(frontier), nodes.mirror(), row_label, col_label, ws.data_ptr(), ws.numel(),
      cur_stream()));
  kept.arm();
  nodes.arm();
  HandedOn edges;
  edges.queue(m, cols, so->sub_indptr, nnz, R, row_label, col_label, values, row_divisor, ws);
  const int64_t k = kept.get();
  edges.finish(k, indptr, sums);
  const int64_t n = nodes.get();
  if (k == 0 && values.has_value()) return {};  // (the operators say what the values of no edges are)
  return std::make_tuple(trim_to(frontier, n), edges.row, edges.col, edges.normalised());
}

void Graph::keep_row_firsts(const torch::Tensor& firsts, const torch::Tensor& edge_rows) {
  if (!firsts.defined()) return;
  row_firsts_ = firsts;
  row_firsts_of_ = edge_rows;
  row_firsts_version_ = (int64_t)edge_rows._version();
  row_firsts_epoch_ = cache_epoch();
}

void Graph::keep_column_zeros(const torch::Tensor& zeros) {
  if (!zeros.defined()) return;
  column_zeros_ = zeros;
  column_zeros_stream_ = cur_stream();
}

// (nothing where they are not this call's to use)
torch::Tensor Graph::take_column_zeros() {
  torch::Tensor zeros;
  std::lock_guard<std::mutex> lock(column_zeros_guard_);
  if (column_zeros_.defined() && column_zeros_.numel() == num_cols_ &&
      column_zeros_stream_ == cur_stream() && !capturing())
    std::swap(zeros, column_zeros_);
  return zeros;
}

// batch * stride for everything that the batches hold.
static torch::Tensor moves_by_batch(const torch::Tensor& bptr, int64_t n, int64_t stride) {
  torch::Tensor e = new_ids(n, bptr);
  GS_CALL(gs_encode_batch_ids(nullptr, cptr(bptr), bptr.numel() - 1, n, stride, mptr(e), cur_stream()));
  return e;
}

torch::Tensor Graph::SliceOffsets::kept_key_offset(const torch::Tensor& bptr) {
  std::lock_guard<std::mutex> lock(guard);
  return key_offset.defined() && key_bptr.is_same(bptr) &&
                 key_bptr_version == (int64_t)bptr._version()
             ? key_offset
             : torch::Tensor();
}
void Graph::SliceOffsets::keep_key_offset(const torch::Tensor& bptr, const torch::Tensor& offset) {
  std::lock_guard<std::mutex> lock(guard);
  key_offset = offset;
  key_bptr = bptr;
  key_bptr_version = (int64_t)bptr._version();
}
torch::Tensor Graph::key_offsets_for(SliceOffsets& so, const torch::Tensor& col_bptr) {
  torch::Tensor offset = so.kept_key_offset(col_bptr);
  if (!offset.defined()) {
    offset = moves_by_batch(col_bptr, so.cols.numel(), num_rows_);
    so.keep_key_offset(col_bptr, offset);
  }
  return offset;
}

// Per batch b: the columns col[col_bptr[b] : col_bptr[b+1]] restricted to the
// rows row[row_bptr[b] : row_bptr[b+1]]; row ids become positions in `row`.
// The returned edge index addresses the parent's edges.  One pass over the
// parent's columns (BatchCSCColRowSlicingCUDA,
// src/cuda/fusion/column_row_slicing.cu:356-362): a batch's rows and the row
// ids of its columns' edges are both moved by batch * num_rows, so one table of
// picked rows serves all batches.
GraphAndIndex Graph::BatchColRowSlcing(torch::Tensor col, torch::Tensor col_bptr,
                                       torch::Tensor row, torch::Tensor row_bptr) {
  col = ids(col, "col");
  row = ids(row, "row");
  col_bptr = ids(col_bptr, "col_bptr");
  row_bptr = ids(row_bptr, "row_bptr");
  TORCH_CHECK(col_bptr.numel() == row_bptr.numel() && col_bptr.numel() >= 2,
              "BatchColRowSlcing: column and row batch pointers must have the same length");
  BatchOffsets::check(col_bptr, col.numel(), "BatchColRowSlicing");
  BatchOffsets::check(row_bptr, row.numel(), "BatchColRowSlicing");
  const Compressed& m = compressed(kCSC);
  const int64_t stride = num_rows_;
  torch::Tensor key_offset, picked;
  if (row.is_same(col) && row_bptr.is_same(col_bptr)) {
    key_offset = new_ids(col.numel(), col_bptr);
    picked = new_ids(row.numel(), row_bptr);
    GS_CALL(gs_pick_batch_ids(cptr(row), row.numel(), nullptr, cptr(row_bptr), row_bptr.numel() - 1,
                              row.numel(), stride, nullptr, mptr(picked), mptr(key_offset),
                              nullptr, cur_stream()));
  } else {
    key_offset = moves_by_batch(col_bptr, col.numel(), stride);
    picked = new_ids(row.numel(), row_bptr);
    GS_CALL(gs_pick_batch_ids(cptr(row), row.numel(), nullptr, cptr(row_bptr), row_bptr.numel() - 1,
                              row.numel(), stride, nullptr, mptr(picked), nullptr, nullptr,
                              cur_stream()));
  }
  const std::shared_ptr<SliceOffsets> shared = slice_offsets_for(col);
  SliceOffsets& so = *shared;
  MajorResult kept;
  if (read_in_place(m, so.nnz, col.numel())) {
    kept = col_row_slice(m, col, so.sub_indptr, so.nnz, key_offset, picked, false);
  } else {
    // the batched column slice with rows moved by batch * num_rows is written and row-sliced
    MajorResult sliced = major_slice(m, col, false, col_bptr, stride);
    Compressed tmp(sliced.indptr, sliced.minor_ids);
    kept = minor_slice(tmp, picked, false);
    kept.select = sliced.select.index_select(0, kept.select);
  }
  auto g = c10::make_intrusive<Graph>(row.numel(), col.numel());
  auto csc = std::make_shared<Compressed>();
  csc->indptr = kept.indptr;
  csc->indices = kept.minor_ids;
  g->csc_ = csc;
  g->num_edges_ = kept.select.numel();
  g->col_bptr_ = col_bptr;
  g->row_bptr_ = row_bptr;
  g->orig_col_ids_ = col;
  g->orig_row_ids_ = row;
  g->edge_bptr_ = taken_offsets(kept.indptr, col_bptr);
  BatchOffsets::trust(g->edge_bptr_, g->num_edges_);
  if (row.is_same(col) && row_bptr.is_same(col_bptr)) {
    g->square_rows_ = kept.minor_ids;
    g->square_rows_version_ = (int64_t)kept.minor_ids._version();
    g->square_rows_epoch_ = cache_epoch();
  }
  return {g, edge_index(m.e_ids, kept.select)};
}

// What a layer-wise sampler asks an encoded slice (BatchColSlicing with encoding) for:
// its rows with where every batch's begin, and the sums of its squared edge values on
// them.  The slice is not written; the picked rows' edges come from EncodedPickedRows.
// Nothing where the slice has to be written after all: values that are no plain float32
// edge data, or keys too many or too few for the pass.
c10::optional<std::tuple<torch::Tensor, torch::Tensor, torch::Tensor>> Graph::EncodedSquareSums(
    torch::Tensor seeds, torch::Tensor col_bptr, torch::Tensor efeat) {
  const Compressed& m = compressed(kCSC);
  if (!m.indices.is_cuda() || !efeat.defined() || !efeat.is_cuda() ||
      efeat.scalar_type() != torch::kFloat32 || efeat.dim() != 1 || !efeat.is_contiguous() ||
      efeat.numel() != m.indices.numel())
    return {};
  seeds = ids(seeds, "seeds");
  col_bptr = ids(col_bptr, "col_bptr");
  const int64_t B = col_bptr.numel() - 1;
  TORCH_CHECK(B >= 1, "BatchColSlicing: col_bptr needs at least two entries");
  BatchOffsets::check(col_bptr, seeds.numel(), "BatchColSlicing");
  const int64_t stride = num_rows_, n = seeds.numel();
  const std::shared_ptr<SliceOffsets> shared = slice_offsets_for(seeds);
  const int64_t nnz = shared->nnz;
  if (!gs_encoded_square_sums_pay(nnz, B, stride)) return {};
  torch::Tensor key_offset = key_offsets_for(*shared, col_bptr);
  torch::Tensor row_bptr = new_ids(B + 1, m.indptr);
  torch::Tensor ws = new_workspace(gs_encoded_square_sums_workspace_bytes(nnz, B, stride), m.indptr);
  const torch::Tensor narrow = m.narrow_indices(2 * nnz);  // the row slice reads them as well
  const torch::Tensor e_ids = m.e_ids.has_value() ? m.e_ids.value() : torch::Tensor();
  int64_t* mirror = OffsetMirror::reserve(row_bptr);
  GS_CALL(gs_encoded_square_sums(cptr(m.indptr), cptr(m.indices),
                                 narrow.defined() ? narrow.data_ptr<int32_t>() : nullptr,
                                 cptr(seeds), n, cptr(shared->sub_indptr), nnz, cptr(key_offset), B,
                                 stride, cptr(e_ids), efeat.data_ptr<float>(), mptr(row_bptr),
                                 mirror, ws.data_ptr(), (size_t)ws.numel(), cur_stream()));
  OffsetMirror::arm(row_bptr);
  const int64_t bound = std::min(nnz, B * stride);
  torch::Tensor rows = new_ids(bound, m.indptr);
  torch::Tensor sums = torch::empty({bound}, efeat.options().requires_grad(false));
  GS_CALL(gs_encoded_square_sums_rows(nnz, B, stride, mptr(rows), sums.data_ptr<float>(),
                                      ws.data_ptr(), (size_t)ws.numel(), cur_stream()));
  const int64_t total = OffsetMirror::values(row_bptr).back();
  BatchOffsets::trust(row_bptr, total);
  return std::make_tuple(trim_to(rows, total), row_bptr, trim_to(sums, total));
}

// BatchRowSlicing of the encoded slice of (seeds, col_bptr) by row_ids, positions in
// `rows` (EncodedSquareSums) that lie in it; the edge index addresses this matrix's edges.
// `picked`: rows[row_ids], moved by batch * num_rows.
GraphAndIndex Graph::encoded_row_slice(const torch::Tensor& seeds, const torch::Tensor& col_bptr,
                                       const torch::Tensor& picked, const torch::Tensor& row_ids,
                                       const torch::Tensor& row_bptr) {
  const Compressed& m = compressed(kCSC);
  const std::shared_ptr<SliceOffsets> shared = slice_offsets_for(seeds);
  torch::Tensor key_offset = key_offsets_for(*shared, col_bptr);
  torch::Tensor firsts, zeros;
  const MajorResult r = col_row_slice(m, seeds, shared->sub_indptr, shared->nnz, key_offset, picked,
                                      true, &firsts, &zeros);
  GraphPtr g = derive(kCSC, kCSC | kCOO, r, row_ids.numel(), seeds.numel());
  g->keep_row_firsts(firsts, r.minor_ids);
  g->keep_column_zeros(zeros);
  g->col_bptr_ = col_bptr;
  g->orig_col_ids_ = seeds;
  g->row_encoding_size_ = num_rows_;
  g->edge_bptr_ = taken_offsets(g->csc_->indptr, col_bptr);
  BatchOffsets::trust(g->edge_bptr_, g->num_edges_);
  g->row_bptr_ = row_bptr;
  g->orig_row_ids_ = row_ids;
  return {g, edge_index(m.e_ids, r.select)};
}

static void check_encoded(torch::Tensor& seeds, torch::Tensor& col_bptr, torch::Tensor& row_ids,
                          torch::Tensor& row_bptr) {
  seeds = ids(seeds, "seeds");
  col_bptr = ids(col_bptr, "col_bptr");
  row_ids = ids(row_ids, "row_ids");
  row_bptr = ids(row_bptr, "row_bptr");
  TORCH_CHECK(col_bptr.numel() == row_bptr.numel() && col_bptr.numel() >= 2,
              "BatchRowSlicing: column and row batch pointers must have the same length");
  BatchOffsets::check(col_bptr, seeds.numel(), "BatchColSlicing");
  BatchOffsets::check(row_bptr, row_ids.numel(), "BatchRowSlicing");
}

// Behind a wait for something queued after the picks' ids.
static void check_picks(const HostFlag& refused, const torch::Tensor& rows) {
  TORCH_CHECK(!refused.raised(), "BatchRowSlicing: a picked row lies outside the ", rows.numel(),
              " rows of the slice");
}

std::tuple<GraphPtr, torch::Tensor, torch::Tensor> Graph::EncodedPickedRows(
    torch::Tensor seeds, torch::Tensor col_bptr, torch::Tensor rows, torch::Tensor row_ids,
    torch::Tensor row_bptr) {
  check_encoded(seeds, col_bptr, row_ids, row_bptr);
  rows = ids(rows, "rows");
  const int64_t n = row_ids.numel();
  torch::Tensor picked = new_ids(n, row_ids), names = new_ids(n, row_ids);
  HostFlag refused;
  GS_CALL(gs_pick_batch_ids(cptr(rows), rows.numel(), cptr(row_ids), cptr(row_bptr),
                            row_bptr.numel() - 1, n, num_rows_, mptr(names), mptr(picked), nullptr,
                            refused.word(), cur_stream()));
  auto got = encoded_row_slice(seeds, col_bptr, picked, row_ids, row_bptr);  // (waits for a count)
  check_picks(refused, rows);
  return {std::get<0>(got), std::get<1>(got), names};
}

static c10::intrusive_ptr<BlockBatch> blocks_of(const HandedOn& edges, const torch::Tensor& indptr,
                                                const torch::Tensor& col_bptr,
                                                const torch::Tensor& seeds) {
  auto out = c10::make_intrusive<BlockBatch>();
  out->num_batches = col_bptr.numel() - 1;
  out->sampled_indptr = indptr;
  out->row = edges.row;
  out->col = edges.col;
  out->col_seeds = seeds;
  out->num_dst_total = seeds.numel();
  out->coo_ptr = taken_offsets(indptr, col_bptr);
  BatchOffsets::trust(out->coo_ptr, edges.row.numel());
  out->col_bptr = col_bptr;
  return out;
}

// Whether the keys of every batch fit the one work-group that labels them: known before
// anything is queued (a batch that does not would be refused behind the whole slice).
static bool batches_fit_labels(const torch::Tensor& col_bptr, const torch::Tensor& row_bptr) {
  const std::vector<int64_t> cols = OffsetMirror::values(col_bptr);
  const std::vector<int64_t>& rows = OffsetMirror::values(row_bptr);
  for (size_t b = 0; b + 1 < cols.size(); ++b)
    if (cols[b + 1] - cols[b] + rows[b + 1] - rows[b] > GS_LIST_LABELS_MAX_KEYS) return false;
  return true;
}

// (every kept edge's row lies in its batch's segment of the list: both are moved by the batch)
c10::optional<std::tuple<c10::intrusive_ptr<BlockBatch>, c10::optional<torch::Tensor>>>
Graph::EncodedBlocks(torch::Tensor seeds, torch::Tensor col_bptr, torch::Tensor rows,
                     torch::Tensor row_ids, torch::Tensor row_bptr,
                     c10::optional<torch::Tensor> values,
                     c10::optional<torch::Tensor> row_divisor) {
  const Compressed& m = compressed(kCSC);
  check_encoded(seeds, col_bptr, row_ids, row_bptr);
  rows = ids(rows, "rows");
  const int64_t R = row_ids.numel(), S = seeds.numel(), B = col_bptr.numel() - 1;
  if (!m.indices.is_cuda() || R == 0 || S == 0 || R + S > B * (GS_LIST_LABELS_MAX_KEYS / 2) ||
      !values_in_passing(m, values, row_divisor, R) || !batches_fit_labels(col_bptr, row_bptr))
    return {};
  const std::shared_ptr<SliceOffsets> so = slice_offsets_for(seeds);
  const int64_t nnz = so->nnz;
  if (nnz < 8 * (R + S) || nnz > kBoundLimit || !gs_col_row_slice_tells_first(nnz, R)) return {};
  torch::Tensor key_offset = key_offsets_for(*so, col_bptr);
  torch::Tensor picked = new_ids(R, row_ids), names = new_ids(R, row_ids);
  HostFlag refused;
  GS_CALL(gs_pick_batch_ids(cptr(rows), rows.numel(), cptr(row_ids), cptr(row_bptr), B, R, num_rows_,
                            mptr(names), mptr(picked), nullptr, refused.word(), cur_stream()));
  const torch::Tensor narrow = narrow_for_slice(m, nnz, S);
  torch::Tensor ws = new_workspace(gs_col_row_slice_first_workspace_bytes(nnz, R), m.indptr);
  torch::Tensor indptr = new_ids(S + 1, m.indptr), unique_ptr = new_ids(B + 1, m.indptr);
  torch::Tensor frontier = new_ids(R + S, m.indptr);
  // first edges and labels of the rows, labels of the columns and their sums, scratch
  torch::Tensor small = new_ids(3 * R + 3 * S + B + 1, m.indptr);
  int64_t* const first = mptr(small);
  int64_t* const row_label = first + R;
  int64_t* const col_label = row_label + R;
  double* const sums = (double*)(col_label + S);
  int64_t* const scratch = col_label + 2 * S;
  AsyncCount kept = AsyncCount::mirrored();
  int64_t* mirror = OffsetMirror::reserve(unique_ptr);
  GS_CALL(gs_col_row_slice_count_batch_labels(
      cptr(m.indptr), cptr(m.indices), narrow.defined() ? narrow.data_ptr<int32_t>() : nullptr,
      cptr(seeds), cptr(key_offset), S, cptr(so->sub_indptr), nnz, cptr(picked), R, mptr(indptr),
      kept.mirror(), first, sums, cptr(col_bptr), cptr(names), cptr(row_bptr), num_rows_, B,
      mptr(frontier), mptr(unique_ptr), mirror, row_label, col_label, scratch, ws.data_ptr(),
      ws.numel(), cur_stream()));
  kept.arm();
  OffsetMirror::arm(unique_ptr);
  HandedOn edges;
  edges.queue(m, seeds, so->sub_indptr, nnz, R, row_label, col_label, values, row_divisor, ws);
  const int64_t k = kept.get();
  check_picks(refused, rows);
  edges.finish(k, indptr, sums);
  c10::intrusive_ptr<BlockBatch> out = blocks_of(edges, indptr, col_bptr, seeds);
  const int64_t total = OffsetMirror::values(unique_ptr).back();
  if (k == 0 && values.has_value()) return {};  // (the operators say what the values of no edges are)
  BatchOffsets::trust(unique_ptr);
  out->frontier_ptr = unique_ptr;
  out->frontier = frontier.narrow(0, 0, total);
  return std::make_tuple(out, edges.normalised());
}

c10::optional<c10::intrusive_ptr<BlockBatch>> Graph::SubgraphBlocks(torch::Tensor nodes,
                                                                    torch::Tensor nodes_ptr) {
  nodes = ids(nodes, "col");
  nodes_ptr = ids(nodes_ptr, "col_bptr");
  const Compressed& m = compressed(kCSC);
  const int64_t n = nodes.numel(), B = nodes_ptr.numel() - 1;
  if (!m.indices.is_cuda() || n == 0 || B < 1) return {};
  BatchOffsets::check(nodes_ptr, n, "BatchColRowSlicing");
  slice_offsets_for(nodes, false);
  torch::Tensor picked = new_ids(n, nodes), key_offset = new_ids(n, nodes);
  GS_CALL(gs_pick_batch_ids(cptr(nodes), n, nullptr, cptr(nodes_ptr), B, n, num_rows_, nullptr,
                            mptr(picked), mptr(key_offset), nullptr, cur_stream()));
  const std::shared_ptr<SliceOffsets> so = slice_offsets_for(nodes);
  const int64_t nnz = so->nnz;
  if (nnz < n || nnz > kBoundLimit) return {};
  const torch::Tensor narrow = narrow_for_slice(m, nnz, n);
  torch::Tensor ws = new_workspace(gs_minor_slice_workspace_bytes(nnz, n), m.indptr);
  torch::Tensor indptr = new_ids(n + 1, m.indptr), label = new_ids(n, m.indptr);
  AsyncCount kept = AsyncCount::mirrored();
  GS_CALL(gs_col_row_slice_count(
      cptr(m.indptr), cptr(m.indices), narrow.defined() ? narrow.data_ptr<int32_t>() : nullptr,
      cptr(nodes), cptr(key_offset), n, cptr(so->sub_indptr), nnz, cptr(picked), n, mptr(indptr),
      kept.mirror(), ws.data_ptr(), ws.numel(), cur_stream()));
  kept.arm();
  // an edge's ends are nodes of the list, so the frontier is the list's unique nodes
  auto of = c10::make_intrusive<Graph>(n, n);
  LabelRequest labels{nullptr, nullptr, mptr(label), nullptr};
  Frontier& f = of->frontier_for(nodes, nodes, nodes_ptr, nodes_ptr, &labels);
  HandedOn edges;
  edges.queue(m, nodes, so->sub_indptr, nnz, n, cptr(label), cptr(label), {}, {}, ws);
  edges.finish(kept.get(), indptr, nullptr);
  c10::intrusive_ptr<BlockBatch> out = blocks_of(edges, indptr, nodes_ptr, nodes);
  out->frontier_ptr = f.unique_ptr;
  out->frontier = f.frontier();
  return out;
}

}  // namespace gs

// batch_graph.cc -- super-batch operators: B independent mini-batches share one
// launch; per-batch boundaries travel as int64[B + 1] pointer arrays
// (col_bptr over the seed columns, edge_bptr over the edges, row_bptr over
// compacted rows).  Mirrors the interface of src/batch_graph.cc of gSampler.
#include "abi_call.h"
#include "graph.h"

namespace gs {

void Graph::copy_batch_state_to(Graph& g, bool with_rows) {
  g.col_bptr_ = col_bptr_;
  g.orig_col_ids_ = orig_col_ids_;
  if (with_rows) {
    g.row_bptr_ = row_bptr_;
    g.orig_row_ids_ = orig_row_ids_;
  }
  g.row_encoding_size_ = row_encoding_size_;
  if (g.csc_ && col_bptr_.defined()) {
    g.edge_bptr_ = g.csc_->indptr.index_select(0, col_bptr_);
    BatchOffsets::trust(g.edge_bptr_);
  }
}

std::tuple<torch::Tensor, torch::Tensor> Graph::BatchGetCSCIndptr() {
  CreateSparseFormat(kCSC);
  return {csc_->indptr, col_bptr_};
}
std::tuple<torch::Tensor, torch::Tensor> Graph::BatchGetCSCIndices() {
  CreateSparseFormat(kCSC);
  return {csc_->indices, edge_bptr_};
}
std::tuple<torch::Tensor, torch::Tensor> Graph::BatchGetCSCEids() {
  CreateSparseFormat(kCSC);
  if (csc_->e_ids.has_value()) return {csc_->e_ids.value(), edge_bptr_};
  return {torch::Tensor(), torch::Tensor()};
}
std::tuple<torch::Tensor, torch::Tensor> Graph::BatchGetCOORows() {
  CreateSparseFormat(kCOO);
  return {coo_->row, edge_bptr_};
}
std::tuple<torch::Tensor, torch::Tensor> Graph::BatchGetCOOCols() {
  CreateSparseFormat(kCOO);
  return {coo_->col, edge_bptr_};
}
std::tuple<torch::Tensor, torch::Tensor> Graph::BatchGetCOOEids() {
  CreateSparseFormat(kCOO);
  if (coo_->e_ids.has_value()) return {coo_->e_ids.value(), edge_bptr_};
  return {torch::Tensor(), torch::Tensor()};
}

static const std::vector<int64_t>& host_offsets(const torch::Tensor& offset) {
  if (offset.scalar_type() != torch::kInt64)
    return OffsetMirror::values(offset.to(torch::kInt64));
  return OffsetMirror::values(offset);
}

std::vector<int64_t> Graph::BatchGetColCounts() {
  TORCH_CHECK(col_bptr_.defined() && col_bptr_.numel() > 0,
              "BatchGetColCounts: no column batch pointer set");
  const std::vector<int64_t>& p = host_offsets(col_bptr_);
  std::vector<int64_t> counts(p.size() - 1);
  for (size_t i = 0; i < counts.size(); ++i) counts[i] = p[i + 1] - p[i];
  return counts;
}

// Decodes ids of the form id + batch * stride (row encoding of batched
// slicing): returns (per-batch offsets into the sorted encoded array, original
// ids).  Counterpart of GetBatchOffsets, src/cuda/batch/encoding_decoding.cu:99.
static std::tuple<torch::Tensor, torch::Tensor> batch_offsets(
    const torch::Tensor& encoded, int64_t num_batches, int64_t stride) {
  const int64_t n = encoded.numel();
  torch::Tensor batch = new_ids(n, encoded), orig = new_ids(n, encoded);
  GS_CALL(gs_decode_batch_ids(cptr(encoded), n, stride, mptr(orig), mptr(batch),
                              cur_stream()));
  torch::Tensor ptr = new_ids(num_batches + 1, encoded);
  GS_CALL(gs_sorted_to_indptr(cptr(batch), n, num_batches, mptr(ptr),
                              cur_stream()));
  return {ptr, orig};
}

// The rows of an encoded slice are numbered through one flag byte per
// (batch, row) while those bytes are cheap next to the edges: clearing and
// reading them back streams at several TB/s, a sort of the edges' keys costs
// about 50 ps per key and pass, ten passes, and a dozen launches.
static bool compact_by_flags(int64_t num_batches, int64_t stride, int64_t nnz) {
  constexpr int64_t kAlways = int64_t(1) << 24, kNever = int64_t(1) << 30;
  if (stride == 0 || num_batches > kNever / stride) return false;
  const int64_t keys = num_batches * stride;
  return keys <= kAlways || keys / 256 <= nnz;
}

// The encoded slice with its rows numbered anew, and those rows: which ids, and
// where every batch's begin (compact.hip).
static MajorResult compact_slice(const Compressed& m, const torch::Tensor& cols,
                                 const torch::Tensor& offsets, int64_t nnz,
                                 const torch::Tensor& col_bptr, int64_t stride,
                                 torch::Tensor* row_bptr, torch::Tensor* rows) {
  const int64_t B = col_bptr.numel() - 1, n = cols.numel();
  MajorResult r;
  r.indptr = offsets;
  torch::Tensor key_offset = new_ids(n, m.indptr);
  *row_bptr = new_ids(B + 1, m.indptr);
  torch::Tensor ws = new_workspace(gs_slice_compact_workspace_bytes(B, stride), m.indptr);
  const torch::Tensor narrow = m.narrow_indices(nnz);  // two passes read every id of the slice
  const int32_t* ids32 = narrow.defined() ? narrow.data_ptr<int32_t>() : nullptr;
  int64_t* mirror = OffsetMirror::reserve(*row_bptr);
  GS_CALL(gs_slice_compact_count(cptr(m.indptr), cptr(m.indices), ids32, cptr(cols), n,
                                 cptr(offsets), nnz, cptr(col_bptr), B, stride, mptr(key_offset),
                                 mptr(*row_bptr), mirror, ws.data_ptr(), ws.numel(),
                                 cur_stream()));
  OffsetMirror::arm(*row_bptr);
  torch::Tensor bound = new_ids(std::min(nnz, B * stride), m.indptr);
  r.minor_ids = new_ids(nnz, m.indptr);
  r.select = new_ids(nnz, m.indptr);
  r.major_ids = new_ids(nnz, m.indptr);
  GS_CALL(gs_slice_compact_fill(cptr(m.indptr), cptr(m.indices), ids32, cptr(cols), n,
                                cptr(offsets), nnz, cptr(key_offset), B, stride, mptr(bound),
                                mptr(r.major_ids), mptr(r.minor_ids), mptr(r.select),
                                ws.data_ptr(), ws.numel(), cur_stream()));
  const int64_t total = OffsetMirror::values(*row_bptr).back();
  BatchOffsets::trust(*row_bptr, total);
  *rows = trim_to(bound, total);
  return r;
}

GraphAndIndex Graph::BatchColSlicing(torch::Tensor seeds, torch::Tensor col_bptr,
                                     bool encoding) {
  seeds = ids(seeds, "seeds");
  col_bptr = ids(col_bptr, "col_bptr");
  const int64_t B = col_bptr.numel() - 1;
  TORCH_CHECK(B >= 1, "BatchColSlicing: col_bptr needs at least two entries");
  BatchOffsets::check(col_bptr, seeds.numel(), "BatchColSlicing");
  const Compressed& m = compressed(kCSC);
  const int64_t stride = num_rows_;
  MajorResult r;
  torch::Tensor row_bptr, orig_rows;
  if (!encoding) {
    r = major_slice(m, seeds, true, col_bptr, 0);
  } else {
    int64_t nnz = 0;
    torch::Tensor offsets = slice_offsets(m, seeds, &nnz);
    if (compact_by_flags(B, stride, nnz)) {
      r = compact_slice(m, seeds, offsets, nnz, col_bptr, stride, &row_bptr, &orig_rows);
    } else {
      // few edges of a huge range of keys: sorted unique + rank of every edge's row
      r = major_slice(m, seeds, true, col_bptr, stride);
      auto uniq = torch::_unique2(r.minor_ids, /*sorted=*/true,
                                  /*return_inverse=*/true, /*return_counts=*/false);
      r.minor_ids = std::get<1>(uniq);
      std::tie(row_bptr, orig_rows) = batch_offsets(std::get<0>(uniq), B, stride);
      BatchOffsets::trust(row_bptr);
    }
  }
  const int64_t new_rows = encoding ? orig_rows.numel() : num_rows_ * B;
  GraphPtr g = derive(kCSC, kCSC | kCOO, r, new_rows, seeds.numel());
  g->col_bptr_ = col_bptr;
  g->orig_col_ids_ = seeds;
  g->edge_bptr_ = taken_offsets(r.indptr, col_bptr);
  BatchOffsets::trust(g->edge_bptr_, g->num_edges_);
  if (encoding) {
    g->row_bptr_ = row_bptr;
    g->orig_row_ids_ = orig_rows;
    g->row_encoding_size_ = stride;
  }
  return {g, edge_index(m.e_ids, r.select)};
}

GraphAndIndex Graph::BatchRowSlicing(torch::Tensor row_ids,
                                     torch::Tensor row_bptr) {
  BatchOffsets::check(ids(row_bptr, "row_bptr"), row_ids.numel(), "BatchRowSlicing");
  auto ret = Slicing(row_ids, 0, kCSC, kCSC | kCOO);
  Graph& g = *std::get<0>(ret);
  copy_batch_state_to(g, false);
  g.row_bptr_ = row_bptr;
  g.orig_row_ids_ = row_ids;
  return ret;
}

GraphAndIndex Graph::BatchRowSampling(int64_t fanout, bool replace) {
  auto ret = Sampling(1, fanout, replace, kCSC, kCSC | kCOO);
  copy_batch_state_to(*std::get<0>(ret), true);
  return ret;
}

GraphAndIndex Graph::BatchRowSamplingProbs(int64_t fanout, bool replace,
                                           torch::Tensor edge_probs) {
  auto ret = SamplingProbs(1, edge_probs, fanout, replace, kCSC, kCSC | kCOO);
  copy_batch_state_to(*std::get<0>(ret), true);
  return ret;
}

// One launch samples the columns of every batch: a column's picks depend on
// its position in the concatenated seed array, never on the batch split.
GraphAndIndex Graph::BatchFusedSlicingSampling(torch::Tensor seeds,
                                               torch::Tensor col_bptr,
                                               int64_t fanout, bool replace) {
  col_bptr = ids(col_bptr, "col_bptr");
  BatchOffsets::check(col_bptr, seeds.numel(), "BatchFusedSlicingSampling");
  EdgeCount::HintScope batch(col_bptr);  // the sampler leaves the edge pointer here
  // compressed by column only: the relabel pass reads the column pointer, and
  // the coordinate form is expanded from it if somebody asks
  auto ret = FusedSlicingSampling(1, seeds, fanout, replace, kCSC, kCSC);
  Graph& g = *std::get<0>(ret);
  g.col_labels_ = EdgeCount::hint().col_labels;
  g.col_bptr_ = col_bptr;
  g.orig_col_ids_ = ids(seeds, "seeds");
  g.edge_bptr_ = EdgeCount::hint().edge_bptr;
  if (!g.edge_bptr_.defined()) g.edge_bptr_ = g.csc_->indptr.index_select(0, col_bptr);
  BatchOffsets::trust(g.edge_bptr_, g.num_edges_);
  return ret;
}

// A compressed-by-column matrix whose coordinate form nobody has asked for
// hands over its column pointer; the coordinate form is then not built at all.
Graph::ColumnOrderedEdges Graph::column_ordered_edges(const char* who) {
  if (csc_ && !coo_) return {csc_->indices, {}, csc_->indptr, csc_->e_ids};
  CreateSparseFormat(kCOO);
  TORCH_CHECK(coo_->col_sorted, who, ": the COO format must be column-sorted");
  return {coo_->row, coo_->col, {}, coo_->e_ids};
}

// Global row ids of every edge as the relabel pass needs them: rows of an
// encoded (compacted) batch graph are decoded back through row_ids.  Rows that the list does
// not have (written by the caller, or a list that is too short) are refused by frontier_of().
torch::Tensor Graph::batch_rows_for_relabel(const torch::Tensor& edge_rows,
                                            const torch::Tensor& row_ids) {
  if (row_ids.numel() == 0) return edge_rows;
  if (!(mapped_out_.defined() && mapped_from_.is_same(edge_rows) &&
        mapped_by_.is_same(row_ids))) {
    torch::Tensor table = ids(row_ids, "row_ids");
    mapped_refused_.emplace();
    mapped_out_ = new_ids(edge_rows.numel(), edge_rows);
    GS_CALL(gs_local_ids(cptr(table), table.numel(), cptr(edge_rows), edge_rows.numel(),
                         row_encoding_size_, mptr(mapped_out_), mapped_refused_->word(),
                         cur_stream()));
    mapped_from_ = edge_rows;
    mapped_by_ = row_ids;
  }
  return mapped_out_;
}

// The frontier, once it has arrived; behind it the kernel that mapped the rows has, too.
const torch::Tensor& Graph::frontier_of(Frontier& f, const char* who) {
  const torch::Tensor& frontier = f.frontier();
  if (!mapped_refused_.has_value()) return frontier;
  const bool refused = mapped_refused_->raised();
  mapped_refused_.reset();
  if (refused) {
    const int64_t listed = mapped_by_.numel();
    mapped_out_ = mapped_from_ = mapped_by_ = torch::Tensor();
    frontier_.reset();
    TORCH_CHECK(false, who, ": the row of an edge lies outside the ", listed, " row ids given");
  }
  return frontier;
}

// A pass over the edges finds the first edge of every listed id: in LDS for a few
// thousand ids, with an atomic in device memory for an edge of one of more, where
// edges soon queue for their id.  all_nodes() and to_dgl_block() together, by the
// list and by the general path, us:
//   4 batches of 192 keys, 512 ids                     56 K edges   78   115
//   16 batches of 192 keys, 2048 ids                  875 K         84   158
//   16 batches of 450 keys, 4800 ids                   48 K         88   109
//                                                     177 K        110   109
//                                                     694 K        262   138
//   64 batches of 192 keys, 8192 ids                  123 K         86   107
//                                                     461 K        136   113
//   64 batches of 1000 keys, 44 800 ids               295 K         91    99
//                                                     4.1 M        647   171
// (rows drawn by a power law, for the last two lines evenly).  Below eight edges a key the
// list is ahead as well (77 against 106 us at 1.6); those calls have always taken the
// general path.  A batch of more than GS_LIST_LABELS_MAX_KEYS is refused by the device
// after both passes: half of that on average leaves room for uneven batches.
static bool list_labels_pay(int64_t ids, int64_t seeds, int64_t edges, int64_t batches) {
  constexpr int64_t kFewEdges = int64_t(1) << 17;
  return edges >= 8 * (ids + seeds) &&
         (ids <= GS_FIRST_POSITION_FEW_IDS || edges <= kFewEdges) &&
         ids + seeds <= batches * (GS_LIST_LABELS_MAX_KEYS / 2);
}

// Frontier and labels by way of the list of row ids, for a matrix whose rows are
// positions in a list with a segment per mini-batch; null where that does not pay
// (`list_labels_pay`) or where an edge's row turns out to lie in another batch's
// segment.  Waits for the size of the frontier, as every caller is about to do.
Graph::BatchListLabels* Graph::batch_list_labels_for(const torch::Tensor& col_seeds,
                                                     const torch::Tensor& row_ids,
                                                     const ColumnOrderedEdges& edges,
                                                     bool want_labels) {
  const int64_t R = row_ids.numel(), S = col_seeds.numel(), E = edges.row.numel();
  const int64_t B = col_bptr_.numel() - 1;
  if (R == 0 || S == 0 || R != num_rows_ || S != num_cols_ || !edges.col.defined() ||
      !row_bptr_.defined() || row_bptr_.numel() != B + 1 || row_encoding_size_ <= 0 ||
      !list_labels_pay(R, S, E, B))
    return nullptr;
  if (batch_list_labels_ && batch_list_labels_->base.is_same(edges.row) &&
      batch_list_labels_->row_ids.is_same(row_ids) &&
      batch_list_labels_->seeds.is_same(col_seeds) &&
      batch_list_labels_->row_ids_version == (int64_t)row_ids._version() &&
      batch_list_labels_->seeds_version == (int64_t)col_seeds._version() &&
      batch_list_labels_->epoch == cache_epoch() &&
      (batch_list_labels_->refused || !want_labels || batch_list_labels_->row.defined()))
    return batch_list_labels_->refused ? nullptr : batch_list_labels_.get();
  auto out = std::make_unique<BatchListLabels>();
  out->base = edges.row;
  out->row_ids = row_ids;
  out->seeds = col_seeds;
  out->row_ids_version = row_ids._version();
  out->seeds_version = col_seeds._version();
  out->epoch = cache_epoch();
  torch::Tensor table = ids(row_ids, "row_ids"), list_ptr = ids(row_bptr_, "row_bptr");
  torch::Tensor first = first_edges(edges.row, R);
  Frontier& f = out->frontier;
  f.num_batches = B;
  f.unique_ptr = new_ids(B + 1, edges.row);
  f.unique_buffer = new_ids(R + S, edges.row);
  out->row = new_ids(E, edges.row);
  out->col = new_ids(E, edges.row);
  torch::Tensor labels = new_ids(R + S, edges.row);
  torch::Tensor scratch = new_ids(R + S + B + 1, edges.row);
  int64_t* mirror = OffsetMirror::reserve(f.unique_ptr);
  GS_CALL(gs_batch_list_labels(cptr(col_seeds), cptr(col_bptr_), S, cptr(table), cptr(list_ptr), R,
                               row_encoding_size_, B, cptr(edges.row), cptr(edges.col),
                               cptr(edge_bptr_), E, cptr(first), mptr(f.unique_buffer),
                               mptr(f.unique_ptr), mirror, mptr(labels), mptr(labels) + R,
                               mptr(out->row), mptr(out->col), mptr(scratch), cur_stream()));
  OffsetMirror::arm(f.unique_ptr);
  out->refused = f.total() < 0;
  batch_list_labels_ = std::move(out);
  if (batch_list_labels_->refused) {
    batch_list_labels_->row = batch_list_labels_->col = torch::Tensor();
    batch_list_labels_->frontier = Frontier{};
    return nullptr;
  }
  BatchOffsets::trust(batch_list_labels_->frontier.unique_ptr);
  return batch_list_labels_.get();
}

// The subgraph that a list of nodes induces (ShaDow): its edges' rows are positions of the
// list that the seeds are, so the frontier is the unique of the seeds alone, and an edge's
// labels are those of two seeds.  Hashing the seeds and two gathers from a small table take
// the place of hashing every edge, which took, us with all_nodes() and to_dgl_block():
//   917 edges between 80 nodes of 2 batches 31, now 25        11 K between 200 34, 27
//   1.4 M between 19 K of 64 65, 42       2.3 M between 19 K of 16 88, 45
//   6.0 M between 80 K of 4 255, 98
bool Graph::rows_are_the_seeds(const torch::Tensor& col_seeds, const torch::Tensor& row_ids,
                               const torch::Tensor& edge_rows) const {
  return square_rows_.defined() && square_rows_.is_same(edge_rows) &&
         square_rows_version_ == (int64_t)edge_rows._version() &&
         square_rows_epoch_ == cache_epoch() && row_ids.is_same(col_seeds) &&
         col_seeds.numel() == num_rows_ && num_rows_ == num_cols_ && row_bptr_.is_same(col_bptr_) &&
         edge_rows.numel() >= num_rows_;
}

// Queues unique (count + fill) and relabel for the super-batch; nothing here
// waits for the device.  The frontier's size is still on its way when this
// returns: f.frontier() waits for it.
Graph::Frontier& Graph::batch_relabel_launch(torch::Tensor& col_seeds,
                                             const torch::Tensor& row_ids,
                                             torch::Tensor* out_row, torch::Tensor* out_col,
                                             c10::optional<torch::Tensor>* e_ids) {
  TORCH_CHECK(edge_bptr_.defined() && edge_bptr_.numel() > 0,
              "BatchGraphRelabel: the graph has no edge batch pointer");
  ColumnOrderedEdges edges = column_ordered_edges("BatchGraphRelabel");
  col_seeds = ids(col_seeds, "col_seeds");
  // the kernels read seeds[col_bptr[b] ...]: the seeds must be the ones the
  // batch pointer was recorded for
  BatchOffsets::check(col_bptr_, col_seeds.numel(), "BatchGraphRelabel");
  if (edges.col_indptr.defined())
    TORCH_CHECK(edges.col_indptr.numel() == col_seeds.numel() + 1,
                "BatchGraphRelabel: ", col_seeds.numel(), " seeds for a matrix of ",
                edges.col_indptr.numel() - 1, " columns");
  if (BatchListLabels* l = batch_list_labels_for(col_seeds, row_ids, edges, true)) {
    // handed out once: they are the caller's to change
    *out_row = std::move(l->row);
    *out_col = std::move(l->col);
    l->row = l->col = torch::Tensor();
    if (e_ids) *e_ids = edges.e_ids;
    return l->frontier;
  }
  if (rows_are_the_seeds(col_seeds, row_ids, edges.row)) {
    const int64_t S = col_seeds.numel(), E = edges.row.numel();
    torch::Tensor seed_label = new_ids(S, edges.row);
    LabelRequest labels{nullptr, nullptr, mptr(seed_label), nullptr};
    Frontier& f = frontier_for(col_seeds, col_seeds, col_bptr_, col_bptr_, &labels);
    if (!labels.done)
      GS_CALL(gs_unique_relabel(cptr(col_seeds), cptr(col_bptr_), S, cptr(col_seeds),
                                cptr(col_bptr_), S, f.num_batches, nullptr, nullptr,
                                mptr(seed_label), nullptr, 0, f.workspace.data_ptr(),
                                f.workspace.numel(), cur_stream()));
    *out_row = new_ids(E, edges.row);
    *out_col = new_ids(E, edges.row);
    GS_CALL(gs_list_edge_labels(cptr(edges.row), edges.col.defined() ? cptr(edges.col) : nullptr,
                                edges.col_indptr.defined() ? cptr(edges.col_indptr) : nullptr, S,
                                E, cptr(seed_label), S, cptr(seed_label), mptr(*out_row),
                                mptr(*out_col), cur_stream()));
    if (e_ids) *e_ids = edges.e_ids;
    return f;
  }
  torch::Tensor rows = batch_rows_for_relabel(edges.row, row_ids);
  const int64_t E = rows.numel();
  *out_row = new_ids(E, rows);
  // the column labels that the sampler left go out as they are wherever a batch
  // has distinct seeds (the relabel pass rewrites the other batches in place)
  const bool prefilled = edges.col_indptr.defined() && col_labels_.defined() &&
                         col_labels_.numel() == E && E > 0;
  *out_col = prefilled ? col_labels_ : new_ids(E, rows);
  LabelRequest labels{edges.col.defined() ? cptr(edges.col) : nullptr,
                      edges.col_indptr.defined() ? cptr(edges.col_indptr) : nullptr,
                      mptr(*out_row), mptr(*out_col), prefilled};
  Frontier& f = frontier_for(col_seeds, rows, col_bptr_, edge_bptr_, &labels);
  if (!labels.done)
    GS_CALL(gs_unique_relabel(cptr(col_seeds), cptr(col_bptr_), col_seeds.numel(),
                              cptr(rows), cptr(edge_bptr_), E, f.num_batches,
                              labels.edge_col, labels.col_indptr, labels.out_row,
                              labels.out_col, prefilled ? 1 : 0, f.workspace.data_ptr(),
                              f.workspace.numel(),
                              cur_stream()));
  if (e_ids) *e_ids = edges.e_ids;
  return f;
}

std::tuple<torch::Tensor, torch::Tensor, torch::Tensor, torch::Tensor,
           c10::optional<torch::Tensor>, torch::Tensor>
Graph::BatchGraphRelabel(torch::Tensor col_seeds, torch::Tensor row_ids) {
  torch::Tensor out_row, out_col;
  c10::optional<torch::Tensor> e_ids;
  Frontier& f = batch_relabel_launch(col_seeds, row_ids, &out_row, &out_col, &e_ids);
  return {frontier_of(f, "BatchGraphRelabel"), f.unique_ptr, out_row, out_col, e_ids, edge_bptr_};
}

std::tuple<torch::Tensor, torch::Tensor> Graph::BatchGetValidNodes(
    torch::Tensor col_seeds, torch::Tensor row_ids) {
  TORCH_CHECK(edge_bptr_.defined() && edge_bptr_.numel() > 0,
              "BatchGetValidNodes: the graph has no edge batch pointer");
  ColumnOrderedEdges edges = column_ordered_edges("BatchGetValidNodes");
  col_seeds = ids(col_seeds, "col_seeds");
  BatchOffsets::check(col_bptr_, col_seeds.numel(), "BatchGetValidNodes");
  if (BatchListLabels* l = batch_list_labels_for(col_seeds, row_ids, edges, false))
    return {l->frontier.frontier(), l->frontier.unique_ptr};
  if (rows_are_the_seeds(col_seeds, row_ids, edges.row)) {
    Frontier& f = frontier_for(col_seeds, col_seeds, col_bptr_, col_bptr_);
    return {f.frontier(), f.unique_ptr};
  }
  torch::Tensor rows = batch_rows_for_relabel(edges.row, row_ids);
  Frontier& f = frontier_for(col_seeds, rows, col_bptr_, edge_bptr_);
  return {frontier_of(f, "BatchGetValidNodes"), f.unique_ptr};
}

// ------------------------------------------------------------ free operators
std::vector<torch::Tensor> SplitByOffset(torch::Tensor data,
                                         torch::Tensor offset) {
  const std::vector<int64_t>& p = host_offsets(offset);
  std::vector<int64_t> sizes;
  for (size_t i = 0; i + 1 < p.size(); ++i) sizes.push_back(p[i + 1] - p[i]);
  return torch::split_with_sizes(data, sizes);
}

// Per-batch indptr arrays rebased to start at 0; batch i covers columns
// [offset[i], offset[i+1]] of the shared indptr
// (src/cuda/batch/batch_split.cu:53-94).
std::vector<torch::Tensor> SplitIndptrByOffset(torch::Tensor indptr,
                                               torch::Tensor offset) {
  indptr = ids(indptr, "indptr");
  offset = ids(offset, "offset");
  const int64_t B = offset.numel() - 1;
  const std::vector<int64_t>& p = host_offsets(offset);
  std::vector<int64_t> sizes;
  int64_t total = 0;
  for (int64_t i = 0; i < B; ++i) {
    sizes.push_back(p[i + 1] - p[i] + 1);
    total += sizes.back();
  }
  torch::Tensor out = new_ids(total, indptr);
  GS_CALL(gs_split_indptr(cptr(indptr), cptr(offset), B, total, mptr(out),
                          cur_stream()));
  return torch::split_with_sizes(out, sizes);
}

}  // namespace gs

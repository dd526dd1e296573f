// graph.h -- the `gs_classes.Graph` operator object: one sparse matrix held in
// up to three formats, plus the super-batch bookkeeping.  Method names,
// argument order and return shapes follow the reference's class
// (src/graph.h:11-232 of gSampler) because its Python layer and JIT address
// them by name and position; the bodies call the C ABI of gsampler_hip.h.
#ifndef GS_HOST_GRAPH_H_
#define GS_HOST_GRAPH_H_

#include <torch/custom_class.h>
#include <torch/script.h>

#include <c10/hip/HIPCachingAllocator.h>

#include "abi_call.h"

#include <atomic>
#include <functional>
#include <memory>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

namespace gs {

// Format bit flags (src/graph_storage.h:31-33).
constexpr int64_t kCOO = 1, kCSC = 2, kCSR = 4;

// A table that operators derive from a matrix on first use and keep with it.  The
// kernel that fills it is queued on the stream of whoever asked first, and its memory
// belongs to that stream: a caller on another one waits for it once, on the host, and
// announces to the allocator that it reads there.  (An event behind the kernel would
// spare that wait and cost every first use a gap on the device.)
class DerivedTable {
 public:
  bool defined() const { return table_.defined(); }
  void drop() { table_ = torch::Tensor(); }
  void set(torch::Tensor t) {
    table_ = std::move(t);
    made_on_ = cur_stream();
    complete_ = false;
  }
  torch::Tensor on_current_stream() {
    if (!table_.defined() || made_on_ == cur_stream()) return table_;
    if (!complete_) {
      const hipError_t e = hipDeviceSynchronize();
      TORCH_CHECK(e == hipSuccess, "HIP error: ", hipGetErrorString(e));
      complete_ = true;
    }
    c10::hip::HIPCachingAllocator::recordStream(table_.storage().data_ptr(),
                                                c10::hip::getCurrentHIPStream());
    return table_;
  }

 private:
  torch::Tensor table_;
  gs_stream_t made_on_ = nullptr;
  bool complete_ = false;
};

// CSC or CSR: `indptr` over the compressed ("major") axis, `indices` holds the
// ids on the other ("minor") axis.
struct Compressed {
  torch::Tensor indptr, indices;
  c10::optional<torch::Tensor> e_ids;
  // Exclusive bound of the ids in `indices` when it is known (a loaded or
  // converted matrix), else -1.
  int64_t num_minor = -1;
  // The tables below belong to the ids they were made from: their version, the cache
  // epoch (invalidate_caches) and their address.  None is made or handed out while
  // the current stream is being captured: the graph would record the kernel that fills
  // the table, or read one that a later edit of the matrix frees.
  //
  // int32 copy of `indices` (half the bytes behind every random pick), of a matrix in
  // device memory whose ids fit.  A sampler makes it on its first call; an operator that
  // gains less tells how many ids it is about to read, and makes the copy once the reads
  // so told come to as many as the matrix has edges.
  torch::Tensor narrow_indices(int64_t reads = -1) const;
  // There are ids on the other axis, known to be below 2^31.
  bool minor_ids_fit_32() const {
    return indices.numel() > 0 && num_minor >= 0 && num_minor < (int64_t(1) << 31);
  }
  // Where the column behind every edge lies (gs_hop_table), for walks over a
  // square matrix; made at the second walk over the same matrix.
  torch::Tensor hop_table() const;
  // Marks of every column (gs_column_marks), for second-order walks over a square matrix
  // with sorted columns; made once calls that go by them have walked enough steps.
  torch::Tensor column_marks(int64_t steps) const;
  struct Derived {
    std::mutex guard;  // a matrix is shared by every handle and sampler thread
    DerivedTable narrow, hops, marks;
    int64_t versions[2] = {-1, -1}, epoch = -1;
    const void* source = nullptr;
    int64_t walks = 0, reads = 0, steps = 0;
    void drop() {
      narrow.drop();
      hops.drop();
      marks.drop();
      walks = reads = steps = 0;
    }
  };
  Compressed() = default;
  Compressed(torch::Tensor indptr, torch::Tensor indices)
      : indptr(std::move(indptr)), indices(std::move(indices)) {}
  Compressed(const Compressed& o)  // derived tables stay with the matrix they were made for
      : indptr(o.indptr), indices(o.indices), e_ids(o.e_ids), num_minor(o.num_minor) {}
  // Call after assigning another `indices` or `indptr` to a matrix that was used.
  void forget_derived() {
    std::lock_guard<std::mutex> lock(derived_.guard);
    derived_.drop();
  }

 private:
  mutable Derived derived_;
  Derived& current_derived() const;  // called under the lock: aged tables dropped
};

struct Coordinate {
  torch::Tensor row, col;
  c10::optional<torch::Tensor> e_ids;
  bool row_sorted = false, col_sorted = false;
};

// Output of an operator that works along the compressed axis.
struct MajorResult {
  torch::Tensor indptr;     // [items + 1]
  torch::Tensor major_ids;  // local id on the compressed axis per edge (COO), may be undefined
  torch::Tensor minor_ids;  // id on the other axis per edge
  torch::Tensor select;     // position of the edge in the parent's `indices`
};

// Process-wide sampler state: every sampling call consumes one call id, so
// successive layers / epochs draw from disjoint Philox streams while a fixed
// seed reproduces a whole run.
struct RandomState {
  uint64_t seed = 7777;  // the reference's literal, src/cuda/sampling.cu:143
  std::atomic<uint64_t> next_call{0};
  int64_t algo = 0;      // GS_ALGO_AUTO
};
RandomState& random_state();
// Takes call ids, the first of which it returns.  Threads share the counter: what one
// has taken is never put back.
uint64_t next_call_id(uint64_t how_many = 1);

// Views of one mini-batch block: (row, col, indptr by destination -- absent for
// a mini-batch whose seeds repeat --, source ids, edge ids if the matrix carries
// any, number of source nodes, number of destination nodes).
using BlockViews = std::tuple<torch::Tensor, torch::Tensor, c10::optional<torch::Tensor>,
                              torch::Tensor, c10::optional<torch::Tensor>, int64_t, int64_t>;

// The same for every block of a layer, one list per field.
using BlockParts =
    std::tuple<std::vector<torch::Tensor>, std::vector<torch::Tensor>,
               std::vector<c10::optional<torch::Tensor>>, std::vector<torch::Tensor>,
               std::vector<c10::optional<torch::Tensor>>, std::vector<int64_t>,
               std::vector<int64_t>>;

// All blocks of one layer of a super-batched sampler (see blocks.cc).  The
// tensors are the layer's concatenated arrays; a block is a set of views.  The
// per-batch offsets reach the host on first use (they are already on their way
// when the object is handed out).
class BlockBatch : public torch::CustomClassHolder {
 public:
  torch::Tensor frontier, frontier_ptr, row, col, coo_ptr, col_bptr, col_seeds;
  torch::Tensor sampled_indptr;    // offsets of the sampled matrix over all its columns
  torch::Tensor indptr, distinct;  // per-block offsets and per-batch flags, made on first use
  c10::optional<torch::Tensor> e_ids;
  int64_t num_batches = 0, num_dst_total = 0;

  int64_t Size() { return num_batches; }
  // (source nodes, destination nodes, edges) over all blocks; no device read
  std::vector<int64_t> Totals();
  // host copies of (frontier_ptr, col_bptr, coo_ptr)
  std::tuple<std::vector<int64_t>, std::vector<int64_t>, std::vector<int64_t>> Offsets();
  BlockViews Block(int64_t b);
  BlockParts Blocks();
  int64_t NumSrcOf(int64_t b);
  bool grouped(int64_t b) const { return grouped_[(size_t)b] != 0; }  // after Offsets()
  torch::Tensor Frontier() { return frontier; }
  torch::Tensor FrontierPtr() { return frontier_ptr; }
  torch::Tensor Row() { return row; }
  torch::Tensor Col() { return col; }
  torch::Tensor Indptr() {
    fetch();
    return indptr;
  }
  torch::Tensor EdgePtr() { return coo_ptr; }
  torch::Tensor ColPtr() { return col_bptr; }
  c10::optional<torch::Tensor> EdgeIds() { return e_ids; }
  // For a producer that has the offsets on the host already: of the frontier, the
  // edges and the columns, and per batch whether its seeds are distinct.
  void set_host_offsets(std::vector<int64_t> f, std::vector<int64_t> e, std::vector<int64_t> c,
                        std::vector<uint8_t> grouped);

 private:
  void fetch();
  bool have_host_ = false;
  std::vector<int64_t> f_off_, e_off_, c_off_;
  std::vector<uint8_t> grouped_;  // per batch: edges grouped by destination in offset order
};

class Graph;
using GraphPtr = c10::intrusive_ptr<Graph>;
using GraphAndIndex = std::tuple<GraphPtr, torch::Tensor>;

class Graph : public torch::CustomClassHolder {
 public:
  Graph(int64_t num_rows, int64_t num_cols)
      : num_rows_(num_rows), num_cols_(num_cols) {}

  // ---- loading and inspection
  void LoadCSC(torch::Tensor indptr, torch::Tensor indices);
  void LoadCOO(torch::Tensor row, torch::Tensor col, bool row_sorted,
               bool col_sorted);
  void LoadCSR(torch::Tensor indptr, torch::Tensor indices);
  int64_t GetNumRows() { return num_rows_; }
  int64_t GetNumCols() { return num_cols_; }
  int64_t GetNumEdges() { return num_edges_; }
  torch::Tensor GetCSCIndptr();
  torch::Tensor GetCSCIndices();
  torch::Tensor GetCSCEids();
  torch::Tensor GetCOORows();
  torch::Tensor GetCOOCols();
  torch::Tensor GetCOOEids();
  torch::Tensor GetCSRIndptr();
  torch::Tensor GetCSRIndices();
  torch::Tensor GetCSREids();
  void CreateSparseFormat(int64_t format);

  // ---- extract / select operators
  GraphAndIndex Slicing(torch::Tensor seeds, int64_t axis, int64_t on_format,
                        int64_t output_format);
  GraphAndIndex Sampling(int64_t axis, int64_t fanout, bool replace,
                         int64_t on_format, int64_t output_format);
  GraphAndIndex SamplingProbs(int64_t axis, torch::Tensor edge_probs,
                              int64_t fanout, bool replace, int64_t on_format,
                              int64_t output_format);
  // Not in the reference: column slice + weighted sampling in one step, on the
  // weights of this (unsliced) matrix.  What gs.jit.compile turns
  // Slicing -> SamplingProbs into; draws go through a persistent CDF of the
  // weights that is built on first use and kept while the same tensor comes in.
  GraphAndIndex FusedSlicingSamplingProbs(int64_t axis, torch::Tensor seeds,
                                          torch::Tensor edge_probs, int64_t fanout,
                                          bool replace, int64_t on_format,
                                          int64_t output_format);
  GraphAndIndex FusedSlicingSampling(int64_t axis, torch::Tensor seeds,
                                     int64_t fanout, bool replace,
                                     int64_t on_format, int64_t output_format);
  // Not in the reference: operators that read the column slice A[:, cols]
  // straight from this matrix instead of from a written slice (fused_slices.cc).
  // out[row] += sum of efeat^2 over the edges of A[:, cols];
  void SlicedESquareSum(torch::Tensor cols, torch::Tensor efeat, torch::Tensor out);
  // The sums alone; nothing where the call is not one for it (see EdgeScore).
  c10::optional<torch::Tensor> SlicedSquareSums(torch::Tensor cols, torch::Tensor efeat);
  // A[rows, cols], the edge index addressing this matrix's edges.
  GraphAndIndex ColRowSlicing(torch::Tensor cols, torch::Tensor rows, int64_t on_format,
                              int64_t output_format);
  GraphAndIndex Compact(int64_t axis);
  torch::Tensor RandomWalk(torch::Tensor seeds, int64_t walk_length);
  torch::Tensor Node2Vec(torch::Tensor seeds, int64_t walk_length, double p,
                         double q);
  void SortCSCIndices();

  // ---- compute operators
  void SDDMM(const std::string& op, torch::Tensor lhs, torch::Tensor rhs,
             torch::Tensor out, int64_t lhs_target, int64_t rhs_target,
             int64_t on_format);
  void SpMM(const std::string& op, const std::string& reduce,
            torch::Tensor ufeat, torch::Tensor efeat, torch::Tensor out,
            torch::Tensor argu, torch::Tensor arge, int64_t u_target,
            int64_t on_format);
  // gs_edge_score over the terms (kinds[k], lhs[k], rhs[k], targets[2 k .. 2 k + 1]);
  // nothing where the call is not one for it: other types, shapes or devices, values
  // that carry gradients, a transform or a mode that has to see torch's operators.
  c10::optional<torch::Tensor> EdgeScore(const std::vector<int64_t>& kinds,
                                         std::vector<torch::Tensor> lhs,
                                         std::vector<torch::Tensor> rhs,
                                         const std::vector<int64_t>& targets,
                                         c10::optional<torch::Tensor> weights,
                                         bool positive_part, double shift, int64_t on_format);
  // gs_normalise_columns; nothing where the call is not one for it (see EdgeScore).
  c10::optional<torch::Tensor> NormaliseColumns(torch::Tensor values,
                                                c10::optional<torch::Tensor> select,
                                                c10::optional<torch::Tensor> row_divisor);
  // For a compiled sampler: the row slice A[rows, cols] as GraphRelabel(cols, rows) of it
  // and, with `values` of this matrix's edges, NormaliseColumns leave it, (frontier, row,
  // column, values), the slice itself not written; nothing where the call is not one for it.
  c10::optional<std::tuple<torch::Tensor, torch::Tensor, torch::Tensor,
                           c10::optional<torch::Tensor>>>
  RelabelledRows(torch::Tensor cols, torch::Tensor rows, c10::optional<torch::Tensor> values,
                 c10::optional<torch::Tensor> row_divisor);
  // The same of a super-batch, as EncodedPickedRows (with `seeds` and the names of the picked
  // rows) and BatchBlocks leave it, and of the subgraphs that lists of nodes induce, as
  // BatchColRowSlcing of a list by itself does.
  c10::optional<std::tuple<c10::intrusive_ptr<BlockBatch>, c10::optional<torch::Tensor>>>
  EncodedBlocks(torch::Tensor seeds, torch::Tensor col_bptr, torch::Tensor rows,
                torch::Tensor row_ids, torch::Tensor row_bptr,
                c10::optional<torch::Tensor> values, c10::optional<torch::Tensor> row_divisor);
  // Queues what an operator that slices these columns would wait for first.
  void PrepareSlice(torch::Tensor cols);
  c10::optional<c10::intrusive_ptr<BlockBatch>> SubgraphBlocks(torch::Tensor nodes,
                                                               torch::Tensor nodes_ptr);
  void FusedUOPV(const std::string& op, torch::Tensor lhs1, torch::Tensor rhs1,
                 torch::Tensor out1, torch::Tensor lhs2, torch::Tensor rhs2,
                 torch::Tensor out2, int64_t on_format);
  void FusedESquareSum(const std::string& op, const std::string& reduce,
                       torch::Tensor ufeat, torch::Tensor efeat,
                       torch::Tensor out, torch::Tensor argu,
                       torch::Tensor arge, int64_t u_target, int64_t on_format);
  void FusedEDivUSum(const std::string& op, const std::string& reduce,
                     torch::Tensor ufeat, torch::Tensor efeat,
                     torch::Tensor out, torch::Tensor argu, torch::Tensor arge,
                     int64_t u_target, int64_t on_format);

  // ---- finalize operators
  std::tuple<torch::Tensor, torch::Tensor, torch::Tensor,
             c10::optional<torch::Tensor>>
  GraphRelabel(torch::Tensor col_seeds, torch::Tensor row_ids);
  torch::Tensor GetValidNodes(torch::Tensor col_seeds, torch::Tensor row_ids);

  // ---- super-batch interface
  void SetEdgeBptr(torch::Tensor p) { edge_bptr_ = p; }
  void SetColBptr(torch::Tensor p) { col_bptr_ = p; }
  void SetRowBptr(torch::Tensor p) { row_bptr_ = p; }
  void SetOrigRowIds(torch::Tensor t) { orig_row_ids_ = t; }
  void SetOrigColIds(torch::Tensor t) { orig_col_ids_ = t; }
  torch::Tensor GetEdgeBptr() { return edge_bptr_; }
  torch::Tensor GetColBptr() { return col_bptr_; }
  torch::Tensor GetRowBptr() { return row_bptr_; }
  std::tuple<torch::Tensor, torch::Tensor> BatchGetRows() {
    return {orig_row_ids_, row_bptr_};
  }
  std::tuple<torch::Tensor, torch::Tensor> BatchGetCols() {
    return {orig_col_ids_, col_bptr_};
  }
  std::tuple<torch::Tensor, torch::Tensor> BatchGetCSCIndptr();
  std::tuple<torch::Tensor, torch::Tensor> BatchGetCSCIndices();
  std::tuple<torch::Tensor, torch::Tensor> BatchGetCSCEids();
  std::tuple<torch::Tensor, torch::Tensor> BatchGetCOORows();
  std::tuple<torch::Tensor, torch::Tensor> BatchGetCOOCols();
  std::tuple<torch::Tensor, torch::Tensor> BatchGetCOOEids();
  std::vector<int64_t> BatchGetColCounts();
  GraphAndIndex BatchColSlicing(torch::Tensor seeds, torch::Tensor col_bptr,
                                bool encoding);
  c10::optional<std::tuple<torch::Tensor, torch::Tensor, torch::Tensor>> EncodedSquareSums(
      torch::Tensor seeds, torch::Tensor col_bptr, torch::Tensor efeat);
  // BatchRowSlicing of that slice by row_ids, positions in its `rows`; and rows[row_ids].
  std::tuple<GraphPtr, torch::Tensor, torch::Tensor> EncodedPickedRows(
      torch::Tensor seeds, torch::Tensor col_bptr, torch::Tensor rows, torch::Tensor row_ids,
      torch::Tensor row_bptr);
  GraphAndIndex BatchColRowSlcing(torch::Tensor col, torch::Tensor col_bptr,
                                  torch::Tensor row, torch::Tensor row_bptr);
  GraphAndIndex BatchRowSlicing(torch::Tensor row_ids, torch::Tensor row_bptr);
  GraphAndIndex BatchRowSampling(int64_t fanout, bool replace);
  GraphAndIndex BatchRowSamplingProbs(int64_t fanout, bool replace,
                                      torch::Tensor edge_probs);
  GraphAndIndex BatchFusedSlicingSamplingProbs(torch::Tensor seeds,
                                               torch::Tensor col_bptr,
                                               torch::Tensor edge_probs,
                                               int64_t fanout, bool replace);
  GraphAndIndex BatchFusedSlicingSampling(torch::Tensor seeds,
                                          torch::Tensor col_bptr,
                                          int64_t fanout, bool replace);
  std::tuple<torch::Tensor, torch::Tensor, torch::Tensor, torch::Tensor,
             c10::optional<torch::Tensor>, torch::Tensor>
  BatchGraphRelabel(torch::Tensor col_seeds, torch::Tensor row_ids);
  std::tuple<torch::Tensor, torch::Tensor> BatchGetValidNodes(
      torch::Tensor col_seeds, torch::Tensor row_ids);
  // Not in the reference: relabel + all mini-batch blocks of the layer (edge
  // list and compressed form) in one call; see blocks.cc.
  c10::intrusive_ptr<BlockBatch> BatchBlocks(torch::Tensor col_seeds, torch::Tensor row_ids);
  // Not in the reference: all layers of a node-wise sampler in one call
  // (layers.cc) -- what gs.jit.compile runs for a chain of slice + sample +
  // relabel.  Per layer: frontier, row and column labels, edge ids (none) ...
  std::vector<c10::optional<torch::Tensor>> SampleLayers(
      torch::Tensor seeds, std::vector<int64_t> fanouts, bool replace,
      c10::optional<torch::Tensor> edge_probs);
  // ... or, for a super-batch, the layer's blocks.
  std::vector<c10::intrusive_ptr<BlockBatch>> BatchSampleLayers(
      torch::Tensor seeds, torch::Tensor col_bptr, std::vector<int64_t> fanouts, bool replace,
      c10::optional<torch::Tensor> edge_probs);
  // ... or their nodes alone: frontier and where every mini-batch's begins, per layer.
  std::vector<torch::Tensor> BatchSampleNodes(torch::Tensor seeds, torch::Tensor col_bptr,
                                              std::vector<int64_t> fanouts, bool replace,
                                              c10::optional<torch::Tensor> edge_probs);
  // The blocks again; `done` takes the finished layers one by one where the host would
  // otherwise only wait for the next one.  Returns the layers it was not called for.
  using LayerDone = std::function<void(c10::intrusive_ptr<BlockBatch>)>;
  std::vector<c10::intrusive_ptr<BlockBatch>> BatchSampleLayersWhile(
      torch::Tensor seeds, torch::Tensor col_bptr, std::vector<int64_t> fanouts, bool replace,
      c10::optional<torch::Tensor> edge_probs, const LayerDone& done);

 private:
  struct Layer;
  // `idle(layers)` runs while the device works on layer layers.size()
  using LayersIdle = std::function<void(std::vector<Layer>& layers, size_t complete)>;
  std::vector<Layer> sample_layers(const torch::Tensor& seeds, const torch::Tensor& col_bptr,
                                   const std::vector<int64_t>& fanouts, bool replace,
                                   const c10::optional<torch::Tensor>& edge_probs, bool blocks,
                                   const LayersIdle& idle, bool labels = true);
  Layer large_layer(const torch::Tensor& cols, const torch::Tensor& col_bptr, int64_t fanout,
                    bool replace, const torch::Tensor& cdf, uint64_t call_id, bool labels,
                    const std::function<void()>& idle);
  // Workspace of the small layers, kept between calls (one per matrix, at most
  // 2^19 positions, 22 MiB, 18 of weighted layers): its tables, two or one, are empty
  // whenever a call has been queued, so the next call on the same stream starts without clearing it.  A call
  // takes it out and puts it back; one that finds none (another thread has it, or it
  // belongs to another stream) makes its own.
  struct LayerWorkspace {
    torch::Tensor ws;
    int64_t positions = 0;
    bool weighted = false;
    gs_stream_t stream = nullptr;
  };
  LayerWorkspace layer_ws_;
  std::mutex layer_ws_guard_;

  // Unique/relabel state shared by all_nodes() and to_dgl_block(): the
  // frontier is computed once, the relabel pass reuses the hash tables.
  struct Frontier {
    torch::Tensor seeds, rows, seeds_ptr, rows_ptr;  // the keys it was built from
    int64_t seeds_version = -1, rows_version = -1, epoch = -1;
    torch::Tensor workspace, unique_ptr;
    int64_t num_batches = 0;
    // The unique keys: filled into a buffer sized by the upper bound, trimmed
    // once the count has arrived (frontier() waits for it).
    torch::Tensor unique_buffer;
    int64_t total() { return OffsetMirror::values(unique_ptr).back(); }
    const torch::Tensor& frontier() {
      if (!unique_.defined()) unique_ = unique_buffer.narrow(0, 0, total());
      return unique_;
    }
    bool matches(const torch::Tensor& s, const torch::Tensor& r,
                 const torch::Tensor& sp, const torch::Tensor& rp) const;

   private:
    torch::Tensor unique_;
  };
  // Labels wanted together with a frontier: when the frontier has to be built,
  // both come from one launch and `done` is set; a frontier that is already there
  // leaves `done` false and the caller labels on its own.
  struct LabelRequest {
    const int64_t* edge_col = nullptr;
    const int64_t* col_indptr = nullptr;
    int64_t* out_row = nullptr;
    int64_t* out_col = nullptr;
    bool col_prefilled = false;  // out_col holds the samplers' column labels
    bool done = false;
  };
  Frontier& frontier_for(const torch::Tensor& seeds, const torch::Tensor& rows,
                         const torch::Tensor& seeds_ptr,
                         const torch::Tensor& rows_ptr, LabelRequest* labels = nullptr);
  const torch::Tensor& frontier_of(Frontier& f, const char* who);
  Frontier& batch_relabel_launch(torch::Tensor& col_seeds, const torch::Tensor& row_ids,
                                 torch::Tensor* out_row, torch::Tensor* out_col,
                                 c10::optional<torch::Tensor>* e_ids);

  const Compressed& compressed(int64_t format);
  // Offsets and size of the column slice A[:, cols], kept for the next operator
  // that is handed the same tensor of columns.  (Sampler threads share the matrix: what
  // one holds stays when another puts its own in its place.)
  struct SliceOffsets {
    torch::Tensor cols, sub_indptr;
    int64_t version = -1, indptr_version = -1, epoch = -1;
    int64_t nnz = -1;        // (waited for under the guard)
    torch::Tensor total;     // where it is on its way to the host from
    void* stream = nullptr;  // whose kernels write the tensors
    std::mutex guard;
    MajorResult written;  // the slice itself, when an operator had to write it
    // of a super-batch cut by key_bptr: what every column's row ids are moved by
    torch::Tensor key_offset, key_bptr;
    int64_t key_bptr_version = -1;
    torch::Tensor kept_key_offset(const torch::Tensor& bptr);
    void keep_key_offset(const torch::Tensor& bptr, const torch::Tensor& offset);
  };
  std::mutex slice_offsets_guard_;
  std::shared_ptr<SliceOffsets> slice_offsets_;
  std::shared_ptr<SliceOffsets> slice_offsets_for(const torch::Tensor& cols, bool wait = true);
  static bool read_in_place(const Compressed& m, int64_t slice_nnz, int64_t num_cols_picked);
  const MajorResult& written_slice(SliceOffsets& so);
  torch::Tensor key_offsets_for(SliceOffsets& so, const torch::Tensor& col_bptr);
  GraphAndIndex encoded_row_slice(const torch::Tensor& seeds, const torch::Tensor& col_bptr,
                                  const torch::Tensor& picked, const torch::Tensor& row_ids,
                                  const torch::Tensor& row_bptr);
  // CDF of edge_probs in the edge order of `format` (cached per weights tensor).
  torch::Tensor weight_cdf_for(const torch::Tensor& edge_probs, int64_t format);
  void check_reduce_operands(const std::string& op, const torch::Tensor& ufeat,
                             const torch::Tensor& efeat, const torch::Tensor& out,
                             int64_t u_target, const char* who) const;
  bool csc_sorted_ = false;  // row ids known to be sorted inside every column
  std::mutex cdf_guard_;
  DerivedTable cdf_;
  torch::Tensor cdf_probs_;
  int64_t cdf_version_ = -1, cdf_format_ = 0, cdf_epoch_ = -1;
  torch::Tensor mapped_rows(const torch::Tensor& base, const torch::Tensor& row_ids);
  GraphAndIndex slice_coo(const torch::Tensor& seeds, int64_t axis,
                          int64_t new_rows, int64_t new_cols);
  GraphPtr derive(int64_t on_format, int64_t output_format,
                  const MajorResult& r, int64_t new_rows, int64_t new_cols);
  torch::Tensor edge_index(const c10::optional<torch::Tensor>& parent_eids,
                           const torch::Tensor& select);
  void copy_batch_state_to(Graph& g, bool with_rows);
  // The edges in column order, for the relabel pass: their row ids and either
  // the column of every edge or the column pointer that implies it.
  struct ColumnOrderedEdges {
    torch::Tensor row;
    torch::Tensor col;         // undefined when col_indptr is given
    torch::Tensor col_indptr;  // undefined when col is given
    c10::optional<torch::Tensor> e_ids;
  };
  ColumnOrderedEdges column_ordered_edges(const char* who);
  torch::Tensor batch_rows_for_relabel(const torch::Tensor& edge_rows,
                                       const torch::Tensor& row_ids);

  int64_t num_rows_ = 0, num_cols_ = 0, num_edges_ = 0;
  std::shared_ptr<Compressed> csc_, csr_;
  std::shared_ptr<Coordinate> coo_;
  torch::Tensor col_bptr_, row_bptr_, edge_bptr_;
  // per edge, the place of its column inside its batch, as the super-batched
  // samplers write it (see EdgeCount::Hint); undefined for any other matrix
  torch::Tensor col_labels_;
  torch::Tensor orig_row_ids_, orig_col_ids_;
  int64_t row_encoding_size_ = 0;
  std::unique_ptr<Frontier> frontier_;
  torch::Tensor mapped_out_, mapped_from_, mapped_by_;
  c10::optional<HostFlag> mapped_refused_;  // while nobody has waited for what mapped them
  // Relabel of a matrix whose rows are positions in a short list of ids
  // (row slicing leaves it that way): label of every list entry and of every
  // seed, computed from the list instead of from every edge.
  struct ListLabels {
    torch::Tensor base, row_ids, seeds;
    int64_t row_ids_version = -1, seeds_version = -1, epoch = -1;
    torch::Tensor label_by_local, seed_label;
    // The unique keys sit at the front of a buffer sized by the bound; how many
    // there are may still be on its way from the device.
    torch::Tensor frontier_bound;
    AsyncCount frontier_count;
    bool counted = false;
    const torch::Tensor& frontier() {
      if (!counted) {
        if (frontier_count.requested())
          frontier_bound = frontier_bound.narrow(0, 0, frontier_count.get());
        counted = true;
      }
      return frontier_bound;
    }
  };
  std::unique_ptr<ListLabels> list_labels_;
  // Which edge of a row slice is the first of each of its rows, as the pass that made the
  // slice has met them; nothing once the rows of the edges have been written to.
  torch::Tensor row_firsts_, row_firsts_of_;
  // A value a column that is zero, for the first sum over columns that asks for one on the
  // stream whose slice cleared them: another stream's kernels would still add to memory
  // that goes back to this one, and a graph that is being recorded would not clear them.
  torch::Tensor column_zeros_;
  gs_stream_t column_zeros_stream_ = nullptr;
  std::mutex column_zeros_guard_;
  void keep_column_zeros(const torch::Tensor& zeros);
  torch::Tensor take_column_zeros();
  int64_t row_firsts_version_ = -1, row_firsts_epoch_ = -1;
  // The rows of the edges of A[list, list], while each is still a position of the list in the
  // segment of its edge's mini-batch: what the slice wrote.
  torch::Tensor square_rows_;
  int64_t square_rows_version_ = -1, square_rows_epoch_ = -1;
  bool rows_are_the_seeds(const torch::Tensor& col_seeds, const torch::Tensor& row_ids,
                          const torch::Tensor& edge_rows) const;
  void keep_row_firsts(const torch::Tensor& firsts, const torch::Tensor& edge_rows);
  torch::Tensor first_edges(const torch::Tensor& edge_rows, int64_t num_ids);
  // The same for a super-batch: the frontier and the labels of every edge.
  struct BatchListLabels {
    torch::Tensor base, row_ids, seeds;
    int64_t row_ids_version = -1, seeds_version = -1, epoch = -1;
    torch::Tensor row, col;  // until a caller takes them
    Frontier frontier;
    bool refused = false;  // the general path serves this matrix
  };
  std::unique_ptr<BatchListLabels> batch_list_labels_;
  BatchListLabels* batch_list_labels_for(const torch::Tensor& col_seeds,
                                         const torch::Tensor& row_ids,
                                         const ColumnOrderedEdges& edges, bool want_labels);
  bool use_list_labels(const torch::Tensor& col_seeds, const torch::Tensor& row_ids) const;
  ListLabels& list_labels_for(const torch::Tensor& col_seeds, const torch::Tensor& row_ids);
};

// Offsets of the slice along the compressed axis by `picked`, and its size.
torch::Tensor slice_offsets(const Compressed& m, const torch::Tensor& picked, int64_t* nnz);
// The same without waiting for the number of edges: it stays with the last of the offsets.
torch::Tensor slice_offsets_ahead(const Compressed& m, const torch::Tensor& picked,
                                  torch::Tensor* total);
// Operators along the compressed axis (graph.cc) and across it (slicing.cc).
MajorResult major_slice(const Compressed& m, const torch::Tensor& picked,
                        bool with_coo, const torch::Tensor& batch_ptr,
                        int64_t encode_stride);
// (call_id: one that the caller has taken already)
MajorResult major_sample_uniform(const Compressed& m, const torch::Tensor& picked,
                                 int64_t fanout, bool replace, bool with_coo,
                                 c10::optional<uint64_t> call_id = c10::nullopt);
MajorResult major_sample_weighted(const Compressed& m, const torch::Tensor& cdf,
                                  const torch::Tensor& picked, int64_t fanout, bool replace,
                                  bool with_coo, c10::optional<uint64_t> call_id = c10::nullopt);
void check_weighted_fanout(int64_t fanout, bool replace, const char* who);
MajorResult minor_slice(const Compressed& m, const torch::Tensor& picked,
                        bool with_coo);
// A float32 tensor on the current device that nothing but its values matters of.
bool plain_values(const torch::Tensor& t, bool gradients_matter);
// First n entries of a buffer sized by an upper bound: a view, or a copy when
// the view would pin a large buffer for a small result.
torch::Tensor trim_to(const torch::Tensor& buffer, int64_t n);

// ---- free operators (gs_ops)
torch::Tensor GatherRows(torch::Tensor table, torch::Tensor ids);
torch::Tensor ListSampling(int64_t num_items, int64_t num_picks, bool replace);
torch::Tensor ListSamplingProbs(torch::Tensor probs, int64_t num_picks,
                                bool replace);
// Either of these for a compiled sampler, with the picks' weights: (index, offsets, weights);
// nothing where the call is not one for it (see Graph::EdgeScore).
c10::optional<std::tuple<torch::Tensor, torch::Tensor, torch::Tensor>> ListSamplingPicked(
    torch::Tensor probs, int64_t num_picks, bool replace, c10::optional<torch::Tensor> range);
std::tuple<torch::Tensor, torch::Tensor> BatchListSamplingProbs(
    torch::Tensor probs, int64_t num_picks, bool replace, torch::Tensor range);
std::tuple<torch::Tensor, torch::Tensor> BatchListSampling(
    int64_t num_picks, bool replace, torch::Tensor range);
std::vector<torch::Tensor> SplitByOffset(torch::Tensor data,
                                         torch::Tensor offset);
std::vector<torch::Tensor> SplitIndptrByOffset(torch::Tensor indptr,
                                               torch::Tensor offset);

}  // namespace gs

#endif  // GS_HOST_GRAPH_H_

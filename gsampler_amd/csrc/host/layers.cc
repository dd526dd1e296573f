// layers.cc -- all layers of a node-wise sampler (slice columns, sample, unique,
// relabel; the frontier is the next layer's columns) in one operator call, for a
// single mini-batch and for a super-batch.
//
// Small layers are three launches each (layers.hip), read the number of their
// columns from the device and are queued one behind the other: the host waits
// once, at the end, for all offsets.  A layer whose bound has grown too large for
// that waits for the one before it first; large layers run on the count / fill /
// unique kernels, with the edges' positions in the matrix left out (nobody asked
// for them), the columns' labels left by the sampler, and the row ids, which end with
// the layer, 32 bits wide where the matrix's are.
#include "abi_call.h"
#include "graph.h"

namespace gs {

struct Graph::Layer {
  torch::Tensor frontier, frontier_ptr, row, col, edge_ptr;
  torch::Tensor block_indptr;    // offsets per block, or
  torch::Tensor sampled_indptr;  // the offsets over all columns they come from
  torch::Tensor cols, col_bptr;
  std::vector<int64_t> f_off, e_off;
  std::vector<uint8_t> distinct;
};

namespace {

// Positions (fanout + 1 per column) up to which a layer takes the three launches:
// beyond, hashing into one table in global memory is slower than partitioning the
// keys first.  And up to which it may be queued on a bound alone, without the host
// knowing the number of its columns: outputs are sized by the bound.
constexpr int64_t kSmallPositions = int64_t(1) << 19;
constexpr int64_t kQueuedPositions = int64_t(1) << 19;

// A small layer on its way: outputs in one buffer, cut up when the sizes are in.
struct Queued {
  torch::Tensor buffer;
  int64_t bound = 0, fanout = 0;
  int64_t at_ptr = 0, at_edge_ptr = 0, at_indptr = 0, at_row = 0, at_col = 0;
  const int64_t* mirror = nullptr;
};

}  // namespace

// One layer on the kernels for large layers; waits for its edge and key counts.
Graph::Layer Graph::large_layer(const torch::Tensor& cols, const torch::Tensor& col_bptr,
                                int64_t fanout, bool replace, const torch::Tensor& cdf,
                                uint64_t call_id, bool labels_wanted,
                                const std::function<void()>& idle) {
  const Compressed& m = compressed(kCSC);
  const int64_t B = col_bptr.numel() - 1, S = cols.numel();
  Layer l;
  EdgeCount::HintScope batch(col_bptr, /*no_select=*/true);
  MajorResult r = cdf.defined() ? major_sample_weighted(m, cdf, cols, fanout, replace, false, call_id)
                                : major_sample_uniform(m, cols, fanout, replace, false, call_id);
  l.sampled_indptr = r.indptr;
  l.edge_ptr = EdgeCount::hint().edge_bptr;
  if (!l.edge_ptr.defined()) l.edge_ptr = r.indptr.index_select(0, col_bptr);
  const torch::Tensor& rows = r.minor_ids;
  const bool rows32 = rows.scalar_type() == torch::kInt32;
  const int64_t E = rows.numel();
  const torch::Tensor labels = EdgeCount::hint().col_labels;
  const bool prefilled = labels_wanted && labels.defined() && labels.numel() == E && E > 0;
  if (labels_wanted) {
    l.row = new_ids(E, cols);
    l.col = prefilled ? labels : new_ids(E, cols);
  }
  torch::Tensor ws = new_workspace(gs_unique_workspace_bytes(S, E, B), cols);
  l.frontier_ptr = new_ids(B + 1, cols);
  int64_t* distinct = PinnedWords::take((size_t)B);
  int64_t* mirror = OffsetMirror::reserve(l.frontier_ptr);
  // the same calls for either width of the row ids
  auto calls = [&](auto* row_ids, auto count, auto fill, auto fill_relabel) {
    GS_CALL(count(cptr(cols), cptr(col_bptr), S, row_ids, cptr(l.edge_ptr), E, B,
                  mptr(l.frontier_ptr), mirror, distinct, ws.data_ptr(), ws.numel(), cur_stream()));
    OffsetMirror::arm(l.frontier_ptr);
    const int64_t bound = S + E <= kBoundLimit ? S + E : OffsetMirror::values(l.frontier_ptr).back();
    l.frontier = new_ids(bound, cols);
    if (labels_wanted)
      GS_CALL(fill_relabel(cptr(cols), cptr(col_bptr), S, row_ids, cptr(l.edge_ptr), E, B,
                           cptr(l.frontier_ptr), mptr(l.frontier), nullptr, cptr(r.indptr),
                           mptr(l.row), mptr(l.col), prefilled ? 1 : 0, ws.data_ptr(), ws.numel(),
                           cur_stream()));
    else
      GS_CALL(fill(cptr(cols), cptr(col_bptr), S, row_ids, cptr(l.edge_ptr), E, B,
                   cptr(l.frontier_ptr), mptr(l.frontier), ws.data_ptr(), ws.numel(), cur_stream()));
  };
  if (rows32)
    calls(E > 0 ? rows.data_ptr<int32_t>() : nullptr, gs_unique_count_distinct_rows32,
          gs_unique_fill_rows32, gs_unique_fill_relabel_rows32);
  else
    calls(cptr(rows), gs_unique_count_distinct, gs_unique_fill, gs_unique_fill_relabel);
  idle();
  l.e_off = OffsetMirror::values(l.edge_ptr);
  l.f_off = OffsetMirror::values(l.frontier_ptr);
  await_words(distinct, (size_t)B, (hipStream_t)cur_stream());
  PinnedWords::arrived();
  l.distinct.assign((size_t)B, 1);
  for (int64_t b = 0; b < B; ++b) l.distinct[(size_t)b] = distinct[b] != 0;
  l.frontier = l.frontier.narrow(0, 0, l.f_off.back());
  return l;
}

std::vector<Graph::Layer> Graph::sample_layers(const torch::Tensor& seeds,
                                               const torch::Tensor& col_bptr,
                                               const std::vector<int64_t>& fanouts, bool replace,
                                               const c10::optional<torch::Tensor>& edge_probs,
                                               bool blocks, const LayersIdle& idle, bool labels) {
  const Compressed& m = compressed(kCSC);
  const bool weighted = edge_probs.has_value();
  const torch::Tensor cdf = weighted ? weight_cdf_for(edge_probs.value(), kCSC) : torch::Tensor();
  const int64_t B = col_bptr.defined() ? col_bptr.numel() - 1 : 1;
  const int64_t num_cols = m.indptr.numel() - 1;
  const int64_t stride = std::max<int64_t>(std::max(num_cols, num_rows_), 1);
  const RandomState& rs = random_state();
  const uint64_t first_call = next_call_id(fanouts.size());  // a second attempt draws by the same ids
  // (rows of a matrix that was loaded or converted are known to lie below num_rows)
  bool small_ok = m.num_minor >= 0 && m.num_minor <= stride && B <= (int64_t)0xFFFFFFFEll / stride &&
                  (weighted || replace || rs.algo != GS_ALGO_RESERVOIR);
  auto fits = [&](int64_t columns, int64_t fanout, int64_t most) {
    return small_ok && columns > 0 && fanout >= 1 && fanout < 64 && columns <= most / (fanout + 1);
  };
  const torch::Tensor narrow = m.narrow_indices();
  const size_t L = fanouts.size();
  for (;;) {
    std::vector<Layer> out(L);
    std::vector<Queued> queued(L);
    const size_t words = (size_t)(3 * B + 3);
    LayerWorkspace lw;
    int64_t* mirrors = nullptr;
    bool retry = false;
    // the layer's columns: exact on the host, or a bound while `known` is false
    torch::Tensor cols = seeds, ptr = col_bptr;
    int64_t n = seeds.numel();
    bool known = true;
    size_t settled = 0;  // layers whose sizes are on the host
    // A layer's labels wait for the next one's picks, beside which they run.
    gs_layer unlabelled{};
    auto label = [&] {
      if (unlabelled.columns)
        GS_CALL(gs_sample_layer_next(&unlabelled, nullptr, cur_stream()));
      unlabelled = gs_layer{};
    };
    auto settle = [&](size_t upto) {
      label();
      for (; settled < upto; ++settled) {
        Queued& q = queued[settled];
        if (!q.buffer.defined()) continue;
        Layer& l = out[settled];
        await_words(q.mirror, words, (hipStream_t)cur_stream());
        const int64_t* w = q.mirror;
        l.f_off.assign(w, w + B + 1);
        l.e_off.assign(w + B + 1, w + 2 * (B + 1));
        l.distinct.resize((size_t)B);
        for (int64_t b = 0; b < B; ++b) l.distinct[(size_t)b] = w[2 * (B + 1) + b] != 0;
        retry = retry || w[3 * B + 2] != 0;
        l.frontier = piece_of(q.buffer, 0, l.f_off.back(), false);
        l.row = piece_of(q.buffer, q.at_row, l.e_off.back(), false);
        l.col = piece_of(q.buffer, q.at_col, l.e_off.back(), false);
        l.frontier_ptr = piece_of(q.buffer, q.at_ptr, B + 1, false);
        l.edge_ptr = piece_of(q.buffer, q.at_edge_ptr, B + 1, false);
        const int64_t columns = settled ? out[settled - 1].f_off.back() : seeds.numel();
        if (blocks) l.block_indptr = piece_of(q.buffer, q.at_indptr, columns + B, false);
      }
    };
    for (size_t i = 0; i < L && !retry; ++i) {
      const int64_t K = fanouts[i];
      if (!known && !fits(n, K, kQueuedPositions)) {
        settle(i);
        if (retry) break;
        n = out[i - 1].f_off.back();
        cols = out[i - 1].frontier;
        ptr = out[i - 1].frontier_ptr;
        known = true;
      }
      Layer& l = out[i];
      l.cols = cols;
      l.col_bptr = ptr;
      if (!fits(n, K, known ? kSmallPositions : kQueuedPositions)) {
        if (!ptr.defined()) {  // a single batch: offsets 0, n
          ptr = torch::arange(0, 2, device_options(m.indptr).dtype(torch::kInt64)) * n;
          BatchOffsets::trust(ptr, n);
        }
        label();
        PinnedWords::arrived();  // every layer queued so far has been settled
        l = large_layer(cols, ptr, K, replace, cdf, first_call + i, labels, [&] { idle(out, i); });
        mirrors = nullptr;  // it has used the thread's pinned words
        l.cols = cols;
        l.col_bptr = ptr;
        cols = l.frontier;
        ptr = l.frontier_ptr;
        n = cols.numel();
        settled = i + 1;
        continue;
      }
      const int64_t positions = n * (K + 1);
      if (!lw.ws.defined()) {
        std::lock_guard<std::mutex> lock(layer_ws_guard_);
        if (layer_ws_.ws.defined() && layer_ws_.stream == cur_stream() &&
            layer_ws_.weighted == weighted)
          std::swap(lw, layer_ws_);
      }
      if (lw.positions < positions) {
        label();
        // room for the layers that can be queued behind this one as well
        int64_t most = positions, bound = positions;
        for (size_t j = i + 1; j < L && fits(bound, fanouts[j], kQueuedPositions); ++j) {
          bound *= fanouts[j] + 1;
          most = std::max(most, bound);
        }
        lw.ws = new_workspace(gs_layer_workspace_bytes(most, weighted ? 1 : 0), m.indptr);
        lw.positions = most;
        lw.weighted = weighted;
        lw.stream = cur_stream();
        GS_CALL(gs_layer_begin(most, weighted ? 1 : 0, lw.ws.data_ptr(), (size_t)lw.ws.numel(),
                               cur_stream()));
      }
      if (!mirrors) mirrors = PinnedWords::take(words * L);
      Queued& q = queued[i];
      auto even = [](int64_t x) { return (x + 1) & ~int64_t(1); };
      int64_t at = even(positions);
      q.at_row = at;
      at += even(n * K);
      q.at_col = at;
      at += even(n * K);
      q.at_ptr = at;
      at += even(B + 1);
      q.at_edge_ptr = at;
      at += even(B + 1);
      q.at_indptr = at;
      at += blocks ? n + B : 0;
      q.buffer = new_ids(at, m.indptr);
      q.mirror = mirrors + words * i;
      int64_t* base = mptr(q.buffer);
      const gs_layer next{
          cptr(m.indptr), num_cols, cptr(m.indices),
          narrow.defined() ? narrow.data_ptr<int32_t>() : nullptr, cptr(cdf), stride, cptr(cols), n,
          cptr(ptr), B, K, replace ? 1 : 0, rs.seed, first_call + i, base, base + q.at_ptr,
          base + q.at_row, base + q.at_col, base + q.at_edge_ptr,
          blocks ? base + q.at_indptr : nullptr, mirrors + words * i, lw.positions, lw.ws.data_ptr(),
          (size_t)lw.ws.numel(), weighted ? 0 : (int)(i & 1)};
      GS_CALL(gs_sample_layer_next(unlabelled.columns ? &unlabelled : nullptr, &next, cur_stream()));
      unlabelled = next;
      // the next layer's columns, as far as they are known
      cols = piece_of(q.buffer, 0, positions, false);
      ptr = piece_of(q.buffer, q.at_ptr, B + 1, false);
      n = positions;
      known = false;
    }
    if (!retry) settle(L);
    if (!retry) {
      PinnedWords::arrived();
      for (size_t i = 1; i < L; ++i)
        if (queued[i - 1].buffer.defined()) {  // the pieces, in place of the bounds
          out[i].cols = out[i - 1].frontier;
          out[i].col_bptr = out[i - 1].frontier_ptr;
        }
      if (lw.ws.defined()) {
        std::lock_guard<std::mutex> lock(layer_ws_guard_);
        if (!layer_ws_.ws.defined() || layer_ws_.stream != lw.stream ||
            layer_ws_.positions <= lw.positions)
          std::swap(lw, layer_ws_);
      }
      for (const Layer& l : out) {
        BatchOffsets::trust(l.frontier_ptr, l.f_off.back());
        BatchOffsets::trust(l.edge_ptr, l.e_off.back());
      }
      return out;
    }
    // a seed that is no id of this matrix: its keys do not fit the small layers' table
    GS_CALL(hipStreamSynchronize((hipStream_t)cur_stream()) == hipSuccess ? GS_OK : GS_ERR_HIP);
    small_ok = false;
  }
}

static void check_layers(const std::vector<int64_t>& fanouts, bool replace, bool weighted) {
  TORCH_CHECK(!fanouts.empty(), "SampleLayers: no layers");
  for (int64_t k : fanouts) {
    TORCH_CHECK(k >= 0, "fanout must be non-negative, got ", k);
    if (weighted) check_weighted_fanout(k, replace, "SampleLayers");
  }
}

std::vector<c10::optional<torch::Tensor>> Graph::SampleLayers(
    torch::Tensor seeds, std::vector<int64_t> fanouts, bool replace,
    c10::optional<torch::Tensor> edge_probs) {
  check_layers(fanouts, replace, edge_probs.has_value());
  seeds = ids(seeds, "seeds");
  std::vector<c10::optional<torch::Tensor>> out;
  if (seeds.numel() == 0) {  // no columns, no edges: layer after layer
    next_call_id(fanouts.size());
    for (size_t i = 0; i < fanouts.size(); ++i) {
      const torch::Tensor none = new_ids(0, compressed(kCSC).indptr);
      out.insert(out.end(), {none, none.clone(), none.clone(), c10::nullopt});
    }
    return out;
  }
  for (Layer& l : sample_layers(seeds, {}, fanouts, replace, edge_probs, false,
                                [](std::vector<Layer>&, size_t) {}))
    out.insert(out.end(), {l.frontier, l.row, l.col, c10::nullopt});
  return out;
}

std::vector<torch::Tensor> Graph::BatchSampleNodes(torch::Tensor seeds, torch::Tensor col_bptr,
                                                   std::vector<int64_t> fanouts, bool replace,
                                                   c10::optional<torch::Tensor> edge_probs) {
  check_layers(fanouts, replace, edge_probs.has_value());
  seeds = ids(seeds, "seeds");
  col_bptr = ids(col_bptr, "col_bptr");
  BatchOffsets::check(col_bptr, seeds.numel(), "BatchSampleNodes");
  std::vector<torch::Tensor> out;
  for (Layer& l : sample_layers(seeds, col_bptr, fanouts, replace, edge_probs, false,
                                [](std::vector<Layer>&, size_t) {}, /*labels=*/false))
    out.insert(out.end(), {l.frontier, l.frontier_ptr});
  return out;
}

std::vector<c10::intrusive_ptr<BlockBatch>> Graph::BatchSampleLayersWhile(
    torch::Tensor seeds, torch::Tensor col_bptr, std::vector<int64_t> fanouts, bool replace,
    c10::optional<torch::Tensor> edge_probs, const LayerDone& done) {
  check_layers(fanouts, replace, edge_probs.has_value());
  seeds = ids(seeds, "seeds");
  col_bptr = ids(col_bptr, "col_bptr");
  BatchOffsets::check(col_bptr, seeds.numel(), "BatchSampleLayers");
  std::vector<int64_t> c_off = OffsetMirror::values(col_bptr);
  auto batch_of = [&](Layer& l) {
    auto b = c10::make_intrusive<BlockBatch>();
    b->num_batches = col_bptr.numel() - 1;
    b->num_dst_total = l.cols.numel();
    b->frontier = l.frontier;
    b->frontier_ptr = l.frontier_ptr;
    b->row = l.row;
    b->col = l.col;
    b->coo_ptr = l.edge_ptr;
    b->col_bptr = l.col_bptr;
    b->col_seeds = l.cols;
    b->sampled_indptr = l.sampled_indptr;
    b->indptr = l.block_indptr;
    std::vector<int64_t> f_off = l.f_off;
    b->set_host_offsets(l.f_off, l.e_off, std::move(c_off), l.distinct);
    c_off = std::move(f_off);
    return b;
  };
  size_t handed = 0;
  auto idle = [&](std::vector<Layer>& layers, size_t complete) {
    if (!done) return;
    for (; handed < complete; ++handed) done(batch_of(layers[handed]));
  };
  std::vector<Layer> layers =
      sample_layers(seeds, col_bptr, fanouts, replace, edge_probs, true, idle);
  std::vector<c10::intrusive_ptr<BlockBatch>> out;
  for (; handed < layers.size(); ++handed) out.push_back(batch_of(layers[handed]));
  return out;
}

std::vector<c10::intrusive_ptr<BlockBatch>> Graph::BatchSampleLayers(
    torch::Tensor seeds, torch::Tensor col_bptr, std::vector<int64_t> fanouts, bool replace,
    c10::optional<torch::Tensor> edge_probs) {
  return BatchSampleLayersWhile(seeds, col_bptr, fanouts, replace, edge_probs, LayerDone());
}

}  // namespace gs

// binding.cpp -- the Python side of the block hand-off, native: a compiled
// super-batched sampler hands out a few hundred Block objects per step, each with
// half a dozen tensors, and a call through torch's custom classes converts every
// one of them through IValue lists.  Here the objects are filled directly, and the
// blocks of the layers that are done are made while the host would otherwise wait
// for the counts of the next one, if nobody else wants the interpreter.
//
//   sample_layers(graph, seeds, fanouts, replace, weights)
//       -> (frontier, row, col, None) per layer, one flat tuple
//   batch_sample_layers(graph, seeds, seeds_ptr, fanouts, replace, weights)
//       -> one BlockBatch per layer
//   batch_sample_nodes(graph, seeds, seeds_ptr, fanouts, replace, weights)
//       -> (frontier, frontier_ptr) per layer, one flat tuple
//   edge_score(graph, kinds, lhs, rhs, targets, weights, positive_part, shift, on_format)
//       -> a value per edge, or None where the call is not one for the kernel
//   list_sampling(probs, num_picks, replace, ranges or None)
//       -> (picks, their offsets, their weights), or None likewise
//   BlockBatch   the operator library's class of that name with its methods, plus
//       make_blocks(): the list of Block objects
//   wrap(batch)  the same around a batch that came through torch
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/api/object.h>
#include <torch/csrc/utils/pybind.h>

#include <structmember.h>

#include <atomic>

#include "../abi_call.h"
#include "../graph.h"

namespace py = pybind11;

namespace {

// gsampler_amd.utils.block.Block and where its slots live in an instance.
struct BlockClass {
  PyTypeObject* type = nullptr;
  Py_ssize_t row, col, num_src, num_dst, srcdata, dstdata, edata, indptr;
};
BlockClass g_block;
PyObject* g_id_key = nullptr;  // "_ID"

Py_ssize_t slot_offset(PyTypeObject* type, const char* name) {
  PyObject* d = PyDict_GetItemString(type->tp_dict, name);  // borrowed
  TORCH_CHECK(d && Py_TYPE(d) == &PyMemberDescr_Type, "Block has no slot '", name, "'");
  return ((PyMemberDescrObject*)d)->d_member->offset;
}

void set_block_class(py::object cls) {
  TORCH_CHECK(PyType_Check(cls.ptr()), "set_block_class: not a class");
  auto* type = (PyTypeObject*)cls.ptr();
  BlockClass b;
  b.type = type;
  b.row = slot_offset(type, "row");
  b.col = slot_offset(type, "col");
  b.num_src = slot_offset(type, "num_src");
  b.num_dst = slot_offset(type, "num_dst");
  b.srcdata = slot_offset(type, "srcdata");
  b.dstdata = slot_offset(type, "dstdata");
  b.edata = slot_offset(type, "edata");
  b.indptr = slot_offset(type, "indptr");
  Py_INCREF(type);
  g_block = b;
  g_id_key = PyUnicode_InternFromString("_ID");
}

// Takes over the reference to `value`.
inline void put(PyObject* object, Py_ssize_t offset, PyObject* value) {
  if (!value) throw py::error_already_set();
  PyObject** at = (PyObject**)((char*)object + offset);
  PyObject* old = *at;
  *at = value;
  Py_XDECREF(old);
}

inline PyObject* wrap_tensor(torch::Tensor t) { return THPVariable_Wrap(std::move(t)); }

class Batch {
 public:
  explicit Batch(c10::intrusive_ptr<gs::BlockBatch> b) : b_(std::move(b)) {}
  gs::BlockBatch& get() { return *b_; }

  // The blocks may be made before anybody asks for them.
  void make_ahead() { ahead_ = make_blocks(); }

  // All blocks of the layer, objects of the caller's own: those made ahead go to the
  // first who asks, another hand-out of the same layer gets others.
  py::list make_blocks() {
    if (ahead_) return py::reinterpret_steal<py::list>(ahead_.release());
    TORCH_CHECK(g_block.type, "the Block class has not been set");
    gs::BlockBatch& b = *b_;
    auto off = b.Offsets();
    const std::vector<int64_t>&f = std::get<0>(off), &c = std::get<1>(off), &e = std::get<2>(off);
    const int64_t n = b.num_batches;
    const torch::Tensor indptr = b.Indptr();
    py::list out((size_t)n);
    for (int64_t i = 0; i < n; ++i) {
      const int64_t ne = e[i + 1] - e[i], nf = f[i + 1] - f[i], nc = c[i + 1] - c[i];
      py::object block = py::reinterpret_steal<py::object>(g_block.type->tp_alloc(g_block.type, 0));
      if (!block) throw py::error_already_set();
      PyObject* o = block.ptr();
      put(o, g_block.row, wrap_tensor(gs::piece_of(b.row, e[i], ne)));
      put(o, g_block.col, wrap_tensor(gs::piece_of(b.col, e[i], ne)));
      put(o, g_block.num_src, PyLong_FromLongLong(nf));
      put(o, g_block.num_dst, PyLong_FromLongLong(nc));
      if (b.grouped(i)) {
        put(o, g_block.indptr, wrap_tensor(gs::piece_of(indptr, c[i] + i, nc + 1)));
      } else {
        Py_INCREF(Py_None);
        put(o, g_block.indptr, Py_None);
      }
      auto with_id = [&](torch::Tensor ids) {
        py::object d = py::reinterpret_steal<py::object>(PyDict_New());
        py::object v = py::reinterpret_steal<py::object>(wrap_tensor(std::move(ids)));
        if (!d || !v || PyDict_SetItem(d.ptr(), g_id_key, v.ptr()) != 0) throw py::error_already_set();
        return d.release().ptr();
      };
      put(o, g_block.srcdata, with_id(gs::piece_of(b.frontier, f[i], nf)));
      put(o, g_block.dstdata, PyDict_New());
      if (b.e_ids.has_value())
        put(o, g_block.edata, with_id(gs::piece_of(b.e_ids.value(), e[i], ne)));
      else
        put(o, g_block.edata, PyDict_New());
      PyList_SET_ITEM(out.ptr(), i, block.release().ptr());
    }
    return out;
  }

 private:
  c10::intrusive_ptr<gs::BlockBatch> b_;
  py::object ahead_;  // a list, or nothing
};

// The C++ object behind a torch custom-class instance.
template <typename T>
c10::intrusive_ptr<T> unwrap(const py::handle& h) {
  const auto& object = py::cast<const torch::jit::Object&>(h);
  return c10::IValue(object._ivalue()).toCustomClass<T>();
}

c10::optional<torch::Tensor> optional_tensor(const py::object& o) {
  if (o.is_none()) return c10::nullopt;
  return py::cast<torch::Tensor>(o);
}

// Whether the interpreter can be had at once: nobody holds it.  (Asked by a thread that
// has let go of it; up to Python 3.11 the running thread's state is the process's, later
// a thread sees its own only, and the answer is whether there is another thread at all.)
class Interpreter {
 public:
  Interpreter() {
#if PY_VERSION_HEX >= 0x030C0000
    alone_ = PyThreadState_Next(PyInterpreterState_ThreadHead(PyThreadState_Get()->interp)) == nullptr;
#endif
  }
  bool is_free() const {
#if PY_VERSION_HEX >= 0x030C0000
    return alone_;
#else
    return _PyThreadState_UncheckedGet() == nullptr;
#endif
  }

 private:
  bool alone_ = true;
};

// Calls of batch_sample_layers under way, in all threads.
std::atomic<int> g_calls{0};
struct CallScope {
  CallScope() { g_calls.fetch_add(1, std::memory_order_relaxed); }
  ~CallScope() { g_calls.fetch_sub(1, std::memory_order_relaxed); }
  static bool only_one() { return g_calls.load(std::memory_order_relaxed) == 1; }
};

py::tuple sample_layers(py::handle graph, torch::Tensor seeds, std::vector<int64_t> fanouts,
                        bool replace, py::object weights) {
  auto g = unwrap<gs::Graph>(graph);
  auto w = optional_tensor(weights);
  std::vector<c10::optional<torch::Tensor>> got;
  {
    py::gil_scoped_release nogil;
    got = g->SampleLayers(std::move(seeds), std::move(fanouts), replace, std::move(w));
  }
  py::tuple out(got.size());
  for (size_t i = 0; i < got.size(); ++i) {
    PyObject* v;
    if (got[i].has_value()) {
      v = wrap_tensor(std::move(*got[i]));
      if (!v) throw py::error_already_set();
    } else {
      Py_INCREF(Py_None);
      v = Py_None;
    }
    PyTuple_SET_ITEM(out.ptr(), (Py_ssize_t)i, v);
  }
  return out;
}

py::tuple batch_sample_nodes(py::handle graph, torch::Tensor seeds, torch::Tensor ptr,
                             std::vector<int64_t> fanouts, bool replace, py::object weights) {
  auto g = unwrap<gs::Graph>(graph);
  auto w = optional_tensor(weights);
  std::vector<torch::Tensor> got;
  {
    py::gil_scoped_release nogil;
    got = g->BatchSampleNodes(std::move(seeds), std::move(ptr), std::move(fanouts), replace,
                              std::move(w));
  }
  py::tuple out(got.size());
  for (size_t i = 0; i < got.size(); ++i) {
    PyObject* v = wrap_tensor(std::move(got[i]));
    if (!v) throw py::error_already_set();
    PyTuple_SET_ITEM(out.ptr(), (Py_ssize_t)i, v);
  }
  return out;
}

// -> the scores, or None where torch's own operators have to do it.
py::object edge_score(py::handle graph, std::vector<int64_t> kinds, py::list lhs, py::list rhs,
                      std::vector<int64_t> targets, py::object weights, bool positive_part,
                      double shift, int64_t on_format) {
  auto g = unwrap<gs::Graph>(graph);
  std::vector<torch::Tensor> l, r;
  for (const py::handle& t : lhs) {
    if (!THPVariable_CheckExact(t.ptr())) return py::none();
    l.push_back(THPVariable_Unpack(t.ptr()));
  }
  for (const py::handle& t : rhs) {
    if (t.is_none()) {
      r.emplace_back();
      continue;
    }
    if (!THPVariable_CheckExact(t.ptr())) return py::none();
    r.push_back(THPVariable_Unpack(t.ptr()));
  }
  c10::optional<torch::Tensor> w;
  if (!weights.is_none()) {
    if (!THPVariable_CheckExact(weights.ptr())) return py::none();
    w = THPVariable_Unpack(weights.ptr());
  }
  c10::optional<torch::Tensor> out;
  {
    py::gil_scoped_release nogil;
    out = g->EdgeScore(kinds, std::move(l), std::move(r), targets, std::move(w), positive_part,
                       shift, on_format);
  }
  if (!out.has_value()) return py::none();
  return py::reinterpret_steal<py::object>(wrap_tensor(std::move(*out)));
}

py::object list_sampling(py::handle probs, int64_t num_picks, bool replace, py::object ranges) {
  if (!THPVariable_CheckExact(probs.ptr())) return py::none();
  torch::Tensor p = THPVariable_Unpack(probs.ptr());
  auto r = optional_tensor(ranges);
  c10::optional<std::tuple<torch::Tensor, torch::Tensor, torch::Tensor>> got;
  {
    py::gil_scoped_release nogil;
    got = gs::ListSamplingPicked(std::move(p), num_picks, replace, std::move(r));
  }
  if (!got.has_value()) return py::none();
  py::tuple out(3);
  torch::Tensor* parts[] = {&std::get<0>(*got), &std::get<1>(*got), &std::get<2>(*got)};
  for (Py_ssize_t i = 0; i < 3; ++i) {
    PyObject* v = wrap_tensor(std::move(*parts[i]));
    if (!v) throw py::error_already_set();
    PyTuple_SET_ITEM(out.ptr(), i, v);
  }
  return out;
}

std::vector<std::shared_ptr<Batch>> batch_sample_layers(py::handle graph, torch::Tensor seeds,
                                                        torch::Tensor ptr,
                                                        std::vector<int64_t> fanouts, bool replace,
                                                        py::object weights) {
  auto g = unwrap<gs::Graph>(graph);
  auto w = optional_tensor(weights);
  std::vector<std::shared_ptr<Batch>> out;
  // called where the host is about to wait for a layer's counts, with the layers
  // before it: their blocks are made now instead of after the wait.  Not while another
  // thread holds the interpreter, which would keep the next layer's launches waiting,
  // nor beside another sampler thread: every tensor of a block lets go of the
  // interpreter when it is freed.  (32 batches of 1024 on 2 M edges, blocks never asked
  // for, 1 and 8 threads: 3020 and 635 passes a second with blocks always made ahead,
  // 3140 and 5130 without.)
  const Interpreter interpreter;
  const CallScope scope;
  auto done = [&](c10::intrusive_ptr<gs::BlockBatch> b) {
    if (g_block.type && CallScope::only_one() && interpreter.is_free()) {
      py::gil_scoped_acquire gil;
      out.push_back(std::make_shared<Batch>(std::move(b)));
      out.back()->make_ahead();
    } else {
      out.push_back(std::make_shared<Batch>(std::move(b)));
    }
  };
  std::vector<c10::intrusive_ptr<gs::BlockBatch>> got;
  {
    py::gil_scoped_release nogil;
    got = g->BatchSampleLayersWhile(std::move(seeds), std::move(ptr), std::move(fanouts), replace,
                                    std::move(w), done);
  }
  for (auto& b : got) out.push_back(std::make_shared<Batch>(std::move(b)));
  return out;
}

}  // namespace

PYBIND11_MODULE(_gs_python, m) {
  m.def("set_block_class", &set_block_class);
  m.def("sample_layers", &sample_layers);
  m.def("batch_sample_layers", &batch_sample_layers);
  m.def("batch_sample_nodes", &batch_sample_nodes);
  m.def("edge_score", &edge_score);
  m.def("list_sampling", &list_sampling);
  m.def("wrap", [](py::handle batch) { return std::make_shared<Batch>(unwrap<gs::BlockBatch>(batch)); });
  py::class_<Batch, std::shared_ptr<Batch>>(m, "BlockBatch")
      .def("make_blocks", &Batch::make_blocks)
      .def("size", [](Batch& b) { return b.get().Size(); })
      .def("totals", [](Batch& b) { return b.get().Totals(); })
      .def("offsets", [](Batch& b) { return b.get().Offsets(); })
      .def("block", [](Batch& b, int64_t i) { return b.get().Block(i); })
      .def("blocks", [](Batch& b) { return b.get().Blocks(); })
      .def("num_src_of", [](Batch& b, int64_t i) { return b.get().NumSrcOf(i); })
      .def("frontier", [](Batch& b) { return b.get().Frontier(); })
      .def("frontier_ptr", [](Batch& b) { return b.get().FrontierPtr(); })
      .def("row", [](Batch& b) { return b.get().Row(); })
      .def("col", [](Batch& b) { return b.get().Col(); })
      .def("indptr", [](Batch& b) { return b.get().Indptr(); })
      .def("edge_ptr", [](Batch& b) { return b.get().EdgePtr(); })
      .def("col_ptr", [](Batch& b) { return b.get().ColPtr(); })
      .def("edge_ids", [](Batch& b) { return b.get().EdgeIds(); });
}

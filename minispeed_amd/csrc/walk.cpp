// Host-side pointer walk for the boundary's segment tables.
//
// At every boundary the engine needs the device address of each parameter's
// gradient (K1 / K3 read them) and of each parameter's storage (K3 writes the
// model copy there).  Done attribute by attribute from Python this costs
// ~0.3 us per tensor before K1 can launch; here it is one call per group.
//
// Both functions take the group's parameters and only look at tensor
// metadata.  They never raise for a bad tensor: they return the index of the
// first parameter that is not on the fast path (wrong dtype, size, device or
// layout), and the caller re-walks from there in Python, which raises the
// precise error or makes the contiguous copy.  Everything on the fast path is
// exactly what the Python walk would have accepted.

#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <pybind11/numpy.h>
#include <pybind11/stl.h>

#include <c10/core/Stream.h>
#include <c10/core/impl/VirtualGuardImpl.h>

#include <algorithm>
#include <array>
#include <cstdint>
#include <cstring>
#include <optional>
#include <utility>
#include <vector>

namespace py = pybind11;

namespace {

at::Tensor unpack(PyObject* obj) {
  if (!THPVariable_Check(obj)) {
    throw py::type_error("expected a torch.Tensor / nn.Parameter");
  }
  return THPVariable_Unpack(obj);
}

bool on_fast_path(const at::Tensor& t, at::ScalarType dtype, int64_t numel, int64_t device_index) {
  return t.scalar_type() == dtype && t.numel() == numel && t.is_cuda() &&
         t.get_device() == device_index && t.is_contiguous();
}

// grad_pointers(params, numels, device_index, out) -> (bad, keep)
//   out[k]  : data_ptr of params[k].grad, 0 when it has none
//   keep[k] : params[k].grad (None when it has none), to hold the storage
//             until the kernels reading it are queued
//   bad     : -1, or the first k whose gradient needs the slow path (then
//             out and keep cover indices < bad only)
py::tuple grad_pointers(py::list params, py::array_t<int64_t, py::array::c_style> numels,
                        int64_t device_index, py::array_t<int64_t, py::array::c_style> out) {
  const Py_ssize_t n = PyList_GET_SIZE(params.ptr());
  if (numels.size() != n || out.size() < n) {
    throw py::value_error("numels / out must have one entry per parameter");
  }
  const int64_t* num = numels.data();
  int64_t* dst = out.mutable_data();
  py::list keep;
  if (n == 0) return py::make_tuple(-1, keep);
  const at::ScalarType dtype = unpack(PyList_GET_ITEM(params.ptr(), 0)).scalar_type();
  for (Py_ssize_t k = 0; k < n; ++k) {
    const at::Tensor p = unpack(PyList_GET_ITEM(params.ptr(), k));
    const at::Tensor& g = p.grad();
    if (!g.defined()) {
      dst[k] = 0;
      keep.append(py::none());
      continue;
    }
    if (!on_fast_path(g, dtype, num[k], device_index)) {
      return py::make_tuple(static_cast<int64_t>(k), keep);
    }
    dst[k] = reinterpret_cast<int64_t>(g.data_ptr());
    keep.append(py::reinterpret_steal<py::object>(THPVariable_Wrap(g)));
  }
  return py::make_tuple(-1, keep);
}

// model_pointers(params, device_index, out[, numels]) -> bad
//   out[k] : data_ptr of params[k] (the cast target), all of the group dtype
//            (params[0]'s), contiguous, on the device and, where numels are
//            given, of that size
//   bad    : -1, or the first k that is not
int64_t model_pointers(py::list params, int64_t device_index,
                       py::array_t<int64_t, py::array::c_style> out,
                       std::optional<py::array_t<int64_t, py::array::c_style>> numels) {
  const Py_ssize_t n = PyList_GET_SIZE(params.ptr());
  if (out.size() < n || (numels && numels->size() != n)) {
    throw py::value_error("numels / out must have one entry per parameter");
  }
  const int64_t* num = numels ? numels->data() : nullptr;
  int64_t* dst = out.mutable_data();
  if (n == 0) return -1;
  const at::ScalarType dtype = unpack(PyList_GET_ITEM(params.ptr(), 0)).scalar_type();
  for (Py_ssize_t k = 0; k < n; ++k) {
    const at::Tensor p = unpack(PyList_GET_ITEM(params.ptr(), k));
    if (!(p.scalar_type() == dtype && p.is_cuda() && p.get_device() == device_index &&
          p.is_contiguous() && (num == nullptr || p.numel() == num[k]))) {
      return static_cast<int64_t>(k);
    }
    dst[k] = reinterpret_cast<int64_t>(p.data_ptr());
  }
  return -1;
}

// Tensor.record_stream on tensors one after another, without a dispatch per
// tensor and once for neighbours in one storage (192 gradients: 23 -> 9 us,
// 2 us in one storage).  The tensors are alive at least as long as this is.
class StreamRecorder {
 public:
  StreamRecorder(int64_t device_type, int64_t device_index, int64_t stream_id)
      : stream_(c10::Stream::UNSAFE,
                c10::Device(static_cast<c10::DeviceType>(device_type),
                            static_cast<c10::DeviceIndex>(device_index)),
                static_cast<c10::StreamId>(stream_id)),
        impl_(stream_.device_type()) {}

  void record(const at::Tensor& t) {
    const c10::Storage& storage = t.storage();
    if (storage.unsafeGetStorageImpl() == last_) return;
    last_ = storage.unsafeGetStorageImpl();
    impl_.recordDataPtrOnStream(storage.data_ptr(), stream_);
  }

 private:
  c10::Stream stream_;
  c10::impl::VirtualGuardImpl impl_;
  const c10::StorageImpl* last_ = nullptr;
};

// record_streams(tensors, device_type, device_index, stream_id) -> count
//   Every device tensor of `tensors` (None entries and host tensors are
//   skipped): the caching allocator then hands their memory out again only
//   after the work queued on that stream by the time they are freed.
int64_t record_streams(py::list tensors, int64_t device_type, int64_t device_index,
                       int64_t stream_id) {
  StreamRecorder recorder(device_type, device_index, stream_id);
  int64_t count = 0;
  const Py_ssize_t n = PyList_GET_SIZE(tensors.ptr());
  for (Py_ssize_t k = 0; k < n; ++k) {
    PyObject* obj = PyList_GET_ITEM(tensors.ptr(), k);
    if (obj == Py_None) continue;
    const at::Tensor t = unpack(obj);
    if (!t.is_cuda()) continue;
    recorder.record(t);
    ++count;
  }
  return count;
}

// param.grad = None for every parameter of the list
void release_grads(py::list params) {
  const Py_ssize_t n = PyList_GET_SIZE(params.ptr());
  for (Py_ssize_t k = 0; k < n; ++k) {
    PyObject* obj = PyList_GET_ITEM(params.ptr(), k);
    if (THPVariable_CheckExact(obj)) {
      const at::Tensor p = THPVariable_Unpack(obj);
      if (p.grad().defined()) p.mutable_grad().reset();
    } else if (PyObject_SetAttrString(obj, "grad", Py_None) != 0) {
      throw py::error_already_set();
    }
  }
}

// Two tables of the same length hold the same bytes
bool same_table(py::array_t<int64_t, py::array::c_style> a,
                py::array_t<int64_t, py::array::c_style> b) {
  return a.size() == b.size() && std::memcmp(a.data(), b.data(), a.size() * sizeof(int64_t)) == 0;
}

// The boundary's segment table over a whole group, one table for K1 and K3:
// the rows (begin, numel) stay, the gradient and model columns are filled in
// place at each boundary.
class BoundaryRows {
 public:
  // (taken from an array at once; as std::vector each entry is a Python int)
  using Ints = py::array_t<int64_t, py::array::c_style | py::array::forcecast>;

  // rows: [n, 4], its first two columns set (copied); index: each row's
  // parameter (the parameter count: the padding row)
  BoundaryRows(py::list params, const Ints& numels, int64_t device_index,
               const py::array_t<int64_t, py::array::c_style>& rows, const Ints& index)
      : params_(std::move(params)), numels_(numels.data(), numels.data() + numels.size()),
        device_(device_index),
        // (a copy of known type; one from the buffer's description takes 11 us
        // in numpy's format parser)
        rows_({rows.shape(), rows.shape() + rows.ndim()}, rows.data()),
        index_(index.data(), index.data() + index.size()) {
    const int64_t n = static_cast<int64_t>(numels_.size());
    if (rows_.ndim() != 2 || rows_.shape(1) != 4 ||
        rows_.shape(0) != static_cast<py::ssize_t>(index_.size())) {
      throw py::value_error("rows must be [n, 4] with one index per row");
    }
    for (int64_t k : index_) {
      if (k < 0 || k > n) throw py::value_error("row index out of range");
    }
  }

  py::array_t<int64_t, py::array::c_style> table() const { return rows_; }

  // Fill the gradient column from param.grad and hold the gradients for
  // kernels on the given stream.  -1, or the first parameter whose gradient
  // needs the slow path; then nothing is held.
  int64_t grads(int64_t device_type, int64_t device_index, int64_t stream_id) {
    std::vector<int64_t> ptrs(numels_.size() + 1, 0);
    held_.clear();
    stream_ = {device_type, device_index, stream_id};
    check_params();
    if (!numels_.empty()) {
      const at::ScalarType dtype = param(0).scalar_type();
      for (size_t k = 0; k < numels_.size(); ++k) {
        const at::Tensor p = param(k);
        const at::Tensor& g = p.grad();
        if (!g.defined()) continue;
        if (!on_fast_path(g, dtype, numels_[k], device_)) {
          held_.clear();
          return static_cast<int64_t>(k);
        }
        ptrs[k] = reinterpret_cast<int64_t>(g.data_ptr());
        held_.push_back(g);
      }
    }
    column(2, ptrs.data());
    return -1;
  }

  // Fill the gradient column with given addresses (one per parameter and a
  // trailing 0 for the padding row).
  void set_grads(py::array_t<int64_t, py::array::c_style> ptrs) {
    check_addresses(ptrs);
    held_.clear();
    column(2, ptrs.data());
  }

  // Fill the model column with the parameters' storages (write false: with
  // zeros).  -1, or the first parameter that is not contiguous storage of the
  // group's dtype and of the parameter's full size on its device: K3 writes
  // whole rows.
  int64_t models(bool write) {
    std::vector<int64_t> ptrs(numels_.size() + 1, 0);
    check_params();
    if (write && !numels_.empty()) {
      const at::ScalarType dtype = param(0).scalar_type();
      for (size_t k = 0; k < numels_.size(); ++k) {
        const at::Tensor p = param(k);
        if (!(p.scalar_type() == dtype && p.is_cuda() && p.get_device() == device_ &&
              p.is_contiguous() && p.numel() == numels_[k])) {
          return static_cast<int64_t>(k);
        }
        ptrs[k] = reinterpret_cast<int64_t>(p.data_ptr());
      }
    }
    column(3, ptrs.data());
    return -1;
  }

  // Fill the model column with given addresses, as set_grads.
  void set_models(py::array_t<int64_t, py::array::c_style> ptrs) {
    check_addresses(ptrs);
    column(3, ptrs.data());
  }

  // Record the stream on the gradients and let go of them (their readers are
  // queued): nothing before the kernels waits for it.
  void drop() {
    if (held_.empty()) return;
    StreamRecorder recorder(stream_[0], stream_[1], stream_[2]);
    for (const at::Tensor& g : held_) recorder.record(g);
    held_.clear();
  }

  // The parameter list is shown to the garbage collector: parameters that
  // refer to the group (an attribute, a hook over the engine) make a cycle
  // through this object, and with it unseen the group's buffers stayed.
  static void collectable(PyHeapTypeObject* heap_type) {
    PyTypeObject* type = &heap_type->ht_type;
    type->tp_flags |= Py_TPFLAGS_HAVE_GC;
    type->tp_traverse = [](PyObject* obj, visitproc visit, void* arg) {
      Py_VISIT(Py_TYPE(obj));
      if (py::detail::is_holder_constructed(obj)) {
        Py_VISIT(py::cast<BoundaryRows&>(py::handle(obj)).params_.ptr());
      }
      return 0;
    };
    type->tp_clear = [](PyObject* obj) {
      if (py::detail::is_holder_constructed(obj)) {
        py::list empty;
        std::swap(py::cast<BoundaryRows&>(py::handle(obj)).params_, empty);
      }
      return 0;
    };
  }

 private:
  at::Tensor param(size_t k) const { return unpack(PyList_GET_ITEM(params_.ptr(), k)); }

  void check_params() const {
    if (PyList_GET_SIZE(params_.ptr()) != static_cast<Py_ssize_t>(numels_.size())) {
      throw py::value_error("the parameter list changed its length");
    }
  }

  void check_addresses(const py::array_t<int64_t, py::array::c_style>& ptrs) const {
    if (ptrs.size() != static_cast<py::ssize_t>(numels_.size()) + 1) {
      throw py::value_error("one address per parameter and one for the padding");
    }
  }

  void column(int c, const int64_t* ptrs) {
    int64_t* rows = rows_.mutable_data();
    for (size_t r = 0; r < index_.size(); ++r) rows[4 * r + c] = ptrs[index_[r]];
  }

  py::list params_;
  std::vector<int64_t> numels_;
  int64_t device_;
  py::array_t<int64_t, py::array::c_style> rows_;
  std::vector<int64_t> index_;
  std::vector<at::Tensor> held_;
  std::array<int64_t, 3> stream_{};   // device type and index, id
};

// The gradients queued for K5 (contiguous gradients), one entry per hook call,
// and the rows K5 takes them in.  A hook runs for every parameter and
// micro-batch; checked, queued and released from Python it took 3.2 us, here
// 0.24 us with the Python call around it (192 parameters, four micro-batches:
// 2.68 ms of host time a window, the kernels 0.2 ms).
class GradQueue {
 public:
  // A group: every parameter's element count, its offset in the fp32 sums at
  // `accum`, and its first statistics slot in `sumsq` / `flag`.
  void add_group(int64_t device_index, const std::vector<int64_t>& numels,
                 const std::vector<int64_t>& offsets, const std::vector<int64_t>& tile0,
                 int64_t accum, int64_t sumsq, int64_t flag) {
    if (offsets.size() != numels.size() || tile0.size() != numels.size()) {
      throw py::value_error("numels, offsets and tile0 must have one entry per parameter");
    }
    Group g{device_index, accum, sumsq, flag, {}};
    for (size_t k = 0; k < numels.size(); ++k) {
      g.params.push_back({numels[k], offsets[k], tile0[k], -1, false, false});
    }
    groups_.push_back(std::move(g));
  }

  // Queue and release param.grad.  Returns the queued elements, kNone when
  // there is no gradient, kSlow for whatever the caller has to look at (a
  // tensor subclass, a gradient of another size, device, dtype or layout) and
  // kAgain when the parameter is queued already; those three change nothing.
  int64_t take(int64_t gi, int64_t k, py::handle param) {
    Param& p = at(gi, k);
    if (!THPVariable_CheckExact(param.ptr())) return kSlow;
    const at::Tensor& t = THPVariable_Unpack(param.ptr());
    const at::Tensor& g = t.grad();
    if (!g.defined()) return kNone;
    if (g.layout() != at::kStrided || g.numel() != p.numel || !g.is_cuda() ||
        g.get_device() != groups_[gi].device || ms_dtype(g.scalar_type()) < 0 ||
        !g.is_contiguous()) {
      return kSlow;
    }
    if (p.queued) return kAgain;
    push(gi, k, p, std::move(t.mutable_grad()));
    return queued_;
  }

  // Queue a gradient that the caller checked and made contiguous.
  int64_t put(int64_t gi, int64_t k, py::handle grad) {
    Param& p = at(gi, k);
    const at::Tensor g = unpack(grad.ptr());
    if (g.numel() != p.numel || ms_dtype(g.scalar_type()) < 0 || !g.is_contiguous()) {
      throw py::value_error("a contiguous f32 / f16 / bf16 gradient of the parameter's size");
    }
    if (p.queued) return kAgain;
    push(gi, k, p, g);
    return queued_;
  }

  bool empty() const { return entries_.empty(); }

  // The queue's content as [(device index, MS_DTYPE_*, rows, gradients)], one
  // item per device and dtype, group by group in the order they came; rows are
  // ms_accum_row_t records (48 bytes).  The queue is empty afterwards.
  py::list rows() {
    struct Batch {
      int64_t device;
      int dtype;
      std::vector<std::array<int64_t, 6>> rows;
      py::list grads;
    };
    std::vector<Batch> batches;
    // a group's rows one after another: K5 takes few buffers in one launch
    std::stable_sort(entries_.begin(), entries_.end(),
                     [](const Entry& a, const Entry& b) { return a.group < b.group; });
    for (Entry& e : entries_) {
      const Group& g = groups_[e.group];
      Param& p = groups_[e.group].params[e.index];
      const int dtype = ms_dtype(e.grad.scalar_type());
      Batch* b = nullptr;
      for (Batch& x : batches) {
        if (x.device == g.device && x.dtype == dtype) b = &x;
      }
      if (b == nullptr) {
        batches.push_back({g.device, dtype, {}, py::list()});
        b = &batches.back();
      }
      b->rows.push_back({g.accum + 4 * p.offset, reinterpret_cast<int64_t>(e.grad.data_ptr()),
                         p.numel, e.first ? 1 : 0, g.sumsq + 8 * p.tile0, g.flag + 4 * p.tile0});
      b->grads.append(py::reinterpret_steal<py::object>(THPVariable_Wrap(e.grad)));
      p.queued = false;
    }
    entries_.clear();
    queued_ = 0;
    py::list out;
    for (Batch& b : batches) {
      py::array_t<int64_t> rows({static_cast<py::ssize_t>(b.rows.size()), py::ssize_t{6}});
      std::memcpy(rows.mutable_data(), b.rows.data(), b.rows.size() * sizeof(b.rows[0]));
      out.append(py::make_tuple(b.device, b.dtype, std::move(rows), std::move(b.grads)));
    }
    return out;
  }

  // out[k]: the address of parameter k's sums, 0 where none came this window
  void pointers(int64_t gi, py::array_t<int64_t, py::array::c_style> out) const {
    const Group& g = groups_.at(gi);
    if (out.size() < static_cast<py::ssize_t>(g.params.size())) {
      throw py::value_error("out must have one entry per parameter");
    }
    int64_t* dst = out.mutable_data();
    for (size_t k = 0; k < g.params.size(); ++k) {
      dst[k] = g.params[k].seen == window_ ? g.accum + 4 * g.params[k].offset : 0;
    }
  }

  // The slot ranges [begin, end) that still hold an earlier window's
  // statistics, of parameters without a gradient in this one; they count as
  // cleared from here on.
  std::vector<std::pair<int64_t, int64_t>> stale_slots(int64_t gi, int64_t tile) {
    std::vector<std::pair<int64_t, int64_t>> out;
    for (Param& p : groups_.at(gi).params) {
      if (!p.stats || p.seen == window_) continue;
      p.stats = false;
      const int64_t end = p.tile0 + (p.numel + tile - 1) / tile;
      if (!out.empty() && out.back().second == p.tile0) {
        out.back().second = end;
      } else if (end > p.tile0) {
        out.emplace_back(p.tile0, end);
      }
    }
    return out;
  }

  // Drop what is queued and start the next window.
  void next_window() {
    for (const Entry& e : entries_) groups_[e.group].params[e.index].queued = false;
    entries_.clear();
    queued_ = 0;
    ++window_;
  }

  // The queue over a copy of the groups' buffers (accum, sumsq, flag of
  // each): the same windows and slots, nothing queued yet.
  GradQueue rebased(const std::vector<std::array<int64_t, 3>>& buffers) const {
    if (buffers.size() != groups_.size() || !entries_.empty()) {
      throw py::value_error("one (accum, sumsq, flag) per group, and an empty queue");
    }
    GradQueue q(*this);
    for (size_t g = 0; g < buffers.size(); ++g) {
      q.groups_[g].accum = buffers[g][0];
      q.groups_[g].sumsq = buffers[g][1];
      q.groups_[g].flag = buffers[g][2];
    }
    return q;
  }

  static constexpr int64_t kNone = -1, kSlow = -2, kAgain = -3;

 private:
  struct Param {
    int64_t numel, offset, tile0, seen;   // seen: the window it last contributed in
    bool queued;
    bool stats;   // its slots hold statistics (not zeros)
  };
  struct Group {
    int64_t device, accum, sumsq, flag;
    std::vector<Param> params;
  };
  struct Entry {
    int64_t group, index;
    at::Tensor grad;
    bool first;   // of its window: K5 overwrites the sums
  };

  static int ms_dtype(at::ScalarType t) {   // MS_DTYPE_F32 / F16 / BF16
    return t == at::kFloat ? 0 : t == at::kHalf ? 1 : t == at::kBFloat16 ? 2 : -1;
  }

  Param& at(int64_t gi, int64_t k) {
    return groups_.at(gi).params.at(k);
  }

  void push(int64_t gi, int64_t k, Param& p, at::Tensor g) {
    entries_.push_back({gi, k, std::move(g), p.seen != window_});
    p.seen = window_;
    p.queued = p.stats = true;
    queued_ += p.numel;
  }

  std::vector<Group> groups_;
  std::vector<Entry> entries_;
  int64_t queued_ = 0, window_ = 0;
};

}  // namespace

PYBIND11_MODULE(_walk, m) {
  m.doc() = "device addresses of parameter gradients / storages for the boundary tables";
  m.def("grad_pointers", &grad_pointers);
  m.def("model_pointers", &model_pointers, py::arg("params"), py::arg("device_index"),
        py::arg("out"), py::arg("numels") = py::none());
  m.def("record_streams", &record_streams);
  m.def("release_grads", &release_grads);
  m.def("same_table", &same_table);
  py::class_<BoundaryRows>(m, "BoundaryRows", py::custom_type_setup(&BoundaryRows::collectable))
      .def(py::init<py::list, const BoundaryRows::Ints&, int64_t,
                    py::array_t<int64_t, py::array::c_style>, const BoundaryRows::Ints&>())
      .def_property_readonly("table", &BoundaryRows::table)
      .def("grads", &BoundaryRows::grads)
      .def("set_grads", &BoundaryRows::set_grads)
      .def("models", &BoundaryRows::models)
      .def("set_models", &BoundaryRows::set_models)
      .def("drop", &BoundaryRows::drop);
  py::class_<GradQueue>(m, "GradQueue")
      .def(py::init<>())
      .def_readonly_static("NONE", &GradQueue::kNone)
      .def_readonly_static("SLOW", &GradQueue::kSlow)
      .def_readonly_static("AGAIN", &GradQueue::kAgain)
      .def("add_group", &GradQueue::add_group)
      .def("take", &GradQueue::take)
      .def("put", &GradQueue::put)
      .def("empty", &GradQueue::empty)
      .def("rows", &GradQueue::rows)
      .def("pointers", &GradQueue::pointers)
      .def("stale_slots", &GradQueue::stale_slots)
      .def("next_window", &GradQueue::next_window)
      .def("rebased", &GradQueue::rebased);
}

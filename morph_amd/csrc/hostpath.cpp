// The host side of an AdamW step over tensors it has stepped before.
//
// A step's work on the host is to look at every gradient (is it there, on the device, of
// the batch's type and size, contiguous), to put its address into the launch descriptors,
// and to make two launches.  In Python a step took 39 us for 6 tensors and 291 us for 326,
// beside 9 and 10.1 us of kernels; here 12 and 30 us (25 without the look at where parameters
// and moments lie).
//
// StepPlan belongs to one descriptor batch (kernels.AdamwBatch) and keeps no check from one
// step to the next: match() looks at every parameter, both its moments and its gradient again
// and says no on anything that is not exactly what the batch was built for (another parameter
// list, a parameter or a moment that lies elsewhere, a gradient missing or new, another type,
// device, size or layout, a tensor subclass, other export buffers); the caller then takes the
// Python path, which rebuilds or raises.
#include <ATen/TensorSubclassLikeUtils.h>
#include <pybind11/pybind11.h>
#include <pybind11/stl.h>
#include <torch/csrc/autograd/python_variable.h>

#include <vector>

#include "../../include/morph_optim.h"

namespace py = pybind11;

namespace {

// at::isTensorSubclassLike without its question for a dispatch mode, which match() asks once.
bool plain(const at::Tensor& t) {
  return (t.key_set() & at::kTensorSubclassLike).empty() && t.has_storage();
}

const at::Tensor* plain_tensor(PyObject* o) {
  if (o == nullptr || !THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && plain(t) ? &t : nullptr;
}

// Whether t is n contiguous elements of `type`.
bool holds(const at::Tensor& t, at::ScalarType type, int64_t n) {
  return t.numel() == n && t.scalar_type() == type && t.is_contiguous();
}

// Whether o is still the n floats at `address` that a descriptor points at.
bool still_at(PyObject* o, const void* address, int64_t n) {
  const at::Tensor* t = plain_tensor(o);
  return t != nullptr && holds(*t, at::kFloat, n) && t->const_data_ptr() == address;
}

// The same for a moment, by its address alone: another size or type there would be a view of
// the moment that the batch was built on, whose memory is as large as it was.  Looking at all
// that still_at does took 326 parameters whose tensors no cache holds 3 us longer.
bool lies_at(PyObject* o, const void* address) {
  if (o == nullptr || !THPVariable_CheckExact(o)) return false;
  const c10::TensorImpl* t = THPVariable_Unpack(o).unsafeGetTensorImpl();
  if (!t->has_storage()) return false;
  if (t->numel() == 0) return address == nullptr;
  const void* base = t->unsafe_storage().unsafeGetStorageImpl()->data();
  return static_cast<const char*>(base) + t->storage_offset() * (int64_t)sizeof(float) == address;
}

// A list's or tuple's items, borrowed; false for anything else.
struct Items {
  PyObject* seq;
  Py_ssize_t n = 0;
  explicit Items(PyObject* o) : seq(o) {
    ok = PyList_CheckExact(o) || PyTuple_CheckExact(o);
    if (ok) n = PySequence_Fast_GET_SIZE(o);
  }
  PyObject* at(Py_ssize_t i) const { return PySequence_Fast_GET_ITEM(seq, i); }
  bool ok;
};

using NonfiniteOrMulti = decltype(&morph_nonfinite_or_multi);
using NonfiniteOrClose = decltype(&morph_nonfinite_or_close);
using AdamwMultiDev = decltype(&morph_adamw_multi_dev);
using NonfiniteTable = decltype(&morph_nonfinite_table);
using AdamwTableDev = decltype(&morph_adamw_table_dev);

struct Entries {  // of the library, by address: it is loaded by the caller
  NonfiniteOrMulti nonfinite_or_multi;
  NonfiniteOrClose nonfinite_or_close;
  AdamwMultiDev adamw_multi_dev;
  NonfiniteTable nonfinite_table;
  AdamwTableDev adamw_table_dev;
};

class StepPlan {
 public:
  // params: every parameter in order; present: those the batch steps, ascending; the
  // descriptors (morph_adamw_tensor[len(present)]) and everything behind the other
  // addresses are kept alive by the batch and the optimizer.
  StepPlan(py::list params, std::vector<int64_t> present, uint64_t descriptors, int grad_dtype,
           int out_dtype, uint64_t table, uint64_t clocks, uint64_t state,
           std::vector<uint64_t> entries)
      : params_(std::move(params)),
        present_(std::move(present)),
        desc_(reinterpret_cast<morph_adamw_tensor*>(descriptors)),
        grad_dtype_(grad_dtype),
        out_dtype_(out_dtype),
        table_(reinterpret_cast<const void*>(table)),
        clocks_(reinterpret_cast<int64_t*>(clocks)),
        state_(reinterpret_cast<morph_step_state*>(state)) {
    if (entries.size() != 5) throw std::invalid_argument("five entry points expected");
    fn_.nonfinite_or_multi = reinterpret_cast<NonfiniteOrMulti>(entries[0]);
    fn_.nonfinite_or_close = reinterpret_cast<NonfiniteOrClose>(entries[1]);
    fn_.adamw_multi_dev = reinterpret_cast<AdamwMultiDev>(entries[2]);
    fn_.nonfinite_table = reinterpret_cast<NonfiniteTable>(entries[3]);
    fn_.adamw_table_dev = reinterpret_cast<AdamwTableDev>(entries[4]);
    const size_t n = present_.size();
    numels_.resize(n);
    ptrs_.resize(n);
    grads_.resize(n);
    for (size_t k = 0; k < n; ++k) {
      const int64_t i = present_[k];
      if (i < 0 || i >= (int64_t)params_.size() || (k > 0 && i <= present_[k - 1]))
        throw std::invalid_argument("present must be ascending parameter indices");
      numels_[k] = desc_[k].numel;
    }
    if (n == 0) throw std::invalid_argument("a plan steps at least one tensor");
    // Any tensor will do here, a subclass's or one under a dispatch mode too: a step that
    // cannot be taken natively is match()'s to refuse.
    PyObject* first = PyList_GET_ITEM(params_.ptr(), present_[0]);
    if (!THPVariable_Check(first)) throw std::invalid_argument("parameters must be tensors");
    device_ = THPVariable_Unpack(first).device();
    type_ = grad_dtype == MORPH_DTYPE_F16    ? at::kHalf
            : grad_dtype == MORPH_DTYPE_BF16 ? at::kBFloat16
                                             : at::kFloat;
  }

  // Whether this step's parameters, moments, gradients and export buffers are what the batch
  // was built for; if so the descriptors now hold the gradients' addresses and the plan holds
  // the gradients (until the next match).  grads: None (each parameter's .grad), or a
  // list or tuple with an entry (or None) per parameter.  state: the optimizer's, {parameter:
  // {exp_avg, exp_avg_sq, ..}} in the parameters' order.
  bool match(py::handle groups, py::handle grads, py::handle exports, py::handle state) {
    const Items gs(groups.ptr()), outs(exports.ptr());
    if (!gs.ok || !outs.ok || !PyDict_Check(state.ptr())) return false;
    if (c10::impl::dispatch_mode_enabled()) return false;
    const bool own = grads.is_none();
    const Items given(own ? groups.ptr() : grads.ptr());
    const Py_ssize_t total = PyList_GET_SIZE(params_.ptr());
    if (!given.ok || (!own && given.n != total)) return false;
    if (outs.n != 0 && outs.n != total) return false;
    Py_ssize_t i = 0, in_state = 0;
    size_t k = 0;
    for (Py_ssize_t g = 0; g < gs.n; ++g) {
      PyObject* group = gs.at(g);
      if (!PyDict_CheckExact(group)) return false;
      static PyObject* key = PyUnicode_InternFromString("params");
      PyObject* list = PyDict_GetItem(group, key);  // borrowed
      if (list == nullptr || !PyList_CheckExact(list)) return false;
      for (Py_ssize_t j = 0; j < PyList_GET_SIZE(list); ++j, ++i) {
        PyObject* po = PyList_GET_ITEM(list, j);
        if (i >= total || po != PyList_GET_ITEM(params_.ptr(), i)) return false;
        PyObject *owner = nullptr, *moments = nullptr;  // borrowed
        if (!PyDict_Next(state.ptr(), &in_state, &owner, &moments) || owner != po) return false;
        const bool want = k < present_.size() && present_[k] == i;
        const at::Tensor* grad = nullptr;
        if (own) {
          const at::Tensor* p = plain_tensor(po);
          if (p == nullptr) return false;
          grad = &p->unsafeGetTensorImpl()->grad();
          if (grad->defined() != want) return false;
          if (want && !plain(*grad)) return false;
        } else {
          PyObject* go = given.at(i);
          if ((go == Py_None) == want) return false;
          if (want) grad = plain_tensor(go);
          if (want && grad == nullptr) return false;
        }
        if (!want) continue;
        static PyObject* const first = PyUnicode_InternFromString("exp_avg");
        static PyObject* const second = PyUnicode_InternFromString("exp_avg_sq");
        const morph_adamw_tensor& d = desc_[k];
        if (!PyDict_Check(moments) || !still_at(po, d.param, d.numel) ||
            !lies_at(PyDict_GetItemWithError(moments, first), d.exp_avg) ||
            !lies_at(PyDict_GetItemWithError(moments, second), d.exp_avg_sq))
          return false;
        if (grad->layout() != at::kStrided || grad->device() != device_ ||
            !holds(*grad, type_, d.numel))
          return false;
        void* out = nullptr;
        if (outs.n != 0) {
          const at::Tensor* o = plain_tensor(outs.at(i));
          if (o == nullptr) return false;
          out = o->data_ptr();
        }
        if (out != d.out) return false;
        ptrs_[k] = grad->const_data_ptr();
        grads_[k] = grad;
        ++k;
      }
    }
    if (i != total || k != present_.size()) return false;
    std::vector<at::Tensor> dropped;  // freed when all is done: that can run any code
    held_.resize(present_.size());
    for (k = 0; k < present_.size(); ++k) {
      desc_[k].grad = ptrs_[k];
      if (held_[k].is_same(*grads_[k])) continue;
      dropped.push_back(std::move(held_[k]));
      held_[k] = *grads_[k];
    }
    return true;
  }

  // Lets go of the last match's gradients.
  void release() {
    std::vector<at::Tensor> dropped;
    dropped.swap(held_);
  }

  // The step's launches on `stream` after match(): the detector (unless `checked`; with the
  // previous step's close when prev_list is not 0), then AdamW.  The status of the first
  // that failed, or 0.  The GIL is released meanwhile, as around every other call of the
  // library: a launch waits when the queue is full.
  int launch(uint64_t stream, int slot, bool checked, uint64_t prev_list, int n_prev,
             uint64_t hps, uint64_t scheds, int n_hp) {
    const py::gil_scoped_release nogil;
    void* s = reinterpret_cast<void*>(stream);
    const int32_t* prev = reinterpret_cast<const int32_t*>(prev_list);
    const int count = (int)present_.size();
    int rc = MORPH_OK;
    closed_ = false;
    if (!checked) {
      if (table_ != nullptr)
        rc = fn_.nonfinite_table(table_, desc_, count, grad_dtype_, state_, slot, clocks_, prev,
                                 n_prev, prev != nullptr, s);
      else if (prev != nullptr)
        rc = fn_.nonfinite_or_close(ptrs_.data(), numels_.data(), count, grad_dtype_, state_, slot,
                                    clocks_, prev, n_prev, s);
      else
        rc = fn_.nonfinite_or_multi(ptrs_.data(), numels_.data(), count, grad_dtype_,
                                    &state_->found_inf[slot], s);
      if (rc != MORPH_OK) return rc;
    }
    closed_ = true;
    const morph_adamw_hp* h = reinterpret_cast<const morph_adamw_hp*>(hps);
    const morph_adamw_sched* c = reinterpret_cast<const morph_adamw_sched*>(scheds);
    if (table_ != nullptr)
      return fn_.adamw_table_dev(table_, desc_, count, grad_dtype_, out_dtype_, h, c, n_hp, clocks_,
                                 state_, slot, nullptr, nullptr, s);
    return fn_.adamw_multi_dev(desc_, count, grad_dtype_, out_dtype_, h, c, n_hp, clocks_, state_,
                               slot, nullptr, nullptr, s);
  }

  // Whether the last launch() got past the detector, which carries the previous step's close.
  bool closed() const { return closed_; }

 private:
  py::list params_;
  std::vector<int64_t> present_;
  morph_adamw_tensor* desc_;
  int grad_dtype_, out_dtype_;
  const void* table_;
  int64_t* clocks_;
  morph_step_state* state_;
  Entries fn_;
  std::vector<int64_t> numels_;
  std::vector<const void*> ptrs_;
  std::vector<const at::Tensor*> grads_;  // during a match
  std::vector<at::Tensor> held_;
  bool closed_ = false;
  at::Device device_{at::kCPU};
  at::ScalarType type_;
};

// Where each tensor of the list lies, its size and whether it is contiguous, for a key.
py::bytes places(const py::list& tensors) {
  std::vector<int64_t> out;
  out.reserve(2 * tensors.size());
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(tensors.ptr()); ++i) {
    PyObject* o = PyList_GET_ITEM(tensors.ptr(), i);
    if (!THPVariable_Check(o)) throw py::type_error("places() takes tensors");
    const at::Tensor t = THPVariable_Unpack(o);
    out.push_back(reinterpret_cast<int64_t>(t.const_data_ptr()));
    out.push_back(t.is_contiguous() ? t.numel() : ~t.numel());
  }
  return py::bytes(reinterpret_cast<const char*>(out.data()), out.size() * sizeof(int64_t));
}

}  // namespace

PYBIND11_MODULE(_hostpath, m) {
  m.def("places", &places);
  py::class_<StepPlan>(m, "StepPlan")
      .def(py::init<py::list, std::vector<int64_t>, uint64_t, int, int, uint64_t, uint64_t, uint64_t,
                    std::vector<uint64_t>>())
      .def("match", &StepPlan::match)
      .def("release", &StepPlan::release)
      .def("closed", &StepPlan::closed)
      .def("launch", &StepPlan::launch);
}

// A repeated call of a `@kernel` function on torch tensors, in native code.
//
// The first call with given arguments goes through dvm_amd/jit.py: shape inference, code generation, binding, launches. When a
// second one like it follows, what came out of it (the arguments' types, shapes and strides, the numbers among them, the
// outputs' shapes, the size of the workspace) is recorded here as the kernel's plan, and while the arguments of a call match it,
// the call is: check them, allocate the outputs and the workspace from torch's caching allocator, write the addresses into the
// compiled programs, launch. No address is kept from one call for the next, and whatever else changes the kernel
// (dvm_rt_plan_stamp) makes the plan stale; any mismatch hands the call back to jit.py, which raises what there is to raise.
// Measured on an MI355X's host, us a call from Python / from the plan: two fp32 tensors added 12.9 / 4.4, an Adam step on 64 x 64
// (four tensors, two numbers, three results) 24.3 / 6.0; of that the launch itself takes 3.5.
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <pybind11/gil.h>

#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <vector>

namespace {

typedef int (*RebindRunFn)(void *rt, uint64_t stamp, void *const *ios, void *const *ptrs, size_t n, void *workspace, void *stream);
typedef uint64_t (*StampFn)(void *rt);
typedef const char *(*LastErrorFn)();

struct TensorSpec {
  at::ScalarType type;
  std::vector<int64_t> sizes, strides;
};

struct ArgSpec {
  bool tensor = false;
  TensorSpec spec;           // a tensor
  bool is_float = false;     // a number: its value, bit for bit
  double f = 0.0;
  int64_t i = 0;
};

struct Recorded {  // what a call is compared with and made from; never changed once it stands
  std::vector<ArgSpec> args;
  std::vector<TensorSpec> outs;
  std::vector<void *> ios;  // the loads behind the tensor arguments, then the stores
  bool many = false;
  uint64_t stamp = 0;
  int64_t ws_bytes = 0;
  c10::DeviceIndex device = -1;
};

struct Plan {
  PyObject_HEAD
  RebindRunFn rebind_run;
  StampFn stamp_of;
  LastErrorFn last_error;
  void *rt;
  std::shared_ptr<const Recorded> *now;  // (empty: nothing recorded, or stale)
  std::vector<ArgSpec> *seen;            // arguments of the last call made from Python (empty: none that can be recorded)
  std::recursive_mutex *launch;          // one thread at a time binds, generates code and launches, from here or from Python
};

bool IsPlainTensor(PyObject *o) { return THPVariable_CheckExact(o); }

bool ReadNumber(PyObject *o, ArgSpec *a) {
  if (PyFloat_CheckExact(o)) {
    a->is_float = true;
    a->f = PyFloat_AS_DOUBLE(o);
    return true;
  }
  if (PyLong_CheckExact(o)) {
    int overflow = 0;
    a->i = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow == 0;
  }
  return false;
}

bool SameNumber(const ArgSpec &a, const ArgSpec &b) {
  return a.is_float == b.is_float && (a.is_float ? std::memcmp(&a.f, &b.f, sizeof(double)) == 0 : a.i == b.i);
}

// strided memory of the plan's device behind an unwrapped tensor, read as it lies
bool Readable(const at::Tensor &t, c10::DeviceIndex device) {
  return t.is_cuda() && t.device().index() == device && t.layout() == at::kStrided && t.has_storage() && !t.is_neg() && !t.is_conj();
}

// Plan(rebind_run, stamp_of, last_error, rt): addresses of the runner's functions and of the runner
PyObject *PlanNew(PyTypeObject *type, PyObject *args, PyObject *) {
  unsigned long long rebind_run = 0, stamp_of = 0, last_error = 0, rt = 0;
  if (!PyArg_ParseTuple(args, "KKKK", &rebind_run, &stamp_of, &last_error, &rt)) return nullptr;
  Plan *p = reinterpret_cast<Plan *>(type->tp_alloc(type, 0));
  if (p == nullptr) return nullptr;
  p->rebind_run = reinterpret_cast<RebindRunFn>(rebind_run);
  p->stamp_of = reinterpret_cast<StampFn>(stamp_of);
  p->last_error = reinterpret_cast<LastErrorFn>(last_error);
  p->rt = reinterpret_cast<void *>(rt);
  p->now = new std::shared_ptr<const Recorded>();
  p->seen = new std::vector<ArgSpec>();
  p->launch = new std::recursive_mutex();
  return reinterpret_cast<PyObject *>(p);
}

void PlanDealloc(PyObject *self) {
  Plan *p = reinterpret_cast<Plan *>(self);
  delete p->now;
  delete p->seen;
  delete p->launch;
  Py_TYPE(self)->tp_free(self);
}

// Whether the arguments of a call are those of `specs`; ptrs: where the tensors among them lie.
bool Matches(const std::vector<ArgSpec> &specs, c10::DeviceIndex device, PyObject *args, void **ptrs) {
  const size_t n = specs.size();
  if (static_cast<size_t>(PyTuple_GET_SIZE(args)) != n) return false;
  for (size_t i = 0; i < n; ++i) {
    PyObject *o = PyTuple_GET_ITEM(args, static_cast<Py_ssize_t>(i));
    const ArgSpec &a = specs[i];
    if (!a.tensor) {
      ArgSpec now;
      if (!ReadNumber(o, &now) || !SameNumber(a, now)) return false;
      continue;
    }
    if (!IsPlainTensor(o)) return false;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!Readable(t, device) || t.scalar_type() != a.spec.type || t.sizes() != at::IntArrayRef(a.spec.sizes) ||
        t.strides() != at::IntArrayRef(a.spec.strides)) return false;
    if (ptrs != nullptr) *ptrs++ = t.data_ptr();
  }
  return true;
}

c10::DeviceIndex DeviceOf(PyObject *args) {
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(args); ++i) {
    PyObject *o = PyTuple_GET_ITEM(args, i);
    if (!IsPlainTensor(o)) continue;
    const at::Tensor &t = THPVariable_Unpack(o);
    return t.is_cuda() ? t.device().index() : static_cast<c10::DeviceIndex>(-1);
  }
  return -1;
}

// repeats(args): whether the call from Python that has just been made was like the one before it. Only then is a plan worth its
// recording: where a number or a shape is another one at every call, what is added to the call is this comparison.
PyObject *PlanRepeats(PyObject *self, PyObject *args) {
  HANDLE_TH_ERRORS
  Plan *p = reinterpret_cast<Plan *>(self);
  if (!PyTuple_Check(args)) {
    PyErr_SetString(PyExc_TypeError, "repeats(args)");
    return nullptr;
  }
  const c10::DeviceIndex device = DeviceOf(args);
  if (!p->seen->empty() && device >= 0 && Matches(*p->seen, device, args, nullptr)) Py_RETURN_TRUE;
  std::vector<ArgSpec> &seen = *p->seen;
  const size_t n = static_cast<size_t>(PyTuple_GET_SIZE(args));
  seen.resize(device >= 0 ? n : 0);
  for (size_t i = 0; i < seen.size(); ++i) {
    PyObject *o = PyTuple_GET_ITEM(args, static_cast<Py_ssize_t>(i));
    ArgSpec &a = seen[i];
    a.tensor = IsPlainTensor(o);
    if (a.tensor) {
      const at::Tensor &t = THPVariable_Unpack(o);
      if (Readable(t, device)) {
        a.spec.type = t.scalar_type();
        a.spec.sizes.assign(t.sizes().begin(), t.sizes().end());
        a.spec.strides.assign(t.strides().begin(), t.strides().end());
        continue;
      }
    } else {
      a.is_float = false;
      if (ReadNumber(o, &a)) continue;
    }
    seen.clear();
    break;
  }
  Py_RETURN_FALSE;
  END_HANDLE_TH_ERRORS
}

// record(args, load handles, outputs, store handles, many, workspace bytes): the call that `repeats` has just been asked about
// becomes the plan, unless another thread has asked about another one meanwhile. False when calls like it cannot go this way.
PyObject *PlanRecord(PyObject *self, PyObject *pyargs) {
  HANDLE_TH_ERRORS
  Plan *p = reinterpret_cast<Plan *>(self);
  PyObject *args, *loads, *outs, *stores;
  int many = 0;
  long long ws_bytes = 0;
  if (!PyArg_ParseTuple(pyargs, "O!O!O!O!pL", &PyTuple_Type, &args, &PyList_Type, &loads, &PyList_Type, &outs, &PyList_Type, &stores, &many, &ws_bytes)) return nullptr;
  p->now->reset();
  if (!Matches(*p->seen, DeviceOf(args), args, nullptr)) Py_RETURN_TRUE;
  auto r = std::make_shared<Recorded>();
  r->args = *p->seen;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(outs); ++i) {
    PyObject *o = PyList_GET_ITEM(outs, i);
    if (!IsPlainTensor(o)) Py_RETURN_FALSE;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!t.is_cuda()) Py_RETURN_FALSE;
    if (r->device < 0) r->device = t.device().index();
    if (!Readable(t, r->device) || !t.is_contiguous()) Py_RETURN_FALSE;
    r->outs.push_back({t.scalar_type(), t.sizes().vec(), {}});
  }
  for (PyObject *list : {loads, stores}) {
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list); ++i) {
      void *h = PyLong_AsVoidPtr(PyList_GET_ITEM(list, i));
      if (h == nullptr) return PyErr_Occurred() ? nullptr : (Py_INCREF(Py_False), Py_False);
      r->ios.push_back(h);
    }
  }
  size_t tensors = r->outs.size();
  for (const ArgSpec &a : r->args) tensors += a.tensor;
  if (tensors != r->ios.size() || tensors > 64 || r->device < 0) Py_RETURN_FALSE;
  r->many = many != 0;
  r->ws_bytes = ws_bytes;
  r->stamp = p->stamp_of(p->rt);
  *p->now = r;
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// call(kernel, args, stream_of): the outputs, or None when the call is not the recorded one. kernel._alive holds the call's
// tensors until the next one: the launches may still be running.
PyObject *PlanCall(PyObject *self, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  Plan *p = reinterpret_cast<Plan *>(self);
  if (argc != 3 || !PyTuple_Check(argv[1])) {
    PyErr_SetString(PyExc_TypeError, "call(kernel, args, stream_of)");
    return nullptr;
  }
  PyObject *kernel = argv[0], *args = argv[1];
  const std::shared_ptr<const Recorded> r = *p->now;  // (another thread may record a plan while this one is at work)
  void *ptrs[64];
  if (!r || !Matches(r->args, r->device, args, ptrs)) Py_RETURN_NONE;
  if (p->stamp_of(p->rt) != r->stamp) {
    p->now->reset();
    Py_RETURN_NONE;
  }
  PyObject *index = PyLong_FromLong(r->device);
  if (index == nullptr) return nullptr;
  PyObject *stream = PyObject_CallOneArg(argv[2], index);
  Py_DECREF(index);
  if (stream == nullptr) return nullptr;
  void *raw = PyLong_AsVoidPtr(stream);
  Py_DECREF(stream);
  if (raw == nullptr && PyErr_Occurred()) return nullptr;
  std::vector<at::Tensor> made;
  made.reserve(r->outs.size() + 1);
  int rc = 1;
  {
    // Other threads run meanwhile: an allocation may have to free memory and wait for the GPU, a launch waits while the
    // stream's queue is full.
    pybind11::gil_scoped_release no_gil;
    const c10::Device device(c10::kCUDA, r->device);
    size_t np = r->ios.size() - r->outs.size();
    void *workspace = nullptr;
    bool memory = true;  // (false: a mode makes something else of an allocation)
    for (const TensorSpec &s : r->outs) {
      made.push_back(at::empty(s.sizes, at::TensorOptions().dtype(s.type).device(device)));
      memory = memory && made.back().has_storage();
      if (memory) ptrs[np++] = made.back().data_ptr();
    }
    if (memory && r->ws_bytes > 0) {
      made.push_back(at::empty({r->ws_bytes}, at::TensorOptions().dtype(at::kByte).device(device)));
      memory = made.back().has_storage();
      if (memory) workspace = made.back().data_ptr();
    }
    if (memory) {
      const std::lock_guard<std::recursive_mutex> one(*p->launch);
      rc = p->rebind_run(p->rt, r->stamp, r->ios.data(), ptrs, np, workspace, raw);
    }
  }
  if (rc != 0) {
    p->now->reset();
    if (rc > 0) Py_RETURN_NONE;
    PyErr_SetString(PyExc_RuntimeError, p->last_error());
    return nullptr;
  }
  const Py_ssize_t n_out = static_cast<Py_ssize_t>(r->outs.size()), n_made = static_cast<Py_ssize_t>(made.size());
  PyObject *alive = PyList_New(static_cast<Py_ssize_t>(1) + n_made);
  if (alive == nullptr) return nullptr;
  Py_INCREF(args);
  PyList_SET_ITEM(alive, 0, args);
  for (Py_ssize_t i = 0; i < n_made; ++i) PyList_SET_ITEM(alive, 1 + i, THPVariable_Wrap(made[static_cast<size_t>(i)]));
  PyObject *result;
  if (r->many) {
    result = PyList_New(n_out);
    for (Py_ssize_t i = 0; result != nullptr && i < n_out; ++i) {
      PyObject *o = PyList_GET_ITEM(alive, 1 + i);
      Py_INCREF(o);
      PyList_SET_ITEM(result, i, o);
    }
  } else {
    result = PyList_GET_ITEM(alive, 1);
    Py_INCREF(result);
  }
  const int set = PyObject_SetAttrString(kernel, "_alive", alive);
  Py_DECREF(alive);
  if (set != 0) Py_CLEAR(result);
  return result;
  END_HANDLE_TH_ERRORS
}

// hold() .. release(): a call from Python, which takes several steps, on a kernel that others may call from this plan
PyObject *PlanHold(PyObject *self, PyObject *) {
  HANDLE_TH_ERRORS
  pybind11::gil_scoped_release no_gil;
  reinterpret_cast<Plan *>(self)->launch->lock();
  END_HANDLE_TH_ERRORS_RET(nullptr)
  Py_RETURN_NONE;
}
PyObject *PlanRelease(PyObject *self, PyObject *) {
  reinterpret_cast<Plan *>(self)->launch->unlock();
  Py_RETURN_NONE;
}

PyMethodDef plan_methods[] = {
    {"hold", PlanHold, METH_NOARGS, nullptr},
    {"release", PlanRelease, METH_NOARGS, nullptr},
    {"repeats", PlanRepeats, METH_O, nullptr},
    {"record", PlanRecord, METH_VARARGS, nullptr},
    {"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(PlanCall)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyTypeObject plan_type = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_torch_call", nullptr, -1, nullptr, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC __attribute__((visibility("default"))) PyInit__torch_call(void) {
  plan_type.tp_name = "dvm_amd._torch_call.Plan";
  plan_type.tp_basicsize = sizeof(Plan);
  plan_type.tp_flags = Py_TPFLAGS_DEFAULT;
  plan_type.tp_new = PlanNew;
  plan_type.tp_dealloc = PlanDealloc;
  plan_type.tp_methods = plan_methods;
  if (PyType_Ready(&plan_type) < 0) return nullptr;
  PyObject *m = PyModule_Create(&module_def);
  if (m == nullptr) return nullptr;
  if (PyModule_AddStringConstant(m, "built_for", DVM_TORCH_CALL_TAG) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  Py_INCREF(&plan_type);
  if (PyModule_AddObject(m, "Plan", reinterpret_cast<PyObject *>(&plan_type)) < 0) {
    Py_DECREF(&plan_type);
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}

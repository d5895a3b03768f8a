// A repeated call of a `@kernel` function on torch tensors, in native code.
//
// The first call with given shapes goes through dvm_amd/jit.py: shape inference, code generation, binding, launches. What
// came out of it (the arguments' types, shapes and strides, the outputs' shapes, the size of the workspace) is recorded here
// as the kernel's plan, and while the arguments of a call match it, the call is: check them, allocate the outputs and the
// workspace from torch's caching allocator, write the addresses into the compiled programs, launch. No address is kept from
// one call for the next, and whatever else changes the kernel (dvm_rt_plan_stamp) makes the plan stale; any mismatch hands
// the call back to jit.py, which raises what there is to raise. Measured on an MI355X's host, us a call: two fp32 tensors
// added 12.8 -> 5.1, a row block's RMSNorm 15.8 -> 4.9; of that the launch itself takes 3.5.
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstring>
#include <string>
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

struct Plan {
  PyObject_HEAD
  RebindRunFn rebind_run;
  StampFn stamp_of;
  LastErrorFn last_error;
  void *rt;
  std::vector<void *> *ios;  // the loads behind the tensor arguments, then the stores
  std::vector<ArgSpec> *args;
  std::vector<TensorSpec> *outs;
  bool valid, many;
  uint64_t stamp;
  int64_t ws_bytes;
  c10::DeviceIndex device;
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
  p->ios = new std::vector<void *>();
  p->args = new std::vector<ArgSpec>();
  p->outs = new std::vector<TensorSpec>();
  p->valid = false;
  return reinterpret_cast<PyObject *>(p);
}

void PlanDealloc(PyObject *self) {
  Plan *p = reinterpret_cast<Plan *>(self);
  delete p->ios;
  delete p->args;
  delete p->outs;
  Py_TYPE(self)->tp_free(self);
}

// record(args, load handles, outputs, store handles, many, workspace bytes): what the call that has just been made was.
// False when calls like it cannot go this way.
PyObject *PlanRecord(PyObject *self, PyObject *pyargs) {
  HANDLE_TH_ERRORS
  Plan *p = reinterpret_cast<Plan *>(self);
  PyObject *args, *loads, *outs, *stores;
  int many = 0;
  long long ws_bytes = 0;
  if (!PyArg_ParseTuple(pyargs, "O!O!O!O!pL", &PyTuple_Type, &args, &PyList_Type, &loads, &PyList_Type, &outs, &PyList_Type, &stores, &many, &ws_bytes)) return nullptr;
  p->valid = false;
  p->ios->clear();
  p->args->clear();
  p->outs->clear();
  c10::DeviceIndex device = -1;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(args); ++i) {
    PyObject *o = PyTuple_GET_ITEM(args, i);
    ArgSpec a;
    if (IsPlainTensor(o)) {
      const at::Tensor &t = THPVariable_Unpack(o);
      if (!t.is_cuda()) Py_RETURN_FALSE;
      if (device < 0) device = t.device().index();
      if (!Readable(t, device)) Py_RETURN_FALSE;
      a.tensor = true;
      a.spec.type = t.scalar_type();
      a.spec.sizes = t.sizes().vec();
      a.spec.strides = t.strides().vec();
    } else if (!ReadNumber(o, &a)) {
      Py_RETURN_FALSE;
    }
    p->args->push_back(std::move(a));
  }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(outs); ++i) {
    PyObject *o = PyList_GET_ITEM(outs, i);
    if (!IsPlainTensor(o)) Py_RETURN_FALSE;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!Readable(t, device) || !t.is_contiguous()) Py_RETURN_FALSE;
    p->outs->push_back({t.scalar_type(), t.sizes().vec(), {}});
  }
  for (PyObject *list : {loads, stores}) {
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list); ++i) {
      void *h = PyLong_AsVoidPtr(PyList_GET_ITEM(list, i));
      if (h == nullptr) return PyErr_Occurred() ? nullptr : (Py_INCREF(Py_False), Py_False);
      p->ios->push_back(h);
    }
  }
  size_t tensors = p->outs->size();
  for (const ArgSpec &a : *p->args) tensors += a.tensor;
  if (tensors != p->ios->size() || device < 0) Py_RETURN_FALSE;
  p->device = device;
  p->many = many != 0;
  p->ws_bytes = ws_bytes;
  p->stamp = p->stamp_of(p->rt);
  p->valid = true;
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
  const size_t n = p->args->size();
  if (!p->valid || static_cast<size_t>(PyTuple_GET_SIZE(args)) != n) Py_RETURN_NONE;
  void *ptrs[64];
  size_t np = 0;
  if (p->ios->size() > 64) Py_RETURN_NONE;
  for (size_t i = 0; i < n; ++i) {
    PyObject *o = PyTuple_GET_ITEM(args, static_cast<Py_ssize_t>(i));
    const ArgSpec &a = (*p->args)[i];
    if (!a.tensor) {
      ArgSpec now;
      if (!ReadNumber(o, &now) || !SameNumber(a, now)) Py_RETURN_NONE;
      continue;
    }
    if (!IsPlainTensor(o)) Py_RETURN_NONE;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!Readable(t, p->device) || t.scalar_type() != a.spec.type || t.sizes() != at::IntArrayRef(a.spec.sizes) ||
        t.strides() != at::IntArrayRef(a.spec.strides)) Py_RETURN_NONE;
    ptrs[np++] = t.data_ptr();
  }
  if (p->stamp_of(p->rt) != p->stamp) {
    p->valid = false;
    Py_RETURN_NONE;
  }
  const c10::Device device(c10::kCUDA, p->device);
  std::vector<at::Tensor> made;
  made.reserve(p->outs->size() + 1);
  for (const TensorSpec &s : *p->outs) {
    made.push_back(at::empty(s.sizes, at::TensorOptions().dtype(s.type).device(device)));
    if (!made.back().has_storage()) Py_RETURN_NONE;  // (a mode that makes something else of an allocation)
    ptrs[np++] = made.back().data_ptr();
  }
  void *workspace = nullptr;
  if (p->ws_bytes > 0) {
    made.push_back(at::empty({p->ws_bytes}, at::TensorOptions().dtype(at::kByte).device(device)));
    if (!made.back().has_storage()) Py_RETURN_NONE;
    workspace = made.back().data_ptr();
  }
  PyObject *index = PyLong_FromLong(p->device);
  if (index == nullptr) return nullptr;
  PyObject *stream = PyObject_CallOneArg(argv[2], index);
  Py_DECREF(index);
  if (stream == nullptr) return nullptr;
  void *raw = PyLong_AsVoidPtr(stream);
  Py_DECREF(stream);
  if (raw == nullptr && PyErr_Occurred()) return nullptr;
  const int rc = p->rebind_run(p->rt, p->stamp, p->ios->data(), ptrs, np, workspace, raw);
  if (rc != 0) {
    p->valid = false;
    if (rc > 0) Py_RETURN_NONE;
    PyErr_SetString(PyExc_RuntimeError, p->last_error());
    return nullptr;
  }
  const Py_ssize_t n_out = static_cast<Py_ssize_t>(p->outs->size()), n_made = static_cast<Py_ssize_t>(made.size());
  PyObject *alive = PyList_New(static_cast<Py_ssize_t>(1) + n_made);
  if (alive == nullptr) return nullptr;
  Py_INCREF(args);
  PyList_SET_ITEM(alive, 0, args);
  for (Py_ssize_t i = 0; i < n_made; ++i) PyList_SET_ITEM(alive, 1 + i, THPVariable_Wrap(made[static_cast<size_t>(i)]));
  PyObject *result;
  if (p->many) {
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

PyMethodDef plan_methods[] = {
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

// fastcall.cpp — the repeated call of a fused-group launcher, in native code.
//
// HipKernelLauncher (fuseml_amd/launcher.py) builds a plan per input signature
// (shapes, strides, dtypes) and from then on a call only checks the signature,
// allocates outputs, writes pointers into the plan's descriptor and calls the C
// ABI.  In Python that took 6-7 us of host time per launch, more than the kernel
// of a decode step (16x4096x1024: 5.5 us); here it takes about 1.  Every call that
// is not of a known signature, or whose tensors are not plain GPU tensors the
// plan can take as they are, is declined and runs through the Python path.
//
// The descriptor is copied to the stack per call, so threads may share a launcher.
#define PY_SSIZE_T_CLEAN
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>

#include <cstdlib>
#include <cstring>
#include <utility>
#include <vector>

#include "fuseml_hip.h"

namespace {

using Entry = int (*)(const fuseml_gemm_desc*, void*);

constexpr int kMaxDim = 4;
constexpr size_t kMaxPlans = 64;  // per launcher; more signatures stay in Python

struct Signature {
  int dim;
  int64_t sizes[kMaxDim], strides[kMaxDim];
  at::ScalarType dtype;

  bool operator==(const Signature& o) const {
    return dim == o.dim && dtype == o.dtype && !std::memcmp(sizes, o.sizes, sizeof(int64_t) * dim) &&
           !std::memcmp(strides, o.strides, sizeof(int64_t) * dim);
  }
};

struct Plan {
  std::vector<Signature> signature;               // one per used input
  fuseml_gemm_desc desc;
  Entry entry;
  int left, right;                                // input index of the GEMM operands
  std::vector<std::pair<int, int>> operands;      // (operand slot, input index)
  bool tile;
  at::ScalarType tile_dtype;
  std::vector<at::ScalarType> extras;
  std::vector<int> reductions;                    // slots of reduce_out
  std::vector<std::pair<char, int>> outputs;      // 't', ('r', reduction), ('e', extra)
};

struct Launcher {
  PyObject_HEAD
  int n_inputs;
  bool guarded;                // an eager fallback is bound: the forced-failure switch applies
  long long count;
  std::vector<int>* used;      // input indices a launch reads
  std::vector<Plan*>* plans;   // the last one that matched first
};

PyObject* g_raw_stream = nullptr;  // torch._C._cuda_getCurrentRawStream

bool plain(PyObject* o) {
  if (!THPVariable_CheckTypeExact(Py_TYPE(o))) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                         c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                         c10::DispatchKey::Negative, c10::DispatchKey::Conjugate,
                                         c10::DispatchKey::ZeroTensor});
  return t.is_cuda() && t.layout() == at::kStrided && t.has_storage() && !t.key_set().has_any(wrapped) &&
         t.dim() <= kMaxDim;
}

Signature signature_of(const at::Tensor& t) {
  Signature s{};
  s.dim = (int)t.dim();
  s.dtype = t.scalar_type();
  for (int i = 0; i < s.dim; ++i) {
    s.sizes[i] = t.sizes()[i];
    s.strides[i] = t.strides()[i];
  }
  return s;
}

bool matches(const Signature& s, const at::Tensor& t) {
  if (t.dim() != s.dim || t.scalar_type() != s.dtype) return false;
  const auto sizes = t.sizes(), strides = t.strides();
  for (int i = 0; i < s.dim; ++i)
    if (sizes[i] != s.sizes[i] || strides[i] != s.strides[i]) return false;
  return true;
}

PyObject* declined() { Py_RETURN_NONE; }

// call(inputs): the outputs, an int error code of the C ABI, or None where the
// Python path has to serve the call.
PyObject* launcher_call(PyObject* self_, PyObject* inputs) {
  HANDLE_TH_ERRORS
  Launcher* self = reinterpret_cast<Launcher*>(self_);
  if (self->plans->empty() || !PyTuple_CheckExact(inputs) || PyTuple_GET_SIZE(inputs) != self->n_inputs)
    return declined();
  if (self->guarded) {
    const char* forced = std::getenv("FUSEML_HIP_FORCE_FAIL");
    if (forced != nullptr && *forced != '\0' && std::strcmp(forced, "0") != 0) return declined();
  }
  const std::vector<int>& used = *self->used;
  const at::Tensor* tensors[FUSEML_MAX_OPERANDS + 2];
  c10::DeviceIndex device = -1;
  for (size_t i = 0; i < used.size(); ++i) {
    PyObject* o = PyTuple_GET_ITEM(inputs, used[i]);
    if (!plain(o)) return declined();
    tensors[i] = &THPVariable_Unpack(o);
    const c10::DeviceIndex d = tensors[i]->device().index();
    if (i > 0 && d != device) return declined();
    device = d;
  }
  std::vector<Plan*>& plans = *self->plans;
  size_t at = 0;
  for (; at < plans.size(); ++at) {
    bool same = true;
    for (size_t i = 0; same && i < used.size(); ++i) same = matches(plans[at]->signature[i], *tensors[i]);
    if (same) break;
  }
  if (at == plans.size()) return declined();
  if (at != 0) std::swap(plans[0], plans[at]);
  const Plan& p = *plans[0];

  const at::Tensor& a = THPVariable_Unpack(PyTuple_GET_ITEM(inputs, p.left));
  const at::Tensor& b = THPVariable_Unpack(PyTuple_GET_ITEM(inputs, p.right));
  const uintptr_t pa = (uintptr_t)a.const_data_ptr(), pb = (uintptr_t)b.const_data_ptr();
  if ((pa | pb) % 16 != 0) return declined();

  fuseml_gemm_desc d = p.desc;
  d.a = (const void*)pa;
  d.b = (const void*)pb;
  for (const auto& [slot, index] : p.operands)
    d.operands[slot].ptr = THPVariable_Unpack(PyTuple_GET_ITEM(inputs, index)).const_data_ptr();
  const auto options = at::TensorOptions().device(a.device());
  at::Tensor tile, extras[FUSEML_MAX_EXTRA_OUT], reds[3];
  d.out.ptr = nullptr;
  if (p.tile) {
    tile = at::empty({d.M, d.N}, options.dtype(p.tile_dtype));
    d.out.ptr = tile.data_ptr();
  }
  for (size_t i = 0; i < p.extras.size(); ++i) {
    extras[i] = at::empty({d.M, d.N}, options.dtype(p.extras[i]));
    d.extra[i].ptr = extras[i].data_ptr();
  }
  for (size_t i = 0; i < p.reductions.size(); ++i) {
    reds[i] = at::empty({d.reduce_axis == 1 ? d.M : d.N}, options.dtype(at::kFloat));
    d.reduce_out[p.reductions[i]] = reds[i].data_ptr<float>();
  }

  PyObject* index = PyLong_FromLong(device);
  if (index == nullptr) return nullptr;
  PyObject* handle = PyObject_CallOneArg(g_raw_stream, index);
  Py_DECREF(index);
  if (handle == nullptr) return nullptr;
  void* stream = PyLong_AsVoidPtr(handle);
  Py_DECREF(handle);
  if (stream == nullptr && PyErr_Occurred()) return nullptr;

  // Another thread may add or reorder plans meanwhile; a plan itself stays until
  // the launcher goes, which this call's caller holds.
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = p.entry(&d, stream);
  Py_END_ALLOW_THREADS
  if (rc != FUSEML_OK) return PyLong_FromLong(rc);
  self->count += 1;

  auto wrap = [&](const std::pair<char, int>& o) {
    return THPVariable_Wrap(o.first == 't' ? tile : o.first == 'r' ? reds[o.second] : extras[o.second]);
  };
  const size_t n_out = p.outputs.size();
  if (n_out == 1) return wrap(p.outputs[0]);
  PyObject* result = PyTuple_New((Py_ssize_t)n_out);
  if (result == nullptr) return nullptr;
  for (size_t i = 0; i < n_out; ++i) {
    PyObject* o = wrap(p.outputs[i]);
    if (o == nullptr) {
      Py_DECREF(result);
      return nullptr;
    }
    PyTuple_SET_ITEM(result, (Py_ssize_t)i, o);
  }
  return result;
  END_HANDLE_TH_ERRORS
}

// add(inputs, desc, entry, left, right, operands, tile, extras, reductions, outputs):
// a plan for the signature of `inputs`.  `desc`: the descriptor (a buffer), `entry`:
// the C function's address, `tile`: the output's dtype or None, `extras`: dtypes,
// the rest as in Plan.  Whether the plan was taken.
PyObject* launcher_add(PyObject* self_, PyObject* args) {
  HANDLE_TH_ERRORS
  Launcher* self = reinterpret_cast<Launcher*>(self_);
  PyObject *inputs, *operands, *tile, *extras, *reductions, *outputs;
  Py_buffer desc;
  unsigned long long entry;
  int left, right;
  if (!PyArg_ParseTuple(args, "O!y*KiiO!OO!O!O!", &PyTuple_Type, &inputs, &desc, &entry, &left, &right, &PyTuple_Type,
                        &operands, &tile, &PyTuple_Type, &extras, &PyTuple_Type, &reductions, &PyTuple_Type,
                        &outputs))
    return nullptr;
  auto p = std::make_unique<Plan>();
  const Py_ssize_t desc_len = desc.len;
  if (desc_len == (Py_ssize_t)sizeof(fuseml_gemm_desc)) std::memcpy(&p->desc, desc.buf, sizeof(fuseml_gemm_desc));
  PyBuffer_Release(&desc);
  const int n = self->n_inputs;
  if (desc_len != (Py_ssize_t)sizeof(fuseml_gemm_desc) || PyTuple_GET_SIZE(inputs) != n || left < 0 || left >= n ||
      right < 0 || right >= n || PyTuple_GET_SIZE(extras) > FUSEML_MAX_EXTRA_OUT || PyTuple_GET_SIZE(reductions) > 3 ||
      self->used->size() > FUSEML_MAX_OPERANDS + 2) {
    PyErr_SetString(PyExc_ValueError, "malformed plan");
    return nullptr;
  }
  if (self->plans->size() >= kMaxPlans) Py_RETURN_FALSE;
  for (int i : *self->used) {
    PyObject* o = PyTuple_GET_ITEM(inputs, i);
    if (!plain(o)) Py_RETURN_FALSE;
    p->signature.push_back(signature_of(THPVariable_Unpack(o)));
  }
  p->entry = reinterpret_cast<Entry>(static_cast<uintptr_t>(entry));
  p->left = left;
  p->right = right;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(operands); ++i) {
    int slot, index;
    if (!PyArg_ParseTuple(PyTuple_GET_ITEM(operands, i), "ii", &slot, &index)) return nullptr;
    if (slot < 0 || slot >= FUSEML_MAX_OPERANDS || index < 0 || index >= n) {
      PyErr_SetString(PyExc_ValueError, "malformed operand");
      return nullptr;
    }
    p->operands.emplace_back(slot, index);
  }
  auto dtype_of = [](PyObject* o) { return reinterpret_cast<THPDtype*>(o)->scalar_type; };
  p->tile = tile != Py_None;
  if (p->tile) {
    if (!THPDtype_Check(tile)) {
      PyErr_SetString(PyExc_TypeError, "tile: a dtype or None");
      return nullptr;
    }
    p->tile_dtype = dtype_of(tile);
  }
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(extras); ++i) {
    if (!THPDtype_Check(PyTuple_GET_ITEM(extras, i))) {
      PyErr_SetString(PyExc_TypeError, "extras: dtypes");
      return nullptr;
    }
    p->extras.push_back(dtype_of(PyTuple_GET_ITEM(extras, i)));
  }
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(reductions); ++i) {
    const long slot = PyLong_AsLong(PyTuple_GET_ITEM(reductions, i));
    if (slot < 0 || slot > 2) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "reduction slot");
      return nullptr;
    }
    p->reductions.push_back((int)slot);
  }
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(outputs); ++i) {
    int kind, index;
    if (!PyArg_ParseTuple(PyTuple_GET_ITEM(outputs, i), "Ci", &kind, &index)) return nullptr;
    const bool ok = kind == 't' ? p->tile : kind == 'r' ? index >= 0 && index < (int)p->reductions.size()
                                                        : kind == 'e' && index >= 0 && index < (int)p->extras.size();
    if (!ok) {
      PyErr_SetString(PyExc_ValueError, "malformed output");
      return nullptr;
    }
    p->outputs.emplace_back((char)kind, index);
  }
  if (p->outputs.empty()) {
    PyErr_SetString(PyExc_ValueError, "a plan has outputs");
    return nullptr;
  }
  self->plans->insert(self->plans->begin(), p.release());
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

PyObject* launcher_count(PyObject* self, void*) {
  return PyLong_FromLongLong(reinterpret_cast<Launcher*>(self)->count);
}

// Launcher(n_inputs, used, guarded)
PyObject* launcher_new(PyTypeObject* type, PyObject* args, PyObject*) {
  HANDLE_TH_ERRORS
  int n_inputs, guarded;
  PyObject* used;
  if (!PyArg_ParseTuple(args, "iO!p", &n_inputs, &PyTuple_Type, &used, &guarded)) return nullptr;
  auto indices = std::make_unique<std::vector<int>>();
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(used); ++i) {
    const long index = PyLong_AsLong(PyTuple_GET_ITEM(used, i));
    if (index < 0 || index >= n_inputs) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "input index out of range");
      return nullptr;
    }
    indices->push_back((int)index);
  }
  if (indices->empty()) {
    PyErr_SetString(PyExc_ValueError, "a launch reads inputs");
    return nullptr;
  }
  auto plans = std::make_unique<std::vector<Plan*>>();
  Launcher* self = reinterpret_cast<Launcher*>(type->tp_alloc(type, 0));
  if (self == nullptr) return nullptr;
  self->n_inputs = n_inputs;
  self->guarded = guarded != 0;
  self->count = 0;
  self->used = indices.release();
  self->plans = plans.release();
  return reinterpret_cast<PyObject*>(self);
  END_HANDLE_TH_ERRORS
}

void launcher_dealloc(PyObject* self_) {
  Launcher* self = reinterpret_cast<Launcher*>(self_);
  for (Plan* p : *self->plans) delete p;
  delete self->plans;
  delete self->used;
  Py_TYPE(self_)->tp_free(self_);
}

PyMethodDef kMethods[] = {
    {"call", launcher_call, METH_O, "call(inputs): outputs, an error code, or None (not served here)"},
    {"add", launcher_add, METH_VARARGS, "add(inputs, desc, entry, ...): a plan; whether it was taken"},
    {nullptr, nullptr, 0, nullptr}};

PyGetSetDef kGetSet[] = {{"count", launcher_count, nullptr, "launches made here", nullptr},
                         {nullptr, nullptr, nullptr, nullptr, nullptr}};

PyTypeObject g_type = {PyVarObject_HEAD_INIT(nullptr, 0) "fuseml_amd._fastcall.Launcher"};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fastcall", "Native calls of fused-group launchers.", -1, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fastcall() {
  g_type.tp_basicsize = sizeof(Launcher);
  g_type.tp_flags = Py_TPFLAGS_DEFAULT;
  g_type.tp_new = launcher_new;
  g_type.tp_dealloc = launcher_dealloc;
  g_type.tp_methods = kMethods;
  g_type.tp_getset = kGetSet;
  if (PyType_Ready(&g_type) < 0) return nullptr;
  PyObject* torch_c = PyImport_ImportModule("torch._C");
  if (torch_c == nullptr) return nullptr;
  g_raw_stream = PyObject_GetAttrString(torch_c, "_cuda_getCurrentRawStream");
  Py_DECREF(torch_c);
  if (g_raw_stream == nullptr) return nullptr;
  PyObject* m = PyModule_Create(&kModule);
  if (m == nullptr) return nullptr;
  Py_INCREF(&g_type);
  if (PyModule_AddObject(m, "Launcher", reinterpret_cast<PyObject*>(&g_type)) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}

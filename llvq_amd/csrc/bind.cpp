// The operator's calls of fused.py for the tensors they are nearly always made with: binary16, contiguous, on the device, of the right size.
//
// A product of a few microseconds is shorter than its call from Python: checks, torch.empty, ctypes and the launch take 6.6 us for one
// projection and 11.5 for a group of three (three results to allocate), where the kernels take 3.8 and 4.9.  Here the same checks, the
// results' allocation and the library's entry point are one call: 3.5 and 4.4, most of it the launch.  What is not such a tensor gets None back, and takes fused.py's own
// lines: they convert, or refuse, as ever; so does a call that the library refuses.
//
// Tensors that only look like one on the device (subclasses, those of a transformation or a tracer), and calls under a mode that wants to
// see what is done, are not taken either.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/EmptyTensor.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/llvq_hip.h"

namespace at::cuda {
c10::Allocator* getCUDADeviceAllocator();  // (ATen/cuda/CUDAContextLight.h, whose other declarations want the device's libraries' headers)
}

namespace {

// The library's entry points, as fused.py loads them (bind_library): this module is not linked to a second copy.
decltype(&llvq_hip_gemv) g_gemv;
decltype(&llvq_hip_gemv_group) g_gemv_group;
decltype(&llvq_hip_gemm) g_gemm;
decltype(&llvq_hip_gemm_group) g_gemm_group;
PyObject *g_handle, *g_d_in, *g_d_out;  // attribute names
constexpr Py_ssize_t kMost = 16;        // projections of a call

// A plain call: no mode or transformation around it.
bool plain_call() {
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  return !(tls.included_.raw_repr() & ~c10::default_included_set.raw_repr()) && !at::impl::torch_function_mode_enabled();
}
// A tensor of that dtype whose memory is what its kernels would read.
bool plain_tensor(PyObject* obj, at::ScalarType type, const at::Tensor** out) {
  if (!THPVariable_CheckExact(obj)) return false;
  const at::Tensor& t = THPVariable_Unpack(obj);
  static const c10::DispatchKeySet allowed =
      c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::AutocastCUDA});
  if ((t.key_set().raw_repr() & ~allowed.raw_repr()) || !t.is_cuda() || t.scalar_type() != type || !t.is_contiguous()) return false;
  *out = &t;
  return true;
}
bool out_type(PyObject* dtype, at::ScalarType* type) {
  if (dtype == Py_None) *type = at::kHalf;
  else if (THPDtype_Check(dtype)) *type = reinterpret_cast<THPDtype*>(dtype)->scalar_type;
  else return false;
  return *type == at::kHalf || *type == at::kFloat;
}
int code_of(at::ScalarType type) { return type == at::kFloat ? LLVQ_F32 : LLVQ_F16; }

struct Proj {
  const llvq_mat* mat;
  int64_t d_in, d_out;
};
bool long_attr(PyObject* obj, PyObject* name, int64_t* v) {
  PyObject* a = PyObject_GetAttr(obj, name);
  if (!a) {
    PyErr_Clear();
    return false;
  }
  const bool ok = PyLong_Check(a);
  if (ok) *v = PyLong_AsLongLong(a);
  Py_DECREF(a);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return ok;
}
bool proj_of(PyObject* obj, Proj* p) {
  int64_t h = 0;
  if (!long_attr(obj, g_handle, &h) || !h || !long_attr(obj, g_d_in, &p->d_in) || !long_attr(obj, g_d_out, &p->d_out)) return false;
  p->mat = reinterpret_cast<const llvq_mat*>(static_cast<uintptr_t>(h));
  return true;
}
bool runtime_of(PyObject* obj, llvq_rt** rt) {
  int64_t h = 0;
  if (!long_attr(obj, g_handle, &h) || !h) return false;
  *rt = reinterpret_cast<llvq_rt*>(static_cast<uintptr_t>(h));
  return true;
}
Py_ssize_t projs_of(PyObject* obj, Proj (&p)[kMost]) {
  if (!PyList_CheckExact(obj) && !PyTuple_CheckExact(obj)) return 0;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(obj);
  if (n > kMost) return 0;
  for (Py_ssize_t i = 0; i < n; ++i)
    if (!proj_of(PySequence_Fast_GET_ITEM(obj, i), &p[i])) return 0;
  return n;
}
// On the current device, which is x's (c10::DeviceGuard).  (What at::empty does behind its dispatch and the guards of its own, which are most of an
// allocation's time: a group of three results 5.4 -> 4.4 us of host time a call, 5.48 -> 4.58 a pass.)
at::Tensor result_like(const at::Tensor& x, int64_t d_out, at::ScalarType type) {
  c10::SmallVector<int64_t, 4> dims(x.sizes().begin(), x.sizes().end());
  dims.back() = d_out;
  return at::Tensor(at::detail::empty_generic(dims, at::cuda::getCUDADeviceAllocator(), c10::DispatchKeySet(c10::DispatchKey::CUDA), type, std::nullopt));
}

// A C++ exception of the allocation is fused.py's to raise: its own lines meet it again.
template <class Fn>
PyObject* guarded(Fn&& fn) {
  try {
    if (PyObject* got = fn()) return got;
  } catch (const std::exception&) {
  }
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
}

// (runtime, projection, x, dtype or None) -> y, or None: not for here
PyObject* forward(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 4) Py_RETURN_NONE;
  return guarded([&]() -> PyObject* {
    llvq_rt* rt;
    Proj p;
    const at::Tensor* x;
    at::ScalarType type;
    if (!plain_call() || !runtime_of(args[0], &rt) || !proj_of(args[1], &p) || !plain_tensor(args[2], at::kHalf, &x) || !out_type(args[3], &type)) return nullptr;
    if (x->dim() < 1 || x->numel() != p.d_in || x->size(-1) != p.d_in) return nullptr;
    const c10::DeviceGuard on(x->device());
    at::Tensor y = result_like(*x, p.d_out, type);
    const void* in = x->const_data_ptr();
    void* out = y.mutable_data_ptr();
    int rc;
    Py_BEGIN_ALLOW_THREADS rc = g_gemv(rt, p.mat, in, out, code_of(type));
    Py_END_ALLOW_THREADS
    return rc ? nullptr : THPVariable_Wrap(std::move(y));
  });
}

// (runtime, projections, x, dtype or None) -> [y], or None
PyObject* forward_group(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 4) Py_RETURN_NONE;
  return guarded([&]() -> PyObject* {
    llvq_rt* rt;
    Proj p[kMost];
    const at::Tensor* x;
    at::ScalarType type;
    if (!plain_call() || !runtime_of(args[0], &rt) || !plain_tensor(args[2], at::kHalf, &x) || !out_type(args[3], &type)) return nullptr;
    const Py_ssize_t n = projs_of(args[1], p);
    if (n < 1 || x->dim() < 1 || x->numel() != p[0].d_in || x->size(-1) != p[0].d_in) return nullptr;
    const c10::DeviceGuard on(x->device());
    at::Tensor y[kMost];
    const llvq_mat* mats[kMost];
    void* outs[kMost];
    for (Py_ssize_t i = 0; i < n; ++i) {
      y[i] = result_like(*x, p[i].d_out, type);
      mats[i] = p[i].mat;
      outs[i] = y[i].mutable_data_ptr();
    }
    const void* in = x->const_data_ptr();
    int rc;
    Py_BEGIN_ALLOW_THREADS rc = g_gemv_group(rt, mats, (int)n, in, outs, code_of(type));
    Py_END_ALLOW_THREADS
    if (rc) return nullptr;
    PyObject* list = PyList_New(n);
    for (Py_ssize_t i = 0; list && i < n; ++i) {
      PyObject* w = THPVariable_Wrap(std::move(y[i]));
      if (!w) Py_CLEAR(list);
      else PyList_SET_ITEM(list, i, w);
    }
    return list;
  });
}

// (runtime, projection, x [M, d_in], dtype or None) -> y [M, d_out], or None
PyObject* forward_batched(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 4) Py_RETURN_NONE;
  return guarded([&]() -> PyObject* {
    llvq_rt* rt;
    Proj p;
    const at::Tensor* x;
    at::ScalarType type;
    if (!plain_call() || !runtime_of(args[0], &rt) || !proj_of(args[1], &p) || !plain_tensor(args[2], at::kHalf, &x) || !out_type(args[3], &type)) return nullptr;
    if (x->dim() != 2 || x->size(1) != p.d_in || x->size(0) < 1 || x->size(0) > INT_MAX) return nullptr;
    const c10::DeviceGuard on(x->device());
    at::Tensor y = result_like(*x, p.d_out, type);
    const void* in = x->const_data_ptr();
    void* out = y.mutable_data_ptr();
    const int rows = (int)x->size(0);
    int rc;
    Py_BEGIN_ALLOW_THREADS rc = g_gemm(rt, p.mat, in, rows, out, code_of(type));
    Py_END_ALLOW_THREADS
    return rc ? nullptr : THPVariable_Wrap(std::move(y));
  });
}

// (runtime, projections, x [M, d_in], [y]) -> True, or None
PyObject* forward_batched_group_into(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 4) Py_RETURN_NONE;
  return guarded([&]() -> PyObject* {
    llvq_rt* rt;
    Proj p[kMost];
    const at::Tensor* x;
    if (!plain_call() || !runtime_of(args[0], &rt) || !plain_tensor(args[2], at::kHalf, &x)) return nullptr;
    if (!PyList_CheckExact(args[3]) && !PyTuple_CheckExact(args[3])) return nullptr;
    const Py_ssize_t n = projs_of(args[1], p);
    if (n < 1 || PySequence_Fast_GET_SIZE(args[3]) != n || x->dim() != 2 || x->size(0) < 1 || x->size(0) > INT_MAX) return nullptr;
    const llvq_mat* mats[kMost];
    void* outs[kMost];
    at::ScalarType type = at::kHalf;
    for (Py_ssize_t i = 0; i < n; ++i) {
      PyObject* obj = PySequence_Fast_GET_ITEM(args[3], i);
      const at::Tensor* y;
      if (i == 0 && THPVariable_CheckExact(obj)) type = THPVariable_Unpack(obj).scalar_type();
      if ((type != at::kHalf && type != at::kFloat) || !plain_tensor(obj, type, &y)) return nullptr;
      if (p[i].d_in != x->size(1) || y->dim() != 2 || y->size(0) != x->size(0) || y->size(1) != p[i].d_out) return nullptr;
      mats[i] = p[i].mat;
      outs[i] = y->mutable_data_ptr();
    }
    const void* in = x->const_data_ptr();
    const int rows = (int)x->size(0);
    int rc;
    Py_BEGIN_ALLOW_THREADS rc = g_gemm_group(rt, mats, (int)n, in, rows, outs, code_of(type));
    Py_END_ALLOW_THREADS
    if (rc) return nullptr;
    Py_RETURN_TRUE;
  });
}

// (addresses of llvq_hip_gemv, _gemv_group, _gemm, _gemm_group)
PyObject* bind_library(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 4) return PyErr_Format(PyExc_TypeError, "four addresses");
  void* at[4];
  for (int i = 0; i < 4; ++i) {
    at[i] = PyLong_AsVoidPtr(args[i]);
    if (PyErr_Occurred()) return nullptr;
  }
  g_gemv = reinterpret_cast<decltype(g_gemv)>(at[0]);
  g_gemv_group = reinterpret_cast<decltype(g_gemv_group)>(at[1]);
  g_gemm = reinterpret_cast<decltype(g_gemm)>(at[2]);
  g_gemm_group = reinterpret_cast<decltype(g_gemm_group)>(at[3]);
  Py_RETURN_NONE;
}

template <class Fn>
PyCFunction fast(Fn* fn) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fn)); }
PyMethodDef kMethods[] = {{"bind_library", fast(bind_library), METH_FASTCALL, nullptr},
                          {"forward", fast(forward), METH_FASTCALL, nullptr},
                          {"forward_group", fast(forward_group), METH_FASTCALL, nullptr},
                          {"forward_batched", fast(forward_batched), METH_FASTCALL, nullptr},
                          {"forward_batched_group_into", fast(forward_batched_group_into), METH_FASTCALL, nullptr},
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() {
  g_handle = PyUnicode_InternFromString("_at");
  g_d_in = PyUnicode_InternFromString("d_in");
  g_d_out = PyUnicode_InternFromString("d_out");
  PyObject* module = g_handle && g_d_in && g_d_out ? PyModule_Create(&kModule) : nullptr;
  // the torch and the interpreter of the build: _ffi.py makes no call here under others
  if (module && PyModule_AddStringConstant(module, "built_for", LLVQ_BUILT_FOR)) Py_CLEAR(module);
  return module;
}

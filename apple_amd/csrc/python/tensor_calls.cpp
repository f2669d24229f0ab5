// tensor_calls: the element entry points of the C ABI called straight from
// torch tensors.
//
// An evaluation of a small body is bound by the host: of 14.8 us per call
// (E, gradient and Hessian diagonal of 5,000 tets) 6.8 were the C entry with
// its two launches, the rest the checks of ten arguments in Python.  Here an
// argument's type, device, shape and contiguity are read from the tensor
// itself: 7.2 us per call, and the device, at 9.1, is the slower side.  Whatever is not a
// plain device tensor that passes all of them (subclasses, wrappers of vmap
// and tracing, symbolic sizes, another dtype, ...) makes the call return None
// before anything has run, and the caller takes its checked path, which
// accepts it or raises the error that names it.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include "../../../include/apple_amd.h"

namespace {

using Eval = decltype(&apl_elem_eval);
using Mixed = decltype(&apl_elem_mixed_activation);
using SetActivation = decltype(&apl_mesh_set_activation);

// What a mesh's tensors have to be
struct Spec {
  c10::ScalarType dtype;
  int64_t device;
  int64_t n_tets, n_verts, n_inst;
};

// Data pointer of a tensor of the given form, NULL of None; false: not plain or not of that form.
// cols 0: one dimension
bool pointer(PyObject* o, c10::ScalarType dtype, int64_t device, int64_t rows, int64_t cols, void** out) {
  *out = nullptr;
  if (o == Py_None) return true;
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  const c10::TensorImpl* impl = t.unsafeGetTensorImpl();
  if (impl->is_python_dispatch() || impl->has_symbolic_sizes_strides() || !impl->has_storage()) return false;
  const c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                     c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize});
  if (impl->key_set().has_any(wrapped) || t.layout() != c10::kStrided) return false;
  if (t.scalar_type() != dtype || !t.is_cuda() || t.get_device() != device) return false;
  const c10::IntArrayRef s = t.sizes();
  if (s.size() != (cols > 0 ? 2u : 1u) || s[0] != rows || (cols > 0 && s[1] != cols)) return false;
  if (!t.is_contiguous()) return false;
  *out = t.mutable_data_ptr();
  return true;
}

bool integer(PyObject* o, int64_t* out) {
  if (!PyLong_Check(o)) return false;
  *out = PyLong_AsLongLong(o);
  return !(*out == -1 && PyErr_Occurred());
}

// An address given as an integer; 0 is not one
template <class T>
bool address(PyObject* o, T* out) {
  if (!PyLong_Check(o)) return false;
  void* p = PyLong_AsVoidPtr(o);
  if (p == nullptr) return false;
  *out = reinterpret_cast<T>(p);
  return true;
}

// (entry, handle, stream, (FP64, device, n_tets, n_verts, n_inst))
template <class F>
bool head(PyObject* const* a, F* f, apl_mesh** mesh, void** stream, Spec* s) {
  int64_t f64;
  if (!address(a[0], f) || !address(a[1], mesh) || !PyLong_Check(a[2]) || !PyTuple_CheckExact(a[3]) ||
      PyTuple_GET_SIZE(a[3]) != 5)
    return false;
  *stream = PyLong_AsVoidPtr(a[2]);
  if (!integer(PyTuple_GET_ITEM(a[3], 0), &f64) || !integer(PyTuple_GET_ITEM(a[3], 1), &s->device) ||
      !integer(PyTuple_GET_ITEM(a[3], 2), &s->n_tets) || !integer(PyTuple_GET_ITEM(a[3], 3), &s->n_verts) ||
      !integer(PyTuple_GET_ITEM(a[3], 4), &s->n_inst))
    return false;
  s->dtype = f64 != 0 ? c10::kDouble : c10::kFloat;
  return true;
}

PyObject* declined() {
  PyErr_Clear();
  Py_RETURN_NONE;
}

// elem_eval(entry, handle, stream, spec, material, accumulate, mu, lam, u, p,
//           energy, grad, hess_diag, hess_prod, hess_quad, dmu, dlam) -> status or None
PyObject* elem_eval(PyObject*, PyObject* const* a, Py_ssize_t n) {
  Eval f;
  apl_mesh* mesh;
  void* stream;
  Spec s;
  int64_t material;
  int acc;
  void *mu, *lam, *u, *p, *energy, *grad, *hess_diag, *hess_prod, *hess_quad, *dmu, *dlam;
  try {
    if (n != 17 || !head(a, &f, &mesh, &stream, &s) || !integer(a[4], &material)) return declined();
    acc = PyObject_IsTrue(a[5]);
    if (acc < 0) return declined();
    if (!pointer(a[6], s.dtype, s.device, s.n_tets, 0, &mu) || !pointer(a[7], s.dtype, s.device, s.n_tets, 0, &lam) ||
        !pointer(a[8], s.dtype, s.device, s.n_verts, 3, &u) || !pointer(a[9], s.dtype, s.device, s.n_verts, 3, &p) ||
        !pointer(a[10], c10::kDouble, s.device, s.n_inst, 0, &energy) ||
        !pointer(a[11], s.dtype, s.device, s.n_verts, 3, &grad) ||
        !pointer(a[12], s.dtype, s.device, s.n_verts, 3, &hess_diag) ||
        !pointer(a[13], s.dtype, s.device, s.n_verts, 3, &hess_prod) ||
        !pointer(a[14], c10::kDouble, s.device, s.n_inst, 0, &hess_quad) ||
        !pointer(a[15], s.dtype, s.device, s.n_tets, 0, &dmu) || !pointer(a[16], s.dtype, s.device, s.n_tets, 0, &dlam))
      return declined();
  } catch (...) {
    return declined();
  }
  const unsigned what = (a[10] != Py_None ? APL_ENERGY : 0u) | (a[11] != Py_None ? APL_GRAD : 0u) |
                        (a[12] != Py_None ? APL_HESS_DIAG : 0u) | (a[13] != Py_None ? APL_HESS_PROD : 0u) |
                        (a[14] != Py_None ? APL_HESS_QUAD : 0u) | (a[15] != Py_None ? APL_MIXED : 0u) |
                        (acc ? APL_ACCUMULATE : 0u);
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = f(mesh, (int)material, mu, lam, u, p, what, (double*)energy, grad, hess_diag, hess_prod, (double*)hess_quad, dmu,
         dlam, stream);
  Py_END_ALLOW_THREADS;
  return PyLong_FromLong(rc);
}

// elem_mixed_activation(entry, handle, stream, spec, accumulate, mu, lam, u, p, dact, dmu, dlam) -> status or None
PyObject* elem_mixed_activation(PyObject*, PyObject* const* a, Py_ssize_t n) {
  Mixed f;
  apl_mesh* mesh;
  void* stream;
  Spec s;
  int acc;
  void *mu, *lam, *u, *p, *dact, *dmu, *dlam;
  try {
    if (n != 12 || !head(a, &f, &mesh, &stream, &s)) return declined();
    acc = PyObject_IsTrue(a[4]);
    if (acc < 0) return declined();
    if (!pointer(a[5], s.dtype, s.device, s.n_tets, 0, &mu) || !pointer(a[6], s.dtype, s.device, s.n_tets, 0, &lam) ||
        !pointer(a[7], s.dtype, s.device, s.n_verts, 3, &u) || !pointer(a[8], s.dtype, s.device, s.n_verts, 3, &p) ||
        !pointer(a[9], s.dtype, s.device, s.n_tets, 6, &dact) || !pointer(a[10], s.dtype, s.device, s.n_tets, 0, &dmu) ||
        !pointer(a[11], s.dtype, s.device, s.n_tets, 0, &dlam))
      return declined();
  } catch (...) {
    return declined();
  }
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = f(mesh, mu, lam, u, p, dact, dmu, dlam, acc, stream);
  Py_END_ALLOW_THREADS;
  return PyLong_FromLong(rc);
}

// set_activation(entry, handle, stream (unused), spec, activation) -> status or None
PyObject* set_activation(PyObject*, PyObject* const* a, Py_ssize_t n) {
  SetActivation f;
  apl_mesh* mesh;
  void* stream;
  Spec s;
  void* act;
  try {
    if (n != 5 || !head(a, &f, &mesh, &stream, &s) || !pointer(a[4], s.dtype, s.device, s.n_tets, 6, &act))
      return declined();
  } catch (...) {
    return declined();
  }
  return PyLong_FromLong(f(mesh, act));
}

PyMethodDef METHODS[] = {
    {"elem_eval", (PyCFunction)(void (*)())elem_eval, METH_FASTCALL, nullptr},
    {"elem_mixed_activation", (PyCFunction)(void (*)())elem_mixed_activation, METH_FASTCALL, nullptr},
    {"set_activation", (PyCFunction)(void (*)())set_activation, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef MODULE = {PyModuleDef_HEAD_INIT, "tensor_calls", nullptr, -1, METHODS, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_tensor_calls() { return PyModule_Create(&MODULE); }

// The usual call of the package in native code: tensors are checked, workspace and results allocated and the C ABI called
// without a round through the interpreter (16-19 us of host time per call there, 8.5 here; top-k 12.6 and 6.2).  Bound: two
// allocations by torch and two kernel launches.
//
// Only what needs no copy and no message is taken: plain tensors on the current device in a layout the kernels
// read.  Everything else returns None, and the Python functions of flash.py, which do the same steps for any input, go on from there.
// Nothing is kept between calls.

#include <Python.h>

#include <ATen/Functions.h>
#include <ATen/core/Tensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>

#include "fcr.h"

namespace {

PyObject* g_check = nullptr;   // _lib.check: raises for a non-zero return code

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kHalf: return FCR_DTYPE_F16;
    case at::kBFloat16: return FCR_DTYPE_BF16;
    case at::kFloat: return FCR_DTYPE_F32;
    default: return -1;
  }
}

// A plain dense tensor that is where its type says (no subclass, no wrapper of a transform).
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage()) return nullptr;
  const c10::DispatchKeySet odd({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                 c10::DispatchKey::Functionalize, c10::DispatchKey::ZeroTensor, c10::DispatchKey::Negative});
  return t.key_set().has_any(odd) ? nullptr : &t;
}

// The layouts of flash.py::_device_layout that need no copy; strides of dimensions of size one as dense ones, which every
// check accepts.
bool layout(const at::Tensor& t, int64_t (&strides)[4]) {
  const int64_t al = 16 / t.element_size();
  const auto size = t.sizes(), stride = t.strides();
  if (size[3] % al != 0 || stride[3] != 1 || (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) != 0) return false;
  int64_t dense = size[3];
  for (int i = 2; i >= 0; --i) {
    strides[i] = size[i] == 1 ? dense : stride[i];
    if (strides[i] % al != 0 || strides[i] < 0) return false;
    dense = strides[i] * size[i];
  }
  strides[3] = 1;
  return strides[2] * t.element_size() < (1 << 25) && (size[2] <= 1 || strides[2] >= size[3]);
}

PyObject* failed(int rc) {
  PyObject* r = PyObject_CallFunction(g_check, "i", rc);
  Py_XDECREF(r);
  if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "libfcr reported an error");
  return nullptr;
}

// reduce(query, key, reduction, is_causal, scale, out_dtype, pair): the result, (sums or means, maxima) with `pair`, or None.
PyObject* reduce(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS   // (C++ exceptions as the Python ones torch raises for them)
  if (n != 7) {
    PyErr_SetString(PyExc_TypeError, "reduce takes seven arguments");
    return nullptr;
  }
  const at::Tensor* const qp = plain(args[0]);
  const at::Tensor* const kp = plain(args[1]);
  if (!qp || !kp || !PyUnicode_Check(args[2])) Py_RETURN_NONE;
  const at::Tensor &q = *qp, &k = *kp;
  int red;
  if (PyUnicode_CompareWithASCIIString(args[2], "sum") == 0) red = FCR_REDUCE_SUM;
  else if (PyUnicode_CompareWithASCIIString(args[2], "mean") == 0) red = FCR_REDUCE_MEAN;
  else if (PyUnicode_CompareWithASCIIString(args[2], "max") == 0) red = FCR_REDUCE_MAX;
  else Py_RETURN_NONE;
  const int code = dtype_code(q.scalar_type());
  if (code < 0 || k.scalar_type() != q.scalar_type() || q.dim() != 4 || k.dim() != 4 || q.device() != k.device()) Py_RETURN_NONE;
  const auto qs = q.sizes(), ks = k.sizes();
  if (qs[0] != ks[0] || qs[1] != ks[1] || qs[3] != ks[3] || q.numel() == 0 || k.numel() == 0) Py_RETURN_NONE;
  if (qs[3] * q.element_size() > 1024 || qs[0] > INT32_MAX || qs[1] > INT32_MAX || qs[2] > INT32_MAX || ks[2] > INT32_MAX) Py_RETURN_NONE;
  at::ScalarType out_type = q.scalar_type();
  if (args[5] != Py_None) {
    if (!THPDtype_Check(args[5])) Py_RETURN_NONE;
    out_type = reinterpret_cast<THPDtype*>(args[5])->scalar_type;
    if (dtype_code(out_type) < 0) Py_RETURN_NONE;
  }
  double scale;
  if (args[4] == Py_None) scale = 1.0 / std::sqrt((double)qs[3]);
  else if (PyFloat_CheckExact(args[4])) scale = PyFloat_AS_DOUBLE(args[4]);
  else Py_RETURN_NONE;
  const int causal = PyObject_IsTrue(args[3]);
  const int pair = PyObject_IsTrue(args[6]);
  if (causal < 0 || pair < 0) return nullptr;
    int64_t qst[4], kst[4];
    if (!layout(q, qst) || !layout(k, kst) || c10::hip::current_device() != q.device().index()) Py_RETURN_NONE;
    const int b = (int)qs[0], h = (int)qs[1], m = (int)qs[2], nk = (int)ks[2], d = (int)qs[3];
    size_t bytes = fcr_workspace_bytes(code, b, h, m, nk, d);
    const size_t least = 4 * (size_t)b * (size_t)h * (size_t)m;
    if (bytes < least) bytes = least;
    const at::Tensor ws = at::empty({(int64_t)(bytes / 4)}, q.options().dtype(at::kFloat));
    const auto options = q.options().dtype(out_type);
    at::Tensor out = at::empty({qs[0], qs[1], ks[2]}, options), out2;
    if (pair) out2 = at::empty({qs[0], qs[1], ks[2]}, options);
    void* const stream = c10::hip::getCurrentHIPStream(q.device().index()).stream();
    const void *const qd = q.const_data_ptr(), *const kd = k.const_data_ptr();
    void *const wd = ws.mutable_data_ptr(), *const od = out.mutable_data_ptr(), *const od2 = pair ? out2.mutable_data_ptr() : nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = fcr_colreduce_ws(qd, kd, od, od2, dtype_code(out_type), wd, bytes, code, b, h, m, nk, d, qst, kst, (float)scale, red, causal, stream);
    Py_END_ALLOW_THREADS
    if (rc) return failed(rc);
    if (!pair) return THPVariable_Wrap(std::move(out));
    PyObject* const a = THPVariable_Wrap(std::move(out));
    PyObject* const z = THPVariable_Wrap(std::move(out2));
    if (a && z) return Py_BuildValue("(NN)", a, z);
    Py_XDECREF(a);
    Py_XDECREF(z);
    return nullptr;
  END_HANDLE_TH_ERRORS
}

// keep(scores, k, with_threshold): the mask, (mask, threshold), or None.
PyObject* keep(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS   // (C++ exceptions as the Python ones torch raises for them)
  if (n != 3) {
    PyErr_SetString(PyExc_TypeError, "keep takes three arguments");
    return nullptr;
  }
  const at::Tensor* const sp = plain(args[0]);
  if (!sp || !PyLong_CheckExact(args[1])) Py_RETURN_NONE;
  const at::Tensor& s = *sp;
  const int code = dtype_code(s.scalar_type());
  int overflow = 0;
  const long long k = PyLong_AsLongLongAndOverflow(args[1], &overflow);
  if (code < 0 || overflow || k > INT32_MAX || k < INT32_MIN || s.dim() < 1 || s.numel() == 0 || !s.is_contiguous()) Py_RETURN_NONE;
  const int with_threshold = PyObject_IsTrue(args[2]);
  if (with_threshold < 0) return nullptr;
  const int64_t cols = s.size(-1), rows = s.numel() / cols;
  if (cols > INT32_MAX) Py_RETURN_NONE;
    if (c10::hip::current_device() != s.device().index()) Py_RETURN_NONE;
    at::Tensor mask = at::empty(s.sizes(), s.options().dtype(at::kBool)), threshold, ws;
    if (with_threshold) threshold = at::empty(s.sizes().slice(0, s.dim() - 1), s.options().dtype(at::kFloat));
    const size_t bytes = fcr_topk_bytes_typed(code, rows, (int)cols);
    if (bytes) ws = at::empty({(int64_t)bytes}, s.options().dtype(at::kByte));
    void* const stream = c10::hip::getCurrentHIPStream(s.device().index()).stream();
    const void* const sd = s.const_data_ptr();
    uint8_t* const md = static_cast<uint8_t*>(mask.mutable_data_ptr());
    float* const td = with_threshold ? static_cast<float*>(threshold.mutable_data_ptr()) : nullptr;
    void* const wd = bytes ? ws.mutable_data_ptr() : nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = fcr_topk_mask_typed(sd, code, md, td, rows, (int)cols, (int)k, wd, bytes, stream);
    Py_END_ALLOW_THREADS
    if (rc) return failed(rc);
    if (!with_threshold) return THPVariable_Wrap(std::move(mask));
    PyObject* const a = THPVariable_Wrap(std::move(mask));
    PyObject* const z = THPVariable_Wrap(std::move(threshold));
    if (a && z) return Py_BuildValue("(NN)", a, z);
    Py_XDECREF(a);
    Py_XDECREF(z);
    return nullptr;
  END_HANDLE_TH_ERRORS
}

PyObject* on_error(PyObject*, PyObject* f) {
  Py_INCREF(f);
  Py_XSETREF(g_check, f);
  Py_RETURN_NONE;
}

PyMethodDef g_methods[] = {
    {"reduce", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(reduce)), METH_FASTCALL, "reduce(query, key, reduction, is_causal, scale, out_dtype, pair)"},
    {"keep", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(keep)), METH_FASTCALL, "keep(scores, k, with_threshold)"},
    {"on_error", on_error, METH_O, "on_error(f): f(rc) raises for a return code of the library"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_host", "the usual call in native code", -1, g_methods};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&g_module); }

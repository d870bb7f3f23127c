// g950_py -- packing of an operator call from Python objects in native code.
//
// launch() turns torch tensors and Python scalars into g950_view / g950_scalar
// records on the stack and calls the C ABI entry (include/g950rt.h) it is
// given.  The same packing through ctypes cost more than most kernels: a
// 4-view, 6-scalar call (rmsnorm of a decoding step) took 35 us of host time
// for a 4 us kernel.  Anything but plain device tensors of the supported
// dtypes and int / bool / float / float32 / packed scalars is left to the
// ctypes path (launch() returns None), which raises the errors or encodes the
// rarer scalar types.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <cstring>

#include "../../include/g950rt.h"

namespace {

typedef int (*launch_fn)(g950_module*, uint32_t, const g950_view*, uint32_t, const g950_scalar*, uint32_t, void*);

constexpr Py_ssize_t kMaxViews = 16, kMaxScalars = 64, kMaxDims = 8;
PyObject* g_scalar_type = nullptr;   // compiler_amd.runtime.Scalar (16 bytes, the buffer protocol)
PyObject* g_float32_type = nullptr;  // numpy.float32

uint32_t dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return G950_DTYPE_FLOAT32;
    case at::kBFloat16: return G950_DTYPE_BFLOAT16;
    case at::kHalf: return G950_DTYPE_FLOAT16;
    case at::kChar: return G950_DTYPE_INT8;
    case at::kByte: return G950_DTYPE_UINT8;
    case at::kShort: return G950_DTYPE_INT16;
    case at::kInt: return G950_DTYPE_INT32;
    case at::kLong: return G950_DTYPE_INT64;
    case at::kDouble: return G950_DTYPE_FLOAT64;
    case at::kBool: return G950_DTYPE_BOOL;
    default: return 0;
  }
}

// 1: packed, 0: not a case of this path, -1: Python error set
int pack_scalar(PyObject* o, g950_scalar& s) {
  if (PyBool_Check(o)) {
    s = {G950_DTYPE_BOOL, 1, o == Py_True ? 1ull : 0ull};
  } else if (PyLong_CheckExact(o)) {
    int overflow = 0;
    const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
    if (overflow) return 0;
    if (v == -1 && PyErr_Occurred()) return -1;
    s = {G950_DTYPE_INT64, 8, (uint64_t)v};
  } else if (PyFloat_CheckExact(o)) {
    const double v = PyFloat_AS_DOUBLE(o);
    s.dtype = G950_DTYPE_FLOAT64;
    s.size = 8;
    memcpy(&s.bits, &v, 8);
  } else if ((PyObject*)Py_TYPE(o) == g_float32_type) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) return -1;
    const float f = (float)v;
    uint32_t b;
    memcpy(&b, &f, 4);
    s = {G950_DTYPE_FLOAT32, 4, b};
  } else if ((PyObject*)Py_TYPE(o) == g_scalar_type) {
    Py_buffer buf;
    if (PyObject_GetBuffer(o, &buf, PyBUF_SIMPLE)) return -1;
    const bool fits = buf.len == (Py_ssize_t)sizeof s;
    if (fits) memcpy(&s, buf.buf, sizeof s);
    PyBuffer_Release(&buf);
    return fits ? 1 : 0;
  } else {
    return 0;
  }
  return 1;
}

// launch(entry, module, op, tensors, outputs, scalars, stream): the entry's
// return code, or None where the call is not one of this path's.  tensors,
// outputs (truth values) and scalars are tuples or lists.
PyObject* py_launch(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 7) {
    PyErr_SetString(PyExc_TypeError, "launch: 7 arguments");
    return nullptr;
  }
  void* entry = PyLong_AsVoidPtr(args[0]);
  void* module = PyLong_AsVoidPtr(args[1]);
  const unsigned long op = PyLong_AsUnsignedLong(args[2]);
  void* stream = PyLong_AsVoidPtr(args[6]);
  if (PyErr_Occurred()) return nullptr;
  for (int i = 3; i <= 5; ++i)
    if (!PyTuple_Check(args[i]) && !PyList_Check(args[i])) Py_RETURN_NONE;
  const Py_ssize_t nv = PySequence_Fast_GET_SIZE(args[3]), ns = PySequence_Fast_GET_SIZE(args[5]);
  if (nv > kMaxViews || ns > kMaxScalars || PySequence_Fast_GET_SIZE(args[4]) != nv) Py_RETURN_NONE;
  PyObject** tensors = PySequence_Fast_ITEMS(args[3]);
  PyObject** outs = PySequence_Fast_ITEMS(args[4]);
  PyObject** scalars = PySequence_Fast_ITEMS(args[5]);
  g950_view views[kMaxViews];
  int64_t shape[kMaxViews][kMaxDims], strides[kMaxViews][kMaxDims];
  g950_scalar sc[kMaxScalars];
  try {
    for (Py_ssize_t i = 0; i < nv; ++i) {
      if (!THPVariable_CheckExact(tensors[i])) Py_RETURN_NONE;
      const at::Tensor& t = THPVariable_Unpack(tensors[i]);
      if (!t.defined() || !t.is_cuda() || !t.has_storage() || t.dim() > kMaxDims) Py_RETURN_NONE;
      const uint32_t dt = dtype_code(t.scalar_type());
      if (!dt) Py_RETURN_NONE;
      const int64_t isz = (int64_t)t.element_size();
      const auto sizes = t.sizes();
      const auto steps = t.strides();
      for (int64_t d = 0; d < t.dim(); ++d) {
        shape[i][d] = sizes[d];
        strides[i][d] = steps[d] * isz;
      }
      const int out = PyObject_IsTrue(outs[i]);
      if (out < 0) return nullptr;
      const c10::Storage& st = t.storage();
      views[i] = {t.mutable_data_ptr(), shape[i], strides[i], (uint64_t)st.nbytes(), dt,
                  (uint32_t)t.dim(), out ? G950_VIEW_OUTPUT : 0u, 0u, st.mutable_data()};
    }
  } catch (...) {
    Py_RETURN_NONE;  // the ctypes path meets and reports it
  }
  for (Py_ssize_t i = 0; i < ns; ++i) {
    const int r = pack_scalar(scalars[i], sc[i]);
    if (r < 0) return nullptr;
    if (!r) Py_RETURN_NONE;
  }
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = ((launch_fn)entry)((g950_module*)module, (uint32_t)op, views, (uint32_t)nv, sc, (uint32_t)ns, stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// init(Scalar, numpy.float32): the scalar types recognised by identity
PyObject* py_init(PyObject*, PyObject* args) {
  PyObject *s, *f;
  if (!PyArg_ParseTuple(args, "OO", &s, &f)) return nullptr;
  Py_INCREF(s);
  Py_INCREF(f);
  g_scalar_type = s;
  g_float32_type = f;
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"launch", (PyCFunction)(void (*)(void))py_launch, METH_FASTCALL, nullptr},
                         {"init", py_init, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef def = {PyModuleDef_HEAD_INIT, "g950_py", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_g950_py(void) {
  PyObject* m = PyModule_Create(&def);
  // launch() reads tensors by this torch's layouts: the loader compares
  if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION)) Py_CLEAR(m);
  return m;
}

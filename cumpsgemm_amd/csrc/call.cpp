// CPython entry to the GEMM calls of the library (cumpsgemm_amd/_call.<suffix>.so).
//
// A small product is bound by what one call costs on the host.  Through ctypes the
// conversion of its 17 arguments takes 1.8 us of the 5.3 us of a 128^3 product in a
// loop of calls; here 0.4 of 4.2.  The functions are called at the
// addresses that `bind` is given (the library that ctypes has loaded).  An argument
// of a type that is not the usual one -- anything but int sizes, float / complex
// scalars, and ints, None or objects with data_ptr() as pointers -- makes a call
// return None with nothing done: ctypes then converts it, or refuses it.  What an
// object's data_ptr() raises is raised by the call.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <cstring>
#include <cumpsgemm/cumpsgemm.h>
#include <cumpsgemm/cumpsgemm_ext.h>

namespace {
struct Functions {
  decltype(&cuMpSGEMM_sgemm) sgemm;
  decltype(&cuMpSGEMM_cgemm) cgemm;
  decltype(&cuMpSGEMM_sgemm_strided_batch) sgemm_strided_batch;
  decltype(&cuMpSGEMM_cgemm_strided_batch) cgemm_strided_batch;
  decltype(&cuMpSGEMM_sgemm_pipeline) sgemm_pipeline;
  decltype(&cuMpSGEMM_cgemm_pipeline) cgemm_pipeline;
  decltype(&cuMpSGEMM_sgemm_Mx2x2) sgemm_Mx2x2;
  decltype(&cuMpSGEMM_cgemm_Mx2x2) cgemm_Mx2x2;
  decltype(&cuMpSGEMM_sgemm_2xNx2) sgemm_2xNx2;
  decltype(&cuMpSGEMM_cgemm_2xNx2) cgemm_2xNx2;
} f;
constexpr Py_ssize_t kFunctions = sizeof(Functions) / sizeof(void *);
PyObject *data_ptr_name;

// The arguments of a call, taken one after the other; `ok` goes false at the first
// one that is not of the usual type, or whose data_ptr() raised (the exception is set).
struct Args {
  PyObject *const *arg;
  bool ok = true;
  uint64_t integer(PyObject *o) {
    if (!PyLong_Check(o)) {
      ok = false;
      return 0;
    }
    const uint64_t v = PyLong_AsUnsignedLongLongMask(o); // (as ctypes: no check of the range)
    if (v == (uint64_t)-1 && PyErr_Occurred()) {
      PyErr_Clear();
      ok = false;
    }
    return v;
  }
  uint64_t u64() { return ok ? integer(*arg++) : 0; }
  hipblasOperation_t op() { return (hipblasOperation_t)(int)u64(); }
  template <class T> T *ptr() {
    if (!ok) return nullptr;
    PyObject *const o = *arg++;
    if (o == Py_None) return nullptr;
    if (PyLong_Check(o)) return reinterpret_cast<T *>(integer(o));
    PyObject *const p = PyObject_CallMethodNoArgs(o, data_ptr_name);
    if (p == nullptr) {
      if (PyErr_ExceptionMatches(PyExc_AttributeError)) PyErr_Clear(); // (no data_ptr)
      ok = false;
      return nullptr;
    }
    const uint64_t v = integer(p);
    Py_DECREF(p);
    return reinterpret_cast<T *>(v);
  }
  void scalar(float &v) {
    if (!ok) return;
    PyObject *const o = *arg++;
    if (PyFloat_CheckExact(o)) v = (float)PyFloat_AS_DOUBLE(o);
    else ok = false;
  }
  void scalar(hipComplex &v) {
    if (!ok) return;
    PyObject *const o = *arg++;
    if (PyComplex_CheckExact(o)) v = {(float)PyComplex_RealAsDouble(o), (float)PyComplex_ImagAsDouble(o)};
    else if (PyFloat_CheckExact(o)) v = {(float)PyFloat_AS_DOUBLE(o), 0.0f};
    else ok = false;
  }
};

template <class Call> PyObject *status(const Args &a, Call &&call) {
  if (!a.ok) {
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
  }
  hipblasStatus_t st;
  Py_BEGIN_ALLOW_THREADS
  st = call();
  Py_END_ALLOW_THREADS
  return PyLong_FromLong((long)st);
}
bool count_is(const Py_ssize_t n, const Py_ssize_t want) {
  if (n == want) return true;
  PyErr_Format(PyExc_TypeError, "%zd arguments, not %zd", want, n);
  return false;
}

// handle, op_a, op_b, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, mode
template <class T, class Fn> PyObject *gemm_of(PyObject *const *args, const Fn fn) {
  Args x{args};
  auto *const h = x.ptr<cuMpSGEMM_handle>();
  const auto op_a = x.op(), op_b = x.op();
  const uint64_t m = x.u64(), n = x.u64(), k = x.u64();
  T alpha{}, beta{};
  x.scalar(alpha);
  T *const a = x.ptr<T>();
  const uint64_t lda = x.u64();
  T *const b = x.ptr<T>();
  const uint64_t ldb = x.u64();
  x.scalar(beta);
  T *const c = x.ptr<T>();
  const uint64_t ldc = x.u64();
  const auto mode = (cuMpSGEMM_compute_mode_t)(int)x.u64();
  return status(x, [&] { return fn(h, op_a, op_b, m, n, k, &alpha, a, lda, b, ldb, &beta, c, ldc, mode); });
}
// ..., a, lda, stride_a, b, ldb, stride_b, beta, c, ldc, stride_c, batch, mode
template <class T, class Fn> PyObject *strided_batch_of(PyObject *const *args, const Fn fn) {
  Args x{args};
  auto *const h = x.ptr<cuMpSGEMM_handle>();
  const auto op_a = x.op(), op_b = x.op();
  const uint64_t m = x.u64(), n = x.u64(), k = x.u64();
  T alpha{}, beta{};
  x.scalar(alpha);
  T *const a = x.ptr<T>();
  const uint64_t lda = x.u64(), stride_a = x.u64();
  T *const b = x.ptr<T>();
  const uint64_t ldb = x.u64(), stride_b = x.u64();
  x.scalar(beta);
  T *const c = x.ptr<T>();
  const uint64_t ldc = x.u64(), stride_c = x.u64(), batch = x.u64();
  const auto mode = (cuMpSGEMM_compute_mode_t)(int)x.u64();
  return status(x, [&] {
    return fn(h, op_a, op_b, m, n, k, &alpha, a, lda, stride_a, b, ldb, stride_b, &beta, c, ldc, stride_c, batch, mode);
  });
}
// ... and restore_ab; returns (status, (three ids))
template <class T, class Fn> PyObject *pipeline_of(PyObject *const *args, const Fn fn) {
  Args x{args};
  auto *const h = x.ptr<cuMpSGEMM_handle>();
  const auto op_a = x.op(), op_b = x.op();
  const uint64_t m = x.u64(), n = x.u64(), k = x.u64();
  T alpha{}, beta{};
  x.scalar(alpha);
  T *const a = x.ptr<T>();
  const uint64_t lda = x.u64(), stride_a = x.u64();
  T *const b = x.ptr<T>();
  const uint64_t ldb = x.u64(), stride_b = x.u64();
  x.scalar(beta);
  T *const c = x.ptr<T>();
  const uint64_t ldc = x.u64(), stride_c = x.u64(), batch = x.u64();
  const auto mode = (cuMpSGEMM_compute_mode_t)(int)x.u64();
  const int restore = (int)x.u64();
  unsigned ids[3] = {};
  PyObject *const st = status(x, [&] {
    return fn(h, op_a, op_b, m, n, k, &alpha, a, lda, stride_a, b, ldb, stride_b, &beta, c, ldc, stride_c, batch, mode,
              restore, ids);
  });
  if (st == nullptr || st == Py_None) return st;
  return Py_BuildValue("N(III)", st, ids[0], ids[1], ids[2]);
}
// handle, op_a, op_b, size, alpha, a, lda, stride_a, b, ldb, stride_b, beta, c, ldc, stride_c, batch
template <class T, class Fn> PyObject *by2x2_of(PyObject *const *args, const Fn fn) {
  Args x{args};
  auto *const h = x.ptr<cuMpSGEMM_handle>();
  const auto op_a = x.op(), op_b = x.op();
  const uint64_t size = x.u64();
  T alpha{}, beta{};
  x.scalar(alpha);
  T *const a = x.ptr<T>();
  const uint64_t lda = x.u64(), stride_a = x.u64();
  T *const b = x.ptr<T>();
  const uint64_t ldb = x.u64(), stride_b = x.u64();
  x.scalar(beta);
  T *const c = x.ptr<T>();
  const uint64_t ldc = x.u64(), stride_c = x.u64(), batch = x.u64();
  return status(x, [&] {
    return fn(h, op_a, op_b, size, &alpha, a, lda, stride_a, b, ldb, stride_b, &beta, c, ldc, stride_c, batch);
  });
}

// every function takes `cplx` first
bool is_complex(PyObject *o, bool &cplx) {
  const int r = PyObject_IsTrue(o);
  cplx = r > 0;
  return r >= 0;
}
PyObject *gemm(PyObject *, PyObject *const *args, Py_ssize_t n) {
  bool cplx;
  if (!count_is(n, 16) || !is_complex(args[0], cplx)) return nullptr;
  return cplx ? gemm_of<hipComplex>(args + 1, f.cgemm) : gemm_of<float>(args + 1, f.sgemm);
}
PyObject *strided_batch(PyObject *, PyObject *const *args, Py_ssize_t n) {
  bool cplx;
  if (!count_is(n, 20) || !is_complex(args[0], cplx)) return nullptr;
  return cplx ? strided_batch_of<hipComplex>(args + 1, f.cgemm_strided_batch)
              : strided_batch_of<float>(args + 1, f.sgemm_strided_batch);
}
PyObject *pipeline(PyObject *, PyObject *const *args, Py_ssize_t n) {
  bool cplx;
  if (!count_is(n, 21) || !is_complex(args[0], cplx)) return nullptr;
  return cplx ? pipeline_of<hipComplex>(args + 1, f.cgemm_pipeline) : pipeline_of<float>(args + 1, f.sgemm_pipeline);
}
PyObject *mx2x2(PyObject *, PyObject *const *args, Py_ssize_t n) {
  bool cplx;
  if (!count_is(n, 17) || !is_complex(args[0], cplx)) return nullptr;
  return cplx ? by2x2_of<hipComplex>(args + 1, f.cgemm_Mx2x2) : by2x2_of<float>(args + 1, f.sgemm_Mx2x2);
}
PyObject *twoxnx2(PyObject *, PyObject *const *args, Py_ssize_t n) {
  bool cplx;
  if (!count_is(n, 17) || !is_complex(args[0], cplx)) return nullptr;
  return cplx ? by2x2_of<hipComplex>(args + 1, f.cgemm_2xNx2) : by2x2_of<float>(args + 1, f.sgemm_2xNx2);
}
// the addresses of the functions, in the order of `Functions`
PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (!count_is(n, kFunctions)) return nullptr;
  void *p[kFunctions];
  for (Py_ssize_t i = 0; i < kFunctions; i++) {
    p[i] = PyLong_AsVoidPtr(args[i]);
    if (p[i] == nullptr) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "no function");
      return nullptr;
    }
  }
  memcpy(&f, p, sizeof f);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
                         {"gemm", (PyCFunction)(void (*)(void))gemm, METH_FASTCALL, nullptr},
                         {"strided_batch", (PyCFunction)(void (*)(void))strided_batch, METH_FASTCALL, nullptr},
                         {"pipeline", (PyCFunction)(void (*)(void))pipeline, METH_FASTCALL, nullptr},
                         {"mx2x2", (PyCFunction)(void (*)(void))mx2x2, METH_FASTCALL, nullptr},
                         {"twoxnx2", (PyCFunction)(void (*)(void))twoxnx2, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};
} // namespace

PyMODINIT_FUNC PyInit__call(void) {
  data_ptr_name = PyUnicode_InternFromString("data_ptr");
  return data_ptr_name == nullptr ? nullptr : PyModule_Create(&module);
}

// The entry points that small calls go through, called with torch tensors directly.
//
// A call on small operands is bound by the host: fbfft1D of 4096 rows of 32 points runs 3.5 us
// on the GPU, and filling two descriptors in Python, finding the stream and crossing ctypes took
// 5 us (fbfft1D then fbifft1D, one pass after the other: 10.3 us by way of ctypes, 6.2 us by way
// of this module).  Here a descriptor is filled from the tensor itself.
//
// Each function takes plain calls only - float32 GPU tensors of exact type Tensor or Parameter and
// rank up to 5 whose extents fit 32 bits, integers that fit, the current stream - and returns
// NotImplemented for any other, which its caller then makes by the general way with that way's
// results and errors.  The C entry point runs without the interpreter lock, as under ctypes.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include <limits>

#include "../../include/fbfft_amd.h"

namespace {

PyObject* getDevice;  // () -> current device
PyObject* rawStream;  // (device) -> the handle of its current stream

bool fits(int64_t v) { return v >= std::numeric_limits<int>::min() && v <= std::numeric_limits<int>::max(); }

bool describe(PyObject* o, fbfft_tensor* d) {
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.is_cuda() || t.layout() != at::kStrided || t.scalar_type() != at::kFloat || t.dim() > FBFFT_MAX_DIM) return false;
  *d = fbfft_tensor{};
  d->dim = (int)t.dim();
  for (int i = 0; i < d->dim; ++i) {
    if (!fits(t.size(i)) || !fits(t.stride(i))) return false;
    d->size[i] = (int)t.size(i);
    d->stride[i] = (int)t.stride(i);
  }
  d->data = static_cast<float*>(t.data_ptr());
  return true;
}

bool integer(PyObject* o, int* v) {
  if (!PyLong_Check(o)) return false;
  int over = 0;
  const long long x = PyLong_AsLongLongAndOverflow(o, &over);
  if (over || !fits(x)) return false;
  *v = (int)x;
  return true;
}

bool real(PyObject* o, float* v) {
  if (!PyFloat_Check(o)) return false;
  *v = (float)PyFloat_AS_DOUBLE(o);
  return true;
}

// device memory of any type: address and bytes
bool memory(PyObject* o, void** p, size_t* bytes) {
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.is_cuda() || t.layout() != at::kStrided) return false;
  *p = t.data_ptr();
  *bytes = (size_t)t.numel() * (size_t)t.element_size();
  return true;
}

// false with a Python error set: the stream could not be found
bool stream(void** s) {
  PyObject* device = PyObject_CallNoArgs(getDevice);
  if (!device) return false;
  PyObject* handle = PyObject_CallOneArg(rawStream, device);
  Py_DECREF(device);
  if (!handle) return false;
  *s = PyLong_AsVoidPtr(handle);
  Py_DECREF(handle);
  return !PyErr_Occurred();
}

// What a tensor has no address or strides for throws; the general way then raises it.
template <class F>
PyObject* guarded(Py_ssize_t given, Py_ssize_t wanted, F body) {
  if (given != wanted || !rawStream) Py_RETURN_NOTIMPLEMENTED;
  try {
    return body();
  } catch (...) {
    PyErr_Clear();
    Py_RETURN_NOTIMPLEMENTED;
  }
}

template <class F>
PyObject* call(F entry) {
  void* s = nullptr;
  if (!stream(&s)) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = entry(s);
  Py_END_ALLOW_THREADS;
  return PyLong_FromLong(rc);
}

// (real, complex, padL)
template <int (*ENTRY)(const fbfft_tensor*, const fbfft_tensor*, int, fbfft_stream_t)>
PyObject* rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 3, [&]() -> PyObject* {
    fbfft_tensor x, y;
    int pad;
    if (!describe(a[0], &x) || !describe(a[1], &y) || !integer(a[2], &pad)) Py_RETURN_NOTIMPLEMENTED;
    return call([&](void* s) { return ENTRY(&x, &y, pad, (fbfft_stream_t)s); });
  });
}

// (source, result, padL, padU)
template <int (*ENTRY)(const fbfft_tensor*, const fbfft_tensor*, int, int, fbfft_stream_t)>
PyObject* planes(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 4, [&]() -> PyObject* {
    fbfft_tensor x, y;
    int padL, padU;
    if (!describe(a[0], &x) || !describe(a[1], &y) || !integer(a[2], &padL) || !integer(a[3], &padU))
      Py_RETURN_NOTIMPLEMENTED;
    return call([&](void* s) { return ENTRY(&x, &y, padL, padU, (fbfft_stream_t)s); });
  });
}

// (A, B, C, conjA, conjB, accumulate, invNorm)
template <int (*ENTRY)(const fbfft_tensor*, const fbfft_tensor*, const fbfft_tensor*, int, int, int, float,
                       fbfft_stream_t)>
PyObject* product(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 7, [&]() -> PyObject* {
    fbfft_tensor A, B, C;
    int conjA, conjB, accumulate;
    float norm;
    if (!describe(a[0], &A) || !describe(a[1], &B) || !describe(a[2], &C) || !integer(a[3], &conjA) ||
        !integer(a[4], &conjB) || !integer(a[5], &accumulate) || !real(a[6], &norm))
      Py_RETURN_NOTIMPLEMENTED;
    return call([&](void* s) { return ENTRY(&A, &B, &C, conjA, conjB, accumulate, norm, (fbfft_stream_t)s); });
  });
}

// (x, y, result, fftSize, workspace)
template <int (*ENTRY)(const fbfft_tensor*, const fbfft_tensor*, const fbfft_tensor*, int, void*, size_t,
                       fbfft_stream_t)>
PyObject* layer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 5, [&]() -> PyObject* {
    fbfft_tensor x, y, out;
    int N;
    void* ws;
    size_t bytes;
    if (!describe(a[0], &x) || !describe(a[1], &y) || !describe(a[2], &out) || !integer(a[3], &N) ||
        !memory(a[4], &ws, &bytes))
      Py_RETURN_NOTIMPLEMENTED;
    return call([&](void* s) { return ENTRY(&x, &y, &out, N, ws, bytes, (fbfft_stream_t)s); });
  });
}

// (input, gradOutput, gradWeight, fftSize, scale, accumulate, workspace)
PyObject* accgrad(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 7, [&]() -> PyObject* {
    fbfft_tensor x, y, out;
    int N, accumulate;
    float scale;
    void* ws;
    size_t bytes;
    if (!describe(a[0], &x) || !describe(a[1], &y) || !describe(a[2], &out) || !integer(a[3], &N) ||
        !real(a[4], &scale) || !integer(a[5], &accumulate) || !memory(a[6], &ws, &bytes))
      Py_RETURN_NOTIMPLEMENTED;
    return call([&](void* s) {
      return fbfft_conv_accgrad(&x, &y, &out, N, scale, accumulate, ws, bytes, (fbfft_stream_t)s);
    });
  });
}

// (getDevice, rawStream): how torch names the current stream; kept for the life of the process
PyObject* setup(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 2) {
    PyErr_SetString(PyExc_TypeError, "setup(getDevice, rawStream)");
    return nullptr;
  }
  Py_INCREF(a[0]);
  Py_INCREF(a[1]);
  Py_XSETREF(getDevice, a[0]);
  Py_XSETREF(rawStream, a[1]);
  Py_RETURN_NONE;
}

#define FBFFT_METHOD(name, ...) \
  {name, (PyCFunction)(void (*)(void))(PyObject * (*)(PyObject*, PyObject* const*, Py_ssize_t))(__VA_ARGS__), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    FBFFT_METHOD("setup", setup),
    FBFFT_METHOD("r2c_1d", rows<fbfft_r2c_1d>),
    FBFFT_METHOD("c2r_1d", rows<fbfft_c2r_1d>),
    FBFFT_METHOD("r2c_2d", planes<fbfft_r2c_2d>),
    FBFFT_METHOD("c2r_2d", planes<fbfft_c2r_2d>),
    FBFFT_METHOD("transpose_mm", product<fbfft_transpose_mm>),
    FBFFT_METHOD("transpose_mm_packed", product<fbfft_transpose_mm_packed>),
    FBFFT_METHOD("conv_fprop", layer<fbfft_conv_fprop>),
    FBFFT_METHOD("conv_bprop", layer<fbfft_conv_bprop>),
    FBFFT_METHOD("conv_accgrad", accgrad),
    {nullptr, nullptr, 0, nullptr}};
#undef FBFFT_METHOD

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding() { return PyModule_Create(&module); }

// The Python side of the C ABI for the calls a program makes per layer and
// step: argument conversion, the operand-size checks and the call itself in
// one CPython call.  A launch of a few microseconds would otherwise be bound
// by the interpreter: ctypes' conversions, a parameter structure read field by
// field and a stream object built per call took 3.5 us of a small layer's 7.9.
//
// Every function takes the entry point's address first (from the library that
// capi.py loaded, so there is one library and one HIP runtime), device
// addresses as integers (None = NULL), and a parameter structure as any object
// with the buffer interface (the ctypes structures of capi.py).  It returns the
// status; operand sizes that do not fit the parameters raise AssertionError
// before anything is launched.  The GIL is released around the call.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstddef>
#include <cstdint>

#include "snn_hip.h"

namespace {

// Arguments of one call, read in order; `ok` turns false with a Python error
// set at the first that does not convert.
class Args {
 public:
  Args(PyObject* const* args, Py_ssize_t n, Py_ssize_t want)
      : args_(args), ok(n == want) {
    if (!ok) PyErr_Format(PyExc_TypeError, "%zd arguments, %zd wanted", n, want);
  }
  ~Args() {
    if (view_.obj != nullptr) PyBuffer_Release(&view_);
  }
  void* pointer() {
    PyObject* const o = args_[next_++];
    if (!ok || o == Py_None) return nullptr;
    void* const p = PyLong_AsVoidPtr(o);
    if (p == nullptr && PyErr_Occurred()) ok = false;
    return p;
  }
  size_t size() {
    PyObject* const o = args_[next_++];
    if (!ok) return 0;
    const size_t v = PyLong_AsSize_t(o);
    if (v == static_cast<size_t>(-1) && PyErr_Occurred()) ok = false;
    return v;
  }
  int integer() {
    PyObject* const o = args_[next_++];
    if (!ok) return 0;
    const long v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) ok = false;
    return static_cast<int>(v);
  }
  template <typename T>
  T params() {
    PyObject* const o = args_[next_++];
    T p = {};
    if (!ok) return p;
    if (PyObject_GetBuffer(o, &view_, PyBUF_SIMPLE) != 0) {
      ok = false;
    } else if (static_cast<size_t>(view_.len) != sizeof(T)) {
      PyErr_SetString(PyExc_TypeError, "parameters of another operator");
      ok = false;
    } else {
      p = *static_cast<const T*>(view_.buf);
    }
    return p;
  }
  void check(bool fits, const char* what) {
    if (ok && !fits) {
      PyErr_SetString(PyExc_AssertionError, what);
      ok = false;
    }
  }

 private:
  PyObject* const* args_;
  Py_ssize_t next_ = 0;
  Py_buffer view_ = {};

 public:
  bool ok;
};

template <typename Call>
PyObject* launch(const Args& a, Call call) {
  if (!a.ok) return nullptr;
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = call();
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(status);
}

struct Sizes {
  long long input, filter, output;
};

Sizes in_order(long long x, long long w, long long y, int direction) {
  if (direction == SNN_HIP_FORWARD) return {x, w, y};
  if (direction == SNN_HIP_INPUT_BACKPROP) return {y, w, x};
  return {x, y, w};
}

Sizes conv_sizes(const snn_hip_conv2d_params& p, int direction) {
  const long long n = p.batch;
  return in_order(n * p.in_rows * p.in_cols * p.channels,
                  static_cast<long long>(p.window_rows) * p.window_cols *
                      p.channels * p.features,
                  n * p.out_rows * p.out_cols * p.features, direction);
}

Sizes depthwise_sizes(const snn_hip_depthwise_params& p, int direction) {
  const long long n = p.batch;
  const long long cm =
      static_cast<long long>(p.channels) * p.channel_multiplier;
  return in_order(n * p.in_rows * p.in_cols * p.channels,
                  static_cast<long long>(p.window_rows) * p.window_cols * cm,
                  n * p.out_rows * p.out_cols * cm, direction);
}

// (fn, direction, input, numel, filter, numel, output, params, algorithm,
//  workspace, elements, stream)
PyObject* conv2d(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n, 12);
  if (!a.ok) return nullptr;
  using Fn = int (*)(const void*, const void*, void*,
                     const snn_hip_conv2d_params*, int, void*, size_t, void*);
  const Fn fn = reinterpret_cast<Fn>(a.pointer());
  const int direction = a.integer();
  const void* const input = a.pointer();
  const size_t n_input = a.size();
  const void* const filter = a.pointer();
  const size_t n_filter = a.size();
  void* const output = a.pointer();
  const auto p = a.params<snn_hip_conv2d_params>();
  const int algorithm = a.integer();
  void* const workspace = a.pointer();
  const size_t elems = a.size();
  void* const stream = a.pointer();
  const Sizes s = conv_sizes(p, direction);
  a.check(static_cast<long long>(n_input) == s.input &&
              static_cast<long long>(n_filter) == s.filter,
          "operand sizes do not fit the convolution's parameters");
  return launch(a, [&] {
    return fn(input, filter, output, &p, algorithm, workspace, elems, stream);
  });
}

// (fn, input, filter, bias, output, params, algorithm, activation, workspace,
//  elements, stream)
PyObject* conv2d_bias_act(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n, 11);
  if (!a.ok) return nullptr;
  using Fn = int (*)(const void*, const void*, const void*, void*,
                     const snn_hip_conv2d_params*, int, int, void*, size_t,
                     void*);
  const Fn fn = reinterpret_cast<Fn>(a.pointer());
  const void* const input = a.pointer();
  const void* const filter = a.pointer();
  const void* const bias = a.pointer();
  void* const output = a.pointer();
  const auto p = a.params<snn_hip_conv2d_params>();
  const int algorithm = a.integer();
  const int activation = a.integer();
  void* const workspace = a.pointer();
  const size_t elems = a.size();
  void* const stream = a.pointer();
  return launch(a, [&] {
    return fn(input, filter, bias, output, &p, algorithm, activation,
              workspace, elems, stream);
  });
}

// (fn, direction, input, numel, filter, numel, output, params, stream)
PyObject* depthwise(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n, 9);
  if (!a.ok) return nullptr;
  using Fn = int (*)(const void*, const void*, void*,
                     const snn_hip_depthwise_params*, void*);
  const Fn fn = reinterpret_cast<Fn>(a.pointer());
  const int direction = a.integer();
  const void* const input = a.pointer();
  const size_t n_input = a.size();
  const void* const filter = a.pointer();
  const size_t n_filter = a.size();
  void* const output = a.pointer();
  const auto p = a.params<snn_hip_depthwise_params>();
  void* const stream = a.pointer();
  const Sizes s = depthwise_sizes(p, direction);
  a.check(static_cast<long long>(n_input) == s.input &&
              static_cast<long long>(n_filter) == s.filter,
          "operand sizes do not fit the depthwise convolution's parameters");
  return launch(a, [&] { return fn(input, filter, output, &p, stream); });
}

// (fn, input, numel, output, params, op, stream)
PyObject* pooling_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n, 7);
  if (!a.ok) return nullptr;
  using Fn = int (*)(const void*, void*, const snn_hip_pooling_params*, int,
                     void*);
  const Fn fn = reinterpret_cast<Fn>(a.pointer());
  const void* const input = a.pointer();
  const size_t n_input = a.size();
  void* const output = a.pointer();
  const auto p = a.params<snn_hip_pooling_params>();
  const int op = a.integer();
  void* const stream = a.pointer();
  a.check(static_cast<long long>(n_input) ==
              static_cast<long long>(p.batch) * p.in_rows * p.in_cols *
                  p.channels,
          "the input's size does not fit the pooling's parameters");
  return launch(a, [&] { return fn(input, output, &p, op, stream); });
}

// (fn, input, output, dy, dx, params, op, stream)
PyObject* pooling_max_grad(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n, 8);
  if (!a.ok) return nullptr;
  using Fn = int (*)(const void*, const void*, const void*, void*,
                     const snn_hip_pooling_params*, int, void*);
  const Fn fn = reinterpret_cast<Fn>(a.pointer());
  const void* const input = a.pointer();
  const void* const output = a.pointer();
  const void* const dy = a.pointer();
  void* const dx = a.pointer();
  const auto p = a.params<snn_hip_pooling_params>();
  const int op = a.integer();
  void* const stream = a.pointer();
  return launch(a, [&] { return fn(input, output, dy, dx, &p, op, stream); });
}

// (fn, dy, dx, params, stream)
PyObject* pooling_avg_grad(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n, 5);
  if (!a.ok) return nullptr;
  using Fn = int (*)(const void*, void*, const snn_hip_pooling_params*, void*);
  const Fn fn = reinterpret_cast<Fn>(a.pointer());
  const void* const dy = a.pointer();
  void* const dx = a.pointer();
  const auto p = a.params<snn_hip_pooling_params>();
  void* const stream = a.pointer();
  return launch(a, [&] { return fn(dy, dx, &p, stream); });
}

// (fn, input, output, items, op, stream)
PyObject* pointwise_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n, 6);
  if (!a.ok) return nullptr;
  using Fn = int (*)(const void*, void*, size_t, int, void*);
  const Fn fn = reinterpret_cast<Fn>(a.pointer());
  const void* const input = a.pointer();
  void* const output = a.pointer();
  const size_t items = a.size();
  const int op = a.integer();
  void* const stream = a.pointer();
  return launch(a, [&] { return fn(input, output, items, op, stream); });
}

// A sequence of dimensions into `dims`; more than kMaxDims are counted but not
// kept (the entry point rejects them).
constexpr int kMaxDims = 8;
bool read_dims(PyObject* o, int* dims, int* count) {
  PyObject* const seq = PySequence_Fast(o, "dimensions are a sequence");
  if (seq == nullptr) return false;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
  for (Py_ssize_t i = 0; i < n && i < kMaxDims; ++i) {
    const long v = PyLong_AsLong(PySequence_Fast_GET_ITEM(seq, i));
    if (v == -1 && PyErr_Occurred()) {
      Py_DECREF(seq);
      return false;
    }
    dims[i] = static_cast<int>(v);
  }
  *count = static_cast<int>(n);
  Py_DECREF(seq);
  return true;
}

// (fn, lhs, rhs, output, lhs_dims, rhs_dims, op, stream)
PyObject* binaryop(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n, 8);
  if (!a.ok) return nullptr;
  using Fn = int (*)(const void*, const void*, void*, const int*, int,
                     const int*, int, int, void*);
  const Fn fn = reinterpret_cast<Fn>(a.pointer());
  const void* const lhs = a.pointer();
  const void* const rhs = a.pointer();
  void* const output = a.pointer();
  int lhs_dims[kMaxDims] = {}, rhs_dims[kMaxDims] = {};
  int n_lhs = 0, n_rhs = 0;
  if (!a.ok || !read_dims(args[4], lhs_dims, &n_lhs) ||
      !read_dims(args[5], rhs_dims, &n_rhs))
    return nullptr;
  Args rest(args + 6, n - 6, 2);
  const int op = rest.integer();
  void* const stream = rest.pointer();
  return launch(rest, [&] {
    return fn(lhs, rhs, output, lhs_dims, n_lhs, rhs_dims, n_rhs, op, stream);
  });
}

#define SNN_PY_METHOD(name)                                              \
  {                                                                      \
    #name,                                                               \
        reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&name)),   \
        METH_FASTCALL, nullptr                                           \
  }
PyMethodDef methods[] = {SNN_PY_METHOD(conv2d),
                         SNN_PY_METHOD(conv2d_bias_act),
                         SNN_PY_METHOD(depthwise),
                         SNN_PY_METHOD(pooling_forward),
                         SNN_PY_METHOD(pooling_max_grad),
                         SNN_PY_METHOD(pooling_avg_grad),
                         SNN_PY_METHOD(pointwise_forward),
                         SNN_PY_METHOD(binaryop),
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }

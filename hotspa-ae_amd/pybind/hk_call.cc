// CPython binding of the operator entry points of hk_rowwise.h, lib/hk_call.so, and, compiled with HT_CALL, of hetu_ops_c.h,
// lib/ht_call.so (two modules, so that a program without the operator layer does not load it).
//
// A call takes the C arguments in order and returns the entry point's code.  Tensors are handed over as they are and
// asked for what is needed (data_ptr(), shape, stride(), dtype, ...): a pointer argument is None or a tensor, an HtArray
// argument likewise (described for the length of the call), an array of integers a tuple or list, a stream None (torch's
// current one), a ctypes.c_void_p or an address.  Integers wrap like C's; a fraction or a text is refused as one.  The interpreter's
// lock is released while the entry point runs.  Built without torch's headers: it calls the methods that a Python caller would.
//
// A small call is bound by this path: with a ctypes object built per argument, RMSNorm with a residual of 16 x 4096 bf16
// (3.4 us of kernel) took 10.0 us a call, so it takes 5.0; a 256 x 1000 mean loss and its gradient 43.7 and 33.8.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <pthread.h>

#include <array>
#include <cstdio>
#include <exception>
#include <new>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include "hetu_ops_c.h"
#include "hk_rowwise.h"

namespace {

PyObject *s_data_ptr, *s_is_contiguous, *s_shape, *s_stride, *s_dtype, *s_is_cuda, *s_get_device, *s_value;
PyObject* g_dtype_codes;      // {torch dtype: code}
PyObject* g_current_stream;   // () -> address of torch's current stream (initialises the device if need be)
PyObject *g_get_device, *g_raw_stream;   // torch's own two steps of the same, once the device is initialised
bool g_initialised = false;   // in this process: a child of fork() asks g_current_stream again, which refuses there

bool to_i64(PyObject* o, int64_t* v) {
  if (PyLong_CheckExact(o)) {
    *v = int64_t(PyLong_AsUnsignedLongLongMask(o));
    return !(*v == -1 && PyErr_Occurred());
  }
  PyObject* i = PyNumber_Index(o);   // an integer of any type; a fraction or a text is none
  if (i == nullptr) return false;
  *v = int64_t(PyLong_AsUnsignedLongLongMask(i));
  Py_DECREF(i);
  return !(*v == -1 && PyErr_Occurred());
}

bool to_address(PyObject* tensor, void** p) {
  *p = nullptr;
  if (tensor == Py_None) return true;
  PyObject* a = PyObject_CallMethodNoArgs(tensor, s_data_ptr);
  if (a == nullptr) return false;
  *p = PyLong_AsVoidPtr(a);
  Py_DECREF(a);
  return !(*p == nullptr && PyErr_Occurred());
}

// f(i, value) for every integer of a sequence; -1 on an error
template <typename F>
Py_ssize_t each_i64(PyObject* seq, F&& f) {
  PyObject* fast = PySequence_Fast(seq, "a sequence of integers is expected");
  if (fast == nullptr) return -1;
  Py_ssize_t i = 0;
  for (; i < PySequence_Fast_GET_SIZE(fast); ++i) {   // (an item's conversion may change a list)
    int64_t v;
    PyObject* item = PySequence_Fast_GET_ITEM(fast, i);
    Py_INCREF(item);
    const bool ok = to_i64(item, &v);
    Py_DECREF(item);
    if (!ok) {
      Py_DECREF(fast);
      return -1;
    }
    f(i, v);
  }
  Py_DECREF(fast);
  return i;
}

int dtype_code_of(PyObject* tensor) {
  PyObject* dt = PyObject_GetAttr(tensor, s_dtype);
  if (dt == nullptr) return -1;
  PyObject* code = PyDict_GetItemWithError(g_dtype_codes, dt);   // borrowed
  if (code == nullptr && !PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, dt);
  Py_DECREF(dt);
  return code == nullptr ? -1 : int(PyLong_AsLong(code));
}

bool current_stream(void** p) {
  PyObject* r;
  if (g_initialised) {
    PyObject* dev = PyObject_CallNoArgs(g_get_device);
    if (dev == nullptr) return false;
    r = PyObject_CallOneArg(g_raw_stream, dev);
    Py_DECREF(dev);
  } else {
    r = PyObject_CallNoArgs(g_current_stream);
    g_initialised = r != nullptr;
  }
  if (r == nullptr) return false;
  *p = PyLong_AsVoidPtr(r);
  Py_DECREF(r);
  return !(*p == nullptr && PyErr_Occurred());
}

// ---- one C argument from one Python object ----
template <typename T> struct Arg;

template <> struct Arg<int> {
  int v;
  bool from(PyObject* o) { int64_t i; if (!to_i64(o, &i)) return false; v = int(i); return true; }
  int get() { return v; }
};
template <> struct Arg<int64_t> {
  int64_t v;
  bool from(PyObject* o) { return to_i64(o, &v); }
  int64_t get() { return v; }
};
template <> struct Arg<uint64_t> {   // size_t as well
  int64_t v;
  bool from(PyObject* o) { return to_i64(o, &v); }
  uint64_t get() { return uint64_t(v); }
};
template <> struct Arg<double> {
  double v;
  bool from(PyObject* o) { v = PyFloat_AsDouble(o); return !(v == -1.0 && PyErr_Occurred()); }
  double get() { return v; }
};
template <> struct Arg<float> : Arg<double> {
  float get() { return float(v); }
};
template <typename P> struct PointerArg {
  void* v;
  bool from(PyObject* o) { return to_address(o, &v); }
  P get() { return static_cast<P>(v); }
};
template <> struct Arg<void*> : PointerArg<void*> {};
template <> struct Arg<const void*> : PointerArg<const void*> {};
template <> struct Arg<float*> : PointerArg<float*> {};
template <> struct Arg<const float*> : PointerArg<const float*> {};
template <> struct Arg<uint8_t*> : PointerArg<uint8_t*> {};
template <> struct Arg<const uint8_t*> : PointerArg<const uint8_t*> {};
// Integers on the host (shape, steps, axes, flags): a tuple, a list or None, never a tensor.
template <typename I> struct HostArray {
  std::array<I, 16> few;
  std::vector<I> many;
  I* v = nullptr;
  bool from(PyObject* o) {
    if (o == Py_None) return true;
    if (!PyTuple_Check(o) && !PyList_Check(o)) {
      PyErr_Format(PyExc_TypeError, "a tuple or list of integers is expected, not %s", Py_TYPE(o)->tp_name);
      return false;
    }
    const Py_ssize_t n = PySequence_Size(o);
    if (n < 0) return false;
    I* dst = few.data();
    if (size_t(n) > few.size()) {
      many.resize(size_t(n));
      dst = many.data();
    }
    const Py_ssize_t got = each_i64(o, [&](Py_ssize_t i, int64_t x) { if (i < n) dst[i] = I(x); });
    if (got >= 0 && got != n) PyErr_SetString(PyExc_ValueError, "a list of integers changed while it was read");
    v = dst;
    return got == n;
  }
  const I* get() { return v; }
};
template <> struct Arg<const int32_t*> : HostArray<int32_t> {};
template <> struct Arg<const int64_t*> : HostArray<int64_t> {};
template <> struct Arg<hkStream_t> {
  void* v = nullptr;
  bool from(PyObject* o) {
    if (o == Py_None) return current_stream(&v);
    if (PyLong_Check(o)) {
      v = PyLong_AsVoidPtr(o);
      return !(v == nullptr && PyErr_Occurred());
    }
    PyObject* a = PyObject_GetAttr(o, s_value);
    if (a == nullptr) return false;
    if (a != Py_None) v = PyLong_AsVoidPtr(a);   // a null c_void_p holds None: the null stream
    Py_DECREF(a);
    return !(v == nullptr && PyErr_Occurred());
  }
  hkStream_t get() { return static_cast<hkStream_t>(v); }
};
template <> struct Arg<HtArray*> {
  HtArray a;
  HtArray* p = nullptr;
  bool from(PyObject* o) {
    if (o == Py_None) return true;
    p = &a;
    PyObject* shape = PyObject_GetAttr(o, s_shape);
    if (shape == nullptr) return false;
    Py_ssize_t n = PySequence_Size(shape);
    if (n > HT_C_MAX_NDIM) {
      Py_DECREF(shape);
      PyErr_Format(PyExc_AssertionError, "an array of %zd dimensions, at most %d are taken", n, HT_C_MAX_NDIM);
      return false;
    }
    n = n < 0 ? n : each_i64(shape, [&](Py_ssize_t i, int64_t x) { if (i < n) a.shape[i] = x; });
    Py_DECREF(shape);
    if (n < 0) return false;
    a.ndim = int32_t(n);
    PyObject* stride = PyObject_CallMethodNoArgs(o, s_stride);
    if (stride == nullptr) return false;
    const Py_ssize_t k = each_i64(stride, [&](Py_ssize_t i, int64_t x) { if (i < n) a.stride[i] = x; });
    Py_DECREF(stride);
    if (k < 0 || !to_address(o, &a.data)) return false;
    a.dtype = dtype_code_of(o);
    if (a.dtype < 0) return false;
    PyObject* cuda = PyObject_GetAttr(o, s_is_cuda);
    if (cuda == nullptr) return false;
    const int on = PyObject_IsTrue(cuda);
    Py_DECREF(cuda);
    if (on < 0) return false;
    a.device_type = on ? HT_DEVICE_ACCEL : HT_DEVICE_CPU;
    a.device_index = 0;
    if (on) {
      PyObject* dev = PyObject_CallMethodNoArgs(o, s_get_device);
      if (dev == nullptr) return false;
      int64_t index = 0;
      const bool ok = to_i64(dev, &index);
      Py_DECREF(dev);
      if (!ok) return false;
      a.device_index = int32_t(index);
    }
    return true;
  }
  HtArray* get() { return p; }
};
template <> struct Arg<const HtArray*> : Arg<HtArray*> {};

// LABELS: the entry point's int64 array is one of labels on the device, a tensor, and never one on the host
template <auto F, bool LABELS> struct Entry;
template <typename... A, int (*F)(A...), bool LABELS> struct Entry<F, LABELS> {
  template <typename T>
  using ArgOf = std::conditional_t<LABELS && std::is_same_v<T, const int64_t*>, PointerArg<const int64_t*>, Arg<T>>;
  template <size_t... I>
  static PyObject* run(PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<ArgOf<A>...> conv;
    try {
      if (!(std::get<I>(conv).from(args[I]) && ...)) return nullptr;
    } catch (const std::bad_alloc&) {
      return PyErr_NoMemory();
    }
    int rc = 0;
    const char* thrown = nullptr;   // an exception of the entry point ends before the lock is taken again
    char text[256];
    bool no_memory = false;
    Py_BEGIN_ALLOW_THREADS
    try {
      rc = F(std::get<I>(conv).get()...);
    } catch (const std::bad_alloc&) {
      no_memory = true;
    } catch (const std::exception& e) {
      std::snprintf(text, sizeof text, "%s", e.what());
      thrown = text;
    } catch (...) {
      thrown = "an entry point ended with an exception";
    }
    Py_END_ALLOW_THREADS
    if (no_memory) return PyErr_NoMemory();
    if (thrown != nullptr) {
      PyErr_SetString(PyExc_RuntimeError, thrown);
      return nullptr;
    }
    return PyLong_FromLong(rc);
  }
  static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != Py_ssize_t(sizeof...(A))) {
      PyErr_Format(PyExc_TypeError, "%zd arguments are expected, %zd given", Py_ssize_t(sizeof...(A)), n);
      return nullptr;
    }
    return run(args, std::index_sequence_for<A...>{});
  }
};

#ifndef HT_CALL
// the entry points that take a block of parameters, with its members as arguments
int dropout_fwd_ex(int itype, int rtype, int wtype, int64_t rows, int64_t cols, int64_t x0_numrows, int64_t z_numrows,
                   const void* x0, const void* x1, const void* residual, const void* gamma, const void* beta,
                   const void* gamma1, const void* beta1, const void* rowscale, const void* colscale, const void* x0_subset,
                   const void* z_subset, void* z, void* z1, void* x, uint8_t* dmask, uint8_t* dmask1, float* mu, float* rs,
                   float dropout_p, float epsilon, float rowscale_const, int is_rms_norm, uint64_t seed, uint64_t offset,
                   hkStream_t stream) {
  const hkDropoutAddLnFwdParams p = {itype, rtype, wtype, rows, cols, x0_numrows, z_numrows, x0, x1, residual, gamma, beta,
                                     gamma1, beta1, rowscale, colscale, static_cast<const int32_t*>(x0_subset),
                                     static_cast<const int32_t*>(z_subset), z, z1, x, dmask, dmask1, mu, rs, dropout_p,
                                     epsilon, rowscale_const, is_rms_norm, seed, offset};
  return hk_dropout_add_ln_fwd_ex(&p, stream);
}
int dropout_bwd_ex(int itype, int rtype, int wtype, int64_t rows, int64_t cols, int64_t x0_numrows, int64_t z_numrows,
                   const void* dz, const void* dz1, const void* dx, const void* x, const void* x0, const uint8_t* dmask,
                   const uint8_t* dmask1, const float* mu, const float* rs, const void* gamma, const void* gamma1,
                   const void* rowscale, const void* colscale, const void* x0_subset, const void* z_subset, void* dx0,
                   void* dx1, void* dresidual, void* dgamma, void* dbeta, void* dgamma1, void* dbeta1, void* dcolscale,
                   void* workspace, size_t workspace_bytes, float dropout_p, float rowscale_const, int is_rms_norm,
                   hkStream_t stream) {
  const hkDropoutAddLnBwdParams p = {itype, rtype, wtype, rows, cols, x0_numrows, z_numrows, dz, dz1, dx, x, x0, dmask,
                                     dmask1, mu, rs, gamma, gamma1, rowscale, colscale,
                                     static_cast<const int32_t*>(x0_subset), static_cast<const int32_t*>(z_subset), dx0,
                                     dx1, dresidual, dgamma, dbeta, dgamma1, dbeta1, dcolscale, workspace, workspace_bytes,
                                     dropout_p, rowscale_const, is_rms_norm};
  return hk_dropout_add_ln_bwd_ex(&p, stream);
}

#endif

// dense(a, b, ...): whether every operand is None or contiguous
PyObject* dense(PyObject*, PyObject* const* args, Py_ssize_t n) {
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (args[i] == Py_None) continue;
    PyObject* c = PyObject_CallMethodNoArgs(args[i], s_is_contiguous);
    if (c == nullptr) return nullptr;
    const int yes = PyObject_IsTrue(c);
    Py_DECREF(c);
    if (yes < 0) return nullptr;
    if (!yes) Py_RETURN_FALSE;
  }
  Py_RETURN_TRUE;
}

// rows_cols(t): (elements / last dimension, last dimension); no rows where there are no elements
PyObject* rows_cols(PyObject*, PyObject* t) {
  PyObject* shape = PyObject_GetAttr(t, s_shape);
  if (shape == nullptr) return nullptr;
  int64_t rows = 1, cols = 1;
  const Py_ssize_t n = each_i64(shape, [&](Py_ssize_t, int64_t v) { rows *= cols; cols = v; });
  Py_DECREF(shape);
  if (n < 0) return nullptr;
  if (n == 0) {
    PyErr_SetString(PyExc_IndexError, "an operand has at least one dimension");
    return nullptr;
  }
  return Py_BuildValue("LL", (long long)(cols == 0 ? 0 : rows), (long long)cols);
}

PyObject* setup(PyObject*, PyObject* args) {
  return PyArg_ParseTuple(args, "OOOO", &g_dtype_codes, &g_current_stream, &g_get_device, &g_raw_stream)
             ? (Py_INCREF(g_dtype_codes), Py_INCREF(g_current_stream), Py_INCREF(g_get_device), Py_INCREF(g_raw_stream),
                Py_INCREF(Py_None), Py_None)
             : nullptr;
}

#define ENTRY(name) {#name, (PyCFunction)(void (*)())Entry<&name, false>::call, METH_FASTCALL, nullptr}
#define LABELS(name) {#name, (PyCFunction)(void (*)())Entry<&name, true>::call, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"setup", setup, METH_VARARGS, nullptr},
    {"dense", (PyCFunction)(void (*)())dense, METH_FASTCALL, nullptr},
    {"rows_cols", rows_cols, METH_O, nullptr},
#ifndef HT_CALL
    ENTRY(dropout_fwd_ex), ENTRY(dropout_bwd_ex), ENTRY(hk_batch_norm_bwd), ENTRY(hk_batch_norm_fwd),
    ENTRY(hk_binary_const), ENTRY(hk_dropout_add_ln_bwd_pitched), ENTRY(hk_dropout_add_ln_fwd_pitched),
    ENTRY(hk_layer_norm_bwd_pitched), ENTRY(hk_layer_norm_fwd_pitched), ENTRY(hk_reduce), ENTRY(hk_sce_dense_bwd),
    ENTRY(hk_sce_dense_bwd_reduced), ENTRY(hk_sce_dense_fwd), LABELS(hk_sce_sparse_bwd_pitched),
    LABELS(hk_sce_sparse_bwd_reduced), LABELS(hk_sce_sparse_fwd_pitched), ENTRY(hk_softmax_bwd),
    ENTRY(hk_softmax_bwd_pitched), ENTRY(hk_softmax_fwd), ENTRY(hk_softmax_fwd_pitched), ENTRY(hk_unary),
#else
    ENTRY(ht_batch_norm), ENTRY(ht_batch_norm_gradient), ENTRY(ht_binary), ENTRY(ht_binary_const),
    ENTRY(ht_broadcast_shape), ENTRY(ht_dropout_add_ln_bwd), ENTRY(ht_dropout_add_ln_fwd),
    ENTRY(ht_dropout_add_ln_parallel_residual_bwd), ENTRY(ht_dropout_add_ln_parallel_residual_fwd),
    ENTRY(ht_fused_layer_norm), ENTRY(ht_fused_layer_norm_gradient), ENTRY(ht_instance_norm),
    ENTRY(ht_instance_norm_gradient), ENTRY(ht_layer_norm), ENTRY(ht_layer_norm_gradient), ENTRY(ht_ndarray_binary),
    ENTRY(ht_ndarray_layernorm), ENTRY(ht_ndarray_norm), ENTRY(ht_ndarray_reduce), ENTRY(ht_ndarray_sceloss),
    ENTRY(ht_ndarray_softmax), ENTRY(ht_ndarray_unary), ENTRY(ht_nll_loss), ENTRY(ht_nll_loss_gradient), ENTRY(ht_norm),
    ENTRY(ht_norm_gradient), ENTRY(ht_reduce), ENTRY(ht_reduce_gradient), ENTRY(ht_sceloss_gradient),
    ENTRY(ht_set_random_seed), ENTRY(ht_softmax), ENTRY(ht_softmax_cross_entropy),
    ENTRY(ht_softmax_cross_entropy_gradient), ENTRY(ht_softmax_cross_entropy_sparse),
    ENTRY(ht_softmax_cross_entropy_sparse_gradient), ENTRY(ht_softmax_gradient), ENTRY(ht_unary),
    ENTRY(ht_vocab_parallel_cross_entropy), ENTRY(ht_vocab_parallel_cross_entropy_gradient),
#endif
    {nullptr, nullptr, 0, nullptr}};

#ifndef HT_CALL
#define MODULE_INIT PyInit_hk_call
#define MODULE_NAME "hk_call"
#else
#define MODULE_INIT PyInit_ht_call
#define MODULE_NAME "ht_call"
#endif
PyModuleDef module = {PyModuleDef_HEAD_INIT, MODULE_NAME, nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC MODULE_INIT(void) {
  const std::pair<PyObject**, const char*> names[] = {
      {&s_data_ptr, "data_ptr"}, {&s_is_contiguous, "is_contiguous"}, {&s_shape, "shape"}, {&s_stride, "stride"},
      {&s_dtype, "dtype"}, {&s_is_cuda, "is_cuda"}, {&s_get_device, "get_device"}, {&s_value, "value"}};
  for (const auto& n : names)
    if ((*n.first = PyUnicode_InternFromString(n.second)) == nullptr) return nullptr;
  pthread_atfork(nullptr, nullptr, [] { g_initialised = false; });
  return PyModule_Create(&module);
}

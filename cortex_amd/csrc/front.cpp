// front.cpp -- the parts of the Python front end that every call passes through, as a CPython extension: the shape algebra
// of plain integers (dimensions.py), the ct_dims of a call and the call of an entry point itself.
//
// A small call from Python (a bias over 128 x 784: a kernel of 2.8 us behind a launch of 2.5 to 3) spent twice that in the
// interpreter: tuples built as keys of tables, lists built of what the tables held, ctypes' conversion of a dozen
// arguments.  Here a function reads the lists as they are and builds its result once; nothing is kept between calls.
// The bias takes 6.4 us a call, 9.1 in Python and ctypes; the 25 calls of a digit network's training step 170, 241 before.
// Each takes what it can decide, exact ints whose products fit 64 bits, and hands everything else (index tensors, other
// number types, shapes that are refused) to the Python function that it stands in for.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/cortex_hip.h"

namespace {

constexpr Py_ssize_t kMost = 8;   // dimensions

PyObject *s_shape, *s_strides, *s_max_shape, *s_dimensions, *s_lib;

struct Plain {
  Py_ssize_t n;
  int64_t shape[kMost], strides[kMost];
};

// The exact ints of a list or tuple; -1 for anything else.
Py_ssize_t read_ints(PyObject* seq, int64_t* out) {
  Py_ssize_t n;
  PyObject** items;
  if (PyList_CheckExact(seq)) {
    n = PyList_GET_SIZE(seq);
    items = reinterpret_cast<PyListObject*>(seq)->ob_item;
  } else if (PyTuple_CheckExact(seq)) {
    n = PyTuple_GET_SIZE(seq);
    items = reinterpret_cast<PyTupleObject*>(seq)->ob_item;
  } else {
    return -1;
  }
  if (n > kMost) return -1;
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (!PyLong_CheckExact(items[i])) return -1;
    int overflow = 0;
    out[i] = PyLong_AsLongLongAndOverflow(items[i], &overflow);
    if (overflow) return -1;
  }
  return n;
}

bool read_shape(PyObject* dims, Plain* p) {
  if (!PyDict_CheckExact(dims)) return false;
  PyObject* shape = PyDict_GetItem(dims, s_shape);
  return shape && (p->n = read_ints(shape, p->shape)) >= 0;
}

// Shape and strides, as many of the one as of the other.
bool read_dims(PyObject* dims, Plain* p) {
  if (!read_shape(dims, p)) return false;
  PyObject* strides = PyDict_GetItem(dims, s_strides);
  return strides && read_ints(strides, p->strides) == p->n;
}

bool multiply(int64_t a, int64_t b, int64_t* out) { return !__builtin_mul_overflow(a, b, out); }

bool product(const int64_t* v, Py_ssize_t n, int64_t* out) {
  int64_t r = 1;
  for (Py_ssize_t i = 0; i < n; ++i)
    if (!multiply(r, v[i], &r)) return false;
  *out = r;
  return true;
}

PyObject* list_of(const int64_t* v, Py_ssize_t n) {
  PyObject* list = PyList_New(n);
  if (!list) return nullptr;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* item = PyLong_FromLongLong(v[i]);
    if (!item) {
      Py_DECREF(list);
      return nullptr;
    }
    PyList_SET_ITEM(list, i, item);
  }
  return list;
}

// {key_a: a, key_b: b}; takes both references.
PyObject* dict_of(PyObject* key_a, PyObject* a, PyObject* key_b, PyObject* b) {
  PyObject* d = a && b ? PyDict_New() : nullptr;
  if (d && (PyDict_SetItem(d, key_a, a) || PyDict_SetItem(d, key_b, b))) Py_CLEAR(d);
  Py_XDECREF(a);
  Py_XDECREF(b);
  return d;
}

PyObject* dims_of(const int64_t* shape, const int64_t* strides, Py_ssize_t n) {
  return dict_of(s_shape, list_of(shape, n), s_strides, list_of(strides, n));
}

// dimensions._dense_plain; 1, 0, or -1 where that hands on.
int dense_plain(const Plain& p) {
  if (p.n == 1) return p.strides[0] == 1;
  int64_t count = 1, largest = 0, extent = 1;
  bool any = false;
  for (Py_ssize_t i = 0; i < p.n; ++i) {
    if (p.shape[i] == 1) continue;
    if (!multiply(count, p.shape[i], &count)) return -1;
    if (!any || p.strides[i] > largest) {
      largest = p.strides[i];
      extent = p.shape[i];
      any = true;
    }
  }
  if (count == 0) return -1;
  int64_t span;
  if (any && !multiply(largest, extent, &span)) return -1;
  return any && span == count;
}

// Shapes and strides brought to one rank (dimensions._max_shape_direct).
struct Aligned {
  Py_ssize_t rank;
  int64_t max_shape[kMost];
  Plain dims[4];
};

bool align(PyObject* const* args, Py_ssize_t n, Aligned* a) {
  if (n < 1 || n > 4) return false;
  a->rank = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (!read_dims(args[i], &a->dims[i]) || a->dims[i].n == 0) return false;
    if (a->dims[i].n > a->rank) a->rank = a->dims[i].n;
  }
  for (Py_ssize_t d = 0; d < a->rank; ++d) a->max_shape[d] = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    Plain& p = a->dims[i];
    const Py_ssize_t pad = a->rank - p.n;
    if (pad) {
      Py_ssize_t at = 0;
      for (Py_ssize_t d = 1; d < p.n; ++d)
        if (p.strides[d] > p.strides[at]) at = d;
      int64_t outer;
      if (!multiply(p.strides[at], p.shape[at], &outer)) return false;
      memmove(p.shape + pad, p.shape, sizeof(int64_t) * p.n);
      memmove(p.strides + pad, p.strides, sizeof(int64_t) * p.n);
      for (Py_ssize_t d = 0; d < pad; ++d) {
        p.shape[d] = 1;
        p.strides[d] = outer;
      }
      p.n = a->rank;
    }
    for (Py_ssize_t d = 0; d < a->rank; ++d)
      if (p.shape[d] > a->max_shape[d]) a->max_shape[d] = p.shape[d];
  }
  return true;
}

// ------------------------------------------------------------------ what stands in for functions of dimensions.py

enum Function { kDirectKey, kEcount, kShape, kDense, kAccessIncreasing, kMaxShape, kCommensurate, kTo2d, kToBatch, kAs2d,
                kAsBatch, kDimsRef, kCall, kFunctions };
PyObject* g_python[kFunctions];   // the functions that these stand in for

PyObject* hand_on(Function f, PyObject* const* args, Py_ssize_t n) {
  return PyObject_Vectorcall(g_python[f], args, n, nullptr);
}

PyObject* direct_key(PyObject*, PyObject* const* args, Py_ssize_t n) {
  PyObject* key = PyTuple_New(n);
  if (!key) return nullptr;
  Plain p;
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (!PyDict_CheckExact(args[i])) break;
    PyObject* parts[2] = {PyDict_GetItem(args[i], s_shape), PyDict_GetItem(args[i], s_strides)};
    if (!parts[0] || !parts[1] || read_ints(parts[0], p.shape) < 0 || read_ints(parts[1], p.strides) < 0) break;
    PyObject* pair = PyTuple_New(2);
    if (!pair) {
      Py_DECREF(key);
      return nullptr;
    }
    PyTuple_SET_ITEM(key, i, pair);
    for (int k = 0; k < 2; ++k) {
      PyObject* t = PySequence_Tuple(parts[k]);
      if (!t) {
        Py_DECREF(key);
        return nullptr;
      }
      PyTuple_SET_ITEM(pair, k, t);
    }
  }
  if (n == 0 || PyTuple_GET_ITEM(key, n - 1)) return key;
  Py_DECREF(key);
  return hand_on(kDirectKey, args, n);
}

PyObject* ecount(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Plain p;
  int64_t count;
  if (n != 1 || !read_shape(args[0], &p) || !product(p.shape, p.n, &count)) return hand_on(kEcount, args, n);
  return PyLong_FromLongLong(count);
}

PyObject* shape(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Plain p;
  if (n != 1 || !read_shape(args[0], &p)) return hand_on(kShape, args, n);
  return list_of(p.shape, p.n);
}

PyObject* dense(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Plain p;
  const int known = n == 1 && read_dims(args[0], &p) && p.n > 0 ? dense_plain(p) : -1;
  return known < 0 ? hand_on(kDense, args, n) : PyBool_FromLong(known);
}

PyObject* access_increasing(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Plain p;
  if (n != 1 || !read_dims(args[0], &p)) return hand_on(kAccessIncreasing, args, n);
  for (Py_ssize_t i = 0; i + 1 < p.n; ++i)
    if (p.strides[i] < p.strides[i + 1]) Py_RETURN_FALSE;
  Py_RETURN_TRUE;
}

PyObject* max_shape(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Aligned a;
  if (!align(args, n, &a)) return hand_on(kMaxShape, args, n);
  PyObject* list = PyList_New(n);
  if (!list) return nullptr;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* d = dims_of(a.dims[i].shape, a.dims[i].strides, a.rank);
    if (!d) {
      Py_DECREF(list);
      return nullptr;
    }
    PyList_SET_ITEM(list, i, d);
  }
  return dict_of(s_max_shape, list_of(a.max_shape, a.rank), s_dimensions, list);
}

// Whether the dimensions are plain and every one divides the largest.
PyObject* commensurate(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Aligned a;
  if (!align(args, n, &a)) return hand_on(kCommensurate, args, n);
  for (Py_ssize_t i = 0; i < n; ++i)
    for (Py_ssize_t d = 0; d < a.rank; ++d)
      if (a.dims[i].shape[d] < 1 || a.max_shape[d] % a.dims[i].shape[d] != 0) return hand_on(kCommensurate, args, n);
  Py_RETURN_TRUE;
}

bool matrix_shape(const Plain& p, bool batch, int64_t* out) {
  if (p.n == 0) return false;
  out[0] = 1;
  out[1] = p.shape[0];
  if (p.n == 1) return true;
  if (batch) {
    out[0] = p.shape[0];
    return product(p.shape + 1, p.n - 1, out + 1);
  }
  out[1] = p.shape[p.n - 1];
  return product(p.shape, p.n - 1, out);
}

template <bool kBatch>
PyObject* to_matrix_shape(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Plain p;
  int64_t m[2];
  if (n != 1 || !read_shape(args[0], &p) || !matrix_shape(p, kBatch, m)) return hand_on(kBatch ? kToBatch : kTo2d, args, n);
  return list_of(m, 2);
}

// A packed tensor as a matrix; others are reshaped in Python.
template <bool kBatch>
PyObject* as_matrix(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Plain p;
  int64_t m[2];
  bool packed = n == 1 && read_dims(args[0], &p) && matrix_shape(p, kBatch, m) && m[0] >= 1 && m[1] >= 1;
  for (Py_ssize_t i = 0; packed && i + 1 < p.n; ++i) packed = p.strides[i] >= p.strides[i + 1];
  if (!packed || dense_plain(p) != 1) return hand_on(kBatch ? kAsBatch : kAs2d, args, n);
  const int64_t strides[2] = {m[1], 1};
  return dims_of(m, strides, 2);
}

// ------------------------------------------------------------------ calls

// The ct_dims of directly addressed dimensions, as bytes.
PyObject* dims_ref(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Plain p;
  if (n != 1 || !read_dims(args[0], &p) || p.n < 1) return hand_on(kDimsRef, args, n);
  static_assert(sizeof(ct_dims::shape) == sizeof(int64_t) * kMost && sizeof(ct_dims::strides) == sizeof(int64_t) * kMost,
                "a ct_dims holds eight dimensions of 64 bits");
  PyObject* bytes = PyBytes_FromStringAndSize(nullptr, sizeof(ct_dims));
  if (!bytes) return nullptr;
  ct_dims* d = reinterpret_cast<ct_dims*>(PyBytes_AS_STRING(bytes));
  memset(d, 0, sizeof(*d));
  d->ndim = (int32_t)p.n;
  memcpy(d->shape, p.shape, sizeof(int64_t) * p.n);
  memcpy(d->strides, p.strides, sizeof(int64_t) * p.n);
  return bytes;
}

// Arguments as ctypes converts them: integers are cut to their type, an address is an int, None or (the struct itself) bytes.
template <class T>
bool convert(PyObject* o, T* out) {
  if constexpr (std::is_pointer<T>::value) {
    if (o == Py_None) {
      *out = nullptr;
      return true;
    }
    if (PyLong_CheckExact(o)) {
      const unsigned long long v = PyLong_AsUnsignedLongLongMask(o);
      if (v == (unsigned long long)-1 && PyErr_Occurred()) return PyErr_Clear(), false;
      *out = reinterpret_cast<T>(v);
      return std::is_void<typename std::remove_pointer<T>::type>::value;
    }
    if (PyBytes_CheckExact(o) && std::is_same<T, const ct_dims*>::value && PyBytes_GET_SIZE(o) == sizeof(ct_dims)) {
      *out = reinterpret_cast<T>(PyBytes_AS_STRING(o));
      return true;
    }
    return false;
  } else if constexpr (std::is_floating_point<T>::value) {
    if (!PyFloat_CheckExact(o)) return false;
    *out = PyFloat_AS_DOUBLE(o);
    return true;
  } else {
    if (!PyLong_CheckExact(o)) return false;
    const unsigned long long v = PyLong_AsUnsignedLongLongMask(o);
    if (v == (unsigned long long)-1 && PyErr_Occurred()) return PyErr_Clear(), false;
    *out = (T)v;
    return true;
  }
}

template <class... A, size_t... I>
bool invoke(int (*f)(A...), PyObject* const* args, int* status, std::index_sequence<I...>) {
  std::tuple<A...> values;
  if (!(convert(args[I], &std::get<I>(values)) && ...)) return false;
  Py_BEGIN_ALLOW_THREADS
  *status = f(std::get<I>(values)...);
  Py_END_ALLOW_THREADS
  return true;
}

// Whether the arguments were ones that this converts; then the call has been made.
template <class... A>
bool invoke_at(void* address, int (*)(A...), PyObject* const* args, Py_ssize_t n, int* status) {
  if (n != (Py_ssize_t)sizeof...(A)) return false;
  return invoke(reinterpret_cast<int (*)(A...)>(address), args, status, std::index_sequence_for<A...>());
}

struct Entry {
  const char* name;
  bool (*invoke)(void* address, PyObject* const* args, Py_ssize_t n, int* status);
  void* address;
};
#define CT_ENTRY(f)                                                                                                   \
  {#f, [](void* at, PyObject* const* args, Py_ssize_t n, int* status) {                                              \
     return invoke_at(at, static_cast<decltype(&f)>(nullptr), args, n, status);                                      \
   }, nullptr}
Entry g_entries[] = {
    CT_ENTRY(ct_memcpy_async), CT_ENTRY(ct_memset), CT_ENTRY(ct_assign_constant), CT_ENTRY(ct_assign), CT_ENTRY(ct_unary_accum),
    CT_ENTRY(ct_unary_op), CT_ENTRY(ct_binary_accum_constant), CT_ENTRY(ct_binary_op_constant), CT_ENTRY(ct_binary_accum),
    CT_ENTRY(ct_binary_op), CT_ENTRY(ct_ternary_op), CT_ENTRY(ct_unary_reduce), CT_ENTRY(ct_activation_gradient),
    CT_ENTRY(ct_softmax_eltwise), CT_ENTRY(ct_softmax_spatial), CT_ENTRY(ct_batch_normalize_update_and_apply_eltwise),
    CT_ENTRY(ct_batch_normalize_update_and_apply_spatial), CT_ENTRY(ct_batch_normalize_gradients_eltwise),
    CT_ENTRY(ct_batch_normalize_gradients_spatial), CT_ENTRY(ct_gemm), CT_ENTRY(ct_gemv), CT_ENTRY(ct_rand),
    CT_ENTRY(ct_dropout_bernoulli_mask), CT_ENTRY(ct_adam_step), CT_ENTRY(ct_adadelta_step), CT_ENTRY(ct_lrn_forward),
    CT_ENTRY(ct_lrn_backward)};
PyObject* g_index;     // name -> index of an entry whose address is known
PyObject* g_library;   // the library that the addresses are of

// Whether capi's library is the one whose addresses are known: a program may put another in its place.
bool bound_library() {
  PyObject* python = g_python[kCall];
  return g_library && PyFunction_Check(python) && PyDict_GetItem(PyFunction_GET_GLOBALS(python), s_lib) == g_library;
}

// capi.call; `check` is called with a status that is not zero, and raises.
PyObject* g_check;
PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
  PyObject* at = n > 0 && PyUnicode_CheckExact(args[0]) ? PyDict_GetItem(g_index, args[0]) : nullptr;
  if (at && bound_library()) {
    const Entry& e = g_entries[PyLong_AsLong(at)];
    int status = 0;
    if (e.invoke(e.address, args + 1, n - 1, &status)) {
      if (status == 0) Py_RETURN_NONE;
      return PyObject_CallFunction(g_check, "i", status);
    }
  }
  return hand_on(kCall, args, n);
}

// bind(library, name, address): whether the entry point is one that `call` knows.  The addresses of one library are known at a
// time.
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 3 || !PyUnicode_Check(args[1])) return PyErr_SetString(PyExc_TypeError, "bind(library, name, address)"), nullptr;
  if (args[0] != g_library) {
    PyDict_Clear(g_index);
    Py_INCREF(args[0]);
    Py_XSETREF(g_library, args[0]);
  }
  for (size_t i = 0; i < sizeof(g_entries) / sizeof(g_entries[0]); ++i)
    if (PyUnicode_CompareWithASCIIString(args[1], g_entries[i].name) == 0) {
      g_entries[i].address = PyLong_AsVoidPtr(args[2]);
      if (PyErr_Occurred()) return nullptr;
      PyObject* at = PyLong_FromSize_t(i);
      const int rc = at ? PyDict_SetItem(g_index, args[1], at) : -1;
      Py_XDECREF(at);
      if (rc) return nullptr;
      Py_RETURN_TRUE;
    }
  Py_RETURN_FALSE;
}

template <class F> PyCFunction as_method(F f) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(f)); }

// Arguments by name are for the Python function.
template <Function kWhich, PyObject* (*kNative)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* entry(PyObject* self, PyObject* const* args, Py_ssize_t n, PyObject* names) {
  return names ? PyObject_Vectorcall(g_python[kWhich], args, n, names) : kNative(self, args, n);
}

PyMethodDef g_functions[kFunctions + 1] = {
    {"direct_key", as_method(entry<kDirectKey, direct_key>), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"ecount", as_method(entry<kEcount, ecount>), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"shape", as_method(entry<kShape, shape>), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"dense", as_method(entry<kDense, dense>), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"access_increasing", as_method(entry<kAccessIncreasing, access_increasing>), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"dimension_seq_to_max_shape", as_method(entry<kMaxShape, max_shape>), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"commensurate_dims", as_method(entry<kCommensurate, commensurate>), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"to_2d_shape", as_method(entry<kTo2d, to_matrix_shape<false>>), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"to_batch_shape", as_method(entry<kToBatch, to_matrix_shape<true>>), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"as_2d", as_method(entry<kAs2d, as_matrix<false>>), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"as_batch", as_method(entry<kAsBatch, as_matrix<true>>), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"dims_ref", as_method(entry<kDimsRef, dims_ref>), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"call", as_method(entry<kCall, call>), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {nullptr, nullptr, 0, nullptr}};

// stand_in(function[, check]): the function of this module of that function's name (without a leading underscore), which hands
// on to it what it does not take.
PyObject* stand_in(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n < 1 || n > 2) return PyErr_SetString(PyExc_TypeError, "stand_in(function[, check])"), nullptr;
  PyObject* name = PyObject_GetAttrString(args[0], "__name__");
  if (!name) return nullptr;
  const char* text = PyUnicode_AsUTF8(name);
  PyObject* result = nullptr;
  for (int f = 0; text && f < kFunctions; ++f)
    if (strcmp(g_functions[f].ml_name, text + (text[0] == '_')) == 0) {
      Py_INCREF(args[0]);
      Py_XSETREF(g_python[f], args[0]);
      if (f == kCall) {
        if (n != 2) break;
        Py_INCREF(args[1]);
        Py_XSETREF(g_check, args[1]);
      }
      result = PyCFunction_New(&g_functions[f], nullptr);
    }
  if (!result && !PyErr_Occurred()) PyErr_Format(PyExc_KeyError, "nothing stands in for %S", name);
  Py_DECREF(name);
  return result;
}

PyMethodDef g_module_methods[] = {{"stand_in", as_method(stand_in), METH_FASTCALL, nullptr},
                                  {"bind", as_method(bind), METH_FASTCALL, nullptr},
                                  {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_front", nullptr, -1, g_module_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__front() {
  s_shape = PyUnicode_InternFromString("shape");
  s_strides = PyUnicode_InternFromString("strides");
  s_max_shape = PyUnicode_InternFromString("max-shape");
  s_dimensions = PyUnicode_InternFromString("dimensions");
  s_lib = PyUnicode_InternFromString("_lib");
  g_index = PyDict_New();
  return s_shape && s_strides && s_max_shape && s_dimensions && s_lib && g_index ? PyModule_Create(&g_module) : nullptr;
}

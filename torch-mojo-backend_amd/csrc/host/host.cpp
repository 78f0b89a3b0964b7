// The host side of an eager op in native code: making mojo tensors, and
// calling the kernel library without ctypes' per-argument conversions.
//
// An eager op is a few microseconds of host work around a kernel of a few
// microseconds, so at small sizes the host sets the pace.  Per op this module
// takes over what every op does: the wrapper tensor with its attributes
// (2.1 -> 1.2 us), the output allocation (3.7 -> 2.6 us), metadata views, and
// the call itself (a 25-argument GEMM call 1.9 -> 0.3 us).
//
// Kernel entry points are bound by address (bind()), each with the parameter
// types that the C header declares.  Arguments convert as in ctypes: None or
// an integer for a pointer, integers, floats; an array parameter also takes a
// tuple or list of numbers, or an object with a buffer (a ctypes array).  The
// GIL is released around the call.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>
#include <string.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "../../../include/mi355x_kernels.h"

#ifndef MI355X_SOURCE_HASH
#define MI355X_SOURCE_HASH "unknown"
#endif

namespace {

constexpr int kMaxRank = 64;   // of a view (torch's own limit)
constexpr int kAllocRank = 8;  // of an allocated mojo tensor
constexpr int kMaxArray = 64;  // numbers in a tuple argument

// ---------------------------------------------------------------------------
// kernel calls
// ---------------------------------------------------------------------------
bool as_i64(PyObject* o, int64_t* v) {
  if (PyLong_CheckExact(o)) {
    *v = PyLong_AsLongLong(o);
  } else {
    PyObject* i = PyNumber_Index(o);
    if (!i) return false;
    *v = PyLong_AsLongLong(i);
    Py_DECREF(i);
  }
  return *v != -1 || !PyErr_Occurred();
}

bool as_ptr(PyObject* o, void** v) {
  if (o == Py_None) {
    *v = nullptr;
    return true;
  }
  if (!PyLong_Check(o)) {
    PyErr_Format(PyExc_TypeError, "expected an address or None, got %s", Py_TYPE(o)->tp_name);
    return false;
  }
  *v = PyLong_AsVoidPtr(o);
  return *v || !PyErr_Occurred();
}

// One converted argument of parameter type T.
template <class T, class = void>
struct Arg;

template <class T>
struct Arg<T, std::enable_if_t<std::is_integral<T>::value>> {
  T v;
  bool set(PyObject* o) {
    int64_t x;
    if (!as_i64(o, &x)) return false;
    v = (T)x;
    return true;
  }
};

template <>
struct Arg<double> {
  double v;
  bool set(PyObject* o) {
    v = PyFloat_AsDouble(o);
    return v != -1.0 || !PyErr_Occurred();
  }
};

template <class T>
struct Arg<T*> {
  typedef std::remove_const_t<T> E;
  static constexpr bool kNumbers = std::is_same<E, int64_t>::value || std::is_same<E, int>::value ||
                                   std::is_same<E, double>::value || std::is_pointer<E>::value;
  T* v;
  Py_buffer view;
  bool held = false;
  std::conditional_t<kNumbers, E, char> items[kNumbers ? kMaxArray : 1];

  bool set(PyObject* o) {
    if (o == Py_None || PyLong_Check(o)) {
      void* p;
      if (!as_ptr(o, &p)) return false;
      v = (T*)p;
      return true;
    }
    if constexpr (kNumbers) {
      if (PyTuple_Check(o) || PyList_Check(o)) {
        const Py_ssize_t n = PySequence_Fast_GET_SIZE(o);
        if (n > kMaxArray) {
          PyErr_Format(PyExc_ValueError, "an array argument of %zd numbers (at most %d)", n, kMaxArray);
          return false;
        }
        for (Py_ssize_t i = 0; i < n; ++i) {
          PyObject* e = PySequence_Fast_GET_ITEM(o, i);
          if constexpr (std::is_pointer<E>::value) {
            void* p;
            if (!as_ptr(e, &p)) return false;
            items[i] = (E)p;
          } else if constexpr (std::is_same<E, double>::value) {
            items[i] = PyFloat_AsDouble(e);
            if (items[i] == -1.0 && PyErr_Occurred()) return false;
          } else {
            int64_t x;
            if (!as_i64(e, &x)) return false;
            items[i] = (E)x;
          }
        }
        v = items;
        return true;
      }
    }
    if (PyObject_GetBuffer(o, &view, PyBUF_SIMPLE)) return false;
    held = true;
    v = (T*)view.buf;
    return true;
  }
  ~Arg() {
    if (held) PyBuffer_Release(&view);
  }
};

template <class Tag>
void* slot = nullptr;  // the bound entry point

template <class F, class Tag>
struct Call;

template <class... A, class R, class Tag>
struct Call<R (*)(A...), Tag> {
  template <size_t... I>
  static PyObject* go(PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<Arg<A>...> a;
    if (!(std::get<I>(a).set(args[I]) && ...)) return nullptr;
    R r;
    Py_BEGIN_ALLOW_THREADS;
    r = ((R(*)(A...))slot<Tag>)(std::get<I>(a).v...);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLongLong((long long)r);
  }
  static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != (Py_ssize_t)sizeof...(A)) {
      PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (%zd given)", Tag::name(), (Py_ssize_t)sizeof...(A), n);
      return nullptr;
    }
    if (!slot<Tag>) {
      PyErr_Format(PyExc_RuntimeError, "%s is not bound", Tag::name());
      return nullptr;
    }
    return go(args, std::index_sequence_for<A...>{});
  }
};

// Every entry point that returns an int or an int64_t.
#define KERNELS(X)                                                                                       \
  X(mi355x_copy) X(mi355x_fill) X(mi355x_arange) X(mi355x_map) X(mi355x_reduce_workspace_bytes)          \
  X(mi355x_reduce) X(mi355x_argreduce) X(mi355x_index_select) X(mi355x_embedding_fwd)                    \
  X(mi355x_embedding_bwd_workspace_bytes) X(mi355x_embedding_bwd) X(mi355x_embedding_bwd_accumulate)     \
  X(mi355x_layer_norm_fwd) X(mi355x_layer_norm_fwd_ex) X(mi355x_add_cast) X(mi355x_layer_norm_fwd_low)   \
  X(mi355x_layer_norm_fwd_add) X(mi355x_layer_norm_apply) X(mi355x_layer_norm_bwd_workspace_bytes)       \
  X(mi355x_layer_norm_bwd) X(mi355x_gelu_fwd) X(mi355x_gelu_bwd) X(mi355x_softmax_fwd)                   \
  X(mi355x_softmax_bwd) X(mi355x_nll_workspace_bytes) X(mi355x_nll_fwd) X(mi355x_nll_bwd)                \
  X(mi355x_cross_entropy_workspace_bytes) X(mi355x_cross_entropy_fwd) X(mi355x_cross_entropy_bwd)        \
  X(mi355x_cross_entropy_fwd_bwd) X(mi355x_fused_adamw) X(mi355x_fused_adamw_ex)                         \
  X(mi355x_foreach_norm_workspace_bytes) X(mi355x_foreach_norm) X(mi355x_foreach_apply)                  \
  X(mi355x_gemm_workspace_bytes) X(mi355x_gemm) X(mi355x_gemm_ex) X(mi355x_attn_fwd)                     \
  X(mi355x_rms_norm_fwd) X(mi355x_rms_norm_bwd) X(mi355x_rope) X(mi355x_geglu_fwd) X(mi355x_geglu_bwd)   \
  X(mi355x_attn_fwd_ex) X(mi355x_attn_bwd_workspace_bytes) X(mi355x_attn_bwd) X(mi355x_attn_fwd_gen)     \
  X(mi355x_attn_bwd_gen_workspace_bytes) X(mi355x_attn_bwd_gen) X(mi355x_attn_bwd_noalloc)

#define TAG(f)                                         \
  struct Tag_##f {                                     \
    static const char* name() { return #f; }           \
  };
KERNELS(TAG)
#undef TAG

struct Entry {
  const char* name;
  void** slot;
};
#define ENTRY(f) {#f, &slot<Tag_##f>},
const Entry kEntries[] = {KERNELS(ENTRY)};
#undef ENTRY

// bind(name, address): the kernel function behind `name`
PyObject* bind(PyObject*, PyObject* args) {
  const char* name;
  PyObject* addr;
  if (!PyArg_ParseTuple(args, "sO", &name, &addr)) return nullptr;
  for (const Entry& e : kEntries)
    if (!strcmp(e.name, name)) {
      if (!as_ptr(addr, e.slot)) return nullptr;
      Py_RETURN_TRUE;
    }
  Py_RETURN_FALSE;
}

// ---------------------------------------------------------------------------
// tensors
// ---------------------------------------------------------------------------
PyTypeObject* g_cls = nullptr;   // TorchMojoTensor
PyObject* g_wrap = nullptr;      // torch.Tensor._make_wrapper_subclass
PyObject* g_torch = nullptr;     // the torch module
PyObject* g_oom = nullptr;       // torch.OutOfMemoryError
PyObject* g_uint8 = nullptr;     // torch.uint8
PyObject* g_strided = nullptr;   // torch.strided
PyObject* g_storage = nullptr;   // device index -> the storage's torch.device
PyObject* g_torch_dev = nullptr; // device index -> torch.device("mojo", index)
PyObject* g_retry = nullptr;     // (size, device index): frees cached blocks and allocates again
PyObject* g_itemsize = nullptr;  // dict: dtype -> itemsize
PyObject *kw_wrap = nullptr, *kw_empty = nullptr;
PyObject *s_holder, *s_ptr, *s_shape, *s_strides, *s_offset, *s_dtype, *s_itemsize, *s_numel, *s_device, *s_tdev,
    *s_contig, *s_data_ptr, *s_empty;

constexpr int kDevices = 64;
PyObject* dev_storage[kDevices];
PyObject* dev_torch[kDevices];

// setup(cls, torch, storage_device, torch_device_of, retry_bytes, itemsizes)
PyObject* setup(PyObject*, PyObject* args) {
  PyObject *cls, *torch, *storage, *tdev, *retry, *sizes;
  if (!PyArg_ParseTuple(args, "OOOOOO", &cls, &torch, &storage, &tdev, &retry, &sizes)) return nullptr;
  PyObject* tensor = PyObject_GetAttrString(torch, "Tensor");
  if (!tensor) return nullptr;
  g_wrap = PyObject_GetAttrString(tensor, "_make_wrapper_subclass");
  Py_DECREF(tensor);
  g_oom = PyObject_GetAttrString(torch, "OutOfMemoryError");
  g_uint8 = PyObject_GetAttrString(torch, "uint8");
  g_strided = PyObject_GetAttrString(torch, "strided");
  if (!g_wrap || !g_oom || !g_uint8 || !g_strided) return nullptr;
  Py_INCREF(cls), Py_INCREF(torch), Py_INCREF(storage), Py_INCREF(tdev), Py_INCREF(retry), Py_INCREF(sizes);
  g_cls = (PyTypeObject*)cls, g_torch = torch, g_storage = storage, g_torch_dev = tdev, g_retry = retry;
  g_itemsize = sizes;
  Py_RETURN_NONE;
}

// forget the storage devices (tests switch where storages live)
PyObject* reset(PyObject*, PyObject*) {
  for (int i = 0; i < kDevices; ++i) Py_CLEAR(dev_storage[i]);
  Py_RETURN_NONE;
}

// Borrowed device object of `index` from its cache, filled by fn(index).
PyObject* device_of(PyObject** cache, PyObject* fn, int64_t index) {
  if (index < 0 || index >= kDevices) {
    PyErr_Format(PyExc_ValueError, "device index %lld", (long long)index);
    return nullptr;
  }
  if (!cache[index]) {
    PyObject* i = PyLong_FromLongLong(index);
    if (!i) return nullptr;
    cache[index] = PyObject_CallOneArg(fn, i);
    Py_DECREF(i);
  }
  return cache[index];
}

// A wrapper tensor with its attributes (new reference).  shape and strides
// are tuples of ints with `nd` items.
PyObject* make_impl(PyObject* holder, PyObject* ptr, PyObject* shape, PyObject* strides, PyObject* offset,
                    PyObject* dtype, PyObject* device, int64_t numel, bool contig) {
  const int64_t index = PyLong_AsLongLong(device);
  if (index == -1 && PyErr_Occurred()) return nullptr;
  PyObject* tdev = device_of(dev_torch, g_torch_dev, index);
  if (!tdev) return nullptr;
  PyObject* itemsize = PyDict_GetItemWithError(g_itemsize, dtype);
  if (!itemsize) {
    if (!PyErr_Occurred()) PyErr_Format(PyExc_TypeError, "unsupported dtype %R", dtype);
    return nullptr;
  }
  PyObject* args[] = {(PyObject*)g_cls, shape, strides, offset, dtype, g_strided, tdev};
  PyObject* t = PyObject_Vectorcall(g_wrap, args, 2, kw_wrap);
  if (!t) return nullptr;
  PyObject** dp = _PyObject_GetDictPtr(t);
  if (dp && !*dp) *dp = PyDict_New();
  PyObject* n = PyLong_FromLongLong(numel);
  if (!dp || !*dp || !n || PyDict_SetItem(*dp, s_holder, holder) || PyDict_SetItem(*dp, s_ptr, ptr) ||
      PyDict_SetItem(*dp, s_shape, shape) || PyDict_SetItem(*dp, s_strides, strides) ||
      PyDict_SetItem(*dp, s_offset, offset) || PyDict_SetItem(*dp, s_dtype, dtype) ||
      PyDict_SetItem(*dp, s_itemsize, itemsize) || PyDict_SetItem(*dp, s_numel, n) ||
      PyDict_SetItem(*dp, s_device, device) || PyDict_SetItem(*dp, s_tdev, tdev) ||
      PyDict_SetItem(*dp, s_contig, contig ? Py_True : Py_False)) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "no attribute dict");
    Py_XDECREF(n);
    Py_DECREF(t);
    return nullptr;
  }
  Py_DECREF(n);
  return t;
}

// A tuple's (or list's) ints; returns their count, -1 on error.
int ints_of(PyObject* o, int64_t* v) {
  if (!PyTuple_Check(o) && !PyList_Check(o)) {
    PyErr_Format(PyExc_TypeError, "expected a tuple of ints, got %s", Py_TYPE(o)->tp_name);
    return -1;
  }
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(o);
  if (n > kMaxRank) {
    PyErr_Format(PyExc_RuntimeError, "rank %zd (at most %d)", n, kMaxRank);
    return -1;
  }
  for (Py_ssize_t i = 0; i < n; ++i)
    if (!as_i64(PySequence_Fast_GET_ITEM(o, i), v + i)) return -1;
  return (int)n;
}

// The same for strides of a shape with nd dimensions, as torch reports it.
bool strides_of(PyObject* o, int64_t* v, int nd) {
  const int n = ints_of(o, v);
  if (n >= 0 && n != nd)
    PyErr_Format(PyExc_RuntimeError, "dimensionality of sizes (%d) must match dimensionality of strides (%d)", nd, n);
  return n == nd;
}

PyObject* tuple_of(const int64_t* v, int n) {
  PyObject* t = PyTuple_New(n);
  if (!t) return nullptr;
  for (int i = 0; i < n; ++i) {
    PyObject* x = PyLong_FromLongLong(v[i]);
    if (!x) {
      Py_DECREF(t);
      return nullptr;
    }
    PyTuple_SET_ITEM(t, i, x);
  }
  return t;
}

// Sizes are Python integers, so a count of elements or bytes may not fit in 64
// bits: then it is refused, as torch refuses it.
bool overflow(const char* what) {
  PyErr_Format(PyExc_RuntimeError, "%s overflows 64 bits", what);
  return false;
}

// The element count of a shape; false with an exception when it does not fit.
bool product(const int64_t* v, int n, int64_t* p) {
  bool over = false;
  *p = 1;
  for (int i = 0; i < n; ++i) {
    if (v[i] == 0) {
      *p = 0;
      return true;
    }
    over |= __builtin_mul_overflow(*p, v[i], p);
  }
  return !over || overflow("the number of elements");
}

bool contiguous(const int64_t* shape, const int64_t* strides, int n) {
  int64_t expected = 1;
  bool over = false;
  for (int i = n - 1; i >= 0; --i) {
    if (shape[i] == 1) continue;
    if (over || strides[i] != expected) return false;
    over = __builtin_mul_overflow(expected, shape[i], &expected);
  }
  return true;
}

// False with an exception when a stride does not fit.
bool row_major(const int64_t* shape, int n, int64_t* strides) {
  int64_t acc = 1;
  bool over = false;
  for (int i = n - 1; i >= 0; --i) {
    if (over) return overflow("a stride");
    strides[i] = acc;
    over = __builtin_mul_overflow(acc, shape[i] > 1 ? shape[i] : 1, &acc);
  }
  return true;
}

// make(holder, ptr, shape, strides, offset, dtype, device, contiguous | None)
PyObject* make(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 8) {
    PyErr_SetString(PyExc_TypeError, "make takes 8 arguments");
    return nullptr;
  }
  int64_t shape[kMaxRank], strides[kMaxRank];
  const int nd = ints_of(a[2], shape);
  if (nd < 0 || !strides_of(a[3], strides, nd)) return nullptr;
  int64_t numel;
  if (!product(shape, nd, &numel)) return nullptr;
  const bool c = a[7] == Py_None ? contiguous(shape, strides, nd) : PyObject_IsTrue(a[7]) == 1;
  PyObject *sh = tuple_of(shape, nd), *st = tuple_of(strides, nd), *t = nullptr;
  if (sh && st) t = make_impl(a[0], a[1], sh, st, a[4], a[5], a[6], numel, c);
  Py_XDECREF(sh), Py_XDECREF(st);
  return t;
}

// A new byte tensor of at least 1 byte on the device's storage device.
PyObject* alloc_bytes(int64_t nbytes, PyObject* device) {
  const int64_t index = PyLong_AsLongLong(device);
  if (index == -1 && PyErr_Occurred()) return nullptr;
  PyObject* dev = device_of(dev_storage, g_storage, index);
  if (!dev) return nullptr;
  PyObject* size = PyLong_FromLongLong(nbytes > 1 ? nbytes : 1);
  if (!size) return nullptr;
  PyObject *args[] = {size, g_uint8, dev}, *h = nullptr, *empty = PyObject_GetAttr(g_torch, s_empty);
  if (empty) {
    h = PyObject_Vectorcall(empty, args, 1, kw_empty);
    Py_DECREF(empty);
  }
  if (!h && PyErr_ExceptionMatches(g_oom)) {
    PyErr_Clear();
    h = PyObject_CallFunctionObjArgs(g_retry, size, device, nullptr);
  }
  Py_DECREF(size);
  return h;
}

// alloc_bytes(nbytes, device)
PyObject* alloc_bytes_py(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t size;
  if (n != 2) {
    PyErr_SetString(PyExc_TypeError, "alloc_bytes takes 2 arguments");
    return nullptr;
  }
  return as_i64(a[0], &size) ? alloc_bytes(size, a[1]) : nullptr;
}

// A new contiguous tensor of the shape (a tuple of ints).
PyObject* alloc_impl(const int64_t* shape, int nd, PyObject* dtype, PyObject* device) {
  PyObject* itemsize = PyDict_GetItemWithError(g_itemsize, dtype);
  if (!itemsize) {
    if (!PyErr_Occurred()) PyErr_Format(PyExc_TypeError, "unsupported dtype %R", dtype);
    return nullptr;
  }
  int64_t strides[kMaxRank], numel, bytes;
  if (!product(shape, nd, &numel) || !row_major(shape, nd, strides)) return nullptr;
  if (__builtin_mul_overflow(numel, (int64_t)PyLong_AsLongLong(itemsize), &bytes)) {
    overflow("the number of bytes");
    return nullptr;
  }
  PyObject* holder = alloc_bytes(bytes, device);
  if (!holder) return nullptr;
  PyObject *t = nullptr, *ptr = PyObject_CallMethodNoArgs(holder, s_data_ptr);
  PyObject *sh = tuple_of(shape, nd), *st = tuple_of(strides, nd), *zero = PyLong_FromLong(0);
  if (ptr && sh && st && zero) t = make_impl(holder, ptr, sh, st, zero, dtype, device, numel, true);
  Py_XDECREF(ptr), Py_XDECREF(sh), Py_XDECREF(st), Py_XDECREF(zero);
  Py_DECREF(holder);
  return t;
}

// alloc(shape, dtype, device)
PyObject* alloc(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 3) {
    PyErr_SetString(PyExc_TypeError, "alloc takes 3 arguments");
    return nullptr;
  }
  int64_t shape[kMaxRank];
  const int nd = ints_of(a[0], shape);
  if (nd > kAllocRank)
    PyErr_Format(PyExc_NotImplementedError, "mojo tensors support at most rank %d, got %d", kAllocRank, nd);
  return nd < 0 || nd > kAllocRank ? nullptr : alloc_impl(shape, nd, a[1], a[2]);
}

// The metadata of a mojo tensor (references are borrowed).
struct Meta {
  PyObject *holder, *ptr, *offset, *dtype, *device, *itemsize;
  int64_t shape[kMaxRank], strides[kMaxRank];
  int64_t numel;
  int nd;
  bool contig;
};

// False without an exception when `t` is no mojo tensor with a payload.
bool read(PyObject* t, Meta* m) {
  if (!PyObject_TypeCheck(t, g_cls)) return false;
  PyObject** dp = _PyObject_GetDictPtr(t);
  if (!dp || !*dp) return false;
  PyObject* d = *dp;
  m->holder = PyDict_GetItemWithError(d, s_holder);
  m->ptr = PyDict_GetItemWithError(d, s_ptr);
  m->offset = PyDict_GetItemWithError(d, s_offset);
  m->dtype = PyDict_GetItemWithError(d, s_dtype);
  m->device = PyDict_GetItemWithError(d, s_device);
  m->itemsize = PyDict_GetItemWithError(d, s_itemsize);
  PyObject* shape = PyDict_GetItemWithError(d, s_shape);
  PyObject* strides = PyDict_GetItemWithError(d, s_strides);
  PyObject* contig = PyDict_GetItemWithError(d, s_contig);
  if (!m->holder || !m->ptr || !m->offset || !m->dtype || !m->device || !m->itemsize || !shape || !strides || !contig)
    return false;
  m->nd = ints_of(shape, m->shape);
  if (m->nd < 0 || ints_of(strides, m->strides) != m->nd) return false;
  m->contig = contig == Py_True;
  return product(m->shape, m->nd, &m->numel);
}

// A view of m with another shape and strides, `delta` elements further on.
PyObject* view_impl(const Meta& m, const int64_t* shape, const int64_t* strides, int nd, int64_t delta, bool contig) {
  int64_t numel;
  if (!product(shape, nd, &numel)) return nullptr;
  PyObject *t = nullptr, *sh = tuple_of(shape, nd), *st = tuple_of(strides, nd);
  PyObject *ptr = m.ptr, *off = m.offset;
  if (delta) {
    int64_t p = PyLong_AsLongLong(m.ptr), o = PyLong_AsLongLong(m.offset), by = PyLong_AsLongLong(m.itemsize);
    ptr = off = nullptr;
    if (__builtin_mul_overflow(delta, by, &by) || __builtin_add_overflow(p, by, &p) ||
        __builtin_add_overflow(o, delta, &o)) {
      overflow("the address of a view");
    } else {
      ptr = PyLong_FromLongLong(p);
      off = PyLong_FromLongLong(o);
    }
  } else {
    Py_INCREF(ptr), Py_INCREF(off);
  }
  if (sh && st && ptr && off) t = make_impl(m.holder, ptr, sh, st, off, m.dtype, m.device, numel, contig);
  Py_XDECREF(sh), Py_XDECREF(st), Py_XDECREF(ptr), Py_XDECREF(off);
  return t;
}

PyObject* not_mojo() {
  if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "expected a mojo tensor");
  return nullptr;
}

// view_of(base, shape, strides, offset, contiguous | None): offset is absolute
PyObject* view_of(PyObject*, PyObject* const* a, Py_ssize_t n) {
  Meta m;
  if (n != 5) {
    PyErr_SetString(PyExc_TypeError, "view_of takes 5 arguments");
    return nullptr;
  }
  if (!read(a[0], &m)) return not_mojo();
  int64_t shape[kMaxRank], strides[kMaxRank], off;
  const int nd = ints_of(a[1], shape);
  if (nd < 0 || !strides_of(a[2], strides, nd) || !as_i64(a[3], &off)) return nullptr;
  int64_t delta;
  if (__builtin_sub_overflow(off, (int64_t)PyLong_AsLongLong(m.offset), &delta)) {
    overflow("the offset of a view");
    return nullptr;
  }
  const bool c = a[4] == Py_None ? contiguous(shape, strides, nd) : PyObject_IsTrue(a[4]) == 1;
  return view_impl(m, shape, strides, nd, delta, c);
}

// alias(t)
PyObject* alias(PyObject*, PyObject* t) {
  Meta m;
  if (!read(t, &m)) return not_mojo();
  return view_impl(m, m.shape, m.strides, m.nd, 0, m.contig);
}

// transpose(t, d0, d1); dims wrap, out-of-range dims raise as torch does
PyObject* transpose(PyObject*, PyObject* const* a, Py_ssize_t n) {
  Meta m;
  if (n != 3) {
    PyErr_SetString(PyExc_TypeError, "transpose takes 3 arguments");
    return nullptr;
  }
  if (!read(a[0], &m)) return not_mojo();
  int64_t d[2];
  const int64_t r = m.nd > 1 ? m.nd : 1;
  for (int i = 0; i < 2; ++i) {
    if (!as_i64(a[1 + i], &d[i])) return nullptr;
    if (d[i] < -r || d[i] >= r) {
      PyErr_Format(PyExc_IndexError, "Dimension out of range (expected to be in range of [%lld, %lld], but got %lld)",
                   (long long)-r, (long long)(r - 1), (long long)d[i]);
      return nullptr;
    }
    if (d[i] < 0) d[i] += r;
  }
  if (m.nd == 0) return view_impl(m, m.shape, m.strides, 0, 0, m.contig);
  std::swap(m.shape[d[0]], m.shape[d[1]]);
  std::swap(m.strides[d[0]], m.strides[d[1]]);
  return view_impl(m, m.shape, m.strides, m.nd, 0, contiguous(m.shape, m.strides, m.nd));
}

// narrow(t, dim, start, length): a step-1 slice with normalised arguments
PyObject* narrow(PyObject*, PyObject* const* a, Py_ssize_t n) {
  Meta m;
  int64_t d, start, len;
  if (n != 4) {
    PyErr_SetString(PyExc_TypeError, "narrow takes 4 arguments");
    return nullptr;
  }
  if (!read(a[0], &m)) return not_mojo();
  if (!as_i64(a[1], &d) || !as_i64(a[2], &start) || !as_i64(a[3], &len)) return nullptr;
  int64_t delta = 0;
  if (d < 0 || d >= m.nd || start < 0 || len < 0 || start > m.shape[d] || len > m.shape[d] - start ||
      __builtin_mul_overflow(start, m.strides[d], &delta)) {
    PyErr_SetString(PyExc_IndexError, "narrow: out of range");
    return nullptr;
  }
  m.shape[d] = len;
  return view_impl(m, m.shape, m.strides, m.nd, delta, contiguous(m.shape, m.strides, m.nd));
}

// reshape_contiguous(t, size): the view of a contiguous tensor, or None when
// the tensor is not contiguous or the size does not fit (the caller reports)
PyObject* reshape_contiguous(PyObject*, PyObject* const* a, Py_ssize_t n) {
  Meta m;
  if (n != 2) {
    PyErr_SetString(PyExc_TypeError, "reshape_contiguous takes 2 arguments");
    return nullptr;
  }
  if (!read(a[0], &m)) return not_mojo();
  if (!m.contig) Py_RETURN_NONE;
  int64_t shape[kMaxRank], strides[kMaxRank];
  const int nd = ints_of(a[1], shape);
  if (nd < 0) return nullptr;
  int unknown = -1;
  int64_t known = 1;
  for (int i = 0; i < nd; ++i) {
    if (shape[i] == -1 && unknown < 0) unknown = i;
    else if (shape[i] < 0 || __builtin_mul_overflow(known, shape[i], &known)) Py_RETURN_NONE;
  }
  if (unknown >= 0) {
    if (known == 0 || m.numel % known) Py_RETURN_NONE;
    shape[unknown] = m.numel / known;
  } else if (known != m.numel) {
    Py_RETURN_NONE;
  }
  if (!row_major(shape, nd, strides)) return nullptr;
  return view_impl(m, shape, strides, nd, 0, true);
}

PyObject* source_hash(PyObject*, PyObject*) { return PyUnicode_FromString(MI355X_SOURCE_HASH); }

#define METHOD(f) {#f, (PyCFunction)(void (*)(void))&Call<decltype(&f), Tag_##f>::call, METH_FASTCALL, nullptr},
#define FAST(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr},
PyMethodDef kMethods[] = {
    KERNELS(METHOD) FAST(make) FAST(alloc) FAST(view_of) FAST(transpose) FAST(narrow) FAST(reshape_contiguous)
    {"alloc_bytes", (PyCFunction)(void (*)(void))alloc_bytes_py, METH_FASTCALL, nullptr},
    {"alias", alias, METH_O, nullptr},
    {"bind", bind, METH_VARARGS, nullptr},
    {"setup", setup, METH_VARARGS, nullptr},
    {"reset", reset, METH_NOARGS, nullptr},
    {"source_hash", source_hash, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", "Native host path of the mojo device.", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
  s_holder = PyUnicode_InternFromString("_holder");
  s_ptr = PyUnicode_InternFromString("_ptr");
  s_shape = PyUnicode_InternFromString("_shape");
  s_strides = PyUnicode_InternFromString("_strides");
  s_offset = PyUnicode_InternFromString("_offset");
  s_dtype = PyUnicode_InternFromString("_dtype");
  s_itemsize = PyUnicode_InternFromString("_itemsize");
  s_numel = PyUnicode_InternFromString("_numel");
  s_device = PyUnicode_InternFromString("_device");
  s_tdev = PyUnicode_InternFromString("_torch_device");
  s_contig = PyUnicode_InternFromString("_is_contiguous");
  s_data_ptr = PyUnicode_InternFromString("data_ptr");
  s_empty = PyUnicode_InternFromString("empty");
  kw_wrap = Py_BuildValue("(sssss)", "strides", "storage_offset", "dtype", "layout", "device");
  kw_empty = Py_BuildValue("(ss)", "dtype", "device");
  if (!kw_wrap || !kw_empty || !s_empty) return nullptr;
  return PyModule_Create(&kModule);
}

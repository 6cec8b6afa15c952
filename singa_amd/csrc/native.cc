// The host side of the singa_wrap mirror that every operation passes through, as a CPython extension
// (singa_amd/_native.so): the memory block behind a tensor, the tensor's fields and accessors, and direct calls into the C ABI.
//
// A training step of a small network is bound by its host work: in Python with ctypes a Mult took 7 us around a launch of
// 2.5 us (argument conversion 2.5, result tensor 2.5, shape checks 1.5).  Here a call converts its arguments from the ABI's
// own prototypes at compile time, and a tensor is allocated in one call.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <dlfcn.h>
#include <stddef.h>
#include <stdint.h>

#include <tuple>
#include <utility>

#include "singa_hip.h"

namespace {

PyObject *g_check;   // singa_amd._lib.check(rc, what): raises the library's message
PyObject *g_open;    // opens the library and returns its dlopen handle
PyObject *g_tensor;  // singa_amd.singa_wrap.Tensor: the class of results
PyObject *g_handle_name;

// The library is opened by the first call into it, not by loading this module: a program may import torch after this
// package, and the library has to find the HIP runtime that torch brought, not put a second one into the process.
void *g_library;

void *entry_point(const char *name) {   // null with an exception set
  if (!g_library) {
    PyObject *h = PyObject_CallFunction(g_open, nullptr);
    if (!h) return nullptr;
    g_library = PyLong_AsVoidPtr(h);
    Py_DECREF(h);
    if (!g_library) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "the library has no handle");
      return nullptr;
    }
  }
  void *p = dlsym(g_library, name);
  if (!p) PyErr_Format(PyExc_AttributeError, "%s is not in the library", name);
  return p;
}

// The address of an entry point with the type that the header declares; SGH_ENTRY(name)::get() is null with an exception
// set when the library cannot be opened
template <class F>
struct EntryOf {
  template <class N>
  static F get() {
    static F found = nullptr;
    if (!found) found = reinterpret_cast<F>(entry_point(N::text));
    return found;
  }
};
#define SGH_ENTRY(name)                                                          \
  struct Entry_##name {                                                          \
    typedef decltype(&::name) type;                                              \
    static constexpr const char *text = #name;                                   \
    static type get() { return EntryOf<type>::template get<Entry_##name>(); }    \
  };
#define SGH_ENTRY3(name) SGH_ENTRY(name##_f32) SGH_ENTRY(name##_f16) SGH_ENTRY(name##_bf16)
// what the methods below call by name
#define SGH_CALLS(ONE, ALL)                                                                                                     \
  ONE(sgh_device_join) ONE(sgh_block_used_on) ALL(sgh_memset) ALL(sgh_relu_fwd) ALL(sgh_relu_bwd) ALL(sgh_relu_bwd_add)         \
  ALL(sgh_add) ALL(sgh_add_relu) ALL(sgh_eltwise_mult) ALL(sgh_axpy) ONE(sgh_axpy_devalpha_f32) ONE(sgh_sub_f32)                \
  ONE(sgh_div_f32) ONE(sgh_add_scalar_f32) ONE(sgh_mult_scalar_f32) ONE(sgh_clamp_f32) ONE(sgh_cast_f32_to_f16)                 \
  ONE(sgh_cast_f16_to_f32) ONE(sgh_cast_f32_to_bf16) ONE(sgh_cast_bf16_to_f32) ONE(sgh_cast_f32_to_i32)                         \
  ONE(sgh_cast_i32_to_f32) ALL(sgh_softmax_ce_bwd) ONE(sgh_softmax_fwd_f32) ONE(sgh_cross_entropy_fwd_f32) ALL(sgh_gemm)        \
  ONE(sgh_linear_fwd_f32) ONE(sgh_linear_bwd_x_f32) ONE(sgh_linear_bwd_wb_f32) ONE(sgh_softmax_ce_fwd_f32)                       \
  ONE(sgh_sum_rows_f32) ONE(sgh_add_row_f32) ONE(sgh_row_max_f32) ONE(sgh_row_max_zero_seeded_f32) ONE(sgh_dot_f32)             \
  ONE(sgh_sum_all_f32) ALL(sgh_sgd_momentum) ONE(sgh_sgd_momentum_multi_f32) ONE(sgh_sgd_momentum_multi_mixed)                  \
  ONE(sgh_sgd_momentum_master_f16) ONE(sgh_sgd_momentum_master_bf16) ALL(sgh_conv_fwd) ALL(sgh_conv_dgrad) ALL(sgh_conv_wgrad)  \
  ALL(sgh_conv_bgrad) ONE(sgh_conv_dgrad_acc_f32) ONE(sgh_conv_dgrad_add_relu_f16) ONE(sgh_conv_dgrad_add_relu_bf16)               \
  ONE(sgh_conv_wgrad_bias_f32) ALL(sgh_bn_fwd_train) ALL(sgh_bn_relu_fwd_train) \
  ALL(sgh_bn_add_relu_fwd_train) ALL(sgh_bn_fwd_infer) ALL(sgh_bn_bwd) ALL(sgh_bn_relu_bwd) ALL(sgh_pool_fwd) ALL(sgh_pool_bwd) \
  ONE(sgh_pool_relu_fwd_f32) ONE(sgh_pool_relu_bwd_f32)
SGH_CALLS(SGH_ENTRY, SGH_ENTRY3)
SGH_ENTRY(sgh_malloc)
SGH_ENTRY(sgh_free)
SGH_ENTRY(sgh_device_fork)

bool failed(int rc, const char *what) {
  if (rc == 0) return false;
  PyObject *r = PyObject_CallFunction(g_check, "is", rc, what);
  Py_XDECREF(r);
  if (r) PyErr_SetString(PyExc_RuntimeError, what);   // (check always raises)
  return true;
}

// ------------------------------------------------------------------------------------ direct calls

template <class T>
struct Arg;
template <class T>
struct Arg<T *> {
  static T *from(PyObject *o) {
    if (o == Py_None) return nullptr;
    if (PyLong_Check(o)) return static_cast<T *>(PyLong_AsVoidPtr(o));
    PyObject *v = PyObject_GetAttrString(o, "value");   // a ctypes.c_void_p, as a caller's own stream may come
    if (!v) return nullptr;
    T *p = v == Py_None ? nullptr : static_cast<T *>(PyLong_AsVoidPtr(v));
    Py_DECREF(v);
    return p;
  }
};
template <>
struct Arg<int> {
  static int from(PyObject *o) {
    const long v = PyLong_AsLong(o);
    if (v != long(int(v))) PyErr_SetString(PyExc_OverflowError, "argument does not fit an int");
    return int(v);
  }
};
template <>
struct Arg<size_t> {
  static size_t from(PyObject *o) {
    PyObject *i = PyNumber_Index(o);   // (whole numbers of numpy as well)
    if (!i) return 0;
    const size_t v = PyLong_AsSize_t(i);
    Py_DECREF(i);
    return v;
  }
};
template <>
struct Arg<float> {
  static float from(PyObject *o) { return float(PyFloat_AsDouble(o)); }
};

template <class E, class F = typename E::type>
struct Call;
template <class E, class... A>
struct Call<E, int (*)(A...)> {
  template <size_t... I>
  static PyObject *with(PyObject *const *args, std::integer_sequence<size_t, I...>) {
    const std::tuple<A...> a{Arg<A>::from(args[I])...};
    if (PyErr_Occurred()) return nullptr;
    const typename E::type f = E::get();
    if (!f) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f(std::get<I>(a)...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
  }
  static PyObject *call(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != Py_ssize_t(sizeof...(A))) {
      PyErr_Format(PyExc_TypeError, "%zd arguments given, %zd expected", n, Py_ssize_t(sizeof...(A)));
      return nullptr;
    }
    return with(args, std::make_integer_sequence<size_t, sizeof...(A)>());
  }
};

// ------------------------------------------------------------------------------------ Block

struct Block {
  PyObject_HEAD
  PyObject *dev, *keepalive, *address;
  sgh_device *handle;
  void *ptr;
  Py_ssize_t nbytes;
  char owned;
};
extern PyTypeObject BlockType;

// A block of the device's pool, or (`external`) around memory that someone else owns, at any address: null as well
Block *block_new(PyTypeObject *type, PyObject *dev, Py_ssize_t nbytes, bool external, void *ptr, PyObject *keepalive) {
  sgh_device *h = nullptr;
  if (!external) {
    PyObject *ho = PyObject_GetAttr(dev, g_handle_name);
    if (!ho) return nullptr;
    h = static_cast<sgh_device *>(PyLong_AsVoidPtr(ho));
    Py_DECREF(ho);
    if (PyErr_Occurred()) return nullptr;
    const Entry_sgh_malloc::type take = Entry_sgh_malloc::get();
    if (!take || !Entry_sgh_free::get()) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS   // (a miss of the pool waits for the driver)
    rc = take(h, &ptr, nbytes > 0 ? size_t(nbytes) : 1);
    Py_END_ALLOW_THREADS
    if (failed(rc, "sgh_malloc")) return nullptr;
  }
  Block *b = reinterpret_cast<Block *>(type->tp_alloc(type, 0));
  if (!b) {
    if (h) Entry_sgh_free::get()(h, ptr);
    return nullptr;
  }
  b->handle = h, b->ptr = ptr, b->nbytes = nbytes, b->owned = !external;
  Py_INCREF(dev);
  b->dev = dev;
  Py_XINCREF(keepalive);
  b->keepalive = keepalive;
  b->address = PyLong_FromVoidPtr(ptr);
  return b;
}

PyObject *block_tp_new(PyTypeObject *type, PyObject *args, PyObject *kw) {
  static const char *names[] = {"dev", "nbytes", "ptr", "keepalive", nullptr};
  PyObject *dev, *ptr = Py_None, *keepalive = nullptr;
  Py_ssize_t nbytes;
  if (!PyArg_ParseTupleAndKeywords(args, kw, "On|OO", const_cast<char **>(names), &dev, &nbytes, &ptr, &keepalive)) return nullptr;
  void *p = ptr == Py_None ? nullptr : PyLong_AsVoidPtr(ptr);
  if (PyErr_Occurred()) return nullptr;
  return reinterpret_cast<PyObject *>(block_new(type, dev, nbytes, ptr != Py_None, p, keepalive));
}

// (the owner of wrapped memory may hold the tensor that keeps it alive)
int block_traverse(PyObject *self, visitproc visit, void *arg) {
  Py_VISIT(reinterpret_cast<Block *>(self)->dev);
  Py_VISIT(reinterpret_cast<Block *>(self)->keepalive);
  return 0;
}

int block_clear(PyObject *self) {
  Py_CLEAR(reinterpret_cast<Block *>(self)->dev);
  Py_CLEAR(reinterpret_cast<Block *>(self)->keepalive);
  return 0;
}

void block_dealloc(PyObject *self) {
  PyObject_GC_UnTrack(self);
  Block *b = reinterpret_cast<Block *>(self);
  if (b->owned && b->ptr) {
    const Entry_sgh_free::type give = Entry_sgh_free::get();   // (found before the block was made)
    Py_BEGIN_ALLOW_THREADS
    give(b->handle, b->ptr);
    Py_END_ALLOW_THREADS
  }
  block_clear(self);
  Py_XDECREF(b->address);
  Py_TYPE(self)->tp_free(self);
}

PyMemberDef block_members[] = {
    {"dev", T_OBJECT, offsetof(Block, dev), READONLY, "device"},
    {"keepalive", T_OBJECT, offsetof(Block, keepalive), READONLY, "owner of memory that is not the pool's"},
    {"ptr", T_OBJECT, offsetof(Block, address), READONLY, "device address"},
    {"nbytes", T_PYSSIZET, offsetof(Block, nbytes), READONLY, "size"},
    {"owned", T_BOOL, offsetof(Block, owned), READONLY, "whether the memory goes back to the pool"},
    {nullptr, 0, 0, 0, nullptr}};

PyTypeObject BlockType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ------------------------------------------------------------------------------------ Tensor

struct Tensor {
  PyObject_HEAD
  PyObject *shape, *dev, *block;
  int dtype;
  char transposed;
};
extern PyTypeObject TensorType;

inline Tensor *as_tensor(PyObject *o) { return reinterpret_cast<Tensor *>(o); }

// product of the extents, -1 with an exception set when `shape` is not a tuple of whole numbers or the product leaves no room
// for an element's size
Py_ssize_t count_of(PyObject *shape) {
  if (!shape || !PyTuple_Check(shape)) {
    PyErr_SetString(PyExc_TypeError, "a tensor's shape is a tuple");
    return -1;
  }
  Py_ssize_t n = 1;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(shape); ++i) {
    const Py_ssize_t e = PyLong_AsSsize_t(PyTuple_GET_ITEM(shape, i));
    if (PyErr_Occurred()) return -1;
    if (__builtin_mul_overflow(n, e, &n) || n > PY_SSIZE_T_MAX / 4) {
      PyErr_SetString(PyExc_OverflowError, "a tensor of this shape cannot be addressed");
      return -1;
    }
  }
  return n;
}

inline Py_ssize_t elem_size(int dtype) { return dtype == 1 || dtype == 100 ? 2 : 4; }   // kFloat16, kBFloat16; kFloat32, kInt

// a dense tensor of the pool
PyObject *tensor_make(PyTypeObject *type, PyObject *shape, PyObject *dev, int dtype) {
  const Py_ssize_t n = count_of(shape);
  if (n < 0 && PyErr_Occurred()) return nullptr;
  Block *b = block_new(&BlockType, dev, n * elem_size(dtype), false, nullptr, nullptr);
  if (!b) return nullptr;
  PyObject *o = type->tp_alloc(type, 0);
  if (!o) {
    Py_DECREF(b);
    return nullptr;
  }
  Tensor *t = as_tensor(o);
  Py_INCREF(shape);
  t->shape = shape;
  Py_INCREF(dev);
  t->dev = dev;
  t->block = reinterpret_cast<PyObject *>(b);
  t->dtype = dtype, t->transposed = 0;
  return o;
}

PyObject *empty(PyObject *, PyObject *const *args, Py_ssize_t n) {   // empty(cls, shape, device, dtype)
  if (n != 4 || !PyType_Check(args[0]) || !PyType_IsSubtype(reinterpret_cast<PyTypeObject *>(args[0]), &TensorType)) {
    PyErr_SetString(PyExc_TypeError, "empty(cls, shape, device, dtype)");
    return nullptr;
  }
  const long dtype = PyLong_AsLong(args[3]);
  if (PyErr_Occurred()) return nullptr;
  return tensor_make(reinterpret_cast<PyTypeObject *>(args[0]), args[1], args[2], int(dtype));
}

PyObject *empty_like(PyObject *, PyObject *o) {   // a dense tensor of o's shape, device and type
  if (!PyObject_TypeCheck(o, &TensorType)) {
    PyErr_SetString(PyExc_TypeError, "a Tensor is expected");
    return nullptr;
  }
  Tensor *t = as_tensor(o);
  if (!t->dev) {
    PyErr_SetString(PyExc_AttributeError, "the tensor has no device");
    return nullptr;
  }
  if (!g_tensor) {
    PyErr_SetString(PyExc_RuntimeError, "no tensor class has been set");
    return nullptr;
  }
  return tensor_make(reinterpret_cast<PyTypeObject *>(g_tensor), t->shape, t->dev, t->dtype);
}

int tensor_traverse(PyObject *self, visitproc visit, void *arg) {
  Tensor *t = as_tensor(self);
  Py_VISIT(t->shape);
  Py_VISIT(t->dev);
  Py_VISIT(t->block);
  return 0;
}

int tensor_clear(PyObject *self) {
  Tensor *t = as_tensor(self);
  Py_CLEAR(t->shape);
  Py_CLEAR(t->dev);
  Py_CLEAR(t->block);
  return 0;
}

void tensor_dealloc(PyObject *self) {
  PyObject_GC_UnTrack(self);
  tensor_clear(self);
  Py_TYPE(self)->tp_free(self);
}

PyObject *tensor_shape(PyObject *self, PyObject *const *args, Py_ssize_t n, PyObject *names) {
  PyObject *shape = as_tensor(self)->shape;
  if (count_of(shape) < 0 && PyErr_Occurred()) return nullptr;
  const Py_ssize_t named = names ? PyTuple_GET_SIZE(names) : 0;   // (their values follow the positional ones)
  const bool known = named == 0 || (named == 1 && PyUnicode_CompareWithASCIIString(PyTuple_GET_ITEM(names, 0), "axis") == 0);
  n += named;
  if (known && (n == 0 || (n == 1 && args[0] == Py_None))) return PySequence_List(shape);
  if (!known || n != 1) {
    PyErr_SetString(PyExc_TypeError, "shape(axis=None)");
    return nullptr;
  }
  return PyObject_GetItem(shape, args[0]);
}

PyObject *tensor_size(PyObject *self, PyObject *) {
  const Py_ssize_t n = count_of(as_tensor(self)->shape);
  return n < 0 && PyErr_Occurred() ? nullptr : PyLong_FromSsize_t(n);
}

PyObject *tensor_memsize(PyObject *self, PyObject *) {
  const Py_ssize_t n = count_of(as_tensor(self)->shape);
  return n < 0 && PyErr_Occurred() ? nullptr : PyLong_FromSsize_t(n * elem_size(as_tensor(self)->dtype));
}

PyObject *tensor_ndim(PyObject *self, PyObject *) {
  PyObject *shape = as_tensor(self)->shape;
  return count_of(shape) < 0 && PyErr_Occurred() ? nullptr : PyLong_FromSsize_t(PyTuple_GET_SIZE(shape));
}

PyObject *tensor_data_type(PyObject *self, PyObject *) { return PyLong_FromLong(as_tensor(self)->dtype); }
PyObject *tensor_transpose(PyObject *self, PyObject *) { return PyBool_FromLong(as_tensor(self)->transposed); }

PyObject *tensor_device(PyObject *self, PyObject *) {
  PyObject *d = as_tensor(self)->dev;
  if (!d) d = Py_None;
  Py_INCREF(d);
  return d;
}

PyObject *tensor_ptr(PyObject *self, void *) {
  PyObject *b = as_tensor(self)->block;
  if (b && Py_TYPE(b) == &BlockType) {
    PyObject *a = reinterpret_cast<Block *>(b)->address;
    Py_INCREF(a);
    return a;
  }
  PyErr_SetString(PyExc_AttributeError, "the tensor has no memory");
  return nullptr;
}

PyMemberDef tensor_members[] = {{"_shape", T_OBJECT, offsetof(Tensor, shape), 0, "tuple of extents"},
                                {"_dev", T_OBJECT, offsetof(Tensor, dev), 0, "device"},
                                {"_block", T_OBJECT, offsetof(Tensor, block), 0, "memory"},
                                {"_dtype", T_INT, offsetof(Tensor, dtype), 0, "data type"},
                                {"_transposed", T_BOOL, offsetof(Tensor, transposed), 0, "view of the stored matrix transposed"},
                                {nullptr, 0, 0, 0, nullptr}};
PyGetSetDef tensor_getset[] = {{"ptr", tensor_ptr, nullptr, "device address", nullptr}, {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyMethodDef tensor_methods[] = {
    {"shape", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(tensor_shape)), METH_FASTCALL | METH_KEYWORDS,
     "extents, or one of them"},
    {"Size", tensor_size, METH_NOARGS, "number of elements"},
    {"MemSize", tensor_memsize, METH_NOARGS, "bytes"},
    {"nDim", tensor_ndim, METH_NOARGS, "number of dimensions"},
    {"data_type", tensor_data_type, METH_NOARGS, "data type"},
    {"transpose", tensor_transpose, METH_NOARGS, "whether this is a transposed view"},
    {"device", tensor_device, METH_NOARGS, "device"},
    {nullptr, nullptr, 0, nullptr}};

PyTypeObject TensorType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ------------------------------------------------------------------------------------ module

PyObject *set_check(PyObject *, PyObject *f) {
  Py_INCREF(f);
  Py_XSETREF(g_check, f);
  Py_RETURN_NONE;
}

PyObject *set_tensor(PyObject *, PyObject *c) {
  if (!PyType_Check(c) || !PyType_IsSubtype(reinterpret_cast<PyTypeObject *>(c), &TensorType)) {
    PyErr_SetString(PyExc_TypeError, "a class derived from TensorBase is expected");
    return nullptr;
  }
  Py_INCREF(c);
  Py_XSETREF(g_tensor, c);
  Py_RETURN_NONE;
}

PyObject *set_open(PyObject *, PyObject *f) {
  Py_INCREF(f);
  Py_XSETREF(g_open, f);
  Py_RETURN_NONE;
}

// fork(handle): the auxiliary stream's address
PyObject *fork_(PyObject *, PyObject *h) {
  void *aux = nullptr;
  sgh_device *d = static_cast<sgh_device *>(PyLong_AsVoidPtr(h));
  if (PyErr_Occurred()) return nullptr;
  const Entry_sgh_device_fork::type split = Entry_sgh_device_fork::get();
  if (!split) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = split(d, &aux);
  Py_END_ALLOW_THREADS
  if (failed(rc, "sgh_device_fork")) return nullptr;
  return PyLong_FromVoidPtr(aux);
}

#define SGH_CALL(name) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(Call<Entry_##name>::call)), METH_FASTCALL, nullptr},
#define SGH_CALL3(name) SGH_CALL(name##_f32) SGH_CALL(name##_f16) SGH_CALL(name##_bf16)

PyMethodDef methods[] = {
    {"set_check", set_check, METH_O, "the function that turns a return code into an exception"},
    {"set_open", set_open, METH_O, "the function that opens the library and returns its handle"},
    {"set_tensor", set_tensor, METH_O, "the class of the tensors that empty_like makes"},
    {"empty", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(empty)), METH_FASTCALL, "empty(cls, shape, device, dtype)"},
    {"empty_like", empty_like, METH_O, "a dense tensor of the same shape, device and type"},
    {"fork", fork_, METH_O, "sgh_device_fork: the auxiliary stream"},
    SGH_CALLS(SGH_CALL, SGH_CALL3)
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "tensors, memory blocks and direct calls into libsinga_hip", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
  BlockType.tp_name = "singa_amd._native.Block";
  BlockType.tp_doc = "Block(dev, nbytes, ptr=None, keepalive=None): a pool allocation, or memory owned elsewhere";
  BlockType.tp_basicsize = sizeof(Block);
  BlockType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC;
  BlockType.tp_new = block_tp_new;
  BlockType.tp_dealloc = block_dealloc;
  BlockType.tp_traverse = block_traverse;
  BlockType.tp_clear = block_clear;
  BlockType.tp_members = block_members;
  TensorType.tp_name = "singa_amd._native.TensorBase";
  TensorType.tp_doc = "the fields of a tensor and their accessors";
  TensorType.tp_basicsize = sizeof(Tensor);
  TensorType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC;
  TensorType.tp_new = PyType_GenericNew;
  TensorType.tp_dealloc = tensor_dealloc;
  TensorType.tp_traverse = tensor_traverse;
  TensorType.tp_clear = tensor_clear;
  TensorType.tp_members = tensor_members;
  TensorType.tp_getset = tensor_getset;
  TensorType.tp_methods = tensor_methods;
  if (PyType_Ready(&BlockType) < 0 || PyType_Ready(&TensorType) < 0) return nullptr;
  g_handle_name = PyUnicode_InternFromString("_handle");
  PyObject *m = PyModule_Create(&module);
  if (!m) return nullptr;
  Py_INCREF(&BlockType);
  PyModule_AddObject(m, "Block", reinterpret_cast<PyObject *>(&BlockType));
  Py_INCREF(&TensorType);
  PyModule_AddObject(m, "TensorBase", reinterpret_cast<PyObject *>(&TensorType));
  return m;
}

// The per-request half of the Python binding (ps-lite_amd/capi.py) as a CPython extension.
//
// A request from Python is a few checks on its arrays and one call of the C ABI. Through ctypes the
// checks cost more than the call: 1.7 us for the address of a numpy array, 3.4 us to wait for torch's
// current stream, 4.7 us of the 8.9 us of a device-resident push of 1,000 keys. Every function here
// takes the arrays themselves and returns None when one of them is not what the quick way takes (a list, another
// dtype, a non-contiguous array): capi.py then goes its general way, which converts or refuses it.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <hip/hip_runtime_api.h>
#define NPY_NO_DEPRECATED_API NPY_1_7_API_VERSION
#include <numpy/arrayobject.h>
#include <stdint.h>

#include "pskv/capi.h"

namespace {

// set once by setup(): torch's types, null when torch is not there
PyObject* g_tensor_type = nullptr;
PyObject *g_int64 = nullptr, *g_uint64 = nullptr, *g_float32 = nullptr, *g_int32 = nullptr;
PyObject* g_raw_stream = nullptr;  // callable: device index -> hipStream_t of torch's current stream, as an int
PyObject *s_dtype, *s_is_cuda, *s_is_contiguous, *s_numel, *s_data_ptr;

enum Kind { kNone = -1, kHost = PSKV_MEM_HOST, kDevice = PSKV_MEM_DEVICE };

// One array argument. `type`: 'k' keys (64-bit), 'f' float32, 'i' int32.
class Arg {
 public:
  ~Arg() {
    if (viewed_) PyBuffer_Release(&view_);
  }
  // 1 taken, 0 not for the quick way, -1 a Python error is set
  int take(PyObject* o, char type) {
    if (o == Py_None) return 1;
    // (a numpy array is looked at itself: its buffer costs 50 ns to ask for and to give back, and a slice of a request has six.
    // The caller's arguments keep it.)
    if (PyArray_CheckExact(o)) return array(reinterpret_cast<PyArrayObject*>(o), type);
    if (g_tensor_type && PyObject_TypeCheck(o, reinterpret_cast<PyTypeObject*>(g_tensor_type))) return tensor(o, type);
    if (!PyObject_CheckBuffer(o)) return 0;
    if (PyObject_GetBuffer(o, &view_, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT) != 0) {
      PyErr_Clear();
      return 0;
    }
    viewed_ = true;
    const char* f = view_.format;
    if (!f || f[0] == 0 || f[1] != 0) return 0;
    const bool fits = type == 'k'   ? (f[0] == 'L' || f[0] == 'Q') && view_.itemsize == 8
                      : type == 'f' ? f[0] == 'f' && view_.itemsize == 4
                                    : f[0] == 'i' && view_.itemsize == 4;
    if (!fits) return 0;
    n = (size_t)(view_.len / view_.itemsize);
    ptr = n ? view_.buf : nullptr;
    kind = kHost;
    return 1;
  }
  void* ptr = nullptr;
  size_t n = 0;
  int kind = kNone;
  PyObject* device_tensor = nullptr;  // borrowed

 private:
  int array(PyArrayObject* a, char type) {
    const int t = PyArray_TYPE(a);
    const bool fits = type == 'k'   ? t == NPY_ULONG || t == NPY_ULONGLONG
                      : type == 'f' ? t == NPY_FLOAT
                                    : t == NPY_INT;
    if (!fits || !PyArray_IS_C_CONTIGUOUS(a) || !PyArray_ISALIGNED(a) || !PyArray_ISNOTSWAPPED(a)) return 0;
    n = (size_t)PyArray_SIZE(a);
    ptr = n ? PyArray_DATA(a) : nullptr;
    kind = kHost;
    return 1;
  }
  int tensor(PyObject* o, char type) {
    PyObject* d = PyObject_GetAttr(o, s_dtype);
    if (!d) return -1;
    Py_DECREF(d);  // (dtypes live as long as torch does)
    const bool fits = type == 'k' ? d == g_int64 || d == g_uint64 : type == 'f' ? d == g_float32 : d == g_int32;
    if (!fits) return 0;
    PyObject* c = PyObject_CallMethodNoArgs(o, s_is_contiguous);
    if (!c) return -1;
    Py_DECREF(c);
    if (c != Py_True) return 0;
    PyObject* cuda = PyObject_GetAttr(o, s_is_cuda);
    if (!cuda) return -1;
    Py_DECREF(cuda);
    PyObject* count = PyObject_CallMethodNoArgs(o, s_numel);
    if (!count) return -1;
    n = PyLong_AsSize_t(count);
    Py_DECREF(count);
    if (n) {
      PyObject* p = PyObject_CallMethodNoArgs(o, s_data_ptr);
      if (!p) return -1;
      ptr = PyLong_AsVoidPtr(p);
      Py_DECREF(p);
    }
    if (PyErr_Occurred()) return -1;
    kind = cuda == Py_True ? kDevice : kHost;
    if (kind == kDevice) device_tensor = o;
    return 1;
  }
  Py_buffer view_;
  bool viewed_ = false;
};

// The C ABI wants device buffers complete before the call; torch fills and copies tensors on its current
// stream, which is waited for here. false: a Python error is set.
bool torch_is_done() {
  int device = 0;
  if (!g_raw_stream || hipGetDevice(&device) != hipSuccess) return true;
  PyObject* at = PyLong_FromLong(device);
  if (!at) return false;
  PyObject* raw = PyObject_CallOneArg(g_raw_stream, at);
  Py_DECREF(at);
  if (!raw) return false;
  void* stream = PyLong_AsVoidPtr(raw);
  Py_DECREF(raw);
  if (!stream && PyErr_Occurred()) return false;
  hipError_t e;
  Py_BEGIN_ALLOW_THREADS;
  e = hipStreamSynchronize(static_cast<hipStream_t>(stream));
  Py_END_ALLOW_THREADS;
  if (e != hipSuccess) {
    PyErr_Format(PyExc_RuntimeError, "waiting for torch's stream: %s", hipGetErrorString(e));
    return false;
  }
  return true;
}

// Takes `count` arrays of the given types; what they agree on goes to *kind. Device tensors are appended to `held`
// (a list, or None), which keeps them until the next wait. 1, 0 or -1 as Arg::take.
int take_all(Arg* args, PyObject* const* objects, const char* types, int count, PyObject* held, int* kind) {
  int k = kNone;
  for (int i = 0; i < count; ++i) {
    const int r = args[i].take(objects[i], types[i]);
    if (r != 1) return r;
    if (args[i].kind == kNone) continue;
    if (k != kNone && k != args[i].kind) return 0;
    k = args[i].kind;
  }
  *kind = k == kNone ? (int)kHost : k;
  if (*kind == kDevice) {
    if (!torch_is_done()) return -1;
    if (held != Py_None)
      for (int i = 0; i < count; ++i)
        if (args[i].device_tensor && PyList_Append(held, args[i].device_tensor) != 0) return -1;
  }
  return 1;
}

#define NOT_QUICK(r)                 \
  do {                               \
    const int r_ = (r);              \
    if (r_ < 0) return nullptr;      \
    if (r_ == 0) Py_RETURN_NONE;     \
  } while (0)

bool want(Py_ssize_t got, Py_ssize_t n) {
  if (got == n) return true;
  PyErr_Format(PyExc_TypeError, "%zd arguments expected, %zd given", n, got);
  return false;
}

// a status, or, for the calls that answer a size: the size when the status is 0, else (status, size)
PyObject* sized(int rc, size_t got) {
  if (rc == PSKV_OK) return PyLong_FromSize_t(got);
  return Py_BuildValue("(in)", rc, (Py_ssize_t)got);
}

// table_push(table, keys, vals, lens, held)
PyObject* table_push(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!want(n, 5)) return nullptr;
  pskv_table* t = static_cast<pskv_table*>(PyLong_AsVoidPtr(a[0]));
  if (PyErr_Occurred()) return nullptr;
  Arg x[3];
  int kind, rc;
  NOT_QUICK(take_all(x, a + 1, "kfi", 3, a[4], &kind));
  Py_BEGIN_ALLOW_THREADS;
  rc = pskv_push(t, static_cast<uint64_t*>(x[0].ptr), x[0].n, static_cast<float*>(x[1].ptr), x[1].n,
                 static_cast<int32_t*>(x[2].ptr), x[2].n, kind);
  Py_END_ALLOW_THREADS;
  return PyLong_FromLong(rc);
}

// table_pull(table, keys, out, out_lens, held)
PyObject* table_pull(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!want(n, 5)) return nullptr;
  pskv_table* t = static_cast<pskv_table*>(PyLong_AsVoidPtr(a[0]));
  if (PyErr_Occurred()) return nullptr;
  Arg x[3];
  int kind, rc;
  size_t got = 0;
  NOT_QUICK(take_all(x, a + 1, "kfi", 3, a[4], &kind));
  Py_BEGIN_ALLOW_THREADS;
  rc = pskv_pull(t, static_cast<uint64_t*>(x[0].ptr), x[0].n, static_cast<float*>(x[1].ptr), x[1].n,
                 static_cast<int32_t*>(x[2].ptr), &got, kind);
  Py_END_ALLOW_THREADS;
  return sized(rc, got);
}

// table_pushpull(table, keys, vals, lens, out, out_lens, held)
PyObject* table_pushpull(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!want(n, 7)) return nullptr;
  pskv_table* t = static_cast<pskv_table*>(PyLong_AsVoidPtr(a[0]));
  if (PyErr_Occurred()) return nullptr;
  Arg x[5];
  int kind, rc;
  size_t got = 0;
  NOT_QUICK(take_all(x, a + 1, "kfifi", 5, a[6], &kind));
  Py_BEGIN_ALLOW_THREADS;
  rc = pskv_pushpull(t, static_cast<uint64_t*>(x[0].ptr), x[0].n, static_cast<float*>(x[1].ptr), x[1].n,
                     static_cast<int32_t*>(x[2].ptr), x[2].n, static_cast<float*>(x[3].ptr), x[3].n,
                     static_cast<int32_t*>(x[4].ptr), &got, kind);
  Py_END_ALLOW_THREADS;
  return sized(rc, got);
}

// The tables of a group and the positions that its calls share: host arrays of S+1 entries (None: null).
struct GroupArgs {
  pskv_table* const* tables;
  size_t S;
  bool parse(PyObject* tables_at, PyObject* count) {
    tables = static_cast<pskv_table* const*>(PyLong_AsVoidPtr(tables_at));
    S = PyLong_AsSize_t(count);
    return !PyErr_Occurred();
  }
  // 1 / 0 / -1: a host array with at least S + 1 entries
  int positions(Arg* p, PyObject* o) {
    const int r = p->take(o, 'k');
    if (r != 1) return r;
    return p->kind == kNone || (p->kind == kHost && p->n >= S + 1) ? 1 : 0;
  }
};

// Every tensor of a group's call lives on the device.
int on_device(const Arg* x, int count) {
  for (int i = 0; i < count; ++i)
    if (x[i].kind == kHost) return 0;
  return 1;
}

// group_push(tables, S, keys, vals, lens, pos, val_pos, held)
PyObject* group_push(PyObject*, PyObject* const* a, Py_ssize_t n) {
  GroupArgs g;
  if (!want(n, 8) || !g.parse(a[0], a[1])) return nullptr;
  Arg x[3], pos, val_pos;
  int kind, rc;
  NOT_QUICK(g.positions(&pos, a[5]));
  NOT_QUICK(g.positions(&val_pos, a[6]));
  NOT_QUICK(take_all(x, a + 2, "kfi", 3, a[7], &kind));
  NOT_QUICK(on_device(x, 3));
  Py_BEGIN_ALLOW_THREADS;
  rc = pskv_push_multi(g.tables, g.S, static_cast<uint64_t*>(x[0].ptr), static_cast<uint64_t*>(pos.ptr),
                       static_cast<float*>(x[1].ptr), static_cast<uint64_t*>(val_pos.ptr),
                       static_cast<int32_t*>(x[2].ptr), PSKV_MEM_DEVICE);
  Py_END_ALLOW_THREADS;
  return PyLong_FromLong(rc);
}

// group_pull(tables, S, keys, out, out_lens, pos, out_pos, sizes, held)
PyObject* group_pull(PyObject*, PyObject* const* a, Py_ssize_t n) {
  GroupArgs g;
  if (!want(n, 9) || !g.parse(a[0], a[1])) return nullptr;
  Arg x[3], pos, out_pos, sizes;
  int kind, rc;
  NOT_QUICK(g.positions(&pos, a[5]));
  NOT_QUICK(g.positions(&out_pos, a[6]));
  NOT_QUICK(sizes.take(a[7], 'k'));
  NOT_QUICK(take_all(x, a + 2, "kfi", 3, a[8], &kind));
  NOT_QUICK(on_device(x, 3));
  Py_BEGIN_ALLOW_THREADS;
  rc = pskv_pull_multi(g.tables, g.S, static_cast<uint64_t*>(x[0].ptr), static_cast<uint64_t*>(pos.ptr),
                       static_cast<float*>(x[1].ptr), static_cast<uint64_t*>(out_pos.ptr),
                       static_cast<int32_t*>(x[2].ptr), static_cast<uint64_t*>(sizes.ptr), PSKV_MEM_DEVICE);
  Py_END_ALLOW_THREADS;
  return PyLong_FromLong(rc);
}

// group_pushpull(tables, S, keys, vals, lens, out, out_lens, pos, val_pos, out_pos, sizes, held)
PyObject* group_pushpull(PyObject*, PyObject* const* a, Py_ssize_t n) {
  GroupArgs g;
  if (!want(n, 12) || !g.parse(a[0], a[1])) return nullptr;
  Arg x[5], pos, val_pos, out_pos, sizes;
  int kind, rc;
  NOT_QUICK(g.positions(&pos, a[7]));
  NOT_QUICK(g.positions(&val_pos, a[8]));
  NOT_QUICK(g.positions(&out_pos, a[9]));
  NOT_QUICK(sizes.take(a[10], 'k'));
  NOT_QUICK(take_all(x, a + 2, "kfifi", 5, a[11], &kind));
  NOT_QUICK(on_device(x, 5));
  Py_BEGIN_ALLOW_THREADS;
  rc = pskv_pushpull_multi(g.tables, g.S, static_cast<uint64_t*>(x[0].ptr), static_cast<uint64_t*>(pos.ptr),
                           static_cast<float*>(x[1].ptr), static_cast<uint64_t*>(val_pos.ptr),
                           static_cast<int32_t*>(x[2].ptr), static_cast<float*>(x[3].ptr),
                           static_cast<uint64_t*>(out_pos.ptr), static_cast<int32_t*>(x[4].ptr),
                           static_cast<uint64_t*>(sizes.ptr), PSKV_MEM_DEVICE);
  Py_END_ALLOW_THREADS;
  return PyLong_FromLong(rc);
}

// slice(device, keys, lens, nvals, range_begin, range_end): (pos, val_pos, used), or a status
PyObject* slice(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!want(n, 6)) return nullptr;
  const long device = PyLong_AsLong(a[0]);
  const size_t nvals = PyLong_AsSize_t(a[3]);
  if (PyErr_Occurred()) {  // (a numpy integer, say)
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  Arg x[2], begin, end;
  int kind, rc;
  NOT_QUICK(begin.take(a[4], 'k'));
  NOT_QUICK(end.take(a[5], 'k'));
  const size_t S = begin.n;
  if (begin.kind != kHost || end.kind != kHost || end.n != S) Py_RETURN_NONE;
  NOT_QUICK(take_all(x, a + 1, "ki", 2, Py_None, &kind));
  npy_intp bounds = (npy_intp)S + 1, ranges = (npy_intp)S;
  PyObject* pos = PyArray_SimpleNew(1, &bounds, NPY_UINT64);
  PyObject* val_pos = PyArray_SimpleNew(1, &bounds, NPY_UINT64);
  PyObject* used = PyArray_SimpleNew(1, &ranges, NPY_UINT8);
  PyObject* result = nullptr;
  if (pos && val_pos && used) {
    uint64_t* p = static_cast<uint64_t*>(PyArray_DATA(reinterpret_cast<PyArrayObject*>(pos)));
    uint64_t* v = static_cast<uint64_t*>(PyArray_DATA(reinterpret_cast<PyArrayObject*>(val_pos)));
    uint8_t* u = static_cast<uint8_t*>(PyArray_DATA(reinterpret_cast<PyArrayObject*>(used)));
    Py_BEGIN_ALLOW_THREADS;
    rc = pskv_slice((int)device, static_cast<uint64_t*>(x[0].ptr), x[0].n, static_cast<int32_t*>(x[1].ptr), x[1].n,
                    nvals, static_cast<uint64_t*>(begin.ptr), static_cast<uint64_t*>(end.ptr), S, p, v, u, kind);
    Py_END_ALLOW_THREADS;
    result = rc ? PyLong_FromLong(rc) : PyTuple_Pack(3, pos, val_pos, used);
  }
  Py_XDECREF(pos);
  Py_XDECREF(val_pos);
  Py_XDECREF(used);
  return result;
}

// match(device, src_keys, src_vals, dst_keys, dst_vals, k, op)
PyObject* match(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!want(n, 7)) return nullptr;
  const long device = PyLong_AsLong(a[0]), op = PyLong_AsLong(a[6]);
  const size_t k = PyLong_AsSize_t(a[5]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  Arg x[4];
  int kind, rc;
  uint64_t got = 0;
  NOT_QUICK(take_all(x, a + 1, "kfkf", 4, Py_None, &kind));
  if (x[1].n != x[0].n * k || x[3].n != x[2].n * k) Py_RETURN_NONE;
  Py_BEGIN_ALLOW_THREADS;
  rc = pskv_match((int)device, static_cast<uint64_t*>(x[0].ptr), x[0].n, static_cast<float*>(x[1].ptr),
                  static_cast<uint64_t*>(x[2].ptr), x[2].n, static_cast<float*>(x[3].ptr), k, (int)op, &got, nullptr,
                  kind);
  Py_END_ALLOW_THREADS;
  return sized(rc, got);
}

// replay_run(recording)
PyObject* replay_run(PyObject*, PyObject* at) {
  pskv_replay* r = static_cast<pskv_replay*>(PyLong_AsVoidPtr(at));
  if (PyErr_Occurred()) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = pskv_replay_run(r);
  Py_END_ALLOW_THREADS;
  return PyLong_FromLong(rc);
}

// setup(tensor_type, int64, uint64, float32, int32, raw_stream)
PyObject* setup(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!want(n, 6)) return nullptr;
  PyObject** to[6] = {&g_tensor_type, &g_int64, &g_uint64, &g_float32, &g_int32, &g_raw_stream};
  for (int i = 0; i < 6; ++i) {
    Py_INCREF(a[i]);
    Py_XDECREF(*to[i]);
    *to[i] = a[i];
  }
  Py_RETURN_NONE;
}

#define FAST(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(setup),      FAST(table_push), FAST(table_pull),     FAST(table_pushpull),
                         FAST(group_push), FAST(group_pull), FAST(group_pushpull), FAST(slice),
                         FAST(match),      {"replay_run", replay_run, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
  import_array();
  s_dtype = PyUnicode_InternFromString("dtype");
  s_is_cuda = PyUnicode_InternFromString("is_cuda");
  s_is_contiguous = PyUnicode_InternFromString("is_contiguous");
  s_numel = PyUnicode_InternFromString("numel");
  s_data_ptr = PyUnicode_InternFromString("data_ptr");
  if (!s_dtype || !s_is_cuda || !s_is_contiguous || !s_numel || !s_data_ptr) return nullptr;
  return PyModule_Create(&module);
}

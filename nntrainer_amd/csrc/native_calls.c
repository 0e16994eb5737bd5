/* SPDX-License-Identifier: Apache-2.0 */
/**
 * @file   native_calls.c
 * @brief  The matmul calls of capi.py as native functions.
 *
 * A decode step makes three library calls a layer of a few microseconds of GPU time each. Through ctypes
 * a call spent 2.0 us (one weight) to 5.4 us (three weights: three arrays of handles, addresses and strides)
 * on marshalling, more than the library's own work for a launch, and the stream ran dry: a token through the
 * 28 layers of a 1024-wide decoder took 450 to 520 us for 415 us of kernels. Here the same calls take 0.3 to
 * 0.6 us. Arguments, defaults and errors are those of the functions' ctypes form in capi.py, which an interpreter
 * without this module uses; the global interpreter lock is released during the call, as ctypes does.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#include "hipq.h"

typedef hipq_weight_t weight_t;
enum { MEM_DEVICE = HIPQ_MEM_DEVICE, MAX_STACK = 16 };

/* the library's entry points; their types are the header's */
static __typeof__(&hipq_matmul) f_matmul;
static __typeof__(&hipq_matmul_each_row) f_each_row;
static __typeof__(&hipq_matmul_noalloc) f_noalloc;
static __typeof__(&hipq_matmul_multi) f_multi;
static __typeof__(&hipq_mlp_swiglu) f_swiglu;
static __typeof__(&hipq_mlp_swiglu_down) f_swiglu_down;
static PyObject *load, *raise_status; /* capi.lib, check */
static PyObject *pointer_of, *int_of; /* capi._pointer_of, _int_of: the rarer forms of a stream and an integer */
static PyObject *s_h, *s_handle, *s_value, *s_n, *s_k, *s_data_ptr, *s_ctypes, *s_data;

/* The address of a buffer as capi._addr takes it: None, an int, a torch tensor, a numpy array; nothing else has one
 * (a numpy scalar, bytes and a ctypes object raise AttributeError). */
static int get_addr(PyObject *x, void **out) {
  if (!x || x == Py_None) {
    *out = NULL;
    return 0;
  }
  if (PyLong_Check(x)) {
    *out = PyLong_AsVoidPtr(x);
    return PyErr_Occurred() ? -1 : 0;
  }
  PyObject *p = PyObject_CallMethodNoArgs(x, s_data_ptr);
  if (!p) {
    if (!PyErr_ExceptionMatches(PyExc_AttributeError)) return -1;
    PyErr_Clear();
    /* .ctypes.data, as numpy's arrays (and no other buffer) have it; a C-contiguous array's is the start of its buffer,
     * which is had without the object that .ctypes makes */
    Py_buffer view;
    if (PyObject_HasAttr((PyObject *)Py_TYPE(x), s_ctypes) && PyObject_CheckBuffer(x)) {
      if (PyObject_GetBuffer(x, &view, PyBUF_SIMPLE) == 0) {
        *out = view.buf;
        PyBuffer_Release(&view);
        return 0;
      }
      PyErr_Clear();
    }
    PyObject *c = PyObject_GetAttr(x, s_ctypes);
    if (!c) return -1;
    p = PyObject_GetAttr(c, s_data);
    Py_DECREF(c);
    if (!p) return -1;
  }
  *out = PyLong_AsVoidPtr(p);
  Py_DECREF(p);
  return PyErr_Occurred() ? -1 : 0;
}

/* A stream: None, an int, or whatever ctypes takes for a c_void_p argument (a c_void_p means its value; an object with
 * _as_parameter_, torch's streams among them, that parameter). */
static int get_stream(PyObject *x, void **out) {
  if (!x || x == Py_None) {
    *out = NULL;
    return 0;
  }
  PyObject *p = NULL;
  if (!PyLong_Check(x) && !(x = p = PyObject_CallOneArg(pointer_of, x))) return -1;
  *out = PyLong_AsVoidPtr(x);
  Py_XDECREF(p);
  return PyErr_Occurred() ? -1 : 0;
}

static int get_int(PyObject *x, int64_t *out) {
  PyObject *p = NULL;
  if (!PyIndex_Check(x) && !(x = p = PyObject_CallOneArg(int_of, x))) return -1; /* a ctypes integer */
  *out = PyLong_AsLongLong(x);
  Py_XDECREF(p);
  return *out == -1 && PyErr_Occurred() ? -1 : 0;
}
static int get_attr_int(PyObject *x, PyObject *name, int64_t *out) {
  PyObject *p = PyObject_GetAttr(x, name);
  if (!p) return -1;
  const int rc = get_int(p, out);
  Py_DECREF(p);
  return rc;
}
/* a stride argument: `dflt` of the weight where it is None or 0 */
static int get_stride(PyObject *x, PyObject *w, PyObject *dflt, int64_t *out) {
  if (x && x != Py_None) {
    if (get_int(x, out)) return -1;
    if (*out) return 0;
  }
  return get_attr_int(w, dflt, out);
}
/* the handle of a capi.Weight: its _h is a ctypes.c_void_p (null once destroyed); of another object its `handle` */
static int get_weight(PyObject *w, weight_t *out) {
  void *p = NULL;
  int rc = 0;
  PyObject *h = PyObject_GetAttr(w, s_h);
  if (h) {
    PyObject *v = PyObject_GetAttr(h, s_value);
    if (!v) rc = -1;
    if (v && v != Py_None) p = PyLong_AsVoidPtr(v);
    Py_XDECREF(v);
  } else {
    if (!PyErr_ExceptionMatches(PyExc_AttributeError)) return -1;
    PyErr_Clear();
    if (!(h = PyObject_GetAttr(w, s_handle))) return -1;
    rc = get_stream(h, &p); /* the forms of a pointer argument */
  }
  Py_DECREF(h);
  *out = (weight_t)p;
  return rc || PyErr_Occurred() ? -1 : 0;
}

/* Positional and keyword arguments into slots by the names of `kw` (null-terminated, `need` required). */
static int parse(const char *fn, const char *const *kw, int need, PyObject *const *args, Py_ssize_t nargs, PyObject *names,
                 PyObject **slot, int nslot) {
  if (nargs > nslot) {
    PyErr_Format(PyExc_TypeError, "%s() takes at most %d arguments (%zd given)", fn, nslot, nargs);
    return -1;
  }
  for (int i = 0; i < nslot; ++i) slot[i] = i < nargs ? args[i] : NULL;
  const Py_ssize_t nk = names ? PyTuple_GET_SIZE(names) : 0;
  for (Py_ssize_t j = 0; j < nk; ++j) {
    PyObject *name = PyTuple_GET_ITEM(names, j);
    int i = 0;
    while (i < nslot && PyUnicode_CompareWithASCIIString(name, kw[i])) ++i;
    if (i == nslot) {
      PyErr_Format(PyExc_TypeError, "%s() got an unexpected keyword argument '%U'", fn, name);
      return -1;
    }
    if (slot[i]) {
      PyErr_Format(PyExc_TypeError, "%s() got multiple values for argument '%U'", fn, name);
      return -1;
    }
    slot[i] = args[nargs + j];
  }
  for (int i = 0; i < need; ++i)
    if (!slot[i]) {
      PyErr_Format(PyExc_TypeError, "%s() missing required argument '%s'", fn, kw[i]);
      return -1;
    }
  return 0;
}

static PyObject *finish(int rc) {
  if (rc == 0) Py_RETURN_NONE;
  PyObject *r = PyObject_CallFunction(raise_status, "i", rc);
  if (r) { /* it raises */
    Py_DECREF(r);
    PyErr_Format(PyExc_RuntimeError, "library status %d", rc);
  }
  return NULL;
}

static int ready(void) { /* the first call loads the library, which binds the entry points */
  if (f_matmul) return 0;
  PyObject *r = load ? PyObject_CallNoArgs(load) : NULL;
  Py_XDECREF(r);
  if (r && f_matmul) return 0;
  if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "the library is not loaded");
  return -1;
}

static PyObject *one_weight(int each_row, PyObject *const *args, Py_ssize_t nargs, PyObject *names) {
  static const char *const kw_m[] = {"w", "a", "m", "c", "lda", "ldc", "mem", "stream"};
  static const char *const kw_r[] = {"w", "a", "rows", "c", "lda", "ldc", "mem", "stream"};
  PyObject *s[8];
  weight_t w;
  void *a, *c, *stream;
  int64_t m, lda, ldc, mem = MEM_DEVICE;
  if (ready() || parse(each_row ? "matmul_each_row" : "matmul", each_row ? kw_r : kw_m, 4, args, nargs, names, s, 8) ||
      get_weight(s[0], &w) || get_addr(s[1], &a) || get_int(s[2], &m) || get_addr(s[3], &c) ||
      get_stride(s[4], s[0], s_k, &lda) || get_stride(s[5], s[0], s_n, &ldc) || (s[6] && get_int(s[6], &mem)) ||
      get_stream(s[7], &stream))
    return NULL;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = (each_row ? f_each_row : f_matmul)(w, (const float *)a, m, lda, (float *)c, ldc, (int)mem, stream);
  Py_END_ALLOW_THREADS
  return finish(rc);
}
static PyObject *matmul(PyObject *self, PyObject *const *args, Py_ssize_t nargs, PyObject *names) {
  return one_weight(0, args, nargs, names);
}
static PyObject *matmul_each_row(PyObject *self, PyObject *const *args, Py_ssize_t nargs, PyObject *names) {
  return one_weight(1, args, nargs, names);
}

static PyObject *matmul_noalloc(PyObject *self, PyObject *const *args, Py_ssize_t nargs, PyObject *names) {
  static const char *const kw[] = {"w", "a", "m", "c", "lda", "ldc", "stream"};
  PyObject *s[7];
  weight_t w;
  void *a, *c, *stream;
  int64_t m, lda, ldc;
  if (ready() || parse("matmul_noalloc", kw, 4, args, nargs, names, s, 7) || get_weight(s[0], &w) || get_addr(s[1], &a) ||
      get_int(s[2], &m) || get_addr(s[3], &c) || get_stride(s[4], s[0], s_k, &lda) || get_stride(s[5], s[0], s_n, &ldc) ||
      get_stream(s[6], &stream))
    return NULL;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f_noalloc(w, (const float *)a, m, lda, (float *)c, ldc, stream);
  Py_END_ALLOW_THREADS
  return finish(rc);
}

static PyObject *matmul_multi(PyObject *self, PyObject *const *args, Py_ssize_t nargs, PyObject *names) {
  static const char *const kw[] = {"ws", "a", "m", "cs", "ldc", "mem", "stream", "lda"};
  PyObject *s[8], *ws = NULL, *cs = NULL, *ld = NULL, *result = NULL;
  if (ready() || parse("matmul_multi", kw, 4, args, nargs, names, s, 8)) return NULL;
  weight_t hs[MAX_STACK], *h = hs;
  float *cps[MAX_STACK], **cp = cps;
  int64_t lds[MAX_STACK], *l = lds;
  void *a, *stream, *heap = NULL;
  int64_t m, lda, mem = MEM_DEVICE;
  const int has_ldc = s[4] && s[4] != Py_None;
  if (!(ws = PySequence_Fast(s[0], "ws is a sequence of weights")) || !(cs = PySequence_Fast(s[3], "cs is a sequence of outputs")) ||
      (has_ldc && !(ld = PySequence_Fast(s[4], "ldc is a sequence of strides"))))
    goto out;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(ws);
  if (n < 1 || PySequence_Fast_GET_SIZE(cs) != n || (has_ldc && PySequence_Fast_GET_SIZE(ld) != n)) {
    PyErr_SetString(PyExc_ValueError, "one output (and stride) for each weight, and at least one");
    goto out;
  }
  if (n > MAX_STACK) {
    if (!(heap = PyMem_Malloc((size_t)n * (sizeof *h + sizeof *cp + sizeof *l)))) {
      PyErr_NoMemory();
      goto out;
    }
    l = (int64_t *)heap;
    h = (weight_t *)(l + n);
    cp = (float **)(h + n);
  }
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject *w = PySequence_Fast_GET_ITEM(ws, i);
    void *p;
    if (get_weight(w, &h[i]) || get_addr(PySequence_Fast_GET_ITEM(cs, i), &p) ||
        (has_ldc ? get_int(PySequence_Fast_GET_ITEM(ld, i), &l[i]) : get_attr_int(w, s_n, &l[i])))
      goto out;
    cp[i] = (float *)p;
  }
  if (get_addr(s[1], &a) || get_int(s[2], &m) || (s[5] && get_int(s[5], &mem)) || get_stream(s[6], &stream) ||
      get_stride(s[7], PySequence_Fast_GET_ITEM(ws, 0), s_k, &lda))
    goto out;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f_multi((int)n, h, (const float *)a, m, lda, cp, l, (int)mem, stream);
  Py_END_ALLOW_THREADS
  result = finish(rc);
out:
  PyMem_Free(heap);
  Py_XDECREF(ws);
  Py_XDECREF(cs);
  Py_XDECREF(ld);
  return result;
}

static PyObject *mlp_swiglu(PyObject *self, PyObject *const *args, Py_ssize_t nargs, PyObject *names) {
  static const char *const kw[] = {"w_act", "w_mul", "a", "m", "out", "lda", "ldo", "mem", "stream"};
  PyObject *s[9];
  weight_t wa, wm;
  void *a, *o, *stream;
  int64_t m, lda, ldo, mem = MEM_DEVICE;
  if (ready() || parse("mlp_swiglu", kw, 5, args, nargs, names, s, 9) || get_weight(s[0], &wa) || get_weight(s[1], &wm) ||
      get_addr(s[2], &a) || get_int(s[3], &m) || get_addr(s[4], &o) || get_stride(s[5], s[0], s_k, &lda) ||
      get_stride(s[6], s[0], s_n, &ldo) || (s[7] && get_int(s[7], &mem)) || get_stream(s[8], &stream))
    return NULL;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f_swiglu(wa, wm, (const float *)a, m, lda, (float *)o, ldo, (int)mem, stream);
  Py_END_ALLOW_THREADS
  return finish(rc);
}

static PyObject *mlp_swiglu_down(PyObject *self, PyObject *const *args, Py_ssize_t nargs, PyObject *names) {
  static const char *const kw[] = {"w_act", "w_mul", "w_down", "a", "m", "out", "lda", "ldo", "mem", "stream"};
  PyObject *s[10];
  weight_t wa, wm, wd;
  void *a, *o, *stream;
  int64_t m, lda, ldo, mem = MEM_DEVICE;
  if (ready() || parse("mlp_swiglu_down", kw, 6, args, nargs, names, s, 10) || get_weight(s[0], &wa) ||
      get_weight(s[1], &wm) || get_weight(s[2], &wd) || get_addr(s[3], &a) || get_int(s[4], &m) || get_addr(s[5], &o) ||
      get_stride(s[6], s[0], s_k, &lda) || get_stride(s[7], s[2], s_n, &ldo) || (s[8] && get_int(s[8], &mem)) ||
      get_stream(s[9], &stream))
    return NULL;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f_swiglu_down(wa, wm, wd, (const float *)a, m, lda, (float *)o, ldo, (int)mem, stream);
  Py_END_ALLOW_THREADS
  return finish(rc);
}

/* setup(lib, check, pointer_of, int_of): the functions of capi.py that are needed here */
static PyObject *setup(PyObject *self, PyObject *args) {
  PyObject *p[4];
  if (!PyArg_ParseTuple(args, "OOOO", &p[0], &p[1], &p[2], &p[3])) return NULL;
  for (int i = 0; i < 4; ++i) Py_INCREF(p[i]);
  Py_XSETREF(load, p[0]);
  Py_XSETREF(raise_status, p[1]);
  Py_XSETREF(pointer_of, p[2]);
  Py_XSETREF(int_of, p[3]);
  Py_RETURN_NONE;
}
/* bind(addresses of the six entry points in the order of the pointers above) */
static PyObject *bind(PyObject *self, PyObject *args) {
  unsigned long long p[6];
  if (!PyArg_ParseTuple(args, "KKKKKK", &p[0], &p[1], &p[2], &p[3], &p[4], &p[5])) return NULL;
  *(void **)&f_matmul = (void *)(uintptr_t)p[0];
  *(void **)&f_each_row = (void *)(uintptr_t)p[1];
  *(void **)&f_noalloc = (void *)(uintptr_t)p[2];
  *(void **)&f_multi = (void *)(uintptr_t)p[3];
  *(void **)&f_swiglu = (void *)(uintptr_t)p[4];
  *(void **)&f_swiglu_down = (void *)(uintptr_t)p[5];
  Py_RETURN_NONE;
}

#define FAST(name, doc) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL | METH_KEYWORDS, doc}
static PyMethodDef methods[] = {
  FAST(matmul, "matmul(w, a, m, c, lda=None, ldc=None, mem=MEM_DEVICE, stream=None)"),
  FAST(matmul_each_row, "matmul_each_row(w, a, rows, c, lda=None, ldc=None, mem=MEM_DEVICE, stream=None)\n\n"
                        "`rows` independent one-row products in one call (the bits of `rows` calls of matmul with m = 1)."),
  FAST(matmul_noalloc, "matmul_noalloc(w, a, m, c, lda=None, ldc=None, stream=None)\n\n"
                       "hipq_matmul on device buffers with the quantized activations in the library's fixed scratch array: no "
                       "device allocation inside the call."),
  FAST(matmul_multi, "matmul_multi(ws, a, m, cs, ldc=None, mem=MEM_DEVICE, stream=None, lda=None)"),
  FAST(mlp_swiglu, "mlp_swiglu(w_act, w_mul, a, m, out, lda=None, ldo=None, mem=MEM_DEVICE, stream=None)\n\n"
                   "out = swiglu(a . w_act^T, a . w_mul^T): the gated half of a dense MLP in one call."),
  FAST(mlp_swiglu_down, "mlp_swiglu_down(w_act, w_mul, w_down, a, m, out, lda=None, ldo=None, mem=MEM_DEVICE, stream=None)\n\n"
                        "out = swiglu(a . w_act^T, a . w_mul^T) . w_down^T: the gated MLP of a decoder layer in one call."),
  {"setup", setup, METH_VARARGS, "setup(lib, check, pointer_of, int_of)"},
  {"bind", bind, METH_VARARGS, "bind(six entry points' addresses)"},
  {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "hipq_native", "The matmul calls of capi.py.", -1, methods};

PyMODINIT_FUNC PyInit_hipq_native(void) {
  s_h = PyUnicode_InternFromString("_h");
  s_handle = PyUnicode_InternFromString("handle");
  s_value = PyUnicode_InternFromString("value");
  s_n = PyUnicode_InternFromString("n");
  s_k = PyUnicode_InternFromString("k");
  s_data_ptr = PyUnicode_InternFromString("data_ptr");
  s_ctypes = PyUnicode_InternFromString("ctypes");
  s_data = PyUnicode_InternFromString("data");
  if (!s_h || !s_handle || !s_value || !s_n || !s_k || !s_data_ptr || !s_ctypes || !s_data) return NULL;
  return PyModule_Create(&module);
}

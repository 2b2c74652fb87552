/* kh_pyops.c - the operator calls of a decoder layer (kuiperllama_amd/ops.py) from Python to the C-ABI without ctypes: checks of
 * the tensors, conversions and the call in one C function each.  A call through ctypes took 4.9 us on the host, 2.5 of them the
 * launch itself; a layer is 14 calls of kernels that run for 2 to 14 us each.
 *
 * Knows nothing of torch's C++ interface: tensors are asked through their Python attributes, as ops.py asked them.  The addresses
 * of the C-ABI's functions come from the ctypes handle (bind), so that there is one libkuiper_hip.so in a process. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

static PyObject *s_dtype, *s_is_cuda, *s_is_contiguous, *s_data_ptr, *s_numel, *s_shape;
/* from bind() */
static PyObject *o_f32, *o_i32, *o_i8, *o_tensor, *o_device, *o_raw_stream, *o_stream, *o_check, *o_arg_error;

typedef int (*add_fn)(const void*, const void*, void*, int32_t, void*);
typedef int (*matmul_fn)(const void*, const void*, void*, int32_t, int32_t, float, void*);
typedef int (*matmul_q8_fn)(const void*, const void*, const void*, int32_t, void*, int32_t, int32_t, void*);
typedef int (*rmsnorm_fn)(const void*, const void*, void*, int32_t, float, void*);
typedef int (*rope_fn)(int32_t, int32_t, int32_t, void*, void*, const void*, int32_t, const void*, const void*, int32_t, void*);
typedef int (*mha_fn)(const void*, int32_t, int32_t, int32_t, int32_t, int32_t, int32_t, int32_t, void*, const void*, void*, const void*,
                      const void*, void*);
static add_fn f_add, f_swiglu;
static matmul_fn f_matmul;
static matmul_q8_fn f_matmul_q8;
static rmsnorm_fn f_rmsnorm;
static rope_fn f_rope;
static mha_fn f_mha;

/* The address of a tensor on the GPU, contiguous and of the type; None: null.  0, or -1 with an exception. */
static int ptr(PyObject* t, PyObject* dtype, void** out) {
  *out = NULL;
  if (t == Py_None) return 0;
  PyObject* v = PyObject_GetAttr(t, s_is_cuda);
  if (!v) return -1;
  int yes = PyObject_IsTrue(v);
  Py_DECREF(v);
  if (yes < 0) return -1;
  if (!yes) {
    PyErr_SetString(PyExc_ValueError, "kuiperllama_amd.ops: tensors must be on the GPU (no CPU fallback)");
    return -1;
  }
  if (!(v = PyObject_VectorcallMethod(s_is_contiguous, &t, 1 | PY_VECTORCALL_ARGUMENTS_OFFSET, NULL))) return -1;
  yes = PyObject_IsTrue(v);
  Py_DECREF(v);
  if (yes < 0) return -1;
  if (!yes) {
    PyErr_SetString(PyExc_ValueError, "kuiperllama_amd.ops: tensors must be contiguous");
    return -1;
  }
  if (!(v = PyObject_GetAttr(t, s_dtype))) return -1;
  yes = v == dtype ? 1 : PyObject_RichCompareBool(v, dtype, Py_EQ);
  if (yes == 0) PyErr_Format(PyExc_TypeError, "expected %S, got %S", dtype, v);
  Py_DECREF(v);
  if (yes <= 0) return -1;
  if (!(v = PyObject_VectorcallMethod(s_data_ptr, &t, 1 | PY_VECTORCALL_ARGUMENTS_OFFSET, NULL))) return -1;
  *out = PyLong_AsVoidPtr(v);
  Py_DECREF(v);
  return *out == NULL && PyErr_Occurred() ? -1 : 0;
}
/* Numbers as ctypes takes them: integers masked to 32 bits, no floats for integers. */
static int wrong(const char* what) {
  PyErr_Clear();
  PyErr_Format(o_arg_error, "%s expected", what);
  return -1;
}
static int i32(PyObject* o, int32_t* out) {
  if (PyFloat_Check(o)) return wrong("int");
  const unsigned long v = PyLong_AsUnsignedLongMask(o);
  if (v == (unsigned long)-1 && PyErr_Occurred()) return wrong("int");
  *out = (int32_t)(uint32_t)v;
  return 0;
}
static int f32(PyObject* o, float* out) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) return wrong("float");
  *out = (float)v;
  return 0;
}
static int numel(PyObject* t, int32_t* out) {
  PyObject* v = PyObject_VectorcallMethod(s_numel, &t, 1 | PY_VECTORCALL_ARGUMENTS_OFFSET, NULL);
  if (!v) return -1;
  const int rc = i32(v, out);
  Py_DECREF(v);
  return rc;
}
/* rows and columns of a matrix */
static int shape2(PyObject* t, int32_t* rows, int32_t* cols) {
  PyObject* v = PyObject_GetAttr(t, s_shape);
  if (!v) return -1;
  int rc = -1;
  if (!PyTuple_Check(v) || PyTuple_GET_SIZE(v) != 2) PyErr_SetString(PyExc_ValueError, "a matrix is expected (two dimensions to unpack)");
  else rc = i32(PyTuple_GET_ITEM(v, 0), rows) || i32(PyTuple_GET_ITEM(v, 1), cols) ? -1 : 0;
  Py_DECREF(v);
  return rc;
}
/* torch's current stream of the current device */
static int stream(void** out) {
  PyObject* v;
  if (o_raw_stream != Py_None) {
    PyObject* d = PyObject_CallNoArgs(o_device);
    if (!d) return -1;
    v = PyObject_CallOneArg(o_raw_stream, d);
    Py_DECREF(d);
  } else {
    v = PyObject_CallNoArgs(o_stream);
  }
  if (!v) return -1;
  *out = PyLong_AsVoidPtr(v);
  Py_DECREF(v);
  return *out == NULL && PyErr_Occurred() ? -1 : 0;
}
/* a device tensor of one int32 or a number */
static int position(PyObject* o, void** d_pos, int32_t* pos) {
  *d_pos = NULL;
  *pos = 0;
  if (!PyLong_CheckExact(o)) {
    const int is = PyObject_IsInstance(o, o_tensor);
    if (is < 0) return -1;
    if (is) return ptr(o, o_i32, d_pos);
    PyObject* v = PyNumber_Long(o);
    if (!v) return -1;
    const int rc = i32(v, pos);
    Py_DECREF(v);
    return rc;
  }
  return i32(o, pos);
}
/* raises what the library reports, else returns a new reference to `out` */
static PyObject* done(int rc, const char* what, PyObject* out) {
  if (rc) {
    PyObject* v = PyObject_CallFunction(o_check, "is", rc, what);
    if (!v) return NULL;
    Py_DECREF(v);
  }
  Py_INCREF(out);
  return out;
}
static int count(Py_ssize_t n, Py_ssize_t want) {
  if (n == want) return 0;
  PyErr_Format(PyExc_TypeError, "%zd arguments expected, got %zd", want, n);
  return -1;
}
#define CALL(rc, ...)       \
  Py_BEGIN_ALLOW_THREADS    \
  rc = __VA_ARGS__;         \
  Py_END_ALLOW_THREADS

static PyObject* elementwise(PyObject* const* a, Py_ssize_t n, add_fn f, const char* name) {
  void *x, *y, *o, *s;
  int32_t len;
  int rc;
  if (count(n, 3) || ptr(a[0], o_f32, &x) || ptr(a[1], o_f32, &y) || ptr(a[2], o_f32, &o) || numel(a[0], &len) || stream(&s)) return NULL;
  CALL(rc, f(x, y, o, len, s))
  return done(rc, name, a[2]);
}
static PyObject* py_add(PyObject* m, PyObject* const* a, Py_ssize_t n) { return elementwise(a, n, f_add, "kh_add_f32"); }
static PyObject* py_swiglu(PyObject* m, PyObject* const* a, Py_ssize_t n) { return elementwise(a, n, f_swiglu, "kh_swiglu_f32"); }
static PyObject* py_matmul(PyObject* m, PyObject* const* a, Py_ssize_t n) { /* x, w, out, scale */
  void *x, *w, *o, *s;
  int32_t K, M;
  float scale;
  int rc;
  if (count(n, 4) || shape2(a[1], &K, &M) || ptr(a[0], o_f32, &x) || ptr(a[1], o_f32, &w) || ptr(a[2], o_f32, &o) || f32(a[3], &scale) ||
      stream(&s))
    return NULL;
  CALL(rc, f_matmul(x, w, o, M, K, scale, s))
  return done(rc, "kh_matmul_f32", a[2]);
}
static PyObject* py_matmul_q8(PyObject* m, PyObject* const* a, Py_ssize_t n) { /* x, w8, scales, group, out */
  void *x, *w, *sc, *o, *s;
  int32_t K, M, group;
  int rc;
  if (count(n, 5) || shape2(a[1], &K, &M) || ptr(a[0], o_f32, &x) || ptr(a[1], o_i8, &w) || ptr(a[2], o_f32, &sc) || i32(a[3], &group) ||
      ptr(a[4], o_f32, &o) || stream(&s))
    return NULL;
  CALL(rc, f_matmul_q8(x, w, sc, group, o, M, K, s))
  return done(rc, "kh_matmul_q8", a[4]);
}
static PyObject* py_rmsnorm(PyObject* m, PyObject* const* a, Py_ssize_t n) { /* x, w, out, eps */
  void *x, *w, *o, *s;
  int32_t len;
  float eps;
  int rc;
  if (count(n, 4) || ptr(a[0], o_f32, &x) || ptr(a[1], o_f32, &w) || ptr(a[2], o_f32, &o) || numel(a[0], &len) || f32(a[3], &eps) || stream(&s))
    return NULL;
  CALL(rc, f_rmsnorm(x, w, o, len, eps, s))
  return done(rc, "kh_rmsnorm_f32", a[2]);
}
static PyObject* py_rope(PyObject* m, PyObject* const* a, Py_ssize_t n) { /* q, k, pos, sin, cos, head_size, mode */
  void *q, *k, *d_pos, *sn, *cs, *s;
  int32_t pos, nq, nk, hs, mode;
  int rc;
  if (count(n, 7) || position(a[2], &d_pos, &pos) || numel(a[0], &nq) || numel(a[1], &nk) || i32(a[5], &hs) || ptr(a[0], o_f32, &q) ||
      ptr(a[1], o_f32, &k) || ptr(a[3], o_f32, &sn) || ptr(a[4], o_f32, &cs) || i32(a[6], &mode) || stream(&s))
    return NULL;
  CALL(rc, f_rope(nq, nk, hs, q, k, d_pos, pos, sn, cs, mode, s))
  return done(rc, "kh_rope_f32", Py_None);
}
/* pos, head_num, layer_index, seq_len, kv_dim, kv_mul, head_size, mha_out, q, score, kcache, vcache */
static PyObject* py_mha(PyObject* m, PyObject* const* a, Py_ssize_t n) {
  void *d_pos, *o, *q, *sc, *k, *v, *s;
  int32_t pos, i[6];
  int rc;
  if (count(n, 12) || position(a[0], &d_pos, &pos)) return NULL;
  for (int j = 0; j < 6; ++j)
    if (i32(a[1 + j], &i[j])) return NULL;
  if (ptr(a[7], o_f32, &o) || ptr(a[8], o_f32, &q) || ptr(a[9], o_f32, &sc) || ptr(a[10], o_f32, &k) || ptr(a[11], o_f32, &v) || stream(&s))
    return NULL;
  CALL(rc, f_mha(d_pos, pos, i[0], i[1], i[2], i[3], i[4], i[5], o, q, sc, k, v, s))
  return done(rc, "kh_mha_f32", a[7]);
}

static void keep(PyObject** at, PyObject* o) {
  Py_INCREF(o);
  Py_XSETREF(*at, o);
}
/* (addresses: add, swiglu, matmul, matmul_q8, rmsnorm, rope, mha), (float32, int32, int8, Tensor, current device, raw stream of a
 * device or None, current stream, check, ctypes.ArgumentError) */
static PyObject* py_bind(PyObject* m, PyObject* const* a, Py_ssize_t n) {
  void* p[7];
  PyObject** o[9] = {&o_f32, &o_i32, &o_i8, &o_tensor, &o_device, &o_raw_stream, &o_stream, &o_check, &o_arg_error};
  if (count(n, 2)) return NULL;
  if (!PyTuple_Check(a[0]) || PyTuple_GET_SIZE(a[0]) != 7 || !PyTuple_Check(a[1]) || PyTuple_GET_SIZE(a[1]) != 9) {
    PyErr_SetString(PyExc_TypeError, "seven addresses and nine objects are expected");
    return NULL;
  }
  for (int j = 0; j < 7; ++j) {
    p[j] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(a[0], j));
    if (!p[j]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "an address is null");
      return NULL;
    }
  }
  f_add = (add_fn)p[0];
  f_swiglu = (add_fn)p[1];
  f_matmul = (matmul_fn)p[2];
  f_matmul_q8 = (matmul_q8_fn)p[3];
  f_rmsnorm = (rmsnorm_fn)p[4];
  f_rope = (rope_fn)p[5];
  f_mha = (mha_fn)p[6];
  for (int j = 0; j < 9; ++j) keep(o[j], PyTuple_GET_ITEM(a[1], j));
  Py_RETURN_NONE;
}

#define METHOD(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, NULL}
static PyMethodDef methods[] = {METHOD(bind), METHOD(add),  METHOD(swiglu), METHOD(matmul), METHOD(matmul_q8),
                                METHOD(rmsnorm), METHOD(rope), METHOD(mha), {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "kh_pyops", NULL, -1, methods};
PyMODINIT_FUNC PyInit_kh_pyops(void) {
  s_dtype = PyUnicode_InternFromString("dtype");
  s_is_cuda = PyUnicode_InternFromString("is_cuda");
  s_is_contiguous = PyUnicode_InternFromString("is_contiguous");
  s_data_ptr = PyUnicode_InternFromString("data_ptr");
  s_numel = PyUnicode_InternFromString("numel");
  s_shape = PyUnicode_InternFromString("shape");
  if (!s_dtype || !s_is_cuda || !s_is_contiguous || !s_data_ptr || !s_numel || !s_shape) return NULL;
  return PyModule_Create(&module);
}

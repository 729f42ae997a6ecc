/* honeycrisp_amd._native: the calls that a program makes once per op, from Python to libhchip.so without ctypes.
 *
 * A method of Context takes the backend and an op's arguments, makes the result's block, makes the library call and returns the
 * result's Data. That is one crossing where ctypes made three (the block, the op, and the block of a result that was let go), and
 * argument conversion in C. Small ops are bound by this: x + y over 16 x 512 fp16 took the front-end 8.6 us before the library was
 * entered and takes 3.4; (x + y).normalize().mul(g + 1, thenAdd: b) over the same, four launches, 34.1 us end to end and now 23.2; a
 * training step of 75 calls 540 and now 478.
 *
 * The interpreter's lock is released around library calls, as ctypes does: a call may wait for the device, and that for a host
 * function in Python.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>
#include <stdint.h>
#include <string.h>

#include "../../include/hchip.h"

#define FUNCTIONS(X)                                                                                                                   \
  X(hc_malloc) X(hc_free) X(hc_binary_op) X(hc_binary_op_scalar) X(hc_mul_add) X(hc_add_mul) X(hc_when) X(hc_cast) X(hc_pow) X(hc_elemwise)  \
  X(hc_reduce) X(hc_cumulative) X(hc_argsort) X(hc_log_softmax) X(hc_log_softmax_grad) X(hc_normalize) X(hc_gather) X(hc_scatter)             \
  X(hc_adamw) X(hc_matmul) X(hc_fill) X(hc_broadcast)

typedef struct {
  PyObject_HEAD
  hc_ctx* ctx;          /* NULL once the backend is closed */
  PyTypeObject* data;   /* the class of results (HIPData) */
#define X(name) __typeof__(&name) name;
  FUNCTIONS(X)
#undef X
} Context;

/* A device buffer that is given back with its last reference. */
typedef struct {
  PyObject_HEAD
  PyObject* backend;
  Context* context;     /* the backend's; NULL: nothing to give back */
  void* ptr;
  Py_ssize_t bytes;
} Data;

static PyObject *s_native, *s_dev, *s_ptr, *s_raise, *s_shape, *s_strides, *s_value;
static PyTypeObject Context_Type, Data_Type;

/* ---------------------------------------------------------------- Data */

static void data_give_back(Data* self) {
  void* ptr = self->ptr;
  Context* c = self->context;
  self->ptr = NULL;
  if (ptr && c && c->ctx) {
    hc_ctx* ctx = c->ctx;
    Py_BEGIN_ALLOW_THREADS
    c->hc_free(ctx, ptr);
    Py_END_ALLOW_THREADS
  }
}

static int data_traverse(Data* self, visitproc visit, void* arg) {
  Py_VISIT(self->backend);
  Py_VISIT(self->context);
  return 0;
}

static int data_clear(Data* self) {   /* (the buffer goes before what it goes through) */
  data_give_back(self);
  Py_CLEAR(self->backend);
  Py_CLEAR(self->context);
  return 0;
}

static void data_dealloc(Data* self) {
  PyObject_GC_UnTrack(self);
  PyObject *type, *value, *traceback;
  PyErr_Fetch(&type, &value, &traceback);
  data_clear(self);
  PyErr_Restore(type, value, traceback);
  Py_TYPE(self)->tp_free((PyObject*)self);
}

static int ptr_of(PyObject* o, void** out) {
  if (o == Py_None) return *out = NULL, 0;
  *out = PyLong_AsVoidPtr(o);
  return PyErr_Occurred() ? -1 : 0;
}

static int data_init(Data* self, PyObject* args, PyObject* kw) {
  static char* names[] = {"backend", "ptr", "byteCount", NULL};
  PyObject *backend, *ptr;
  Py_ssize_t bytes;
  void* p;
  if (!PyArg_ParseTupleAndKeywords(args, kw, "OOn", names, &backend, &ptr, &bytes) || ptr_of(ptr, &p)) return -1;
  PyObject* context = PyObject_GetAttr(backend, s_native);
  if (!context) PyErr_Clear();
  Py_INCREF(backend);
  Py_XSETREF(self->backend, backend);
  Py_XSETREF(self->context, context && Py_IS_TYPE(context, &Context_Type) ? (Context*)context : (Py_XDECREF(context), NULL));
  self->ptr = p;
  self->bytes = bytes;
  return 0;
}

static PyObject* data_get_ptr(Data* self, void* unused) {
  if (!self->ptr) Py_RETURN_NONE;
  return PyLong_FromVoidPtr(self->ptr);
}
static int data_set_ptr(Data* self, PyObject* value, void* unused) {
  if (!value) return PyErr_SetString(PyExc_AttributeError, "ptr"), -1;
  return ptr_of(value, &self->ptr);
}
static PyObject* data_get_backend(Data* self, void* unused) {
  PyObject* backend = self->backend ? self->backend : Py_None;
  Py_INCREF(backend);
  return backend;
}
static int data_set_backend(Data* self, PyObject* value, void* unused) {
  Py_XINCREF(value);
  Py_XSETREF(self->backend, value);
  return 0;
}
static PyObject* data_get_bytes(Data* self, void* unused) { return PyLong_FromSsize_t(self->bytes); }
static int data_set_bytes(Data* self, PyObject* value, void* unused) {
  const Py_ssize_t bytes = value ? PyLong_AsSsize_t(value) : -1;
  if (bytes == -1 && PyErr_Occurred()) return -1;
  self->bytes = bytes;
  return 0;
}
static PyGetSetDef data_getset[] = {{"ptr", (getter)data_get_ptr, (setter)data_set_ptr, NULL, NULL},
                                    {"backend", (getter)data_get_backend, (setter)data_set_backend, NULL, NULL},
                                    {"byteCount", (getter)data_get_bytes, (setter)data_set_bytes, NULL, NULL},
                                    {NULL, NULL, NULL, NULL, NULL}};

static PyTypeObject Data_Type = {
    PyVarObject_HEAD_INIT(NULL, 0).tp_name = "honeycrisp_amd._native.Data",
    .tp_basicsize = sizeof(Data),
    .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC,
    .tp_new = PyType_GenericNew,
    .tp_init = (initproc)data_init,
    .tp_dealloc = (destructor)data_dealloc,
    .tp_traverse = (traverseproc)data_traverse,
    .tp_clear = (inquiry)data_clear,
    .tp_getset = data_getset,
};

/* ---------------------------------------------------------------- an op's arguments and its result */

typedef struct {
  Context* c;
  PyObject* backend;
  PyObject* kept[6];    /* foreign operands as they were uploaded */
  int n_kept;
  int failed;           /* an exception is set */
} Call;

static Call begin(Context* c, PyObject* const* a, Py_ssize_t n, Py_ssize_t want) {
  Call call = {.c = c, .backend = n > 0 ? a[0] : NULL};
  if (n != want) {
    PyErr_Format(PyExc_TypeError, "%zd arguments instead of %zd", n, want);
    call.failed = 1;
  }
  return call;
}

static int64_t whole(Call* call, PyObject* o) {
  if (call->failed) return 0;
  PyObject* value = NULL;
  if (!PyLong_Check(o) && !PyIndex_Check(o)) {   /* a ctypes integer */
    value = o = PyObject_GetAttr(o, s_value);
    if (!value) return PyErr_SetString(PyExc_TypeError, "an integer is wanted"), call->failed = 1, 0;
  }
  const int64_t v = PyLong_AsLongLong(o);
  Py_XDECREF(value);
  if (v == -1 && PyErr_Occurred()) call->failed = 1;
  return v;
}

static float real(Call* call, PyObject* o) {
  if (call->failed) return 0;
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) call->failed = 1;
  return (float)v;
}

/* the address of an operand on the device; anything but a plain buffer of this backend goes through the backend's _dev */
static void* operand(Call* call, PyObject* o) {
  if (call->failed) return NULL;
  if (Py_IS_TYPE(o, call->c->data) && ((Data*)o)->backend == call->backend) return ((Data*)o)->ptr;
  PyObject* dev = PyObject_CallMethodOneArg(call->backend, s_dev, o);
  PyObject* value = dev ? PyObject_GetAttr(dev, s_ptr) : NULL;
  void* p = NULL;
  if (!value || ptr_of(value, &p)) call->failed = 1;
  Py_XDECREF(value);
  if (dev) call->kept[call->n_kept++] = dev;
  return p;
}
static void* operand_or_null(Call* call, PyObject* o) { return o == Py_None ? NULL : operand(call, o); }

static int64_t times(Call* call, int64_t a, int64_t b) {
  int64_t v = 0;
  if (!call->failed && __builtin_mul_overflow(a, b, &v)) v = INT64_MAX;   /* (more than there is: hc_malloc says so) */
  return v;
}

/* BroadcastStrides -> its descriptor; the number of elements of the virtual shape */
static int64_t strides(Call* call, PyObject* o, hc_strides* out) {
  if (call->failed) return 0;
  int64_t count = 1;
  PyObject *shape = PyObject_GetAttr(o, s_shape), *steps = shape ? PyObject_GetAttr(o, s_strides) : NULL;
  PyObject *f = steps ? PySequence_Fast(shape, "a shape is a sequence") : NULL, *g = f ? PySequence_Fast(steps, "strides are a sequence") : NULL;
  if (!g) {
    call->failed = 1;
  } else if (PySequence_Fast_GET_SIZE(f) > HC_MAX_DIMS) {
    PyErr_Format(PyExc_ValueError, "at most %d axes are supported, got shape %S", HC_MAX_DIMS, shape);
    call->failed = 1;
  } else if (PySequence_Fast_GET_SIZE(f) != PySequence_Fast_GET_SIZE(g)) {
    PyErr_SetString(PyExc_ValueError, "shape and strides differ in length");
    call->failed = 1;
  } else {
    memset(out, 0, sizeof(*out));
    out->ndim = (uint32_t)PySequence_Fast_GET_SIZE(f);
    for (uint32_t i = 0; i < out->ndim && !call->failed; i++) {
      out->shape[i] = whole(call, PySequence_Fast_GET_ITEM(f, i));
      out->strides[i] = whole(call, PySequence_Fast_GET_ITEM(g, i));
      count = times(call, count, out->shape[i]);
    }
  }
  Py_XDECREF(g);
  Py_XDECREF(f);
  Py_XDECREF(steps);
  Py_XDECREF(shape);
  return count;
}

static int64_t bytes_of(Call* call, int64_t count, int64_t dtype) {
  static const int64_t size[] = {8, 1, 2, 4};   /* HC_I64, HC_BOOL, HC_F16, HC_F32 */
  if (!call->failed && (dtype < 0 || dtype > 3)) {
    PyErr_Format(PyExc_ValueError, "no data type %lld", (long long)dtype);
    call->failed = 1;
  }
  return call->failed ? 0 : times(call, count, size[dtype]);
}

static PyObject* new_data(Call* call, void* ptr, int64_t bytes) {
  Data* d = (Data*)call->c->data->tp_alloc(call->c->data, 0);
  if (!d) return NULL;
  Py_INCREF(call->backend);
  Py_INCREF(call->c);
  d->backend = call->backend;
  d->context = call->c;
  d->ptr = ptr;
  d->bytes = (Py_ssize_t)bytes;
  return (PyObject*)d;
}

static PyObject* raise_status(Call* call, int status) {
  PyObject* r = PyObject_CallMethod(call->backend, "_raise", "i", status);
  if (r) {
    Py_DECREF(r);
    PyErr_Format(PyExc_RuntimeError, "status %d", status);
  }
  return NULL;
}

static PyObject* end(Call* call, PyObject* result) {
  for (int i = 0; i < call->n_kept; i++) Py_DECREF(call->kept[i]);
  return result;
}

/* n buffers of `bytes` into out[], then `expr`; the results, or the backend's exception (also once it is closed: hc_malloc refuses a null context) */
#define RUN(n, bytes, expr)                                                            \
  hc_ctx* const ctx = c->ctx;                                                          \
  void* out[n] = {NULL};                                                               \
  int made = 0, status = HC_OK;                                                        \
  PyObject* result = NULL;                                                             \
  if (!call.failed) {                                                                  \
    const size_t size = (bytes) > 0 ? (size_t)(bytes) : 0;                             \
    Py_BEGIN_ALLOW_THREADS                                                             \
    for (; made < n && status == HC_OK; made++) status = c->hc_malloc(ctx, size, &out[made]); \
    if (status == HC_OK) status = (expr);                                              \
    Py_END_ALLOW_THREADS                                                               \
    if (status != HC_OK) raise_status(&call, status);                                  \
    else result = n == 1 ? new_data(&call, out[0], bytes) : PyTuple_New(n);            \
    for (int i = 0; i < n && n > 1 && result; i++) {                                   \
      PyObject* d = new_data(&call, out[i], bytes);                                    \
      if (d) PyTuple_SET_ITEM(result, i, d), out[i] = NULL;                            \
      else Py_CLEAR(result);                                                           \
    }                                                                                  \
    if (!result) {                                                                     \
      PyObject *type, *value, *traceback;                                              \
      PyErr_Fetch(&type, &value, &traceback);                                          \
      Py_BEGIN_ALLOW_THREADS                                                           \
      for (int i = 0; i < n; i++)                                                      \
        if (out[i]) c->hc_free(ctx, out[i]);                                           \
      Py_END_ALLOW_THREADS                                                             \
      PyErr_Restore(type, value, traceback);                                           \
    }                                                                                  \
  }                                                                                    \
  return end(&call, result)

/* ---------------------------------------------------------------- the ops; a[0] is the backend */
#define OP(name, want) \
  static PyObject* name(Context* c, PyObject* const* a, Py_ssize_t n) { \
    Call call = begin(c, a, n, want);                                   \
    if (call.failed) return NULL;

OP(op_alloc, 2)
  const int64_t bytes = whole(&call, a[1]);
  RUN(1, bytes, HC_OK);
}

OP(op_binary, 7)   /* op, dtype, data, strides, data, strides */
  hc_strides sx, sy;
  const int op = (int)whole(&call, a[1]), dtype = (int)whole(&call, a[2]);
  const void *x = operand(&call, a[3]), *y = operand(&call, a[5]);
  const int64_t bytes = bytes_of(&call, strides(&call, a[4], &sx), dtype);
  strides(&call, a[6], &sy);
  RUN(1, bytes, c->hc_binary_op(ctx, op, dtype, x, &sx, y, &sy, out[0]));
}

OP(op_binary_scalar, 8)   /* op, dtype, data, float, int, scalar first, count */
  const int op = (int)whole(&call, a[1]), dtype = (int)whole(&call, a[2]), first = (int)whole(&call, a[6]);
  const void* x = operand(&call, a[3]);
  const float f = real(&call, a[4]);
  const int64_t i = whole(&call, a[5]), count = whole(&call, a[7]), bytes = bytes_of(&call, count, dtype);
  RUN(1, bytes, c->hc_binary_op_scalar(ctx, op, dtype, x, f, i, first, out[0], (size_t)count));
}

#define THREE(name)   /* dtype, three times data, strides */                                     \
  OP(op_##name, 8)                                                                              \
    hc_strides sx, sy, sz;                                                                      \
    const int dtype = (int)whole(&call, a[1]);                                                  \
    const void *x = operand(&call, a[2]), *y = operand(&call, a[4]), *z = operand(&call, a[6]); \
    const int64_t bytes = bytes_of(&call, strides(&call, a[3], &sx), dtype);                    \
    strides(&call, a[5], &sy);                                                                  \
    strides(&call, a[7], &sz);                                                                  \
    RUN(1, bytes, c->hc_##name(ctx, dtype, x, &sx, y, &sy, z, &sz, out[0]));                    \
  }
THREE(mul_add)
THREE(add_mul)
THREE(when)

OP(op_broadcast, 4)   /* dtype, data, strides */
  hc_strides sx;
  const int dtype = (int)whole(&call, a[1]);
  const void* x = operand(&call, a[2]);
  const int64_t bytes = bytes_of(&call, strides(&call, a[3], &sx), dtype);
  RUN(1, bytes, c->hc_broadcast(ctx, dtype, x, &sx, out[0]));
}

OP(op_fill, 5)   /* dtype, float, int, count */
  const int dtype = (int)whole(&call, a[1]);
  const float f = real(&call, a[2]);
  const int64_t i = whole(&call, a[3]), count = whole(&call, a[4]), bytes = bytes_of(&call, count, dtype);
  RUN(1, bytes, c->hc_fill(ctx, dtype, f, i, out[0], (size_t)count));
}

OP(op_cast, 5)   /* data, count, from, to */
  const void* x = operand(&call, a[1]);
  const int64_t count = whole(&call, a[2]);
  const int from = (int)whole(&call, a[3]), to = (int)whole(&call, a[4]);
  const int64_t bytes = bytes_of(&call, count, to);
  RUN(1, bytes, c->hc_cast(ctx, x, from, out[0], to, (size_t)count));
}

OP(op_pow, 9)   /* dtype, data, exponent: float, scale: float, exponent: int, scale: int, scales, count */
  const int dtype = (int)whole(&call, a[1]);
  const void *x = operand(&call, a[2]), *scales = operand_or_null(&call, a[7]);
  const float bf = real(&call, a[3]), sf = real(&call, a[4]);
  const int64_t bi = whole(&call, a[5]), si = whole(&call, a[6]), count = whole(&call, a[8]), bytes = bytes_of(&call, count, dtype);
  RUN(1, bytes, c->hc_pow(ctx, dtype, x, bf, sf, bi, si, scales, out[0], (size_t)count));
}

OP(op_elemwise, 6)   /* op, dtype, data, scales, count */
  const int op = (int)whole(&call, a[1]), dtype = (int)whole(&call, a[2]);
  const void *x = operand(&call, a[3]), *scales = operand_or_null(&call, a[4]);
  const int64_t count = whole(&call, a[5]), bytes = bytes_of(&call, count, dtype);
  RUN(1, bytes, c->hc_elemwise(ctx, op, dtype, x, scales, out[0], (size_t)count));
}

/* (outer, reduce, inner) at a[at] and after */
#define DIMS(at) \
  const int64_t outer = whole(&call, a[at]), reduce = whole(&call, a[at + 1]), inner = whole(&call, a[at + 2]), total = times(&call, times(&call, outer, reduce), inner)

OP(op_reduce, 8)   /* op, dtype, result's dtype, data, dims */
  const int op = (int)whole(&call, a[1]), dtype = (int)whole(&call, a[2]), to = (int)whole(&call, a[3]);
  const void* x = operand(&call, a[4]);
  const int64_t outer = whole(&call, a[5]), reduce = whole(&call, a[6]), inner = whole(&call, a[7]), bytes = bytes_of(&call, times(&call, outer, inner), to);
  RUN(1, bytes, c->hc_reduce(ctx, op, dtype, x, out[0], outer, reduce, inner));
}

OP(op_cumulative, 9)   /* op, dtype, data, dims, exclusive, reverse */
  const int op = (int)whole(&call, a[1]), dtype = (int)whole(&call, a[2]), exclusive = (int)whole(&call, a[7]), reverse = (int)whole(&call, a[8]);
  const void* x = operand(&call, a[3]);
  DIMS(4);
  const int64_t bytes = bytes_of(&call, total, dtype);
  RUN(1, bytes, c->hc_cumulative(ctx, op, dtype, x, out[0], outer, reduce, inner, exclusive, reverse));
}

OP(op_argsort, 7)   /* dtype, data, dims, descending */
  const int dtype = (int)whole(&call, a[1]), descending = (int)whole(&call, a[6]);
  const void* x = operand(&call, a[2]);
  DIMS(3);
  const int64_t bytes = times(&call, total, 8);
  RUN(1, bytes, c->hc_argsort(ctx, dtype, x, out[0], outer, reduce, inner, descending));
}

OP(op_log_softmax, 6)   /* dtype, data, dims */
  const int dtype = (int)whole(&call, a[1]);
  const void* x = operand(&call, a[2]);
  DIMS(3);
  const int64_t bytes = bytes_of(&call, total, dtype);
  RUN(1, bytes, c->hc_log_softmax(ctx, dtype, x, out[0], outer, reduce, inner));
}

OP(op_log_softmax_grad, 7)   /* dtype, data, gradient, dims */
  const int dtype = (int)whole(&call, a[1]);
  const void *x = operand(&call, a[2]), *g = operand(&call, a[3]);
  DIMS(4);
  const int64_t bytes = bytes_of(&call, total, dtype);
  RUN(1, bytes, c->hc_log_softmax_grad(ctx, dtype, x, g, out[0], outer, reduce, inner));
}

OP(op_normalize, 7)   /* dtype, data, dims, eps */
  const int dtype = (int)whole(&call, a[1]);
  const void* x = operand(&call, a[2]);
  DIMS(3);
  const float eps = real(&call, a[6]);
  const int64_t bytes = bytes_of(&call, total, dtype);
  RUN(1, bytes, c->hc_normalize(ctx, dtype, x, out[0], outer, reduce, inner, eps));
}

OP(op_gather, 9)   /* dtype, data, indices, their strides, outer, middle, out count, inner */
  hc_strides si;
  const int dtype = (int)whole(&call, a[1]);
  const void *x = operand(&call, a[2]), *indices = operand(&call, a[3]);
  const int64_t bytes = bytes_of(&call, strides(&call, a[4], &si), dtype);
  const int64_t outer = whole(&call, a[5]), middle = whole(&call, a[6]), count = whole(&call, a[7]), inner = whole(&call, a[8]);
  RUN(1, bytes, c->hc_gather(ctx, dtype, x, indices, &si, out[0], outer, middle, count, inner));
}

OP(op_scatter, 10)   /* dtype, data, indices, their strides, outer, middle, out count, inner, unique */
  hc_strides si;
  const int dtype = (int)whole(&call, a[1]);
  const void *x = operand(&call, a[2]), *indices = operand(&call, a[3]);
  strides(&call, a[4], &si);
  const int64_t outer = whole(&call, a[5]), middle = whole(&call, a[6]), count = whole(&call, a[7]), inner = whole(&call, a[8]);
  const int unique = (int)whole(&call, a[9]);
  const int64_t bytes = bytes_of(&call, times(&call, times(&call, outer, middle), inner), dtype);
  RUN(1, bytes, c->hc_scatter(ctx, dtype, x, indices, &si, out[0], outer, middle, count, inner, unique));
}

OP(op_adamw, 13)   /* dtype, parameter, gradient, two moments, six numbers, count */
  const int dtype = (int)whole(&call, a[1]);
  const void *p = operand(&call, a[2]), *g = operand(&call, a[3]), *m = operand(&call, a[4]), *v = operand(&call, a[5]);
  const float beta1 = real(&call, a[6]), beta2 = real(&call, a[7]), eps = real(&call, a[8]), decay = real(&call, a[9]), lr = real(&call, a[10]), step = real(&call, a[11]);
  const int64_t count = whole(&call, a[12]), bytes = bytes_of(&call, count, dtype);
  RUN(3, bytes, c->hc_adamw(ctx, dtype, p, g, m, v, beta1, beta2, eps, decay, lr, step, (size_t)count, out[0], out[1], out[2]));
}

OP(op_matmul, 11)   /* dtype, batch, data, transposed, data, transposed, result transposed, rows, inner, columns */
  const int dtype = (int)whole(&call, a[1]), ta = (int)whole(&call, a[4]), tb = (int)whole(&call, a[6]), to = (int)whole(&call, a[7]);
  const int64_t batch = whole(&call, a[2]), rows = whole(&call, a[8]), inner = whole(&call, a[9]), cols = whole(&call, a[10]);
  const void *x = operand(&call, a[3]), *y = operand(&call, a[5]);
  const int64_t bytes = bytes_of(&call, times(&call, times(&call, batch, rows), cols), dtype);
  RUN(1, bytes, c->hc_matmul(ctx, dtype, batch, x, ta, y, tb, to, rows, inner, cols, out[0]));
}

/* ---------------------------------------------------------------- Context */

static int context_init(Context* self, PyObject* args, PyObject* kw) {
  const char* path;
  PyObject *ctx, *data;
  if (!PyArg_ParseTuple(args, "sOO!", &path, &ctx, &PyType_Type, &data)) return -1;
  if (!PyType_IsSubtype((PyTypeObject*)data, &Data_Type)) return PyErr_SetString(PyExc_TypeError, "not a class of Data"), -1;
  void* p;
  if (ptr_of(ctx, &p)) return -1;
  void* lib = dlopen(path, RTLD_NOW | RTLD_NOLOAD);   /* (the caller has loaded it, and keeps it) */
  if (!lib) return PyErr_Format(PyExc_ImportError, "%s is not loaded", path), -1;
  dlclose(lib);
#define X(name)                                                                                          \
  if (!(self->name = (__typeof__(&name))dlsym(lib, #name))) return PyErr_Format(PyExc_ImportError, "%s has no %s", path, #name), -1;
  FUNCTIONS(X)
#undef X
  Py_INCREF(data);
  Py_XSETREF(self->data, (PyTypeObject*)data);
  self->ctx = p;
  return 0;
}

static PyObject* context_close(Context* self, PyObject* unused) {
  self->ctx = NULL;
  Py_RETURN_NONE;
}

static int context_traverse(Context* self, visitproc visit, void* arg) {
  Py_VISIT(self->data);
  return 0;
}
static int context_clear(Context* self) {
  Py_CLEAR(self->data);
  return 0;
}
static void context_dealloc(Context* self) {
  PyObject_GC_UnTrack(self);
  context_clear(self);
  Py_TYPE(self)->tp_free((PyObject*)self);
}

#define M(name) {#name, (PyCFunction)(void (*)(void))op_##name, METH_FASTCALL, NULL}
static PyMethodDef context_methods[] = {
    M(alloc), M(binary), M(binary_scalar), M(mul_add), M(add_mul), M(when), M(broadcast), M(fill), M(cast), M(pow), M(elemwise), M(reduce), M(cumulative), M(argsort),
    M(log_softmax), M(log_softmax_grad), M(normalize), M(gather), M(scatter), M(adamw), M(matmul),
    {"close", (PyCFunction)context_close, METH_NOARGS, NULL}, {NULL, NULL, 0, NULL}};

static PyTypeObject Context_Type = {
    PyVarObject_HEAD_INIT(NULL, 0).tp_name = "honeycrisp_amd._native.Context",
    .tp_basicsize = sizeof(Context),
    .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC,
    .tp_new = PyType_GenericNew,
    .tp_init = (initproc)context_init,
    .tp_dealloc = (destructor)context_dealloc,
    .tp_traverse = (traverseproc)context_traverse,
    .tp_clear = (inquiry)context_clear,
    .tp_methods = context_methods,
};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, .m_name = "_native", .m_size = -1};

PyMODINIT_FUNC PyInit__native(void) {
  s_native = PyUnicode_InternFromString("_native");
  s_dev = PyUnicode_InternFromString("_dev");
  s_ptr = PyUnicode_InternFromString("ptr");
  s_raise = PyUnicode_InternFromString("_raise");
  s_shape = PyUnicode_InternFromString("shape");
  s_strides = PyUnicode_InternFromString("strides");
  s_value = PyUnicode_InternFromString("value");
  PyObject* m = PyModule_Create(&module);
  if (!m || PyModule_AddType(m, &Data_Type) || PyModule_AddType(m, &Context_Type)) return NULL;
  return m;
}

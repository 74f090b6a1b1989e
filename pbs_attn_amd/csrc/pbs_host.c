/* The call of a short prompt inside one segment, from tensors to launch: a CPython function around pbs_one_segment_attn_fwd.
 *
 * Such a call takes the GPU 4 to 10 us, and what Python took to read three tensors and hand over 28 arguments took longer: 32 / 8 heads x
 * 77 tokens 9.4 -> 6.6 us a call, of which the launch takes 3 and the allocation of the output 1.3.  Tensors are read through their Python attributes, the same ones in the same sense as
 * ops.prefill_attn_fwd reads them, so nothing here depends on torch's C++ interface.
 *
 * Whatever is not the plain case returns None with nothing done, and the general path in Python takes the call, or refuses it with its message. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <math.h>
#include <stdint.h>

typedef int (*one_segment_fn)(const void* q, const void* k, const void* v, void* out, int B, int Hq, int Hkv, int S, int head_dim,
                              int block_size, int segment_size, int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t k_sb, int64_t k_sh,
                              int64_t k_ss, int64_t v_sb, int64_t v_sh, int64_t v_ss, int64_t o_sb, int64_t o_sh, int64_t o_ss,
                              float softmax_scale, void* stream);

enum { BLOCK = 128, HEAD_DIM = 128, MAX_BLOCKS = 256, NOT_ONE_LAUNCH = -3 };

static one_segment_fn launch;
static PyObject *tensor_type, *bfloat16, *current_device, *current_stream, *check;
static PyObject *s_shape, *s_stride, *s_data_ptr, *s_is_cuda, *s_dtype, *s_new_empty;

/* n integers out of a tuple of that length: 0 if it is something else */
static int read_ints(PyObject* t, long long* x, Py_ssize_t n) {
  if (!t || !PyTuple_Check(t) || PyTuple_GET_SIZE(t) != n) return 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    x[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(t, i));
    if (x[i] == -1 && PyErr_Occurred()) return 0;
  }
  return 1;
}

static int read_address(PyObject* t, uint64_t* address) {
  PyObject* p = PyObject_CallMethodNoArgs(t, s_data_ptr);
  if (!p) return 0;
  *address = PyLong_AsUnsignedLongLong(p);
  Py_DECREF(p);
  return !PyErr_Occurred();
}

static int attr_is(PyObject* t, PyObject* name, PyObject* want) {
  PyObject* x = PyObject_GetAttr(t, name);
  const int same = x == want;
  Py_XDECREF(x);
  return same;
}

/* a bf16 tensor of (B, H, S, 128) on the GPU whose rows the kernels read where they are */
static int read_tensor(PyObject* t, long long shape[4], long long stride[4], uint64_t* address) {
  if ((PyObject*)Py_TYPE(t) != tensor_type || !attr_is(t, s_is_cuda, Py_True) || !attr_is(t, s_dtype, bfloat16)) return 0;
  PyObject* x = PyObject_GetAttr(t, s_shape);
  const int has_shape = read_ints(x, shape, 4);
  Py_XDECREF(x);
  if (!has_shape) return 0;
  x = PyObject_CallMethodNoArgs(t, s_stride);
  const int has_stride = read_ints(x, stride, 4);
  Py_XDECREF(x);
  return has_stride && read_address(t, address) && stride[3] == 1 && *address % 16 == 0 && stride[0] % 8 == 0 && stride[1] % 8 == 0 &&
         stride[2] % 8 == 0;
}

static int is_pool_mode(PyObject* mode) {
  return PyUnicode_Check(mode) && (!PyUnicode_CompareWithASCIIString(mode, "mean") || !PyUnicode_CompareWithASCIIString(mode, "max"));
}

static PyObject* not_taken(void) {
  if (PyErr_Occurred() && !PyErr_ExceptionMatches(PyExc_Exception)) return NULL;   /* an interrupt, an exit */
  PyErr_Clear();   /* the general path meets the same error again */
  Py_RETURN_NONE;
}

/* one_segment(q, k, v, block_size, segment_size, threshold, causal, use_triton, query_pool_mode, key_pool_mode) -> tensor or None */
static PyObject* one_segment(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  long long qs[4], ks[4], vs[4], qt[4], kt[4], vt[4];
  uint64_t q, k, v, o, stream;
  (void)self;
  if (n != 10) {
    PyErr_SetString(PyExc_TypeError, "one_segment takes ten arguments");
    return NULL;
  }
  if (!launch || !PyLong_CheckExact(args[3]) || !PyLong_CheckExact(args[4]) || !PyFloat_CheckExact(args[5]) || args[6] != Py_True ||
      args[7] != Py_True || !is_pool_mode(args[8]) || !is_pool_mode(args[9]))
    return not_taken();
  const long long block = PyLong_AsLongLong(args[3]), segment = PyLong_AsLongLong(args[4]);   /* (an overflow is -1) */
  if (block != BLOCK || segment <= 0 || segment % BLOCK || segment > INT32_MAX) return not_taken();
  if (!read_tensor(args[0], qs, qt, &q)) return not_taken();
  const long long B = qs[0], Hq = qs[1], S = qs[2];
  if (B <= 0 || Hq <= 0 || S <= 0 || S > segment || qs[3] != HEAD_DIM || B > MAX_BLOCKS || Hq > MAX_BLOCKS || S > MAX_BLOCKS * BLOCK ||
      B * Hq * ((S + BLOCK - 1) / BLOCK) > MAX_BLOCKS)
    return not_taken();
  if (!read_tensor(args[1], ks, kt, &k) || !read_tensor(args[2], vs, vt, &v)) return not_taken();
  const long long Hkv = ks[1];
  if (Hkv <= 0 || Hq % Hkv || ks[0] != B || ks[2] != S || ks[3] != HEAD_DIM || vs[0] != B || vs[1] != Hkv || vs[2] != S || vs[3] != HEAD_DIM)
    return not_taken();

  PyObject* device = PyObject_CallNoArgs(current_device);
  PyObject* raw = device ? PyObject_CallOneArg(current_stream, device) : NULL;
  Py_XDECREF(device);
  if (!raw) return not_taken();
  stream = PyLong_AsUnsignedLongLong(raw);
  Py_DECREF(raw);
  if (PyErr_Occurred()) return not_taken();
  PyObject* shape = PyObject_GetAttr(args[0], s_shape);
  PyObject* out = shape ? PyObject_CallMethodOneArg(args[0], s_new_empty, shape) : NULL;
  Py_XDECREF(shape);
  if (!out) return NULL;
  if (!read_address(out, &o)) {
    Py_DECREF(out);
    return NULL;
  }
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = launch((const void*)(uintptr_t)q, (const void*)(uintptr_t)k, (const void*)(uintptr_t)v, (void*)(uintptr_t)o, (int)B, (int)Hq, (int)Hkv, (int)S,
              HEAD_DIM, BLOCK, (int)segment, qt[0], qt[1], qt[2], kt[0], kt[1], kt[2], vt[0], vt[1], vt[2], Hq * S * HEAD_DIM, S * HEAD_DIM,
              HEAD_DIM, (float)(1.0 / sqrt((double)HEAD_DIM)), (void*)(uintptr_t)stream);
  Py_END_ALLOW_THREADS
  if (!rc) return out;
  Py_DECREF(out);
  if (rc == NOT_ONE_LAUNCH) Py_RETURN_NONE;
  return PyObject_CallFunction(check, "is", rc, "pbs_one_segment_attn_fwd");   /* raises */
}

/* setup(tensor type, torch.bfloat16, current device, its current raw stream, check, address of pbs_one_segment_attn_fwd), once */
static PyObject* setup(PyObject* self, PyObject* args) {
  PyObject *t, *dtype, *dev, *st, *ck;
  unsigned long long address;
  (void)self;
  if (!PyArg_ParseTuple(args, "OOOOOK", &t, &dtype, &dev, &st, &ck, &address)) return NULL;
  Py_INCREF(t), Py_INCREF(dtype), Py_INCREF(dev), Py_INCREF(st), Py_INCREF(ck);
  tensor_type = t, bfloat16 = dtype, current_device = dev, current_stream = st, check = ck;
  launch = (one_segment_fn)(uintptr_t)address;
  Py_RETURN_NONE;
}

static PyMethodDef methods[] = {{"one_segment", (PyCFunction)(void (*)(void))one_segment, METH_FASTCALL, NULL},
                                {"setup", setup, METH_VARARGS, NULL},
                                {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pbs_host", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__pbs_host(void) {
  s_shape = PyUnicode_InternFromString("shape");
  s_stride = PyUnicode_InternFromString("stride");
  s_data_ptr = PyUnicode_InternFromString("data_ptr");
  s_is_cuda = PyUnicode_InternFromString("is_cuda");
  s_dtype = PyUnicode_InternFromString("dtype");
  s_new_empty = PyUnicode_InternFromString("new_empty");
  if (!s_shape || !s_stride || !s_data_ptr || !s_is_cuda || !s_dtype || !s_new_empty) return NULL;
  return PyModule_Create(&module);
}

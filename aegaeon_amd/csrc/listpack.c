/* Host-side packing of the reference's per-step request lists into the flat
 * arrays aegkv_prepare_inputs uploads (the lists Worker._prepare_model_inputs
 * walks, aegaeon/aegaeon/worker.py:596-646: RequestMeta tuples
 * (request_id, tokens, seq_len, context_len), aegaeon/aegaeon/request.py:96-102,
 * and one block table per request).  Python's iteration over those lists
 * costs ~30 ns per element; reading them through the CPython API costs a few.
 *
 *   pack_tables(tables) -> (ids: bytearray of int32, offsets: bytearray of int64)
 *       request b's table is ids[offsets[b]:offsets[b + 1]]
 *   pack_requests(requests) -> (seq_lens: bytearray of int32,
 *                               context_lens: bytearray of int32,
 *                               tokens: bytearray of int64)
 *       the new tokens of every request, in order; a request whose token list
 *       does not hold seq_len - context_len tokens raises ValueError
 *
 * Both accept lists or tuples (any sequence) of Python ints and raise
 * TypeError / OverflowError for anything else.
 *
 *   step_counts(offsets, seq_lens, context_lens) ->
 *       (seq_lens as a list, new tokens, longest decode table, prefills,
 *        prefill tokens, longest new part, longest prefill, longest decode)
 *       of such buffers (requests of context 0 are prefills; a maximum over
 *       none is 0): the step's counts that the host keeps, in one pass
 *   address(buffer) -> its address as an int (None when empty); the caller
 *       keeps the buffer alive while it uses the address */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <stdint.h>
#include <string.h>

static int long_in_range(PyObject* o, long long lo, long long hi, long long* out) {
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) return -1;
  if (v < lo || v > hi) {
    PyErr_SetString(PyExc_OverflowError, "value out of range for its packed type");
    return -1;
  }
  *out = v;
  return 0;
}

static PyObject* pack_tables(PyObject* self, PyObject* arg) {
  (void)self;
  PyObject* outer = PySequence_Fast(arg, "block tables must be a sequence");
  if (!outer) return NULL;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(outer);
  PyObject** rows = PySequence_Fast_ITEMS(outer);
  PyObject* offsets = PyByteArray_FromStringAndSize(NULL, (n + 1) * (Py_ssize_t)sizeof(int64_t));
  PyObject* ids = NULL;
  PyObject** fast = NULL;
  if (!offsets) goto fail;
  fast = (PyObject**)PyMem_Calloc(n ? (size_t)n : 1, sizeof(PyObject*));
  if (!fast) {
    PyErr_NoMemory();
    goto fail;
  }
  int64_t* off = (int64_t*)PyByteArray_AS_STRING(offsets);
  off[0] = 0;
  for (Py_ssize_t b = 0; b < n; ++b) {
    fast[b] = PySequence_Fast(rows[b], "a block table must be a sequence");
    if (!fast[b]) goto fail;
    off[b + 1] = off[b] + PySequence_Fast_GET_SIZE(fast[b]);
  }
  ids = PyByteArray_FromStringAndSize(NULL, (Py_ssize_t)(off[n] * (int64_t)sizeof(int32_t)));
  if (!ids) goto fail;
  int32_t* dst = (int32_t*)PyByteArray_AS_STRING(ids);
  for (Py_ssize_t b = 0; b < n; ++b) {
    const Py_ssize_t m = PySequence_Fast_GET_SIZE(fast[b]);
    PyObject** items = PySequence_Fast_ITEMS(fast[b]);
    for (Py_ssize_t i = 0; i < m; ++i) {
      long long v;
      if (long_in_range(items[i], INT32_MIN, INT32_MAX, &v)) goto fail;
      *dst++ = (int32_t)v;
    }
  }
  for (Py_ssize_t b = 0; b < n; ++b) Py_DECREF(fast[b]);
  PyMem_Free(fast);
  Py_DECREF(outer);
  return Py_BuildValue("(NN)", ids, offsets);
fail:
  if (fast) {
    for (Py_ssize_t b = 0; b < n; ++b) Py_XDECREF(fast[b]);
    PyMem_Free(fast);
  }
  Py_XDECREF(ids);
  Py_XDECREF(offsets);
  Py_DECREF(outer);
  return NULL;
}

static PyObject* pack_requests(PyObject* self, PyObject* arg) {
  (void)self;
  PyObject* outer = PySequence_Fast(arg, "requests must be a sequence");
  if (!outer) return NULL;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(outer);
  PyObject** reqs = PySequence_Fast_ITEMS(outer);
  PyObject* seq = PyByteArray_FromStringAndSize(NULL, n * (Py_ssize_t)sizeof(int32_t));
  PyObject* ctx = PyByteArray_FromStringAndSize(NULL, n * (Py_ssize_t)sizeof(int32_t));
  PyObject* toks = NULL;
  PyObject** fast = NULL;
  if (!seq || !ctx) goto fail;
  fast = (PyObject**)PyMem_Calloc(n ? (size_t)n : 1, sizeof(PyObject*));
  if (!fast) {
    PyErr_NoMemory();
    goto fail;
  }
  int32_t* s = (int32_t*)PyByteArray_AS_STRING(seq);
  int32_t* c = (int32_t*)PyByteArray_AS_STRING(ctx);
  Py_ssize_t total = 0;
  for (Py_ssize_t b = 0; b < n; ++b) {
    PyObject* r = reqs[b];
    if (!PySequence_Check(r) || PySequence_Size(r) < 4) {
      PyErr_SetString(PyExc_TypeError,
                      "a request must be (request_id, tokens, seq_len, context_len)");
      goto fail;
    }
    PyObject* t = PySequence_GetItem(r, 1);
    PyObject* sl = PySequence_GetItem(r, 2);
    PyObject* cl = PySequence_GetItem(r, 3);
    long long sv = 0, cv = 0;
    const int bad = !t || !sl || !cl || long_in_range(sl, INT32_MIN, INT32_MAX, &sv) ||
                    long_in_range(cl, INT32_MIN, INT32_MAX, &cv);
    Py_XDECREF(sl);
    Py_XDECREF(cl);
    if (bad) {
      Py_XDECREF(t);
      goto fail;
    }
    fast[b] = PySequence_Fast(t, "a request's tokens must be a sequence");
    Py_DECREF(t);
    if (!fast[b]) goto fail;
    s[b] = (int32_t)sv;
    c[b] = (int32_t)cv;
    if ((long long)PySequence_Fast_GET_SIZE(fast[b]) != sv - cv) {
      PyErr_SetString(PyExc_ValueError,
                      "a request's tokens must be its seq_len - context_len new tokens");
      goto fail;
    }
    total += PySequence_Fast_GET_SIZE(fast[b]);
  }
  toks = PyByteArray_FromStringAndSize(NULL, total * (Py_ssize_t)sizeof(int64_t));
  if (!toks) goto fail;
  int64_t* dst = (int64_t*)PyByteArray_AS_STRING(toks);
  for (Py_ssize_t b = 0; b < n; ++b) {
    const Py_ssize_t m = PySequence_Fast_GET_SIZE(fast[b]);
    PyObject** items = PySequence_Fast_ITEMS(fast[b]);
    for (Py_ssize_t i = 0; i < m; ++i) {
      long long v;
      if (long_in_range(items[i], INT64_MIN, INT64_MAX, &v)) goto fail;
      *dst++ = (int64_t)v;
    }
  }
  for (Py_ssize_t b = 0; b < n; ++b) Py_DECREF(fast[b]);
  PyMem_Free(fast);
  Py_DECREF(outer);
  return Py_BuildValue("(NNN)", seq, ctx, toks);
fail:
  if (fast) {
    for (Py_ssize_t b = 0; b < n; ++b) Py_XDECREF(fast[b]);
    PyMem_Free(fast);
  }
  Py_XDECREF(seq);
  Py_XDECREF(ctx);
  Py_XDECREF(toks);
  Py_DECREF(outer);
  return NULL;
}

static PyObject* step_counts(PyObject* self, PyObject* args) {
  (void)self;
  Py_buffer off, seq, ctx;
  if (!PyArg_ParseTuple(args, "y*y*y*", &off, &seq, &ctx)) return NULL;
  PyObject* list = NULL;
  PyObject* out = NULL;
  const Py_ssize_t n = seq.len / (Py_ssize_t)sizeof(int32_t);
  if (n == 0 || ctx.len != seq.len || off.len != (n + 1) * (Py_ssize_t)sizeof(int64_t)) {
    PyErr_SetString(PyExc_ValueError, "one context length and one table per request");
    goto done;
  }
  list = PyList_New(n);
  if (!list) goto done;
  const int64_t* o = (const int64_t*)off.buf;
  const int32_t* s = (const int32_t*)seq.buf;
  const int32_t* c = (const int32_t*)ctx.buf;
  /* unsigned sums: any lengths, also ones the call then refuses */
  uint64_t total = 0, prompt_total = 0;
  int64_t prompts = 0, longest_new = INT64_MIN;
  int64_t width = INT64_MIN, longest_prompt = INT64_MIN, longest_decode = INT64_MIN;
  for (Py_ssize_t b = 0; b < n; ++b) {
    const int64_t fresh = (int64_t)s[b] - c[b];
    PyObject* v = PyLong_FromLong(s[b]);
    if (!v) goto done;
    PyList_SET_ITEM(list, b, v);
    total += (uint64_t)fresh;
    if (fresh > longest_new) longest_new = fresh;
    if (c[b] == 0) {
      ++prompts;
      prompt_total += (uint64_t)fresh;
      if (s[b] > longest_prompt) longest_prompt = s[b];
    } else {
      const int64_t w = (int64_t)((uint64_t)o[b + 1] - (uint64_t)o[b]);
      if (w > width) width = w;
      if (s[b] > longest_decode) longest_decode = s[b];
    }
  }
  if (prompts == n) width = longest_decode = 0;
  if (prompts == 0) longest_prompt = 0;
  out = Py_BuildValue("(OLLLLLLL)", list, (long long)total, (long long)width, (long long)prompts,
                      (long long)prompt_total, (long long)longest_new, (long long)longest_prompt,
                      (long long)longest_decode);
done:
  Py_XDECREF(list);
  PyBuffer_Release(&off);
  PyBuffer_Release(&seq);
  PyBuffer_Release(&ctx);
  return out;
}

static PyObject* address(PyObject* self, PyObject* arg) {
  (void)self;
  Py_buffer b;
  if (PyObject_GetBuffer(arg, &b, PyBUF_SIMPLE)) return NULL;
  PyObject* out;
  if (b.len == 0) {
    out = Py_None;
    Py_INCREF(out);
  } else {
    out = PyLong_FromVoidPtr(b.buf);
  }
  PyBuffer_Release(&b);
  return out;
}

static PyMethodDef methods[] = {
    {"pack_tables", pack_tables, METH_O,
     "pack_tables(tables) -> (int32 ids bytearray, int64 offsets bytearray)"},
    {"pack_requests", pack_requests, METH_O,
     "pack_requests(requests) -> (int32 seq_lens, int32 context_lens, int64 tokens) bytearrays"},
    {"step_counts", step_counts, METH_VARARGS,
     "step_counts(offsets, seq_lens, context_lens) -> (list, seven counts)"},
    {"address", address, METH_O, "address(buffer) -> int, None when it is empty"},
    {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_listpack",
                                    "Packing of the per-step request lists", -1, methods,
                                    NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__listpack(void) { return PyModule_Create(&module); }

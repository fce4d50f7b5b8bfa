// Host-side work on Python token lists, as a CPython extension module (mvsd._hostops): what the
// penalties need to know of each request's history, gathered without converting every list to an
// array first.  32 requests of 650 tokens: 4.0 ms with numpy (np.unique per request), 0.17 here.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

static uint64_t mix(uint64_t x) {
  x ^= x >> 31;
  x *= 0x9e3779b97f4a7c15ull;
  return x ^ (x >> 29);
}

// The place of token t among this request's entries [0, *n), added when it is new: an
// open-addressing table of mask + 1 slots (a power of two) that hold a place + 1, or 0.
static int32_t place_of(int32_t* slots, size_t mask, int64_t* keys, int32_t* n, int64_t t) {
  size_t i = (size_t)mix((uint64_t)t) & mask;
  while (slots[i]) {
    const int32_t at = slots[i] - 1;
    if (keys[at] == t) return at;
    i = (i + 1) & mask;
  }
  keys[*n] = t;
  slots[i] = *n + 1;
  return (*n)++;
}

// Adds the first `len` tokens of a fast sequence to the request's entries: of its prompt (kind 0),
// output (1) or drafts (2).  0 where a token is no integer (the exception is set).
static int add_tokens(PyObject* seq, Py_ssize_t len, int kind, int32_t* slots, size_t mask,
                      int64_t* keys, int32_t* info, int32_t* n) {
  // a list can change while __index__ of an element runs: look at it afresh each time
  for (Py_ssize_t i = 0; i < len && i < PySequence_Fast_GET_SIZE(seq); ++i) {
    PyObject* item = PySequence_Fast_GET_ITEM(seq, i);
    int64_t t;
    if (PyLong_CheckExact(item)) {
      t = PyLong_AsLongLong(item);
    } else {
      Py_INCREF(item);
      PyObject* whole = PyNumber_Index(item);
      t = whole ? PyLong_AsLongLong(whole) : -1;
      Py_XDECREF(whole);
      Py_DECREF(item);
    }
    if (t == -1 && PyErr_Occurred()) return 0;
    const int32_t before = *n;
    const int32_t at = place_of(slots, mask, keys, n, t);
    if (at == before) info[at] = 0;
    if (kind == 0) info[at] |= (int32_t)0x80000000u;
    if (kind == 1) ++info[at];
  }
  return 1;
}

// penalty_entries(prompts, outputs, specs, buffer) -> number of entries E
//
// prompts, outputs: sequences of token sequences (missing tail requests count as empty); specs: one
// token sequence per request.  For request r the distinct tokens of its prompt, output and drafts
// are entries [off[r], off[r + 1]); buffer (writable int32) receives off [B + 1], then the tokens
// [E], then, per entry, the token's count in the output | (in the prompt) << 31.  The buffer has
// room for B + 1 + 2 * (all tokens).  TypeError where a token is no integer.
static PyObject* penalty_entries(PyObject* self, PyObject* args) {
  PyObject* lists[3];
  Py_buffer buf;
  if (!PyArg_ParseTuple(args, "OOOw*", &lists[0], &lists[1], &lists[2], &buf)) return NULL;
  PyObject* outer[3] = {NULL, NULL, NULL};
  PyObject* result = NULL;
  int64_t* keys = NULL;
  int32_t* info = NULL;
  int32_t* slots = NULL;
  size_t slots_room = 0, keys_cap = 0;
  for (int s = 0; s < 3; ++s) {
    outer[s] = PySequence_Fast(lists[s], "a sequence of token sequences is expected");
    if (!outer[s]) goto out;
  }
  {
    const Py_ssize_t B = PySequence_Fast_GET_SIZE(outer[2]);
    const int64_t room = (int64_t)(buf.len / 4);
    int32_t* off = (int32_t*)buf.buf;
    int32_t* tok = off + B + 1;  // tokens, then (moved behind them at the end) the infos
    int64_t total = 0;           // entries so far
    if (room < B + 1) {
      PyErr_SetString(PyExc_ValueError, "buffer too small");
      goto out;
    }
    // infos are collected here, since their place follows the last token
    size_t info_cap = (size_t)((room - B - 1) / 2);
    info = (int32_t*)malloc((info_cap ? info_cap : 1) * sizeof(int32_t));
    if (!info) {
      PyErr_NoMemory();
      goto out;
    }
    off[0] = 0;
    for (Py_ssize_t r = 0; r < B; ++r) {
      PyObject* inner[3] = {NULL, NULL, NULL};
      Py_ssize_t len[3] = {0, 0, 0};
      size_t all = 0;
      int ok = 1;
      for (int s = 0; s < 3 && ok; ++s) {
        if (r >= PySequence_Fast_GET_SIZE(outer[s])) continue;
        inner[s] = PySequence_Fast(PySequence_Fast_GET_ITEM(outer[s], r),
                                   "a token sequence is expected");
        if (!inner[s]) ok = 0;
        else all += (size_t)(len[s] = PySequence_Fast_GET_SIZE(inner[s]));
      }
      if (ok && (total + (int64_t)all) > (int64_t)info_cap) {
        PyErr_SetString(PyExc_ValueError, "buffer too small");
        ok = 0;
      }
      // The table has this request's own size, so that a short history after a long one clears a
      // small one; at most a quarter full (half full: 0.20 ms instead of 0.17 for 32 requests).
      size_t cap = 16;
      while (cap < 4 * all) cap *= 2;
      if (ok && cap > slots_room) {
        free(slots);
        slots = (int32_t*)malloc(cap * sizeof(int32_t));
        slots_room = slots ? cap : 0;
      }
      if (ok && all > keys_cap) {
        free(keys);
        keys_cap = all;
        keys = (int64_t*)malloc(keys_cap * sizeof(int64_t));
      }
      if (ok && (!slots || (all && !keys))) {
        PyErr_NoMemory();
        ok = 0;
      }
      if (ok) {
        memset(slots, 0, cap * sizeof(int32_t));
        int32_t n = 0;
        for (int s = 0; s < 3 && ok; ++s)
          ok = !inner[s] || add_tokens(inner[s], len[s], s, slots, cap - 1, keys, info + total, &n);
        for (int32_t e = 0; ok && e < n; ++e) tok[total + e] = (int32_t)keys[e];
        total += ok ? n : 0;
        off[r + 1] = (int32_t)total;
      }
      for (int s = 0; s < 3; ++s) Py_XDECREF(inner[s]);
      if (!ok) goto out;
    }
    memcpy(tok + total, info, (size_t)total * sizeof(int32_t));
    result = PyLong_FromLongLong(total);
  }
out:
  for (int s = 0; s < 3; ++s) Py_XDECREF(outer[s]);
  free(slots);
  free(keys);
  free(info);
  PyBuffer_Release(&buf);
  return result;
}

static PyMethodDef methods[] = {
    {"penalty_entries", penalty_entries, METH_VARARGS,
     "penalty_entries(prompts, outputs, specs, buffer) -> number of entries"},
    {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_hostops", NULL, -1, methods,
                                    NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__hostops(void) { return PyModule_Create(&module); }

// Host-side work on Python token lists, as a CPython extension module (mvsd._hostops): what the
// penalties need to know of each request's history, gathered without converting every list to an
// array first.  32 requests of 650 tokens: 4.0 ms with numpy (np.unique per request), 0.2 here.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

// One request's distinct tokens: an open-addressing table of places in the entry arrays.
typedef struct {
  int32_t* slot;    // place + 1, 0 = free
  size_t cap;       // slots in use for this request, a power of two
  size_t room;      // slots allocated
} Table;

static uint64_t mix(uint64_t x) {
  x ^= x >> 31;
  x *= 0x9e3779b97f4a7c15ull;
  return x ^ (x >> 29);
}

// The place of token t among this request's entries [0, *n), added when it is new.
static int32_t place_of(Table* tb, int64_t* keys, int32_t* n, int64_t t) {
  size_t i = (size_t)mix((uint64_t)t) & (tb->cap - 1);
  while (tb->slot[i]) {
    const int32_t at = tb->slot[i] - 1;
    if (keys[at] == t) return at;
    i = (i + 1) & (tb->cap - 1);
  }
  keys[*n] = t;
  tb->slot[i] = *n + 1;
  return (*n)++;
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
  Table tb = {NULL, 0, 0};
  size_t keys_cap = 0;
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
      size_t cap = 16;
      while (cap < 2 * all) cap *= 2;
      tb.cap = cap;  // its own size: a short history after a long one clears a small table
      if (ok && cap > tb.room) {
        free(tb.slot);
        tb.slot = (int32_t*)malloc(cap * sizeof(int32_t));
        tb.room = tb.slot ? cap : 0;
      }
      if (ok && all > keys_cap) {
        free(keys);
        keys_cap = all;
        keys = (int64_t*)malloc(keys_cap * sizeof(int64_t));
      }
      if (ok && (!tb.slot || (all && !keys))) {
        PyErr_NoMemory();
        ok = 0;
      }
      if (ok) {
        memset(tb.slot, 0, tb.cap * sizeof(int32_t));
        int32_t n = 0;
        for (int s = 0; s < 3 && ok; ++s) {
          // a list can change while __index__ of an element runs: look at it afresh each time
          for (Py_ssize_t i = 0; inner[s] && i < len[s] && i < PySequence_Fast_GET_SIZE(inner[s]);
               ++i) {
            PyObject* item = PySequence_Fast_GET_ITEM(inner[s], i);
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
            if (t == -1 && PyErr_Occurred()) {
              ok = 0;
              break;
            }
            const int32_t before = n;
            const int32_t at = place_of(&tb, keys, &n, t);
            if (at == before) info[total + at] = 0;
            if (s == 0) info[total + at] |= (int32_t)0x80000000u;
            if (s == 1) ++info[total + at];
          }
        }
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
  free(tb.slot);
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

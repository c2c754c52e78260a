/* CPython entry points for the calls an eager program makes per layer: the integers and floats
 * of a C ABI call go straight from Python objects to the library, without ctypes' per-argument
 * conversion (measured on MI355X with the slimmer Python beside it, whole calls: flash_decoding
 * on a 2 x 4 x 1024 x 64 cache 20.7 -> 10.5 us, int4_gemm 16 x 4096 x 4096 11.4 -> 9.0 us).
 * Built by build.py against the product library (linked by path, so the process shares the one
 * copy that _pk loaded); _pk takes the ctypes functions when the module is missing or the
 * library was loaded from elsewhere. Same calls, same kernels, same bits. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>
#include <string.h>

#include "pico_kernels_amd.h"

/* strips_run(handle, a, c, ldc, M, stream) -> status (PK_OK or a PK_E* code) */
static PyObject* pkcall_strips_run(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  (void)self;
  if (nargs != 6) {
    PyErr_SetString(PyExc_TypeError, "strips_run(handle, a, c, ldc, M, stream) takes 6 integers");
    return NULL;
  }
  void* h = PyLong_AsVoidPtr(args[0]);
  const void* a = PyLong_AsVoidPtr(args[1]);
  void* c = PyLong_AsVoidPtr(args[2]);
  const long long ldc = PyLong_AsLongLong(args[3]);
  const long m = PyLong_AsLong(args[4]);
  void* stream = PyLong_AsVoidPtr(args[5]);
  if (PyErr_Occurred()) return NULL;
  if (m < INT32_MIN || m > INT32_MAX) {
    PyErr_SetString(PyExc_OverflowError, "strips_run: M out of range");
    return NULL;
  }
  return PyLong_FromLong(pk_w4a16_strips_run(h, a, c, (int64_t)ldc, (int)m, stream));
}

/* One converted argument of the calls below. */
typedef union {
  void* p;
  int64_t l;
  int i;
  uint32_t u;
  float f;
} Arg;

/* Converts `args` by `kinds`: p pointer (an integer, or None for NULL), l int64, i int, u uint32,
 * f float. Returns 0, or -1 with a Python error set. */
static int convert(const char* name, const char* kinds, PyObject* const* args, Py_ssize_t nargs,
                   Arg* out) {
  Py_ssize_t n = 0;
  for (; kinds[n]; ++n) {
    if (n >= nargs) break;
    PyObject* a = args[n];
    switch (kinds[n]) {
      case 'p':
        out[n].p = a == Py_None ? NULL : PyLong_AsVoidPtr(a);
        break;
      case 'l':
        out[n].l = PyLong_AsLongLong(a);
        break;
      case 'f':
        out[n].f = (float)PyFloat_AsDouble(a);
        break;
      default: {
        const long long v = PyLong_AsLongLong(a);
        const long long lo = kinds[n] == 'i' ? INT32_MIN : 0;
        const long long hi = kinds[n] == 'i' ? INT32_MAX : UINT32_MAX;
        if (v < lo || v > hi) {
          if (!PyErr_Occurred())
            PyErr_Format(PyExc_OverflowError, "%s: argument %zd out of range", name, n + 1);
          return -1;
        }
        if (kinds[n] == 'i') out[n].i = (int)v;
        else out[n].u = (uint32_t)v;
      }
    }
  }
  if (kinds[n] || n != nargs) {
    PyErr_Format(PyExc_TypeError, "%s takes %zu arguments (got %zd)", name, strlen(kinds), nargs);
    return -1;
  }
  return PyErr_Occurred() ? -1 : 0;
}

/* NAME(args...) -> status, the GIL released during the call as ctypes does. */
#define PKCALL(NAME, KINDS, CALL)                                                          \
  static PyObject* call_##NAME(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {  \
    Arg a[sizeof(KINDS)];                                                                  \
    int rc;                                                                                \
    (void)self;                                                                            \
    if (convert(#NAME, KINDS, args, nargs, a)) return NULL;                                \
    Py_BEGIN_ALLOW_THREADS                                                                 \
    rc = CALL;                                                                             \
    Py_END_ALLOW_THREADS                                                                   \
    return PyLong_FromLong(rc);                                                            \
  }

PKCALL(pk_w4a16_gemm, "plplpi" "fpil" "iiii" "plp",
       pk_w4a16_gemm(a[0].p, a[1].l, a[2].p, a[3].l, a[4].p, a[5].i, a[6].f, a[7].p, a[8].i, a[9].l,
                     a[10].i, a[11].i, a[12].i, a[13].i, a[14].p, (size_t)a[15].l, a[16].p))
PKCALL(pk_w4a16_gemm_bias, "plplpi" "fpipil" "iiii" "plp",
       pk_w4a16_gemm_bias(a[0].p, a[1].l, a[2].p, a[3].l, a[4].p, a[5].i, a[6].f, a[7].p, a[8].i,
                          a[9].p, a[10].i, a[11].l, a[12].i, a[13].i, a[14].i, a[15].i, a[16].p,
                          (size_t)a[17].l, a[18].p))
PKCALL(pk_w4a16_gemm_tiled, "plppi" "fpipil" "iiii" "plp",
       pk_w4a16_gemm_tiled(a[0].p, a[1].l, a[2].p, a[3].p, a[4].i, a[5].f, a[6].p, a[7].i, a[8].p,
                           a[9].i, a[10].l, a[11].i, a[12].i, a[13].i, a[14].i, a[15].p,
                           (size_t)a[16].l, a[17].p))
PKCALL(pk_w4a16_strips_run_rows, "pppl" "ip",
       pk_w4a16_strips_run_rows(a[0].p, a[1].p, a[2].p, a[3].l, a[4].i, a[5].p))
PKCALL(pk_w4a16_gemm_strips_rows, "plpp" "ifpi" "pil" "iiip",
       pk_w4a16_gemm_strips_rows(a[0].p, a[1].l, a[2].p, a[3].p, a[4].i, a[5].f, a[6].p, a[7].i,
                                 a[8].p, a[9].i, a[10].l, a[11].i, a[12].i, a[13].i, a[14].p))
PKCALL(pk_w4a16_prep_checked, "pilpf" "plii" "ppup",
       pk_w4a16_prep_checked(a[0].p, a[1].i, a[2].l, a[3].p, a[4].f, a[5].p, a[6].l, a[7].i, a[8].i,
                             a[9].p, a[10].p, a[11].u, a[12].p))
PKCALL(pk_flash_decode, "pll" "plll" "plll" "iiiii" "f" "pplp",
       pk_flash_decode(a[0].p, a[1].l, a[2].l, a[3].p, a[4].l, a[5].l, a[6].l, a[7].p, a[8].l,
                       a[9].l, a[10].l, a[11].i, a[12].i, a[13].i, a[14].i, a[15].i, a[16].f,
                       a[17].p, a[18].p, (size_t)a[19].l, a[20].p))

#define ENTRY(NAME) \
  {#NAME, (PyCFunction)(void (*)(void))call_##NAME, METH_FASTCALL, #NAME "(...) -> status"}
static PyMethodDef pkcall_methods[] = {
    {"strips_run", (PyCFunction)(void (*)(void))pkcall_strips_run, METH_FASTCALL,
     "pk_w4a16_strips_run(handle, a, c, ldc, M, stream) -> status"},
    ENTRY(pk_w4a16_gemm), ENTRY(pk_w4a16_gemm_bias), ENTRY(pk_w4a16_gemm_tiled),
    ENTRY(pk_w4a16_strips_run_rows), ENTRY(pk_w4a16_gemm_strips_rows), ENTRY(pk_w4a16_prep_checked), ENTRY(pk_flash_decode),
    {NULL, NULL, 0, NULL},
};

static struct PyModuleDef pkcall_module = {PyModuleDef_HEAD_INIT, "_pkcall", NULL, -1,
                                           pkcall_methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__pkcall(void) { return PyModule_Create(&pkcall_module); }

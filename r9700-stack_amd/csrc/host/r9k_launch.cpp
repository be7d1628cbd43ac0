// r9k_launch.cpp -- the Python bindings' launch helpers as a CPython extension (r9700_vllm/kernels/_r9k_launch.*.so):
//
//   call(spec, *args) -> int         a libr9k C entry; spec is its address (8 bytes) and one kind letter an argument
//   empty(like, dtype, *sizes)       torch.empty(sizes) of a torch.dtype on like's device
//   TORCH                            the torch version it was built against
//
// Kinds: p a device pointer (a tensor passes its data pointer, an int itself), o the same or None (0), l a long, i an int.
// Numbers go through __index__ and wrap to their C width, as ctypes converts them: a 0-d integer tensor in an l or i
// position is its value, never its address, and None is a number nowhere.
//
// A decode step is a handful of launches of a few microseconds, and its host side was bound by the bindings: a ctypes
// call converts each argument by its argtype (a 20-argument launch with its data_ptr() calls ~5 us beside the ~3 us the
// launch itself takes), torch.empty 1.7 us an output. Measured on MI355X's host, Python loop over one entry: see the
// figures in kernels/moe.py. Entries with a floating-point argument stay on ctypes.
//
// Every libr9k entry takes long and int arguments only and returns int. They are called here through a type of as many
// longs as arguments were given: on x86-64 an int parameter is the low half of the same register or stack slot.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <utility>

#if !defined(__x86_64__)
#error "the calling convention above is x86-64's"
#endif

namespace {

constexpr int MAX_ARGS = 28;

template <size_t>
using Long = long;

template <size_t... I>
int call_n(long fn, const long* v, std::index_sequence<I...>) {
  return reinterpret_cast<int (*)(Long<I>...)>(fn)(v[I]...);
}

template <size_t N>
int dispatch(size_t n, long fn, const long* v) {
  if (n == N) return call_n(fn, v, std::make_index_sequence<N>{});
  if constexpr (N < MAX_ARGS) return dispatch<N + 1>(n, fn, v);
  return -1000;
}

// A number argument as ctypes takes it: anything with __index__, wrapped to 64 bits.
bool number(PyObject* a, long* v) {
  PyObject* n = PyNumber_Index(a);
  if (!n) return false;
  *v = (long)PyLong_AsUnsignedLongMask(n);
  Py_DECREF(n);
  return !(*v == -1 && PyErr_Occurred());
}

PyObject* py_call(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs < 1 || !PyBytes_Check(args[0]) || PyBytes_GET_SIZE(args[0]) <= (Py_ssize_t)sizeof(long)) {
    PyErr_SetString(PyExc_TypeError, "call(spec, *args): spec is an entry's address and its argument kinds, as bytes");
    return nullptr;
  }
  const char* kind = PyBytes_AS_STRING(args[0]) + sizeof(long);
  const Py_ssize_t want = PyBytes_GET_SIZE(args[0]) - (Py_ssize_t)sizeof(long);
  if (want > MAX_ARGS || nargs - 1 != want) {
    PyErr_Format(PyExc_TypeError, "call: the entry takes %zd arguments (at most %d), got %zd", want, MAX_ARGS, nargs - 1);
    return nullptr;
  }
  long fn;
  std::memcpy(&fn, PyBytes_AS_STRING(args[0]), sizeof fn);
  if (fn == 0) {
    PyErr_SetString(PyExc_ValueError, "call: null entry address");
    return nullptr;
  }
  long v[MAX_ARGS];
  for (Py_ssize_t i = 0; i < want; i++) {
    PyObject* a = args[i + 1];
    int over = 0;
    if (PyLong_CheckExact(a) && (v[i] = PyLong_AsLongAndOverflow(a, &over), over == 0)) {
      if (kind[i] == 'i') v[i] = (int)v[i];
    } else if ((kind[i] == 'p' || kind[i] == 'o') && THPVariable_Check(a)) {
      v[i] = reinterpret_cast<long>(THPVariable_Unpack(a).data_ptr());
    } else if (kind[i] == 'o' && a == Py_None) {
      v[i] = 0;
    } else if (!number(a, &v[i])) {
      if (PyErr_ExceptionMatches(PyExc_TypeError))
        PyErr_Format(PyExc_TypeError, "call: argument %zd (kind %c) is a %s", i + 1, kind[i], Py_TYPE(a)->tp_name);
      return nullptr;
    } else if (kind[i] == 'i') {
      v[i] = (int)v[i];
    }
  }
  // without the GIL, as ctypes calls it: a launch waits while its queue is full, and another thread may have to run first
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = dispatch<1>((size_t)want, fn, v);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

PyObject* py_empty(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs < 3 || nargs > 6 || !THPVariable_Check(args[0]) || !THPDtype_Check(args[1])) {
    PyErr_SetString(PyExc_TypeError, "empty(like, dtype, *sizes): a tensor, a torch.dtype and 1 to 4 ints");
    return nullptr;
  }
  const at::Tensor& like = THPVariable_Unpack(args[0]);
  int64_t sz[4];
  for (Py_ssize_t i = 2; i < nargs; i++) {
    sz[i - 2] = PyLong_AsLong(args[i]);
    if (sz[i - 2] == -1 && PyErr_Occurred()) return nullptr;
  }
  return THPVariable_Wrap(at::empty(at::IntArrayRef(sz, (size_t)nargs - 2),
                                    at::TensorOptions().dtype(reinterpret_cast<THPDtype*>(args[1])->scalar_type)
                                        .device(like.device())));
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_call)), METH_FASTCALL,
     "call(spec, *args) -> int: a libr9k entry, its address and argument kinds in spec, on tensors, numbers and None"},
    {"empty", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_empty)), METH_FASTCALL,
     "empty(like, dtype, *sizes) -> an uninitialised tensor on like's device"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_r9k_launch", "Launch helpers of the libr9k bindings.", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__r9k_launch(void) {
  PyObject* m = PyModule_Create(&kModule);
  if (m && PyModule_AddStringConstant(m, "TORCH", R9K_TORCH)) Py_CLEAR(m);
  return m;
}

// Calls of the kernel library's C functions from Python, without ctypes' conversions.
//
// A launch passes up to 38 integers, pointers and floats, and ctypes makes an object of each: 0.9 us for the rotary embedding's 19
// arguments, 1.2 us for decode attention's 34, where a launch itself takes 3.3.  Here they are read straight from the Python objects:
// 0.1 us.  An argument of any other kind than an int, a float or None (a ctypes object, a numpy number) sends the call through
// the ctypes function, which converts or refuses it as before.
//
// One call takes any signature: on x86-64 Linux integers and pointers take the six integer registers and then the stack, floats
// the eight vector registers, each in their own order.  A function of both can be called with its integers first and eight floats after
// them, as long as it has no more than eight.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <array>
#include <utility>

#if !defined(__x86_64__) || !defined(__linux__)
#error "the calling convention below is that of x86-64 Linux"
#endif

namespace {

constexpr int MOST_INTS = 48, MOST_FLOATS = 8, MOST = MOST_INTS + MOST_FLOATS;

struct Function {
  void* address = nullptr;            // null: through ctypes alone
  PyObject* by_ctypes = nullptr;
  int n = 0, ints = 0;
  char kind[MOST] = {};               // P: pointer, I: int, L: long, F: float
};

template <size_t> using Int = long;
template <size_t... I> int invoke(void* address, const long* v, const float* f, std::index_sequence<I...>) {
  using Fn = int (*)(Int<I>..., float, float, float, float, float, float, float, float);
  return reinterpret_cast<Fn>(address)(v[I]..., f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7]);
}
using Invoke = int (*)(void*, const long*, const float*);
template <size_t N> int invoke_n(void* address, const long* v, const float* f) {
  return invoke(address, v, f, std::make_index_sequence<N>());
}
template <size_t... N> constexpr std::array<Invoke, sizeof...(N)> invokes(std::index_sequence<N...>) { return {invoke_n<N>...}; }
constexpr auto INVOKES = invokes(std::make_index_sequence<MOST_INTS + 1>());

PyObject *functions, *missing;        // name -> capsule of a Function; called with a name that is not there, raises

bool through_ctypes(const Function& fn, PyObject* const* args, Py_ssize_t n, long& result) {
  PyObject* r = PyObject_Vectorcall(fn.by_ctypes, args, (size_t)n, nullptr);
  if (!r) return false;
  result = PyLong_AsLong(r);
  Py_DECREF(r);
  return result != -1 || !PyErr_Occurred();
}

// args: the function's own
bool run_bound(const Function& fn, PyObject* const* args, Py_ssize_t n, long& result) {
  if (n != fn.n || !fn.address) return through_ctypes(fn, args, n, result);
  long v[MOST_INTS];
  float f[MOST_FLOATS] = {};
  int nv = 0, nf = 0;
  for (int i = 0; i < fn.n; ++i) {
    PyObject* a = args[i];
    if (fn.kind[i] == 'F') {
      if (PyFloat_Check(a)) f[nf++] = (float)PyFloat_AS_DOUBLE(a);
      else if (PyLong_Check(a)) {
        const double d = PyLong_AsDouble(a);
        if (d == -1.0 && PyErr_Occurred()) return false;
        f[nf++] = (float)d;
      } else return through_ctypes(fn, args, n, result);
    } else if (PyLong_Check(a)) {
      v[nv++] = (long)PyLong_AsUnsignedLongMask(a);     // (the lower bits, as ctypes takes them)
    } else if (a == Py_None && fn.kind[i] == 'P') {
      v[nv++] = 0;
    } else {
      return through_ctypes(fn, args, n, result);
    }
  }
  Py_BEGIN_ALLOW_THREADS                                // (a launch waits where a queue is full)
  result = INVOKES[fn.ints](fn.address, v, f);
  Py_END_ALLOW_THREADS
  return true;
}

// args: the name, then the function's own
bool run(PyObject* const* args, Py_ssize_t n, long& result) {
  if (n < 1) {
    PyErr_SetString(PyExc_TypeError, "the first argument is a function's name");
    return false;
  }
  PyObject* capsule = PyDict_GetItemWithError(functions, args[0]);
  if (!capsule) {
    if (!PyErr_Occurred()) Py_XDECREF(PyObject_CallOneArg(missing, args[0]));
    if (!PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, args[0]);
    return false;
  }
  // (another thread, which runs while this one has given up the interpreter's lock, can bind the name anew)
  Py_INCREF(capsule);
  const bool answered = run_bound(*static_cast<Function*>(PyCapsule_GetPointer(capsule, nullptr)), args + 1, n - 1, result);
  Py_DECREF(capsule);
  return answered;
}

// call(name, *args): raises unless the function answers 0
PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
  long result;
  if (!run(args, n, result)) return nullptr;
  if (result != 0) {
    PyErr_Format(PyExc_RuntimeError, "%U failed with code %ld", args[0], result);
    return nullptr;
  }
  Py_RETURN_NONE;
}

// value(name, *args): the function's answer
PyObject* value(PyObject*, PyObject* const* args, Py_ssize_t n) {
  long result;
  return run(args, n, result) ? PyLong_FromLong(result) : nullptr;
}

void free_function(PyObject* capsule) {
  Function* fn = static_cast<Function*>(PyCapsule_GetPointer(capsule, nullptr));
  Py_XDECREF(fn->by_ctypes);
  delete fn;
}

// bind(name, address, kinds, ctypes function): an int function; a name that is bound again is replaced
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *name, *by_ctypes;
  unsigned long long address;
  const char* kinds;
  Py_ssize_t n;
  if (!PyArg_ParseTuple(args, "UKs#O", &name, &address, &kinds, &n, &by_ctypes)) return nullptr;
  Function* fn = new Function;
  int floats = 0;
  for (Py_ssize_t i = 0; i < n; ++i) (kinds[i] == 'F' ? floats : fn->ints)++;
  if (fn->ints <= MOST_INTS && floats <= MOST_FLOATS) {
    fn->address = reinterpret_cast<void*>(address);
    for (Py_ssize_t i = 0; i < n; ++i) fn->kind[i] = kinds[i];
  }
  fn->n = (int)n;
  Py_INCREF(by_ctypes);
  fn->by_ctypes = by_ctypes;
  PyObject* capsule = PyCapsule_New(fn, nullptr, free_function);
  if (!capsule) {
    Py_DECREF(by_ctypes);
    delete fn;
    return nullptr;
  }
  const int rc = PyDict_SetItem(functions, name, capsule);
  Py_DECREF(capsule);
  if (rc != 0) return nullptr;
  Py_RETURN_NONE;
}

PyObject* on_missing(PyObject*, PyObject* callable) {
  Py_INCREF(callable);
  Py_XSETREF(missing, callable);
  Py_RETURN_NONE;
}

PyMethodDef METHODS[] = {
    {"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(call)), METH_FASTCALL, "call(name, *args): raises unless the function answers 0"},
    {"value", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(value)), METH_FASTCALL, "value(name, *args): the function's answer"},
    {"bind", bind, METH_VARARGS, "bind(name, address, kinds, ctypes function)"},
    {"on_missing", on_missing, METH_O, "on_missing(callable): called with the name of a function that is not bound, raises"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef MODULE = {PyModuleDef_HEAD_INIT, "_vda_call", "Calls of C functions by name", -1, METHODS, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__vda_call() {
  functions = PyDict_New();
  if (!functions) return nullptr;
  Py_INCREF(Py_None);
  missing = Py_None;
  return PyModule_Create(&MODULE);
}

// What every launch of a kernel does on the host, natively: its operands checked, its result allocated, its entry point called.
//
// A step that is not replayed as a graph issues 100 to 350 launches, and in Python the checks (0.47 us a tensor), the allocation (1.7),
// the stream (0.35) and the call through ctypes (1.5 beyond the launch itself) of each took longer than most of the kernels.
// Here: 0.06, 1.5, 0.13 and 0.25.
//
//   check(tensor, name, shape = None, dtype = None)      nothing if the tensor is on the GPU, contiguous and as expected; anything else is
//                                                    handed to the Python check, whose errors it raises
//   empty(shape, dtype, like)                        an uninitialised tensor on like's device
//   stream()                                         torch's current stream of the current device, as a number
//   call(module, function, types, *arguments)        the library's function with these arguments, as ctypes would call it; an error code is
//                                                    handed to the Python side; whatever is not plain (other types, other objects) is
//                                                    left to ctypes
//   connect(check, call, failed, entry, array)       the Python functions for all that, and the type of ctypes' arrays
//
// The call: by the C calling convention of x86-64 the first six whole numbers and pointers of a call are in registers, the first eight
// floating-point ones in others, and all further whole numbers on the stack in order, whatever stands between them.  So one function type
// with six, eight and STACK of them calls every function of up to that many.
#include <Python.h>

#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <string>
#include <vector>

#if !defined(__x86_64__)
#error "host_calls.cpp knows the calling convention of x86-64 only"
#endif

namespace {

constexpr int REGISTERS = 6, FLOATS = 8, STACK = 32;

struct Entry {
  void* function;
  std::string types;        // p: pointer (a tensor's address, a number, None), a: a ctypes array's address, i: 32 bits, l: 64 bits, f: float
  std::vector<PyObject*> elements;        // of the arrays, in order
  ~Entry() {
    for (PyObject* e : elements) Py_DECREF(e);
  }
};

struct WithoutGil {
  PyThreadState* state = PyEval_SaveThread();
  ~WithoutGil() { PyEval_RestoreThread(state); }
};

PyObject *slow_check = nullptr, *slow_call = nullptr, *call_failed = nullptr, *make_entry = nullptr, *array_type = nullptr, *entries_name = nullptr,
         *type_name = nullptr;

bool as_expected(PyObject* const* a, Py_ssize_t n) {
  if (!THPVariable_Check(a[0])) return false;
  const at::Tensor& t = THPVariable_Unpack(a[0]);
  if (!t.is_cuda() || !t.is_contiguous()) return false;
  if (n > 3 && a[3] != Py_None) {
    if (!THPDtype_Check(a[3]) || reinterpret_cast<THPDtype*>(a[3])->scalar_type != t.scalar_type()) return false;
  }
  if (n > 2 && a[2] != Py_None) {
    if (!PyTuple_Check(a[2]) || PyTuple_GET_SIZE(a[2]) != t.dim()) return false;
    for (int64_t i = 0; i < t.dim(); ++i) {
      PyObject* want = PyTuple_GET_ITEM(a[2], i);
      if (want == Py_None) continue;
      if (!PyLong_CheckExact(want)) return false;
      const long long v = PyLong_AsLongLong(want);
      if (v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
      }
      if (v != t.size(i)) return false;
    }
  }
  return true;
}

PyObject* check(PyObject*, PyObject* const* a, Py_ssize_t n, PyObject* keywords) {
  if (!keywords && n >= 2 && n <= 4 && as_expected(a, n)) Py_RETURN_NONE;
  return PyObject_Vectorcall(slow_check, a, n, keywords);
}

PyObject* empty(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 3 || !PyTuple_Check(a[0]) || !THPDtype_Check(a[1]) || !THPVariable_Check(a[2])) {
    PyErr_SetString(PyExc_TypeError, "empty(shape: tuple, dtype: torch.dtype, like: torch.Tensor)");
    return nullptr;
  }
  int64_t sizes[8];
  const Py_ssize_t dims = PyTuple_GET_SIZE(a[0]);
  if (dims > 8) {
    PyErr_SetString(PyExc_TypeError, "empty: at most eight dimensions");
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < dims; ++i) {
    sizes[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(a[0], i));
    if (sizes[i] == -1 && PyErr_Occurred()) return nullptr;
  }
  HANDLE_TH_ERRORS
  const at::TensorOptions options = at::TensorOptions().dtype(reinterpret_cast<THPDtype*>(a[1])->scalar_type).device(THPVariable_Unpack(a[2]).device());
  at::Tensor made;
  {
    WithoutGil released;        // (an allocation may wait)
    made = at::empty(at::IntArrayRef(sizes, dims), options);
  }
  return THPVariable_Wrap(std::move(made));
  END_HANDLE_TH_ERRORS
}

PyObject* stream(PyObject*, PyObject*) {
  HANDLE_TH_ERRORS
  return PyLong_FromVoidPtr((void*)c10::hip::getCurrentHIPStream().stream());
  END_HANDLE_TH_ERRORS
}

void free_entry(PyObject* capsule) { delete static_cast<Entry*>(PyCapsule_GetPointer(capsule, "entry")); }

// entry(address, types, elements): what ``call`` keeps of a function, or None where the types do not fit the one call there is
PyObject* entry(PyObject*, PyObject* const* a, Py_ssize_t n) {
  const char* types = n == 3 && PyTuple_Check(a[2]) ? PyUnicode_AsUTF8(a[1]) : nullptr;
  if (!types) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "entry(address, types, elements: tuple)");
    return nullptr;
  }
  int floats = 0, others = 0, arrays = 0;
  for (const char* c = types; *c; ++c) {
    if (*c == 'f') ++floats;
    else if (*c == 'p' || *c == 'a' || *c == 'i' || *c == 'l') ++others;
    else Py_RETURN_NONE;
    arrays += *c == 'a';
  }
  if (floats > FLOATS || others > REGISTERS + STACK) Py_RETURN_NONE;
  if (arrays != PyTuple_GET_SIZE(a[2])) {
    PyErr_SetString(PyExc_TypeError, "entry: an element type for every array");
    return nullptr;
  }
  void* function = PyLong_AsVoidPtr(a[0]);
  if (!function) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "entry: no address");
    return nullptr;
  }
  Entry* made = new Entry{function, types, {}};
  for (int i = 0; i < arrays; ++i) {
    PyObject* e = PyTuple_GET_ITEM(a[2], i);
    Py_INCREF(e);
    made->elements.push_back(e);
  }
  PyObject* capsule = PyCapsule_New(made, "entry", free_entry);
  if (!capsule) delete made;
  return capsule;
}

typedef uint64_t W;
typedef int (*Function)(W, W, W, W, W, W, double, double, double, double, double, double, double, double,  //
                        W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W);

// The buffers that a call's arguments were taken from, held until it is over.
struct Buffers {
  Py_buffer views[REGISTERS + STACK];
  int n = 0;
  ~Buffers() {
    while (n > 0) PyBuffer_Release(&views[--n]);
  }
};

// Whether v is a ctypes array of these elements, as a pointer to them takes it: other objects with a buffer, a ctypes pointer among them, hold something else there.
bool is_array_of(PyObject* v, PyObject* element) {
  if (!PyType_IsSubtype(Py_TYPE(v), reinterpret_cast<PyTypeObject*>(array_type))) return false;
  PyObject* of = PyObject_GetAttr(reinterpret_cast<PyObject*>(Py_TYPE(v)), type_name);
  if (!of) {
    PyErr_Clear();
    return false;
  }
  Py_DECREF(of);        // (its type keeps it)
  return of == element;
}

// The arguments as words; false: one is not plain
bool words(const Entry& entry, PyObject* const* a, W* whole, double* floats, Buffers& buffers) {
  const std::string& types = entry.types;
  int w = 0, f = 0;
  for (size_t i = 0; i < types.size(); ++i) {
    PyObject* v = a[i];
    if (types[i] == 'f') {
      double d;
      if (PyFloat_CheckExact(v)) d = PyFloat_AS_DOUBLE(v);
      else if (PyLong_CheckExact(v)) d = PyLong_AsDouble(v);
      else return false;
      const float s = (float)d;
      W bits = 0;
      memcpy(&bits, &s, sizeof(s));
      memcpy(&floats[f++], &bits, sizeof(bits));
    } else if (types[i] == 'p') {
      if (THPVariable_Check(v)) {
        const at::Tensor& t = THPVariable_Unpack(v);
        if (!t.has_storage()) return false;
        whole[w++] = (W)t.data_ptr();
      } else if (v == Py_None) whole[w++] = 0;
      else if (PyLong_CheckExact(v)) whole[w++] = (W)PyLong_AsVoidPtr(v);
      else return false;
    } else if (types[i] == 'a') {
      if (!is_array_of(v, entry.elements[buffers.n])) return false;
      Py_buffer* view = &buffers.views[buffers.n];
      if (PyObject_GetBuffer(v, view, PyBUF_SIMPLE) != 0) {
        PyErr_Clear();
        return false;
      }
      ++buffers.n;
      whole[w++] = (W)view->buf;
    } else {
      if (!PyLong_Check(v)) return false;        // (True and False among them)
      whole[w++] = (W)PyLong_AsLongLong(v);
    }
  }
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

PyObject* call_or_throw(PyObject* const* a, Py_ssize_t n) {
  if (n < 3) {
    PyErr_SetString(PyExc_TypeError, "call(module, function, types, *arguments)");
    return nullptr;
  }
  PyObject* entries = PyObject_GetAttr(a[0], entries_name);
  if (!entries) return nullptr;
  PyObject* found = PyDict_CheckExact(entries) ? PyDict_GetItemWithError(entries, a[1]) : nullptr;
  Py_DECREF(entries);        // (the module keeps it)
  if (!found) {
    if (PyErr_Occurred()) return nullptr;
    found = PyObject_CallFunctionObjArgs(make_entry, a[0], a[1], a[2], nullptr);        // (which keeps it in the module's entries)
    if (!found) return nullptr;
    Py_DECREF(found);
  }
  if (found != Py_None) {
    const Entry* e = static_cast<const Entry*>(PyCapsule_GetPointer(found, "entry"));
    if (!e) return nullptr;
    W w[REGISTERS + STACK] = {};
    double d[FLOATS] = {};
    Buffers buffers;
    if ((size_t)(n - 3) == e->types.size() && words(*e, a + 3, w, d, buffers)) {
      const Function f = reinterpret_cast<Function>(e->function);
      int rc;
      Py_BEGIN_ALLOW_THREADS
      rc = f(w[0], w[1], w[2], w[3], w[4], w[5], d[0], d[1], d[2], d[3], d[4], d[5], d[6], d[7],  //
             w[6], w[7], w[8], w[9], w[10], w[11], w[12], w[13], w[14], w[15], w[16], w[17], w[18], w[19], w[20], w[21], w[22], w[23], w[24],
             w[25], w[26], w[27], w[28], w[29], w[30], w[31], w[32], w[33], w[34], w[35], w[36], w[37]);
      Py_END_ALLOW_THREADS
      if (rc == 0) Py_RETURN_NONE;
      PyObject* code = PyLong_FromLong(rc);
      if (!code) return nullptr;
      PyObject* r = PyObject_CallFunctionObjArgs(call_failed, a[0], a[1], code, nullptr);
      Py_DECREF(code);
      return r;
    }
  }
  return PyObject_Vectorcall(slow_call, a, n, nullptr);
}

PyObject* call(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  return call_or_throw(a, n);
  END_HANDLE_TH_ERRORS
}

PyObject* connect(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 5 || !PyType_Check(a[4])) {
    PyErr_SetString(PyExc_TypeError, "connect(check, call, failed, entry, array: type)");
    return nullptr;
  }
  PyObject** to[5] = {&slow_check, &slow_call, &call_failed, &make_entry, &array_type};
  for (int i = 0; i < 5; ++i) {
    Py_INCREF(a[i]);
    Py_XDECREF(*to[i]);
    *to[i] = a[i];
  }
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"check", (PyCFunction)(void*)check, METH_FASTCALL | METH_KEYWORDS, nullptr},
                         {"empty", (PyCFunction)(void*)empty, METH_FASTCALL, nullptr},
                         {"stream", (PyCFunction)stream, METH_NOARGS, nullptr},
                         {"entry", (PyCFunction)(void*)entry, METH_FASTCALL, nullptr},
                         {"call", (PyCFunction)(void*)call, METH_FASTCALL, nullptr},
                         {"connect", (PyCFunction)(void*)connect, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef definition = {PyModuleDef_HEAD_INIT, "host_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_host_calls() {
  entries_name = PyUnicode_InternFromString("entries");
  type_name = PyUnicode_InternFromString("_type_");
  return entries_name && type_name ? PyModule_Create(&definition) : nullptr;
}

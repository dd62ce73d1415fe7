// Calls of the kernel library's C entry points from Python without ctypes' conversions.
//
// A launcher takes 20 to 45 plain numbers and pointers; ctypes spends 2 to 4.4 us on turning them into C
// (0.1 us an argument), as much as the launch itself and up to a third of a small step's host time.  Here an
// argument costs about 10 ns: 41 arguments (eia_linear_scan) 4.4 -> 0.5 us.  Whatever is not a plain number of the
// declared kind (ctypes objects, arrays, a wrong count) goes to the ctypes function that the object was made
// from, so that what is accepted and what is refused stays as it is there.
#include <pybind11/pybind11.h>

#include <cstdint>
#include <cstring>
#include <structmember.h>

namespace py = pybind11;

#if !defined(__x86_64__) || defined(_WIN32)
#error "the argument passing below is that of the System V x86-64 ABI"
#endif

namespace {

constexpr int MAX_ARGS = 64, MAX_FLOATS = 8;

struct KernelCall {
  PyObject_HEAD
  vectorcallfunc call;
  void* entry;
  PyObject* plain;                          // the ctypes function
  int n;
  char kinds[MAX_ARGS];                     // 'p' pointer, 'l' long, 'i' int, 'f' float
};

// Integers and pointers of a call take registers and then 8-byte stack places in their own order, whatever their
// width, and up to eight floats take xmm registers in theirs; a callee does not see places behind its own.  So
// one prototype per count of integers, rounded up, serves every entry point.
template <class... T> int invoke(void* f, const float* x, T... a) {
  using Fn = int (*)(T..., float, float, float, float, float, float, float, float);
  return reinterpret_cast<Fn>(f)(a..., x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7]);
}
template <size_t... I> int spread(void* f, const uint64_t* a, const float* x, std::index_sequence<I...>) {
  return invoke(f, x, a[I]...);
}

// One argument; false: not a plain number of its kind.
inline bool convert(char kind, PyObject* o, uint64_t& i, float& f) {
  if (kind == 'f') {
    if (PyFloat_CheckExact(o)) {
      f = static_cast<float>(PyFloat_AS_DOUBLE(o));
      return true;
    }
    if (!PyLong_CheckExact(o)) return false;
    const double d = PyLong_AsDouble(o);
    if (d == -1.0 && PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
    f = static_cast<float>(d);
    return true;
  }
  if (kind == 'p' && o == Py_None) {
    i = 0;
    return true;
  }
  if (!PyLong_CheckExact(o) && !(kind != 'p' && PyBool_Check(o))) return false;
  i = PyLong_AsUnsignedLongLongMask(o);
  if (kind == 'i') i &= 0xffffffffu;
  return true;
}

PyObject* kernel_call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kw) {
  auto* k = reinterpret_cast<KernelCall*>(self);
  const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
  uint64_t ints[MAX_ARGS];
  float floats[MAX_FLOATS] = {};
  int ni = 0, nf = 0;
  bool ok = n == k->n && kw == nullptr;
  for (Py_ssize_t j = 0; ok && j < n; ++j) {
    uint64_t i = 0;
    float f = 0.f;
    ok = convert(k->kinds[j], args[j], i, f);
    if (k->kinds[j] == 'f') floats[nf++] = f;
    else ints[ni++] = i;
  }
  if (!ok) return PyObject_Vectorcall(k->plain, args, nargsf & ~PY_VECTORCALL_ARGUMENTS_OFFSET, kw);
  const int end = ni <= 8 ? 8 : ni <= 16 ? 16 : ni <= 32 ? 32 : ni <= 48 ? 48 : 64;
  while (ni < end) ints[ni++] = 0;
  int r;
  Py_BEGIN_ALLOW_THREADS                    // (as ctypes does)
  switch (end) {
    case 8: r = spread(k->entry, ints, floats, std::make_index_sequence<8>()); break;
    case 16: r = spread(k->entry, ints, floats, std::make_index_sequence<16>()); break;
    case 32: r = spread(k->entry, ints, floats, std::make_index_sequence<32>()); break;
    case 48: r = spread(k->entry, ints, floats, std::make_index_sequence<48>()); break;
    default: r = spread(k->entry, ints, floats, std::make_index_sequence<64>()); break;
  }
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(r);
}

PyObject* kernel_new(PyTypeObject* type, PyObject* args, PyObject* kw) {
  unsigned long long entry = 0;
  const char* kinds = nullptr;
  PyObject* plain = nullptr;
  if (kw && PyDict_GET_SIZE(kw)) {
    PyErr_SetString(PyExc_TypeError, "KernelCall: positional arguments");
    return nullptr;
  }
  if (!PyArg_ParseTuple(args, "KsO", &entry, &kinds, &plain)) return nullptr;
  const size_t n = std::strlen(kinds);
  size_t nf = 0;
  bool known = true;
  for (size_t i = 0; i < n; ++i) {
    known &= std::strchr("plif", kinds[i]) != nullptr;
    nf += kinds[i] == 'f';
  }
  if (!entry || !known || n > MAX_ARGS || nf > MAX_FLOATS || !PyCallable_Check(plain)) {
    PyErr_SetString(PyExc_ValueError, "KernelCall: entry point or argument kinds");
    return nullptr;
  }
  auto* k = reinterpret_cast<KernelCall*>(type->tp_alloc(type, 0));
  if (!k) return nullptr;
  k->call = kernel_call;
  k->entry = reinterpret_cast<void*>(entry);
  Py_INCREF(plain);
  k->plain = plain;
  k->n = static_cast<int>(n);
  std::memcpy(k->kinds, kinds, n);
  return reinterpret_cast<PyObject*>(k);
}

void kernel_dealloc(PyObject* self) {
  PyTypeObject* type = Py_TYPE(self);
  Py_XDECREF(reinterpret_cast<KernelCall*>(self)->plain);
  type->tp_free(self);
  Py_DECREF(type);
}

PyMemberDef members[] = {
    {"__vectorcalloffset__", T_PYSSIZET, offsetof(KernelCall, call), READONLY, nullptr},
    {"plain", T_OBJECT_EX, offsetof(KernelCall, plain), READONLY, nullptr},
    {nullptr, 0, 0, 0, nullptr}};
PyType_Slot slots[] = {{Py_tp_new, reinterpret_cast<void*>(kernel_new)},
                       {Py_tp_dealloc, reinterpret_cast<void*>(kernel_dealloc)},
                       {Py_tp_call, reinterpret_cast<void*>(PyVectorcall_Call)},
                       {Py_tp_members, members},
                       {0, nullptr}};
PyType_Spec spec = {"_eia_runtime.KernelCall", sizeof(KernelCall), 0,
                    Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL, slots};

}  // namespace

void register_kernel_call(py::module_& m) {
  m.attr("KernelCall") = py::reinterpret_steal<py::object>(PyType_FromSpec(&spec));
}

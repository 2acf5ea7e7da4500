// Calls from the Python binding into the C ABI: an extension module whose
// functions do in C++ what the binding did per call in Python (argument
// conversion with the device and contiguity checks, the current stream, output
// allocation, the status check). A small projection is two launches of about
// 3 us each; the Python side of it took longer than the GPU.
//
//   entry(address, kinds): a handle for launch and value; kinds has one
//     letter per parameter, 'p' pointer or 'i' integer.
//   launch(entry, *args): entry(args.., current stream). A pointer argument is
//     a tensor (its device pointer), None (NULL) or an int address; an integer
//     is anything with __index__, as through ctypes. A nonzero status goes to
//     the function given to set_check, which raises.
//   value(entry, *args): entry(args..) as int64 (size functions).
//   pointer(tensor): its device pointer, checked as an argument is.
//   empty(like, dtype, *sizes): torch.empty on like's device.
//
// Every entry takes integers and pointers only, which the x86-64 calling
// convention passes in 64-bit registers and stack slots.
#include <Python.h>

#include <ATen/ops/empty.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstring>
#include <deque>
#include <utility>

#include "build_id.inc"  // CLEF_BUILD_ID, generated by the Makefile
#include "host_abi.inc"  // CLEF_TORCH_VERSION, likewise

namespace {

constexpr int kMaxArgs = 24;

struct Entry {
  void* f;
  uint32_t pointers;  // bit i: parameter i is a pointer
  int args;
};
std::deque<Entry> g_entries;  // handles are addresses of its elements; kept for the process

PyObject* g_check = nullptr;       // called with a nonzero status
PyObject* g_device = nullptr;      // torch._C._cuda_getDevice
PyObject* g_raw_stream = nullptr;  // torch._C._cuda_getCurrentRawStream

template <size_t... I>
int64_t invoke(void* f, const int64_t* v, std::index_sequence<I...>) {
  return reinterpret_cast<int64_t (*)(decltype((void)I, int64_t{})...)>(f)(v[I]...);
}
using Invoker = int64_t (*)(void*, const int64_t*);
template <size_t N>
int64_t invoke_n(void* f, const int64_t* v) {
  return invoke(f, v, std::make_index_sequence<N>{});
}
template <size_t... N>
constexpr Invoker pick(size_t n, std::index_sequence<N...>) {
  constexpr Invoker table[] = {&invoke_n<N>...};
  return table[n];
}

bool tensor_pointer(PyObject* o, int64_t& out) {
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.is_cuda() || !t.is_contiguous()) {
    PyErr_SetString(PyExc_AssertionError, "device tensors must be contiguous CUDA tensors");
    return false;
  }
  out = reinterpret_cast<int64_t>(t.data_ptr());
  return true;
}

bool convert(PyObject* o, bool pointer, int64_t& out) {
  if (PyLong_Check(o)) {
    // device addresses and sizes below 2^64
    out = static_cast<int64_t>(PyLong_AsUnsignedLongLongMask(o));
    return !PyErr_Occurred();
  }
  if (pointer && o == Py_None) {
    out = 0;
    return true;
  }
  if (pointer && THPVariable_Check(o)) return tensor_pointer(o, out);
  if (!pointer && PyIndex_Check(o)) {
    PyObject* i = PyNumber_Index(o);
    if (i == nullptr) return false;
    out = static_cast<int64_t>(PyLong_AsUnsignedLongLongMask(i));
    Py_DECREF(i);
    return !PyErr_Occurred();
  }
  PyErr_Format(PyExc_TypeError, "unsupported argument type %s", Py_TYPE(o)->tp_name);
  return false;
}

// The handle args[0] and the arguments behind it, `missing` fewer than the
// entry has.
bool arguments(PyObject* const* args, Py_ssize_t n, int missing, const Entry*& entry, int64_t* v) {
  entry = n < 1 ? nullptr : static_cast<const Entry*>(PyLong_AsVoidPtr(args[0]));
  if (entry == nullptr) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "no entry");
    return false;
  }
  if (n - 1 != entry->args - missing) {
    PyErr_Format(PyExc_TypeError, "entry takes %d arguments (%zd given)", entry->args - missing, n - 1);
    return false;
  }
  for (Py_ssize_t i = 1; i < n; ++i)
    if (!convert(args[i], (entry->pointers >> (i - 1)) & 1, v[i - 1])) return false;
  return true;
}

PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2) {
    PyErr_SetString(PyExc_TypeError, "entry(address, kinds) expected");
    return nullptr;
  }
  Entry e{PyLong_AsVoidPtr(args[0]), 0, 0};
  Py_ssize_t count = 0;
  const char* kinds = PyErr_Occurred() ? nullptr : PyUnicode_AsUTF8AndSize(args[1], &count);
  if (kinds == nullptr) return nullptr;
  if (e.f == nullptr || count > kMaxArgs) {
    PyErr_SetString(PyExc_ValueError, "no entry, or more than 24 parameters");
    return nullptr;
  }
  e.args = static_cast<int>(count);
  for (int i = 0; i < e.args; ++i) e.pointers |= static_cast<uint32_t>(kinds[i] == 'p') << i;
  g_entries.push_back(e);
  return PyLong_FromVoidPtr(&g_entries.back());
  END_HANDLE_TH_ERRORS
}

PyObject* launch(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Entry* entry;
  int64_t v[kMaxArgs];
  if (!arguments(args, n, 1, entry, v)) return nullptr;
  PyObject* device = PyObject_CallNoArgs(g_device);
  if (device == nullptr) return nullptr;
  PyObject* stream = PyObject_CallOneArg(g_raw_stream, device);
  Py_DECREF(device);
  if (stream == nullptr) return nullptr;
  const bool ok = convert(stream, true, v[n - 1]);
  Py_DECREF(stream);
  if (!ok) return nullptr;
  const Invoker call = pick(static_cast<size_t>(n), std::make_index_sequence<kMaxArgs + 1>{});
  int32_t rc;
  Py_BEGIN_ALLOW_THREADS
  rc = static_cast<int32_t>(call(entry->f, v));
  Py_END_ALLOW_THREADS
  if (rc != 0) {
    PyObject* r = PyObject_CallFunction(g_check, "i", rc);
    if (r == nullptr) return nullptr;
    Py_DECREF(r);
  }
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

PyObject* value(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Entry* entry;
  int64_t v[kMaxArgs];
  if (!arguments(args, n, 0, entry, v)) return nullptr;
  return PyLong_FromLongLong(pick(static_cast<size_t>(n - 1), std::make_index_sequence<kMaxArgs + 1>{})(entry->f, v));
  END_HANDLE_TH_ERRORS
}

PyObject* pointer(PyObject*, PyObject* o) {
  HANDLE_TH_ERRORS
  int64_t p;
  if (!THPVariable_Check(o)) {
    PyErr_SetString(PyExc_TypeError, "tensor expected");
    return nullptr;
  }
  if (!tensor_pointer(o, p)) return nullptr;
  return PyLong_FromUnsignedLongLong(static_cast<uint64_t>(p));
  END_HANDLE_TH_ERRORS
}

PyObject* empty(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n < 3 || n > 6 || !THPVariable_Check(args[0]) || !THPDtype_Check(args[1])) {
    PyErr_SetString(PyExc_TypeError, "empty(like, dtype, *sizes) expects a tensor, a dtype and one to four sizes");
    return nullptr;
  }
  int64_t sizes[4];
  for (Py_ssize_t i = 2; i < n; ++i) {
    sizes[i - 2] = PyLong_AsLongLong(args[i]);
    if (sizes[i - 2] == -1 && PyErr_Occurred()) return nullptr;
  }
  const at::Tensor& like = THPVariable_Unpack(args[0]);
  at::Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    out = at::empty(at::IntArrayRef(sizes, static_cast<size_t>(n - 2)),
                    at::TensorOptions().device(like.device()).dtype(
                        reinterpret_cast<THPDtype*>(args[1])->scalar_type));
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

PyObject* set_check(PyObject*, PyObject* o) {
  Py_XINCREF(o);
  Py_XSETREF(g_check, o);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"entry", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry)), METH_FASTCALL, nullptr},
    {"launch", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&launch)), METH_FASTCALL, nullptr},
    {"value", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&value)), METH_FASTCALL, nullptr},
    {"pointer", &pointer, METH_O, nullptr},
    {"empty", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&empty)), METH_FASTCALL, nullptr},
    {"set_check", &set_check, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "clef_host", nullptr, -1, methods};

}  // namespace

namespace {

// The functions above use torch's and Python's class layouts as their headers
// gave them: no other version of either loads this module. (Written with
// functions of Python's stable interface only.)
bool built_for_this_process() {
#define CLEF_STR2(x) #x
#define CLEF_STR(x) CLEF_STR2(x)
  constexpr const char* python = CLEF_STR(PY_MAJOR_VERSION) "." CLEF_STR(PY_MINOR_VERSION) ".";
  PyObject* torch = PyImport_ImportModule("torch");
  PyObject* version = torch != nullptr ? PyObject_GetAttrString(torch, "__version__") : nullptr;
  PyObject* text = version != nullptr ? PyObject_Str(version) : nullptr;
  const char* found = text != nullptr ? PyUnicode_AsUTF8AndSize(text, nullptr) : nullptr;
  const bool same = found != nullptr && std::strcmp(found, CLEF_TORCH_VERSION) == 0 &&
                    std::strncmp(Py_GetVersion(), python, std::strlen(python)) == 0;
  if (found != nullptr && !same)
    PyErr_Format(PyExc_ImportError,
                 "the call module was built for torch %s and Python %sx, this is torch %s and Python %s; run `make -C "
                 "clef-hrx_amd`",
                 CLEF_TORCH_VERSION, python, found, Py_GetVersion());
  Py_XDECREF(text);
  Py_XDECREF(version);
  Py_XDECREF(torch);
  return same;
}

}  // namespace

PyMODINIT_FUNC PyInit_clef_host() {
  if (!built_for_this_process()) return nullptr;
  PyObject* c = PyImport_ImportModule("torch._C");
  if (c == nullptr) return nullptr;
  g_device = PyObject_GetAttrString(c, "_cuda_getDevice");
  g_raw_stream = g_device != nullptr ? PyObject_GetAttrString(c, "_cuda_getCurrentRawStream") : nullptr;
  Py_DECREF(c);
  if (g_raw_stream == nullptr) return nullptr;
  PyObject* m = PyModule_Create(&module_def);
  if (m != nullptr) PyModule_AddStringConstant(m, "build_id", CLEF_BUILD_ID);
  return m;
}

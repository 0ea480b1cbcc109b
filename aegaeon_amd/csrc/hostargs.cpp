// aegaeon_amd._hostargs: the argument tables of a move, read from Python
// objects in one pass.
//
// A copy over 72 backing tensors asks each for its device, layout, size and
// address. Asked from Python one attribute at a time that is 50 us, several
// times what the copy of one block takes; here it is 2. Both functions return
// None for anything but the plain case (a list of dense device tensors, a
// list of Python integers), and the caller then takes the general path, which
// names what is wrong or converts other kinds of sequences.

#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstring>

namespace {

struct Ref {  // owned reference
  PyObject* p;
  explicit Ref(PyObject* o) : p(o) {}
  ~Ref() { Py_XDECREF(p); }
  PyObject* release() {
    PyObject* o = p;
    p = nullptr;
    return o;
  }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
};

// A list or tuple, whose items stay where they are while none of the code
// here runs Python code.
bool plain_sequence(PyObject* o) { return PyList_CheckExact(o) || PyTuple_CheckExact(o); }

// segment_table(segments, num_blocks) -> (device index, num_blocks, addresses,
// page bytes), the last two as packed 8-byte values, or None. num_blocks None:
// the first tensor's leading size. A page is a tensor's bytes / num_blocks.
PyObject* segment_table(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 2) {
    PyErr_SetString(PyExc_TypeError, "segment_table(segments, num_blocks)");
    return nullptr;
  }
  PyObject* seq = args[0];
  if (!plain_sequence(seq)) Py_RETURN_NONE;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
  PyObject** items = PySequence_Fast_ITEMS(seq);
  if (n == 0) Py_RETURN_NONE;
  int64_t blocks = 0;
  if (args[1] != Py_None) {
    if (!PyLong_CheckExact(args[1])) Py_RETURN_NONE;
    int overflow = 0;
    blocks = PyLong_AsLongLongAndOverflow(args[1], &overflow);
    if (overflow) Py_RETURN_NONE;
  }
  Ref bases(PyBytes_FromStringAndSize(nullptr, n * 8));
  Ref pages(PyBytes_FromStringAndSize(nullptr, n * 8));
  if (!bases.p || !pages.p) return nullptr;
  int device = -1;
  try {
    for (Py_ssize_t i = 0; i < n; ++i) {
      if (!THPVariable_CheckExact(items[i])) Py_RETURN_NONE;
      const at::Tensor& t = THPVariable_Unpack(items[i]);
      if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.is_contiguous())
        Py_RETURN_NONE;
      const int on = static_cast<int>(t.get_device());
      if (i == 0) {
        device = on;
        if (args[1] == Py_None) {
          if (t.dim() == 0) Py_RETURN_NONE;
          blocks = t.size(0);
        }
        if (blocks <= 0) Py_RETURN_NONE;
      }
      if (on != device) Py_RETURN_NONE;
      const int64_t page = static_cast<int64_t>(t.nbytes()) / blocks;
      const void* base = t.data_ptr();
      std::memcpy(PyBytes_AS_STRING(bases.p) + 8 * i, &base, 8);
      std::memcpy(PyBytes_AS_STRING(pages.p) + 8 * i, &page, 8);
    }
  } catch (...) {
    Py_RETURN_NONE;  // the general path meets the same error and reports it
  }
  return Py_BuildValue("iLNN", device, static_cast<long long>(blocks), bases.release(),
                       pages.release());
}

// pack_ids(ids) -> the packed 8-byte values of a list of Python integers, or None.
PyObject* pack_ids(PyObject*, PyObject* seq) {
  if (!plain_sequence(seq)) Py_RETURN_NONE;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
  PyObject** items = PySequence_Fast_ITEMS(seq);
  Ref out(PyBytes_FromStringAndSize(nullptr, n * 8));
  if (!out.p) return nullptr;
  char* to = PyBytes_AS_STRING(out.p);
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (!PyLong_CheckExact(items[i])) Py_RETURN_NONE;  // booleans and numpy integers too
    int overflow = 0;
    const long long v = PyLong_AsLongLongAndOverflow(items[i], &overflow);
    if (overflow) Py_RETURN_NONE;
    std::memcpy(to + 8 * i, &v, 8);
  }
  return out.release();
}

// pack_ids32(ids, limit) -> the packed 4-byte values of a list of Python
// integers, each in [0, limit), or None.
PyObject* pack_ids32(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 2) {
    PyErr_SetString(PyExc_TypeError, "pack_ids32(ids, limit)");
    return nullptr;
  }
  const int64_t limit = PyLong_AsLongLong(args[1]);
  if (limit == -1 && PyErr_Occurred()) return nullptr;
  PyObject* seq = args[0];
  if (!plain_sequence(seq)) Py_RETURN_NONE;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
  PyObject** items = PySequence_Fast_ITEMS(seq);
  Ref out(PyBytes_FromStringAndSize(nullptr, n * 4));
  if (!out.p) return nullptr;
  char* to = PyBytes_AS_STRING(out.p);
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (!PyLong_CheckExact(items[i])) Py_RETURN_NONE;
    int overflow = 0;
    const long long v = PyLong_AsLongLongAndOverflow(items[i], &overflow);
    if (overflow || v < 0 || v >= limit || v > INT32_MAX) Py_RETURN_NONE;
    const int32_t x = static_cast<int32_t>(v);
    std::memcpy(to + 4 * i, &x, 4);
  }
  return out.release();
}

template <typename F>
PyCFunction as_method(F* f) {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f));
}

PyMethodDef methods[] = {
    {"segment_table", as_method(segment_table), METH_FASTCALL, nullptr},
    {"pack_ids32", as_method(pack_ids32), METH_FASTCALL, nullptr},
    {"pack_ids", pack_ids, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_hostargs", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

// torch_version: the torch whose tensor layout this was compiled against.
PyMODINIT_FUNC PyInit__hostargs() {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", AEGKV_TORCH_VERSION) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}

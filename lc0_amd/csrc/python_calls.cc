// The calls that a Python program makes once per position, as a CPython extension: through ctypes a call costs several times the copy
// that it asks for. lc0_amd/backend.py takes these where the arguments are plain arrays and falls back to its own checks and
// conversions, and to the library's error messages, for everything else.
// us for 300 positions with their moves, one at a time: ctypes 720, this 176.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <cstring>

#include "../../include/lc0mi.h"

namespace {

constexpr long kDone = 0, kNotHandled = 1, kError = -1;
constexpr Py_ssize_t kPlanes = 112;

// A C-contiguous native array of `dims` dimensions and one of the given element formats.
class Array {
 public:
  Array(PyObject* o, int dims, Py_ssize_t itemsize, const char* formats) {
    if (PyObject_GetBuffer(o, &view_, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT) != 0) {
      PyErr_Clear();
      return;
    }
    held_ = true;
    const char* f = view_.format;
    ok_ = view_.ndim == dims && view_.itemsize == itemsize && f != nullptr && f[0] != 0 && f[1] == 0 && std::strchr(formats, f[0]) != nullptr;
  }
  Array(const Array&) = delete;
  Array& operator=(const Array&) = delete;
  ~Array() {
    if (held_) PyBuffer_Release(&view_);
  }
  bool ok() const { return ok_; }
  Py_ssize_t size(int dim) const { return view_.shape[dim]; }
  template <typename T>
  const T* data() const { return static_cast<const T*>(view_.buf); }

 private:
  Py_buffer view_;
  bool held_ = false, ok_ = false;
};

lc0mi_comp* Handle(PyObject* o) {
  void* h = PyLong_AsVoidPtr(o);
  if (h == nullptr) PyErr_Clear();
  return static_cast<lc0mi_comp*>(h);
}

// add_inputs(computation, masks u64 [n][112], values f32 [n][112])
PyObject* AddInputs(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  if (n_args != 3) return PyLong_FromLong(kNotHandled);
  lc0mi_comp* comp = Handle(args[0]);
  Array masks(args[1], 2, 8, "LQ"), values(args[2], 2, 4, "f");
  if (comp == nullptr || !masks.ok() || !values.ok() || masks.size(1) != kPlanes || values.size(1) != kPlanes ||
      masks.size(0) != values.size(0) || masks.size(0) < 1 || masks.size(0) > INT32_MAX) {
    return PyLong_FromLong(kNotHandled);
  }
  const int n = static_cast<int>(masks.size(0));
  const uint64_t* m = masks.data<uint64_t>();
  const float* v = values.data<float>();
  int rc;
  if (n <= 16) {
    rc = lc0mi_comp_add_inputs(comp, n, m, v);
  } else {   // (a copy long enough for other threads to run meanwhile)
    Py_BEGIN_ALLOW_THREADS
    rc = lc0mi_comp_add_inputs(comp, n, m, v);
    Py_END_ALLOW_THREADS
  }
  return PyLong_FromLong(rc == 0 ? kDone : kError);
}

// add_legal_moves(computation, ids u16 [n])
PyObject* AddLegalMoves(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  if (n_args != 2) return PyLong_FromLong(kNotHandled);
  lc0mi_comp* comp = Handle(args[0]);
  Array ids(args[1], 1, 2, "H");
  if (comp == nullptr || !ids.ok() || ids.size(0) < 1 || ids.size(0) > INT32_MAX) return PyLong_FromLong(kNotHandled);
  return PyLong_FromLong(lc0mi_comp_add_legal_moves(comp, static_cast<int>(ids.size(0)), ids.data<uint16_t>()) == 0 ? kDone : kError);
}

PyMethodDef kMethods[] = {
    {"add_inputs", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(AddInputs)), METH_FASTCALL, nullptr},
    {"add_legal_moves", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(AddLegalMoves)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() { return PyModule_Create(&kModule); }
